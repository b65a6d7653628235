"""The double-precision core in the whole-grid order against the split form in memory order."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns", [(2, 2, 2), (3, 71, 3), (4, 72, 33), (5, 73, 128), (3, 97, 515), (2, 150, 1201)])
@pytest.mark.parametrize("coeff", ["", "eh"])
def test_whole_grid_equals_split_form(ns, coeff):
    from fdtd_accelerate_amd import Core, Fields
    from fdtd_accelerate_amd.core import CoreSplit
    out = []
    for cls in (Core, CoreSplit):
        rng = np.random.default_rng(9)
        f = Fields(*ns, coeff_use=coeff, precision_float="double", segment_nbytes=16)
        cls(f)
        f.set_ehs(*[rng.standard_normal(ns) for _ in range(6)])
        if coeff:
            f.set_ces(*[rng.uniform(0.1, 0.5, ns) for _ in range(3)])
            f.set_chs(*[rng.uniform(0.1, 0.5, ns) for _ in range(3)])
        for _ in range(3):
            f.update_e()
            f.update_h()
        out.append(f.ehs)
    for x, y in zip(*out):
        assert torch.equal(x.view(torch.int64), y.view(torch.int64))
