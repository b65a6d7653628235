"""The float core on grids that it takes in memory order (planes of few rows, planes of nearly
a multiple of 8 blocks) and next to them, against the split form, byte for byte."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns", [
    (64, 138, 116),   # 47 quads short of two rounds of 8 blocks
    (66, 110, 74),    # 42 quads past one
    (97, 112, 76),    # 80 past
    (96, 72, 113),    # 40 past, the fewest rows with stripes
    (62, 71, 120),    # too few rows for stripes
    (60, 96, 96),     # 256 past: the whole-grid order
])
@pytest.mark.parametrize("coeff,index", [("", False), ("eh", False), ("e", True)])
def test_memory_order_equals_split_form(ns, coeff, index):
    from fdtd_accelerate_amd import Core, Fields
    from fdtd_accelerate_amd.core import CoreSplit
    out = []
    for cls in (Core, CoreSplit):
        gen = torch.Generator(device="cuda").manual_seed(12)
        f = Fields(*ns, coeff_use=coeff)
        cls(f)
        f.set_ehs(*[torch.randn(ns, device="cuda", generator=gen) for _ in range(6)])
        vals = torch.from_numpy((0.5 / np.random.default_rng(2).uniform(1, 6, 9)).astype(np.float32)).cuda()
        pick = lambda: vals[torch.randint(0, 9, ns, device="cuda", generator=gen)]
        if "e" in coeff:
            f.set_ces(*[pick() for _ in range(3)])
        if "h" in coeff:
            f.set_chs(*[pick() for _ in range(3)])
        if index and cls is Core:
            assert f.compress_ce()
        for _ in range(2):
            f.update_e()
            f.update_h()
        out.append(f.ehs)
    for x, y in zip(*out):
        assert torch.equal(x.view(torch.int32), y.view(torch.int32))
