"""Time functions of the 4th-order sources."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_time_functions_are_called_in_the_order_of_the_steps():
    """run() calls the sources' functions as step() does: step after step, stage after stage,
    source after source, so functions that share a state (one random generator here) give the
    same values."""
    from fdtd_accelerate_amd.s4 import S4Sim
    out, calls = [], []
    for whole in (True, False):
        g = S4Sim(24, 20, 18, npml=4)
        rng = np.random.default_rng(5)
        seen = []

        def noise(which):
            def f(t):
                seen.append((which, round(t, 3)))
                return rng.standard_normal()
            return f

        g.add_source("ez", (12, 10, 9), (12, 10, 9), noise(0))
        g.add_source("ex", (8, 9, 9), (9, 10, 9), noise(1), 0.5)
        if whole:
            g.run(3)
        else:
            for _ in range(3):
                g.step()
        calls.append(seen)
        out.append(g.ehs)
    assert calls[0] == calls[1]
    for x, y in zip(*out):
        assert torch.equal(x.view(torch.int32), y.view(torch.int32)) and x.abs().max() > 0
