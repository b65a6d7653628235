"""The double core where planes of few rows keep memory order: the range kernel's values and
masks against the fields' own definition in float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _update_e(e, h, c):
    ex, ey, ez = (x.copy() for x in e)
    hx, hy, hz = h
    i, j, k = slice(0, -1), slice(0, -1), slice(0, -1)
    ex[:, j, k] += c[0][:, j, k] * ((hz[:, 1:, k] - hz[:, j, k]) - (hy[:, j, 1:] - hy[:, j, k]))
    ey[i, :, k] += c[1][i, :, k] * ((hx[i, :, 1:] - hx[i, :, k]) - (hz[1:, :, k] - hz[i, :, k]))
    ez[i, j] += c[2][i, j] * ((hy[1:, j] - hy[i, j]) - (hx[i, 1:] - hx[i, j]))
    ex[:, j, -1] *= 0.0  # the core's masked cells
    ey[i, :, -1] *= 0.0
    return ex, ey, ez


@pytest.mark.parametrize("ns", [(2, 2, 2), (3, 71, 4), (3, 72, 4), (5, 7, 130), (4, 70, 515), (9, 40, 66)])
@pytest.mark.parametrize("coeff", ["", "e"])
def test_small_planes_equal_the_definition(ns, coeff):
    from fdtd_accelerate_amd import Core, Fields
    rng = np.random.default_rng(6)
    f = Fields(*ns, coeff_use=coeff, precision_float="double", segment_nbytes=16)
    Core(f)
    eh = [rng.standard_normal(ns) for _ in range(6)]
    ce = [rng.uniform(0.1, 0.5, ns) if coeff else np.full(ns, 0.5) for _ in range(3)]
    f.set_ehs(*eh)
    if coeff:
        f.set_ces(*ce)
    f.update_e()
    want = _update_e(eh[:3], eh[3:], ce)
    for x, y in zip(f.ehs[:3], want):
        assert np.array_equal(x.cpu().numpy()[:, :, :ns[2]], y)
