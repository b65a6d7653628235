"""The fused engine's whole-grid steps and the rules that choose them and the sweep's tile."""
import numpy as np
import pytest
import torch

from fdtd_accelerate_amd import autotune

NAMES = ("ex", "ey", "ez", "hx", "hy", "hz")


@pytest.mark.parametrize("n", [(2, 2, 16), (7, 300, 64), (24, 20, 48), (130, 31, 96), (256, 256, 256), (384, 384, 384),
                               (512, 512, 512), (1000, 700, 1024), (3000, 90, 64)])
@pytest.mark.parametrize("npml", [0, 4, 12])
def test_tile_rule(n, npml):
    """The chosen tile has rows and planes inside the box and fits the LDS with the largest
    CE table (MAX_CE_TRI triples)."""
    from fdtd_accelerate_amd import _lib
    T, CX = autotune.heuristic(*n, npml)
    assert 1 <= T <= 13 and 1 <= CX <= min(64, n[0])
    assert T == 1 or T <= n[1] // 2
    assert autotune.lds_fits(T, CX, True) and autotune.lds_fits(T, CX, True, _lib.MAX_CE_TRI)


def _sims(ns, npml, ce, feature, probe, kw):
    from fdtd_accelerate_amd import Drude, Pbc, Tfsf
    from fdtd_accelerate_amd.sim import YeeSim
    from fdtd_accelerate_amd.sources import gaussian_pulse
    rng = np.random.default_rng(11)
    nx, ny, nz = ns
    eh = [rng.standard_normal(ns).astype(np.float32) for _ in range(6)]
    cc = [(0.5 / rng.integers(1, 7, ns)).astype(np.float32) for _ in range(3)]
    out = []
    for engine in ("kemp", "fused"):
        faces = ("", "", "fb") if "pbc" in feature else ("fb", "fb", "fb")
        s = YeeSim(*ns, npml=npml, coeff_use="" if ce == "none" else "e", engine=engine, cpml_faces=faces,
                   fused_params=kw if engine == "fused" else None)
        s.fields.set_ehs(*eh)
        if ce != "none":
            s.set_ce(*cc)
            if ce == "index":
                assert s.fields.compress_ce()
        if "pbc" in feature:
            Pbc(s.fields, "xy")
        if "drude" in feature:
            Drude(s.fields, [2, 1, 3], [nx - 3, ny // 2, nz - 2], 0.5, 0.05)
        if "tfsf" in feature:
            Tfsf(s.fields, [nx // 4, ny // 4, nz // 4], [nx - nx // 4, ny - ny // 4, nz - nz // 4], ("fb", "fb", "fb"),
                 9.0, ("normal", "xyz"[nz % 3]))
        c = (nx // 2, ny // 2, nz // 2)
        s.add_source("ez", c, c, gaussian_pulse(4.0, 3.0, 5.0))
        s.add_source("hx", c, (c[0] + 1, c[1], c[2] + 4), gaussian_pulse(3.0, 3.0, 5.0), 0.5)
        s.add_probe("ex", probe)
        s.add_probe("hz", (nx // 2, ny // 2, nz // 2))
        out.append(s)
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("ns,npml,ce,feature,kw", [
    ((24, 75, 130), 5, "index", "", {}),
    ((23, 40, 57), 4, "float", "drude", {}),
    ((30, 73, 131), 6, "index", "tfsf", {}),
    ((31, 28, 96), 4, "none", "tfsf drude", {"z_phase": 20}),
    ((20, 26, 45), 0, "float", "tfsf", {}),
    ((25, 22, 64), 0, "index", "drude", {}),
    ((21, 74, 160), 5, "index", "pbc", {}),
    ((22, 24, 61), 0, "none", "pbc", {}),
    ((28, 80, 320), 12, "float", "pbc", {"z_phase": 8}),
])
def test_whole_grid_equals_inplace(ns, npml, ce, feature, kw):
    """Whole-grid steps equal the in-place engine in every field, psi, current, line and
    probe value (0 == -0), also after a sweep run in between."""
    a, b = _sims(ns, npml, ce, feature, (1, ns[1] // 2, ns[2] // 3), dict(kw, whole_grid=True))
    same = lambda x, y: torch.equal(x, y) and not torch.isnan(x).any()
    for steps in (3, 4):
        ra, rb = a.run(steps), b.run(steps)
        assert b._fused.whole_grid
        assert np.array_equal(ra, rb)
        for n in NAMES:
            assert same(a.field(n), b.field(n)), n
        if npml:
            assert same(a.cpml.psiE_buf, b.cpml.psiE_buf) and same(a.cpml.psiH_buf, b.cpml.psiH_buf)
        for x, y in zip(a.fields.instance_list, b.fields.instance_list):
            for name in ("line_e", "line_h", "abc"):
                if hasattr(x, name):
                    assert same(getattr(x, name), getattr(y, name)), name
            for u, v in zip(getattr(x, "J", ()), getattr(y, "J", ())):
                assert same(u, v)
        a.run(1)  # a timed run takes the sweep and leaves the state in the other buffers
        b._fused.run(1, None, time_kernel=True)
        b.tstep += 1


@pytest.mark.gpu
def test_whole_grid_choice():
    """Small grids step over the whole grid by default, a tile that the caller gives keeps the
    sweep, and step pairs exclude whole-grid steps."""
    from fdtd_accelerate_amd.sim import YeeSim
    s = YeeSim(40, 40, 40, npml=6, coeff_use="", engine="fused")
    s.run(1)
    assert s._fused.whole_grid
    s = YeeSim(40, 40, 40, npml=6, coeff_use="", engine="fused", fused_params={"rows_per_thread": 3})
    s.run(1)
    assert not s._fused.whole_grid
    s = YeeSim(40, 40, 40, npml=6, coeff_use="", engine="fused", fused_params={"step_pairs": True, "whole_grid": True})
    with pytest.raises(ValueError, match="pairs"):
        s.run(1)
