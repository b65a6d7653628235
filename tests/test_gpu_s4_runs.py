"""Whole 4th-order runs against the oracle, byte for byte, at the sizes where the stages' quads
change: one quad a row, slabs that end on a quad and within one, more rows than the stripe
limit, material indices and float coefficients."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

NAMES = ("ex", "ey", "ez", "hx", "hy", "hz")


@pytest.mark.parametrize("shape,npml,kind", [
    ((4, 6, 5), 0, "float"), ((16, 20, 18), 0, "const"), ((24, 26, 28), 7, "index"), ((64, 71, 24), 8, "const"),
    ((68, 72, 26), 10, "float"), ((132, 75, 30), 9, "index"), ((40, 80, 33), 12, "float"), ((260, 30, 26), 5, "index"),
])
def test_run_equals_oracle(shape, npml, kind):
    from fdtd_accelerate_amd.s4 import S4Sim
    nx, ny, nz = shape
    S = 0.6
    rng = np.random.default_rng(sum(shape))
    c0 = np.float32(S / 24)
    ces = None
    if kind == "index":
        vals = (c0 / np.array([1, 2, 4, 6], np.float32)).astype(np.float32)
        ces = [np.asfortranarray(vals[rng.integers(0, 4, shape)]) for _ in range(3)]
    elif kind == "float":
        ces = [np.asfortranarray((c0 / rng.uniform(1, 5, shape)).astype(np.float32)) for _ in range(3)]
    chs = [np.asfortranarray((c0 * rng.uniform(0.5, 1, shape)).astype(np.float32)) for _ in range(3)] if kind == "float" else None
    o = O.OracleS4Sim(nx, ny, nz, S, npml=npml, ces=ces, chs=chs)
    g = S4Sim(nx, ny, nz, S=S, npml=npml)
    if ces is not None:
        g.set_ce(*ces)
        assert kind != "index" or g.ce_mat is not None
    if chs is not None:
        g.set_ch(*chs)
    for k, name in enumerate(NAMES):
        f = np.asfortranarray(rng.standard_normal(shape).astype(np.float32))
        o.ehs[k][:] = f
        g.set_field(name, f)
    tf = lambda t: O.pulse(t, 3.0, 2.0, 4.0)  # noqa: E731
    for s in (o, g):
        s.add_source("ez", (1, 2, 3), (1, 2, 3), tf)
        s.add_source("ex", (0, ny // 2, 1), (nx - 1, ny // 2, 2), tf,
                     np.linspace(0.1, 1.0, 2 * nx, dtype=np.float32).reshape(nx, 1, 2))
        s.add_probe("ey", (nx - 1, 1, nz // 2))
        s.add_probe("hx", (nx // 2, ny - 2, 2))
    series = g.run(3)
    o.run(3)
    for k, name in enumerate(NAMES):
        assert o.ehs[k].tobytes() == np.asfortranarray(g.field(name).cpu().numpy()).tobytes(), name
    assert series.tobytes() == np.array(o.series, np.float32).tobytes()
    for key in (o.psiE if npml else {}):
        for c in range(2):
            for od, gd in ((o.psiE, g.psiE), (o.psiH, g.psiH)):
                got = np.asfortranarray(gd[key][c].cpu().numpy().transpose(2, 1, 0))
                assert od[key][c].tobytes() == got.tobytes(), (key, c)
