"""The 4th-order stage kernels at the sizes where their quads can go wrong: rows of one quad
run, rows cut at lines with CPML slabs that do and do not end on one, more and fewer rows
than the stripe limit, sources and probes at the edges; whole steps against the oracle byte
for byte, and the one-call form against the single stage calls."""
import ctypes
import os
import subprocess

import numpy as np
import pytest
import torch

from oracle import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _pair(shape, npml, kind, seed=4):
    from fdtd_accelerate_amd.s4 import S4Sim
    rng = np.random.default_rng(seed)
    S = 0.6
    fields = [rng.standard_normal(shape).astype(np.float32) for _ in range(6)]
    if kind == "index":
        ce = [(np.float32(S / 24) / rng.integers(1, 7, shape).astype(np.float32)).astype(np.float32) for _ in range(3)]
    else:
        ce = [(np.float32(S / 24) / rng.uniform(1, 5, shape)).astype(np.float32) for _ in range(3)]
    sims = []
    for _ in range(2):
        g = S4Sim(*shape, S=S, npml=npml)
        if kind != "const":
            g.set_ce(*ce)
            assert kind != "index" or g.ce_mat is not None
        for n, f in zip(("ex", "ey", "ez", "hx", "hy", "hz"), fields):
            g.set_field(n, f)
        nx, ny, nz = shape
        tf = lambda t: O.pulse(t, 3.0, 2.0, 4.0)  # noqa: E731
        g.add_source("ez", (1, 2, 3), (1, 2, 3), tf)
        g.add_source("ex", (0, ny // 2, 1), (nx - 1, ny // 2, 2), tf,
                     np.linspace(0.1, 1.0, 2 * nx, dtype=np.float32).reshape(nx, 1, 2))
        g.add_probe("ey", (nx - 1, 1, nz // 2))
        g.add_probe("hx", (nx // 2, ny - 2, 2))
        g.add_probe("ez", (1, 2, 3))
        sims.append(g)
    return sims


@pytest.mark.gpu
@pytest.mark.parametrize("shape,npml,kind", [
    ((4, 6, 5), 0, "float"), ((16, 20, 18), 0, "const"), ((24, 26, 28), 7, "index"), ((64, 71, 24), 8, "const"),
    ((68, 72, 26), 10, "float"), ((132, 75, 30), 9, "index"), ((40, 80, 33), 12, "float"), ((260, 30, 26), 5, "index"),
])
def test_whole_steps_equal_stage_calls(shape, npml, kind):
    a, b = _pair(shape, npml, kind)
    steps = 3
    ra = a.run(steps)
    buf = torch.zeros((steps, 3), dtype=torch.float32, device="cuda")
    for t in range(steps):
        b.step(buf, t)
    assert ra.tobytes() == buf.cpu().numpy().tobytes()
    assert a.tstep == b.tstep
    for x, y in zip(a.ehs, b.ehs):
        assert torch.equal(x.view(torch.int32), y.view(torch.int32))
    for key in (a.psiE if npml else {}):
        for q in range(2):
            assert torch.equal(a.psiE[key][q].view(torch.int32), b.psiE[key][q].view(torch.int32))
            assert torch.equal(a.psiH[key][q].view(torch.int32), b.psiH[key][q].view(torch.int32))


@pytest.mark.gpu
def test_more_sources_than_one_call_holds():
    """Five sources: run() falls back to single stages, with the same result as source by source."""
    from fdtd_accelerate_amd.s4 import S4Sim
    g = S4Sim(32, 24, 20, npml=4)
    for n in range(5):
        g.add_source("ez", (8 + n, 9, 10), (8 + n, 9, 10), lambda t: O.pulse(t, 2.0, 2.0, 4.0))
    g.add_probe("ez", (10, 9, 10))
    s = g.run(4)
    assert s.shape == (4, 1) and np.isfinite(s).all() and np.abs(s).max() > 0


def test_descriptor_mirrors_header(tmp_path):
    """The ctypes mirror of mifdtd_s4_desc has the header's size and offsets."""
    from fdtd_accelerate_amd import _lib
    names = [f for f, _ in _lib.S4Desc._fields_]
    src = tmp_path / "p.c"
    src.write_text('#include <stdio.h>\n#include <stddef.h>\n#include "mifdtd.h"\nint main(void){printf("%zu",sizeof(mifdtd_s4_desc));'
                   + "".join(f'printf(" %zu",offsetof(mifdtd_s4_desc,{n}));' for n in names) + "return 0;}\n")
    exe = tmp_path / "p"
    subprocess.run(["gcc", "-std=c11", "-I", os.path.join(ROOT, "include"), "-I", "/opt/rocm/include", str(src), "-o", str(exe)],
                   check=True, capture_output=True)
    got = [int(v) for v in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()]
    assert got == [ctypes.sizeof(_lib.S4Desc)] + [getattr(_lib.S4Desc, n).offset for n in names]
