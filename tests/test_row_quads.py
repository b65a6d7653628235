"""The thread order of the whole-grid passes (csrc/row_quads.hpp), checked on the host, and
the passes on the GPU at the sizes where that order changes."""
import os
import subprocess

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_rows_are_covered(tmp_path):
    """Every quad of the grid is taken by exactly one thread, z-slab quads only in their own
    runs, and the neighbour flags hold exactly between neighbours (tests/row_cover.cpp)."""
    exe = str(tmp_path / "row_cover")
    subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "-std=c++17", "-O1", "-I",
                    os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "row_cover.cpp"), "-o", exe], check=True,
                   capture_output=True, timeout=600)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and "row cover ok" in out.stdout, out.stdout + out.stderr


def _pair(ns, npml, ce):
    from fdtd_accelerate_amd.sim import YeeSim
    from fdtd_accelerate_amd.sources import gaussian_pulse
    rng = np.random.default_rng(5)
    eh = [rng.standard_normal(ns).astype(np.float32) for _ in range(6)]
    cc = [(0.5 / rng.integers(1, 7, ns)).astype(np.float32) for _ in range(3)]
    out = []
    for engine in ("kemp", "slab"):
        s = YeeSim(*ns, npml=npml, coeff_use="" if ce == "none" else "e", engine=engine)
        s.fields.set_ehs(*eh)
        if ce != "none":
            s.set_ce(*cc)
            if ce == "index":
                assert s.fields.compress_ce()
        nx, ny, nz = ns
        s.add_source("ez", (nx // 2, ny // 2, 1), (nx // 2, ny // 2, nz - 2), gaussian_pulse(4.0, 3.0, 5.0))
        s.add_source("hx", (0, 1, 0), (nx - 1, 1, 2), gaussian_pulse(3.0, 3.0, 5.0), 0.5)
        s.add_probe("ex", (1, ny - 2, nz - 1))
        s.add_probe("hz", (nx - 1, ny // 2, 0))
        out.append(s)
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("ns,npml,ce", [
    ((5, 71, 33), 0, "none"), ((6, 72, 16), 0, "float"), ((7, 73, 30), 0, "index"),
    ((20, 75, 26), 8, "float"), ((21, 97, 64), 9, "index"), ((19, 80, 131), 6, "none"),
    ((26, 130, 57), 12, "index"), ((18, 72, 260), 4, "float"), ((12, 40, 1041), 3, "index"),
])
def test_slab_rows_equal_inplace(ns, npml, ce):
    """The slab engine equals the in-place one byte for byte around the stripe limit, with
    rows of one to five blocks, z slabs that end within a quad, and no z runs at all."""
    a, b = _pair(ns, npml, ce)
    ra, rb = a.run(5), b.run(5)
    assert ra.tobytes() == rb.tobytes()
    for x, y in zip(a.fields.ehs, b.fields.ehs):
        assert torch.equal(x.view(torch.int32), y.view(torch.int32))
    if npml:
        assert torch.equal(a.cpml.psiE_buf.view(torch.int32), b.cpml.psiE_buf.view(torch.int32))
        assert torch.equal(a.cpml.psiH_buf.view(torch.int32), b.cpml.psiH_buf.view(torch.int32))


@pytest.mark.gpu
def test_batch_groups_equal_single_runs():
    """Instances that fill more than one launch group (200 MiB of working set each) end as
    the same simulations run alone."""
    from fdtd_accelerate_amd.batch import BatchedYee
    shapes = [(150, 141, 150), (60, 50, 40), (131, 160, 170), (40, 90, 33)]
    pairs = [_pair(ns, 8, "float") for ns in shapes]
    bt = BatchedYee([b for _, b in pairs])
    series = bt.run(3)
    for (a, b), rb in zip(pairs, series):
        assert a.run(3).tobytes() == rb.tobytes()
        for x, y in zip(a.fields.ehs, b.fields.ehs):
            assert torch.equal(x.view(torch.int32), y.view(torch.int32))
    bt.close()
