"""What the joined half steps read and write beyond the cells they update."""
import ctypes
import os
import subprocess

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_z_face_loads_stay_in_the_z_faces(tmp_path):
    """With CPML on z alone no psi load leaves the z faces (tests/zface_reach.cpp)."""
    exe = str(tmp_path / "zface_reach")
    subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "-std=c++17", "-O1", "-I",
                    os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "zface_reach.cpp"), "-o", exe], check=True,
                   capture_output=True, timeout=600)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and "zface reach ok" in out.stdout, out.stdout + out.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("ns,npml", [((10, 11, 33), 4), ((14, 75, 40), 6), ((8, 9, 24), 1)])
def test_psi_of_the_z_faces_alone(ns, npml):
    """A psi allocation of the z faces only, in their packed order, gives the separate calls'
    fields and psi byte for byte."""
    from fdtd_accelerate_amd import Fields, _lib
    out = []
    for joined in (True, False):
        torch.manual_seed(2)
        f = Fields(*ns, coeff_use="")
        nx, ny, nzp = f.ns_pitch
        size = nx * ny * npml
        for t in f.ehs:
            t[:, :, :ns[2]].normal_()
        psi = [torch.randn(4 * size, device=f.device) for _ in range(2)]
        tab = torch.rand(2, 2 * (npml + 1), device=f.device)
        halves = []
        for p in psi:
            h = _lib.CpmlHalf()
            h.npml, h.b, h.a = npml, tab[0].data_ptr(), tab[1].data_ptr()
            for face, (o1, o2) in ((4, (0, 1)), (5, (2, 3))):
                h.psi1[face], h.psi2[face] = p.data_ptr() + 4 * size * o1, p.data_ptr() + 4 * size * o2
            halves.append(h)
        E, N, st = f.ptrs(f.ehs), (None,) * 3, _lib.stream_handle(f.stream)
        grid = (nx, ny, nzp, f.pad)
        torch.cuda.synchronize()
        for _ in range(2):
            if joined:
                _lib.call("mifdtd_half_e", *grid, ctypes.byref(halves[0]), *E, *N, *N, None, None, st)
                _lib.call("mifdtd_half_h", *grid, ctypes.byref(halves[1]), *E, *N, st)
            else:
                _lib.call("mifdtd_update_e", *grid, *E, *N, st)
                _lib.call("mifdtd_cpml_e", *grid, ctypes.byref(halves[0]), *E, *N, st)
                _lib.call("mifdtd_update_h", *grid, *E, *N, st)
                _lib.call("mifdtd_cpml_h", *grid, ctypes.byref(halves[1]), *E, *N, st)
        torch.cuda.synchronize()
        out.append([*f.ehs, *psi])
    for x, y in zip(*out):
        assert torch.equal(x.view(torch.int32), y.view(torch.int32))
