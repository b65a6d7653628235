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


def _shared(shape, first, second):
    """Arrays first and second of one allocation, the last plane of the one the first plane of
    the other."""
    n, plane = shape[0], shape[1] * shape[2]
    block = torch.empty((2 * n - 1) * plane, device="cuda")
    a, b = block[:n * plane].view(shape), block[(n - 1) * plane:].view(shape)
    a.copy_(first)
    b.copy_(second)
    return a, b


def _check_shared(call, arrays, out, inner, written):
    """``call`` on the six arrays, with the last plane of out[0] being the first plane of
    out[1]: it leaves one of the two alone, so both orders of writing give the plane of the
    array ``written``."""
    want = [t.clone() for t in arrays]
    call(want)
    got = [t.clone() for t in arrays]
    got[out[0]], got[out[1]] = _shared(arrays[0].shape, arrays[out[0]], arrays[out[1]])
    keep = -1 if written == 0 else 0
    if written == 0:  # the first array's last plane is the one that is updated
        got[out[0]][-1].copy_(arrays[out[0]][-1])
    call(got)
    torch.cuda.synchronize()
    same = lambda x, y: torch.equal(x.view(torch.int32), y.view(torch.int32))
    assert same(got[out[written]][keep], want[out[written]][keep])
    for c in inner:
        x, y = got[c], want[c]
        if c == out[0]:
            x, y = x[:-1], y[:-1]
        elif c == out[1]:
            x, y = x[1:], y[1:]
        assert same(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("ns,npml", [((6, 80, 20), 0), ((8, 30, 64), 0), ((24, 75, 40), 5), ((300, 80, 256), 0)])
def test_planes_not_updated_are_not_written(ns, npml):
    """update_e leaves ey of the last plane alone and update_h hy of the first, also with the
    CPML in the same pass: a plane that is such a one of one array and an updated one of
    another ends as the update leaves it."""
    from fdtd_accelerate_amd import Core, Fields, _lib
    from fdtd_accelerate_amd.cpml import Cpml
    f = Fields(*ns, coeff_use="")
    Core(f)
    cp = Cpml(f, npml) if npml else None
    torch.manual_seed(4)
    arrays = [torch.randn(tuple(f.ns_pitch), device=f.device) for _ in range(6)]
    st, N, grid = torch.cuda.current_stream().cuda_stream, (None,) * 3, (*f.ns_pitch, f.pad)

    def half(e):
        def call(a):
            p = [t.data_ptr() for t in a]
            if cp is None:
                _lib.call("mifdtd_update_e" if e else "mifdtd_update_h", *grid, *p, *N, st)
            elif e:
                cp.reset()
                _lib.call("mifdtd_half_e", *grid, cp._descE, *p, *N, *N, None, None, st)
            else:
                cp.reset()
                _lib.call("mifdtd_half_h", *grid, cp._descH, *p, *N, st)
        return call

    torch.cuda.synchronize()
    _check_shared(half(True), arrays, (1, 0), (0, 1, 2), 1)   # ey's last plane, ex's first
    _check_shared(half(False), arrays, (3, 4), (3, 4, 5), 0)  # hx's last plane, hy's first


@pytest.mark.gpu
@pytest.mark.parametrize("n", [(40, 80, 12), (16, 20, 9)])
def test_s4_rows_not_updated_are_not_written(n):
    """The 4th-order stages leave the last z plane alone: the same with that of ex and the
    first of ez, and of hx and hz."""
    from fdtd_accelerate_amd import _lib
    torch.manual_seed(5)
    arrays = [torch.randn(n[2], n[1], n[0], device="cuda") for _ in range(6)]
    st, N = torch.cuda.current_stream().cuda_stream, (None,) * 3

    def stage(name):
        def call(a):
            _lib.call(name, *n, 0.3, *[t.data_ptr() for t in a], *N, 0.03, st)
        return call

    torch.cuda.synchronize()
    _check_shared(stage("mifdtd_s4_update_e"), arrays, (0, 2), (0, 1, 2), 1)
    _check_shared(stage("mifdtd_s4_update_h"), arrays, (3, 5), (3, 4, 5), 1)
