"""The in-place half steps in one pass (core and CPML) against the range kernels of the split
core followed by the CPML face kernels, byte for byte."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

ALL = ("fb", "fb", "fb")


def _fields(ns, npml, coeff, faces, index, split, seed=3):
    from fdtd_accelerate_amd import Core, Fields
    from fdtd_accelerate_amd.core import CoreSplit
    from fdtd_accelerate_amd.cpml import Cpml
    rng = np.random.default_rng(seed)
    f = Fields(*ns, coeff_use=coeff)
    (CoreSplit if split else Core)(f)
    cp = Cpml(f, npml, faces) if npml else None
    f.set_ehs(*[rng.standard_normal(ns).astype(np.float32) for _ in range(6)])
    vals = (0.5 / rng.uniform(1, 6, 9)).astype(np.float32)
    if "e" in coeff:
        f.set_ces(*[vals[rng.integers(0, 9, ns)] for _ in range(3)])
    if "h" in coeff:
        f.set_chs(*[vals[rng.integers(0, 9, ns)] for _ in range(3)])
    if index and not split:
        assert f.compress_ce()
    if cp is not None:  # psi on the cells that the update reaches or keeps
        for buf in (cp.psiE_buf, cp.psiH_buf):
            buf.copy_(torch.from_numpy(rng.standard_normal(buf.numel()).astype(np.float32)))
    return f, cp


@pytest.mark.parametrize("ns,npml,coeff,faces,index", [
    ((2, 2, 3), 0, "", ALL, False), ((3, 72, 16), 0, "eh", ALL, False), ((5, 73, 61), 0, "h", ALL, False),
    ((4, 100, 260), 0, "e", ALL, True), ((60, 70, 127), 0, "eh", ALL, False), ((64, 128, 64), 0, "h", ALL, False),
    ((18, 17, 33), 4, "", ALL, False), ((21, 75, 61), 5, "eh", ALL, False),
    ((26, 130, 57), 12, "e", ALL, True), ((20, 22, 64), 6, "h", ALL, False), ((19, 80, 48), 5, "e", ("", "", "fb"), False),
    ((17, 74, 131), 4, "e", ("fb", "", ""), True), ((24, 28, 50), 6, "eh", ("fb", "fb", ""), False),
    ((20, 76, 45), 5, "e", ("fb", "b", "fb"), True), ((20, 20, 40), 3, "", ("f", "", "b"), False),
])
def test_half_steps_equal_separate_kernels(ns, npml, coeff, faces, index):
    (a, ca), (b, cb) = (_fields(ns, npml, coeff, faces, index, split) for split in (False, True))
    for _ in range(3):
        for f in (a, b):
            f.update_e()
            f.update_h()
    for x, y in zip(a.ehs, b.ehs):
        assert torch.equal(x.view(torch.int32), y.view(torch.int32))
    if npml:
        assert torch.equal(ca.psiE_buf.view(torch.int32), cb.psiE_buf.view(torch.int32))
        assert torch.equal(ca.psiH_buf.view(torch.int32), cb.psiH_buf.view(torch.int32))


@pytest.mark.parametrize("ns,npml,coeff,faces,index,box", [
    ((18, 17, 33), 4, "", ALL, False, ((0, 0, 0), (17, 16, 32))),          # the whole grid, walls and slabs
    ((21, 75, 61), 5, "eh", ALL, False, ((3, 2, 7), (19, 70, 50))),        # rows off the 16-byte lines
    ((26, 130, 57), 12, "e", ALL, True, ((5, 60, 4), (6, 60, 55))),        # one row
    ((19, 80, 48), 5, "e", ("", "", "fb"), False, ((2, 1, 8), (17, 78, 39))),
    ((20, 26, 45), 5, "e", ("fb", "b", "fb"), False, ((4, 4, 5), (9, 20, 30))),  # separate calls
])
def test_half_steps_with_a_drude_region(ns, npml, coeff, faces, index, box):
    from fdtd_accelerate_amd import Drude
    out = []
    for split in (False, True):
        f, cp = _fields(ns, npml, coeff, faces, index, split)
        d = Drude(f, *box, 0.5, 0.05)
        rng = np.random.default_rng(8)
        for t in d.J:
            t.copy_(torch.from_numpy(rng.standard_normal(tuple(t.shape)).astype(np.float32)))
        assert f._joined() == (0 if split else 3)
        for _ in range(3):
            f.update_e()
            f.update_h()
        out.append([*f.ehs, *d.J, cp.psiE_buf, cp.psiH_buf])
    for x, y in zip(*out):
        assert torch.equal(x.view(torch.int32), y.view(torch.int32))


def test_replaced_updates_run_by_themselves():
    """An update method that a program replaces, on an instance or in a subclass, is called."""
    from fdtd_accelerate_amd import Core, Fields
    from fdtd_accelerate_amd.cpml import Cpml

    class Counting(Cpml):
        calls = 0

        def update_e(self):
            Counting.calls += 1
            super().update_e()

    f = Fields(16, 16, 16, coeff_use="")
    Core(f)
    Counting(f, 4)
    f.update_e()
    assert Counting.calls == 1
    f = Fields(16, 16, 16, coeff_use="")
    core = Core(f)
    Cpml(f, 4)
    seen = []
    core.update_h = lambda: seen.append(1)
    f.update_h()
    assert seen == [1]


@pytest.mark.parametrize("count", [1, 31, 32, 33, 70])
def test_record_takes_any_number_of_probes(count):
    from fdtd_accelerate_amd.sim import YeeSim
    rng = np.random.default_rng(count)
    s = YeeSim(9, 8, 18, npml=0, coeff_use="")
    s.fields.set_ehs(*[rng.standard_normal((9, 8, 18)).astype(np.float32) for _ in range(6)])
    pts = [(("ex", "ey", "ez", "hx", "hy", "hz")[rng.integers(6)], tuple(int(rng.integers(n)) for n in (9, 8, 18)))
           for _ in range(count)]
    for name, p in pts:
        s.add_probe(name, p)
    series = s.run(2)
    assert series.shape == (2, count)
    assert np.array_equal(series[-1], np.array([s.field(n)[p].item() for n, p in pts], np.float32))
