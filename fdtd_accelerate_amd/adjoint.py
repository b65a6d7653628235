"""Adjoint gradients of a field objective with respect to the permittivity of a design box.

Problem (``DesignProblem``): a Yee + CPML simulation on the in-place engine's
arithmetic (here stepped by the slab engine, which is bit-identical) with CE = 0.5 in
vacuum and CE = 0.5/eps_r on every E component of each design voxel, soft sources,
and the objective

    J = sum over steps n in [n0, nsteps] of sum over the monitor plane x = im of
        ex^2 + ey^2 + ez^2   (E after step n)

The gradient needs, of each step, the curl of H on the design box before it.
``forward(eps)`` runs the steps once and stores these curls for as many of the last steps
as there is memory for (``curl_bytes``: no more in all than checkpoints of every segment
would take, or a share of the free memory); of the segments of ``ckpt``
steps before those it keeps a checkpoint of the full state (fields and psi), and of the
objective window the monitor-plane E.  ``backward()`` walks the segments in reverse: where
the curls are not stored it restores a checkpoint and recomputes the segment with its
curls, then it runs the hand-written adjoint step (``mifdtd_adjoint_step``) back through
it, accumulating dJ/dCE in double precision; dJ/deps = -0.5/eps^2 * sum over the three
components.  ``FdtdObjective`` is the torch.autograd.Function around it.
"""
from __future__ import annotations

import ctypes

import numpy as np
import torch

from . import _lib
from .fused import SlabStepper
from .sim import YeeSim
from .sources import gaussian_pulse


def curl_bytes(nsteps, ckpt, state, curl, room):
    """Bytes of curls (``curl`` a step) to store for as many of the last steps as there is
    memory for: whole segments of ``ckpt`` steps, such that the curls, the checkpoints
    (``state`` each) of the segments before them and the buffer to recompute one of these take
    no more than checkpoints of all segments with that buffer, or than ``room``."""
    limit = max(-(-nsteps // ckpt) * state + ckpt * curl, room)
    for kept in range(0, nsteps, ckpt):
        curls = (nsteps - kept) * curl
        if curls + kept // ckpt * state + (ckpt * curl if kept else 0) <= limit:
            return curls
    return 0


class DesignProblem:
    def __init__(self, n=(160, 160, 160), npml=10, box=(48, 48, 48, 64, 64, 64), src_plane=20,
                 monitor=140, nsteps=800, window=200, ckpt=50, tfunc=None, src_box=None):
        nx, ny, nz = n
        self.n = n
        self.npml = npml
        self.box = tuple(int(v) for v in box)
        self.monitor = int(monitor)
        self.nsteps = int(nsteps)
        self.n0 = self.nsteps - int(window) + 1  # first step of the objective window
        self.ckpt = int(ckpt)
        self.tfunc = tfunc if tfunc is not None else gaussian_pulse()
        i0, j0, k0, di, dj, dk = self.box
        if not (0 < i0 and i0 + di < nx and 0 < j0 and j0 + dj < ny - 1 and 0 < k0 and k0 + dk < nz - 1):
            raise ValueError(f"design box {self.box} must lie inside the grid {n}")
        # the adjoint's gradient has no term for the CPML correction of E (-/+CE*psi), so
        # the box keeps off every E slab plane: [npml, n-1-npml) on each axis
        if npml and not (i0 >= npml and i0 + di <= nx - 1 - npml and j0 >= npml and j0 + dj <= ny - 1 - npml
                         and k0 >= npml and k0 + dk <= nz - 1 - npml):
            raise ValueError(f"design box {self.box} overlaps a CPML slab (npml {npml}) of the grid {n}")
        self.sim = YeeSim(nx, ny, nz, npml=npml, coeff_use="e")
        # Ez soft line source on the plane x = src_plane: the line y = ny/2 along z over the
        # non-CPML interior
        if src_box is None:
            src_box = ((src_plane, ny // 2, npml), (src_plane, ny // 2, nz - npml - 1))
        self.src = self.sim.add_source("ez", src_box[0], src_box[1], self.tfunc)
        self.stepper = SlabStepper(self.sim)
        f = self.sim.fields
        self.dbox = _lib.DesignBox(*self.box)
        self.dev = f.device
        self.stream = f.stream
        self._eps = None

    # -------------------------------------------------------------- state helpers
    def _state(self):
        f = self.sim.fields
        cp = self.sim.cpml
        return list(f.ehs) + ([cp.psiE_buf, cp.psiH_buf] if cp is not None else [])

    def _reset(self):
        for t in self._state():
            t.zero_()
        self.src.tstep = 1

    def _set_eps(self, eps):
        eps = torch.as_tensor(eps, dtype=torch.float32, device=self.dev)
        i0, j0, k0, di, dj, dk = self.box
        if tuple(eps.shape) != (di, dj, dk):
            raise ValueError(f"eps shape {tuple(eps.shape)} != design box {(di, dj, dk)}")
        ce = 0.5 / eps
        f = self.sim.fields
        for c in f.ces:
            c[i0:i0 + di, j0:j0 + dj, k0:k0 + dk] = ce
        f.ce_mat = f.ce_lut = None  # material indices of the previous CE no longer hold
        self._eps = eps.clone()

    def _plane(self, out):
        f = self.sim.fields
        torch.stack([f.ehs[c][self.monitor] for c in range(3)], out=out)  # (3, ny, nzp)

    def _curl_budget(self):
        """Bytes of curls that a forward run may hold (curl_bytes), with the room left on the
        GPU beside what backward() allocates.  A run of 160^3 cells, 800 steps and a 64^3 box
        takes 2.5 GB of curls or 2.0 GB of checkpoints and recomputes nothing: 193 -> 135 ms
        for forward and backward."""
        size = lambda ts: sum(t.numel() * t.element_size() for t in ts)
        curl = 12 * int(np.prod(self.box[3:]))
        free, total = torch.cuda.mem_get_info(self.dev)
        free += torch.cuda.memory_reserved(self.dev) - torch.cuda.memory_allocated(self.dev)
        state = size(self._state())
        return curl_bytes(self.nsteps, self.ckpt, state, curl, min(total // 32, (free - state - 2 * curl) // 2))

    def _alloc_curls(self):
        """Curls of the steps after ``self.kept`` (a segment start), or None and no such step."""
        shape = (3, *self.box[3:])
        keep = min(self.nsteps, self._curl_budget() // (4 * int(np.prod(shape))))
        kept = -(-(self.nsteps - keep) // self.ckpt) * self.ckpt
        curls = None
        if kept < self.nsteps:
            try:
                curls = torch.empty((self.nsteps - kept, *shape), dtype=torch.float32, device=self.dev)
                curls.record_stream(self.stream)
            except torch.OutOfMemoryError:
                pass
        return (kept, curls) if curls is not None else (self.nsteps, None)

    # ------------------------------------------------------------------- forward
    def forward(self, eps):
        """Run the simulation for eps (design box values); returns J (float)."""
        self._set_eps(eps)
        try:
            return self._forward(True)
        except torch.OutOfMemoryError:
            if self.curls is None:
                raise
        return self._forward(False)

    def _forward(self, keep_curls):
        self._reset()
        self.ckpts = {}
        nwin = self.nsteps - self.n0 + 1
        f = self.sim.fields
        self.planes = self.curls = None  # the last run's, before the new ones are allocated
        self.planes = torch.empty((nwin, 3, f.ny, f.nz_pitch), dtype=torch.float32, device=self.dev)
        self.kept, self.curls = self._alloc_curls() if keep_curls else (self.nsteps, None)
        n = 0
        while n < self.nsteps:
            if n < self.kept and n % self.ckpt == 0:
                self.ckpts[n] = [t.clone() for t in self._state()]
            # to the next checkpoint, the first kept curl or the objective's first plane
            stop = self.nsteps
            if n < self.kept:
                stop = min(stop, (n // self.ckpt + 1) * self.ckpt, self.kept)
            stop = min(stop, self.n0 - 1) if n + 1 < self.n0 else n + 1
            design = None if n < self.kept else (self.box, self.curls[n - self.kept:stop - self.kept])
            self.stepper._call(stop - n, None, design=design)
            n = stop
            if n >= self.n0:
                self._plane(self.planes[n - self.n0])
        p = self.planes.double()
        return float((p * p).sum())

    # ------------------------------------------------------------------ backward
    def backward(self):
        """dJ/deps on the design box (float64 tensor, box shape) of the last forward."""
        try:
            return self._backward()
        except torch.OutOfMemoryError:
            if self.curls is None:
                raise
        self._set_eps(self._eps)
        self._forward(False)  # the same run with checkpoints in place of the curls
        return self._backward()

    def _backward(self):
        f = self.sim.fields
        cp = self.sim.cpml
        i0, j0, k0, di, dj, dk = self.box
        nbox = di * dj * dk
        lam = [torch.zeros_like(t) for t in f.ehs]
        lpE = torch.zeros_like(cp.psiE_buf) if cp is not None else None
        lpH = torch.zeros_like(cp.psiH_buf) if cp is not None else None
        grad = torch.zeros((3, di, dj, dk), dtype=torch.float64, device=self.dev)
        segment = torch.empty((self.ckpt, 3, di, dj, dk), dtype=torch.float32, device=self.dev) if self.ckpts else None
        lamp = (ctypes.c_void_p * 6)(*[t.data_ptr() for t in lam])
        cep = (ctypes.c_void_p * 3)(*[c.data_ptr() for c in f.ces])
        tabs = (cp.bE.data_ptr(), cp.aE.data_ptr(), cp.bH.data_ptr(), cp.aH.data_ptr()) if cp is not None else (None,) * 4
        st = _lib.stream_handle(self.stream)
        for s0 in reversed(range(0, self.nsteps, self.ckpt)):
            s1 = min(s0 + self.ckpt, self.nsteps)
            if s0 >= self.kept:
                curls = self.curls[s0 - self.kept:s1 - self.kept]
            else:  # recompute, keeping curl(H^{n-1}) on the box
                for t, c in zip(self._state(), self.ckpts[s0]):
                    t.copy_(c)
                self.src.tstep = s0 + 1
                curls = segment[:s1 - s0]
                self.stepper._call(s1 - s0, None, design=(self.box, curls))
            for n in range(s1, s0, -1):
                ep = self.planes[n - self.n0].data_ptr() if n >= self.n0 else None
                _lib.call("mifdtd_adjoint_step", f.nx, f.ny, f.nz_pitch, f.pad, ctypes.byref(lamp), ctypes.byref(cep),
                          cp.npml if cp is not None else 0,
                          None if lpE is None else lpE.data_ptr(), None if lpH is None else lpH.data_ptr(),
                          *tabs, ep, self.monitor, ctypes.byref(self.dbox), curls[n - s0 - 1].data_ptr(),
                          grad.data_ptr(), st)
        eps = self._eps.double()
        self.grad_ce = grad
        return grad.sum(0) * (-0.5 / (eps * eps))


class FdtdObjective(torch.autograd.Function):
    """J(eps) with the adjoint gradient: ``FdtdObjective.apply(eps, problem)``."""

    @staticmethod
    def forward(ctx, eps, problem):
        J = problem.forward(eps.detach())
        ctx.problem = problem
        return torch.tensor(J, dtype=torch.float64, device=eps.device)

    @staticmethod
    def backward(ctx, gJ):
        g = ctx.problem.backward()
        return (gJ * g).to(torch.float32), None
