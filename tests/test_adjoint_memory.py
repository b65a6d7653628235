"""How much memory the stored curls of a design problem take, and what happens without it."""
import numpy as np
import pytest
import torch


def _peak(nsteps, ckpt, state, curl, room):
    """Curls, checkpoints and recomputation buffer of a run under curl_bytes."""
    from fdtd_accelerate_amd.adjoint import curl_bytes
    got = curl_bytes(nsteps, ckpt, state, curl, room)
    assert got % curl == 0
    kept = nsteps - got // curl  # the steps without a stored curl: whole segments, or all steps
    assert 0 <= kept <= nsteps and (kept % ckpt == 0 or kept == nsteps)
    return got, got + -(-kept // ckpt) * state + (ckpt * curl if kept else 0)


@pytest.mark.parametrize("n,box,nsteps,ckpt", [
    (512, 320, 2000, 50), (400, 256, 2000, 25), (160, 64, 800, 50), (160, 64, 801, 50), (64, 40, 300, 7), (64, 8, 300, 300),
    (96, 90, 100, 1000), (48, 24, 37, 1),
])
@pytest.mark.parametrize("room", [-10 ** 9, 0, 10 ** 8, 9 * 10 ** 9, 10 ** 12])
def test_curls_stay_within_the_checkpoints_or_the_room(n, box, nsteps, ckpt, room):
    state, curl = 24 * n ** 3, 12 * box ** 3
    checkpoints = -(-nsteps // ckpt) * state + ckpt * curl  # a run that stores no curls
    got, peak = _peak(nsteps, ckpt, state, curl, room)
    assert peak <= max(checkpoints, room)
    if nsteps * curl <= max(checkpoints, room):
        assert got == nsteps * curl  # all of them where they fit


@pytest.mark.gpu
def test_gradient_where_memory_runs_out():
    """Where an allocation beside the stored curls fails, in forward or in backward, the run
    gives them up and the gradient is the same to the last bit."""
    from fdtd_accelerate_amd.adjoint import DesignProblem
    box = (10, 9, 8, 8, 7, 12)
    eps = np.random.default_rng(3).uniform(1, 4, box[3:]).astype(np.float32)
    out = []
    for fail in (None, "forward", "backward"):
        p = DesignProblem(n=(32, 30, 28), npml=5, box=box, src_plane=7, monitor=24, nsteps=60, window=20, ckpt=9)
        if fail:
            name = "_" + fail
            whole = getattr(p, name)

            def once(*args):
                setattr(p, name, whole)
                whole(*args)
                raise torch.OutOfMemoryError("planned")

            if fail == "forward":
                setattr(p, name, once)
        J = p.forward(eps)
        assert (p.curls is None) == (fail == "forward")
        if fail == "backward":
            p._backward = once
        g = p.backward()
        assert (p.curls is None) == (fail is not None)
        out.append((J, g.cpu().numpy().tobytes()))
    assert out[0] == out[1] == out[2]
