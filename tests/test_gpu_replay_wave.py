"""Replay with a wavefront per replica, against the CPU oracle: bit-exact spins,
rand() draw counts and final libc states, at the edges of its batches of 64
attempts, its blocks of 31 outputs, its row widths and its dispatch."""
import numpy as np
import pytest

import oracle as O
from conftest import init_confs

pytestmark = pytest.mark.gpu


def _rows(N, Z, seed, model):
    rng = np.random.RandomState(seed)
    nbs = np.zeros((N, Z, 2))
    nbs[:, :, 0] = rng.randint(0, N, (N, Z))  # spins of their own row and named twice included
    nbs[:, :, 1] = rng.choice([-1.0, 1.0], (N, Z)) if model == "pm" else rng.normal(0.0, 1.0, (N, Z))
    nbs[rng.rand(N, Z) < 0.2] = 0.0           # ragged rows
    return nbs


def _orders(N, G, rng, repeats):
    return np.array([rng.randint(0, N, N) if repeats else rng.permutation(N) for _ in range(G)])


def _device(gpu, nbs, confs, perms, rseeds):
    import torch
    from piqmc import device
    return (device.Problem(nbs), torch.tensor(np.stack(confs), device=gpu),
            torch.tensor(np.stack(perms, axis=2).astype(np.int16), device=gpu),
            torch.tensor(np.stack([O.Type3(s).st for s in rseeds]).view(np.int32), device=gpu))


@pytest.mark.parametrize("N,Z,P,M,T,model,repeats", [
    (1, 1, 2, 1, 0.5, "pm", False), (31, 4, 3, 2, 0.3, "pm", False), (63, 5, 4, 1, 0.05, "gauss", False),
    (64, 4, 2, 1, 1.0, "pm", True), (65, 6, 5, 2, 0.2, "gauss", False), (129, 8, 3, 1, 0.02, "gauss", True),
    (130, 7, 6, 1, 3.0, "gauss", False), (70, 9, 4, 1, 0.2, "gauss", False), (2100, 3, 4, 1, 0.1, "pm", False)])
def test_qa_wave(gpu, N, Z, P, M, T, model, repeats):
    S, R = 6, 5
    nbs = _rows(N, Z, N + Z, model)
    rng = np.random.RandomState(N)
    sched = np.linspace(3.0, 1e-8, S)
    confs = [init_confs(N, P, rng) for _ in range(R)]
    perms = [_orders(N, S * M, rng, repeats) for _ in range(R)]
    pb, c8, pd, rs = _device(gpu, nbs, [c.T.astype(np.int8) for c in confs], perms, range(3, 3 + R))
    draws, _ = pb.qa_replay(c8, sched, M, T, pd, rs)
    for r in range(R):
        t3 = O.Type3(3 + r)
        assert int(draws[r]) == O.qa_compat(sched, M, P, T, N, confs[r], nbs, perms[r], t3)
        assert np.array_equal(c8[r].cpu().numpy(), confs[r].T.astype(np.int8))
        assert np.array_equal(rs[r].cpu().numpy().view(np.uint32), t3.st)


@pytest.mark.parametrize("N,Z,repeats", [(1, 1, False), (64, 4, True), (65, 5, False), (127, 6, False), (200, 8, True)])
def test_sa_wave(gpu, N, Z, repeats):
    # temperatures at which the quotient is infinite, zero, positive, or neither
    sched = np.array([3.0, np.inf, 1.0, 0.0, -1.0, 1e-30, 0.3, 1e30])
    M, R = 2, 5
    nbs = _rows(N, Z, N * Z, "gauss")
    rng = np.random.RandomState(N)
    sv = [rng.randint(0, 2, N) * 2.0 - 1.0 for _ in range(R)]
    perms = [_orders(N, len(sched) * M, rng, repeats) for _ in range(R)]
    pb, s8, pd, rs = _device(gpu, nbs, [v.astype(np.int8) for v in sv], perms, range(3, 3 + R))
    draws, _ = pb.sa_replay(s8, sched, M, pd, rs)
    for r in range(R):
        t3 = O.Type3(3 + r)
        assert int(draws[r]) == O.sa_compat(sched, M, sv[r], nbs, perms[r], t3)
        assert np.array_equal(s8[r].cpu().numpy(), sv[r].astype(np.int8))
        assert np.array_equal(rs[r].cpu().numpy().view(np.uint32), t3.st)


@pytest.mark.parametrize("R", [8192, 8193])
def test_dispatch_line(gpu, R):
    """The largest call a wavefront takes and the smallest a lane takes agree."""
    import torch
    N, P, S, K = 40, 3, 4, 16
    nbs = _rows(N, 4, 1, "gauss")
    rng = np.random.RandomState(2)
    sched = np.linspace(3.0, 1e-8, S)
    confs = [init_confs(N, P, rng) for _ in range(K)]
    perms = [_orders(N, S, rng, False) for _ in range(K)]
    pb, c8, pd, rs = _device(gpu, nbs, [c.T.astype(np.int8) for c in confs], perms, range(K))
    pick = torch.arange(R, device=gpu) % K
    c, p, s = c8[pick].contiguous(), pd[:, :, pick].contiguous(), rs[pick].contiguous()
    pb.qa_replay(c, sched, 1, 0.2, p, s)
    ref, st = [], []
    for r in range(K):
        t3 = O.Type3(r)
        O.qa_compat(sched, 1, P, 0.2, N, confs[r], nbs, perms[r], t3)
        ref.append(confs[r].T.astype(np.int8))
        st.append(t3.st.copy().view(np.int32))
    assert torch.equal(c, torch.tensor(np.stack(ref), device=gpu)[pick])
    assert torch.equal(s, torch.tensor(np.stack(st), device=gpu)[pick])
