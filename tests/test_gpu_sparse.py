"""The sparse real-coupling sweep (weighted-count filter, queued exact
attempts) and its classical-chain form, bit for bit against the CPU twin."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _nbs(kind, rng):
    """Neighbour tables whose rows have up to 4, 6, 8 and 16 nonzero entries."""
    from piqmc import instances
    if kind == "bare":                       # fields only: one color, no couplings
        N = 70
        return instances.neighbors(N, np.arange(N), np.arange(N), rng.randn(N))
    L, dim = {"square": (8, 2), "odd": (7, 2), "field": (9, 2), "cubic": (4, 3), "cubicfield": (5, 3),
              "random": (8, 2), "tiny": (2, 2), "huge": (6, 2)}[kind]
    N, r, c, v = instances.lattice_pm_j(L, dim, rng, 0.5 if "field" in kind else 0.0)
    off = r != c
    v = np.where(off, rng.randn(v.size), v)
    if kind == "random":                     # long ragged rows, a field and a zero coupling among them
        a, b = rng.randint(0, N, 120), rng.randint(0, N, 120)
        m = a < b
        r, c, v = np.r_[r, a[m], 3], np.r_[c, b[m], 3], np.r_[v, 2 * rng.randn(int(m.sum())), 0.7]
        v[5] = 0.0
    if kind == "huge":                       # couplings of very different sizes
        v = v * 10.0 ** rng.randint(-9, 9, v.size)
    return instances.neighbors(N, r, c, v)


@pytest.mark.parametrize("kind", ["square", "odd", "field", "cubic", "cubicfield", "random", "bare", "tiny", "huge"])
@pytest.mark.parametrize("P,T,M,block,rpw", [(2, 0.3, 1, 0, 0), (20, 0.01, 2, 0, 0), (64, 1 / 64, 1, 64, 3),
                                             (66, 1.5, 1, 192, 2), (128, 1 / 128, 1, 1024, 0)])
def test_sparse_sweep_matches_oracle(gpu, kind, P, T, M, block, rpw):
    import torch
    from piqmc import device
    rng = np.random.RandomState(P + len(kind))
    nbs = _nbs(kind, rng)
    pb = device.Problem(nbs)
    pb.set_sweep_path("word")
    N, R, color = nbs.shape[0], 4, pb.coloring()
    sched = np.r_[np.linspace(3.0, 1e-8, 7), 0.0]   # the last field: J_perp is infinite
    init = (2 * rng.randint(2, size=(R, P, N)) - 1).astype(np.int8)
    got = []
    for trace in (False, True):
        d = torch.from_numpy(init.copy()).to(gpu)
        et = pb.qa_colored(d, sched, M, T, 99 + P, replica_base=5, sweep_base=3, trace=trace, block=block, rpw=rpw)
        got.append(d.cpu().numpy())
    for r in range(R):
        ref = init[r].copy()
        etr = O.qa_colored(sched, M, P, T, ref, nbs, color, pb.ncolors, 99 + P, replica=5 + r, sweep_base=3,
                           trace=True)
        assert np.array_equal(got[0][r], ref) and np.array_equal(got[1][r], ref)
        # sums of N rows in another order
        np.testing.assert_allclose(et[r].cpu().numpy(), etr, rtol=1e-12, atol=1e-12 * np.abs(nbs[:, :, 1]).sum())


@pytest.mark.parametrize("kind,C", [("square", 2), ("odd", 62), ("cubicfield", 130), ("random", 64), ("bare", 6),
                                    ("square", 1536)])
def test_sparse_chains_match_oracle(gpu, kind, C):
    import torch
    from piqmc import device
    rng = np.random.RandomState(C)
    nbs = _nbs(kind, rng)
    pb = device.Problem(nbs)
    pb.set_sweep_path("word")
    sched = np.linspace(3.0, 0.01, 5)
    ref = (2 * rng.randint(2, size=(C, nbs.shape[0])) - 1).astype(np.int8)
    d = torch.from_numpy(ref.copy()).to(gpu)
    pb.sa_colored(d, sched, 2, seed=31, replica_base=2, sweep_base=1)
    O.sa_colored(sched, 2, ref, nbs, pb.coloring(), pb.ncolors, 31, replica_base=2, sweep_base=1)
    assert np.array_equal(d.cpu().numpy(), ref)


@pytest.mark.parametrize("scale,T", [(1e-28, 1e9), (1e-28, 1.0), (1e-20, 1e20), (1e20, 1e-3), (1e27, 1e9)])
def test_scales_past_float_products(gpu, scale, T):
    """Couplings and temperatures of which a product (weight scale times J_perp or
    T) leaves float's range: the filter then decides nothing wrongly."""
    import torch
    from piqmc import device, instances
    rng = np.random.RandomState(3)
    N, r, c, v = instances.lattice_pm_j(6, 2, rng, 0.0)
    nbs = instances.neighbors(N, r, c, scale * rng.randn(v.size))
    pb = device.Problem(nbs)
    P, R, sched = 20, 3, np.array([3.0, 1.0, 1e-3, 1e-8])
    init = (2 * rng.randint(2, size=(R, P, N)) - 1).astype(np.int8)
    d = torch.from_numpy(init.copy()).to(gpu)
    pb.qa_colored(d, sched, 2, T, 9)
    for k in range(R):
        ref = init[k].copy()
        O.qa_colored(sched, 2, P, T, ref, nbs, pb.coloring(), pb.ncolors, 9, replica=k)
        assert np.array_equal(d[k].cpu().numpy(), ref)
