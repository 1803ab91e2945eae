"""The blocked dense sweep, bit for bit against the CPU twin: partial blocks,
one block only, every register width, both word sizes, fields, traces and the
schedules on which its float thresholds do not apply."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _dense(N, rng, sparse=False, field=False):
    """Couplings on a grid of 2^-12 (every row sums exactly), some zero."""
    from piqmc import instances
    r, c = np.triu_indices(N, 1)
    v = np.round(rng.randn(r.size) / np.sqrt(N) * 4096) / 4096
    if sparse:
        v[rng.rand(v.size) < 0.5] = 0.0
    if field:
        r, c = np.r_[r, np.arange(N)], np.r_[c, np.arange(N)]
        v = np.r_[v, np.round(rng.randn(N) * 1024) / 4096]
    return instances.neighbors(N, r, c, v)


@pytest.mark.parametrize("N", [5, 16, 17, 33, 64, 100, 130, 200, 256])
@pytest.mark.parametrize("P,T,M", [(2, 0.2, 1), (18, 1 / 18, 2), (64, 1 / 64, 1), (66, 0.5, 1), (128, 1 / 128, 1)])
def test_blocked_sweep_matches_oracle(gpu, N, P, T, M):
    import torch
    from piqmc import device
    rng = np.random.RandomState(N * 131 + P)
    nbs = _dense(N, rng, sparse=N == 33, field=N in (17, 100))
    pb = device.Problem(nbs)
    pb.set_sweep_path("dense")
    assert pb.exact_rows
    R, color = 2, pb.coloring()
    # the last field has infinite J_perp: every decision is made in double
    sched = np.r_[np.linspace(3.0, 1e-8, 5), 0.0]
    init = (2 * rng.randint(2, size=(R, P, N)) - 1).astype(np.int8)
    for trace in (False, True):
        d = torch.from_numpy(init.copy()).to(gpu)
        et = pb.qa_colored(d, sched, M, T, 7 + P, replica_base=3, sweep_base=9, trace=trace)
        for r in range(R):
            ref = init[r].copy()
            etr = O.qa_colored(sched, M, P, T, ref, nbs, color, pb.ncolors, 7 + P, replica=3 + r, sweep_base=9,
                               trace=True)
            assert np.array_equal(d[r].cpu().numpy(), ref)
            if trace:
                np.testing.assert_allclose(et[r].cpu().numpy(), etr, rtol=1e-12, atol=1e-9)


@pytest.mark.parametrize("N,C", [(24, 10), (70, 128)])
def test_blocked_chains_match_oracle(gpu, N, C):
    import torch
    from piqmc import device
    rng = np.random.RandomState(N)
    nbs = _dense(N, rng)
    pb = device.Problem(nbs)
    sched = np.linspace(2.0, 0.05, 6)
    ref = (2 * rng.randint(2, size=(C, N)) - 1).astype(np.int8)
    d = torch.from_numpy(ref.copy()).to(gpu)
    pb.sa_colored(d, sched, 2, seed=5)
    O.sa_colored(sched, 2, ref, nbs, pb.coloring(), pb.ncolors, 5)
    assert np.array_equal(d.cpu().numpy(), ref)


@pytest.mark.parametrize("variant", ["auto", "wave", "split", "workgroup", "pipe4", "fields"])
def test_no_field_steps(gpu, variant):
    """A call without field steps is the identity on every dense layout, with
    and without a scratch region, and leaves no error for the call after it."""
    import ctypes as C
    import torch
    from piqmc import _lib, device
    rng = np.random.RandomState(1)
    nbs = _dense(48, rng)
    pb = device.Problem(nbs)
    pb.set_dense_variant(variant)
    init = (2 * rng.randint(2, size=(3, 16, 48)) - 1).astype(np.int8)
    d = torch.from_numpy(init.copy()).to(gpu)
    none = np.zeros(0)
    for _ in range(2):
        assert pb.qa_colored(d, none, 1, 0.1, 1, trace=True).shape == (3, 0)
        _lib.call("piqmc_qa_colored_noalloc", pb._h, 3, 16, 0, 1, 0.1, none.ctypes.data, d.data_ptr(), 1, 0, 0, None,
                  0, 0, C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert np.array_equal(d.cpu().numpy(), init)
    sched = np.linspace(3.0, 1e-8, 4)
    pb.qa_colored(d, sched, 1, 1 / 16, 7)
    ref = init[0].copy()
    O.qa_colored(sched, 1, 16, 1 / 16, ref, nbs, pb.coloring(), pb.ncolors, 7)
    assert np.array_equal(d[0].cpu().numpy(), ref)


SWITCHES = ("PIQMC_DENSE_WG", "PIQMC_DENSE_PIPE", "PIQMC_DENSE_PIPE_WAVES", "PIQMC_FIELDS_SPLIT")


@pytest.mark.parametrize("P,switch,value,items", [
    (16, None, "", 8), (66, None, "", 8), (16, "PIQMC_DENSE_WG", "0", 2), (66, "PIQMC_DENSE_WG", "0", 2),
    (16, "PIQMC_FIELDS_SPLIT", "0", 2), (66, "PIQMC_FIELDS_SPLIT", "0", 2), (66, "PIQMC_FIELDS_SPLIT", "1", 2),
    (16, "PIQMC_FIELDS_SPLIT", "1", 8)])
def test_layout_switches_reach_a_batch(gpu, monkeypatch, P, switch, value, items):
    """A replica per work item in the blocked sweep, four in the layouts that the
    switches compare (one where the replica's 8 slices a parity are split over the
    four wavefronts; 33 are not); the same spins from all of them."""
    import torch
    from piqmc import device
    for s in SWITCHES:
        monkeypatch.delenv(s, raising=False)
    if switch:
        monkeypatch.setenv(switch, value)
    rng = np.random.RandomState(2)
    nbs = _dense(24, rng)
    pb = device.Problem(nbs)
    init = (2 * rng.randint(2, size=(8, P, 24)) - 1).astype(np.int8)
    d = torch.from_numpy(init.copy()).to(gpu)
    sched = np.linspace(3.0, 1e-8, 5)
    b = device.Batch()
    b.add(pb, d, sched, 1, 1.0 / P, 7)
    b.run()
    assert b.info()["items"] == items
    for r in range(8):
        ref = init[r].copy()
        O.qa_colored(sched, 1, P, 1.0 / P, ref, nbs, pb.coloring(), pb.ncolors, 7, replica=r)
        assert np.array_equal(d[r].cpu().numpy(), ref)


def test_scratch_counts_what_the_blocked_sweep_takes(gpu, monkeypatch):
    """The region of the allocation-free entry holds 300 replicas of 256 spins at
    P=128 (4 KiB each); cached fields, 257 KiB a replica more, would not fit it."""
    import ctypes as C
    import torch
    from piqmc import _lib, device
    for s in SWITCHES:
        monkeypatch.delenv(s, raising=False)
    rng = np.random.RandomState(5)
    pb = device.Problem(_dense(256, rng))
    P, sched = 128, np.linspace(3.0, 1e-8, 2)
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)

    def noalloc(d, R):
        _lib.call("piqmc_qa_colored_noalloc", pb._h, R, P, 2, 1, 1.0 / P, sched.ctypes.data, d.data_ptr(), 9, 0, 0, None,
                  0, 0, st)

    a = torch.from_numpy((2 * rng.randint(2, size=(300, P, 256)) - 1).astype(np.int8)).to(gpu)
    b = a.clone()
    noalloc(a, 300)
    pb.qa_colored(b, sched, 1, 1.0 / P, 9)
    assert torch.equal(a, b)
    need = 20000 * 8 * 2 * 256 + 256      # refused before any device work
    with pytest.raises(ValueError, match=" %d bytes" % need):
        noalloc(a, 20000)
    monkeypatch.setenv("PIQMC_FIELDS_SPLIT", "0")
    with pytest.raises(ValueError, match=" %d bytes" % (need + 20000 * 8 * 2 * 64 * 257)):
        noalloc(a, 20000)
