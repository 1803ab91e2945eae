"""+-1 lattices with fields of which some are exactly zero or tiny: a balanced
bit's energy change is then zero, or too small for any draw to reject."""
import numpy as np
import pytest

import oracle as O
from conftest import pm_j_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,dim,P,T", [(4, 3, 32, 1 / 32), (4, 3, 128, 1 / 128), (6, 2, 32, 0.1), (5, 3, 66, 0.02),
                                       (6, 3, 16, 2.0), (4, 3, 8, 200.0)])
def test_zero_and_tiny_fields(gpu, L, dim, P, T):
    import torch
    from piqmc import device
    N, nbs, _, _, _ = pm_j_problem(L, dim=dim, seed=L + P, field_sigma=0.3)
    nbs = nbs.copy()
    own = nbs[:, :, 0].astype(int) == np.arange(N)[:, None]
    own &= nbs[:, :, 1] != 0
    nbs[own & (np.arange(N) % 3 == 0)[:, None], 1] = 0.0
    nbs[own & (np.arange(N) % 3 == 1)[:, None], 1] = 2.0 ** -27
    R, S, M = 3, 12, 2
    sched = np.linspace(3.0, 1e-8, S)
    pb = device.Problem(nbs)
    assert pb.pm_j_fields
    color = pb.coloring()
    conf = (2 * np.random.RandomState(P).randint(2, size=(R, P, N)) - 1).astype(np.int8)
    c8 = torch.tensor(conf, device=gpu)
    pb.qa_colored(c8, sched, M, T, 7)
    for r in range(R):
        ref = conf[r].copy()
        O.qa_colored(sched, M, P, T, ref, nbs, color, int(color.max()) + 1, 7, replica=r)
        assert np.array_equal(c8[r].cpu().numpy(), ref)


@pytest.mark.parametrize("L,dim,P,T,block,rpw", [
    (6, 2, 128, 1 / 128, 0, 0), (8, 2, 66, 0.02, 64, 3), (14, 2, 64, 1 / 64, 64, 2), (16, 2, 100, 0.3, 128, 0),
    (10, 3, 40, 0.05, 256, 1), (12, 3, 128, 1 / 128, 512, 2), (12, 3, 20, 0.05, 0, 0), (8, 3, 2, 0.2, 128, 5)])
def test_open_bits_queue(gpu, L, dim, P, T, block, rpw):
    """Two-colored square and cubic lattices: whole and partial passes, word
    widths on both sides of 32 slices, several replicas a workgroup, traced."""
    import torch
    from piqmc import device
    N, nbs, _, _, _ = pm_j_problem(L, dim=dim, seed=L + P, field_sigma=0.1)
    R, S, M = 5, 6, 2
    sched = np.linspace(3.0, 1e-8, S)
    pb = device.Problem(nbs)
    assert pb.pm_j_fields
    color = pb.coloring()
    conf = (2 * np.random.RandomState(P).randint(2, size=(R, P, N)) - 1).astype(np.int8)
    c8 = torch.tensor(conf, device=gpu)
    et = pb.qa_colored(c8, sched, M, T, 11, replica_base=3, sweep_base=9, trace=True, block=block, rpw=rpw)
    for r in (0, R - 1):
        ref = conf[r].copy()
        e = O.qa_colored(sched, M, P, T, ref, nbs, color, int(color.max()) + 1, 11, replica=3 + r, sweep_base=9,
                         trace=True)
        assert np.array_equal(c8[r].cpu().numpy(), ref)
        np.testing.assert_allclose(et[r].cpu().numpy(), e, rtol=1e-12, atol=1e-12)
