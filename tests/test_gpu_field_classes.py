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
