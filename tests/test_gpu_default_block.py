"""Default workgroup sizes of the +-1 sweep on uniform lattices: 512 and 256
threads with more than two colors, 1024 where two colors of up to 2048 spins
stay cached.  Same spins as the CPU twin on every side of the lines."""
import numpy as np
import pytest

import oracle as O
from conftest import pm_j_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,dim,P,R", [(25, 2, 40, 256), (25, 2, 70, 257), (9, 3, 20, 3), (44, 2, 20, 5), (46, 2, 20, 3),
                                       (64, 2, 66, 2), (64, 2, 8, 2048), (66, 2, 10, 2)])
def test_default_block(gpu, L, dim, P, R):
    import torch
    from piqmc import device
    N, nbs, _, _, _ = pm_j_problem(L, dim=dim, seed=L + P)
    S, T = 4, 1.0 / P
    sched = np.linspace(3.0, 1e-8, S)
    pb = device.Problem(nbs)
    color = pb.coloring()
    g = torch.Generator(device=gpu).manual_seed(L)
    c8 = torch.randint(0, 2, (R, P, N), generator=g, dtype=torch.int8, device=gpu) * 2 - 1
    init = c8.cpu().numpy().copy()
    pb.qa_colored(c8, sched, 1, T, 5)
    for r in (0, R - 1):
        ref = init[r].copy()
        O.qa_colored(sched, 1, P, T, ref, nbs, color, int(color.max()) + 1, 5, replica=r)
        assert np.array_equal(c8[r].cpu().numpy(), ref)


@pytest.mark.parametrize("L,dim,P,R", [(99, 2, 20, 300), (65, 2, 128, 600), (17, 3, 20, 600), (25, 2, 64, 1000),
                                       (33, 2, 100, 301), (33, 2, 20, 2048)])
def test_default_block_is_near_the_best(gpu, L, dim, P, R):
    """More than two colors: the kernel time of the default workgroup size against
    that of 256 and of 512 threads."""
    _near_the_best(gpu, L, dim, P, R, (256, 512))


def _near_the_best(gpu, L, dim, P, R, blocks):
    import torch
    from piqmc import device
    N, nbs, _, _, _ = pm_j_problem(L, dim=dim, seed=L + P)
    pb = device.Problem(nbs)
    c8 = torch.ones((R, P, N), dtype=torch.int8, device=gpu)
    sched = np.linspace(3.0, 1e-8, 20)

    best = dict.fromkeys((0,) + blocks, np.inf)
    for _ in range(6):                   # in turn, the first round to warm up
        for block in best:
            c8.fill_(1)
            pb.qa_colored(c8, sched, 1, 1.0 / P, 5, block=block)
            best[block] = min(best[block], device.last_kernel_ms())
    assert best.pop(0) <= 1.1 * min(best.values())


@pytest.mark.parametrize("L,dim,P,R", [(46, 2, 20, 600), (14, 3, 20, 1000), (46, 2, 64, 100), (46, 2, 128, 600),
                                       (64, 2, 64, 600), (46, 2, 20, 2048)])
def test_default_block_of_two_large_colors(gpu, L, dim, P, R):
    _near_the_best(gpu, L, dim, P, R, (512, 1024))
