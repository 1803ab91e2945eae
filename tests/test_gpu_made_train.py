"""The fused training step at the edges of its tiles: ragged sizes, batches
after larger ones (stale padding), and the size from which the separate
passes run."""
import numpy as np
import pytest

import made_oracle as MO

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,H1,H2,B", [(2, 1, 1, 1), (37, 70, 129, 67), (64, 64, 64, 64), (65, 191, 63, 65),
                                       (100, 192, 256, 500), (256, 512, 512, 1024), (20, 24, 28, 32900)])
def test_training_gradients_match_oracle(gpu, N, H1, H2, B):
    import torch
    from piqmc.made import MADE
    rng = np.random.RandomState(N + B)
    S = (2 * rng.randint(2, size=(B, N)) - 1).astype(np.int8)
    Sd = torch.tensor(S, device=gpu)
    a, b = MADE(N, H1, H2, seed=3), MADE(N, H1, H2, seed=3)
    b.train_step(torch.cat([Sd, Sd, Sd[:1]]), 0.0)   # larger buffers, their rows full
    p = a.params()
    nll = a.train_step(Sd, 0.0)
    cache, ref = MO.forward(p, S, round_bf16=True)
    # bf16 activations and gradients: 2^-8 a rounding, a few of them in a row
    assert abs(nll - ref.mean()) < 2e-2 * N ** 0.5
    go = MO.backward([MO.bf16(x) if i % 2 == 0 else x for i, x in enumerate(p)], cache)
    for x, y in zip(a.grads(), go):
        assert np.linalg.norm(x - y) <= 3e-2 * max(np.linalg.norm(y), 1e-12)
    # the buffers' size does not enter the result
    assert b.train_step(Sd, 0.0) == nll
    for net in (a, b):
        for _ in range(2):
            net.train_step(Sd, 1e-3)
    for x, y in zip(a.params() + a.grads(), b.params() + b.grads()):
        assert np.array_equal(x, y)
