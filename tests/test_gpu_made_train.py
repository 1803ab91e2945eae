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


def test_forward_passes_allocate_no_training_buffers(gpu):
    import torch
    from piqmc.made import MADE
    N, H1, H2, B = 100, 300, 200, 200000
    rng = np.random.RandomState(1)
    Sd = torch.tensor((2 * rng.randint(2, size=(B, N)) - 1).astype(np.int8), device=gpu)
    out = torch.empty(B, dtype=torch.float64, device=gpu)
    net = MADE(N, H1, H2, seed=3)
    net.logprob(Sd[:1])
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    out = net.logprob(Sd)
    torch.cuda.synchronize()
    took = before - torch.cuda.mem_get_info()[0]
    # spins and both hidden layers in bf16 at pitches of 128, 320 and 256, the logits
    # in fp32, a double and a row of spins
    need = B * (2 * (128 + 320 + 256) + 4 * N + 8 + N)
    assert took < 1.05 * need + (64 << 20)
    assert torch.isfinite(out).all()


@pytest.mark.parametrize("N,H1,H2", [(37, 70, 129), (64, 64, 64), (100, 191, 63)])
def test_training_after_larger_forward_passes(gpu, N, H1, H2):
    """Forward buffers that grow between training steps (their rows then hold
    other data past the sizes) leave the steps unchanged."""
    import torch
    from piqmc.made import MADE
    rng = np.random.RandomState(N)
    Sd = torch.tensor((2 * rng.randint(2, size=(7000, N)) - 1).astype(np.int8), device=gpu)
    a, b = MADE(N, H1, H2, seed=5), MADE(N, H1, H2, seed=5)
    for k, B in enumerate((67, 130, 64)):
        junk = torch.full((1 << 24,), float("nan"), dtype=torch.bfloat16, device=gpu)
        del junk
        torch.cuda.empty_cache()          # memory of NaN for the next allocation to find
        lb = b.logprob(Sd[:1000 * (2 * k + 1)])
        assert a.train_step(Sd[:B], 1e-3) == b.train_step(Sd[:B], 1e-3)
        assert torch.isfinite(lb).all()
    for x, y in zip(a.params() + a.grads(), b.params() + b.grads()):
        assert np.array_equal(x, y)
    assert torch.equal(a.logprob(Sd), b.logprob(Sd))
