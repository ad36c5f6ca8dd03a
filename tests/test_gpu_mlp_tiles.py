"""The network's gradient at the edges of its 16-sample tiles and of the 256
blocks that share them, against the FP64 reference of the same network.  The
targets lie 1 above or below the reference's predictions, so that a first
layer activation on the other side of a BF16 rounding boundary (a change of
about 1e-3 of a prediction, at most 5e-3) moves a gradient by at most 1e-2 of
itself.  Two passes over the same samples must give the same bits."""
import numpy as np
import pytest

import mlp_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 4095, 4096, 4097, 12345])
def test_gradient_at_tile_edges(n):
    import torch
    from harm_finalwham_amd import harmgpu
    print("case gradient tiles", n, flush=True)
    rng = np.random.default_rng(n)
    w = mlp_ref.random_params(6).astype(np.float32)
    X = rng.normal(0.0, 1.5, (n, 8)).astype(np.float32)
    y, _ = mlp_ref.forward(w.astype(np.float64), X, quant=True)
    Y = (y + rng.choice([-1.0, 1.0], n)).astype(np.float32)
    m = harmgpu.Mlp(seed=1)
    m.set_params(w)
    Xd, Yd = torch.from_numpy(X).cuda(), torch.from_numpy(Y).cuda()
    g, loss = m.gradient(Xd, Yd)
    lr, gr = mlp_ref.loss_grad(w.astype(np.float64), X, Y, quant=True)
    assert abs(loss - lr) <= 1e-2 * lr
    for a, b in ((0, 512), (512, 576), (576, 4672), (4672, 4736), (4736, 4800), (4800, 4801)):
        # sums of signed terms are compared with the size of their terms
        scale = max(np.linalg.norm(gr[a:b]), np.linalg.norm(gr[:mlp_ref.NTRAIN]) * 1e-1)
        assert np.linalg.norm(g[a:b] - gr[a:b]) <= 1e-2 * scale, (a, b)
    assert np.all(g[mlp_ref.NTRAIN:] == 0.0)
    g2, loss2 = m.gradient(Xd, Yd)
    assert np.array_equal(g, g2) and loss == loss2


def test_training_follows_the_reference():
    """Three Adam steps, the last of a ragged minibatch, against the reference."""
    import torch
    from harm_finalwham_amd import harmgpu
    print("case training steps", flush=True)
    rng = np.random.default_rng(9)
    n, batch, lr = 2 * 1000 + 333, 1000, 1e-3
    w = mlp_ref.random_params(8).astype(np.float32)
    X = rng.normal(0.0, 1.5, (n, 8)).astype(np.float32)
    Y = rng.normal(0.0, 2.0, n).astype(np.float32)
    m = harmgpu.Mlp(seed=1)
    m.set_params(w)
    loss = m.train(torch.from_numpy(X).cuda(), torch.from_numpy(Y).cuda(), epochs=1, batch=batch, lr=lr)
    ref, m1, m2, ls = w.astype(np.float64), 0.0, 0.0, []
    for t, a in enumerate(range(0, n, batch)):
        l, g = mlp_ref.loss_grad(ref, X[a:a + batch], Y[a:a + batch], quant=True)
        ls.append(l)
        m1, m2 = 0.9 * m1 + 0.1 * g, 0.999 * m2 + 0.001 * g * g
        ref = ref - lr * (m1 / (1 - 0.9 ** (t + 1))) / (np.sqrt(m2 / (1 - 0.999 ** (t + 1))) + 1e-8)
    assert abs(loss - np.mean(ls)) <= 1e-2 * np.mean(ls)
    # each step moves a weight by about lr; gradients agree to 1e-2 of
    # themselves, a few near zero by their sign
    moved, off = ref - w, m.params() - ref
    assert np.linalg.norm(off) <= 5e-2 * np.linalg.norm(moved)
    y = m.forward(torch.from_numpy(X).cuda()).cpu().numpy()
    yr, _ = mlp_ref.forward(m.params().astype(np.float64), X, quant=True)
    assert np.median(np.abs(y - yr)) <= 1e-5 * max(1.0, np.abs(yr).max())
