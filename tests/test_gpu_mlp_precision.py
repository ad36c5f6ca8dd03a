"""Training keeps its 64 bits: two epochs of minibatches, the last one ragged,
against the same Adam steps in FP64 with the network's own number formats
(hidden weights and activations rounded to BF16, the input a BF16 pair)."""
import numpy as np
import pytest

import mlp_ref

pytestmark = pytest.mark.gpu

N, BATCH = 15 * 512 + 131, 512


def _bf(v):
    return mlp_ref.bf16(np.asarray(v, np.float32)).astype(np.float64)


def _adam64(w, X, Y, epochs, lr):
    """The parameters after each epoch of Adam in FP64, and the last one's mean minibatch loss."""
    mu, sd, w = w[4801:4809].astype(np.float64), w[4809:].astype(np.float64), w[:4801].astype(np.float64)
    x = (X.astype(np.float64) - mu) / sd
    x = _bf(x) + _bf(x - _bf(x))
    y = Y.astype(np.float64)
    m1, m2, t, out = np.zeros_like(w), np.zeros_like(w), 0, []
    for _ in range(epochs):
        ls = []
        for a in range(0, len(y), BATCH):
            xb, yb = x[a:a + BATCH], y[a:a + BATCH]
            W1, W2, w3 = _bf(w[:512]).reshape(8, 64), _bf(w[576:4672]).reshape(64, 64), w[4736:4800]
            h1 = np.tanh(xb @ W1 + w[512:576])
            h2 = np.tanh(_bf(h1) @ W2 + w[4672:4736])
            r = h2 @ w3 + w[4800] - yb
            ls.append(np.mean(r * r))
            d = 2.0 * r / len(yb)
            d2 = d[:, None] * w3 * (1.0 - h2 * h2)
            d1 = (d2 @ W2.T) * (1.0 - h1 * h1)
            g = np.concatenate([(xb.T @ d1).ravel(), d1.sum(0), (_bf(h1).T @ d2).ravel(), d2.sum(0), h2.T @ d,
                                [d.sum()]])
            t += 1
            m1, m2 = 0.9 * m1 + 0.1 * g, 0.999 * m2 + 0.001 * g * g
            w = w - lr * (m1 / (1 - 0.9 ** t)) / (np.sqrt(m2 / (1 - 0.999 ** t)) + 1e-8)
        out.append(w)
    return out, np.mean(ls)


def _samples(seed):
    rng = np.random.default_rng(seed)
    w = mlp_ref.random_params(seed).astype(np.float32)
    X = rng.normal(0.0, 1.5, (N, 8)).astype(np.float32)
    Y = rng.normal(0.0, 2.0, N).astype(np.float32)
    return w, X, Y


def _net(w):
    from harm_finalwham_amd import harmgpu
    m = harmgpu.Mlp(seed=1)
    m.set_params(w)
    return m


# 2^-8 and 2^-30 are the same numbers in FP32 and FP64.  At 2^-8 the weights move
# by 0.1 and the BF16 roundings change; at 2^-30 a step is a thirtieth of an ulp
# of a weight of 0.3, and only what the weights carry below FP32 moves them.
@pytest.mark.parametrize("lr", [2.0 ** -8, 2.0 ** -30])
def test_training_is_the_64_bit_training(lr):
    import torch
    print("case training in 64 bits, rate", lr, flush=True)
    w, X, Y = _samples(12)
    ref, ls = _adam64(w, X, Y, 2, lr)
    m = _net(w)
    loss = m.train(torch.from_numpy(X).cuda(), torch.from_numpy(Y).cuda(), epochs=2, batch=BATCH, lr=lr)
    # the parameters' rounding to FP32, and 1e-9 for the sums' order
    off = np.abs(m.params()[:4801] - ref[-1])
    print("off by", off.max(), "relative", (off / np.abs(ref[-1]).clip(1e-3)).max(), flush=True)
    assert (off <= 2.0 ** -24 * np.abs(ref[-1]) + 1e-9).all()
    assert abs(loss - ls) <= 1e-6 * ls


def test_gradient_is_that_of_64_bits():
    import torch
    print("case gradient in 64 bits", flush=True)
    w, X, Y = _samples(13)
    mu, sd = w[4801:4809].astype(np.float64), w[4809:].astype(np.float64)
    x = (X.astype(np.float64) - mu) / sd
    x = _bf(x) + _bf(x - _bf(x))
    v = w[:4801].astype(np.float64)
    W1, W2, w3 = _bf(v[:512]).reshape(8, 64), _bf(v[576:4672]).reshape(64, 64), v[4736:4800]
    h1 = np.tanh(x @ W1 + v[512:576])
    h2 = np.tanh(_bf(h1) @ W2 + v[4672:4736])
    r = h2 @ w3 + v[4800] - Y.astype(np.float64)
    d = 2.0 * r / N
    d2 = d[:, None] * w3 * (1.0 - h2 * h2)
    d1 = (d2 @ W2.T) * (1.0 - h1 * h1)
    ref = np.concatenate([(x.T @ d1).ravel(), d1.sum(0), (_bf(h1).T @ d2).ravel(), d2.sum(0), h2.T @ d, [d.sum()]])
    g, loss = _net(w).gradient(torch.from_numpy(X).cuda(), torch.from_numpy(Y).cuda())
    # FP32 rounding of each entry, and the sums' order at the size of the largest
    assert (np.abs(g[:4801] - ref) <= 2.0 ** -23 * np.abs(ref) + 1e-9 * np.abs(ref).max()).all()
    assert abs(loss - np.mean(r * r)) <= 1e-6 * np.mean(r * r)
