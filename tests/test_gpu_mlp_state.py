"""What a caller can read of a network in training: setting the parameters it
reads back changes nothing, and hg_mlp_gradient differentiates at them."""
import numpy as np
import pytest

import mlp_ref

pytestmark = pytest.mark.gpu


def _samples(n=3 * 256 + 40):
    import torch
    rng = np.random.default_rng(31)
    X = torch.from_numpy(rng.normal(0.0, 1.5, (n, 8)).astype(np.float32)).cuda()
    Y = torch.from_numpy(rng.normal(0.0, 2.0, n).astype(np.float32)).cuda()
    return X, Y


def _net(w):
    from harm_finalwham_amd import harmgpu
    m = harmgpu.Mlp(seed=1)
    m.set_params(w)
    return m


# at 2^-30 a step is far below the FP32 spacing of a weight
@pytest.mark.parametrize("lr", [2.0 ** -8, 2.0 ** -30])
def test_parameters_set_as_read_leave_training_alone(lr):
    print("case parameters set as read, rate", lr, flush=True)
    w = mlp_ref.random_params(3).astype(np.float32)
    X, Y = _samples()
    a, b = _net(w), _net(w)
    for k in range(4):
        la = a.train(X, Y, epochs=2, batch=256, lr=lr)
        lb = b.train(X, Y, epochs=2, batch=256, lr=lr)
        assert la == lb
        b.set_params(b.params())
    assert not np.array_equal(a.params()[:4801], w[:4801])
    assert np.array_equal(a.params(), b.params())


def test_other_parameters_start_without_the_old_remainders():
    print("case other parameters", flush=True)
    w, v = (mlp_ref.random_params(s).astype(np.float32) for s in (4, 5))
    X, Y = _samples()
    a = _net(w)
    a.train(X, Y, epochs=2, batch=256, lr=2.0 ** -8)
    a.set_params(v)
    b = _net(v)
    ga, la = a.gradient(X, Y)
    gb, lb = b.gradient(X, Y)
    assert la == lb and np.array_equal(ga, gb)


def test_gradient_after_training_is_at_the_parameters_read():
    print("case gradient after training", flush=True)
    w = mlp_ref.random_params(6).astype(np.float32)
    X, Y = _samples()
    a = _net(w)
    a.train(X, Y, epochs=2, batch=256, lr=2.0 ** -8)
    b = _net(a.params())
    ga, la = a.gradient(X, Y)
    gb, lb = b.gradient(X, Y)
    assert la == lb and np.array_equal(ga, gb)
