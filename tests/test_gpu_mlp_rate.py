"""Training takes the rate it is given: hg_mlp_train the FP32 number,
hg_mlp_train_rate (and Mlp.train) the FP64 one, neither a decimal near it."""
import ctypes as C

import numpy as np
import pytest

import mlp_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lr", [2e-3, 1.0 / 3.0, 1e-2])
def test_the_rate_given_is_the_rate_taken(lr):
    import torch
    from harm_finalwham_amd import harmgpu
    print("case rate", lr, flush=True)
    rng = np.random.default_rng(17)
    n, batch, epochs = 20 * 256, 256, 4
    X = torch.from_numpy(rng.normal(0.0, 1.5, (n, 8)).astype(np.float32)).cuda()
    Y = torch.from_numpy(rng.normal(0.0, 2.0, n).astype(np.float32)).cuda()
    w = mlp_ref.random_params(9).astype(np.float32)

    def params(train):
        m = harmgpu.Mlp(seed=1)
        m.set_params(w)
        train(m)
        return m.params()

    def in_float(m):
        loss = C.c_float()
        assert harmgpu.lib().hg_mlp_train(m.h, n, C.c_void_p(X.data_ptr()), C.c_void_p(Y.data_ptr()), epochs, batch,
                                          C.c_float(lr), C.byref(loss), None) == 0

    f = params(in_float)
    as_float = params(lambda m: m.train(X, Y, epochs=epochs, batch=batch, lr=float(np.float32(lr))))
    as_double = params(lambda m: m.train(X, Y, epochs=epochs, batch=batch, lr=lr))
    assert np.array_equal(f, as_float)
    # the two rates are 1e-8 to 5e-8 apart: some weights of a training's end are too
    assert not np.array_equal(f, as_double)
