"""A state goes in and out of a context's own device, whichever device the
caller has set, as a copy of memory does."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(20, 12, 1), (130, 40, 24)])  # one piece, several with threads
def test_states_move_with_another_device_set(size):
    import torch
    from harm_finalwham_amd import harmgpu
    if torch.cuda.device_count() < 2:
        pytest.skip("needs two GPUs: with one there is no other device to set")
    print("case state copies, another device", size, flush=True)
    with torch.cuda.device(1):
        g = harmgpu.Grid(*size, nb=6)
    p = np.random.default_rng(2).normal(size=g.shape)
    with torch.cuda.device(0):
        g.set_prims(p)
        assert np.array_equal(g.get_prims(), p)
        assert torch.cuda.current_device() == 0
    g.close()
