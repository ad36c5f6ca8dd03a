"""FP64 inversions whose Newton iteration meets a step that is not finite:
magnetisations up to 1e20 and guesses whose energy is off by up to 1e8 either
way, where the determinant of the Jacobian is lost to rounding.  Such a step is
no convergence: the reference takes W back and goes on, so failure codes,
iteration counts and solutions are the oracle's, bit for bit, and the converged
root keeps the codes."""
import numpy as np
import pytest

from c2p_sample import sample_c2p

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gam", [4.0 / 3.0, 5.0 / 3.0])
def test_infinite_steps_are_not_convergence(gam):
    import torch
    import pyoracle
    from harm_finalwham_amd import harmgpu
    n = 1 << 17
    print("case infinite steps, gam", gam, flush=True)
    rng = np.random.default_rng(404)
    gcov, gcon, gdet, gpert, p, guess = sample_c2p(n, rng, sigma=(1e-4, 1e20))
    guess[:, 1] *= 10.0 ** rng.uniform(-8, 8, n)
    U = pyoracle.primtoU_batch(gcov, gcon, gdet, gpert, p, gam)
    po, fo, io = pyoracle.c2p_batch(gcov, gcon, gdet, gpert, U, gam, guess)
    assert (fo == 0).sum() > n // 10 and (fo != 0).sum() > n // 10
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).to("cuda:0")
    args = [t(U.T), t(gcov.reshape(n, 16).T), t(gcon.reshape(n, 16).T), t(gdet), t(gpert[:, 0])]
    for mode in (harmgpu.HG_C2P_FP64, harmgpu.HG_C2P_REFINED):
        pr = t(guess.T)
        pflag = torch.zeros(n, dtype=torch.int32, device="cuda:0")
        iters = torch.zeros_like(pflag)
        harmgpu.utoprim_batch(*args, pr, pflag, iters, gam=gam, mode=mode)
        f, it = pflag.cpu().numpy(), iters.cpu().numpy()
        print("mode", mode, "codes that differ", int((f != fo).sum()), flush=True)
        assert np.array_equal(f, fo)
        if mode == harmgpu.HG_C2P_FP64:
            assert np.array_equal(it, io)
            assert np.array_equal(pr.cpu().numpy().T, po, equal_nan=True)
