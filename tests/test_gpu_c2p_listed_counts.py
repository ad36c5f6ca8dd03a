"""The step counts of zones that the FP32 phase leaves to the list: those of
HG_C2P_REFINED, which inverts them.  At scales outside FP32's range every zone
is on the list, so every count, code and solved zone can be compared."""
import numpy as np
import pytest

from test_gpu_newton_ranges import N, _batch, _solve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gam", [4.0 / 3.0, 5.0 / 3.0])
@pytest.mark.parametrize("exp4", [-75, 75])
def test_listed_zones_have_the_converged_roots_counts(exp4, gam):
    from harm_finalwham_amd import harmgpu
    print("case listed counts, 4 **", exp4, "gam", gam, flush=True)
    rec = _batch(exp4, gam)
    pr, fr, ir = _solve(rec, gam, harmgpu.HG_C2P_REFINED)
    pm, fm, im = _solve(rec, gam, harmgpu.HG_C2P_MIXED)
    listed = harmgpu.c2p_fallbacks()
    print("listed", listed, "of", N, "counts that differ", int((im != ir).sum()), flush=True)
    # the others failed in the set-up, without a step in either mode
    assert listed >= N - int((ir == 0).sum())
    assert np.array_equal(im, ir)
