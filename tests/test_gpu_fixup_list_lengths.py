"""post_fixup of a small grid takes one launch while its lists are short and four
while they are long: calls with no, few, many, all and few zones failed or
fast, on one context, so that each way follows the other, against the oracle.
Primitives and codes bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CODES = np.array([101, 4, 2, 9, 10, 11])


@pytest.mark.parametrize("shape", [(61, 47, 1), (24, 16, 11)])
def test_lists_of_changing_length_match_oracle(shape):
    import pyoracle
    from harm_finalwham_amd import harmgpu
    nb = 3
    g = harmgpu.Grid(*shape, nb=nb, lim=harmgpu.HG_LIM_MC, fluxmethod=harmgpu.HG_FLUX_LAXF)
    g.build_mks_geometry()
    g.init_torus(rin=6.0, rmax=12.0, kappa=1e-3, beta=100.0, randfact=4e-2, seed=3)
    geo = harmgpu.mks_geometry_tables(*shape, nb)
    cfg = g.config()
    og = pyoracle.Grid(*shape, nb, 0, 0, cfg.gam, cfg.cour, list(cfg.dx), geo["gcov"], geo["gcon"],
                       geo["gcovpert"], geo["gdet"], geo["conn"], geo["r_cent"])
    rng = np.random.default_rng(sum(shape))
    start = g.get_prims()
    c = tuple(slice(nb, -nb) if n > 1 else slice(None) for n in shape)
    for call, (failing, fast) in enumerate([(0.0, 0.0), (0.02, 0.02), (0.6, 0.0), (0.6, 0.1), (0.0, 0.0), (1.0, 1.0),
                                            (0.01, 1.0), (0.02, 0.02), (0.02, 0.0)]):
        print("case lists", shape, "failing", failing, "fast", fast, flush=True)
        p = start.copy()
        p[..., 2][rng.random(p.shape[:-1]) < fast] += 3.0
        codes = np.where(rng.random(shape) < failing, rng.choice(CODES, shape), 0).astype(np.int32)
        g.set_prims(p)
        g.post_fixup(codes=codes, finalstep=call % 2)
        po, fo = og.post_fixup_sequence(p, codes, call % 2)
        assert np.array_equal(g.get_pflag(), fo[c]), call
        assert np.array_equal(g.get_prims(), po), call
    g.close()
