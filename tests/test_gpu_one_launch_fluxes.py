"""The fluxes of all directions in one launch (small grids, default launch
shapes) against the launches per direction, which a tuned context takes
(hg_set_tune concurrent 0): one step of every scheme with one, two and three
active directions, on both sides of the size where the rule ends, plain and
replayed from a captured graph.  State, dt and counters bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SCHEMES = [("HG_LIM_WENO5BND", "HG_FLUX_HLL", 2, False), ("HG_LIM_MC", "HG_FLUX_LAXF", 2, False),
           ("HG_LIM_PARA", "HG_FLUX_HLL", 4, True), ("HG_LIM_WENO5BND", "HG_FLUX_HLL", 2, True)]
SHAPES = [(33, 1, 1), (1, 17, 1), (20, 13, 1), (21, 1, 9), (1, 9, 8), (19, 11, 7), (130, 66, 40)]


@pytest.mark.parametrize("scheme", SCHEMES, ids=lambda s: "%s-%s-%d-%s" % s)
@pytest.mark.parametrize("shape", SHAPES)
def test_one_launch_matches_launches_per_direction(scheme, shape):
    import torch
    from harm_finalwham_amd import harmgpu
    lim, flux, to, fv = scheme
    print("case one launch", scheme, shape, flush=True)
    out = []
    for concurrent in (0, 1):
        g = harmgpu.Grid(*shape, nb=6, lim=getattr(harmgpu, lim), fluxmethod=getattr(harmgpu, flux), timeorder=to,
                         doenoflux=harmgpu.HG_ENOFINITEVOLUME if fv else harmgpu.HG_NOENOFLUX)
        g.build_mks_geometry()
        if 1 in shape[:2]:
            g.set_prims(np.broadcast_to([0.1, 0.01, 0.0, 0.0, 0.05, 0.01, 0.0, 0.01], g.shape).copy())
            g.bound_prim()
            dt = 1e-3
        else:
            dt = g.init_torus(rin=6.0, rmax=12.0, kappa=1e-3, beta=100.0, randfact=4e-2, seed=2)
        g.set_tune(harmgpu.HgTune(bs_flux=256, bs_emf=256, bs_update=256, bs_invert=256, weno_xwaves=4,
                                  concurrent=concurrent))
        dt, nf, it = g.step_ch(dt)
        p1 = g.get_prims()
        graph = harmgpu.Graph([g], 1)
        graph.launch()
        torch.cuda.synchronize()
        out.append((dt, nf, it, p1, g.get_prims()))
        graph.close()
        g.close()
    assert out[0][:3] == out[1][:3]
    assert np.array_equal(out[0][3], out[1][3])
    assert np.array_equal(out[0][4], out[1][4])
