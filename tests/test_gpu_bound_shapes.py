"""The ghost fill in one launch (bounds.fishmon.c:29) over grid shapes where its
blocks meet: one to three directions, extents equal to the ghost layers, more
ghost layers than lanes per row end, extents on both sides of a block.  Every
zone of the array, the rows POLEDEATH clears included, is the oracle's bit for
bit, on a first and on a repeated call."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [((37, 1, 1), 3), ((2, 12, 1), 9), ((12, 9, 1), 9), ((6, 6, 6), 6), ((19, 13, 7), 6), ((5, 11, 11), 10),
          ((1, 8, 8), 3), ((64, 33, 3), 3), ((3, 3, 130), 3)]


@pytest.mark.parametrize("shape,nb", SHAPES)
def test_ghost_fill_matches_oracle(shape, nb):
    import pyoracle
    from harm_finalwham_amd import harmgpu
    n1, n2, n3 = shape
    print("case ghost fill", shape, nb, flush=True)
    g = harmgpu.Grid(n1, n2, n3, nb=nb, lim=harmgpu.HG_LIM_MC, fluxmethod=harmgpu.HG_FLUX_LAXF)
    # two zones and nine ghost layers: a narrow ring far out, so that no ghost is inside the hole
    ring = dict(Rin=20.0, Rout=24.0) if n1 == 2 else {}
    g.build_mks_geometry(**ring)
    geo = harmgpu.mks_geometry_tables(n1, n2, n3, nb, **ring)
    cfg = g.config()
    og = pyoracle.Grid(n1, n2, n3, nb, 0, 0, cfg.gam, cfg.cour, list(cfg.dx), geo["gcov"], geo["gcon"],
                       geo["gcovpert"], geo["gdet"], geo["conn"], geo["r_cent"])
    rng = np.random.default_rng(n1 * 1000 + n2 * 10 + n3)
    p = rng.uniform(0.1, 1.0, og.shape)
    p[..., 2:5] = rng.normal(0.0, 0.3, og.shape[:-1] + (3,))
    p[..., 5:8] = rng.normal(0.0, 0.1, og.shape[:-1] + (3,))
    p[..., 3][rng.random(og.shape[:-1]) < 0.1] = -0.0
    g.set_prims(p)
    for call in range(2):
        g.bound_prim()
        p = og.bound(p)
        q = g.get_prims()
        assert np.array_equal(q, p), (call, np.argwhere(q != p)[:8])
        assert np.array_equal(np.signbit(q), np.signbit(p)), call
    g.close()
