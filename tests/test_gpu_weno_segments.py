"""The split of the marching reconstruction's lines into segments over grids at
the rule's ends: fewer points than a segment's least length times two, one
segment, many segments with a short last one, the length from which two is the
least.  One RK2 step, the oracle's bit for bit (a segment's result does not
depend on where it starts)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(8, 6, 1), (6, 6, 6), (33, 35, 1), (7, 94, 1), (300, 13, 1), (5, 8, 94)])
def test_segmented_reconstruction_step_matches_oracle(shape):
    import pyoracle
    from harm_finalwham_amd import harmgpu
    n1, n2, n3 = shape
    nb = 6
    print("case weno segments", shape, flush=True)
    ring = dict(Rin=6.0, Rout=20.0) if n1 < 16 else {}
    g = harmgpu.Grid(n1, n2, n3, nb=nb)
    g.build_mks_geometry(**ring)
    dt = g.init_torus(rin=6.0, rmax=12.0, kappa=1e-3, beta=100.0, randfact=4e-2, seed=9)
    geo = harmgpu.mks_geometry_tables(n1, n2, n3, nb, **ring)
    cfg = g.config()
    og = pyoracle.Grid(n1, n2, n3, nb, 1, 1, cfg.gam, cfg.cour, list(cfg.dx), geo["gcov"], geo["gcon"],
                       geo["gcovpert"], geo["gdet"], geo["conn"], geo["r_cent"])
    p, dto, nfo, ito = og.step(g.get_prims(), dt)
    dtg, nf, it = g.step_ch(dt)
    assert (dtg, nf, it) == (dto, nfo, ito)
    assert np.array_equal(g.get_prims(), p)
    g.close()
