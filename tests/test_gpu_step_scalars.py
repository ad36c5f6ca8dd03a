"""hg_step's scalars (dt in; dt, failures and iterations out) and the ndt slots
that its substeps hand on: whatever ran on the context before a step, the step
gives the oracle's state, dt and iteration count bit for bit.  MC and PARA
reset the slots in different launches on the first and on later substeps; the
orders 2, 3 and 4 have one to three later substeps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [("HG_LIM_MC", 2, 0), ("HG_LIM_MC", 3, 0), ("HG_LIM_PARA", 4, 2), ("HG_LIM_WENO5BND", 2, 1)]


@pytest.mark.parametrize("lim,to,olim", CASES)
def test_step_after_anything_matches_oracle(lim, to, olim):
    import torch
    import pyoracle
    from harm_finalwham_amd import harmgpu
    n1, n2, n3, nb = 21, 13, 1, 6
    print("case step scalars", lim, to, flush=True)
    g = harmgpu.Grid(n1, n2, n3, nb=nb, lim=getattr(harmgpu, lim), fluxmethod=harmgpu.HG_FLUX_HLL, timeorder=to)
    g.build_mks_geometry()
    dt = g.init_torus(rin=6.0, rmax=12.0, kappa=1e-3, beta=100.0, randfact=4e-2, seed=5)
    geo = harmgpu.mks_geometry_tables(n1, n2, n3, nb)
    cfg = g.config()
    og = pyoracle.Grid(n1, n2, n3, nb, olim, 1, cfg.gam, cfg.cour, list(cfg.dx), geo["gcov"], geo["gcon"],
                       geo["gcovpert"], geo["gdet"], geo["conn"], geo["r_cent"], timeorder=to, slim=3)
    p = g.get_prims()
    dto = dt
    graph = harmgpu.Graph([g], 1)
    before = [lambda: None, lambda: g.fluxcalc(), lambda: g.step_async(1), lambda: graph.launch(), lambda: None]
    for n, run in enumerate(before):
        run()
        torch.cuda.synchronize()
        g.set_prims(p)
        dt, nf, it = g.step_ch(dt)
        p, dto, nfo, ito = og.step(p, dto)
        assert (dt, nf, it) == (dto, nfo, ito), n
        assert np.array_equal(g.get_prims(), p), n
    graph.close()
    g.close()
