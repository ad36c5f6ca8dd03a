"""The flux kernels that park one side's results in LDS, a place per wavefront of
the launch: one step with blocks of one and two wavefronts against blocks of
four, for every such kernel and both forms of the metric.  State, dt and
counters bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lim,fv", [("HG_LIM_WENO5BND", False), ("HG_LIM_WENO5BND", True), ("HG_LIM_PARA", False),
                                    ("HG_LIM_PARA", True)])
@pytest.mark.parametrize("captured", [False, True])  # a captured step takes the full metric's kernels
def test_parked_fluxes_by_block_size(lim, fv, captured):
    import torch
    from harm_finalwham_amd import harmgpu
    print("case flux blocks", lim, fv, captured, flush=True)
    out = []
    for bs in (256, 128, 64):
        g = harmgpu.Grid(67, 35, 9, nb=6, lim=getattr(harmgpu, lim), fluxmethod=harmgpu.HG_FLUX_HLL,
                         doenoflux=harmgpu.HG_ENOFINITEVOLUME if fv else harmgpu.HG_NOENOFLUX)
        g.build_mks_geometry()
        dt = g.init_torus(rin=6.0, rmax=12.0, kappa=1e-3, beta=100.0, randfact=4e-2, seed=4)
        g.set_tune(harmgpu.HgTune(bs_flux=bs, bs_emf=256, bs_update=256, bs_invert=256, weno_xwaves=4, concurrent=0))
        if captured:
            g.set_dt(dt)
            graph = harmgpu.Graph([g], 1)
            graph.launch()
            torch.cuda.synchronize()
            graph.close()
            out.append(((g.get_dt(),), g.get_prims()))
        else:
            out.append((g.step_ch(dt), g.get_prims()))
        g.close()
    for o in out[1:]:
        assert o[0] == out[0][0]
        assert np.array_equal(o[1], out[0][1])
