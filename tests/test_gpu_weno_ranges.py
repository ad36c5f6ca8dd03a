"""WENO5BND reads the monotonicity indicator and its weights' quotients off
their operands where those decide the result, and takes the reference's own
divisions elsewhere.  Lines that sit on both sides of each of those lines:
blocks that are constant, that vary by a rounding error, by the indicator's
cutoff and its neighbourhood, and by much more; fields and velocities that
are zero or so small that their squares underflow.  The interface states of
every direction, and so the fluxes and time-step limits, must be the
oracle's bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

AMPS = [0.0, 1.2e-16, 3e-14, 1e-13, 4e-13, 1e-11, 1e-3, 0.4]
SCALES = [0.0, 1e-200, 1e-163, 1e-155, 1e-148, 1e-120, 1e-80, 1e-30, 1e-3]


def blocky(rng, shape, values, size):
    """One of `values` per block of size^3 zones."""
    b = [(-(-n // size)) for n in shape]
    v = np.array(values)[rng.integers(len(values), size=b)]
    for ax in range(3):
        v = np.repeat(v, size, axis=ax)
    return v[:shape[0], :shape[1], :shape[2]]


@pytest.mark.parametrize("size,seed", [((40, 21, 9), 1), ((61, 70, 1), 2), ((17, 12, 33), 3)])
def test_reconstruction_at_its_decisions(size, seed):
    import pyoracle
    from harm_finalwham_amd import harmgpu as h
    print("case WENO ranges", size, seed, flush=True)
    nb = 6
    g = h.Grid(*size, nb=nb)
    g.build_mks_geometry()
    cfg = g.config()
    t = h.mks_geometry_tables(*size, nb)
    og = pyoracle.Grid(*size, nb, 1, 1, cfg.gam, cfg.cour, list(cfg.dx), t["gcov"], t["gcon"], t["gcovpert"],
                       t["gdet"], t["conn"], t["r_cent"])
    rng = np.random.default_rng(seed)
    p = np.empty(g.shape)
    sh = g.shape[:3]
    for pl, base in enumerate((1e-3, 1e-4, 1e-2, 1e-3, 1e-3, 1e-3, 1e-3, 1e-3)):
        noise = 1.0 + blocky(rng, sh, AMPS, 4) * rng.uniform(-1, 1, sh)
        if pl >= 2:
            noise *= blocky(rng, sh, SCALES, 7) / 1e-3 * blocky(rng, sh, [1.0, 1.0, -1.0], 3)
        p[..., pl] = base * noise
    p = og.bound(p)
    g.set_prims(p)
    F, ndt = g.fluxcalc()
    oF, ondt = og.fluxcalc(p)
    assert np.array_equal(ndt, ondt)
    c = [slice(nb, -nb) if n > 1 else slice(None) for n in size]
    for k in range(3):
        if size[k] > 1:
            assert np.isfinite(oF[k]).all()
            assert np.array_equal(F[k][tuple(c)], oF[k][tuple(c)]), k
    g.close()
