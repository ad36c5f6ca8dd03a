"""The conserved totals are the reference's sequential double sums: the device
adds blocks of numbers out of order where the rounding of every addition is
known beforehand.  States whose sums stay in one binade, cross binades all the
time (fields of alternating sign, magnitudes over many decades), meet ties
(numbers of few bits), cancel to zero and stay zero, over counts that no block
or piece divides, against a sequential sum of the oracle's conserved
densities, bit for bit; and the div B maximum with its first place."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def state(kind, shape, rng):
    p = np.zeros(shape + (8,))
    p[..., 0], p[..., 1] = 1e-2, 1e-3
    if kind == "torus":
        return None
    if kind == "decades":
        p[..., 0] = 10.0 ** rng.uniform(-12, 0, shape)
        p[..., 1] = p[..., 0] * 10.0 ** rng.uniform(-6, 0, shape)
        p[..., 2:5] = rng.normal(0, 0.05, shape + (3,)) / np.array([1.0, 10.0, 10.0])
        p[..., 5:] = rng.choice([-1.0, 1.0], shape + (3,)) * 10.0 ** rng.uniform(-14, -2, shape + (3,))
    if kind == "waves":
        x = np.arange(np.prod(shape)).reshape(shape)
        for c, period in ((5, 2), (6, 64), (7, 1500)):
            p[..., c] = 1e-3 * np.sin(2 * np.pi * x / period) * (1 + 1e-3 * rng.normal(size=shape))
    if kind == "ties":
        p[..., 5:] = rng.integers(-3, 4, shape + (3,)) * 2.0 ** rng.integers(-12, 0, shape + (3,))
        p[..., 0] = 2.0 ** -rng.integers(1, 8, shape)
        p[..., 1] = 2.0 ** -10
    return p


@pytest.mark.parametrize("size", [(40, 30, 13), (131, 65, 1), (9, 7, 1)])
@pytest.mark.parametrize("kind", ["torus", "decades", "waves", "ties"])
def test_totals_are_sequential_sums(size, kind):
    import pyoracle
    from harm_finalwham_amd import harmgpu as h
    print("case ordered sums", size, kind, flush=True)
    nb = 3
    g = h.Grid(*size, nb=nb, lim=h.HG_LIM_MC, fluxmethod=h.HG_FLUX_LAXF)
    g.build_mks_geometry()
    cfg = g.config()
    t = h.mks_geometry_tables(*size, nb)
    og = pyoracle.Grid(*size, nb, 0, 0, cfg.gam, cfg.cour, list(cfg.dx), t["gcov"], t["gcon"], t["gcovpert"],
                       t["gdet"], t["conn"], t["r_cent"])
    p = state(kind, g.shape[:3], np.random.default_rng(5))
    if p is None:
        g.init_torus(rin=6.0, rmax=12.0, kappa=1e-3, beta=100.0, randfact=4e-2, seed=3)
        p = g.get_prims()
    p = og.bound(p)
    g.set_prims(p)
    g.fluxcalc()
    d = g.diagnostics()
    U = np.asarray(og.cons_from_prims(p))
    if U.shape == p.shape:
        c = [slice(nb, -nb) if n > 1 else slice(None) for n in size]
        U = U[tuple(c)]
    dv = cfg.dx[1] * cfg.dx[2] * cfg.dx[3]
    for pl in range(8):
        terms = (U[..., pl] * dv).ravel()
        ref = np.cumsum(np.concatenate([[0.0], terms]))[-1]
        assert d["cons"][pl] == ref, (pl, d["cons"][pl], ref)
    assert np.isfinite(d["divbmax"]) and d["divbmax"] >= d["divbavg"] >= 0.0
    # a second call on the same state says the same
    e = g.diagnostics()
    assert np.array_equal(d["cons"], e["cons"]) and d["divbmax_ijk"] == e["divbmax_ijk"]
    assert np.array_equal(d["pdotterms"], e["pdotterms"])
    g.close()
