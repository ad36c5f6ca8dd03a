"""The kernels that leave out the zeros of the Kerr-Schild metric against the
ones that read the whole metric, on the same tables: one of those zeros is
made -0 in a corner ghost zone, which sends the grid to the general kernels
and changes no number.  A metric with every entry nonzero is compared with the
oracle, and a graph whose grids change their geometry after it was made with
the grids' own steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SCHEMES = [
    ("MC + LaxF, RK2, 33x17", (33, 17, 1), 3, ("HG_LIM_MC", "HG_FLUX_LAXF", 2, 0), "HG_C2P_FP64"),
    ("PARA + HLL, RK4, finite volume, 21x13x5", (21, 13, 5), 3, ("HG_LIM_PARA", "HG_FLUX_HLL", 4, 3), "HG_C2P_FP64"),
    ("WENO5BND + HLL, RK2, 19x12x7", (19, 12, 7), 6, ("HG_LIM_WENO5BND", "HG_FLUX_HLL", 2, 0), "HG_C2P_FP64"),
    ("WENO5BND + HLL, RK3, mixed inversion, 70x9", (70, 9, 1), 6, ("HG_LIM_WENO5BND", "HG_FLUX_HLL", 3, 0),
     "HG_C2P_MIXED"),
]


def grid(size, nb, scheme, seed=11, a=0.9375):
    from harm_finalwham_amd import harmgpu as h
    lim, flux, to, fv = scheme
    g = h.Grid(*size, nb=nb, lim=getattr(h, lim), fluxmethod=getattr(h, flux), timeorder=to, doenoflux=fv)
    g.build_mks_geometry(a=a)
    dt = g.init_torus(rin=6.0, rmax=12.0, kappa=1e-3, beta=100.0, randfact=4e-2, seed=seed)
    return g, dt


def tables(size, nb, general, a=0.9375):
    from harm_finalwham_amd import harmgpu as h
    t = h.mks_geometry_tables(*size, nb, a=a)
    t.pop("dx")
    if general:
        assert t["gcov"][0, 0, 6, 0, 2] == 0.0
        t["gcov"][0, 0, 6, 0, 2] = -0.0
    return t


@pytest.mark.parametrize("case", SCHEMES, ids=[c[0] for c in SCHEMES])
def test_general_kernels_give_the_same_numbers(case):
    from harm_finalwham_amd import harmgpu as h
    label, size, nb, scheme, mode = case
    print("case metric forms", label, flush=True)
    out = []
    for general in (False, True):
        g, dt = grid(size, nb, scheme)
        g.upload_geometry(**tables(size, nb, general))
        g.set_inversion(getattr(h, mode))
        F, ndt = g.fluxcalc()
        got = [ndt, *F]
        for _ in range(3):
            dt, nf, it = g.step_ch(dt)
            got += [dt, nf, it]
        out.append(got + [g.get_prims(), g.diagnostics()["cons"]])
        g.close()
    for k, (a, b) in enumerate(zip(*out)):
        assert np.array_equal(a, b), k


def test_full_metric_matches_oracle():
    import pyoracle
    from harm_finalwham_amd import harmgpu as h
    size, nb = (22, 14, 6), 6
    print("case full metric", flush=True)
    g, dt0 = grid(size, nb, ("HG_LIM_WENO5BND", "HG_FLUX_HLL", 2, 0))
    t = tables(size, nb, False)
    # every entry nonzero: theta mixed with the others by a hundredth of the
    # diagonal, symmetric, with the inverse and the lapse that belong to it
    gc = t["gcov"]
    d = np.sqrt(np.abs(np.einsum("...ii->...i", gc)))
    gc += 0.01 * np.where(gc == 0.0, d[..., :, None] * d[..., None, :], 0.0)
    t["gcov"] = 0.5 * (gc + gc.swapaxes(-1, -2))
    gi = np.linalg.inv(t["gcov"])
    t["gcon"] = 0.5 * (gi + gi.swapaxes(-1, -2))
    t["gcovpert"][..., 0] = 1.0 + t["gcov"][..., 0, 0]
    g.upload_geometry(**t)
    cfg = g.config()
    og = pyoracle.Grid(*size, nb, 1, 1, cfg.gam, cfg.cour, list(cfg.dx), t["gcov"], t["gcon"], t["gcovpert"],
                       t["gdet"], t["conn"], t["r_cent"])
    p = og.bound(g.get_prims())
    g.set_prims(p)
    F, ndt = g.fluxcalc()
    oF, ondt = og.fluxcalc(p)[:2]
    assert np.array_equal(ndt, ondt)
    c = [slice(nb, -nb)] * 3
    for k in range(3):
        assert np.array_equal(F[k][tuple(c)], oF[k][tuple(c)]), k
    dt, _, _ = g.step_ch(dt0)
    po, dto, _, _ = og.step(p, dt0)
    assert dt == dto
    assert np.array_equal(g.get_prims(), po)
    g.close()


@pytest.mark.parametrize("grouped", [False, True])
def test_graph_follows_a_changed_geometry(grouped):
    import torch
    from harm_finalwham_amd import harmgpu as h
    print("case graph with a changed geometry", grouped, flush=True)
    scheme, nb = ("HG_LIM_WENO5BND", "HG_FLUX_HLL", 2, 0), 6
    sizes = [(24, 16, 1), (17, 12, 7)]
    batch = [grid(s, nb, scheme) for s in sizes]
    alone = [grid(s, nb, scheme) for s in sizes]
    for (b, dt), (a, _) in zip(batch, alone):
        b.set_dt(dt)
        a.set_dt(dt)
    graph = h.Graph([b for b, _ in batch], 2, grouped=grouped)

    def both():
        graph.launch()
        for a, _ in alone:
            a.step_async(2)
        torch.cuda.synchronize()
        for (b, _), (a, _) in zip(batch, alone):
            assert b.get_dt() == a.get_dt()
            assert np.array_equal(b.get_prims(), a.get_prims())

    both()
    # the same numbers through the general kernels, then another spin
    batch[1][0].upload_geometry(**tables(sizes[1], nb, True))
    both()
    for pair in (batch, alone):
        pair[0][0].upload_geometry(**tables(sizes[0], nb, True, a=0.5))
    both()
    graph.close()
    for g, _ in batch + alone:
        g.close()
