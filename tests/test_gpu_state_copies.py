"""States that pass between the host and the device in several pieces: rows
and row lengths that no piece or tile divides, in 3-D and 2-D, against the
oracle stepping the same state; two threads reading one context."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(70, 40, 9), (201, 151, 1), (13, 100, 17)])
def test_states_of_several_pieces(size):
    import pyoracle
    from harm_finalwham_amd import harmgpu as h
    print("case state copies", size, flush=True)
    nb = 6
    g = h.Grid(*size, nb=nb)
    assert np.prod(g.shape) * 8 > 2 << 20
    g.build_mks_geometry()
    dt0 = g.init_torus(rin=6.0, rmax=12.0, kappa=1e-3, beta=100.0, randfact=4e-2, seed=3)
    p0 = g.get_prims()
    cfg = g.config()
    t = h.mks_geometry_tables(*size, nb)
    og = pyoracle.Grid(*size, nb, 1, 1, cfg.gam, cfg.cour, list(cfg.dx), t["gcov"], t["gcon"], t["gcovpert"],
                       t["gdet"], t["conn"], t["r_cent"])
    mark = np.arange(p0.size, dtype=np.float64).reshape(p0.shape)
    g.set_prims(mark)
    got = [None, None]

    def read(k):
        got[k] = g.get_prims()

    team = [threading.Thread(target=read, args=(k,)) for k in range(2)]
    for t_ in team:
        t_.start()
    for t_ in team:
        t_.join()
    assert np.array_equal(got[0], mark) and np.array_equal(got[1], mark)
    g.set_prims(p0)
    dt, _, _ = g.step_ch(dt0)
    p, dto, _, _ = og.step(p0, dt0)
    assert dt == dto
    assert np.array_equal(g.get_prims(), p)
    g.close()
