"""hg_autotune leaves alone what the step does not read: the block size of the
separate inversion kernel where update and inversion are one kernel."""
import pytest

pytestmark = pytest.mark.gpu


def test_autotune_does_not_time_unread_shapes():
    from harm_finalwham_amd import harmgpu as h
    print("case autotune axes", flush=True)
    g = h.Grid(24, 16, 1, nb=6)
    g.build_mks_geometry()
    g.set_dt(g.init_torus())
    for bs in (64, 128, 256):
        t = g.tune()
        t.bs_invert = bs
        g.set_tune(t)
        for _ in range(3):
            assert g.autotune(1).bs_invert == bs
    g.close()
