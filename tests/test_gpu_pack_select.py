"""The pack selection's bound from its wavefronts' first maxima: quotas on both
sides of the 16 wavefronts, and scenes where fewer of them than the quota hold
any power at all."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots", [1, 2, 15, 16, 17])
@pytest.mark.parametrize("powered", [3, 40, 600, 0])
def test_bounded_selection_equals_plain(rad, slots, powered):
    """Powers in `powered` consecutive patches (0: in all), in few levels, so
    that most keys differ by their index only."""
    sc = rad.Scene.boxes(nboxes=10, room=(6.0, 3.0, 6.0), target_tris=6000, nlights=4, seed=2)
    rng = np.random.default_rng(100 * slots + powered)
    u = rng.integers(1, 4, size=(sc.npatch, 3)).astype(np.float32)
    if powered:
        at = int(rng.integers(0, sc.npatch - powered))
        u[:at] = 0
        u[at + powered:] = 0
    z = np.zeros_like(u)
    out = []
    for pack in (True, False):
        s = rad.Solver(hemicube=16, hemicubes=slots)
        s.set_deterministic(True)
        if pack:
            s.pack_upload([sc], [slots])
        else:
            s.upload(sc)
        s.set_state(u, z, u)
        if pack:
            s.pack_begin(1e-9)
        s.step(2)
        if pack:
            s.pack_status()
        else:
            s.finish()
        out.append(s.state())
        s.close()
    for a, b in zip(*out):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
