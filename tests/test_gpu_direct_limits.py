"""The direct rasterizer at the limits of the passes it takes, against the
binned one: item buffers and depths are the same bits.  Which of the two drew
a pass shows in its entry count, 0 without bins."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def room(rad):
    return rad.Scene.boxes(nboxes=96, room=(12.0, 3.5, 12.0), target_tris=60000, nlights=4, seed=8)


# hemicube side, shooters, the most triangles drawn directly: tiles of 16 in one
# round of workgroups, of 32 in one and in more
@pytest.mark.parametrize("W,K,most", [(128, 1, 49152), (64, 5, 28800), (256, 1, 34816),
                                      (128, 5, 28800), (128, 8, 8192), (256, 2, 8192)])
def test_at_the_limit(rad, room, W, K, most):
    # shooters on triangles that are left out see into the room as well
    sh = np.linspace(0, room.npatch - 1, K + 2).astype(np.uint32)[1:-1]
    first = (room.ntri - most) // 2
    for n in (most, most + 1):
        cut = slice(first, first + n)
        sc = rad.Scene(room.tri[cut], room.tri_patch[cut], room.frame, room.refl, room.area,
                       room.emission, room.shot0)
        print(f"direct limit: W={W} K={K} triangles={n}", flush=True)
        out = []
        for tile in (0, 32):
            s = rad.Solver(hemicube=W, hemicubes=K, tile_px=tile)
            s.upload(sc)
            out.append(s.render(sh, depth=True))
            direct = s.debug_counters()["entries"] == 0
            assert direct == (tile == 0 and n == most)
            s.close()
        (ia, za), (ib, zb) = out
        assert (ia > 0).any()
        assert np.array_equal(ia, ib) and np.array_equal(za.view(np.uint32), zb.view(np.uint32))
