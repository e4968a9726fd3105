"""The direct rasterizer (small passes of contexts without a chosen tile
side) against the binned one (tile_px given): the item buffers and depths
are the same bits, and the rows and states agree to float rounding."""
import sys

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _soup(rad, ntri, seed, scale=1.0, shift=0.0):
    """ntri random triangles around the origin (slivers, tiny ones and some
    through the viewpoints among them), one patch each."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(-4, 4, (ntri, 1, 3))
    size = np.exp(rng.uniform(np.log(0.01), np.log(3.0), (ntri, 1, 1)))
    tri = c + size * rng.uniform(-1, 1, (ntri, 3, 3))
    tri[::7, 2] = tri[::7, 1] + 1e-3 * rng.uniform(-1, 1, (len(tri[::7]), 3))
    tri = (tri * scale + shift).astype(np.float32)
    n = rng.normal(size=(ntri, 3))
    n /= np.linalg.norm(n, axis=1, keepdims=True)
    up = np.cross(n, rng.normal(size=(ntri, 3)))
    up /= np.linalg.norm(up, axis=1, keepdims=True)
    up[::5] = rng.normal(size=(len(up[::5]), 3))  # not orthogonal: no culls
    frame = np.concatenate([tri.mean(1), n, up], 1)
    one = np.ones((ntri, 3), np.float32)
    return rad.Scene(tri, np.arange(ntri), frame, 0.5 * one, np.ones(ntri), one, 0 * one)


def _pair(rad, sc, W, K, tile=16, **kw):
    out = []
    for t in (0, tile):
        s = rad.Solver(hemicube=W, hemicubes=K, tile_px=t, **kw)
        s.upload(sc)
        out.append(s)
    return out


@pytest.mark.parametrize("W", [2, 6, 16, 30, 34, 64, 90, 130, 256])
def test_item_buffers_equal_binned(rad, W):
    """Hemicube sides that do and do not divide into tiles, triangle counts
    around the runs of 16 and 64 and the two-level cull."""
    for ntri in (1, 15, 16, 17, 63, 64, 65, 1000, 3071, 3073):
        sc = _soup(rad, ntri, W + ntri)
        k = min(ntri, 3)
        say(f"direct W={W} triangles={ntri}")
        a, b = _pair(rad, sc, W, k)
        sh = np.linspace(0, ntri - 1, k).astype(np.uint32)
        ia, za = a.render(sh, depth=True)
        ib, zb = b.render(sh, depth=True)
        assert np.array_equal(ia, ib) and np.array_equal(za.view(np.uint32), zb.view(np.uint32))
        a.close()
        b.close()


@pytest.mark.parametrize("scale,shift", [(0.01, 0.0), (100.0, 0.0), (1.0, 3000.0), (20.0, -500.0)])
def test_item_buffers_equal_binned_far_and_small(rad, scale, shift):
    """Scenes at other scales and far from the origin, where the culls'
    margins carry the rounding of the clip transform."""
    sc = _soup(rad, 4000, 11, scale, shift)
    a, b = _pair(rad, sc, 128, 4)
    sh = np.arange(4, dtype=np.uint32) * 997
    assert np.array_equal(a.render(sh), b.render(sh))


def test_box_room_at_the_limit(rad):
    """A furnished room just below the triangle limit (meshed walls: the runs
    share planes, so the plane and back-face culls act) and just above."""
    for n in (48000, 60000):
        sc = rad.Scene.boxes(nboxes=96, room=(12.0, 3.5, 12.0), target_tris=n, nlights=4, seed=8)
        say(f"direct limit: {sc.ntri} triangles")
        a, b = _pair(rad, sc, 128, 8, 32)
        sh = np.linspace(0, sc.npatch - 1, 8).astype(np.uint32)
        ia = a.render(sh)
        assert np.array_equal(ia, b.render(sh))
        res = a.tex_res
        want = O.render_hemicube(128, sc.tri, sc.tri_patch, sc.frame[sh[3]])
        assert np.array_equal(ia[3 * res:4 * res], want)


@pytest.mark.parametrize("det", [False, True])
def test_states_match_binned(rad, det):
    sc = rad.Scene.boxes(nboxes=20, room=(8.0, 3.0, 8.0), target_tris=5000, nlights=4, seed=3)
    for K, graph in ((1, 0), (5, 0), (16, 4)):
        out = []
        for s in _pair(rad, sc, 50, K, 16, graph_passes=graph):
            s.set_deterministic(det)
            s.set_state(sc.emission, sc.shot0, sc.emission)
            s.step(12)
            s.finish()
            out.append(s.state())
        for x, y in zip(*out):
            # F entries of a few hundred texels summed in another grouping
            assert np.abs(x - y).max() <= 1e-5 * np.abs(y).max()


def test_pack_matches_binned(rad):
    scenes = [rad.Scene.boxes(nboxes=3 + i, room=(5.0, 3.0, 5.0), target_tris=700 + 900 * i,
                              nlights=3, seed=20 + i) for i in range(3)]
    out = []
    for t in (0, 16):
        s = rad.Solver(hemicube=64, hemicubes=6, tile_px=t)
        s.pack_upload(scenes, [1, 2, 3])
        s.pack_hemicubes([16, 34, 64])
        s.pack_begin(1e-9)
        s.step(6)
        s.pack_status()
        out.append(s.state())
    for x, y in zip(*out):
        assert np.abs(x - y).max() <= 1e-5 * np.abs(y).max()


def test_debug_bins_after_a_direct_pass(rad):
    """The bin counts are those of the binned rasterizer."""
    sc = rad.Scene.boxes(nboxes=20, room=(8.0, 3.0, 8.0), target_tris=5000, nlights=4, seed=3)
    s = rad.Solver(hemicube=64, hemicubes=4)
    s.upload(sc)
    sh = [5, 1000, 2000, 4000]
    s.render(sh)
    bins, tile = s.debug_bins()
    b = rad.Solver(hemicube=64, hemicubes=4, tile_px=tile)
    b.upload(sc)
    b.render(sh)
    assert np.array_equal(bins, b.debug_bins()[0])
