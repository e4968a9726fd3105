"""Scenes near the rasterizer's capacities: the launch shapes and tile sides
that the library takes by itself refuse none that others take."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _scene(rad, tri, eyes):
    n = len(eyes)
    frame = np.concatenate([eyes, np.tile([[0.0, 0, 1, 0, 1, 0]], (n, 1))], 1)
    one = np.ones((n, 3), np.float32)
    return rad.Scene(tri.astype(np.float32), np.sort(np.arange(len(tri)) % n), frame, 0.5 * one,
                     np.ones(n), one, 0 * one)


def test_many_triangles_to_clip(rad):
    """One shooter, 100,000 triangles (a workgroup takes all five faces of
    them), 70,000 of which cross the near plane."""
    rng = np.random.default_rng(2)
    c = np.concatenate([rng.uniform(-0.002, 0.002, (70000, 1, 2)), np.full((70000, 1, 1), 0.01)], 2)
    d = rng.uniform(-8e-4, 8e-4, (70000, 3, 3))
    d[:, 0, 2], d[:, 1, 2] = -6e-4, 6e-4
    far = rng.uniform(-4, 4, (30000, 1, 3)) + rng.uniform(-0.05, 0.05, (30000, 3, 3))
    sc = _scene(rad, np.concatenate([c + d, far]), np.zeros((1, 3)))
    print("triangles to clip", flush=True)
    s = rad.Solver(hemicube=64, hemicubes=1)
    s.upload(sc)
    ids = s.render([0])
    assert s.debug_counters()["clip"] >= 70000
    assert np.array_equal(ids, O.render_hemicube(64, sc.tri, sc.tri_patch, sc.frame[0]))


def _large(rad, n):
    """n shooters amid 3,000 large triangles, all of them seen from the middle."""
    rng = np.random.default_rng(3)
    c = rng.normal(size=(3000, 1, 3))
    c[:, :, 2] = np.abs(c[:, :, 2])
    c *= rng.uniform(3, 5, (3000, 1, 1)) / np.linalg.norm(c, axis=2, keepdims=True)
    tri = c + 2.0 * rng.uniform(-1, 1, (3000, 3, 3))
    back = (np.cross(tri[:, 2] - tri[:, 0], tri[:, 1] - tri[:, 0]) * tri.mean(1)).sum(1) > 0
    tri[back] = tri[back][:, [0, 2, 1]]
    return _scene(rad, tri, rng.uniform(-0.1, 0.1, (n, 3)))


def test_entries_of_small_tiles(rad):
    """Twelve shooters: in tiles of 32, the entries fit; in tiles of 16, which
    the library takes, they are more than that limit."""
    sc = _large(rad, 12)
    sh = np.arange(12)
    out = []
    for tile in (32, 0):
        print(f"entries, tile {tile}", flush=True)
        s = rad.Solver(hemicube=128, hemicubes=12, tile_px=tile)
        s.upload(sc)
        ids = s.render(sh)
        out.append((ids, s.debug_counters(), s.debug_bins()[1]))
        s.close()
    assert out[1][2] == 16 and out[1][1]["entries"] > out[0][1]["entry_cap"]
    assert np.array_equal(out[0][0], out[1][0])


def test_entries_of_a_whole_pass(rad):
    """24 shooters in 4,608 tiles of 16, drawn whole: more entries than each
    half of a split pass may have, and fewer than both."""
    sc = _large(rad, 24)
    print("entries of a whole pass", flush=True)
    s = rad.Solver(hemicube=128, hemicubes=24, tile_px=16)
    s.upload(sc)
    ids = s.render(np.arange(24))
    c = s.debug_counters()
    assert c["entry_cap"] < c["entries"] < 2 * c["entry_cap"]
    res = s.tex_res
    for k in (0, 23):
        assert np.array_equal(ids[k * res:(k + 1) * res],
                              O.render_hemicube(128, sc.tri, sc.tri_patch, sc.frame[k]))
