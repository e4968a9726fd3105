"""The binned setup's culls (faces by the largest coordinate, triangles seen
from behind) drop nothing that the oracle draws."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _soup(rad, ntri, scale, shift, seed):
    """Triangles of all sizes around the viewpoints, from slivers and ones of a
    thousandth of a pixel to ones around the eye; a third nearly edge-on to
    the first viewpoint, on either side."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(-4, 4, (ntri, 1, 3))
    size = np.exp(rng.uniform(np.log(1e-4), np.log(4.0), (ntri, 1, 1)))
    tri = c + size * rng.uniform(-1, 1, (ntri, 3, 3))
    tri[::7, 2] = tri[::7, 1] + 1e-3 * rng.uniform(-1, 1, (len(tri[::7]), 3))
    # edge-on: the third vertex close to the plane of the eye and the others
    t = rng.uniform(0.2, 0.8, (len(tri[::3]), 1))
    tri[::3, 2] = (t * tri[::3, 0] + (1 - t) * tri[::3, 1]) * rng.uniform(0.5, 1.5, t.shape)
    tri[::3, 2] += np.exp(rng.uniform(np.log(1e-6), np.log(1e-1), t.shape)) * rng.normal(size=(len(t), 3))
    tri = tri * scale + shift
    n = rng.normal(size=(ntri, 3))
    n /= np.linalg.norm(n, axis=1, keepdims=True)
    up = np.cross(n, rng.normal(size=(ntri, 3)))
    up /= np.linalg.norm(up, axis=1, keepdims=True)
    eye = tri.mean(1)
    eye[0] = shift
    up[::5] = rng.normal(size=(len(up[::5]), 3))  # not orthogonal: no culls
    up[0] = np.cross(n[0], [0.3, 0.5, 0.8])
    one = np.ones((ntri, 3), np.float32)
    return rad.Scene(tri.astype(np.float32), np.arange(ntri),
                     np.concatenate([eye, n, up], 1).astype(np.float32), 0.5 * one, np.ones(ntri),
                     one, 0 * one)


@pytest.mark.parametrize("scale,shift", [(1.0, 0.0), (0.01, 0.0), (100.0, 0.0), (1.0, 3000.0)])
@pytest.mark.parametrize("W,K", [(16, 2), (90, 6), (256, 6)])
def test_culls_against_the_oracle(rad, W, K, scale, shift):
    """K 2: a workgroup per face; K 6: all faces in one."""
    sc = _soup(rad, 3000, scale, shift, W)
    print(f"setup culls: W={W} K={K} scale={scale} shift={shift}", flush=True)
    s = rad.Solver(hemicube=W, hemicubes=K, tile_px=16)
    s.upload(sc)
    sh = np.arange(K, dtype=np.uint32) * 401
    ids = s.render(sh)
    res = s.tex_res
    for k in range(K):
        want = O.render_hemicube(W, sc.tri, sc.tri_patch, sc.frame[sh[k]])
        assert np.array_equal(ids[k * res:(k + 1) * res], want), k
