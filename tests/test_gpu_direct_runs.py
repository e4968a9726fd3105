"""The direct rasterizer's culls of whole runs of triangles, where the normals
of a run differ: a fold whose first triangles are seen from behind and whose
others are seen."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _fold(n, back, front):
    """A strip of n triangles across the view of a shooter at the origin (looking
    along +z, up +y): the first half slopes `back` degrees away from it, the
    others `front` degrees towards it."""
    x = np.linspace(-2.0, 2.0, n // 2 + 1)
    tri = []
    for i in range(n // 2):
        s = np.tan(np.radians(-back if i < n // 4 else front))
        a, b, c, d = [(u, s * (z - 4.5), z) for u, z in
                      ((x[i], 4.1), (x[i + 1], 4.1), (x[i + 1], 4.9), (x[i], 4.9))]
        tri += [(a, b, c), (a, c, d)]
    return np.array(tri)


@pytest.mark.parametrize("n,pad", [(16, 0), (64, 3200)])
@pytest.mark.parametrize("back,front", [(2.5, 3.0), (1.2, 4.2), (0.02, 0.01), (3.0, -3.0)])
def test_folded_run(rad, n, pad, back, front):
    """A group of 16 alone; a cluster of 64 among triangles behind the shooter,
    enough of them for the clusters to be tested before their groups.  The
    last fold is a plane."""
    rng = np.random.default_rng(4)
    behind = rng.uniform(-1, 1, (pad, 3, 3)) - [0.0, 0.0, 5.0]
    tri = np.concatenate([_fold(n, back, front), behind]).astype(np.float32)
    n = len(tri)
    frame = np.tile(np.array([0, 0, 0, 0, 0, 1, 0, 1, 0], np.float32), (n, 1))
    one = np.ones((n, 3), np.float32)
    sc = rad.Scene(tri, np.arange(n), frame, 0.5 * one, np.ones(n), one, 0 * one)
    print(f"folded run: {n} triangles, {back} and {front} degrees", flush=True)
    s = rad.Solver(hemicube=256, hemicubes=1)
    s.upload(sc)
    ids = s.render([0])
    assert s.debug_counters()["entries"] == 0  # drawn without bins
    want = O.render_hemicube(256, sc.tri, sc.tri_patch, sc.frame[0])
    assert ((want > 0).sum() > 0) == (front > 1.0)
    assert np.array_equal(ids, want)
