"""The setup's cull of triangles seen from behind drops the same triangles
whether a workgroup looks at one face or at all five."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

# Triangles just behind their drawn side, each on two or more faces of a shooter
# at the origin looking along +z (up +y) and with a vertex at the near plane: on
# some face the clipped polygon has a counter-clockwise part of some pixels
# (found by a search over 947 million triangles near the cull's threshold).
# Nine coordinates each, hexadecimal.
TRIANGLES = """
    1.a1aeecp-5 1.d83594p-5 1.a87ceap-6 1.e42f9ap-5 1.4799dp-7 1.143a4cp-7 1.319144p-4 1.c0abe2p-5 1.de960ep-6
    1.55e892p-5 1.0fa8fp-3 1.06fb3ep-3 1.1085e6p-4 1.614a0ep-3 1.4c11c4p-2 1.b0c2ep-8 1.47982ap-7 1.57ff18p-2
    1.4a01p-6 1.32ed74p-5 1.027c46p-5 1.a648dp-6 1.cedc4p-6 1.a20f82p-5 1.7bcc4ep-6 1.47a052p-7 1.d8f12cp-5
    -1.52f708p-6 -1.85fab6p-5 1.3ad5acp-5 -1.45a47ap-5 -1.22bd08p-4 1.af0a78p-4 -1.2411f8p-7 -1.47a968p-7 1.4dcc08p-4
    -1.b69ec4p-6 -1.47abfcp-7 1.1ceddap-5 -1.2a0c74p-5 -1.912712p-6 1.656e3cp-5 -1.200d68p-5 -1.2a398p-5 1.21f146p-5
    1.3b93c4p-9 -1.66ce12p-5 1.167d4ap-5 -1.0dcebep-9 -1.ca4978p-5 1.141f32p-4 -1.dc184cp-8 -1.47a5cep-7 1.066862p-4
    -1.4134c2p-4 1.4ec386p-6 1.2f8d72p-4 -1.47a086p-7 1.7fe714p-6 1.2547a8p-4 -1.6d0c0cp-4 1.7932aap-6 1.b0313ep-4
    -1.dcd06ep-5 -1.867d38p-5 1.b66b14p-5 -1.47a8cap-7 -1.89abd2p-4 1.a9a0d2p-4 -1.e21deap-5 -1.ab0344p-4 1.b3d84ep-4
    -1.ec6aeap-5 1.b98486p-6 1.57670ep-5 -1.47a3c2p-7 1.1657ccp-6 1.0ed698p-4 -1.0626f2p-4 1.eaa0f6p-6 1.17723ap-4
    1.c7b3e8p-5 -1.826612p-6 1.b7a76p-5 1.ccbcb8p-5 -1.0bcf0cp-4 1.939206p-4 1.47ad24p-7 -1.e0e022p-5 1.2557dp-4
    1.915b6cp-5 1.242ddap-7 1.5320c4p-5 1.5dcc28p-5 1.1f439ep-5 1.55e9aep-4 1.478bdap-7 1.e8e302p-6 1.ba59bcp-5
    1.47aaaep-7 -1.4c27dep-5 1.7a193p-9 1.15b0ccp-5 -1.032e6cp-4 -1.6247c6p-8 1.6a71aap-5 -1.580e52p-5 -1.2dea2ap-6
    1.dcc2f4p-6 1.35fa1ep-5 1.429e2ap-5 1.c2cc6cp-6 1.07532p-4 1.15bcf8p-5 1.d1f916p-7 1.25e356p-4 1.479604p-7
    1.a995a8p+0 1.76497ep-3 1.47a406p-7 1.a9cf9ep+0 1.6b9e5cp-2 1.e023ep-1 1.67d1d6p-1 1.65369ep-2 1.1884e8p+0
    1.0683e2p-3 -1.6402cp-7 1.47a87p-7 1.0cab32p-3 -1.31d97ep-6 1.d48ba4p-4 1.cc99e2p-5 -1.56aeaep-8 1.eaefecp-5
"""


def test_faces_apart_and_together(rad):
    tri = np.array([[float.fromhex(x) for x in t.split()]
                    for t in TRIANGLES.strip().splitlines()], np.float32)
    n = len(tri)
    frame = np.tile(np.array([0, 0, 0, 0, 0, 1, 0, 1, 0], np.float32), (n, 1))
    one = np.ones((n, 3), np.float32)
    sc = rad.Scene(tri, np.arange(n), frame, 0.5 * one, np.ones(n), one, 0 * one)
    out = []
    for k in (1, 8):  # one face a workgroup; all five
        print(f"cull, {k} shooters", flush=True)
        s = rad.Solver(hemicube=256, hemicubes=k, tile_px=32)
        s.upload(sc)
        ids = s.render([0])
        bins, _ = s.debug_bins()
        out.append((ids, bins[0]))
        s.close()
    assert out[1][1].sum() >= n
    assert np.array_equal(out[0][1], out[1][1])
    want = O.render_hemicube(256, sc.tri, sc.tri_patch, sc.frame[0])
    for ids, _ in out:
        assert np.array_equal(ids, want)
