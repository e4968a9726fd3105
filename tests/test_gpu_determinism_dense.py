"""Deterministic F rows where many screen tiles are full: more than one bin in
16 holds the records from which the float path draws a bin as quadrants."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_full_tiles_identical_run_to_run(rad):
    """64 shooters over a 100,000-triangle room at hemicube 128, 3,072 tiles of
    32: two runs give the same bits."""
    sc = rad.Scene.boxes(nboxes=200, room=(14.0, 4.0, 14.0), target_tris=100000, nlights=16, seed=3)
    runs = []
    for rep in range(2):
        print(f"deterministic, full tiles: run {rep}", flush=True)
        s = rad.Solver(hemicube=128, hemicubes=64, tile_px=32)
        s.set_deterministic(True)
        s.upload(sc)
        s.step(6)
        s.finish()
        bins, _ = s.debug_bins()
        runs.append(s.state())
        s.close()
    # the case the quadrants' rule is about
    assert 512 < bins.size <= 4096 and (bins >= 1536).sum() > bins.size // 16
    for a, b in zip(*runs):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
