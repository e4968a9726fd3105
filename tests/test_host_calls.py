"""What the host code allocates and launches, on the CPU: it runs against a
stand-in for the HIP runtime (device_double.cpp) that counts allocations and
names launches."""
import os
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="session")
def on_double(tmp_path_factory):
    """Runs a program against the stand-in, in a process of its own: D is the
    stand-in, R the package, np numpy."""
    so = str(tmp_path_factory.mktemp("double") / "device_double.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I",
                    "/opt/rocm/include", os.path.join(ROOT, "tests", "device_double.cpp"), "-o", so],
                   check=True)

    def run(code):
        head = f"""
            import ctypes as C, numpy as np
            D = C.CDLL({so!r}, mode=C.RTLD_GLOBAL)
            D.double_live.restype = D.double_live_bytes.restype = C.c_size_t
            D.double_limit.argtypes = D.double_largest.argtypes = [C.c_size_t]
            import radiosity_amd as R
            """
        p = subprocess.run([sys.executable, "-c", textwrap.dedent(head) + textwrap.dedent(code)],
                           cwd=ROOT, capture_output=True, text=True, timeout=300)
        assert p.returncode == 0, p.stdout + p.stderr

    return run


def test_close_returns_every_allocation(on_double):
    """Plain scenes, a replaced scene, a pack, the deterministic rows, a dense
    matrix with its solve, a graph."""
    on_double("""
        def boxes(n, seed=3):
            return R.Scene.boxes(nboxes=4, room=(5.0, 3.0, 5.0), target_tris=n, nlights=2, seed=seed)
        for kw in (dict(hemicube=16, hemicubes=1), dict(hemicube=64, hemicubes=16, graph_passes=4)):
            s = R.Solver(**kw)
            s.set_deterministic(True)
            s.upload(boxes(600))
            s.upload(boxes(3000))
            s.prepare()
            s.step(9)
            s.autotune(1)
            s.dense_upload(np.zeros((s.npatch, s.npatch), np.float32))
            s.dense_apply(np.zeros((3, s.npatch), np.float32))
            s.pack_upload([boxes(300 + 200 * i, i + 1) for i in range(3)], [1, 1, 1])
            s.step(2)
            assert D.double_live() > 30
            s.close()
            assert D.double_live() == 0, (kw, D.double_live(), D.double_live_bytes())
        """)


def test_capacities_of_every_launch_shape(on_double):
    """What a pass may hold (records beyond their regions, entries, triangles to
    clip) counts a region of 768 records for each 256 triangles, shooter and,
    up to four shooters, face; four times the entries where a side of 16 was
    taken for four shooters or more."""
    on_double("""
        def caps(W, K, ntri, tile):
            s = R.Solver(hemicube=W, hemicubes=K, tile_px=tile)
            s.upload(R.Scene(np.zeros((ntri, 9)), np.zeros(ntri), np.eye(3).reshape(1, 9),
                             np.ones((1, 3)), np.ones(1), np.ones((1, 3)), np.ones((1, 3))))
            c, (_, side) = s.debug_counters(), s.debug_bins()
            s.close()
            return c, side
        seen = set()
        for W in (16, 64, 128, 256):
            for K in (1, 3, 4, 5, 12, 32, 64):
                for ntri in (1, 700, 3000, 24000, 60000, 120000):
                    for tile in (0, 32):
                        if K * ntri > 1000000:
                            continue
                        c, side = caps(W, K, ntri, tile)
                        slots = -(-ntri // 256) * K * (5 if K <= 4 else 1) * 768
                        spill = slots // 8 + 65536
                        entries = 2 * (slots + spill)
                        if not tile and K >= 4 and side == 16:
                            entries *= 4
                        seen.add((tile, K >= 4, side))
                        assert c["clip_cap"] == spill // 2, (W, K, ntri, tile)
                        assert c["spill_cap"] >= spill, (W, K, ntri, tile)
                        assert c["entry_cap"] == entries, (W, K, ntri, tile)
        assert (0, True, 16) in seen and (0, True, 32) in seen
        """)


def test_lists_in_the_memory_there_is(on_double):
    """An upload, and another tile side later, without memory for the tiles'
    lists at their full size take smaller ones; without any, the context has no
    scene.  No launch gets a missing list."""
    on_double("""
        sc = R.Scene.boxes(nboxes=8, room=(6.0, 3.0, 6.0), target_tris=6000, nlights=2, seed=3)
        tiles = []
        def note(name, args):
            if b"k_tile_raster" in name:
                tiles.append([C.cast(args[i], C.POINTER(C.c_void_p))[0] for i in (7, 8)])
        CB = C.CFUNCTYPE(None, C.c_char_p, C.POINTER(C.c_void_p))
        D.double_on_launch(cb := CB(note))

        def solver(limit):
            D.double_limit(limit)
            s = R.Solver(hemicube=64, hemicubes=40, tile_px=32)
            s.upload(sc)
            return s

        s = solver(1 << 62)
        full = D.double_live_bytes()
        s.close()
        lists = 4 * 40 * 12 * 8192  # 40 x 12 tiles, 16 x 6,000 / 12 entries and up
        assert full > lists
        # the upload, with a quarter of the lists' memory
        s = solver(full - lists * 3 // 4)
        assert D.double_live_bytes() < full - lists // 2
        s.step(3)
        s.close()
        # other tiles later, with a quarter; and with none
        s = solver(1 << 62)
        D.double_largest(lists // 4)
        s.autotune(1)
        s.step(3)
        s.close()
        D.double_largest(1 << 62)
        s = solver(1 << 62)
        D.double_largest(70000)
        for call, word in ((lambda: s.autotune(1), "out of memory"), (lambda: s.step(1), "no scene")):
            try:
                call()
                raise SystemExit("done without lists")
            except R.RadError as e:
                assert word in str(e), e
        D.double_largest(1 << 62)
        s.upload(sc)
        s.step(3)
        s.close()
        assert len(tiles) > 20 and all(p for t in tiles for p in t)
        """)


def test_autotune_times_direct_passes_with_the_limit_it_chose(on_double):
    """The stand-in's times grow with every call, so the first candidate's
    limit of 16 pixels is chosen."""
    on_double("""
        limits = []
        def note(name, args):
            if b"k_direct" in name:
                limits.append(C.cast(args[0], C.POINTER(C.c_uint32))[5])  # DirectArgs::small_px
        CB = C.CFUNCTYPE(None, C.c_char_p, C.POINTER(C.c_void_p))
        D.double_on_launch(cb := CB(note))
        s = R.Solver(hemicube=64, hemicubes=8)
        s.upload(R.Scene.boxes(nboxes=4, room=(5.0, 3.0, 5.0), target_tris=2000, nlights=2, seed=3))
        s.step(1)
        assert limits == [64]
        assert s.autotune(2)[1] == 16
        assert limits == [64] + 3 * [16], limits
        """)


def test_second_stream_where_passes_may_be_split(on_double):
    """A context has the second half's stream from 16 shooters and 8,192 tiles
    on, at whatever tile side it comes to that."""
    on_double("""
        for f in (D.double_streams, D.double_unstreamed):
            f.restype = C.c_size_t
        sc = R.Scene.boxes(nboxes=4, room=(5.0, 3.0, 5.0), target_tris=3000, nlights=2, seed=3)
        def run(streams, tune=None, **kw):
            s = R.Solver(**kw)
            s.upload(sc)
            s.step(3)
            assert D.double_streams() == streams, (kw, D.double_streams())
            if tune:
                s.autotune(1)  # tiles of 16 and 32
                s.step(3)
                assert D.double_streams() == tune, (kw, D.double_streams())
            s.close()
            assert D.double_streams() == 0
        run(1, hemicube=16, hemicubes=1)
        run(1, hemicube=128, hemicubes=64, tune=2)
        run(1, hemicube=512, hemicubes=15, tune=1)
        run(2, hemicube=256, hemicubes=64, graph_passes=2)
        assert D.double_unstreamed() == 0
        """)
