"""Shooter selection at the edges of its kernels: the reference's list rule
(chunks of 1,024 patches, one or four list entries per lane) against the
oracle's list, ties and zeros included; a pack's per-scene selection (64
keys at once, single rounds beyond) against a plain context's."""
import sys

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _points(rad, n):
    """n patches without triangles: only the selection looks at them."""
    frame = np.tile(np.eye(3, dtype=np.float32).reshape(9), (n, 1))
    z = np.zeros((n, 3))
    return rad.Scene(np.zeros((0, 9)), np.zeros(0), frame, z + 0.5, np.ones(n), z, z)


@pytest.mark.parametrize("K", [2, 10, 63, 64, 65, 200, 256])
def test_reference_list_rule(rad, K):
    rng = np.random.default_rng(K)
    for n in (1, 2, 63, 64, 65, 1023, 1024, 1025, 3000):
        s = rad.Solver(hemicube=16, hemicubes=K, mode=rad.RAD_MODE_REFERENCE,
                       select=rad.RAD_SELECT_REFERENCE)
        s.upload(_points(rad, n))
        say(f"list rule K={K} n={n}")
        for levels, first in ((2, 0), (4, 1), (40, 2), (100000, 0)):
            # few levels: long runs of equal keys; first: patch 0's, below
            # which the rule takes nothing
            u = rng.integers(0, levels, size=(n, 3)).astype(np.float32)
            u[0] = first
            s.set_state(u, np.zeros_like(u), u)
            ids, got = s.select(K)
            want, wn = O.select_reference(u, K)
            assert got == wn and np.array_equal(ids, want), (n, levels, first)
        # increasing keys: every patch enters the list
        u = np.arange(3 * n, dtype=np.float32).reshape(n, 3)
        s.set_state(u, np.zeros_like(u), u)
        ids, got = s.select(K)
        want, wn = O.select_reference(u, K)
        assert got == wn and np.array_equal(ids, want), n
        s.close()


@pytest.mark.parametrize("slots", [1, 5, 63, 64, 65, 100])
def test_pack_selection_equals_plain(rad, slots):
    """A pack of one scene shoots what a plain context with as many hemicubes
    shoots: with fixed-point form factors the states agree bit for bit."""
    sc = rad.Scene.boxes(nboxes=10, room=(6.0, 3.0, 6.0), target_tris=2500, nlights=4, seed=2)
    rng = np.random.default_rng(slots)
    # few power levels with equal areas: ties go to the lower index
    u = rng.integers(0, 6, size=(sc.npatch, 3)).astype(np.float32)
    z = np.zeros_like(u)
    say(f"pack selection of {slots} slots")
    p = rad.Solver(hemicube=16, hemicubes=slots)
    p.set_deterministic(True)
    p.pack_upload([sc], [slots])
    p.set_state(u, z, u)
    p.pack_begin(1e-9)
    p.step(3)
    done, res, passes, rem = p.pack_status()
    assert passes == 3 and rem == 1 and p.pack_shooters[0] == 3 * slots
    q = rad.Solver(hemicube=16, hemicubes=slots)
    q.set_deterministic(True)
    q.upload(sc)
    q.set_state(u, z, u)
    q.step(3)
    q.finish()
    for a, b in zip(p.state(), q.state()):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    # the residual of the last selection is the state's before that pass
    q.set_state(u, z, u)
    q.step(2)
    assert res[0] == pytest.approx(q.residual(), rel=1e-12)


@pytest.mark.parametrize("K,graph,select", [(1, 0, 0), (1, 0, 1), (1, 5, 0), (1, 5, 1), (3, 0, 0),
                                            (7, 4, 0), (24, 0, 1), (64, 0, 1), (70, 0, 1)])
def test_passes_in_a_row_equal_single_passes(rad, K, graph, select):
    """A call of several passes selects and prepares each from what the one
    before left; single-pass calls select from the stored state.  With
    fixed-point form factors the states agree bit for bit, stopped cycles
    (whose later passes shoot nobody) included."""
    sc = rad.Scene.boxes(nboxes=12, room=(7.0, 3.0, 7.0), target_tris=3000, nlights=6, seed=4)
    say(f"passes in a row K={K} graph={graph} select={select}")
    out = []
    for one in (False, True):
        s = rad.Solver(hemicube=32, hemicubes=K, graph_passes=0 if one else graph, select=select)
        s.set_deterministic(True)
        s.upload(sc)
        for _ in range(2):
            if one:
                for _ in range(11):
                    s.step(1)
            else:
                s.step(11)
        s.finish()
        out.append(s.state() + (s.shot_count(),))
        st = s.run_cycle(4, 1e9) if not one else None
        if st:
            assert st.passes == 1 and st.stopped == 1
    for a, b in zip(out[0][:2], out[1][:2]):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    assert out[0][2] == out[1][2]
