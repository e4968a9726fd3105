"""Performance cases: the work a user of this library has it do, through the
Python binding's public calls, from the reference's default Cornell box to the
200,000-patch room.

Every case is a dict of plain values; "kind" picks the path:

  cycle   the drop-in's cycle (Solver.run_cycle) in the reference's own mode
  shoot   progressive shooting of one scene from its emission (Solver.run)
  pack    many small scenes in one context (Solver.pack_*)
  rows    the two-step API: item buffers, then ProcessHemicube over them
  dense   dense form factors from hemicubes, then the gather (global solve)
  gather  the gather over a matrix the program already has, many lightings
  apply   one product with that matrix

A pass starts by handing over the emission (a relighting program's call), so
every pass of a state does the same work, and ends with the results in host
memory, where these calls put them.
"""
import numpy as np
import torch

import radiosity_amd as R


def listed():
    return [
        # the reference program as it starts: Cornell quads, hemicube 16, 10
        # hemicubes per pass, its own selection and shooting rules
        dict(name="cycle_cornell772_w16_k10", kind="cycle", area=0.3127, w=16, k=10, passes=20),
        # the single-shooter drop-in on the Cornell box, 100 shots
        dict(name="plain_cornell1500_w128", kind="shoot", scene="cornell", area=0.3127, w=128, k=1,
             graph=0, passes=100, det=False),
        # the same box finely subdivided, hemicube 256
        dict(name="plain_cornell20k_w256", kind="shoot", scene="cornell", area=0.0232, w=256, k=1,
             graph=0, passes=200, det=False),
        # the single-shooter drop-in on the largest room
        dict(name="plain_room200k_w256", kind="shoot", scene="boxes", n=200000, w=256, k=1,
             graph=0, passes=60, det=False),
        # batched shooting replayed from captured graphs: a small room, a
        # middle one and the largest
        dict(name="batch_room6k_w64_k16", kind="shoot", scene="boxes", n=6000, w=64, k=16,
             graph=8, passes=64, det=False),
        dict(name="batch_room33k_w128_k64", kind="shoot", scene="boxes", n=32768, w=128, k=64,
             graph=10, passes=60, det=False),
        dict(name="batch_room200k_w256_k64", kind="shoot", scene="boxes", n=200000, w=256, k=64,
             graph=10, passes=60, det=False),
        # reproducible results (fixed-point form factors), plain launches
        dict(name="det_room20k_w128_k32", kind="shoot", scene="boxes", n=20000, w=128, k=32,
             graph=0, passes=30, det=True),
        # a service's batch of uneven rooms, each at its own hemicube side
        dict(name="pack32_w256_k64", kind="pack", scenes=32, lo=500, hi=20000, k=64, graph=8,
             passes=24),
        # form-factor rows of chosen patches for a program of its own
        dict(name="rows_room10k_w64_k24", kind="rows", n=10000, w=64, k=24),
        # the global solve: every hemicube into a dense matrix, then BF16
        # Jacobi sweeps with refinement
        dict(name="dense_room16k_w128", kind="dense", n=16384, w=128, k=64, target=1e-3),
        # relighting over a stored matrix: 64 lightings x RGB
        dict(name="gather_8k_r192", kind="gather", n=8192, r=192, target=1e-4),
    ]


def _log(rng, lo, hi):
    return int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))


def _side(rng, lo, hi):
    return 2 * _log(rng, lo / 2, hi / 2)


def draw(rng):
    kind = rng.choice(["cycle", "plain", "batch", "batch", "det", "pack", "rows", "dense",
                       "gather", "apply"])
    if kind == "cycle":
        return dict(kind="cycle", area=_log(rng, 400, 20000) / 10000.0, w=_side(rng, 8, 64),
                    k=rng.randint(2, 24), passes=rng.randint(8, 30))
    if kind == "plain":
        if rng.random() < 0.5:
            return dict(kind="shoot", scene="cornell", area=_log(rng, 230, 10000) / 10000.0,
                        w=_side(rng, 32, 256), k=1, graph=rng.choice([0, 0, 8]),
                        passes=rng.randint(40, 120), det=False)
        return dict(kind="shoot", scene="boxes", n=_log(rng, 700, 200000), w=_side(rng, 32, 256),
                    k=1, graph=rng.choice([0, 0, 8]), passes=rng.randint(20, 60), det=False)
    if kind in ("batch", "det"):
        det = kind == "det"
        return dict(kind="shoot", scene="boxes", n=_log(rng, 1500, 60000 if det else 200000),
                    w=_side(rng, 32, 256), k=_log(rng, 2, 64 if det else 100),
                    graph=0 if det else rng.choice([0, 8, 10]), passes=rng.randint(16, 40), det=det)
    if kind == "pack":
        lo = _log(rng, 500, 2000)
        return dict(kind="pack", scenes=_log(rng, 5, 48), lo=lo, hi=_log(rng, 4000, 20000),
                    k=_log(rng, 24, 160), graph=rng.choice([0, 8]), passes=rng.randint(8, 24))
    if kind == "rows":
        return dict(kind="rows", n=_log(rng, 1500, 40000), w=_side(rng, 16, 128),
                    k=_log(rng, 1, 48))
    if kind == "dense":
        return dict(kind="dense", n=_log(rng, 1500, 18000), w=_side(rng, 32, 128),
                    k=_log(rng, 16, 64), target=1e-3)
    return dict(kind=kind, n=_log(rng, 700, 8192), r=_log(rng, 1, 192),
                **(dict(target=1e-4) if kind == "gather" else dict(split=rng.random() < 0.5)))


# ------------------------------------------------------------------ inputs

def _paint(sc, seed):
    """The scene with this seed's reflectances and light strengths, turned by a
    quarter turn about the vertical and scaled as this seed says."""
    rng = np.random.default_rng(seed)
    turn = np.linalg.matrix_power(np.array([[0, 0, 1], [0, 1, 0], [-1, 0, 0]]),
                                  int(rng.integers(4))).astype(np.float32)
    scale = np.float32(rng.uniform(0.8, 1.25))
    frame = sc.frame.reshape(-1, 3, 3) @ turn.T
    frame[:, 0] *= scale
    lit = sc.emission.max(1) > 0
    emission = sc.emission.copy()
    emission[lit] = rng.uniform(5.0, 20.0, (int(lit.sum()), 3))
    return R.Scene(sc.tri.reshape(-1, 3) @ turn.T * scale, sc.tri_patch, frame,
                   rng.uniform(0.1, 0.8, sc.refl.shape), sc.area * scale * scale, emission,
                   sc.shot0)


def _boxes(n, seed):
    """A furnished room of about n triangle patches (the 200,000-patch room is
    20 x 5 x 20 with 400 boxes), lit by 16 ceiling triangles."""
    side = 5.0 + 15.0 * (n / 200000.0) ** 0.5
    return _paint(R.Scene.boxes(nboxes=max(2, n // 500),
                                room=(side, 3.0 + 2.0 * n / 200000.0, side), target_tris=n,
                                nlights=16, seed=3), seed)


def _cornell_quads(area, seed):
    """The reference's Cornell box with the wall colours and the light's
    strength of this seed."""
    quads, color, emission, shot0 = R.cornell_faces()
    rng = np.random.default_rng(seed)
    color = np.where(color > 0, rng.uniform(0.2, 0.9, color.shape), color).astype(np.float32)
    emission = (emission * rng.uniform(0.5, 2.0, (1, 3))).astype(np.float32)
    return R.Scene.faces(quads, area, R.RAD_FACES_QUADS, color, emission, shot0)


def _matrix(n, seed):
    """Form factors of a closed scene of n patches: every row sums to 0.98,
    most of it in a few near or large patches."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    m = torch.exp(2.0 * torch.randn(n, n, device="cuda", generator=g))
    m.fill_diagonal_(0.0)
    return m * (0.98 / m.sum(1, keepdim=True))


def _gather_inputs(case, seed):
    """(matrix on the GPU, reflectances n x 3, columns r x n)."""
    rng = np.random.default_rng(seed)
    n, r = case["n"], case["r"]
    rho = rng.uniform(0.1, 0.8, (n, 3)).astype(np.float32)
    if case["kind"] == "apply":
        x = rng.uniform(0.0, 2.0, (r, n))
    else:
        # lightings: a few of 32 candidate lights on in each
        x = np.zeros((r, n))
        lights = rng.choice(n, 32, replace=False)
        for c in range(r):
            on = rng.choice(lights, 6, replace=False)
            x[c, on] = rng.uniform(5.0, 20.0, 6)
    return _matrix(n, seed), rho, x.astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "cycle":
        s = R.Solver(hemicube=case["w"], hemicubes=case["k"], mode=R.RAD_MODE_REFERENCE,
                     select=R.RAD_SELECT_REFERENCE)
        sc = _cornell_quads(case["area"], seed)
        s.upload(sc)
        return dict(case=case, solver=s, scene=sc)
    if kind == "shoot":
        if case["scene"] == "cornell":
            sc = _paint(R.Scene.cornell(case["area"], triangle_patches=True, physical=True, seed=1),
                        seed)
        else:
            sc = _boxes(case["n"], seed)
        s = R.Solver(hemicube=case["w"], hemicubes=case["k"], graph_passes=case["graph"])
        if case["det"]:
            s.set_deterministic(True)
        s.upload(sc)
        s.prepare()
        return dict(case=case, solver=s, scene=sc)
    if kind == "pack":
        sizes = np.exp(np.random.default_rng(5).uniform(np.log(case["lo"]), np.log(case["hi"]),
                                                        case["scenes"]))
        scenes, sides, slots = [], [], []
        for i, n in enumerate(sizes.astype(int)):
            edge = 5.0 + 7.0 * n / 20000.0
            sc = R.Scene.boxes(nboxes=max(2, int(n) // 400), room=(edge, 3.0 + n / 10000.0, edge),
                               target_tris=int(n), nlights=4, seed=1000 + i)
            scenes.append(_paint(sc, 1000 * seed + i))
            np_ = scenes[-1].npatch
            sides.append(64 if np_ < 1500 else (128 if np_ < 6000 else 256))
            slots.append(int(min(16, max(1, -(-np_ // 2000)))))
        s = R.Solver(hemicube=256, hemicubes=case["k"], graph_passes=case["graph"])
        s.pack_upload(scenes, slots)
        s.pack_hemicubes(sides)
        s.pack_begin(1e-3)
        s.prepare()
        return dict(case=case, solver=s,
                    emission=np.concatenate([sc.emission for sc in scenes]),
                    shot0=np.concatenate([sc.shot0 for sc in scenes]))
    if kind in ("rows", "dense"):
        sc = _boxes(case["n"], seed)
        s = R.Solver(hemicube=case["w"], hemicubes=case["k"])
        s.upload(sc)
        rng = np.random.default_rng(seed)
        return dict(case=case, solver=s,
                    shooters=rng.choice(sc.npatch, case["k"], replace=False).astype(np.uint32))
    m, rho, x = _gather_inputs(case, seed)
    n = case["n"]
    # the matrix is the program's own; its scene carries no triangles
    sc = R.Scene(np.zeros((0, 9)), np.zeros(0), np.tile(np.eye(3, dtype=np.float32).reshape(9),
                                                        (n, 1)),
                 rho, np.ones(n), np.zeros((n, 3)), np.zeros((n, 3)))
    s = R.Solver(hemicube=16, hemicubes=1)
    s.upload(sc)
    s.dense_upload(m.cpu().numpy())
    return dict(case=case, solver=s, x=x)


# -------------------------------------------------------------------- runs

def run(state):
    case, s = state["case"], state["solver"]
    kind = case["kind"]
    if kind == "cycle":
        sc = state["scene"]
        s.set_state(sc.emission, sc.shot0, sc.emission)
        st = s.run_cycle(case["passes"])
        unshot, shot = s.state()
        return dict(unshot=unshot, shot=shot, passes=int(st.passes), shooters=int(st.shooters))
    if kind == "shoot":
        sc = state["scene"]
        s.set_state(sc.emission, sc.shot0, sc.emission)
        st = s.run(case["passes"], 0.0)
        unshot, shot = s.state()
        return dict(unshot=unshot, shot=shot, residual=float(st.residual),
                    shooters=int(st.shooters))
    if kind == "pack":
        s.set_state(state["emission"], state["shot0"], state["emission"])
        s.step(case["passes"])
        done, residual, _, _ = s.pack_status()
        unshot, shot = s.state()
        return dict(unshot=unshot, shot=shot, residual=residual)
    if kind == "rows":
        ids = s.render(state["shooters"])
        hits, ff = s.process(case["k"])
        return dict(ids=ids, hits=hits, ff=ff)
    if kind == "dense":
        s.dense_build()
        b, st = s.gather(target=case["target"])
        return dict(b=b)
    if kind == "gather":
        b, st = s.gather(state["x"], target=case["target"])
        return dict(b=b)
    return dict(y=s.dense_apply(state["x"], split=case["split"]))


def exact(case, seed):
    """64-bit results of the matrix paths.  The hemicube paths have none: what
    a texel sees is decided on vertices snapped to 1/256 pixel and on float
    depths, choices that 64-bit arithmetic would make differently."""
    if case["kind"] not in ("gather", "apply"):
        return None
    m, rho, x = _gather_inputs(case, seed)
    m, x = m.double(), torch.from_numpy(x).cuda().double()
    if case["kind"] == "apply":
        return dict(y=(x @ m.T).cpu())
    # column r solves (I - diag(rho[:, r % 3]) M) b = x_r; the solver stops at
    # the case's target, which bounds how near it comes
    b = torch.empty_like(x)
    for ch in range(3):
        a = torch.eye(case["n"], dtype=torch.float64, device="cuda")
        a -= torch.from_numpy(rho[:, ch]).cuda().double()[:, None] * m
        if x[ch::3].numel():
            b[ch::3] = torch.linalg.solve(a, x[ch::3].T).T
    return dict(b=b.cpu())


def work(case):
    """Scene and state once in and the results once out; a transform per
    (triangle, shooter) and a depth test and a weight per texel of every
    shooting pass."""
    kind, k = case["kind"], case.get("k", 1)
    if kind in ("gather", "apply"):
        n, r = case["n"], case["r"]
        halves = 2 if case.get("split", True) else 1
        return dict(bytes=2.0 * halves * n * n + 8.0 * r * n, flops=2.0 * r * n * n)
    if kind == "pack":
        n = case["scenes"] * 1.4 * (case["lo"] * case["hi"]) ** 0.5
        tris, texels = case["k"] * n / case["scenes"], case["k"] * 3.0 * 128 * 128
    else:
        n = case["n"] if "n" in case else (8.0 if kind == "shoot" else 4.0) * 60.0 / case["area"]
        tris, texels = k * n, k * 3.0 * case["w"] ** 2
    if kind == "rows":
        return dict(bytes=40.0 * n + 4.0 * texels + 8.0 * k * n, flops=40.0 * tris + 8.0 * texels)
    if kind == "dense":
        texels = n * 3.0 * case["w"] ** 2
        return dict(bytes=4.0 * n * n, flops=40.0 * n * n + 8.0 * texels + 6.0 * n * n)
    passes = case["passes"]
    return dict(bytes=124.0 * n, flops=passes * (40.0 * tris + 8.0 * texels))
