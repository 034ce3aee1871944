"""Performance cases: the work a program has this library do, through its
public Python entry points, with inputs made from a seed.

listed()            the named cases
draw(rng)           one more case of the same ranges
prepare(case, seed) inputs and handles a program has in hand before the call
run(state)          one pass, returning its outputs whole
work(case)          bytes and flops a pass cannot do without
exact(case, seed)   run's outputs in 64 bits from plain numpy / torch

Sizes and settings are those of the repository's scenes, tests and
benchmark: particles of r = 0.01 (coarse sets of the upsamplers 0.02) at the
scenes' density, cells of 0.0404, 3 stabilisation and 5 or 10 solver sweeps,
8 fine particles per coarse one, Adam batches of a few hundred to a few
thousand pairs.
"""
import math

import numpy as np
import torch

L = np.float32(0.0404)
DENSITY = np.float32(238732.4146)  # m = 1 <=> r = 0.01
R_COARSE = 0.02
UP_DT = 0.002


# ---- the cases ----------------------------------------------------------------
def listed():
    return [
        # the smallest scene anyone steps (the smoke test's size): launches
        # and latency decide
        _step("step_2k", 12, 12, 12, solver=5, mu=0.0, steps=10),
        # the plain box's default size, replayed from a captured step
        _step("step_graph_33k", 32, 32, 32, solver=10, mu=0.5, steps=10, graph=True),
        # about the reference scenes' 100,000 particles, a ragged block
        _step("step_111k", 61, 37, 49, solver=5, mu=0.0, steps=4),
        # the headline workload: 1M particles, friction, 3 + 10 sweeps
        _step("step_1m", 100, 100, 100, solver=10, mu=0.5, steps=2),
        # a parameter sweep: many scenes of uneven size in one set, captured,
        # lists refreshed inside the step
        _scenes("scenes_16", 16, 900_000, steps=2),
        # merge / split every step on a bed that is coarse inside and fine at
        # its surface
        _adaptive("adaptive_140k", 100, 90, steps=2),
        # a frame of the plain upsampler: fine sort and advection pass
        _fine("fine_2m", 63, 63, 63),
        # the learned upsampler on a small set and at the size it is for
        _learned("learned_27k", 30, 30, 30),
        _learned("learned_1m", 100, 100, 100),
        # training data: cell sort, features and fine-run targets of a
        # coarse run and its fine twin
        _pairs("pairs_59k", 41, 35, 41),
        # training: minibatches at the default batch and a large one, with
        # the validation forward
        _train("train_512", 512, steps=4, rows=2048),
        _train("train_8k", 8192, steps=1, rows=8192),
    ]


def _step(name, nx, ny, nz, solver, mu, steps, graph=False):
    return {"name": name, "kind": "step", "nx": nx, "ny": ny, "nz": nz, "solver": solver,
            "mu": mu, "steps": steps, "graph": graph}


def _scenes(name, count, total, steps):
    return {"name": name, "kind": "scenes", "count": count, "total": total, "steps": steps}


def _adaptive(name, nx, nz, steps):
    return {"name": name, "kind": "adaptive", "nx": nx, "nz": nz, "steps": steps}


def _fine(name, nx, ny, nz):
    return {"name": name, "kind": "fine", "nx": nx, "ny": ny, "nz": nz}


def _learned(name, nx, ny, nz):
    return {"name": name, "kind": "learned", "nx": nx, "ny": ny, "nz": nz}


def _pairs(name, nx, ny, nz):
    return {"name": name, "kind": "pairs", "nx": nx, "ny": ny, "nz": nz}


def _train(name, batch, steps, rows):
    return {"name": name, "kind": "train", "batch": batch, "steps": steps, "rows": rows}


def draw(rng):
    def log_int(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    def block(lo, hi):
        """Three ragged lattice sides with a product in about [lo, hi]."""
        side = log_int(lo, hi) ** (1.0 / 3.0)
        nx = max(3, int(round(side * rng.uniform(0.75, 1.3))))
        nz = max(3, int(round(side * rng.uniform(0.75, 1.3))))
        ny = max(3, int(min(side ** 3, hi) / (nx * nz)))
        return nx, ny, nz

    kind = rng.choice(["step", "step", "scenes", "adaptive", "fine", "learned", "pairs", "train"])
    if kind == "step":
        nx, ny, nz = block(500, 900_000)
        n = nx * ny * nz
        c = _step("", nx, ny, nz, solver=rng.choice([5, 10]), mu=rng.choice([0.0, 0.3, 0.5]),
                  steps=10 if n < 50_000 else (4 if n < 200_000 else 2),
                  graph=rng.random() < 0.4)
    elif kind == "scenes":
        c = _scenes("", rng.randint(2, 16), log_int(20_000, 850_000), steps=2)
    elif kind == "adaptive":
        c = _adaptive("", rng.randint(14, 100), rng.randint(14, 90), steps=2)
    elif kind == "fine":
        c = _fine("", *block(1_000, 240_000))
    elif kind == "learned":
        c = _learned("", *block(1_000, 900_000))
    elif kind == "pairs":
        c = _pairs("", *block(1_000, 58_000))
    else:
        b = rng.choice([log_int(64, 1024), log_int(1024, 8192)])
        c = _train("", b, steps=4 if b <= 1024 else 1, rows=log_int(256, 8192))
    del c["name"]
    return c


# ---- inputs -------------------------------------------------------------------
def _cells(space):
    return tuple(int(math.ceil(float(np.float32(s) / L))) for s in space)


def _shell(space):
    """Wall particles of a closed box: two per cell and axis on its faces."""
    m = [2 * c for c in _cells(space)]
    ix, iy, iz = np.meshgrid(*[np.arange(k) for k in m], indexing="ij")
    on = ((ix == 0) | (ix == m[0] - 1) | (iy == 0) | (iy == m[1] - 1) | (iz == 0)
          | (iz == m[2] - 1))
    idx = np.stack([ix[on], iy[on], iz[on]], 1).astype(np.float64)
    s = np.asarray(space, np.float64)
    return (0.005 * s + 0.99 * s * idx / (np.asarray(m, np.float64) - 1)).astype(np.float32)


def _cell_id(pos, cells):
    q = np.floor(pos / L)
    c = np.asarray(cells, np.float32)
    ok = ((q >= 0) & (q < c)).all(axis=1)
    k = np.where(ok[:, None], q, 0).astype(np.int64)
    cid = (k[:, 0] * cells[1] + k[:, 1]) * cells[2] + k[:, 2]
    return np.where(ok, cid, cells[0] * cells[1] * cells[2])


def _lattice(nx, ny, nz, spacing, origin, jitter, rng):
    ix, iy, iz = np.meshgrid(np.arange(nx), np.arange(ny), np.arange(nz), indexing="ij")
    p = np.stack([ix.ravel(), iy.ravel(), iz.ravel()], 1).astype(np.float32) * np.float32(spacing)
    p += np.asarray(origin, np.float32)
    return p + (rng.random(p.shape, dtype=np.float32) * 2 - 1) * np.float32(jitter)


def _pile_velocity(pos, rng):
    """Particles of a pile that is still compacting: everything creeps and
    jostles, the upper part falls faster."""
    v = rng.standard_normal(pos.shape, dtype=np.float32) * np.float32(0.1)
    h = (pos[:, 1] - pos[:, 1].min()) / max(float(np.ptp(pos[:, 1])), 1e-6)
    v[:, 1] -= np.float32(0.1) + np.float32(0.5) * h
    return v


def _block_scene(nx, ny, nz, r, rng):
    """A block of nx * ny * nz particles of radius r resting on the floor of a
    closed box, slightly overlapping, in the cell order of the step before."""
    s = 1.97 * r
    space = tuple(float(np.float32(max(1.2 * s * k, s * (k - 1) + 0.25))) for k in (nx, ny, nz))
    x0 = [0.5 * (space[a] - s * (k - 1)) for a, k in ((0, nx), (2, nz))]
    pos = _lattice(nx, ny, nz, s, (x0[0], 0.005 * space[1] + 0.01 + r, x0[1]), 0.1 * r, rng)
    vel = _pile_velocity(pos, rng)
    return _scene(pos, vel, np.full(pos.shape[0], (r / 0.01) ** 3, np.float32), space, r)


def _scene(pos, vel, mass, space, r, dt=0.002):
    from granular_gpu_amd import scenes
    cells = _cells(space)
    order = np.argsort(_cell_id(pos - np.float32(dt) * vel, cells), kind="stable")
    pos, vel, mass = (np.ascontiguousarray(a[order]) for a in (pos, vel, mass))
    return scenes.Scene(name="block", pos=pos, vel=vel, mass=mass, boundary=_shell(space),
                        space=space, cell_length=L, cells=cells, dt=np.float32(dt),
                        gravity=(0.0, -9.8, 0.0), density=DENSITY, radius=r)


def _scene_sides(case):
    """Lattice sides of a batch (the case's own, whatever the inputs' seed):
    particle counts log-uniform over a factor of 64, scaled so that they add
    up to about the case's total."""
    shape = np.random.default_rng([case["count"], case["total"]])
    u = np.exp(shape.random(case["count"]) * math.log(64.0))
    return [max(6, int(round((case["total"] * w / u.sum()) ** (1.0 / 3.0)))) for w in u]


def _bed(nx, nz, rng):
    """A bed as merging and splitting leave it: particles of 2r deep inside,
    r above them, r / 2 in the two surface layers."""
    sx, sz = 0.02 * nx, 0.02 * nz
    space = tuple(float(np.float32(v)) for v in (sx + 0.3, 1.0, sz + 0.3))
    parts, y = [], 0.005 * space[1] + 0.01
    for spacing, layers, m in ((0.04, 6, 8.0), (0.02, 6, 1.0), (0.01, 2, 0.125)):
        kx, kz = int(sx / spacing), int(sz / spacing)
        p = _lattice(kx, layers, kz, 0.99 * spacing, (0.15, y + 0.5 * spacing, 0.15),
                     0.04 * spacing, rng)
        parts.append((p, np.full(p.shape[0], m, np.float32)))
        y += spacing * layers
    pos = np.concatenate([p for p, _ in parts])
    mass = np.concatenate([m for _, m in parts])
    vel = rng.standard_normal(pos.shape, dtype=np.float32) * np.float32(0.05)
    return _scene(pos, vel, mass, space, 0.01)


def _scenes_of(case, rng):
    sides = _scene_sides(case)
    scs = [_block_scene(k, k, k, 0.01, rng) for k in sides]
    fr = [(float(m), 0.8 * float(m)) for m in 0.3 + 0.4 * rng.random(len(sides))]
    return scs, fr


TEMPLATE = np.array([[(k >> 2) & 1, (k >> 1) & 1, k & 1] for k in range(8)], np.float32) - 0.5


def _smooth_velocity(pos, rng):
    """A coarse flow: a few long waves and some noise per particle."""
    v = np.zeros(pos.shape, np.float32)
    for _ in range(3):
        k = rng.normal(0.0, 3.0, 3).astype(np.float32)
        a = rng.normal(0.0, 0.5, 3).astype(np.float32)
        v += np.sin(pos @ k + np.float32(rng.uniform(0, 6)))[:, None] * a
    return v + rng.standard_normal(pos.shape, dtype=np.float32) * np.float32(0.05)


def _coarse(case, rng):
    sc = _block_scene(case["nx"], case["ny"], case["nz"], R_COARSE, rng)
    sc.vel = _smooth_velocity(sc.pos, rng)
    return sc


def _fine_of(sc, rng, spread):
    """8 fine particles per coarse one: its template corners, spread about."""
    n = sc.n
    fp = sc.pos[:, None, :] + np.float32(R_COARSE) * TEMPLATE[None]
    fp = (fp + (rng.random((n, 8, 3), dtype=np.float32) * 2 - 1) * np.float32(spread)
          ).reshape(-1, 3).astype(np.float32)
    fv = (np.repeat(sc.vel, 8, axis=0)
          + rng.standard_normal((8 * n, 3), dtype=np.float32) * np.float32(0.05))
    order = np.argsort(_cell_id(fp - np.float32(UP_DT) * fv, sc.cells), kind="stable")
    return np.ascontiguousarray(fp[order]), np.ascontiguousarray(fv[order])


DIMS = ((96, 128), (128, 128), (128, 128), (128, 32))
OFFS = ((0, 0), (12288, 128), (28672, 256), (45056, 384))  # weights, biases per layer


def _weights(rng):
    W, b = np.zeros(49152, np.float32), np.zeros(416, np.float32)
    for l, (k_in, n_out) in enumerate(DIMS):
        a = math.sqrt(6.0 / k_in) * (0.1 if l == 3 else 1.0)
        w = (rng.random((n_out, k_in), dtype=np.float32) * 2 - 1) * np.float32(a)
        c = rng.standard_normal(n_out, dtype=np.float32) * np.float32(0.02)
        if l == 3:
            w[24:] = 0.0
            c[24:] = 0.0
        wo, bo = OFFS[l]
        W[wo:wo + n_out * k_in] = w.ravel()
        b[bo:bo + n_out] = c
    return W, b


def _bf16_bits(x):
    u = np.ascontiguousarray(x, np.float32).view(np.uint32).astype(np.uint64)
    return (((u + 0x7FFF + ((u >> 16) & 1)) >> 16) & 0xFFFF).astype(np.uint16)


def _train_inputs(case, rng):
    """Mid-training: weights, Adam moments after some hundred steps, pairs
    whose features look like 16 neighbours within a few radii."""
    W, b = _weights(rng)
    m = case["steps"] * case["batch"]

    def features(rows):
        f = rng.standard_normal((rows, 16, 6), dtype=np.float32)
        f[:, :, :3] *= np.linspace(1.0, 2.2, 16, dtype=np.float32)[None, :, None]
        f[:, :, 3:] *= np.float32(0.2)
        return _bf16_bits(f.reshape(rows, 96)).view(np.int16)

    x, xe = features(m), features(case["rows"])
    t = rng.standard_normal((m, 24), dtype=np.float32) * np.float32(0.1)
    mom = [rng.standard_normal(W.size, dtype=np.float32) * np.float32(1e-3),
           (rng.random(W.size, dtype=np.float32) + np.float32(0.5)) * np.float32(1e-5),
           rng.standard_normal(b.size, dtype=np.float32) * np.float32(1e-3),
           (rng.random(b.size, dtype=np.float32) + np.float32(0.5)) * np.float32(1e-5)]
    return W, b, mom, x, t, xe


TRAIN_STEP0 = 300
LR = 1e-3


# ---- prepare / run -------------------------------------------------------------
def prepare(case, seed):
    return _PREPARE[case["kind"]](case, np.random.default_rng(seed))


def run(state):
    return _RUN[state["kind"]](state)


class _Saved:
    """A sim's arrays as they were, written back before each pass (a program
    that tries settings from one saved state), in one launch."""

    def __init__(self, live):
        self.live = live
        self.keep = [t.clone() for t in live]

    def restore(self):
        torch._foreach_copy_(self.live, self.keep)


def _prepare_step(case, rng):
    from granular_gpu_amd.device import PlainSim
    sc = _block_scene(case["nx"], case["ny"], case["nz"], 0.01, rng)
    sim = PlainSim(sc, stab=3, solver=case["solver"], mu_s=case["mu"], mu_k=0.8 * case["mu"])
    graph = sim.graph(1) if case["graph"] else None
    return {"kind": "step", "sim": sim, "saved": _Saved([sim.pos, sim.vel]), "graph": graph,
            "steps": case["steps"]}


def _run_step(st):
    st["saved"].restore()
    if st["graph"] is not None:
        st["graph"].launch(st["steps"])
    else:
        st["sim"].step(st["steps"])
    s = st["sim"]
    return [s.pos, s.vel, s.mass, s.p2c, s.cs]


def _prepare_scenes(case, rng):
    from granular_gpu_amd._lib import GG_FLAG_LIST_REFRESH
    from granular_gpu_amd.device import SceneBatch
    scs, fr = _scenes_of(case, rng)
    sb = SceneBatch(scs, fr, stab=3, solver=10, flags=GG_FLAG_LIST_REFRESH)
    sb.capture(1)
    return {"kind": "scenes", "sim": sb, "saved": _Saved([sb.pos, sb.vel]),
            "steps": case["steps"]}


def _run_scenes(st):
    st["saved"].restore()
    sb = st["sim"]
    sb.launch(st["steps"])
    return [sb.pos, sb.vel, sb.mass, sb.p2c, sb.cs]


def _prepare_adaptive(case, rng):
    from granular_gpu_amd._lib import GG_FLAG_LIST_REFRESH
    from granular_gpu_amd.device import AdaptiveSim
    sc = _bed(case["nx"], case["nz"], rng)
    sim = AdaptiveSim(sc, capacity=2 * sc.n, max_mass=8.0, merge_first=True, stab=3, solver=5,
                      gmax=160, bmax=96, flags=GG_FLAG_LIST_REFRESH)
    sim.params.adaptive_rules = 1
    for key, v in dict(min_mass=0.125, split_mass=0.125, merge_dist=1.75, merge_depth=3.0,
                       split_depth=2.0).items():
        setattr(sim.params, key, v)
    live = [sim.pos, sim.vel, sim.mass, sim.adl, sim.remove, sim.merge, sim.mcount, sim.mv,
            sim.surface, sim.sd]
    return {"kind": "adaptive", "sim": sim, "saved": _Saved(live), "n": sc.n,
            "steps": case["steps"]}


def _run_adaptive(st):
    sim = st["sim"]
    st["saved"].restore()
    sim.n = sim.set.n = st["n"]
    sim.step(st["steps"])
    # the count depends on the inputs: the arrays come at their capacity, with
    # the rows past the particles cleared
    n, before = sim.n, sim.stats[-1][2]
    out = [sim.pos, sim.vel, sim.mass, sim.adl, sim.remove, sim.merge, sim.mcount]
    flags = [sim.surface, sim.sd]
    torch._foreach_zero_([t[n:] for t in out] + [t[before:] for t in flags])
    return out + flags + [n]


def _coarse_sim(sc):
    from granular_gpu_amd.device import PlainSim
    sim = PlainSim(sc, stab=3, solver=5)
    sim.grid_build()
    return sim


def _prepare_fine(case, rng):
    from granular_gpu_amd.device import FineSet
    sc = _coarse(case, rng)
    fp, fv = _fine_of(sc, rng, 0.5 * R_COARSE)
    fs = FineSet(_coarse_sim(sc), fp, fv)
    return {"kind": "fine", "fs": fs, "saved": _Saved([fs.pos, fs.vel])}


def _run_fine(st):
    fs = st["fs"]
    st["saved"].restore()
    fs.sort()
    fs.upsample()
    return [fs.pos, fs.vel, fs.p2c]


def _prepare_learned(case, rng):
    from granular_gpu_amd.learned import LearnedUpsampler, MlpNet
    sc = _coarse(case, rng)
    sim = _coarse_sim(sc)
    up = LearnedUpsampler(MlpNet(master=_weights(rng)))
    out = [torch.empty((sc.n, 24), dtype=torch.float32, device="cuda") for _ in range(2)]
    return {"kind": "learned", "sim": sim, "up": up, "out": out}


def _run_learned(st):
    st["up"].infer(st["sim"], fine_pos=st["out"][0], fine_vel=st["out"][1])
    return st["out"]


def _prepare_pairs(case, rng):
    from granular_gpu_amd.device import PlainSim
    from granular_gpu_amd.learned import LearnedUpsampler, MlpNet
    sc, fine = _twins(case, rng)
    sim, fsim = PlainSim(sc, stab=3, solver=5), PlainSim(fine, stab=3, solver=5)
    return {"kind": "pairs", "sim": sim, "fsim": fsim, "up": LearnedUpsampler(MlpNet(seed=1)),
            "saved": _Saved([sim.pos, sim.vel, fsim.pos, fsim.vel])}


def _twins(case, rng):
    sc = _coarse(case, rng)
    fp, fv = _fine_of(sc, rng, 0.1 * R_COARSE)
    return sc, _scene(fp, fv, np.ones(fp.shape[0], np.float32), sc.space, 0.01)


def _run_pairs(st):
    from granular_gpu_amd.learned import fine_targets
    sim, fsim, up = st["sim"], st["fsim"], st["up"]
    st["saved"].restore()
    sim.grid_build()
    fsim.grid_build()
    feat, flags, knn = up.features(sim)
    y, d2, match = fine_targets(sim, fsim, up.cfg)
    return [feat, flags, knn, y, d2, match, sim.pos, fsim.pos]


def _prepare_train(case, rng):
    from granular_gpu_amd.learned import MlpNet, Trainer
    W, b, mom, x, t, xe = _train_inputs(case, rng)
    net = MlpNet(master=(W, b))
    for live, v in zip((net.m_w, net.v_w, net.m_b, net.v_b), mom):
        live.copy_(torch.from_numpy(v))
    net.step = TRAIN_STEP0
    tr = Trainer(net, batch=case["batch"])
    B = case["batch"]
    x, t = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
    mini = [(x[k * B:(k + 1) * B].contiguous(), t[k * B:(k + 1) * B].contiguous())
            for k in range(case["steps"])]
    return {"kind": "train", "tr": tr, "mini": mini, "xe": torch.from_numpy(xe).cuda()}


def _run_train(st):
    tr = st["tr"]
    for x, t in st["mini"]:
        tr.grad(x, t)
        tr.adam(lr=LR)
    y = tr.forward(st["xe"])
    n = tr.net
    return [tr.dW, tr.db, tr.sq, n.w_master, n.b_master, n.m_w, n.v_w, y]


_PREPARE = {"step": _prepare_step, "scenes": _prepare_scenes, "adaptive": _prepare_adaptive,
            "fine": _prepare_fine, "learned": _prepare_learned, "pairs": _prepare_pairs,
            "train": _prepare_train}
_RUN = {"step": _run_step, "scenes": _run_scenes, "adaptive": _run_adaptive, "fine": _run_fine,
        "learned": _run_learned, "pairs": _run_pairs, "train": _run_train}


# ---- work -----------------------------------------------------------------------
def _box_counts(nx, ny, nz, r):
    s = 1.97 * r
    space = [max(1.2 * s * k, s * (k - 1) + 0.25) for k in (nx, ny, nz)]
    c = _cells(space)
    m = [2 * k for k in c]
    walls = m[0] * m[1] * m[2] - (m[0] - 2) * (m[1] - 2) * (m[2] - 2)
    return c[0] * c[1] * c[2], walls


# per particle and sweep: about 6 contacts of some 40 operations each
SWEEP_FLOPS = 240
# multiply-adds of one sample through the network
MLP_FMA = 96 * 128 + 2 * 128 * 128 + 128 * 24


def work(case):
    k = case["kind"]
    if k == "step":
        n = case["nx"] * case["ny"] * case["nz"]
        c, w = _box_counts(case["nx"], case["ny"], case["nz"], 0.01)
        per = 28 * n + 32 * n + 16 * w + 8 * c  # state in and out, walls, tables
        return {"bytes": case["steps"] * per,
                "flops": case["steps"] * n * ((3 + case["solver"]) * SWEEP_FLOPS + 100)}
    if k == "scenes":
        n = case["total"]
        return {"bytes": case["steps"] * 64 * n, "flops": case["steps"] * n * (13 * SWEEP_FLOPS + 100)}
    if k == "adaptive":
        area = 0.0004 * case["nx"] * case["nz"]
        n = int(area * (6 / 0.0016 + 6 / 0.0004 + 2 / 0.0001))
        return {"bytes": case["steps"] * 110 * n,
                "flops": case["steps"] * n * (8 * SWEEP_FLOPS + 4 * 30 * 20)}
    n = 0 if k == "train" else case["nx"] * case["ny"] * case["nz"]
    if k == "fine":
        c, w = _box_counts(case["nx"], case["ny"], case["nz"], R_COARSE)
        return {"bytes": 8 * n * 52 + 24 * n + 12 * w + 8 * c, "flops": 8 * n * 27 * 20}
    if k == "learned":
        c, w = _box_counts(case["nx"], case["ny"], case["nz"], R_COARSE)
        return {"bytes": 24 * n + 8 * n * 24 + 12 * w + 8 * c, "flops": n * (2 * MLP_FMA + 27 * 8)}
    if k == "pairs":
        return {"bytes": n * (48 + 192 + 4 + 64 + 96 + 64) + 8 * n * 48,
                "flops": n * (27 * 8 + 8 * 216 * 8)}
    m, rows = case["steps"] * case["batch"], case["rows"]
    return {"bytes": (m + rows) * (192 + 96) + case["steps"] * 49152 * 4 * 7,
            "flops": 2 * MLP_FMA * (3 * m + rows)}


# ---- exact ----------------------------------------------------------------------
def exact(case, seed):
    """None for the steps: whether a pair that the sweep before left exactly
    touching counts as a contact is decided by the last bit, so a run in 64
    bits takes other decisions and is no reference for a whole step."""
    fn = _EXACT.get(case["kind"])
    return fn(case, np.random.default_rng(seed)) if fn else None


def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Sorted:
    """A point set in stable cell order with its cell table, on the device."""

    def __init__(self, pos, cells, *more):
        cid = _cell_id(pos, cells)
        self.order = np.argsort(cid, kind="stable")
        self.cid = cid
        self.cells = cells
        count = np.bincount(cid, minlength=cells[0] * cells[1] * cells[2] + 1)
        self.cs = torch.from_numpy(np.concatenate([[0], np.cumsum(count)])).to(_dev())
        self.pos = torch.from_numpy(pos[self.order].astype(np.float64)).to(_dev())
        self.more = [torch.from_numpy(m[self.order].astype(np.float64)).to(_dev()) for m in more]


def _stencil(near, base):
    """Indices (-1: none) of the members of near in the 27 cells around each
    base cell, ascending."""
    cx, cy, cz = near.cells
    z0 = (base[:, 2] - 1).clamp(min=0)
    z1 = (base[:, 2] + 1).clamp(max=cz - 1)
    starts, lens = [], []
    for dx in (-1, 0, 1):
        for dy in (-1, 0, 1):
            x, y = base[:, 0] + dx, base[:, 1] + dy
            ok = (x >= 0) & (x < cx) & (y >= 0) & (y < cy) & (z0 <= z1)
            c = torch.where(ok, (x * cy + y) * cz, torch.zeros_like(x))
            a = near.cs[torch.where(ok, c + z0, torch.zeros_like(x))]
            b = near.cs[torch.where(ok, c + z1 + 1, torch.zeros_like(x))]
            starts.append(a)
            lens.append(torch.where(ok, b - a, torch.zeros_like(a)))
    width = max(1, int(torch.stack(lens).max()))
    k = torch.arange(width, device=base.device)
    return torch.cat([torch.where(k[None] < n[:, None], a[:, None] + k[None], -1)
                      for a, n in zip(starts, lens)], 1)


def _chunks(n, rows=65536):
    return [(a, min(n, a + rows)) for a in range(0, n, rows)]


def _base(pos32):
    """floor(p / L) with the single-precision quotient the cells are defined by."""
    return torch.from_numpy(np.floor(pos32 / L).astype(np.int64)).to(_dev())


def _advect(p, v, base, coarse, walls):
    """The plain upsampler's update of fine particles in 64 bits (its
    constants: gg_upsample_params)."""
    r9 = float(np.float32(493.8271605))
    g = torch.zeros(3, dtype=torch.float64, device=p.device)
    g[1] = float(np.float32(-9.8)) * float(np.float32(UP_DT))
    brad, dt = float(np.float32(0.015)), float(np.float32(UP_DT))
    out_p, out_v = torch.empty_like(p), torch.empty_like(v)
    for a, b in _chunks(p.shape[0]):
        P, V = p[a:b], v[a:b]
        j = _stencil(coarse, base[a:b])
        d2 = ((P[:, None] - coarse.pos[j.clamp(min=0)]) ** 2).sum(-1)
        w = (1.0 - d2 * r9).clamp(min=0.0) ** 3 * (j >= 0)
        gw = w.sum(1)
        mean = (w[..., None] * coarse.more[0][j.clamp(min=0)]).sum(1) / gw.clamp(min=1e-30)[:, None]
        keep = (1.0 - w.max(1).values).clamp(min=0.0)[:, None]
        j = _stencil(walls, base[a:b])
        t = P[:, None] - walls.pos[j.clamp(min=0)]
        d = t.square().sum(-1).sqrt()
        hit = (d < brad) & (j >= 0)
        f = torch.where(hit, 3.0 * (brad - d) / brad / (d + 1e-6), torch.zeros_like(d))
        push = (t * f[..., None]).sum(1)
        near = hit.any(1)
        free = V + g
        damped = free * 0.8
        damped[:, 1] = torch.where(P[:, 1] < 0.1, damped[:, 1] * 0.5, damped[:, 1])
        alone = torch.where(near[:, None], damped, free)
        u = torch.where((gw > 1e-6)[:, None], keep * free + (1.0 - keep) * mean, alone) + push
        u = u.clamp(-7.0, 7.0)
        q = P + u * dt
        low = q[:, 1] < float(np.float32(0.04))
        q[:, 1] = torch.where(low, float(np.float32(0.04)), q[:, 1])
        u[:, 1] = torch.where(low, 0.0, u[:, 1])
        for ax in (0, 2):
            u[:, ax] = torch.where(low, u[:, ax] * float(np.float32(0.95)), u[:, ax])
            out = q[:, ax] < 0.0
            q[:, ax] = torch.where(out, 0.0, q[:, ax])
            u[:, ax] = torch.where(out, 0.0, u[:, ax])
        out_p[a:b], out_v[a:b] = q, u
    return out_p, out_v


def _exact_fine(case, rng):
    sc = _coarse(case, rng)
    fp, fv = _fine_of(sc, rng, 0.5 * R_COARSE)
    coarse, walls = _Sorted(sc.pos, sc.cells, sc.vel), _Sorted(sc.boundary, sc.cells)
    fine = _Sorted(fp, sc.cells, fv)
    p, v = _advect(fine.pos, fine.more[0], _base(fp[fine.order]), coarse, walls)
    return [p, v, None]


def _bf16(x):
    return x.to(torch.float32).to(torch.bfloat16).to(torch.float64)


def _layers(W, b):
    out = []
    for (k_in, n_out), (wo, bo) in zip(DIMS, OFFS):
        w = W[wo:wo + n_out * k_in].reshape(n_out, k_in)
        out.append((_bf16(w), b[bo:bo + n_out]))
    return out


def _network(x, layers):
    """Hidden activations, pre-activations and the 24 outputs, with the
    bfloat16 weights the network holds and nothing else rounded."""
    hs, zs = [x], []
    for l, (w, c) in enumerate(layers):
        z = hs[-1] @ w.T + c
        zs.append(z)
        if l < 3:
            hs.append(z.clamp(min=0.0))
    return hs, zs, zs[3][:, :24]


def _exact_learned(case, rng):
    sc = _coarse(case, rng)
    W, b = (torch.from_numpy(a).to(_dev()).double() for a in _weights(rng))
    layers = _layers(W, b)
    coarse, walls = _Sorted(sc.pos, sc.cells, sc.vel), _Sorted(sc.boundary, sc.cells)
    P, V = coarse.pos, coarse.more[0]
    base = _base(sc.pos[coarse.order])
    n = P.shape[0]
    R, dt = float(np.float32(R_COARSE)), float(np.float32(UP_DT))
    T = torch.from_numpy(TEMPLATE.astype(np.float64)).to(P.device)
    fp = torch.empty((n, 8, 3), dtype=torch.float64, device=P.device)
    fv = torch.empty_like(fp)
    flag = torch.zeros(n, dtype=torch.bool, device=P.device)
    for lo, hi in _chunks(n):
        p, v = P[lo:hi], V[lo:hi]
        j = _stencil(coarse, base[lo:hi])
        d2 = ((p[:, None] - coarse.pos[j.clamp(min=0)]) ** 2).sum(-1)
        me = torch.arange(lo, hi, device=P.device)[:, None]
        d2 = torch.where((j >= 0) & (j != me), d2, float("inf"))
        if d2.shape[1] < 16:
            pad = 16 - d2.shape[1]
            d2 = torch.nn.functional.pad(d2, (0, pad), value=float("inf"))
            j = torch.nn.functional.pad(j, (0, pad), value=-1)
        order = torch.argsort(d2, dim=1, stable=True)[:, :16]
        d2, j = torch.gather(d2, 1, order), torch.gather(j, 1, order)
        has = torch.isfinite(d2)[..., None]
        k = j.clamp(min=0)
        f = torch.cat([torch.where(has, (P[k] - p[:, None]) / R, 0.0),
                       torch.where(has, V[k] - v[:, None], 0.0)], -1)
        _, _, y = _network(f.reshape(hi - lo, 96), layers)
        fv[lo:hi] = v[:, None] + y.reshape(-1, 8, 3)
        fp[lo:hi] = p[:, None] + R * T[None] + dt * fv[lo:hi]
        j = _stencil(walls, base[lo:hi])
        d2 = ((p[:, None] - walls.pos[j.clamp(min=0)]) ** 2).sum(-1)
        flag[lo:hi] = ((d2 < 0.0025) & (j >= 0)).any(1)
    flag |= (P[:, 1] < 0.08) | (P[:, 0] < 0.05) | (P[:, 2] < 0.05)
    at = torch.nonzero(flag).flatten()
    if at.numel():
        p32 = sc.pos[coarse.order][at.cpu().numpy()]
        q32 = (p32[:, None, :] + np.float32(R_COARSE) * TEMPLATE[None]).reshape(-1, 3)
        q, u = _advect(torch.from_numpy(q32.astype(np.float64)).to(P.device),
                       V[at].repeat_interleave(8, 0), _base(q32), coarse, walls)
        fp[at], fv[at] = q.reshape(-1, 8, 3), u.reshape(-1, 8, 3)
    return [fp.reshape(n, 24), fv.reshape(n, 24)]


def _exact_pairs(case, rng):
    sc, fine = _twins(case, rng)
    coarse = _Sorted(sc.pos, sc.cells, sc.vel)
    fs = _Sorted(fine.pos, sc.cells, fine.vel)
    p32 = sc.pos[coarse.order]
    q32 = (p32[:, None, :] + np.float32(R_COARSE) * TEMPLATE[None]).reshape(-1, 3)
    q, base = torch.from_numpy(q32.astype(np.float64)).to(_dev()), _base(q32)
    y, d2 = torch.empty_like(q), torch.empty(q.shape[0], dtype=torch.float64, device=q.device)
    for a, b in _chunks(q.shape[0], 32768):
        j = _stencil(fs, base[a:b])
        d = ((q[a:b, None] - fs.pos[j.clamp(min=0)]) ** 2).sum(-1)
        best = torch.where(j >= 0, d, float("inf")).min(1)
        d2[a:b] = best.values
        at = torch.gather(j, 1, best.indices[:, None])[:, 0]
        v = coarse.more[0][torch.arange(a, b, device=q.device) // 8]
        y[a:b] = torch.where((at >= 0)[:, None], fs.more[0][at.clamp(min=0)] - v, 0.0)
    n = p32.shape[0]
    return [None, None, None, y.reshape(n, 24), d2.reshape(n, 8), None, coarse.pos, fs.pos]


def _exact_train(case, rng):
    W, b, mom, x, t, xe = _train_inputs(case, rng)
    dev = _dev()
    W, b, mw, vw, mb, vb = (torch.from_numpy(a).to(dev).double() for a in (W, b, *mom))

    def rows(bits):
        u = np.ascontiguousarray(bits).view(np.uint16).astype(np.uint32) << 16
        return torch.from_numpy(u.view(np.float32).astype(np.float64)).to(dev)

    x, xe, t = rows(x), rows(xe), torch.from_numpy(t).to(dev).double()
    B = case["batch"]
    b1, b2, eps, lr = (float(np.float32(v)) for v in (0.9, 0.999, 1e-8, LR))
    for k in range(case["steps"]):
        xb, tb = x[k * B:(k + 1) * B], t[k * B:(k + 1) * B]
        layers = _layers(W, b)
        hs, zs, y = _network(xb, layers)
        e = y - tb
        sq = e.square().sum(1)
        g = torch.zeros((B, 32), dtype=torch.float64, device=dev)
        g[:, :24] = e * (2.0 / (24 * B))
        dW, db = torch.zeros_like(W), torch.zeros_like(b)
        for l in (3, 2, 1, 0):
            (k_in, n_out), (wo, bo) = DIMS[l], OFFS[l]
            dW[wo:wo + n_out * k_in] = (g.T @ hs[l]).reshape(-1)
            db[bo:bo + n_out] = g.sum(0)
            if l:
                g = (g @ layers[l][0]) * (zs[l - 1] > 0)
        s = TRAIN_STEP0 + k + 1
        c1, c2 = 1.0 / (1.0 - b1 ** s), 1.0 / (1.0 - b2 ** s)
        mw, vw = b1 * mw + (1 - b1) * dW, b2 * vw + (1 - b2) * dW * dW
        mb, vb = b1 * mb + (1 - b1) * db, b2 * vb + (1 - b2) * db * db
        W = W - lr * (mw * c1) / ((vw * c2).sqrt() + eps)
        b = b - lr * (mb * c1) / ((vb * c2).sqrt() + eps)
    y = _network(xe, _layers(W, b))[2]
    return [dW, db, sq, W, b, mw, vw, y]


_EXACT = {"fine": _exact_fine, "learned": _exact_learned, "pairs": _exact_pairs,
          "train": _exact_train}
