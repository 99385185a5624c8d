"""The framework's measured cases: renders, batched jobs and the proposal network, through the
entry points a user's program calls.

A render case is what the CLI's main loop does: load a scene, create a renderer, run `iters`
progressive 1-spp iterations and read the mean image. Its fields are the command line's: scene
(kind of gpuupbp_amd.workloads.scene, or "predefined" with its -s id), resolution, maximum path
length, techniques, initial radius, light paths as a share of the pixels, beam types, and whether
the iteration is replayed from a captured graph or guided by installed proposal lobes. A batch case
renders a round of independent jobs; the mlp cases run the proposal's network on host arrays.
"""
import math
import os
import tempfile

import numpy as np

from gpuupbp_amd import capi
from gpuupbp_amd import workloads as wl
from gpuupbp_amd.renderer import Batch, Mlp, Renderer

ALL_SIX = "upbp_bpt+surf+pp3d+pb2d+bb1d+bp2d"
# iterations a render cycles through: successive passes are successive iterations of the radius
# schedule, and the work of a pass stays the same however many passes are made
CYCLE = 4


def render(scene, scene_seed, w, h, l, alg, r, iters=1, light=1.0, qbt="L", pbt="S", graph=False, guide=False):
    return {"kind": "render", "scene": scene, "scene_seed": scene_seed, "w": w, "h": h, "l": l, "alg": alg, "r": r,
            "iters": iters, "light": light, "qbt": qbt, "pbt": pbt, "graph": graph, "guide": guide}


def listed():
    cases = [
        # the smallest call: one preview iteration of the box thumbnail
        ("box_preview", render("box", 0, 64, 64, 8, ALL_SIX, 0.01)),
        # the CPU-runnable box workload at its own size, four iterations
        ("box", render("box", 0, 256, 256, 8, ALL_SIX, 0.01, iters=4)),
        # dense anisotropic fog at an odd size, long photon beams, replayed from a captured graph
        ("boxfog_graph", render("boxfog", 0, 333, 217, 12, "upbp_all", 0.01, iters=4, pbt="L", graph=True)),
        # glass, water and ice spheres in a weak fog: the reference's predefined scenes
        ("predefined", render("predefined", 27, 320, 240, 10, "upbp_all", 0.01, iters=2)),
        # bidirectional path tracing alone: connections and occlusion rays over 184k triangles
        ("bpt", render("blobs_small", 5, 640, 360, 10, "upbp_bpt", 0.01, iters=2)),
        # photon points only (surface, P-P3D, P-B2D) with few light paths and short query beams
        ("points", render("blobs_small", 2, 501, 283, 12, "upbp_bpt+surf+pp3d+pb2d", 0.02, light=0.5, qbt="S")),
        # the learned proposal's workload: the dense g = 0.9 slab, plain, at three quarters of its size
        ("slabroom", render("slabroom", 3, 960, 540, 16, "upbp_all", 0.01)),
        # the same kind of room with a proposal installed: guided sampling and its pdf in every merge
        ("guided", render("slabroom_small", 1, 256, 256, 12, "upbp_all", 0.01, iters=2, guide=True)),
        # the largest: the blob grid of bench.py, 1.31M triangles, three media, 900k light paths
        ("blobs", render("blobs", 1, 1280, 720, 12, "upbp_all", 0.005, light=900000 / (1280 * 720))),
        # independent jobs of uneven sizes in one launch per stage, the round replayed from a graph
        ("batch", {"kind": "batch", "jobs": 12, "mix": 2, "graph": True}),
        # one training step of the proposal's network on the online trainer's batch
        ("mlp_train", {"kind": "mlp_train", "n": 65536}),
        # its outputs at the centres of the 64^3 record grid
        ("mlp_forward", {"kind": "mlp_forward", "n": 262144}),
    ]
    return [dict(c, name=name) for name, c in cases]


# largest width drawn, so that no drawn case costs more than the largest listed one
DRAWN_SCENES = [("box", 900), ("boxfog", 640), ("blobs_small", 900), ("slabroom_small", 400), ("slabroom", 640),
                ("predefined", 640), ("blobs", 960)]
DRAWN_ALGS = [ALL_SIX, "upbp_all", "upbp_all", "upbp_bpt", "upbp_bpt+surf", "upbp_bpt+surf+pp3d+pb2d",
              "upbp_bpt+pb2d+bb1d"]
DRAWN_PREDEFINED = [1, 2, 5, 7, 8, 11, 15, 21, 27, 28, 30, 33, 36, 39, 40]


def log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["render", "mlp_train", "mlp_forward", "batch"], [16, 2, 2, 1])[0]
    if kind == "mlp_train":
        return {"kind": kind, "n": log_uniform(rng, 256, 65536)}
    if kind == "mlp_forward":
        return {"kind": kind, "n": log_uniform(rng, 1, 262144)}
    if kind == "batch":
        return {"kind": kind, "jobs": rng.randint(2, 10), "mix": rng.randint(1, 1000), "graph": rng.random() < 0.5}
    scene, wmax = rng.choices(DRAWN_SCENES, [4, 3, 4, 3, 2, 4, 1])[0]
    w = log_uniform(rng, 48, wmax)
    h = max(16, int(w * rng.uniform(0.5, 1.0)))
    seed = {"blobs_small": rng.randint(0, 11), "slabroom_small": rng.randint(0, 3), "slabroom": 3, "blobs": 1,
            "predefined": rng.choice(DRAWN_PREDEFINED)}.get(scene, 0)
    return render(scene, seed, w, h, rng.randint(4, 16), rng.choice(DRAWN_ALGS),
                  0.005 if scene == "blobs" else round(rng.uniform(0.005, 0.02), 4),
                  iters=1 if scene in ("blobs", "slabroom") else rng.randint(1, 3),
                  light=rng.choice([0.25, 0.5, 1.0, 1.0]), qbt=rng.choice("LLS"), pbt=rng.choice("SSL"),
                  graph=rng.random() < 0.3, guide=rng.random() < 0.15)


def scene_dir():
    d = os.path.join(tempfile.gettempdir(), "upbp_case_scenes_%d" % os.getuid())
    os.makedirs(d, exist_ok=True)
    return d


def light_paths(case):
    return max(1, int(round(case["light"] * case["w"] * case["h"])))


def stream_offset(seed):
    """The -ioff of a seed: random streams shared with no other seed's."""
    return str((int(seed) % (1 << 24)) * 64)


def prepare_render(case, seed):
    if case["scene"] == "predefined":
        path, head = case["scene_seed"], ["-s", str(case["scene_seed"])]
    else:
        path = wl.scene(scene_dir(), case["scene"], case["scene_seed"])
        head = ["-s", "-1", path]
    rc, cfg = capi.parse_args(head + ["-r", "%dx%d" % (case["w"], case["h"]), "-l", str(case["l"]),
                                      "-pcpi", str(light_paths(case)), "-a", case["alg"], "-r_initial", str(case["r"]),
                                      "-qbt", case["qbt"], "-pbt", case["pbt"], "-ioff", stream_offset(seed)])
    if rc != 0:
        raise ValueError("command line rejected: %r" % (case,))
    sh = capi.SceneHandle(path, cfg.res_x, cfg.res_y)
    r = Renderer(sh.ptr, cfg)
    if case["graph"]:
        r.set_tuning(graph=1)
    if case["guide"]:
        # sharp to broad lobes in random directions on a coarse grid over the scene's cube
        rng = np.random.default_rng(seed)
        res = 8
        n = res ** 3 * 8
        mu = rng.normal(size=(n, 3))
        lobes = np.hstack([mu / np.linalg.norm(mu, axis=1, keepdims=True), np.exp(rng.uniform(-2, 4, (n, 1))),
                           rng.uniform(0.05, 1, (n, 1))]).astype(np.float32)
        c, rad = np.array(list(sh.scene.scene_center)), sh.scene.scene_radius
        r.set_guide_lobes(lobes, res, c - rad, c + rad, 0.65)
    sh.close()
    return {"kind": "render", "renderer": r, "iters": case["iters"], "done": 0}


def prepare_batch(case, seed):
    rs = []
    for obj, argv, _, _, _ in wl.batch_mix(scene_dir(), case["jobs"], case["mix"]):
        rc, cfg = capi.parse_args(argv + ["-ioff", stream_offset(seed)])
        if rc != 0:
            raise ValueError("command line rejected: %r" % (argv,))
        sh = capi.SceneHandle(obj, cfg.res_x, cfg.res_y)
        rs.append(Renderer(sh.ptr, cfg))
        sh.close()
    return {"kind": "batch", "batch": Batch(rs, use_graph=case["graph"]), "renderers": rs, "done": 0}


def mlp_samples(case, seed):
    """Positions in the unit cube, arrival directions (zero in the online trainer's samples, which
    learn incident radiance); a training sample adds the scattered direction, gathered around a
    direction that turns with the position, and a positive weight with a long tail."""
    rng = np.random.default_rng(seed)
    n = case["n"]
    x = rng.uniform(0, 1, (n, 3))
    arrive = np.zeros((n, 3))
    if case["kind"] == "mlp_forward":
        return np.ascontiguousarray(np.hstack([x, arrive]), np.float32)
    axis = np.stack([np.cos(4 * x[:, 0]), np.sin(4 * x[:, 0]), x[:, 1] - 0.5], 1)
    d = axis + 0.6 * rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return np.ascontiguousarray(np.hstack([x, arrive, d, rng.gamma(0.5, 2.0, (n, 1)) + 1e-3]), np.float32)


def prepare(case, seed):
    if case["kind"] == "render":
        return prepare_render(case, seed)
    if case["kind"] == "batch":
        return prepare_batch(case, seed)
    return {"kind": case["kind"], "mlp": Mlp(seed=3), "samples": mlp_samples(case, seed)}


def run(state):
    if state["kind"] == "mlp_forward":
        return state["mlp"].forward(state["samples"])
    if state["kind"] == "mlp_train":
        loss = state["mlp"].train_step(state["samples"], LEARNING_RATE)
        return {"loss": loss, "params": state["mlp"].params()}
    if state["kind"] == "batch":
        state["batch"].run([state["done"] % CYCLE] * len(state["renderers"]))
        state["done"] += 1
        return [r.read_accum(state["done"]) for r in state["renderers"]]
    for _ in range(state["iters"]):
        state["renderer"].run_iteration(state["done"] % CYCLE, want_stats=False)
        state["done"] += 1
    return state["renderer"].read_accum(state["done"])


# ---- what a pass cannot do without -----------------------------------------------------------------
TRIANGLES = {"box": 1292, "boxfog": 1292, "slabroom_small": 770, "slabroom": 194982, "blobs": 1314566,
             "blobs_small": 83206, "predefined": 40}
# accepted beam-beam pairs per (pixel x light path x unit of radius), from the renderer's own counters
BEAM_PAIRS = {"box": 0.02, "boxfog": 0.1, "blobs_small": 0.05, "slabroom_small": 0.2, "slabroom": 0.2, "blobs": 0.06,
              "predefined": 0.05}
WEIGHTS = 64 * 64 + 64 * 64 + 64 * 64 + 48 * 64


def render_work(scene, w, h, l, alg, r, light, iters):
    """Scene read and image written once; per iteration a box test per tree level, a hit and its
    scattering per path segment (four segments a path), and each beam pair's estimator."""
    px, tris = w * h, TRIANGLES[scene]
    segments = 4 if l >= 4 else l
    flops = (px + light) * segments * (48 * math.log2(tris + 1) + 800.0)
    if "all" in alg or "bb1d" in alg:
        flops += 250.0 * BEAM_PAIRS[scene] * r * px * light
    return {"bytes": 92.0 * tris + 24.0 * px, "flops": float(iters) * flops}


def work(case):
    if case["kind"] == "render":
        return render_work(case["scene"], case["w"], case["h"], case["l"], case["alg"], case["r"], light_paths(case),
                           case["iters"])
    if case["kind"] == "batch":
        out = {"bytes": 0.0, "flops": 0.0}
        for _, argv, px, kind, length in wl.batch_mix(scene_dir(), case["jobs"], case["mix"]):
            side = int(round(math.sqrt(px)))
            one = render_work(kind, side, side, length, "upbp_all", 0.01, px, 1)
            out = {k: out[k] + one[k] for k in out}
        return out
    n = case["n"]
    if case["kind"] == "mlp_forward":
        return {"bytes": n * (24.0 + 160.0) + 2.0 * WEIGHTS, "flops": 2.0 * WEIGHTS * n}
    return {"bytes": n * 40.0 + 3 * 2 * 4.0 * 14248, "flops": 6.0 * WEIGHTS * n}


def tolerance(case):
    # Renders and the network's outputs are the same paths and products in FP32 sums whose order
    # the atomics choose; a path whose FP32 decision falls the other way moves a few pixels.
    if case["kind"] == "mlp_forward":
        return {"rel": 1e-3, "max": 0.05}  # BF16 operands, FP32 sums
    if case["kind"] == "mlp_train":
        return {"rel": 1e-3, "max": 0.05}
    return {"rel": 2e-3, "max": 0.9}


# ---- the network in 64 bits ------------------------------------------------------------------------
LEARNING_RATE = 8e-3
SHAPES = [(64, 51), (64, 64), (64, 64), (40, 64)]


def split(p):
    ws, bs, at = [], [], 0
    for rows, cols in SHAPES:
        ws.append(p[at:at + rows * cols].reshape(rows, cols))
        at += rows * cols
        bs.append(p[at:at + rows])
        at += rows
    return ws, bs


def initial_params(seed=3):
    """He initialisation: Box-Muller over a splitmix64 stream of the seed, biases zero."""
    mask = (1 << 64) - 1
    st = (0x9E3779B97F4A7C15 * (seed + 1)) & mask

    def nxt():
        nonlocal st
        st = (st + 0x9E3779B97F4A7C15) & mask
        z = st
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        return ((z ^ (z >> 31)) >> 11) / 9007199254740992.0

    out = []
    for rows, cols in SHAPES:
        sd = math.sqrt(2.0 / cols)
        for _ in range(rows * cols):
            u1, u2 = max(nxt(), 1e-300), nxt()
            out.append(sd * math.sqrt(-2.0 * math.log(u1)) * math.cos(2.0 * math.pi * u2))
        out += [0.0] * rows
    return np.array(out, np.float32).astype(np.float64)


def encode(s):
    f = np.zeros((len(s), 51))
    for j in range(3):
        for k in range(8):
            a = (2.0 ** k) * math.pi * s[:, j]
            f[:, (j * 8 + k) * 2] = np.sin(a)
            f[:, (j * 8 + k) * 2 + 1] = np.cos(a)
    f[:, 48:] = s[:, 3:6]
    return f


def exact(case, seed):
    if case["kind"] not in ("mlp_forward", "mlp_train"):
        return None  # a Monte Carlo render has no plain 64-bit counterpart
    s = mlp_samples(case, seed).astype(np.float64)
    p = initial_params()
    ws, bs = split(p)
    acts = [encode(s)]
    for k in range(3):
        acts.append(np.maximum(acts[-1] @ ws[k].T + bs[k], 0.0))
    o = acts[3] @ ws[3].T + bs[3]
    if case["kind"] == "mlp_forward":
        return o
    n = len(s)
    o5 = o.reshape(n, 8, 5)
    d, weight = s[:, 6:9], s[:, 9]
    norm = np.linalg.norm(o5[:, :, :3], axis=2)
    mu = o5[:, :, :3] / norm[:, :, None]
    kap = np.logaddexp(0.0, o5[:, :, 3]) + 0.01
    e = np.exp(o5[:, :, 4] - o5[:, :, 4].max(axis=1, keepdims=True))
    pi = e / e.sum(axis=1, keepdims=True)
    cd = np.einsum("nlk,nk->nl", mu, d)
    v = kap / (2 * math.pi * -np.expm1(-2 * kap)) * np.exp(kap * (cd - 1))
    q = (pi * v).sum(axis=1)
    gam = pi * v / q[:, None]
    g = np.zeros((n, 8, 5))
    g[:, :, 4] = pi - gam
    g[:, :, 3] = -gam * (1 / kap - 2 / np.expm1(2 * kap) + cd - 1) / (1 + np.exp(-o5[:, :, 3]))
    g[:, :, :3] = (d[:, None, :] - mu * cd[:, :, None]) * (-gam * kap / norm)[:, :, None]
    delta = (g * (weight / n)[:, None, None]).reshape(n, 40)
    gw, gb = [None] * 4, [None] * 4
    for k in (3, 2, 1, 0):
        gw[k], gb[k] = delta.T @ acts[k], delta.sum(axis=0)
        if k:
            delta = (delta @ ws[k]) * (acts[k] > 0)
    grad = np.concatenate([np.concatenate([a.ravel(), b]) for a, b in zip(gw, gb)])
    # Adam's first step: both moments over their bias corrections are the gradient and its square
    return {"loss": float(np.mean(weight * -np.log(q))),
            "params": p - LEARNING_RATE * grad / (np.abs(grad) + 1e-8)}
