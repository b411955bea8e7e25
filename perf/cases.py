"""The work a user of this framework has it do, as cases that can be timed.

Each case is one pass through the public entry points of `lyapunov3d_amd`:
lambda at points and over volumes, frames rendered one by one or as a batch,
views and volume blocks in one launch, and a burst of requests through the
serving loop. Sizes, boxes, sequences and iteration counts are those of the
seeded workloads the tests and the benchmark use, of the reference-shaped
driver (the default scene), or odd sizes of the same kind. A seed moves the
inputs within the same distribution: points and boxes are shifted, cameras
turned, batches drawn again.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import lyapunov3d_amd as lyap

CENTER = (3.0, 3.0, 3.0)
PRECISIONS = {"plain": lyap.PREC_PLAIN, "product": lyap.PREC_PRODUCT, "fp64": lyap.PREC_FP64}
#: Volume re-evaluation rules: (fp64_margin, converge_tau, converge_band).
RULES = {"none": (0.0, 0.0, 0.0), "margin": (0.01, 0.0, 0.0), "strict": (0.01, 1e-4, 0.2)}
#: Mean lambda evaluations per pixel of the march scenes (samples up to the
#: first opaque one, refinement, normal; rays that miss the box have none).
EVALS_PER_PIXEL = 20.0

_ctx = None


def context():
    """The one context a program on this device keeps."""
    global _ctx
    if _ctx is None:
        _ctx = lyap.Context(0)
    return _ctx


# ------------------------------------------------------------------ cases ----

def listed():
    return [
        # a probe of a few points under the cursor: the smallest call, latency
        dict(name="points_probe", kind="points", n=61, precision="plain", rule="none", seq="BCABA",
             settle=18, accum=1008, d=2.1, lo=2.0, edge=2.0),
        # a scattered point set (an isosurface tool's samples), ragged count
        dict(name="points_scattered", kind="points", n=100003, precision="product", rule="margin",
             seq="ABCABCCA", settle=200, accum=2000, d=2.1, lo=2.5, edge=1.5),
        # the plain volume workload: a preview volume
        dict(name="volume_preview", kind="volume", nx=64, ny=64, nz=64, precision="product",
             rule="none", seq="ABBAC", settle=100, accum=400, d=2.1, lo=2.0, edge=2.0),
        # the reference's volume program: default scene, per-step log, box [0, 4)
        dict(name="volume_reference", kind="volume", nx=128, ny=128, nz=128, precision="plain",
             rule="none", seq="BCABA", settle=18, accum=1008, d=2.1, lo=0.0, edge=4.0),
        # a ragged block in double, with a twelve-letter sequence
        dict(name="volume_fp64_ragged", kind="volume", nx=101, ny=67, nz=45, precision="fp64",
             rule="none", seq="AABCBBACCABC", settle=100, accum=600, d=2.1, lo=2.0, edge=2.0),
        # the precision volume workload, FP64 near lambda = 0
        dict(name="volume_precision", kind="volume", nx=256, ny=256, nz=256, precision="product",
             rule="margin", seq="ABCABCCA", settle=200, accum=2000, d=2.1, lo=2.5, edge=1.5),
        # the same under the rule that meets both accuracy bars
        dict(name="volume_strict", kind="volume", nx=256, ny=256, nz=256, precision="product",
             rule="strict", seq="ABCABCCA", settle=200, accum=2000, d=2.1, lo=2.5, edge=1.5),
        # one frame of the viewer: default scene and the reference's method
        # (per-step log, refinement walk, jitter, near step), iterations and
        # depth turned down as one does while moving about
        dict(name="frame_viewer", kind="frame", method="walk", w=320, h=200, precision="plain",
             margin=0.0, seq="BCABA", settle=18, accum=120, depth=256.0),
        # the benchmark's frame
        dict(name="frame_512", kind="frame", method="bisect", w=512, h=512, precision="product",
             margin=0.0, seq="AABAB", settle=100, accum=300, depth=500.0),
        # 64 mixed views in one launch, the batched workload: the largest pass
        dict(name="batch_64", kind="batch", views=64, blocks=0, edge=0, accum_lo=200,
             accum_hi=2000, precision="product"),
        # views and volume blocks in one launch sequence
        dict(name="mixed_8_4", kind="batch", views=8, blocks=4, edge=96, accum_lo=200,
             accum_hi=2000, precision="product"),
        # a burst of requests through the serving loop, both kinds
        dict(name="serve_burst", kind="serve", requests=24, accum_lo=200, accum_hi=4000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _letters(rng, lo=3, hi=12):
    return "".join(rng.choice("ABC") for _ in range(rng.randint(lo, hi)))


def draw(rng):
    kind = rng.choice(["points", "volume", "volume", "volume", "frame", "frame", "frame", "batch", "batch",
                       "serve"])
    if kind in ("points", "volume"):
        precision = rng.choice(["plain", "product", "product", "product", "fp64"])
        rule = rng.choice(["none", "margin", "strict"]) if precision == "product" else "none"
        lo, edge = rng.choice([(0.0, 4.0), (2.0, 2.0), (2.5, 1.5)])
        c = dict(kind=kind, precision=precision, rule=rule, seq=_letters(rng),
                 settle=rng.choice([18, 100, 200]), accum=_log_int(rng, 200, 2000), d=2.1, lo=lo,
                 edge=edge)
        if kind == "points":
            c["n"] = _log_int(rng, 33, 400000)
        else:
            for k in ("nx", "ny", "nz"):
                c[k] = _log_int(rng, 24, 200)
        return c
    if kind == "frame":
        method = rng.choice(["bisect", "bisect", "walk"])
        precision = rng.choice(["plain", "product", "product", "fp64"])
        margin = rng.choice([0.0, 0.01]) if method == "bisect" and precision == "product" else 0.0
        return dict(kind=kind, method=method, w=_log_int(rng, 64, 1024), h=_log_int(rng, 64, 1024),
                    precision=precision, margin=margin, seq=_letters(rng), settle=rng.choice([18, 100]),
                    accum=_log_int(rng, 120, 1000), depth=256.0 if method == "walk" else 500.0)
    if kind == "batch":
        return dict(kind=kind, views=rng.randint(1, 24), blocks=rng.randint(0, 4),
                    edge=_log_int(rng, 32, 128), accum_lo=200, accum_hi=_log_int(rng, 400, 2000),
                    precision="product")
    return dict(kind=kind, requests=rng.randint(2, 24), accum_lo=200, accum_hi=_log_int(rng, 400, 4000))


# ----------------------------------------------------------------- inputs ----

def _empty(shape, dtype):
    return torch.empty(shape, dtype=dtype, device="cuda")


def _params(case):
    return lyap.make_params(settle=case["settle"], accum=case["accum"], d=case["d"])


def _box(case, rng):
    """The case's cube, moved by up to 0.05 (kept inside [0, 4])."""
    lo, hi = [], []
    for _ in range(3):
        s = float(rng.uniform(0.0, 0.05))
        if case["lo"] > 0.0:
            lo.append(case["lo"] - s)
            hi.append(case["lo"] - s + case["edge"])
        else:
            lo.append(0.0)
            hi.append(case["edge"] - s)
    return tuple(lo), tuple(hi)


def _volume_mode(precision, rule):
    m, tau, band = RULES[rule]
    return lyap.volume_mode(PRECISIONS[precision], fp64_margin=m, converge_tau=tau, converge_band=band)


def _lights(lights, n):
    raw = np.frombuffer(bytearray(bytes(lights)), dtype=np.uint8)[:n * 224].copy()
    return torch.from_numpy(raw).cuda()


def _image(w, h):
    return dict(rgba=_empty((h, w, 4), torch.uint8), points=_empty((h, w, 9), torch.float32),
                depth=_empty((h, w), torch.float32), lam=_empty((h, w), torch.float32),
                evals=_empty((h, w), torch.int32))


def _sphere_camera(rng, w, h):
    """A camera on a sphere of radius 3 to 6 about the centre, looking at it."""
    radius = float(rng.uniform(3.0, 6.0))
    d = rng.normal(size=3)
    d = d / np.linalg.norm(d)
    eye = tuple(float(CENTER[k] + radius * d[k]) for k in range(3))
    return lyap.cam_look_at(eye, CENTER, math.tan(math.radians(22.5)), w, h)


def _march_params(settle, accum, depth):
    return lyap.make_params(settle=settle, accum=accum, stepMethod=1, depth=depth, jitter=0.0,
                            nearMultiplier=1.0, opaqueThreshold=0.0, lMin=2.0, lMax=4.0)


#: Output buffers of a view: name, values per pixel, type.
FULL = (("rgba", 4, torch.uint8), ("points", 9, torch.float32), ("depth", 1, torch.float32),
        ("lam", 1, torch.float32), ("evals", 1, torch.int32))


def _views(rng, shapes, lights, n_lights, full):
    """Seeded views over the given (side, accum, sequence) shapes; their outputs lie one view
    after the other in one buffer per kind of output."""
    pixels = sum(side * side for side, _, _ in shapes)
    buf = {name: _empty((pixels, k), dtype) for name, k, dtype in FULL if full or name in ("rgba", "lam")}
    views, at = [], 0
    for side, accum, seq in shapes:
        ptr = {name: b.data_ptr() + at * b.shape[1] * b.element_size() for name, b in buf.items()}
        views.append(lyap.make_view(_sphere_camera(rng, side, side), _march_params(100, accum, 500.0), seq, side,
                                    side, lights=lights.data_ptr(), num_lights=n_lights, **ptr))
        at += side * side
    return views, buf


def _shapes(n, sides, accum_lo, accum_hi):
    """The views' sides, iterations and sequences: fixed for a case, so its work is its own."""
    rng = np.random.default_rng(4)
    out = []
    for _ in range(n):
        side = int(rng.choice(sides))
        accum = int(rng.integers(accum_lo, accum_hi + 1))
        out.append((side, accum, "".join("ABC"[int(i)] for i in rng.integers(0, 3, int(rng.integers(3, 13))))))
    return out


BATCH_SIDES = (128, 256, 384, 512, 768, 1024)
SERVE_SIDES = (256, 512, 1024)
SERVE_EDGES = (32, 64, 128, 256)


def _requests(case):
    """Kinds and sizes of a burst: seven views in ten, else volume blocks."""
    rng = np.random.default_rng(5)
    out = []
    for i in range(case["requests"]):
        accum = int(rng.integers(case["accum_lo"], case["accum_hi"] + 1))
        seq = "".join("ABC"[int(k)] for k in rng.integers(0, 3, int(rng.integers(3, 13))))
        side, edge = int(rng.choice(SERVE_SIDES)), int(rng.choice(SERVE_EDGES))
        out.append(("view", side, accum, seq) if rng.random() < 0.7 else ("volume", edge, accum, seq))
    return out


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    s = dict(kind=kind, ctx=context(), case=case)
    if kind == "points":
        g = torch.Generator(device="cuda")
        g.manual_seed(int(seed))
        s["xyz"] = torch.rand((case["n"], 3), generator=g, device="cuda") * case["edge"] + case["lo"]
        s["out"] = _empty((case["n"],), torch.float32)
        s["prm"], s["seq"] = _params(case), lyap.convert_sequence(case["seq"])
        s["mode"] = _volume_mode(case["precision"], case["rule"])
    elif kind == "volume":
        s["lo"], s["hi"] = _box(case, rng)
        s["n"] = (case["nx"], case["ny"], case["nz"])
        s["out"] = _empty((case["nz"], case["ny"], case["nx"]), torch.float32)
        s["prm"], s["seq"] = _params(case), lyap.convert_sequence(case["seq"])
        s["mode"] = _volume_mode(case["precision"], case["rule"])
    elif kind == "frame":
        prm, cam, lights, n = lyap.params_init()
        w, h = case["w"], case["h"]
        if case["method"] == "bisect":
            # camera 4 from the box's centre along a seeded quaternion's axis
            q = rng.normal(size=4)
            q = q / np.linalg.norm(q)
            cam.Q.x, cam.Q.y, cam.Q.z, cam.Q.w = (float(v) for v in q)
            fwd = lyap.quat_transform(cam.Q, (0.0, 0.0, 1.0))
            cam.C.x, cam.C.y, cam.C.z = (CENTER[k] - 4.0 * fwd[k] for k in range(3))
            cam.M = math.tan(math.radians(22.5))
            prm = _march_params(case["settle"], case["accum"], case["depth"])
            s["mode"] = lyap.render_mode(refine=lyap.REFINE_BISECT, bisect_steps=8, normal_h=1e-3,
                                         precision=PRECISIONS[case["precision"]],
                                         fp64_margin=case["margin"])
        else:
            # the default scene, the camera panned a little
            prm.settle, prm.accum, prm.depth = case["settle"], case["accum"], case["depth"]
            cam.C.x += float(rng.uniform(-0.05, 0.05))
            cam.C.y += float(rng.uniform(-0.05, 0.05))
            cam.C.z += float(rng.uniform(-0.05, 0.05))
            s["mode"] = lyap.render_mode(precision=PRECISIONS[case["precision"]])
        lyap.cam_recalculate(cam, w, h, 1)
        lyap.lights_recalculate(lights, n)
        s.update(image=_image(w, h), cam=cam, prm=prm, seq=lyap.convert_sequence(case["seq"]),
                 lights=_lights(lights, n), n_lights=n)
    else:
        _, _, lights, n = lyap.params_init()
        lyap.lights_recalculate(lights, n)
        s["lights"] = _lights(lights, n)
        if kind == "batch":
            shapes = _shapes(case["views"], BATCH_SIDES, case["accum_lo"], case["accum_hi"])
            s["views"], s["out"] = _views(rng, shapes, s["lights"], n, True)
            s["blocks"], e = [], case["edge"]
            if case["blocks"]:
                s["out"]["volumes"] = _empty((case["blocks"], e, e, e), torch.float32)
            for k in range(case["blocks"]):
                lo = tuple(float(2.5 + rng.uniform(0.0, 0.75)) for _ in range(3))
                s["blocks"].append(lyap.make_block(lyap.make_params(settle=200, accum=2000), "ABCABCCA", lo,
                                                   tuple(x + 0.75 for x in lo), e,
                                                   s["out"]["volumes"][k].data_ptr()))
            s["mode"] = lyap.render_mode(refine=lyap.REFINE_BISECT, bisect_steps=8, normal_h=1e-3,
                                         precision=PRECISIONS[case["precision"]])
            s["vol_mode"] = _volume_mode("product", "margin")
        else:
            s["server"] = lyap.Server(s["ctx"], lyap.server_config(vol_mode=_volume_mode("product", "margin")))
            asked = _requests(case)
            views, s["out"] = _views(rng, [r[1:] for r in asked if r[0] == "view"], s["lights"], n, False)
            voxels = sum(r[1] ** 3 for r in asked if r[0] == "volume")
            if voxels:
                s["out"]["volumes"] = _empty((voxels,), torch.float32)
            s["requests"], views, at = [], iter(views), 0
            for what, size, accum, seq in asked:
                if what == "view":
                    s["requests"].append(lyap.view_request(next(views)))
                    continue
                edge = float(rng.uniform(0.25, 2.0))
                lo = tuple(float(2.0 + rng.uniform(0.0, 2.0 - edge)) for _ in range(3))
                s["requests"].append(lyap.volume_request(
                    lyap.make_params(settle=100, accum=accum), seq, lo, tuple(x + edge for x in lo), size,
                    s["out"]["volumes"].data_ptr() + 4 * at))
                at += size ** 3
    return s


# -------------------------------------------------------------------- run ----

def run(state):
    ctx, kind = state["ctx"], state["kind"]
    if kind == "points":
        ctx.calc_points(state["out"].data_ptr(), state["xyz"].data_ptr(), state["xyz"].shape[0], state["prm"],
                        state["seq"], state["mode"])
        return state["out"]
    if kind == "volume":
        ctx.calc_volume(state["out"].data_ptr(), state["prm"], state["seq"], state["lo"], state["hi"],
                        state["n"], state["mode"])
        return state["out"]
    if kind == "frame":
        im, case = state["image"], state["case"]
        ctx.calc_render(im["rgba"].data_ptr(), im["points"].data_ptr(), state["cam"], state["prm"], state["seq"],
                        state["lights"].data_ptr(), state["n_lights"], case["w"], case["h"],
                        im["depth"].data_ptr(), im["lam"].data_ptr(), im["evals"].data_ptr(), state["mode"])
        return im
    if kind == "batch":
        if state["blocks"]:
            ctx.run_batch(state["views"], state["blocks"], state["mode"], state["vol_mode"])
        else:
            ctx.render_batch(state["views"], state["mode"])
        return state["out"]
    server = state["server"]
    tickets = [server.submit(r) for r in state["requests"]]
    server.drain(60000.0)
    for t in tickets:
        if server.poll(t).status != lyap.OK:
            raise RuntimeError("request %d did not finish" % t)
        server.release(t)
    return state["out"]


# ---------------------------------------------------------- work and exact ----

def _flops(settle, accum):
    """Of one lambda evaluation: x - x*x and the product with r per step; the
    derivative and the accumulation per accumulated step besides."""
    return 3.0 * settle + 6.0 * accum


def work(case):
    kind = case["kind"]
    if kind == "points":
        return {"bytes": 16.0 * case["n"], "flops": case["n"] * _flops(case["settle"], case["accum"])}
    if kind == "volume":
        n = float(case["nx"]) * case["ny"] * case["nz"]
        return {"bytes": 4.0 * n, "flops": n * _flops(case["settle"], case["accum"])}
    if kind == "frame":
        n = float(case["w"]) * case["h"]
        return {"bytes": 52.0 * n, "flops": n * EVALS_PER_PIXEL * _flops(case["settle"], case["accum"])}
    b = f = 0.0
    if kind == "batch":
        for side, accum, _ in _shapes(case["views"], BATCH_SIDES, case["accum_lo"], case["accum_hi"]):
            b += 52.0 * side * side
            f += EVALS_PER_PIXEL * side * side * _flops(100, accum)
        n = float(case["blocks"]) * case["edge"] ** 3
        return {"bytes": b + 4.0 * n, "flops": f + n * _flops(200, 2000)}
    for what, size, accum, _ in _requests(case):
        if what == "view":
            b += 8.0 * size * size
            f += EVALS_PER_PIXEL * size * size * _flops(100, accum)
        else:
            b += 4.0 * size ** 3
            f += float(size) ** 3 * _flops(100, accum)
    return {"bytes": b, "flops": f}


def _lambda64(x, y, z, seq, settle, accum, d):
    """The exponent in double with the reference's operation order; x, y, z are FP32 coordinates."""
    r = {0: x.double(), 1: y.double(), 2: z.double(), 3: torch.full_like(x, d).double()}
    period = [int(k) for k in seq if int(k) >= 0]
    v = torch.full_like(r[0], 0.5)
    for k in range(settle):
        c = r[period[k % len(period)]]
        v = (c * v) * (1.0 - v)
    guard = (v - 0.5).abs() < 1e-8
    s = torch.zeros_like(v)
    prod, left = torch.ones_like(v), 8
    for k in range(settle, settle + accum):
        c = r[period[k % len(period)]]
        v = (c * v) * (1.0 - v)
        prod = prod * (c * (1.0 - 2.0 * v)).abs()
        left -= 1
        if left == 0:
            s, prod, left = s + prod.log(), torch.ones_like(v), 8
    lam = (s + prod.log()) / accum
    lam = torch.where(guard, torch.zeros_like(lam), lam)
    return torch.where(torch.isfinite(lam), lam, torch.full_like(lam, math.nan))


def exact(case, seed):
    """Points and volumes in double; a frame's march, its refinement and its
    colours have no closed value that plain torch gives in seconds."""
    if case["kind"] == "points":
        s = prepare(case, seed)
        x, y, z = (s["xyz"][:, k].contiguous() for k in range(3))
        return _lambda64(x, y, z, s["seq"], case["settle"], case["accum"], case["d"])
    if case["kind"] == "volume":
        lo, hi = _box(case, np.random.default_rng(seed))
        axes = []
        for k, n in enumerate((case["nx"], case["ny"], case["nz"])):
            a, b = np.float32(lo[k]), np.float32(hi[k])
            i = np.arange(n, dtype=np.float32)
            axes.append(torch.from_numpy(a + ((b - a) * i) / np.float32(n)).cuda())
        shape = (case["nz"], case["ny"], case["nx"])
        x = axes[0].view(1, 1, -1).expand(shape).contiguous()
        y = axes[1].view(1, -1, 1).expand(shape).contiguous()
        z = axes[2].view(-1, 1, 1).expand(shape).contiguous()
        return _lambda64(x, y, z, lyap.convert_sequence(case["seq"]), case["settle"], case["accum"], case["d"])
    return None
