"""Timed cases of the hair ray tracer: what a program that uses the library has it do, through the
Python entry points, from a 64x64 probe of a small groom to a path-traced batch of views.

The hair of every case is a seeded random walk of strands grown outward from the upper half of a
sphere and pulled down (root radius 100, 1.5 units a step, fibre radius 0.04 at the root and 0.01
at the tip), made here with torch; cameras and light samples vary with the seed too.

Kinds of case:
  trace     a buffer of rays against phantom curves (closest hit, FP64 polish, accurate normals)
  frame     one rendered frame: primary rays and shadow rays, RGBA8 image and primitive ids
  rebuild   one frame of a groom that moves: strand vertices -> lines -> curves -> BLAS -> TLAS,
            then camera rays traced through it
  batch     path tracing of many views of several models at once
  gradient  the loss gradient of the shadow-visibility MLP over a set of samples
"""
import math

import torch

import vkhrt_amd as V

SPHERE, STEP, GRAVITY, CURL, R_ROOT, R_TIP = 100.0, 1.5, 0.3, 0.2, 0.04, 0.01
TMIN, TMAX = 0.001, 10000.0
MODES = {"phantom": V.GEOMETRY_PHANTOM_CURVES, "lss": V.GEOMETRY_LSS, "dots": V.GEOMETRY_DOTS}
PIECES = 4  # linear pieces per cubic segment in the LSS and DOTS forms
VIEW_SIZES = ((512, 512), (1024, 576), (1280, 720), (1920, 1080))
TINTS = [(0.9, 0.7, 0.5), (0.6, 0.4, 0.3), (0.8, 0.8, 0.7), (0.5, 0.3, 0.2)]
NEURAL_THRESHOLD = 0.2499

_context = None


def context():
    """The device context such a program creates once."""
    global _context
    if _context is None:
        torch.cuda.init()
        _context = V.Context(0)
    return _context


def stream():
    return torch.cuda.current_stream().cuda_stream


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # picking or probing a groom under the cursor: one small buffer of rays, where the
        # launches and the longest walk are the time
        {"name": "trace_probe", "kind": "trace", "strands": 1000, "segments": 16, "rays": 4096},
        # the small frame: thumbnail or preview of a 1,000-strand groom
        {"name": "frame_small", "kind": "frame", "mode": "phantom", "strands": 1000, "segments": 16, "width": 256,
         "height": 256, "accurate": False, "light": "sun", "samples": 1, "head": False},
        # the headline frame: 100k strands at 1080p, accurate normals
        {"name": "frame_100k", "kind": "frame", "mode": "phantom", "strands": 100000, "segments": 32, "width": 1920,
         "height": 1080, "accurate": True, "light": "sun", "samples": 1, "head": False},
        # the same hair in the two other geometry modes, 12.8M pieces
        {"name": "frame_lss", "kind": "frame", "mode": "lss", "strands": 100000, "segments": 32, "width": 1920,
         "height": 1080, "accurate": False, "light": "sun", "samples": 1, "head": False},
        {"name": "frame_dots", "kind": "frame", "mode": "dots", "strands": 100000, "segments": 32, "width": 1920,
         "height": 1080, "accurate": False, "light": "sun", "samples": 1, "head": False},
        # hair on a triangle-mesh head in one TLAS, as an asset loads
        {"name": "frame_head", "kind": "frame", "mode": "phantom", "strands": 100000, "segments": 32, "width": 1920,
         "height": 1080, "accurate": False, "light": "sun", "samples": 1, "head": True},
        # the largest model, two area-light samples per hit: exact, and with the neural shadows
        {"name": "frame_area", "kind": "frame", "mode": "phantom", "strands": 500000, "segments": 32, "width": 1920,
         "height": 1080, "accurate": False, "light": "area", "samples": 2, "head": False},
        {"name": "frame_neural", "kind": "frame", "mode": "phantom", "strands": 500000, "segments": 32, "width": 1920,
         "height": 1080, "accurate": False, "light": "neural", "samples": 2, "head": False},
        # a moving groom, rebuilt every frame: a small one (launches and waits) and a full one
        {"name": "rebuild_small", "kind": "rebuild", "strands": 1000, "segments": 16, "rays": 4096},
        {"name": "rebuild_100k", "kind": "rebuild", "strands": 100000, "segments": 32, "rays": 262144},
        # reference images of several models from many sides: 16 views, 4 bounces, 9.7M segments
        {"name": "batch_16", "kind": "batch", "strands": 200000, "segments": 32, "views": 16, "bounces": 4},
        # one training step's gradient of the shadow MLP
        {"name": "gradient_64k", "kind": "gradient", "samples": 65536},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["trace", "frame", "frame", "frame", "frame", "rebuild", "rebuild", "batch", "gradient"])
    if kind == "trace":
        return {"kind": kind, "strands": _log(rng, 700, 100000), "segments": rng.randint(8, 32),
                "rays": _log(rng, 1000, 300000)}
    if kind == "rebuild":
        return {"kind": kind, "strands": _log(rng, 700, 100000), "segments": rng.randint(8, 32),
                "rays": _log(rng, 1000, 262144)}
    if kind == "batch":
        return {"kind": kind, "strands": _log(rng, 2000, 150000), "segments": rng.randint(8, 32),
                "views": rng.randint(2, 15), "bounces": rng.randint(0, 4)}
    if kind == "gradient":
        return {"kind": kind, "samples": _log(rng, 1000, 1000000)}
    mode = rng.choice(["phantom", "phantom", "phantom", "lss", "dots"])
    light = rng.choice(["sun", "sun", "area", "neural"]) if mode == "phantom" else rng.choice(["sun", "area"])
    head = light == "sun" and rng.random() < 0.3
    return {"kind": kind, "mode": mode, "strands": _log(rng, 1000, 300000 if mode == "phantom" else 80000),
            "segments": rng.randint(8, 32), "width": _log(rng, 100, 1920), "height": _log(rng, 100, 1080),
            "accurate": mode == "phantom" and rng.random() < 0.5, "light": light,
            "samples": rng.randint(1, 3) if light != "sun" else 1, "head": head}


# ------------------------------------------------------------------ inputs
def _gen(seed, stream_id):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + stream_id)
    return g


def _normalize(v):
    return v * (1.0 / v.norm(dim=1, keepdim=True))


def strand_vertices(strands, segments, seed):
    """(strands, segments + 1, 4): x, y, z, radius of every strand vertex."""
    g = _gen(seed, 1)
    d = _normalize(torch.randn(strands, 3, generator=g, device="cuda"))
    d[:, 1].abs_()
    p = d * SPHERE
    out = torch.empty(strands, segments + 1, 4, device="cuda")
    pull = torch.tensor([0.0, -GRAVITY, 0.0], device="cuda")
    for k in range(segments + 1):
        if k:
            d = _normalize(d + pull + (torch.rand(strands, 3, generator=g, device="cuda") * 2.0 - 1.0) * CURL)
            p = p + d * STEP
        out[:, k, :3] = p
        out[:, k, 3] = R_ROOT - (R_ROOT - R_TIP) * (k / segments)
    return out


def bezier_curves(verts):
    """Catmull-Rom through the strand vertices as cubic Bezier segments: (n, 4, 4)."""
    a, b = verts[:, :-1], verts[:, 1:]
    prev = torch.cat([a[:, :1], a[:, :-1]], 1)
    nxt = torch.cat([b[:, 1:], b[:, -1:]], 1)
    return torch.stack([a, a + (b - prev) / 6.0, b - (nxt - a) / 6.0, b], 2).reshape(-1, 4, 4)


def aimed_rays(curves, count, seed):
    """Rays from 5 to 400 units away, aimed into the fibres at random curve points."""
    g = _gen(seed, 2)

    def rand(*s):
        return torch.rand(*s, generator=g, device="cuda", dtype=torch.float64)

    c = curves[(rand(count) * curves.shape[0]).long()].double()
    t = rand(count, 1) * 0.8 + 0.1
    u = 1.0 - t
    w = torch.stack([u ** 3, 3 * u * u * t, 3 * u * t * t, t ** 3], 1)
    p = (c * w).sum(1)
    tan = _normalize(c[:, 3, :3] - c[:, 0, :3])
    d = torch.randn(count, 3, generator=g, device="cuda", dtype=torch.float64)
    d = _normalize(d - 0.7 * (d * tan).sum(1, keepdim=True) * tan)
    aim = p[:, :3] + (rand(count, 3) - 0.5) * 0.6 * p[:, 3:4]
    rays = torch.empty(count, 8, device="cuda")
    rays[:, 4:7] = _normalize(d.float())
    rays[:, :3] = aim - rays[:, 4:7].double() * (5.0 + 395.0 * rand(count, 1))
    rays[:, 3] = TMIN
    rays[:, 7] = TMAX
    return rays


def camera(seed, width, height, k=0, of=1, cx=0.0):
    """A view of the hair from around it; `of` views stand in a ring."""
    a = 2.0 * math.pi * ((seed * 0.6180339887) % 1.0 + k / of)
    eye = (cx + 300.0 * math.sin(a), 60.0 + 25.0 * math.sin(3.0 * a), 300.0 * math.cos(a))
    return V.camera_look_at(eye, (cx, 40.0, 0.0), fov_deg=60.0, aspect=width / height)


def build(curves, mode="phantom", transform=None, material=0):
    """BLAS of the curves in one geometry mode."""
    ctx, sp, n = context(), stream(), curves.shape[0]
    prims, flags = curves, V.BLAS_PER_POINT_RADIUS
    if mode != "phantom":
        lines = torch.empty(n * PIECES, 8, device="cuda")
        ctx.curves_to_lines(curves.data_ptr(), n, PIECES, lines.data_ptr(), stream=sp)
        prims, n = lines, n * PIECES
        if mode == "lss":
            prims = torch.empty(n, 8, device="cuda")
            ctx.generate_lss(lines.data_ptr(), n, prims.data_ptr(), stream=sp)
    return V.BottomLevelAccelerationStructure(ctx, MODES[mode], prims.data_ptr(), n, flags=flags, transform=transform,
                                              material_index=material, stream=sp)


def head_mesh(rows=96, columns=192, radius=99.0):
    """A sphere of triangles under the hair: 8 floats a vertex, u32 triples."""
    i, j = torch.meshgrid(torch.arange(rows + 1, device="cuda"), torch.arange(columns + 1, device="cuda"), indexing="ij")
    th, ph = math.pi * i.double() / rows, 2.0 * math.pi * j.double() / columns
    n = torch.stack([th.sin() * ph.cos(), th.cos(), th.sin() * ph.sin()], 2)
    verts = torch.cat([radius * n, n, (j.double() / columns)[..., None], (i.double() / rows)[..., None]], 2).float()
    a = (i[:-1, :-1] * (columns + 1) + j[:-1, :-1]).reshape(-1)
    b = a + columns + 1
    tris = torch.cat([torch.stack([a, b, a + 1], 1), torch.stack([a + 1, b, b + 1], 1)]).int().contiguous()
    return verts.reshape(-1, 8).contiguous(), tris


MLP_SHAPES = ((64, 96), (64,), (64, 64), (64,), (64, 64), (64,), (64, 64), (64,), (64,), (1,))


def mlp_weights(seed):
    """He-uniform weights and small biases, flat in the library's order (CPU, float32)."""
    g = torch.Generator().manual_seed(seed * 7919 + 5)
    parts = []
    for k, s in enumerate(MLP_SHAPES):
        lim = math.sqrt(6.0 / s[1]) if len(s) == 2 else (math.sqrt(6.0 / 64) if k == 8 else 0.05)
        parts.append(((torch.rand(s, generator=g) * 2.0 - 1.0) * lim).reshape(-1))
    return torch.cat(parts)


BOX_MIN, BOX_MAX = (-160.0, -20.0, -160.0), (160.0, 170.0, 160.0)


def mlp(seed):
    net = V.ShadowMLP(context(), BOX_MIN, BOX_MAX, seed=1)
    net.set_params(mlp_weights(seed).tolist())
    return net


def mlp_samples(count, seed):
    """Points around the hair, directions toward a light above, and whether they are lit."""
    g = _gen(seed, 4)
    p = _normalize(torch.randn(count, 3, generator=g, device="cuda"))
    p[:, 1].abs_()
    p = p * (SPHERE + 45.0 * torch.rand(count, 1, generator=g, device="cuda"))
    light = (torch.rand(count, 3, generator=g, device="cuda") * 2.0 - 1.0) * 100.0
    light[:, 1] = 260.0
    smp = torch.zeros(count, 8, device="cuda")
    smp[:, :3] = p
    smp[:, 4:7] = _normalize(light - p)
    lit = (p.norm(dim=1) / 145.0) ** 4 > torch.rand(count, generator=g, device="cuda")
    return smp, lit.float()


def prepare(case, seed):
    ctx, kind = context(), case["kind"]
    st = {"case": case, "ctx": ctx, "stream": stream()}
    if kind == "gradient":
        st["smp"], st["lit"] = mlp_samples(case["samples"], seed)
        st["mlp"] = mlp(seed)
        st["grad"] = torch.empty(V.SHADOW_MLP_PARAMS, device="cuda")
        return st
    if kind == "batch":
        models = [max(1, int(case["strands"] * f)) for f in (0.02, 0.1, 0.4, 1.0)]
        blases = []
        for k, ns in enumerate(models):
            curves = bezier_curves(strand_vertices(ns, case["segments"], seed * 4 + k))
            xf = [1.0, 0.0, 0.0, 500.0 * k - 750.0, 0.0, 1.0, 0.0, 0.0, 0.0, 0.0, 1.0, 0.0]
            blases.append(build(curves, transform=xf, material=k))
        st["tlas"] = V.TopLevelAccelerationStructure(ctx, blases, stream=st["stream"])
        st["images"], st["views"] = [], []
        for v in range(case["views"]):
            w, h = VIEW_SIZES[(v + v // 4) % 4]
            img = torch.empty(h, w, dtype=torch.int32, device="cuda")
            st["images"].append(img)
            st["views"].append((camera(seed, w, h, v, case["views"], 500.0 * (v % 4) - 750.0), w, h, img.data_ptr()))
        st["seed"] = seed
        return st
    verts = strand_vertices(case["strands"], case["segments"], seed)
    curves = bezier_curves(verts)
    n = curves.shape[0]
    if kind in ("trace", "rebuild"):
        count = case["rays"]
        st["rays"], st["hits"] = aimed_rays(curves, count, seed), torch.empty(count, 8, device="cuda")
        st["out"] = {"t": st["hits"][:, 0], "ids": st["hits"].view(torch.int32)[:, 1:3], "u": st["hits"][:, 3],
                     "normal": st["hits"][:, 4:7], "v": st["hits"][:, 7]}
        if kind == "trace":
            st["tlas"] = V.TopLevelAccelerationStructure(ctx, [build(curves)], stream=st["stream"])
        else:
            st["verts"] = verts
            st["lines"], st["curves"] = torch.empty(n, 8, device="cuda"), torch.empty(n, 16, device="cuda")
            st["blas"] = st["tlas"] = None
        return st
    w, h = case["width"], case["height"]
    blases = [build(curves, case["mode"])]
    if case["head"]:
        mv, mi = head_mesh()
        blases.append(V.BottomLevelAccelerationStructure(ctx, V.GEOMETRY_TRIANGLES, mv.data_ptr(), mi.shape[0],
                                                         indices_ptr=mi.data_ptr(), vertex_count=mv.shape[0],
                                                         material_index=1, stream=st["stream"]))
    st["tlas"] = V.TopLevelAccelerationStructure(ctx, blases, stream=st["stream"])
    st["camera"] = camera(seed, w, h)
    st["image"] = torch.empty(h, w, dtype=torch.int32, device="cuda")
    st["ids"] = torch.empty(h, w, dtype=torch.int32, device="cuda")
    st["flags"] = V.RENDER_SHADOWS | V.RENDER_RGBA8
    if case["mode"] == "phantom":
        st["flags"] |= V.RENDER_FP64_POLISH | (V.RENDER_ACCURATE_NORMALS if case["accurate"] else 0)
    st["more"] = {}
    if case["light"] != "sun":
        st["more"]["area_light"] = V.area_light((0.0, 260.0, 0.0), (100.0, 0.0, 0.0), (0.0, 0.0, 100.0),
                                                samples=case["samples"], seed=seed)
    if case["light"] == "neural":
        st["flags"] |= V.RENDER_NEURAL_SHADOWS
        st["more"].update(shadow_mlp=mlp(seed), variance_threshold=NEURAL_THRESHOLD)
    return st


# ------------------------------------------------------------------ one pass
def run(st):
    case, ctx, sp = st["case"], st["ctx"], st["stream"]
    kind = case["kind"]
    if kind == "frame":
        ctx.render(st["tlas"], st["camera"], case["width"], case["height"], st["image"].data_ptr(), flags=st["flags"],
                   prim_ids_ptr=st["ids"].data_ptr(), stream=sp, **st["more"])
        return st["image"], st["ids"]
    if kind == "batch":
        ctx.render_batch(st["tlas"], st["views"], bounces=case["bounces"], seed=st["seed"],
                         environment=(0.25, 0.3, 0.35), flags=V.BATCH_RGBA8 | V.BATCH_FP64_POLISH,
                         material_albedo=TINTS, stream=sp)
        return st["images"]
    if kind == "gradient":
        loss = st["mlp"].gradient(st["smp"].data_ptr(), st["lit"].data_ptr(), case["samples"], st["grad"].data_ptr(),
                                  stream=sp)
        return {"gradient": st["grad"], "loss": loss}
    if kind == "rebuild":
        ns, nseg = case["strands"], case["segments"]
        n = ns * nseg
        ctx.generate_lines(st["verts"].data_ptr(), ns, nseg, st["lines"].data_ptr(), stream=sp)
        ctx.generate_curves(st["lines"].data_ptr(), n, st["curves"].data_ptr(), stream=sp)
        old = st["tlas"], st["blas"]
        st["blas"] = V.BottomLevelAccelerationStructure(ctx, V.GEOMETRY_PHANTOM_CURVES, st["curves"].data_ptr(), n,
                                                        flags=V.BLAS_PER_POINT_RADIUS, stream=sp)
        st["tlas"] = V.TopLevelAccelerationStructure(ctx, [st["blas"]], stream=sp)
        for x in old:
            if x is not None:
                x.close()
    ctx.trace_rays(st["tlas"], st["rays"].data_ptr(), case["rays"], st["hits"].data_ptr(),
                   V.TRACE_FP64_POLISH | V.TRACE_ACCURATE_NORMALS, stream=sp)
    return st["out"]


# ------------------------------------------------------------------ what a pass cannot do without
# Candidates per ray (primitives whose box the ray enters before its hit) and hits per primary ray
# of the 100k-strand frame; operations of one intersection in each mode (phantom: the iteration
# over both ends, 12.5 steps on average).
CANDIDATES, SHADOW_CANDIDATES, HIT_SHARE = 1.2, 3.8, 0.17
INTERSECT_FLOPS = {"phantom": 2003, "lss": 180, "dots": 340}
RECORD_BYTES = {"phantom": 64, "lss": 32, "dots": 64}


def work(case):
    kind = case["kind"]
    if kind == "gradient":
        n = case["samples"]
        return {"bytes": 36.0 * n + 8.0 * V.SHADOW_MLP_PARAMS, "flops": 111000.0 * n}
    if kind == "batch":
        paths = sum(w * h for w, h in (VIEW_SIZES[(v + v // 4) % 4] for v in range(case["views"])))
        # of the paths 18% hit; about three quarters of the hits send the shadow ray and each
        # bounce ray, and a bounce ray hits again about 70% of the time
        hits, rays = 0.18 * paths, 0.0
        for _ in range(case["bounces"] + 1):
            rays += 1.75 * hits
            hits *= 0.7
        cand = CANDIDATES * paths + SHADOW_CANDIDATES * rays
        return {"bytes": 4.0 * paths + 64.0 * cand, "flops": 2003.0 * cand}
    if kind == "frame":
        pix, rec = case["width"] * case["height"], RECORD_BYTES[case["mode"]]
        cand = CANDIDATES * pix
        if case["light"] != "neural":
            cand += SHADOW_CANDIDATES * HIT_SHARE * pix * case["samples"]
        flops = INTERSECT_FLOPS[case["mode"]] * cand
        if case["light"] == "neural":
            flops += 37000.0 * HIT_SHARE * pix * case["samples"]
        return {"bytes": 8.0 * pix + rec * cand, "flops": float(flops)}
    rays = case["rays"]
    w = {"bytes": (64.0 + 64.0 * CANDIDATES) * rays, "flops": 2003.0 * CANDIDATES * rays}
    if kind == "rebuild":
        # vertices in; lines and curves out and in again; records, ids, radii and nodes out
        w["bytes"] += (16.0 + 2 * 32.0 + 2 * 64.0 + 64.0 + 12.0 + 24.0) * case["strands"] * case["segments"]
        w["flops"] += 200.0 * case["strands"] * case["segments"]
    return w


def tolerance(case):
    if case["kind"] == "gradient":
        # FP32 sums of bf16 products in another order, and the bf16 roundings that flip with them
        return {"rel": 3e-5}
    if case["kind"] == "frame" and case["light"] == "neural":
        # the same in the network's forward pass, seen through the 8-bit image
        return {"differ": 2e-4}
    return "exact"  # the hit rules fix every bit: the image bytes, ids and hit records


# ------------------------------------------------------------------ 64-bit results
def _exact_gradient(case, seed):
    smp, lit = mlp_samples(case["samples"], seed)
    parts, at, flat = [], 0, mlp_weights(seed).double().cuda()
    for s in MLP_SHAPES:
        parts.append(flat[at:at + math.prod(s)].reshape(s).requires_grad_())
        at += math.prod(s)
    lo = torch.tensor(BOX_MIN, dtype=torch.float64, device="cuda")
    hi = torch.tensor(BOX_MAX, dtype=torch.float64, device="cuda")
    n, total = smp.shape[0], 0.0
    for k in range(0, n, 1 << 18):
        s = smp[k:k + (1 << 18)].double()
        x = torch.cat([(s[:, :3] - 0.5 * (lo + hi)) * (2.0 / (hi - lo)), s[:, 4:7]], 1)
        a = x[:, :, None] * (math.pi * 2.0 ** torch.arange(8, device="cuda", dtype=torch.float64))
        h = torch.stack([a.sin(), a.cos()], 3).reshape(-1, 96)
        for L in range(4):
            h = torch.relu(h @ parts[2 * L].t() + parts[2 * L + 1])
        z = h @ parts[8] + parts[9]
        y = lit[k:k + (1 << 18)].double()
        loss = torch.nn.functional.binary_cross_entropy_with_logits(z, y, reduction="sum") / n
        loss.backward()
        total += float(loss.detach())
    return {"gradient": torch.cat([p.grad.reshape(-1) for p in parts]), "loss": total}


def exact(case, seed):
    if case["kind"] == "gradient":
        return _exact_gradient(case, seed)
    # Images are bytes. Hit records have no 64-bit counterpart: a ray whose FP32 iteration does not
    # converge on a curve within its eight steps misses it by definition (12% of the aimed rays),
    # and t, u and the normal of the next curve behind are another hit's.
    return None
