"""GPU tests of the neural shadow-visibility MLP (BF16 MFMA kernels) against the oracle
(oracle/oracle_mlp.hpp), and of the neural shadow form of the render against the exact one."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SCENE_MIN = (-150.0, -110.0, -150.0)
SCENE_MAX = (150.0, 190.0, 150.0)


@pytest.fixture(scope="module")
def O():
    import oracle_lib
    return oracle_lib


def _box(O):
    center = np.array([(a + b) / 2 for a, b in zip(SCENE_MIN, SCENE_MAX)], np.float32)
    inv_half = np.array([2.0 / (b - a) for a, b in zip(SCENE_MIN, SCENE_MAX)], np.float32)
    return center, inv_half


def _samples(n, seed):
    rng = np.random.default_rng(seed)
    s = np.zeros((n, 8), np.float32)
    s[:, :3] = rng.uniform(SCENE_MIN, SCENE_MAX, (n, 3))
    d = rng.normal(size=(n, 3))
    s[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    return s


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def test_forward_matches_oracle(gpu_ctx, O):
    import vkhrt_amd as V
    mlp = V.ShadowMLP(gpu_ctx, SCENE_MIN, SCENE_MAX, seed=3)
    P = O.mlp_init(11)
    P[O.MLP_OFF["b1"]:O.MLP_OFF["b1"] + 64] = 0.1
    P[O.MLP_OFF["b5"]] = -0.3
    mlp.set_params(P)
    assert np.array_equal(np.array(mlp.get_params(), np.float32), P)
    smp = _samples(5000, 12)
    ds = _dev(smp)
    out = torch.empty(5000, dtype=torch.float32, device="cuda")
    print("[mlp forward] 5000 samples", flush=True)
    mlp.infer(ds.data_ptr(), 5000, out.data_ptr())
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    center, inv_half = _box(O)
    ref = O.mlp_forward(P, center, inv_half, smp)
    exact = O.mlp_forward(P, center, inv_half, smp, fp64=True)
    err = np.abs(got - ref)
    print(f"forward |gpu - oracle(bf16)| max {err.max():.3g} mean {err.mean():.3g}; "
          f"|gpu - fp64| max {np.abs(got - exact).max():.3g}")
    # Both sides round every activation to bf16 and accumulate in fp32; the MFMA and the oracle
    # sum in different orders, so an activation near a bf16 rounding boundary can round to the
    # neighbouring value (one bf16 ulp, 2^-8 relative). Such flips are rare and bounded: the mean
    # error stays at fp32 rounding level, the largest at a few 1e-4 (measured 2.2e-4, mean 1e-7).
    assert err.max() < 2e-3 and err.mean() < 1e-5
    assert np.abs(got - exact).max() < 0.05


def test_gradient_matches_oracle(gpu_ctx, O):
    import vkhrt_amd as V
    mlp = V.ShadowMLP(gpu_ctx, SCENE_MIN, SCENE_MAX, seed=4)
    P = O.mlp_init(21)
    P[O.MLP_OFF["b1"]:O.MLP_OFF["b1"] + 64] = 0.05
    mlp.set_params(P)
    n = 1000  # not a multiple of 64: exercises the partial chunk
    smp = _samples(n, 22)
    tgt = (np.random.default_rng(23).random(n) < 0.4).astype(np.float32)
    ds, dt = _dev(smp), _dev(tgt)
    grad = torch.zeros(V.SHADOW_MLP_PARAMS, dtype=torch.float32, device="cuda")
    print("[mlp gradient] 1000 samples", flush=True)
    loss = mlp.gradient(ds.data_ptr(), dt.data_ptr(), n, grad.data_ptr())
    torch.cuda.synchronize()
    g = grad.cpu().numpy()
    center, inv_half = _box(O)
    gref, lref = O.mlp_grad(P, center, inv_half, smp, tgt)
    assert abs(loss - lref) < 1e-5 * max(1.0, abs(lref)), (loss, lref)
    rel = np.linalg.norm(g - gref) / np.linalg.norm(gref)
    print(f"gradient relative L2 error vs oracle {rel:.3g}; loss {loss:.6f} vs {lref:.6f}")
    assert rel < 1e-4  # measured 5.9e-6: the same bf16 rounding flips as the forward pass
    for name, size in [("W1", 6144), ("W2", 4096), ("W3", 4096), ("W4", 4096), ("w5", 64)]:
        a = g[O.MLP_OFF[name]:O.MLP_OFF[name] + size]
        b = gref[O.MLP_OFF[name]:O.MLP_OFF[name] + size]
        cos = float(a @ b / (np.linalg.norm(a) * np.linalg.norm(b) + 1e-30))
        assert cos > 0.99999, (name, cos)
    # the same parameters are untouched by a gradient evaluation
    assert np.array_equal(np.array(mlp.get_params(), np.float32), P)


@pytest.mark.parametrize("n", [1, 15, 64, 65, 16385, 20000])
def test_gradient_at_chunk_edges(gpu_ctx, O, n):
    """One sample, part of a wave's 16, a chunk of 64 and one more, one chunk more than 256 blocks
    take in their first pass: the gradient matches the oracle's in every parameter block, biases and
    output layer among them, and a second evaluation gives the same bits."""
    import vkhrt_amd as V
    mlp = V.ShadowMLP(gpu_ctx, SCENE_MIN, SCENE_MAX, seed=4)
    P = O.mlp_init(21)
    P[O.MLP_OFF["b1"]:O.MLP_OFF["b1"] + 64] = 0.05
    mlp.set_params(P)
    smp = _samples(n, 24)
    tgt = (np.random.default_rng(25).random(n) < 0.4).astype(np.float32)
    ds, dt = _dev(smp), _dev(tgt)
    runs = []
    for _ in range(2):
        grad = torch.zeros(V.SHADOW_MLP_PARAMS, dtype=torch.float32, device="cuda")
        loss = mlp.gradient(ds.data_ptr(), dt.data_ptr(), n, grad.data_ptr())
        torch.cuda.synchronize()
        runs.append(grad.cpu().numpy())
    assert runs[0].tobytes() == runs[1].tobytes()
    center, inv_half = _box(O)
    gref, lref = O.mlp_grad(P, center, inv_half, smp, tgt)
    assert abs(loss - lref) < 1e-5 * max(1.0, abs(lref)), (loss, lref)
    # a bf16 rounding that falls the other way moves one of 64 inputs by 2^-8: 5e-4 of a layer's
    # output for a single sample; a few samples of 64 flip (4e-4 of the gradient measured), and over
    # thousands the flips average out
    tol = 2e-3 if n <= 65 else 2e-4
    for name, size in [("W1", 6144), ("b1", 64), ("W2", 4096), ("b2", 64), ("W3", 4096), ("b3", 64), ("W4", 4096),
                       ("b4", 64), ("w5", 64), ("b5", 1)]:
        a, b = (x[O.MLP_OFF[name]:O.MLP_OFF[name] + size] for x in (runs[0], gref))
        rel = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)
        assert rel < tol, (name, rel)


def test_training_learns_a_half_space(gpu_ctx, O):
    """Visibility = [y_normalized > 0.2]: Adam on the device drives the loss down and the
    classifier right on held-out samples."""
    import vkhrt_amd as V
    mlp = V.ShadowMLP(gpu_ctx, SCENE_MIN, SCENE_MAX, seed=5)
    n = 1 << 16
    smp = _samples(n, 31)
    center, inv_half = _box(O)
    y = ((smp[:, 1] - center[1]) * inv_half[1] > 0.2).astype(np.float32)
    ds, dt = _dev(smp), _dev(y)
    print("[mlp train] half space", flush=True)
    l0 = mlp.train(ds.data_ptr(), dt.data_ptr(), n, batch=8192, epochs=1, learning_rate=3e-3)
    l1 = mlp.train(ds.data_ptr(), dt.data_ptr(), n, batch=8192, epochs=15, learning_rate=3e-3)
    hold = _samples(20000, 32)
    yh = ((hold[:, 1] - center[1]) * inv_half[1] > 0.2)
    out = torch.empty(20000, dtype=torch.float32, device="cuda")
    mlp.infer(_dev(hold).data_ptr(), 20000, out.data_ptr())
    torch.cuda.synchronize()
    acc = float(((out.cpu().numpy() > 0.5) == yh).mean())
    print(f"loss after 1 epoch {l0:.4f}, after 16 {l1:.4f}; held-out accuracy {acc:.4f}")
    assert l1 < 0.5 * l0 and l1 < 0.1
    assert acc > 0.97


def _hair_tlas(ctx, nstrands, seed):
    import gpu_util as G
    import oracle_lib as O
    import vkhrt_amd as V
    curves = O.hair_curves(seed, nstrands, 16)
    blas = G.build_blas(ctx, V.GEOMETRY_PHANTOM_CURVES, curves, per_point=True)
    return blas, V.TopLevelAccelerationStructure(ctx, [blas])


def _shadow_samples(ctx, tlas, mlp, eyes, W, H):
    """Training data from the exact tracer: primary hits of each view -> shadow ray toward
    the light -> traced visibility."""
    import vkhrt_amd as V
    samples, targets = [], []
    for eye in eyes:
        cam = V.camera_look_at(eye, (0.0, 40.0, 0.0), aspect=W / H)
        n = W * H
        rays = torch.empty(n * 8, dtype=torch.float32, device="cuda")
        hits = torch.empty(n * 8, dtype=torch.float32, device="cuda")
        ctx.generate_camera_rays(cam, W, H, rays.data_ptr())
        ctx.trace_rays(tlas, rays.data_ptr(), n, hits.data_ptr())
        srays = torch.empty(n * 8, dtype=torch.float32, device="cuda")
        cnt = torch.zeros(1, dtype=torch.int32, device="cuda")
        ctx.generate_shadow_rays(rays.data_ptr(), hits.data_ptr(), n, srays.data_ptr(), cnt.data_ptr())
        torch.cuda.synchronize()
        m = int(cnt.item())
        s = torch.empty(m * 8, dtype=torch.float32, device="cuda")
        t = torch.empty(m, dtype=torch.float32, device="cuda")
        mlp.collect(tlas, srays.data_ptr(), m, s.data_ptr(), t.data_ptr())
        samples.append(s.view(m, 8))
        targets.append(t)
    torch.cuda.synchronize()
    return torch.cat(samples).contiguous(), torch.cat(targets).contiguous()


def test_neural_shadow_render(gpu_ctx):
    """Trained on shadow rays the exact tracer labels from 8 views, the MLP renders a held-out
    view at PSNR >= 40 dB against the exact image while tracing only the uncertain shadow
    rays; an untrained network at the same threshold does worse. Threshold 0 reproduces the
    exact image bit for bit; 0.25 traces no shadow ray."""
    import gpu_util as G
    import vkhrt_amd as V
    ctx = gpu_ctx
    blas, tlas = _hair_tlas(ctx, 20000, 77)
    mlp = V.ShadowMLP(ctx, SCENE_MIN, SCENE_MAX, seed=9)
    untrained = V.ShadowMLP(ctx, SCENE_MIN, SCENE_MAX, seed=9)
    eyes = [(300 * math.sin(a), 60.0 + 80 * math.cos(3 * a), 300 * math.cos(a))
            for a in np.linspace(0, 2 * math.pi, 8, endpoint=False)]
    print("[neural render] collecting", flush=True)
    smp, tgt = _shadow_samples(ctx, tlas, mlp, eyes, 384, 384)
    n = smp.shape[0]
    print(f"[neural render] training on {n} shadow rays ({float(tgt.mean()):.3f} lit)", flush=True)
    loss = mlp.train(smp.data_ptr(), tgt.data_ptr(), n, batch=16384, epochs=30, learning_rate=3e-3)
    W = H = 512
    cam = V.camera_look_at((120.0, 90.0, 330.0), (0.0, 40.0, 0.0), aspect=1.0)  # not a training view
    exact, ids = G.render(ctx, tlas, cam, W, H, V.RENDER_SHADOWS)
    _, queries, traced = ctx.render_stats()

    def neural(net, thr):
        img = torch.zeros(W * H * 4, dtype=torch.float32, device="cuda")
        ctx.render(tlas, cam, W, H, img.data_ptr(), flags=V.RENDER_SHADOWS | V.RENDER_NEURAL_SHADOWS,
                   shadow_mlp=net, variance_threshold=thr, stream=G.stream_ptr())
        torch.cuda.synchronize()
        _, q, tr = ctx.render_stats()
        return img.cpu().numpy().reshape(H, W, 4), q, tr

    same, q0, t0 = neural(mlp, 0.0)
    assert np.array_equal(same, exact) and t0 == q0 == queries
    _, _, tnone = neural(mlp, 0.25)
    assert tnone == 0
    thr = 0.05
    img, q, tr = neural(mlp, thr)
    uimg, _, utr = neural(untrained, thr)
    p_trained = G.psnr(img[..., :3], exact[..., :3])
    p_untrained = G.psnr(uimg[..., :3], exact[..., :3])
    p_all, _, _ = neural(mlp, 0.25)
    p_nofallback = G.psnr(p_all[..., :3], exact[..., :3])
    print(f"train loss {loss:.4f}; shadow queries {q}: traced exactly {tr} ({tr / q:.3f}) trained, "
          f"{utr} untrained; PSNR trained {p_trained:.2f} dB, untrained {p_untrained:.2f} dB, "
          f"trained without fallback {p_nofallback:.2f} dB")
    assert p_trained >= 40.0
    assert tr < q  # the network answers part of the queries
    assert tr < utr or p_trained > p_untrained + 3.0


@pytest.mark.parametrize("area", [False, True], ids=["directional", "area2"])
def test_wave_fallback_equals_persistent_lanes(gpu_ctx, area):
    """The neural form's exact fallback gives the same image whether its queue is walked by lane
    groups (8, 16 or 64 lanes per ray, forced for every queue length here) or by the persistent
    lanes (wave limit 0): bit for bit at every threshold, FP64 polish on. At
    threshold 0 every query takes the fallback, and the image equals the exact frame. An
    untrained network is deterministic and uncertain, so the thresholds split the queries."""
    import gpu_util as G
    import vkhrt_amd as V
    ctx = gpu_ctx
    blas, tlas = _hair_tlas(ctx, 20000, 78)
    mlp = V.ShadowMLP(ctx, SCENE_MIN, SCENE_MAX, seed=12)
    W = H = 384
    cam = V.camera_look_at((120.0, 90.0, 330.0), (0.0, 40.0, 0.0), aspect=1.0)
    light = V.area_light((0.0, 260.0, 0.0), (100.0, 0.0, 0.0), (0.0, 0.0, 100.0), samples=2, seed=3) if area else None
    flags = V.RENDER_SHADOWS | V.RENDER_FP64_POLISH

    def frame(net, thr):
        img = torch.zeros(W * H * 4, dtype=torch.float32, device="cuda")
        f = flags | (V.RENDER_NEURAL_SHADOWS if net is not None else 0)
        ctx.render(tlas, cam, W, H, img.data_ptr(), flags=f, shadow_mlp=net, variance_threshold=thr,
                   area_light=light, stream=G.stream_ptr())
        torch.cuda.synchronize()
        _, q, tr = ctx.render_stats()
        return img.cpu().numpy(), q, tr

    exact, _, _ = frame(None, 0.0)
    partial = False
    try:
        for thr in (0.0, 0.2, 0.24, 0.245, 0.249, 0.2499):
            ctx.set_option(V.OPTION_SHADOW_WAVE_LIMIT, 0)
            b, q, tr = frame(mlp, thr)
            ctx.set_option(V.OPTION_SHADOW_WAVE_LIMIT, 1 << 20)
            for lanes in (8, 16, 64):
                ctx.set_option(V.OPTION_SHADOW_GROUP_LANES, lanes)
                a, q2, tr2 = frame(mlp, thr)
                print(f"[wave fallback] threshold {thr}, {lanes} lanes per ray: {tr2}/{q2} queries traced", flush=True)
                assert (q, tr) == (q2, tr2)
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (thr, lanes)
            if thr == 0.0:
                assert tr == q and np.array_equal(a.view(np.uint32), exact.view(np.uint32))
            partial = partial or 0 < tr < q
    finally:
        ctx.set_option(V.OPTION_SHADOW_WAVE_LIMIT, 65536)
        ctx.set_option(V.OPTION_SHADOW_GROUP_LANES, 16)
    assert partial
    for opt, v in ((V.OPTION_SHADOW_WAVE_LIMIT, -1), (V.OPTION_SHADOW_WAVE_LIMIT, (1 << 20) + 1),
                   (V.OPTION_SHADOW_GROUP_LANES, 4), (V.OPTION_SHADOW_GROUP_LANES, 24)):
        with pytest.raises(V.VkhrtError):
            ctx.set_option(opt, v)
    mlp.close()
    tlas.close()
    blas.close()
