"""The persistent lanes' leaf and intersection queues at their edges, through the C-ABI against
the oracle: every geometry mode, leaves of 1 to 3 records (a node test can yield 24), ray counts
around the 64-lane wavefront, equal hits of several instances and rays with a negative tmin."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


@pytest.fixture(scope="module")
def curves():
    import scenes
    return scenes.dense_ball_curves(nstrands=300)


def _add(S, oracle, G, ctx, mode, curves, leaf_size=0, transform=None):
    """One instance of `curves` in a mode: into the oracle scene, and as a BLAS."""
    import scenes
    import vkhrt_amd as V
    if mode == "mesh":
        import torch
        verts, idx = scenes.uv_sphere(11.0, 24, 48)
        S.add_mesh(verts, idx, transform=transform)
        dv, di = G.dev(verts), G.dev(idx)
        b = V.BottomLevelAccelerationStructure(ctx, V.GEOMETRY_TRIANGLES, dv.data_ptr(), idx.shape[0],
                                               indices_ptr=di.data_ptr(), vertex_count=verts.shape[0],
                                               leaf_size=leaf_size, transform=transform, stream=G.stream_ptr())
        torch.cuda.synchronize()
        return b
    if mode.startswith("phantom"):
        point = mode == "phantom"
        S.add(oracle.MODE_PHANTOM, curves, per_point=point, transform=transform)
        return G.build_blas(ctx, V.GEOMETRY_PHANTOM_CURVES, curves, per_point=point, leaf_size=leaf_size,
                            transform=transform)
    lines = scenes.lines_from_curves(curves, 4)
    if mode == "lss":
        prims = oracle.generate_lss(lines)
        S.add(oracle.MODE_LSS, prims, transform=transform)
        return G.build_blas(ctx, V.GEOMETRY_LSS, prims, leaf_size=leaf_size, transform=transform)
    S.add(oracle.MODE_DOTS, lines, per_point=True, transform=transform)
    return G.build_blas(ctx, V.GEOMETRY_DOTS, lines, per_point=True, leaf_size=leaf_size, transform=transform)


@pytest.mark.parametrize("count", [1, 63, 64, 65, 4097])
@pytest.mark.parametrize("modes,leaf", [(("phantom",), 3), (("lss",), 1), (("lss",), 3), (("dots",), 2), (("mesh",), 3),
                                        (("phantom", "mesh"), 2), (("phantom", "phantom const", "lss", "dots", "mesh"), 3)])
def test_lanes_match_oracle(gpu_ctx, G, oracle, curves, modes, leaf, count):
    import scenes
    import vkhrt_amd as V
    S = oracle.Scene()
    tlas = V.TopLevelAccelerationStructure(gpu_ctx, [_add(S, oracle, G, gpu_ctx, m, curves, leaf) for m in modes])
    rays = scenes.targeted_rays(curves, count, seed=31, dist=(1.0, 60.0))
    assert (S.trace(rays)["prim"] != 0xFFFFFFFF).sum() * 4 > count or count < 64
    G.compare_hits(G.trace(gpu_ctx, tlas, rays), S.trace(rays), f"{modes} x {count}")
    g = G.trace(gpu_ctx, tlas, rays, flags=V.TRACE_TERMINATE_ON_FIRST_HIT)
    r = S.trace(rays, flags=oracle.F_ANY_HIT)
    assert np.array_equal(g["prim"] == 0xFFFFFFFF, r["prim"] == 0xFFFFFFFF)
    polish = S.trace(rays, flags=oracle.F_POLISH)
    G.compare_hits(G.trace(gpu_ctx, tlas, rays, flags=V.TRACE_FP64_POLISH), polish, f"{modes} x {count}, polished")


@pytest.mark.parametrize("copies", [2, 17])
@pytest.mark.parametrize("mode", ["phantom", "lss", "dots", "mesh"])
def test_equal_hits_of_instances(gpu_ctx, G, oracle, curves, mode, copies):
    """The same geometry several times over: equal t goes to the lowest instance (up to 16
    instances are staged in LDS, more are not), with another mode's instance among them."""
    import scenes
    import vkhrt_amd as V
    other = "mesh" if mode != "mesh" else "lss"
    far = np.array([1, 0, 0, 40.0, 0, 1, 0, 0, 0, 0, 1, 0], np.float32)
    for extra in (False, True):
        S = oracle.Scene()
        blases = [_add(S, oracle, G, gpu_ctx, other, curves, transform=far)] if extra else []
        blases += [_add(S, oracle, G, gpu_ctx, mode, curves) for _ in range(copies)]
        tlas = V.TopLevelAccelerationStructure(gpu_ctx, blases)
        rays = scenes.targeted_rays(curves, 1500, seed=32, dist=(1.0, 60.0))
        ref = S.trace(rays)
        assert set(np.unique(ref["inst"])) >= {int(extra)}
        G.compare_hits(G.trace(gpu_ctx, tlas, rays), ref, f"{copies} x {mode}")


@pytest.mark.parametrize("mode", ["lss", "dots", "mesh", "phantom"])
def test_negative_tmin(gpu_ctx, G, oracle, curves, mode):
    """Hits behind the origin (t < 0) order like the others: rays from inside the hair whose
    interval starts 40 units behind them."""
    import scenes
    import vkhrt_amd as V
    S = oracle.Scene()
    tlas = V.TopLevelAccelerationStructure(gpu_ctx, [_add(S, oracle, G, gpu_ctx, mode, curves)])
    rays = scenes.targeted_rays(curves, 3000, seed=33, dist=(-25.0, 25.0))
    rays[:, 3] = -40.0
    rays[:, 7] = 30.0
    ref = S.trace(rays)
    if mode != "phantom":  # a phantom hit lies in front of the origin
        assert (ref["t"][ref["prim"] != 0xFFFFFFFF] < 0).sum() > 100
    G.compare_hits(G.trace(gpu_ctx, tlas, rays), ref, f"{mode}, negative tmin")


@pytest.mark.parametrize("more", [-1, 0, 1])
def test_shared_out_and_claimed_rays_agree(gpu_ctx, G, curves, more):
    """As many rays as a grid of one block per CU has lanes, one fewer and one more: shared out
    evenly up to there, claimed from counters beyond; the default grid shares out all three."""
    import scenes
    import torch
    import vkhrt_amd as V
    tlas = V.TopLevelAccelerationStructure(gpu_ctx, [G.build_blas(gpu_ctx, V.GEOMETRY_PHANTOM_CURVES, curves, per_point=True)])
    count = torch.cuda.get_device_properties(0).multi_processor_count * 256 + more
    rays = scenes.targeted_rays(curves, count, seed=37, dist=(1.0, 60.0))
    for flags in (V.TRACE_FP64_POLISH, V.TRACE_TERMINATE_ON_FIRST_HIT):
        ref = G.trace(gpu_ctx, tlas, rays, flags=flags)
        gpu_ctx.set_option(V.OPTION_BLOCKS_PER_CU, 1)
        try:
            got = G.trace(gpu_ctx, tlas, rays, flags=flags)
        finally:
            gpu_ctx.set_option(V.OPTION_BLOCKS_PER_CU, 0)
        if flags == V.TRACE_FP64_POLISH:
            assert got.tobytes() == ref.tobytes()
        else:
            assert np.array_equal(got["prim"] == 0xFFFFFFFF, ref["prim"] == 0xFFFFFFFF)
    tlas.close()


def _mesh(G, ctx, S, verts, idx):
    """A triangle soup as a BLAS and in the oracle scene."""
    import torch
    import vkhrt_amd as V
    v = np.zeros((len(verts), 8), np.float32)
    v[:, :3] = verts
    v[:, 5] = 1.0
    idx = np.ascontiguousarray(idx, np.uint32)
    S.add_mesh(v, idx)
    dv, di = G.dev(v), G.dev(idx)
    b = V.BottomLevelAccelerationStructure(ctx, V.GEOMETRY_TRIANGLES, dv.data_ptr(), idx.shape[0],
                                           indices_ptr=di.data_ptr(), vertex_count=v.shape[0], stream=G.stream_ptr())
    torch.cuda.synchronize()
    return b


@pytest.mark.parametrize("half", [1e3, 1e12, 1e14, 1e15])
def test_axis_parallel_rays_in_wide_scenes(gpu_ctx, G, oracle, half):
    """A ray parallel to an axis takes 1e20 for the reciprocal of its zero direction components; the
    planes of a node 2e15 units wide are then 1e33 or more apart in t, and none of them may overflow
    on the way. Triangles of a 10000th of the scene, each with an axis-parallel ray at its middle (the
    triangle test forms size^2 x distance, which stays below 1e37 so)."""
    import vkhrt_amd as V
    rng = np.random.default_rng(41)
    n = 500
    mid = rng.uniform(-half, half, (n, 1, 3))
    tri = mid + rng.normal(size=(n, 3, 3)) * (half / 10000.0)
    S = oracle.Scene()
    tlas = V.TopLevelAccelerationStructure(gpu_ctx, [_mesh(G, gpu_ctx, S, tri.reshape(-1, 3), np.arange(3 * n).reshape(n, 3))])
    axis, sign = rng.integers(0, 3, n), rng.choice([-1.0, 1.0], n)
    rays = np.zeros((n, 8), np.float32)
    rays[:, :3] = tri.mean(1)
    rays[np.arange(n), axis] -= sign * half / 20.0
    rays[np.arange(n), 4 + axis] = sign
    rays[:, 7] = 3e38
    ref = S.trace(rays)
    assert (ref["prim"] != 0xFFFFFFFF).mean() > 0.9
    for persistent in (1, 0):
        gpu_ctx.set_option(V.OPTION_PERSISTENT, persistent)
        try:
            G.compare_hits(G.trace(gpu_ctx, tlas, rays), ref, f"scene of +-{half:g}")
            got = G.trace(gpu_ctx, tlas, rays, flags=V.TRACE_TERMINATE_ON_FIRST_HIT)
        finally:
            gpu_ctx.set_option(V.OPTION_PERSISTENT, 1)
        assert np.array_equal(got["prim"] == 0xFFFFFFFF, ref["prim"] == 0xFFFFFFFF)


@pytest.mark.parametrize("mode", ["phantom", "lss"])
def test_wide_scenes_take_their_own_route(gpu_ctx, G, oracle, curves, mode):
    """Two records 1e14 units away make the scene wide, and the kernels others; what is near gives the same
    records, statistics, frames (polished, accurate, with an area light) and path-traced images."""
    import scenes
    import torch
    import vkhrt_amd as V
    if mode == "phantom":
        near, m = np.asarray(curves, np.float32).reshape(-1, 16), V.GEOMETRY_PHANTOM_CURVES
        far = np.zeros((2, 4, 4), np.float32)
        far[:, :, 0] = np.array([[1.0], [-1.0]]) * np.linspace(1e14, 1.1e14, 4)
        far[:, :, 3] = 0.02
        far = far.reshape(2, 16)
    else:
        near, m = oracle.generate_lss(scenes.lines_from_curves(curves, 4)).reshape(-1, 8), V.GEOMETRY_LSS
        far = np.array([[1e14, 0, 0, 0.1, 1.1e14, 0, 0, 0.1], [-1e14, 0, 0, 0.1, -1.1e14, 0, 0, 0.1]], np.float32)
    rays = scenes.targeted_rays(curves, 3000, seed=46, dist=(1.0, 60.0))
    W, H = 160, 120
    cam = V.camera_look_at((0.0, 20.0, 45.0), (0.0, 8.0, 0.0), fov_deg=60.0, aspect=W / H)
    light = V.area_light((0.0, 60.0, 0.0), (20.0, 0.0, 0.0), (0.0, 0.0, 20.0), samples=2, seed=3)
    polish = V.RENDER_SHADOWS | V.RENDER_FP64_POLISH
    runs = []
    for records in (near, np.concatenate([near, far])):
        tlas = V.TopLevelAccelerationStructure(gpu_ctx, [G.build_blas(gpu_ctx, m, records, per_point=mode == "phantom")])
        out = [G.trace(gpu_ctx, tlas, rays), G.trace(gpu_ctx, tlas, rays, V.TRACE_FP64_POLISH | V.TRACE_ACCURATE_NORMALS),
               G.trace(gpu_ctx, tlas, rays, V.TRACE_TERMINATE_ON_FIRST_HIT)["prim"] == 0xFFFFFFFF]
        for flags, al in ((polish, None), (polish | V.RENDER_ACCURATE_NORMALS, None), (polish, light)):
            image = torch.zeros(W * H, dtype=torch.int32, device="cuda")
            gpu_ctx.render(tlas, cam, W, H, image.data_ptr(), flags=flags | V.RENDER_RGBA8, area_light=al, stream=G.stream_ptr())
            out.append(image.cpu().numpy())
        image = torch.zeros(W * H, dtype=torch.int32, device="cuda")
        gpu_ctx.render_batch(tlas, [(cam, W, H, image.data_ptr())], bounces=2, seed=5,
                             flags=V.BATCH_RGBA8 | V.BATCH_FP64_POLISH, stream=G.stream_ptr())
        out.append(image.cpu().numpy())
        r, h = G.dev(rays), torch.zeros(len(rays) * 8, device="cuda")
        st = torch.zeros(len(rays) * 2, dtype=torch.int32, device="cuda")
        gpu_ctx.trace_stats(tlas, r.data_ptr(), len(rays), h.data_ptr(), st.data_ptr(), stream=G.stream_ptr())
        out.append(h.cpu().numpy())
        gpu_ctx.synchronize(G.stream_ptr())
        runs.append(out)
    assert (runs[0][0]["prim"] != 0xFFFFFFFF).mean() > 0.25
    for k, (a, b) in enumerate(zip(*runs)):
        assert a.tobytes() == b.tobytes(), k


@pytest.mark.parametrize("length", [1e-12, 1e15, 1e30, 1e36])
def test_directions_of_any_length(gpu_ctx, G, oracle, length):
    """t is in units of the direction's length; the node test keeps its bits down to the least normal
    numbers (t near 1e-35 for a direction of 1e36). (Components below 1e-20 are taken for 1e-20: the
    shortest length here keeps all but 1 in 10^8 of them above.)"""
    import vkhrt_amd as V
    rng = np.random.default_rng(45)
    n = 4000
    tri = rng.uniform(-50.0, 50.0, (n, 1, 3)) + rng.normal(size=(n, 3, 3)) * 0.3
    S = oracle.Scene()
    tlas = V.TopLevelAccelerationStructure(gpu_ctx, [_mesh(G, gpu_ctx, S, tri.reshape(-1, 3), np.arange(3 * n).reshape(n, 3))])
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    rays = np.zeros((n, 8), np.float32)
    rays[:, :3] = tri.mean(1) - d * rng.uniform(0.0, 60.0, (n, 1))
    rays[:, 4:7] = d * length
    rays[:, 7] = 3e38
    ref = S.trace(rays)
    assert (ref["prim"] != 0xFFFFFFFF).mean() > 0.9
    G.compare_hits(G.trace(gpu_ctx, tlas, rays), ref, f"directions of {length:g}")


def test_zero_distances_of_either_sign_are_equal(gpu_ctx, G, oracle):
    """A ray that starts in the plane of two triangles of opposite winding hits one at t = +0 and the
    other at t = -0 (the numerator cancels to +0, the determinants have opposite signs; all numbers
    here are exact): equal distances, so the lower triangle wins, whichever of them it is."""
    import vkhrt_amd as V
    a, b = [[-1, -1, 0], [2, -1, 0], [-1, 2, 0]], [[-1, -1, 0], [-1, 2, 0], [2, -1, 0]]
    rays = np.zeros((4, 8), np.float32)
    rays[:, :2] = [[0.25, 0.125], [0.25, -0.5], [-0.5, 0.25], [0.0625, 0.125]]
    rays[:, 4:7] = [[1.0, 0.5, 0.25], [1.0, 0.5, -0.25], [-1.0, 0.25, 0.5], [0.25, 1.0, -0.5]]
    rays[:, 7] = 10.0
    for tris in ([a, b], [b, a]):
        S = oracle.Scene()
        verts, idx = np.array(tris, np.float32).reshape(-1, 3), np.arange(6).reshape(2, 3)
        one = _mesh(G, gpu_ctx, S, verts, idx)
        ref = S.trace(rays)
        assert (ref["t"] == 0.0).all() and (ref["prim"] == 0).all()
        G.compare_hits(G.trace(gpu_ctx, V.TopLevelAccelerationStructure(gpu_ctx, [one]), rays), ref, "one mesh")
        S = oracle.Scene()
        parts = [_mesh(G, gpu_ctx, S, np.array(t, np.float32), np.arange(3).reshape(1, 3)) for t in tris]
        ref = S.trace(rays)
        assert (ref["t"] == 0.0).all() and (ref["inst"] == 0).all()
        G.compare_hits(G.trace(gpu_ctx, V.TopLevelAccelerationStructure(gpu_ctx, parts), rays), ref, "two instances")


@pytest.mark.parametrize("modes", [("lss",), ("dots",), ("mesh",), ("lss", "lss"), ("phantom", "mesh"),
                                   ("phantom", "lss", "dots")])
def test_any_hit_record_is_the_rays_own(gpu_ctx, G, oracle, curves, modes):
    """The record that an any-hit trace of these modes returns is the first hit of the ray's own walk:
    the same whole and in parts, in any order, and with one thread per ray."""
    import scenes
    import vkhrt_amd as V
    tlas = V.TopLevelAccelerationStructure(gpu_ctx, [_add(oracle.Scene(), oracle, G, gpu_ctx, m, curves) for m in modes])
    rays = scenes.targeted_rays(curves, 300001, seed=43, dist=(1.0, 60.0))
    for flags in (V.TRACE_TERMINATE_ON_FIRST_HIT, V.TRACE_TERMINATE_ON_FIRST_HIT | V.TRACE_FP64_POLISH):
        gpu_ctx.set_option(V.OPTION_PERSISTENT, 0)
        try:
            ref = G.trace(gpu_ctx, tlas, rays, flags=flags)
        finally:
            gpu_ctx.set_option(V.OPTION_PERSISTENT, 1)
        assert (ref["prim"] != 0xFFFFFFFF).mean() > 0.25
        whole = G.trace(gpu_ctx, tlas, rays, flags=flags)
        assert whole.tobytes() == ref.tobytes(), (whole["prim"] != ref["prim"]).sum()
        order = np.random.default_rng(44).permutation(len(rays))
        mixed = np.empty_like(ref)
        mixed[order] = G.trace(gpu_ctx, tlas, rays[order], flags=flags)
        assert mixed.tobytes() == ref.tobytes()
        cut = 4099
        assert G.trace(gpu_ctx, tlas, rays[:cut], flags=flags).tobytes() == ref[:cut].tobytes()


def test_work_counters_tell_leaf_rounds_from_steps():
    """The counting build's tool: records are tested in leaf rounds of at most 64, whose cycles are not
    the steps'. (In a process of its own, which loads the counting library.)"""
    import json
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-m", "vkhrt_amd.workcount", "--frames", "1", "--strands", "3000", "--width", "320",
                        "--height", "240"], cwd=root, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    out = json.loads(r.stdout.strip().splitlines()[-1])
    for kind in ("primary", "shadow"):
        c = out[kind]["per_frame"]
        assert 0 < c["leaf_rounds"] <= c["leaf_tests"] <= 64 * c["leaf_rounds"]
        assert c["node_tests"] <= c["step_lanes"] and c["cycles_leaf"] > 0 and c["cycles_steps"] > 0
        share = out[kind]["cycle_share"]
        assert abs(sum(share.values()) - 1.0) < 1e-3 and share["leaf_rounds"] > 0
        assert c["rounds"] + c["leaf_rounds"] <= c["iterations"]
