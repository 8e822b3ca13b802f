"""BLAS builds at the edges of their kernels, through the C-ABI: record counts around a wave's and a
tile's share of the sort (4 and 16 keys per thread) and the aligned runs of the boxes, equal sort
keys, and blocks that one build leaves to the next (sizes growing and shrinking, two threads, a BLAS
that outlives its context)."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    import gpu_util
    return gpu_util


def capsules(n, seed, same=False):
    """n short LSS records scattered in a box, or all at one place but for their length."""
    rng = np.random.default_rng(seed)
    a = np.zeros((n, 8), np.float32)
    a[:, :3] = rng.uniform(-50.0, 50.0, (1 if same else n, 3))
    a[:, 4:7] = a[:, :3] + (np.array([1.0, 0.5, 0.25], np.float32) if same else rng.uniform(-1.0, 1.0, (n, 3)))
    a[:, 3] = a[:, 7] = rng.uniform(0.02, 0.1, n)
    return a


def rays_at(caps, idx, seed):
    """Rays into the middle of the capsules `idx` from 0.3 units away."""
    rng = np.random.default_rng(seed)
    d = rng.standard_normal((len(idx), 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    r = np.zeros((len(idx), 8), np.float32)
    r[:, :3] = 0.5 * (caps[idx, :3] + caps[idx, 4:7]) - 0.3 * d
    r[:, 3] = 0.0
    r[:, 4:7] = d
    r[:, 7] = 1000.0
    return r


def check(ctx, G, oracle, caps, blas, label):
    import vkhrt_amd as V
    n = len(caps)
    idx = np.unique(np.concatenate([np.arange(min(n, 300)), np.arange(max(0, n - 300), n),
                                    np.linspace(0, n - 1, 400).astype(int)]))
    rays = rays_at(caps, idx, 5)
    tlas = V.TopLevelAccelerationStructure(ctx, [blas])
    S = oracle.Scene()
    S.add(oracle.MODE_LSS, caps)
    ref = S.trace(rays)
    assert (ref["prim"] != 0xFFFFFFFF).mean() > 0.9
    G.compare_hits(G.trace(ctx, tlas, rays), ref, label)
    assert blas.info()["leaf_records"] == n
    tlas.close()


@pytest.mark.parametrize("n", [1, 2, 3, 9, 63, 64, 65, 127, 128, 129, 1023, 1025, 4097, 16383, 520193, 520192, 524289])
def test_counts(gpu_ctx, G, oracle, n):
    import vkhrt_amd as V
    caps = capsules(n, n)
    blas = G.build_blas(gpu_ctx, V.GEOMETRY_LSS, caps)
    check(gpu_ctx, G, oracle, caps, blas, f"{n} records")
    blas.close()


@pytest.mark.parametrize("leaf", [1, 3])
def test_equal_keys(gpu_ctx, G, oracle, leaf):
    """Records with one sort key: the tree splits them by index."""
    import vkhrt_amd as V
    caps = capsules(3000, 7, same=True)
    blas = G.build_blas(gpu_ctx, V.GEOMETRY_LSS, caps, leaf_size=leaf)
    check(gpu_ctx, G, oracle, caps, blas, f"equal keys, leaves of {leaf}")
    blas.close()


@pytest.mark.parametrize("collapse,width,leaf", [(2, 8, 1), (4, 8, 3), (1, 5, 2), (2, 4, 3), (4, 7, 1), (0, 4, 1), (0, 5, 3),
                                                 (0, 7, 2)])
def test_collapse_rules(G, oracle, collapse, width, leaf):
    """The SAH-optimal collapse (costs per round, the slots it records) and the greedy one at the
    widths and leaf sizes that the options allow: every record is in the tree and found."""
    import vkhrt_amd as V
    ctx = V.Context(0)
    ctx.set_option(V.OPTION_BVH_COLLAPSE, collapse)
    ctx.set_option(V.OPTION_BVH_WIDTH, width)
    for n in (1, 2, 9, 129, 4097, 3000):
        caps = capsules(n, n, same=n == 3000)  # 3000: equal sort keys
        blas = G.build_blas(ctx, V.GEOMETRY_LSS, caps, leaf_size=leaf)
        info = blas.info()
        assert info["node_count"] >= -(-n // (width * leaf)) and (n == 1 or info["node_count"] < n)
        check(ctx, G, oracle, caps, blas, f"{n} records, collapse {collapse}, width {width}, leaves of {leaf}")
        blas.close()
    ctx.close()


def test_collapse_rules_give_other_trees(G):
    """The options reach the build: the SAH rule and the width change the tree."""
    import vkhrt_amd as V
    ctx = V.Context(0)
    counts = {}
    for collapse, width in ((0, 8), (4, 8), (0, 4), (4, 4)):
        ctx.set_option(V.OPTION_BVH_COLLAPSE, collapse)
        ctx.set_option(V.OPTION_BVH_WIDTH, width)
        blas = G.build_blas(ctx, V.GEOMETRY_LSS, capsules(20000, 3), leaf_size=3)
        counts[collapse, width] = blas.info()["node_count"]
        blas.close()
    assert len(set(counts.values())) == 4, counts
    ctx.close()


def test_blocks_pass_from_build_to_build(G, oracle):
    """Sizes that grow and shrink, all above the least that the pool keeps (1 MiB: 6000 records of
    scratch, 30000 of records), then more sizes than it holds blocks, so that the oldest go."""
    import vkhrt_amd as V
    ctx = V.Context(0)
    keep = []
    for k, n in enumerate([70000, 72000, 150000, 300, 71000, 140000, 70000] + [30000 * 4 ** i // 3 ** i for i in range(6)]):
        caps = capsules(n, 100 + k)
        blas = G.build_blas(ctx, V.GEOMETRY_LSS, caps)
        keep.append((caps, blas))
        if len(keep) == 3:  # two builds old: its memory goes to later ones
            keep.pop(0)[1].close()
        for c, b in keep:
            check(ctx, G, oracle, c, b, f"build {k}")
    ctx.close()
    for _, b in keep:
        b.close()


def test_device_bytes_counts_the_blocks(G):
    """What a BLAS holds: its nodes with room for a sixteenth more, records and ids; a smaller one that
    takes over the blocks of a destroyed one holds as much."""
    import vkhrt_amd as V
    ctx = V.Context(0)
    held = []
    for n in (200000, 190000):
        blas = G.build_blas(ctx, V.GEOMETRY_LSS, capsules(n, 9))
        info = blas.info()
        held.append(info["device_bytes"])
        assert held[-1] >= n * 36 + info["node_count"] * 85
        blas.close()
    assert held[0] == held[1] < 200000 * (36 + 85)
    ctx.close()


@pytest.mark.parametrize("mode,other", [("relaxed", False), ("relaxed", True), ("thread_local", True)])
def test_destroyed_during_a_capture(G, mode, other):
    """A BLAS that is destroyed while a graph is recorded, by this thread or another, leaves the capture
    whole: every replay gives the eager records, with builds in the freed memory in between."""
    import torch
    import vkhrt_amd as V
    ctx = V.Context(0)
    caps = capsules(70000, 21)
    tlas = V.TopLevelAccelerationStructure(ctx, [G.build_blas(ctx, V.GEOMETRY_LSS, caps)])
    extra = G.build_blas(ctx, V.GEOMETRY_LSS, caps[::-1])
    rays = G.dev(rays_at(caps, np.arange(5000), 6))
    hits = torch.zeros(5000 * 8, dtype=torch.float32, device="cuda")

    def trace():
        ctx.trace_rays(tlas, rays.data_ptr(), 5000, hits.data_ptr(), 0, G.stream_ptr())

    trace()
    torch.cuda.synchronize()
    ref = hits.cpu().numpy().tobytes()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode=mode):
        trace()
        if other:
            t = threading.Thread(target=extra.close)
            t.start()
            t.join()
        else:
            extra.close()
    for k in range(3):
        hits.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert hits.cpu().numpy().tobytes() == ref
        G.build_blas(ctx, V.GEOMETRY_LSS, capsules(70000, 30 + k)).close()
    ctx.close()


def test_destroying_a_blas_waits_for_the_device(G):
    """A BLAS's memory goes to the next build only when the GPU is done with it: its destruction waits
    for work on any stream (here a copy loop of some 20 ms on a stream of its own)."""
    import time
    import torch
    import vkhrt_amd as V
    ctx = V.Context(0)
    blas = G.build_blas(ctx, V.GEOMETRY_LSS, capsules(70000, 22))
    a = torch.zeros(1 << 28, dtype=torch.float32, device="cuda")
    stream = torch.cuda.Stream()
    done = torch.cuda.Event()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for _ in range(40):
            a.add_(1.0)
        done.record()
    assert not done.query()
    t0 = time.perf_counter()
    blas.close()
    waited = time.perf_counter() - t0
    assert done.query() and waited > 1e-3
    ctx.close()


def test_builds_in_two_threads(G, oracle):
    import torch
    import vkhrt_amd as V
    ctx = V.Context(0)
    # scratch of 12 to 17 MB, records of 2 to 3 MB and nodes of 1 MB or more: all blocks are pooled
    sets = [[capsules(70000 + 9000 * i, 10 * t + i) for i in range(4)] for t in range(2)]
    dev = [[G.dev(c) for c in s] for s in sets]
    streams = [torch.cuda.Stream() for _ in sets]
    torch.cuda.synchronize()
    built = [[], []]

    def work(t):
        for c, d in zip(sets[t], dev[t]):
            old = V.BottomLevelAccelerationStructure(ctx, V.GEOMETRY_LSS, d.data_ptr(), c.shape[0],
                                                     stream=streams[t].cuda_stream)
            old.close()
            built[t].append(V.BottomLevelAccelerationStructure(ctx, V.GEOMETRY_LSS, d.data_ptr(), c.shape[0],
                                                               stream=streams[t].cuda_stream))

    threads = [threading.Thread(target=work, args=(t,)) for t in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for t in range(2):
        assert len(built[t]) == 4
        for c, b in zip(sets[t], built[t]):
            check(ctx, G, oracle, c, b, f"thread {t}")
            b.close()
    ctx.close()
