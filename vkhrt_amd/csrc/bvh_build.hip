// GPU builder for the bottom-level structure (replaces the driver-internal build behind
// vkCmdBuildAccelerationStructuresKHR, bottom_level_acceleration_structure.cpp:34-78).
//
// Pipeline (all on one stream, in one scratch block):
//   1. primitive boxes (GenerateAABBs semantics, geometry_processor.cpp:422-436, plus a
//      small conservative pad) and centroid bounds (wave reduction + ordered-int atomics)
//   2. 63-bit Morton codes of box centroids
//   3. stable LSD radix sort of (key, index), 9 bits per pass: counts per tile, row scans,
//      scatter of tiles put in digit order in LDS (wave ballots rank equal digits)
//   4. boxes of the aligned power-of-two runs of the sorted order
//   5. Karras (HPG 2012) binary radix tree, one thread per internal node, each node's box
//      combined from those runs
//   6. top-down collapse to 8-wide nodes, one level per launch, by one of two rules:
//      SAH: level-synchronous rounds compute, for every binary node, the least SAH cost
//      of covering its subtree with at most j child slots (j = 1..width), and each wide node is
//      opened along those choices (Ylitie, Karras, Laine, HPG 2017);
//      greedy (default, fewer node visits per ray on hair): each binary subtree is opened by
//      largest surface area until `width` (<= 8)
//      children, and subtrees with at most `leaf_max` primitives become leaf children.
//      Child slots are ordered per ray octant; child boxes are quantized to 8 bits against
//      power-of-two scales (outward rounding)
//   7. gather primitive records into leaf order
#include <hip/hip_runtime.h>

#include <stddef.h>

#include <algorithm>
#include <string>
#include <type_traits>
#include <vector>

#include "build.hpp"
#include "device_math.hpp"
#include "internal.hpp"

namespace vk {

namespace {

constexpr int kBlock = 256;
constexpr uint32_t kLeafFlag = 0x80000000u;

__device__ __forceinline__ uint32_t f2ord(float f) {
    uint32_t b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float ord2f(uint32_t u) {
    uint32_t b = (u & 0x80000000u) ? (u & 0x7fffffffu) : ~u;
    return __uint_as_float(b);
}

__global__ void k_init_bounds(uint32_t* cb) {
    if (threadIdx.x < 3) {
        cb[threadIdx.x] = 0xFFFFFFFFu;  // min (ordered)
        cb[3 + threadIdx.x] = 0u;       // max (ordered)
    }
}

// Conservative pad added to every primitive box: 1e-4 + 4e-7 * max|coordinate|.
__device__ __forceinline__ float box_pad(float lo[3], float hi[3]) {
    float m = 0.0f;
    for (int k = 0; k < 3; ++k) m = fmaxf(m, fmaxf(fabsf(lo[k]), fabsf(hi[k])));
    return 1e-4f + 4e-7f * m;
}

// Grid-stride over the records (a fixed grid), so the centroid bounds take one set of atomics
// per block: per-wave atomics on the same 6 words serialized large builds.
__global__ __launch_bounds__(kBlock) void k_prim_boxes(const float4* __restrict__ prims, uint32_t n, int mode,
                                                       int radius_mode, float radius, float4* __restrict__ box,
                                                       uint32_t* __restrict__ cbounds) {
    float cmn[3] = {INFINITY, INFINITY, INFINITY}, cmx[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    float c[3] = {0, 0, 0};
    {
        if (mode == kPhantom) {
            float4 p[4];
            for (int k = 0; k < 4; ++k) p[k] = prims[size_t(i) * 4 + k];
            float r = radius;
            if (radius_mode == 1) r = gmax(gmax(p[0].w, p[1].w), gmax(p[2].w, p[3].w));
            const float px[4] = {p[0].x, p[1].x, p[2].x, p[3].x};
            const float py[4] = {p[0].y, p[1].y, p[2].y, p[3].y};
            const float pz[4] = {p[0].z, p[1].z, p[2].z, p[3].z};
            const float* pc[3] = {px, py, pz};
            for (int k = 0; k < 3; ++k) {
                // glm::min(glm::min(start, end), glm::min(cp1, cp2)) - r
                lo[k] = gmin(gmin(pc[k][0], pc[k][3]), gmin(pc[k][1], pc[k][2])) - r;
                hi[k] = gmax(gmax(pc[k][0], pc[k][3]), gmax(pc[k][1], pc[k][2])) + r;
            }
        } else if (mode == kLss) {
            float4 a = prims[size_t(i) * 2], b = prims[size_t(i) * 2 + 1];
            float ra = fabsf(a.w), rb = b.w;
            lo[0] = fminf(a.x - ra, b.x - rb);
            lo[1] = fminf(a.y - ra, b.y - rb);
            lo[2] = fminf(a.z - ra, b.z - rb);
            hi[0] = fmaxf(a.x + ra, b.x + rb);
            hi[1] = fmaxf(a.y + ra, b.y + rb);
            hi[2] = fmaxf(a.z + ra, b.z + rb);
        } else if (mode == kTriangles) {
            for (int v = 0; v < 3; ++v) {
                const float4 q = prims[size_t(i) * 3 + v];
                const float a[3] = {q.x, q.y, q.z};
                for (int k = 0; k < 3; ++k) {
                    lo[k] = fminf(lo[k], a[k]);
                    hi[k] = fmaxf(hi[k], a[k]);
                }
            }
        } else {
            float4 P[4];
            for (int k = 0; k < 4; ++k) P[k] = prims[size_t(i) * 4 + k];
            // the 6 distinct vertices of the two quads: start +- v r0, end +- v r1
            for (int f = 0; f < 2; ++f) {
                float4 v = P[2 + f];
                for (int sgn = -1; sgn <= 1; sgn += 2) {
                    float s0 = float(sgn) * P[0].w, s1 = float(sgn) * P[1].w;
                    float a[3] = {P[0].x + v.x * s0, P[0].y + v.y * s0, P[0].z + v.z * s0};
                    float b[3] = {P[1].x + v.x * s1, P[1].y + v.y * s1, P[1].z + v.z * s1};
                    for (int k = 0; k < 3; ++k) {
                        lo[k] = fminf(lo[k], fminf(a[k], b[k]));
                        hi[k] = fmaxf(hi[k], fmaxf(a[k], b[k]));
                    }
                }
            }
        }
        float pad = box_pad(lo, hi);
        for (int k = 0; k < 3; ++k) {
            lo[k] -= pad;
            hi[k] += pad;
            c[k] = 0.5f * lo[k] + 0.5f * hi[k];
        }
        box[size_t(i) * 2] = make_float4(lo[0], lo[1], lo[2], 0.0f);
        box[size_t(i) * 2 + 1] = make_float4(hi[0], hi[1], hi[2], 0.0f);
    }
    for (int k = 0; k < 3; ++k) {
        cmn[k] = fminf(cmn[k], c[k]);
        cmx[k] = fmaxf(cmx[k], c[k]);
    }
    }
    // centroid bounds: wave reduction, block reduction in LDS, one atomic per block and word
    __shared__ float s_mn[kBlock / 64][3], s_mx[kBlock / 64][3];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int k = 0; k < 3; ++k) {
        float mn = cmn[k], mx = cmx[k];
        for (int off = 32; off > 0; off >>= 1) {
            mn = fminf(mn, __shfl_xor(mn, off));
            mx = fmaxf(mx, __shfl_xor(mx, off));
        }
        if (lane == 0) {
            s_mn[wave][k] = mn;
            s_mx[wave][k] = mx;
        }
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        const int k = threadIdx.x;
        float mn = s_mn[0][k], mx = s_mx[0][k];
        for (int w = 1; w < kBlock / 64; ++w) {
            mn = fminf(mn, s_mn[w][k]);
            mx = fmaxf(mx, s_mx[w][k]);
        }
        if (mn <= mx) {
            atomicMin(&cbounds[k], f2ord(mn));
            atomicMax(&cbounds[3 + k], f2ord(mx));
        }
    }
}

__device__ __forceinline__ uint64_t spread21(uint64_t x) {
    x &= 0x1fffffull;
    x = (x | (x << 32)) & 0x1f00000000ffffull;
    x = (x | (x << 16)) & 0x1f0000ff0000ffull;
    x = (x | (x << 8)) & 0x100f00f00f00f00full;
    x = (x | (x << 4)) & 0x10c30c30c30c30c3ull;
    x = (x | (x << 2)) & 0x1249249249249249ull;
    return x;
}

__global__ void k_morton(const float4* __restrict__ box, uint32_t n, const uint32_t* __restrict__ cbounds,
                         uint64_t* __restrict__ keys, uint32_t* __restrict__ vals) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 a = box[size_t(i) * 2], b = box[size_t(i) * 2 + 1];
    float c[3] = {0.5f * a.x + 0.5f * b.x, 0.5f * a.y + 0.5f * b.y, 0.5f * a.z + 0.5f * b.z};
    uint64_t q[3];
    for (int k = 0; k < 3; ++k) {
        float lo = ord2f(cbounds[k]), hi = ord2f(cbounds[3 + k]);
        float ext = hi - lo;
        float x = ext > 0.0f ? (c[k] - lo) / ext : 0.0f;
        x = fminf(fmaxf(x, 0.0f), 1.0f);
        q[k] = uint64_t(fminf(x * 2097152.0f, 2097151.0f));
    }
    keys[i] = (spread21(q[0]) << 2) | (spread21(q[1]) << 1) | spread21(q[2]);
    vals[i] = i;
}

// ------------------------------------------------------------------ radix sort
// Stable LSD passes of 9 bits over the 63-bit keys, three launches each: digit counts per tile, an
// exclusive scan of each digit's row over the tiles, and the scatter, which scans the 512 digit
// totals itself. A wave ranks its share of a tile alone (its own digit counters, no barriers), the
// tile is put in digit order in LDS, and neighbouring lanes write neighbouring addresses.
// 3.2M keys: 359 us (scatter 36 us a pass, its 77 MB at 2.2 TB/s); 8 passes of 8 bits with a block
// barrier every 256 keys, direct scatter and 5 launches each took 652 us. 16k keys: 85 against 227.
constexpr int kRsBits = 9, kRsDigits = 1 << kRsBits, kRsPasses = 7;
static_assert(kRsBits * kRsPasses >= 63 && kRsDigits == 2 * kBlock, "two digits per thread");

template <int ITEMS>
__global__ __launch_bounds__(kBlock) void k_rs_hist(const uint64_t* __restrict__ keys, uint32_t n, int shift,
                                                    uint32_t* __restrict__ hist, uint32_t ntiles) {
    __shared__ uint32_t h[kRsDigits];
    h[threadIdx.x] = h[threadIdx.x + kBlock] = 0;
    __syncthreads();
    const uint32_t base = blockIdx.x * (kBlock * ITEMS);
    for (int it = 0; it < ITEMS; ++it) {
        const uint32_t idx = base + it * kBlock + threadIdx.x;
        if (idx < n) atomicAdd(&h[uint32_t(keys[idx] >> shift) & (kRsDigits - 1)], 1u);
    }
    __syncthreads();
    for (int d = threadIdx.x; d < kRsDigits; d += kBlock) hist[size_t(d) * ntiles + blockIdx.x] = h[d];
}

// Exclusive prefix sum of one value per thread over the block; `total` gets the sum. Called by all
// threads; `s_wave` is kBlock / 64 words.
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* s_wave, uint32_t& total) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t x = v;
    for (uint32_t k = 1; k < 64u; k <<= 1) {
        const uint32_t y = __shfl_up(x, k);
        if (lane >= k) x += y;
    }
    __syncthreads();
    if (lane == 63u) s_wave[wave] = x;
    __syncthreads();
    uint32_t before = 0;
    total = 0;
    for (uint32_t w = 0; w < kBlock / 64; ++w) {
        const uint32_t t = s_wave[w];
        before += w < wave ? t : 0u;
        total += t;
    }
    return before + x - v;
}

// One block per digit: its counts over the tiles become their exclusive prefix sum, `totals` its sum.
__global__ __launch_bounds__(kBlock) void k_rs_rows(uint32_t* __restrict__ hist, uint32_t ntiles,
                                                    uint32_t* __restrict__ totals) {
    __shared__ uint32_t s_wave[kBlock / 64];
    uint32_t* row = hist + size_t(blockIdx.x) * ntiles;
    uint32_t run = 0;
    for (uint32_t t0 = 0; t0 < ntiles; t0 += kBlock) {
        const uint32_t t = t0 + threadIdx.x;
        uint32_t sum;
        const uint32_t x = block_scan(t < ntiles ? row[t] : 0u, s_wave, sum);
        if (t < ntiles) row[t] = run + x;
        run += sum;
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = run;
}

template <int ITEMS>
__global__ __launch_bounds__(kBlock) void k_rs_scatter(const uint64_t* __restrict__ kin, const uint32_t* __restrict__ vin,
                                                       uint64_t* __restrict__ kout, uint32_t* __restrict__ vout, uint32_t n,
                                                       int shift, const uint32_t* __restrict__ offs,
                                                       const uint32_t* __restrict__ totals, uint32_t ntiles) {
    constexpr uint32_t kTile = kBlock * ITEMS, kWaves = kBlock / 64;
    __shared__ uint64_t s_key[kTile];
    __shared__ uint32_t s_val[kTile];
    __shared__ uint32_t s_cnt[kWaves][kRsDigits];  // per wave: counts, then first local position
    __shared__ uint32_t s_glob[kRsDigits];         // output position of a digit's first key minus its local position
    __shared__ uint32_t s_wave[kWaves];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6;
    const uint64_t lt = (1ull << lane) - 1ull;
    const uint32_t tile = blockIdx.x * kTile, count = min(kTile, n - tile);
    for (uint32_t i = tid; i < kWaves * kRsDigits; i += kBlock) (&s_cnt[0][0])[i] = 0u;
    __syncthreads();
    // rank within the wave: its ITEMS * 64 consecutive keys, 64 at a time
    uint64_t key[ITEMS];
    uint32_t val[ITEMS], rank[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        const uint32_t i = (w * ITEMS + it) * 64u + lane;
        key[it] = i < count ? kin[tile + i] : 0ull;
        val[it] = i < count ? vin[tile + i] : 0u;
    }
    volatile uint32_t* cnt = s_cnt[w];
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        const bool valid = (w * ITEMS + it) * 64u + lane < count;
        const uint32_t digit = uint32_t(key[it] >> shift) & (kRsDigits - 1);
        uint64_t peers = __builtin_amdgcn_ballot_w64(valid);
        for (int b = 0; b < kRsBits; ++b) {
            const bool bit = (digit >> b) & 1u;
            const uint64_t m = __builtin_amdgcn_ballot_w64(bit);
            peers &= bit ? m : ~m;
        }
        const uint32_t before = valid ? cnt[digit] : 0u;
        rank[it] = before + uint32_t(__popcll(peers & lt));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (valid && (peers & lt) == 0ull) cnt[digit] = before + uint32_t(__popcll(peers));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // digits 2 tid and 2 tid + 1: where each starts in the tile and in the output
    {
        uint32_t c[2] = {0, 0}, sum;
        for (uint32_t k = 0; k < kWaves; ++k)
            for (uint32_t h = 0; h < 2; ++h) c[h] += s_cnt[k][2 * tid + h];
        const uint32_t local = block_scan(c[0] + c[1], s_wave, sum);
        const uint32_t t0 = totals[2 * tid], t1 = totals[2 * tid + 1];
        const uint32_t first = block_scan(t0 + t1, s_wave, sum);
        uint32_t at = local;
        for (uint32_t h = 0; h < 2; ++h) {
            const uint32_t d = 2 * tid + h;
            s_glob[d] = (h ? first + t0 : first) + offs[size_t(d) * ntiles + blockIdx.x] - at;
            for (uint32_t k = 0; k < kWaves; ++k) {
                const uint32_t x = s_cnt[k][d];
                s_cnt[k][d] = at;
                at += x;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < ITEMS; ++it)
        if ((w * ITEMS + it) * 64u + lane < count) {
            const uint32_t at = s_cnt[w][uint32_t(key[it] >> shift) & (kRsDigits - 1)] + rank[it];
            s_key[at] = key[it];
            s_val[at] = val[it];
        }
    __syncthreads();
    for (uint32_t i = tid; i < count; i += kBlock) {
        const uint64_t k = s_key[i];
        const uint32_t to = s_glob[uint32_t(k >> shift) & (kRsDigits - 1)] + i;
        kout[to] = k;
        vout[to] = s_val[i];
    }
}

// ------------------------------------------------------------------ boxes of sorted ranges
struct Box {
    float lo[3], hi[3];
};
__device__ __forceinline__ void grow(Box& a, const Box& b) {
    for (int k = 0; k < 3; ++k) {
        a.lo[k] = fminf(a.lo[k], b.lo[k]);
        a.hi[k] = fmaxf(a.hi[k], b.hi[k]);
    }
}

// Boxes of the aligned power-of-two runs of the sorted primitives: entry l of level k is the box of
// the sorted primitives [l << k, (l + 1) << k); runs that reach past the end are left out. Every
// binary node covers a range of the sorted order, so its box follows from at most two entries per
// level, without its children's boxes: no node waits for another and no launch per tree level is
// needed. (min and max do not depend on the order, so the boxes are those of a bottom-up refit.)
// 3.2M curves: 134 us here and 194 us for the tree with its boxes, where the tree and 32 refit
// rounds took 102 + 455 us and a wait for every 8 rounds.
constexpr int kBoxLevels = 32;
struct BoxTree {
    Box* box;
    size_t off[kBoxLevels];  // first entry of each level
};
constexpr int kBoxPass = 7;  // levels made per launch: a wave's 64 lanes hold 2 entries each

__device__ __forceinline__ Box range_box(const BoxTree& T, uint32_t first, uint32_t last) {
    Box r;
    for (int k = 0; k < 3; ++k) {
        r.lo[k] = INFINITY;
        r.hi[k] = -INFINITY;
    }
    uint32_t l = first, e = last + 1;
    for (int k = 0; l < e; ++k) {
        const Box* b = T.box + T.off[k];
        if (l & 1u) grow(r, b[l++]);
        if (e & 1u) grow(r, b[--e]);
        l >>= 1;
        e >>= 1;
    }
    return r;
}

// Levels level + 1 .. level + 7 from level `level`; the first launch (level 0) also gathers level 0,
// the primitive boxes in sorted order.
__global__ __launch_bounds__(kBlock) void k_box_levels(BoxTree T, uint32_t n, int level, const uint32_t* __restrict__ vals,
                                                       const float4* __restrict__ prim_box) {
    const uint32_t count = n >> level;  // entries of the input level
    const uint32_t i = (blockIdx.x * kBlock + threadIdx.x) * 2u;
    Box b[2];
    for (uint32_t h = 0; h < 2; ++h) {
        if (i + h < count) {
            if (level == 0) {
                const uint32_t p = vals[i + h];
                const float4 lo = prim_box[size_t(p) * 2], hi = prim_box[size_t(p) * 2 + 1];
                b[h] = Box{{lo.x, lo.y, lo.z}, {hi.x, hi.y, hi.z}};
                T.box[T.off[0] + i + h] = b[h];
            } else {
                b[h] = T.box[T.off[level] + i + h];
            }
        } else {
            b[h] = Box{{INFINITY, INFINITY, INFINITY}, {-INFINITY, -INFINITY, -INFINITY}};
        }
    }
    grow(b[0], b[1]);
    for (int k = 1; k <= kBoxPass; ++k) {
        const int lv = level + k;
        if (lv >= kBoxLevels || (n >> lv) == 0) break;
        const uint32_t l = i >> k;
        if ((threadIdx.x & ((1u << (k - 1)) - 1u)) == 0u && l < (n >> lv)) T.box[T.off[lv] + l] = b[0];
        if (k == kBoxPass) break;
        Box o;
        for (int c = 0; c < 3; ++c) {
            o.lo[c] = __shfl_xor(b[0].lo[c], 1 << (k - 1));
            o.hi[c] = __shfl_xor(b[0].hi[c], 1 << (k - 1));
        }
        grow(b[0], o);
    }
}

// ------------------------------------------------------------------ Karras LBVH
struct BinNode {
    Box box;
    uint32_t child[2];  // internal index, or kLeafFlag | sorted index
    uint32_t first, count;  // its range of the sorted order
};

__device__ __forceinline__ int delta(const uint64_t* k, int n, int i, int j) {
    if (j < 0 || j >= n) return -1;
    uint64_t a = k[i], b = k[j];
    if (a == b) return 64 + __clz(uint32_t(i ^ j));
    return __clzll(a ^ b);
}

__global__ __launch_bounds__(kBlock) void k_karras(const uint64_t* __restrict__ keys, int n, BoxTree T,
                                                   BinNode* __restrict__ bin) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) > 0 ? 1 : -1;
    int dmin = delta(keys, n, i, i - d);
    int lmax = 2;
    while (delta(keys, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
    int j = i + l * d;
    int dnode = delta(keys, n, i, j);
    int s = 0, t = l;
    do {
        t = (t + 1) >> 1;
        if (delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    int gamma = i + s * d + min(d, 0);
    int lo = min(i, j), hi = max(i, j);
    BinNode b;
    b.child[0] = (lo == gamma) ? (kLeafFlag | uint32_t(gamma)) : uint32_t(gamma);
    b.child[1] = (hi == gamma + 1) ? (kLeafFlag | uint32_t(gamma + 1)) : uint32_t(gamma + 1);
    b.first = uint32_t(lo);
    b.count = uint32_t(hi - lo + 1);
    b.box = range_box(T, uint32_t(lo), uint32_t(hi));
    bin[i] = b;
}

__device__ __forceinline__ float box_area(const float lo[3], const float hi[3]) {
    const float dx = hi[0] - lo[0], dy = hi[1] - lo[1], dz = hi[2] - lo[2];
    return dx * dy + dy * dz + dz * dx;
}

// SAH-optimal collapse (Ylitie, Karras, Laine, "Efficient Incoherent Ray Traversal on GPUs
// Through Compressed Wide BVHs", HPG 2017). Every binary node n gets the least SAH cost C(n, j)
// of covering its subtree with at most j child slots of a wide node (j = 1..width):
//   C(n, 1) = min(as a leaf slot: A(n) cnt(n) c_prim, if cnt(n) <= leaf_max;
//                 as a wide node: A(n) c_node + D(n, width))
//   C(n, j) = min(C(n, j - 1), D(n, j)),   D(n, j) = min over k of C(left, k) + C(right, j - k)
// with A the half surface area of the box; a binary leaf (one primitive) costs A c_prim for any
// j. The choices are recorded, and the top-down pass opens each wide node along them.
struct SahCost {
    float c[8];      // C(n, j), j = 1..width
    uint8_t dec[8];  // dec[0]: 1 leaf slot, 0 wide node; dec[j - 1] (j >= 2): 0 = C(n, j - 1), else the k of D(n, j)
    uint32_t kint;   // the k of D(n, width): slots of the wide node rooted at n from the left child
    uint32_t pad;
};
struct SahParams {
    SahCost* cost;  // null: greedy collapse
    int leaf_max, width;
    float c_node, c_prim;
};

__device__ __forceinline__ void sah_node(const SahParams& sp, int i, const BinNode& b, const Box* leaf_box) {
    const int W = sp.width;
    float cl[8], cr[8], dist[9];
    uint8_t dk[9];
    auto side = [&](uint32_t ref, int j) {
        if (!(ref & kLeafFlag)) return sp.cost[ref].c[j - 1];
        const Box& q = leaf_box[ref & ~kLeafFlag];
        return box_area(q.lo, q.hi) * sp.c_prim;
    };
#pragma unroll
    for (int j = 1; j <= 8; ++j) {
        cl[j - 1] = j <= W ? side(b.child[0], j) : 0.0f;
        cr[j - 1] = j <= W ? side(b.child[1], j) : 0.0f;
    }
    for (int j = 2; j <= W; ++j) {
        float best = INFINITY;
        uint8_t bk = 1;
        for (int k = 1; k < j; ++k) {
            const float v = cl[k - 1] + cr[j - k - 1];
            if (v < best) {
                best = v;
                bk = uint8_t(k);
            }
        }
        dist[j] = best;
        dk[j] = bk;
    }
    const float A = box_area(b.box.lo, b.box.hi);
    const uint32_t cnt = b.count;
    const float c_leaf = cnt <= uint32_t(sp.leaf_max) ? A * float(cnt) * sp.c_prim : INFINITY;
    const float c_int = A * sp.c_node + dist[W];
    SahCost out;
    out.c[0] = fminf(c_leaf, c_int);
    out.dec[0] = c_leaf <= c_int ? 1 : 0;
    for (int j = 2; j <= 8; ++j) {
        if (j <= W && dist[j] < out.c[j - 2]) {
            out.c[j - 1] = dist[j];
            out.dec[j - 1] = dk[j];
        } else {
            out.c[j - 1] = out.c[j - 2];
            out.dec[j - 1] = 0;
        }
    }
    out.kint = dk[W];
    out.pad = 0;
    sp.cost[i] = out;
}

// SAH costs, one round per launch: an internal node whose children were finished in earlier rounds
// (leaves always are) gets its costs and records the round. Rounds = tree height. The kernel
// boundary makes the children's costs visible, so the rounds need no atomics or fences.
__global__ void k_sah_round(int nint, const BinNode* __restrict__ bin, const Box* __restrict__ leaf_box,
                            uint32_t* __restrict__ done, uint32_t round, SahParams sp) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nint || done[i]) return;
    const BinNode b = bin[i];
    for (int k = 0; k < 2; ++k)
        if (!(b.child[k] & kLeafFlag) && (done[b.child[k]] == 0u || done[b.child[k]] >= round)) return;
    sah_node(sp, i, b, leaf_box);
    done[i] = round;
}

// ------------------------------------------------------------------ collapse to 8-wide
__device__ __forceinline__ uint32_t fexp_for(float extent) {
    // smallest power of two s with 255 * s >= extent; returns the biased exponent byte
    float x = extent / 255.0f;
    if (!(x > 0.0f)) return 1u;
    int e;
    frexpf(x, &e);  // x = m * 2^e, m in [0.5, 1)  =>  2^e >= x
    int b = e + 127;
    return uint32_t(max(1, min(254, b)));
}

// Top-down collapse, one tree level per launch. Eight lanes make one wide node: lane e of the group
// holds child e, so the opening, the slot order and the quantization run one child per lane in
// registers. (One thread per node kept the eight boxes in scratch memory and walked them in
// series: 2666 us for the 10 levels of 3.2M curves, 73 us per level even for a few nodes; now 772
// and about 15. Bound by the chain of dependent loads while a node is opened, at one block of 16
// waves per CU: 82 registers, the SAH rule's stack among them.)
// The nodes of a level are consecutive, bounds[level] .. bounds[level + 1], and tasks[w] is the
// binary node that wide node w covers; a block allocates the children and leaf records of its 128
// nodes with one atomic on the packed counter (nodes in the low, records in the high half): atomics
// on one address take about 18 ns each, one after the other, which with 32 nodes per block was the
// time of the large levels. The last working block to finish records where the next level ends.
constexpr uint32_t kCollapseBlock = 1024;
constexpr uint32_t kCollapseNodes = kCollapseBlock / 8;  // wide nodes per block and pass
constexpr uint32_t kMaxWideLevels = 128;         // a binary tree over 64-bit keys and 32-bit ties is at most 96 deep

struct CollapseState {
    unsigned long long alloc;  // wide nodes | leaf records << 32
    uint32_t bounds[kMaxWideLevels + 2];
    uint32_t done[kMaxWideLevels];  // blocks finished per level
};

// Value of a lane in another part of the caller's eight lanes, step 0: its neighbour, 1: the other
// pair of the four, 2: the other four (mirrored: which of the four does not matter once steps 0 and
// 1 have made them equal). Register moves, where a shuffle goes through the LDS.
template <int STEP, class T>
__device__ __forceinline__ T group_other(T v) {
    constexpr int ctrl = STEP == 0 ? 0xB1 : STEP == 1 ? 0x4E : 0x141;  // quad_perm 1,0,3,2; 2,3,0,1; row_half_mirror
    return __builtin_bit_cast(T, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), ctrl, 0xf, 0xf, true));
}
template <class F>
__device__ __forceinline__ void group_steps(F&& f) {
    f(std::integral_constant<int, 0>{});
    f(std::integral_constant<int, 1>{});
    f(std::integral_constant<int, 2>{});
}
__device__ __forceinline__ float group_min8(float v) {
    group_steps([&](auto k) { v = fminf(v, group_other<decltype(k)::value>(v)); });
    return v;
}
__device__ __forceinline__ float group_max8(float v) {
    group_steps([&](auto k) { v = fmaxf(v, group_other<decltype(k)::value>(v)); });
    return v;
}
__device__ __forceinline__ uint32_t group_or8(uint32_t v) {
    group_steps([&](auto k) { v |= group_other<decltype(k)::value>(v); });
    return v;
}

__global__ __launch_bounds__(kCollapseBlock) void k_collapse(uint32_t level, CollapseState* __restrict__ state,
                                                     uint32_t* __restrict__ tasks, uint32_t n, int leaf_max, int width,
                                                     const BinNode* __restrict__ bin, const Box* __restrict__ leaf_box,
                                                     const uint32_t* __restrict__ vals, WideNode* __restrict__ nodes,
                                                     uint32_t* __restrict__ prim_slots, SahParams sp) {
    __shared__ uint32_t s_node[kCollapseNodes * sizeof(WideNode) / 4];
    __shared__ uint32_t s_nint[kCollapseNodes], s_nprim[kCollapseNodes];  // then their offsets
    const uint32_t begin = state->bounds[level], end = min(state->bounds[level + 1], n);
    const uint32_t sub = threadIdx.x & 7u, grp = threadIdx.x >> 3;
    const int lane0 = int(threadIdx.x & 56u);  // first lane of the group
    for (uint32_t base = begin + blockIdx.x * kCollapseNodes; base < end; base += gridDim.x * kCollapseNodes) {
        const uint32_t w = base + grp;
        const bool live = w < end;
        // child `sub`: reference, box, range and (internal) its own children
        uint32_t ref = 0, cnt = 0, first = 0, c0 = 0, c1 = 0;
        Box box{{INFINITY, INFINITY, INFINITY}, {-INFINITY, -INFINITY, -INFINITY}};
        bool is_int = false;
        uint32_t ne = 0;
        auto load = [&](uint32_t r) {
            ref = r;
            if (r & kLeafFlag) {
                cnt = 1;
                first = r & ~kLeafFlag;
                box = leaf_box[first];
            } else {
                const BinNode b = bin[r];
                cnt = b.count;
                first = b.first;
                box = b.box;
                c0 = b.child[0];
                c1 = b.child[1];
            }
        };
        const uint32_t bref = live ? tasks[w] : kLeafFlag;
        const bool single = (bref & kLeafFlag) != 0;  // a tree of one primitive
        if (live && single) {
            if (sub == 0) load(bref);
            ne = 1;
        } else if (live && sp.cost) {
            // the slots recorded by the cost pass: D(root, width) split, each side expanded along
            // its choices (a binary leaf, or one slot, ends the expansion)
            uint2 stk[16];
            int sn = 0;
            const BinNode& b = bin[bref];
            const int k = int(sp.cost[bref].kint);
            stk[sn++] = make_uint2(b.child[1], uint32_t(width - k));
            stk[sn++] = make_uint2(b.child[0], uint32_t(k));
            while (sn > 0 && ne < 8) {
                const uint2 t = stk[--sn];
                const uint32_t m = t.x;
                const int j = int(t.y);
                if ((m & kLeafFlag) || j <= 1) {
                    if (sub == ne) {
                        load(m);
                        is_int = !(m & kLeafFlag) && sp.cost[m].dec[0] == 0;
                    }
                    ++ne;
                    continue;
                }
                const int d = sp.cost[m].dec[j - 1];
                if (d == 0) {
                    stk[sn++] = make_uint2(m, uint32_t(j - 1));
                } else if (sn + 2 <= 16) {
                    stk[sn++] = make_uint2(bin[m].child[1], uint32_t(j - d));
                    stk[sn++] = make_uint2(bin[m].child[0], uint32_t(d));
                }
            }
        } else if (live) {
            if (sub < 2) load(bin[bref].child[sub]);
            ne = 2;
        }
        if (!sp.cost) {
            // greedy: open the child of the largest area (the first of equals) until `width`
            bool more = live && !single && ne < uint32_t(width);
            while (__ballot(more)) {
                float a = -1.0f;
                if (more && sub < ne && !(ref & kLeafFlag) && cnt > uint32_t(leaf_max)) {
                    const float q = box_area(box.lo, box.hi);
                    if (q > a) a = q;  // not a NaN
                }
                uint32_t best = sub;
                group_steps([&](auto k) {
                    const float oa = group_other<decltype(k)::value>(a);
                    const uint32_t ob = group_other<decltype(k)::value>(best);
                    if (oa > a || (oa == a && ob < best)) {
                        a = oa;
                        best = ob;
                    }
                });
                const uint32_t r1 = __shfl(c1, lane0 + int(best));
                more = more && a >= 0.0f;
                if (more) {
                    if (sub == best || sub == ne) load(sub == best ? c0 : r1);
                    more = ++ne < uint32_t(width);
                }
            }
            is_int = live && !single && sub < ne && !(ref & kLeafFlag) && cnt > uint32_t(leaf_max);
        }
        const bool mine = sub < ne;
        // node box, and the child's centre relative to the node's
        Box nb;
        float off[3];
        for (int k = 0; k < 3; ++k) {
            nb.lo[k] = group_min8(box.lo[k]);
            nb.hi[k] = group_max8(box.hi[k]);
            off[k] = (0.5f * box.lo[k] + 0.5f * box.hi[k]) - (0.5f * nb.lo[k] + 0.5f * nb.hi[k]);
        }
        // octant slot assignment: slot s should hold the child met first along direction
        // d_s = ((s&1)?-1:1, (s&2)?-1:1, (s&4)?-1:1), i.e. the lowest dot(centroid offset, d_s);
        // per round the lowest cost of all free children and slots is placed (ties: the first
        // child, its first slot; NaN costs take the first free pair)
        uint32_t slot = 8, used = 0;
        for (int round = 0; round < 8; ++round) {
            float bc = INFINITY;
            uint32_t bs = __ffs(~used) - 1u;
            if (mine && slot == 8u)
                for (uint32_t s = 0; s < 8; ++s) {
                    const float c = ((s & 1) ? -off[0] : off[0]) + ((s & 2) ? -off[1] : off[1]) +
                                    ((s & 4) ? -off[2] : off[2]);
                    if (!((used >> s) & 1u) && c < bc) {
                        bc = c;
                        bs = s;
                    }
                }
            uint32_t be = (mine && slot == 8u ? sub : sub + 8u) | (bs << 8);  // placed children lose every tie
            group_steps([&](auto k) {
                const float oc = group_other<decltype(k)::value>(bc);
                const uint32_t oe = group_other<decltype(k)::value>(be);
                if (oc < bc || (oc == bc && (oe & 255u) < (be & 255u))) {
                    bc = oc;
                    be = oe;
                }
            });
            if ((be & 255u) < 8u) {
                if (sub == (be & 255u)) slot = be >> 8;
                used |= 1u << (be >> 8);
            }
        }
        // quantization frame
        uint32_t ebyte[3];
        float scale[3];
        for (int k = 0; k < 3; ++k) {
            uint32_t eb = fexp_for(nb.hi[k] - nb.lo[k]);
            for (;;) {
                float s = __uint_as_float(eb << 23);
                if (!(nb.lo[k] + 255.0f * s < nb.hi[k]) || eb >= 254) break;
                ++eb;
            }
            ebyte[k] = eb;
            scale[k] = __uint_as_float(eb << 23);
        }
        // children in slot order: internal children ranked, leaf records by their counts (1..3)
        const uint32_t imask = group_or8(mine && is_int ? 1u << slot : 0u);
        const uint32_t counts = group_or8(mine && !is_int ? cnt << (2u * slot) : 0u);
        const uint32_t below = (1u << slot) - 1u;
        uint32_t poff = 0, n_prims = 0;
        for (uint32_t s = 0; s < 8; ++s) {
            const uint32_t c = (counts >> (2u * s)) & 3u;
            n_prims += c;
            poff += s < slot ? c : 0u;
        }
        if (sub == 0) {
            s_nint[grp] = live ? __popc(imask) : 0u;
            s_nprim[grp] = live ? n_prims : 0u;
        }
        for (uint32_t i = threadIdx.x; i < kCollapseNodes * sizeof(WideNode) / 4; i += kCollapseBlock) s_node[i] = 0u;
        __syncthreads();
        if (threadIdx.x < 64u) {  // one wave scans two nodes per lane
            static_assert(kCollapseNodes == 128, "two nodes per lane");
            const uint32_t i = 2u * threadIdx.x;
            const uint32_t a0 = s_nint[i], a1 = s_nint[i + 1], b0 = s_nprim[i], b1 = s_nprim[i + 1];
            uint32_t sa = a0 + a1, sb = b0 + b1;
            for (uint32_t k = 1; k < 64u; k <<= 1) {
                const uint32_t xa = __shfl_up(sa, k), xb = __shfl_up(sb, k);
                if (threadIdx.x >= k) {
                    sa += xa;
                    sb += xb;
                }
            }
            unsigned long long at = 0;
            if (threadIdx.x == 63u) at = atomicAdd(&state->alloc, (static_cast<unsigned long long>(sb) << 32) | sa);
            at = __shfl(at, 63);
            s_nint[i] = uint32_t(at) + sa - a0 - a1;
            s_nint[i + 1] = uint32_t(at) + sa - a1;
            s_nprim[i] = uint32_t(at >> 32) + sb - b0 - b1;
            s_nprim[i + 1] = uint32_t(at >> 32) + sb - b1;
        }
        __syncthreads();
        const uint32_t cbase = s_nint[grp], pbase = s_nprim[grp];
        // capacity guards (a consistent tree never trips them; the host checks the counters)
        const bool fits = cbase + __popc(imask) <= n && pbase + n_prims <= n;
        if (live && mine && fits) {
            uint8_t* q = reinterpret_cast<uint8_t*>(s_node + grp * (sizeof(WideNode) / 4)) + slot;
            for (int k = 0; k < 3; ++k) {
                const float org = nb.lo[k];
                int q0 = int(floorf((box.lo[k] - org) / scale[k]));
                q0 = max(0, min(255, q0));
                while (q0 > 0 && org + float(q0) * scale[k] > box.lo[k]) --q0;
                int q1 = int(ceilf((box.hi[k] - org) / scale[k]));
                q1 = max(0, min(255, q1));
                while (q1 < 255 && org + float(q1) * scale[k] < box.hi[k]) ++q1;
                q[offsetof(WideNode, qlo_x) + 8 * k] = uint8_t(q0);
                q[offsetof(WideNode, qhi_x) + 8 * k] = uint8_t(q1);
            }
            if (is_int) {
                q[offsetof(WideNode, meta)] = 0x80u;
                tasks[cbase + __popc(imask & below)] = ref;
            } else {
                q[offsetof(WideNode, meta)] = uint8_t((cnt << 5) | poff);
                for (uint32_t j = 0; j < cnt; ++j) prim_slots[pbase + poff + j] = vals[first + j];
            }
            if (sub == 0) {
                uint32_t* h = s_node + grp * (sizeof(WideNode) / 4);
                h[0] = __float_as_uint(nb.lo[0]);
                h[1] = __float_as_uint(nb.lo[1]);
                h[2] = __float_as_uint(nb.lo[2]);
                h[3] = ebyte[0] | (ebyte[1] << 8) | (ebyte[2] << 16) | (imask << 24);
                h[4] = cbase;
                h[5] = pbase;
            }
        }
        __syncthreads();
        const uint32_t words = min(kCollapseNodes, end - base) * uint32_t(sizeof(WideNode) / 4);
        uint32_t* dst = reinterpret_cast<uint32_t*>(nodes + base);
        for (uint32_t i = threadIdx.x; i < words; i += kCollapseBlock) dst[i] = s_node[i];
        __syncthreads();
    }
    const uint32_t working = max(1u, min(gridDim.x, (end - begin + kCollapseNodes - 1) / kCollapseNodes));
    if (threadIdx.x == 0 && blockIdx.x < working) {
        __threadfence();
        if (atomicAdd(&state->done[level], 1u) == working - 1)
            state->bounds[level + 2] = uint32_t(atomicAdd(&state->alloc, 0ull));
    }
}

__global__ void k_gather(const float4* __restrict__ in, const uint32_t* __restrict__ slots, uint32_t n, int rec,
                         float4* __restrict__ out) {
    const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= uint64_t(n) * uint32_t(rec)) return;
    const uint32_t s = uint32_t(i / uint32_t(rec)), k = uint32_t(i % uint32_t(rec));
    out[i] = in[size_t(slots[s]) * rec + k];
}

// The curve records in leaf order, four lanes per record (lane k of the four moves control point k),
// with what belongs to each: its early-out cylinder radius (hair_intersection.rint:21-22),
// CurveDistanceToCylinder(curve, SampleCurvePoint(curve, 0.5)) + radius, with the same IEEE
// sequence as the intersector (no contraction), so the per-ray test is unchanged bit for bit, and
// the slot of its primitive. (One pass over the records instead of three: 3.2M curves 117 us
// against 174; bound by the gather's memory traffic.)
__global__ __launch_bounds__(kBlock) void k_leaf_curves(const float4* __restrict__ in, const uint32_t* __restrict__ slots,
                                                        uint32_t n, int radius_mode, float radius,
                                                        float4* __restrict__ out, float* __restrict__ rmax,
                                                        uint32_t* __restrict__ slot_of) {
    const uint64_t i = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    const uint32_t s = uint32_t(i >> 2), k = uint32_t(i) & 3u;
    const bool valid = s < n;
    const uint32_t p = valid ? slots[s] : 0u;
    const float4 q = in[size_t(p) * 4 + k];
    if (valid) out[i] = q;
    // control point j of the four lanes' record, in each of them
    auto point = [&](auto j) {
        constexpr int ctrl = decltype(j)::value * 0x55;
        auto get = [&](float v) {
            return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), ctrl, 0xf, 0xf, true));
        };
        return make_float4(get(q.x), get(q.y), get(q.z), get(q.w));
    };
    const float4 a = point(std::integral_constant<int, 0>{}), b = point(std::integral_constant<int, 1>{}),
                 c = point(std::integral_constant<int, 2>{}), d = point(std::integral_constant<int, 3>{});
    const f3 p0 = f3{a.x, a.y, a.z}, p1 = f3{b.x, b.y, b.z}, p2 = f3{c.x, c.y, c.z}, p3 = f3{d.x, d.y, d.z};
    float rpad = radius;
    if (radius_mode == 1) rpad = gmax(gmax(a.w, b.w), gmax(c.w, d.w));
    // SampleCurvePoint(curve, 0.5)
    const float t = 0.5f, u = 1.0f - t, tt = t * t, uu = u * u, uuu = uu * u, ttt = tt * t;
    const float w1 = 3.0f * uu * t, w2 = 3.0f * u * tt;
    const f3 mid = f3{uuu * p0.x + w1 * p1.x + w2 * p2.x + ttt * p3.x, uuu * p0.y + w1 * p1.y + w2 * p2.y + ttt * p3.y,
                      uuu * p0.z + w1 * p1.z + w2 * p2.z + ttt * p3.z};
    float r = len3(cross3(sub(mid, p0), sub(mid, p3))) / len3(sub(p3, p0));
    r += rpad;
    if (valid && k == 0u) {
        rmax[s] = r;
        if (p < n) slot_of[p] = s;
    }
}

__global__ void k_set_u32(uint32_t* p, uint32_t v, uint32_t n) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_collapse_init(CollapseState* state, uint32_t* tasks, uint32_t root) {
    for (uint32_t i = threadIdx.x; i < kMaxWideLevels; i += blockDim.x) state->done[i] = 0u;
    if (threadIdx.x == 0) {
        state->alloc = 1ull;  // the root
        state->bounds[0] = 0u;
        state->bounds[1] = 1u;
        tasks[0] = root;
    }
}

// Hands out 256-byte aligned parts of one block; with a null base it only adds up their sizes.
struct Carver {
    char* base;
    size_t at = 0;
    template <class T>
    void part(T** p, size_t count) {
        at = (at + 255) & ~size_t(255);
        *p = base ? reinterpret_cast<T*>(base + at) : nullptr;
        at += std::max<size_t>(1, count) * sizeof(T);
    }
};

inline uint32_t blocks(uint64_t n, int b = kBlock) { return uint32_t((n + b - 1) / b); }

}  // namespace

#define VK_TRY(x)                                  \
    do {                                           \
        hipError_t e_ = (x);                       \
        if (e_ != hipSuccess) {                    \
            err = std::string(#x) + ": " + hipGetErrorString(e_); \
            goto fail;                             \
        }                                          \
    } while (0)

hipError_t build_bvh(int mode, const float4* prims_in, uint32_t n, int radius_mode, float radius, int leaf_max,
                     int width, int collapse, MemPool& pool, hipStream_t st, BuiltBvh* out, std::string& err) {
    const int rec = mode == kLss ? 2 : mode == kTriangles ? 3 : 4;
    float4* box = nullptr;
    uint32_t *cb = nullptr, *v0 = nullptr, *v1 = nullptr, *hist = nullptr, *totals = nullptr, *tasks = nullptr, *done = nullptr;
    uint64_t *k0 = nullptr, *k1 = nullptr;
    BoxTree tree{};
    BinNode* bin = nullptr;
    SahParams sp{};
    struct Head {  // read back together: the collapse's state and the root node
        CollapseState state;
        alignas(16) WideNode root;
    };
    Head* head = nullptr;
    WideNode* nodes = nullptr;
    MemPool::Block scratch, records, node_block;
    BuiltBvh built;
    Head fin{};
    hipError_t rc = hipSuccess;
    uint32_t tiles = 0;
    bool small = false;
    size_t boxes = 0;
    *out = BuiltBvh{};
    if (n == 0) return hipSuccess;
    if (leaf_max < 1) leaf_max = 1;
    if (leaf_max > 3) leaf_max = 3;
    if (width < 2) width = 2;
    if (width > 8) width = 8;
    // tiles of 16 keys per thread; of 4 where those would leave more than half of the 256 CUs idle (16k keys:
    // a scatter of 4 tiles took 15 us, of 16 tiles 6)
    small = blocks(n, kBlock * 16) < 128u;
    tiles = blocks(n, kBlock * (small ? 4 : 16));
    for (int k = 0; k < kBoxLevels; ++k) {
        tree.off[k] = boxes;
        boxes += n >> k;
    }

    // One scratch block. The wide nodes (at most n) take the place of the primitive boxes and of the
    // keys' first buffer, which are done with when the collapse starts.
    for (int pass = 0; pass < 2; ++pass) {
        Carver c{static_cast<char*>(scratch.p)};
        c.part(&head, 1);
        c.at = offsetof(Head, root);  // head comes first in the block; the nodes follow its state, from `root` on
        nodes = scratch.p ? &head->root : nullptr;
        {
            Carver early{c.base, c.at};
            early.part(&box, size_t(n) * 2);
            early.part(&k0, n);
            early.part(&v0, n);
            c.at = std::max(early.at, c.at + size_t(n) * sizeof(WideNode));
        }
        c.part(&k1, n);
        c.part(&v1, n);
        c.part(&cb, 6);
        c.part(&hist, size_t(tiles) * kRsDigits);
        c.part(&totals, kRsDigits);
        c.part(&tree.box, boxes);
        c.part(&bin, n);
        c.part(&tasks, n);
        if (collapse > 0 && n >= 2) {
            c.part(&sp.cost, n);
            c.part(&done, n);
        }
        if (pass == 0) VK_TRY(pool.acquire(c.at, &scratch));
    }
    sp.leaf_max = leaf_max;
    sp.width = width;
    sp.c_node = 1.0f;
    sp.c_prim = 0.25f * float(collapse);
    for (int pass = 0; pass < 2; ++pass) {
        Carver c{static_cast<char*>(records.p)};
        c.part(&built.prims, size_t(n) * rec);
        c.part(&built.prim_ids, n);
        if (mode == kPhantom) {
            c.part(&built.aux, n);
            c.part(&built.slot_of, n);
        }
        if (pass == 0) VK_TRY(pool.acquire(c.at, &records));
    }
    VK_TRY(MemPool::make_fence(&built.fence));

    hipLaunchKernelGGL(k_init_bounds, dim3(1), dim3(64), 0, st, cb);
    hipLaunchKernelGGL(k_prim_boxes, dim3(std::min<uint32_t>(blocks(n), 2048u)), dim3(kBlock), 0, st, prims_in, n, mode,
                       radius_mode, radius, box, cb);
    hipLaunchKernelGGL(k_morton, dim3(blocks(n)), dim3(kBlock), 0, st, box, n, cb, k0, v0);
    VK_TRY(hipGetLastError());
    static_assert(kRsPasses % 2 == 1, "the sorted keys end in the second buffer");
    for (int pass = 0; pass < kRsPasses; ++pass) {
        const int shift = pass * kRsBits;
        if (small)
            hipLaunchKernelGGL(k_rs_hist<4>, dim3(tiles), dim3(kBlock), 0, st, k0, n, shift, hist, tiles);
        else
            hipLaunchKernelGGL(k_rs_hist<16>, dim3(tiles), dim3(kBlock), 0, st, k0, n, shift, hist, tiles);
        hipLaunchKernelGGL(k_rs_rows, dim3(kRsDigits), dim3(kBlock), 0, st, hist, tiles, totals);
        if (small)
            hipLaunchKernelGGL(k_rs_scatter<4>, dim3(tiles), dim3(kBlock), 0, st, k0, v0, k1, v1, n, shift, hist, totals,
                               tiles);
        else
            hipLaunchKernelGGL(k_rs_scatter<16>, dim3(tiles), dim3(kBlock), 0, st, k0, v0, k1, v1, n, shift, hist, totals,
                               tiles);
        std::swap(k0, k1);
        std::swap(v0, v1);
    }
    VK_TRY(hipGetLastError());
    for (int lv = 0; lv == 0 || (n >> lv) > 1; lv += kBoxPass)
        hipLaunchKernelGGL(k_box_levels, dim3(blocks(n >> lv, 2 * kBlock)), dim3(kBlock), 0, st, tree, n, lv, v0, box);
    if (n >= 2) hipLaunchKernelGGL(k_karras, dim3(blocks(n - 1)), dim3(kBlock), 0, st, k0, int(n), tree, bin);
    VK_TRY(hipGetLastError());
    if (sp.cost) {
        hipLaunchKernelGGL(k_set_u32, dim3(blocks(n)), dim3(kBlock), 0, st, done, 0u, n);
        // rounds in groups of 8; the root is the last node to finish
        uint32_t root_done = 0;
        for (uint32_t round = 1; !root_done; round += 8) {
            if (round > 8192) {
                err = "BVH cost rounds did not reach the root";
                rc = hipErrorUnknown;
                goto fail;
            }
            for (uint32_t r = round; r < round + 8; ++r)
                hipLaunchKernelGGL(k_sah_round, dim3(blocks(n - 1)), dim3(kBlock), 0, st, int(n - 1), bin, tree.box, done, r,
                                   sp);
            VK_TRY(hipGetLastError());
            VK_TRY(hipMemcpyAsync(&root_done, done, 4, hipMemcpyDeviceToHost, st));
            VK_TRY(hipStreamSynchronize(st));
        }
    }
    hipLaunchKernelGGL(k_collapse_init, dim3(1), dim3(64), 0, st, &head->state, tasks, n >= 2 ? 0u : kLeafFlag);
    {
        // as many levels as an evenly filled tree of this size has and three more, then four at a time; level L has
        // at most 8^L nodes
        uint32_t level = 0, until = 3;
        for (uint64_t m = 1; m < n; m *= 8) ++until;
        while (built.depth == 0) {
            if (until > kMaxWideLevels) {
                err = "BVH collapse did not reach the leaves";
                rc = hipErrorUnknown;
                goto fail;
            }
            for (; level < until; ++level) {
                const uint64_t most = level < 10 ? std::min<uint64_t>(n, 1ull << (3 * level)) : n;
                hipLaunchKernelGGL(k_collapse, dim3(std::min<uint32_t>(blocks(most, kCollapseNodes), 2048u)), dim3(kCollapseBlock),
                                   0, st, level, &head->state, tasks, n, leaf_max, width, bin, tree.box, v0, nodes,
                                   built.prim_ids, sp);
            }
            VK_TRY(hipGetLastError());
            VK_TRY(hipMemcpyAsync(&fin, head, sizeof(fin), hipMemcpyDeviceToHost, st));
            VK_TRY(hipStreamSynchronize(st));
            for (uint32_t l = 1; l <= level && !built.depth; ++l)
                if (fin.state.bounds[l + 1] == fin.state.bounds[l]) built.depth = l;
            until = level + 4;
        }
    }
    built.nnodes = uint32_t(fin.state.alloc);
    built.root = fin.root;
    if (uint32_t(fin.state.alloc >> 32) != n || built.nnodes > n) {
        err = "BVH collapse placed " + std::to_string(uint32_t(fin.state.alloc >> 32)) + " of " + std::to_string(n) +
              " primitives";
        rc = hipErrorUnknown;
        goto fail;
    }
    {
        // a sixteenth more, so that the next frame of a moving groom fits the block too
        const size_t bytes = size_t(built.nnodes) * sizeof(WideNode);
        VK_TRY(pool.acquire(bytes + bytes / 16, &node_block));
        built.nodes = static_cast<WideNode*>(node_block.p);
        VK_TRY(hipMemcpyAsync(built.nodes, nodes, bytes, hipMemcpyDeviceToDevice, st));
    }
    if (mode == kPhantom)
        hipLaunchKernelGGL(k_leaf_curves, dim3(blocks(uint64_t(n) * 4)), dim3(kBlock), 0, st, prims_in, built.prim_ids, n,
                           radius_mode, radius, built.prims, built.aux, built.slot_of);
    else
        hipLaunchKernelGGL(k_gather, dim3(blocks(uint64_t(n) * rec)), dim3(kBlock), 0, st, prims_in, built.prim_ids, n, rec,
                           built.prims);
    VK_TRY(hipGetLastError());
    VK_TRY(hipStreamSynchronize(st));
    pool.release(scratch, true);
    built.mem[0] = records;
    built.mem[1] = node_block;
    *out = built;
    return hipSuccess;
fail:
    if (rc == hipSuccess) rc = hipErrorUnknown;
    (void)hipFree(built.fence);
    pool.release(scratch, false);
    pool.release(records, false);
    pool.release(node_block, false);
    return rc;
}

}  // namespace vk
