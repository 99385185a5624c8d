// LBVH construction on gfx950: centroid bounds -> Morton codes (30 bits, photon trees 32) -> stable
// LSD radix sort (8-bit digits, LDS histograms, wave64 ballot ranking) -> Karras
// (HPG 2012) hierarchy, each node's child boxes looked up in a pyramid over the sorted boxes ->
// 8-wide collapse of the photon trees.
// Replaces the per-iteration OptiX GAS/IAS builds of nolmoonen/gpuupbp
// gpuupbp/renderer/renderer.cpp:201-307 and the scene GAS build of
// gpuupbp/renderer/renderer_init.cpp:31-289.
#include "lbvh.h"

#include <algorithm>

using namespace upbp;

namespace {

constexpr int kSortThreads = 256;
constexpr int kSortItems = 8;
constexpr int kSortTile = kSortThreads * kSortItems;
constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;

__device__ __forceinline__ uint32_t f2ord(float f)
{
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ord2f(uint32_t u)
{
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

__global__ void k_fill_u32(uint32_t* p, uint32_t v, uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// centroid bounds: bounds[0..2] = ordered min, bounds[3..5] = ordered max
// n_dev (when given): the count in device memory, at most n
__device__ __forceinline__ uint32_t dev_count(uint32_t n, const uint32_t* n_dev) { return n_dev ? min(*n_dev, n) : n; }

__global__ void k_centroid_bounds(const float4* lo, const float4* hi, uint32_t cap, const uint32_t* n_dev,
                                  uint32_t* bounds)
{
    __shared__ float smin[3][256], smax[3][256];
    const uint32_t n = dev_count(cap, n_dev);
    const uint32_t t = threadIdx.x;
    float mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (uint32_t i = blockIdx.x * blockDim.x + t; i < n; i += gridDim.x * blockDim.x) {
        const float4 a = lo[i], b = hi[i];
        const float c[3] = {(a.x + b.x) * .5f, (a.y + b.y) * .5f, (a.z + b.z) * .5f};
        for (int k = 0; k < 3; k++) {
            mn[k] = fminf(mn[k], c[k]);
            mx[k] = fmaxf(mx[k], c[k]);
        }
    }
    for (int k = 0; k < 3; k++) {
        smin[k][t] = mn[k];
        smax[k][t] = mx[k];
    }
    __syncthreads();
    for (uint32_t s = blockDim.x / 2; s > 0; s >>= 1) {
        if (t < s)
            for (int k = 0; k < 3; k++) {
                smin[k][t] = fminf(smin[k][t], smin[k][t + s]);
                smax[k][t] = fmaxf(smax[k][t], smax[k][t + s]);
            }
        __syncthreads();
    }
    if (t == 0)
        for (int k = 0; k < 3; k++) {
            atomicMin(&bounds[k], f2ord(smin[k][0]));
            atomicMax(&bounds[3 + k], f2ord(smax[k][0]));
        }
}

__device__ __forceinline__ uint32_t spread10(uint32_t v)
{
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

// one axis of the Morton grid: [0, 1] over the centroids' range [l, h]. With a region of interest
// [c - r, c + r] (r > 0), what lies outside it shares an eighth of the axis at either end, ever
// coarser with the distance, so that a few primitives far away do not take the grid's resolution
// from the region. Beams of a fog that fills all space reach hundreds of scene radii, and a linear
// grid over them puts the scene in a handful of cells, whose primitives keep their list order.
__device__ __forceinline__ float morton_axis(float x, float l, float h, float c, float r)
{
    const float a = r > 0.f ? fmaxf(l, c - r) : l, b = r > 0.f ? fminf(h, c + r) : h;
    if (!(a < b)) return h > l ? (x - l) / (h - l) : 0.5f;
    const float fl = l < a ? 0.125f : 0.f, fh = h > b ? 0.125f : 0.f;
    if (x < a) return fl / (1.f + (a - x) / r);
    if (x > b) return 1.f - fh / (1.f + (x - b) / r);
    return fl + (x - a) / (b - a) * (1.f - fl - fh);
}

// keys: 30 bits, and with a region of interest 32 (a bit more of x and y: four 8-bit sort passes
// either way)
__global__ void k_morton(const float4* lo, const float4* hi, uint32_t cap, const uint32_t* n_dev, const uint32_t* bounds,
                         float4 region, uint32_t* keys, uint32_t* vals)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= dev_count(cap, n_dev)) return;
    const float4 a = lo[i], b = hi[i];
    const float c[3] = {(a.x + b.x) * .5f, (a.y + b.y) * .5f, (a.z + b.z) * .5f};
    const float rc[3] = {region.x, region.y, region.z};
    uint32_t q[3];
    for (int k = 0; k < 3; k++) {
        const float u = morton_axis(c[k], ord2f(bounds[k]), ord2f(bounds[3 + k]), rc[k], region.w);
        q[k] = uint32_t(fminf(fmaxf(u * 2048.f, 0.f), 2047.f));
    }
    const uint32_t key = (spread10(q[0] >> 1) << 2) | (spread10(q[1] >> 1) << 1) | spread10(q[2] >> 1);
    keys[i] = region.w > 0.f ? (key << 2) | ((q[0] & 1u) << 1) | (q[1] & 1u) : key;
    vals[i] = i;
}

// ---- radix sort ----------------------------------------------------------------
__global__ void __launch_bounds__(kSortThreads) k_radix_hist(const uint32_t* keys, uint32_t cap,
                                                             const uint32_t* n_dev, int shift, uint32_t* hist,
                                                             uint32_t nblocks)
{
    __shared__ uint32_t h[256];
    const uint32_t n = dev_count(cap, n_dev);
    h[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t base = blockIdx.x * kSortTile;
    for (int r = 0; r < kSortItems; r++) {
        const uint32_t i = base + r * kSortThreads + threadIdx.x;
        if (i < n) atomicAdd(&h[(keys[i] >> shift) & 0xffu], 1u);
    }
    __syncthreads();
    hist[threadIdx.x * nblocks + blockIdx.x] = h[threadIdx.x];
}

// Stable scatter: element order within a tile is preserved (round r, then thread id).
__global__ void __launch_bounds__(kSortThreads) k_radix_scatter(const uint32_t* keys_in, const uint32_t* vals_in,
                                                                uint32_t* keys_out, uint32_t* vals_out, uint32_t cap,
                                                                const uint32_t* n_dev, int shift,
                                                                const uint32_t* offsets, uint32_t nblocks)
{
    constexpr int kWaves = kSortThreads / 64;
    const uint32_t n = dev_count(cap, n_dev);
    __shared__ uint32_t running[256];
    __shared__ uint32_t wave_hist[kWaves][256];
    const uint32_t t = threadIdx.x;
    const uint32_t lane = t & 63u, wave = t >> 6;
    running[t] = offsets[t * nblocks + blockIdx.x];
    for (int w = 0; w < kWaves; w++) wave_hist[w][t] = 0;
    __syncthreads();
    const uint32_t base = blockIdx.x * kSortTile;
    const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    for (int r = 0; r < kSortItems; r++) {
        const uint32_t i = base + r * kSortThreads + t;
        const bool valid = i < n;
        const uint32_t key = valid ? keys_in[i] : 0u;
        const uint32_t val = valid ? vals_in[i] : 0u;
        const uint32_t d = (key >> shift) & 0xffu;
        uint64_t match = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bb = __ballot(bit);
            match &= bit ? bb : ~bb;
        }
        const uint32_t rank = __popcll(match & lt_mask);
        const bool leader = valid && (match & lt_mask) == 0ull;
        if (leader) wave_hist[wave][d] = __popcll(match);
        __syncthreads();
        if (valid) {
            uint32_t off = running[d] + rank;
            for (uint32_t w = 0; w < wave; w++) off += wave_hist[w][d];
            keys_out[off] = key;
            vals_out[off] = val;
        }
        __syncthreads();
        uint32_t tot = 0;
        for (int w = 0; w < kWaves; w++) {
            tot += wave_hist[w][t];
            wave_hist[w][t] = 0;
        }
        running[t] += tot;
        __syncthreads();
    }
}

// ---- exclusive scan (reduce, scan of block sums, downsweep) ----------------------
__global__ void __launch_bounds__(kScanThreads) k_scan_reduce(const uint32_t* in, uint32_t n, uint32_t* sums)
{
    __shared__ uint32_t s[kScanThreads];
    uint32_t acc = 0;
    const uint32_t base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    for (int k = 0; k < kScanItems; k++)
        if (base + k < n) acc += in[base + k];
    s[threadIdx.x] = acc;
    __syncthreads();
    for (uint32_t st = kScanThreads / 2; st > 0; st >>= 1) {
        if (threadIdx.x < st) s[threadIdx.x] += s[threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0) sums[blockIdx.x] = s[0];
}

// Scans one tile per block; adds block_offsets[blockIdx] if given. Writes the grand total of
// block 0's tile into *total when there is a single block.
__global__ void __launch_bounds__(kScanThreads) k_scan_tile(const uint32_t* in, uint32_t* out, uint32_t n,
                                                            const uint32_t* block_offsets, uint32_t* total)
{
    __shared__ uint32_t s[kScanThreads];
    const uint32_t base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    uint32_t v[kScanItems];
    uint32_t acc = 0;
    for (int k = 0; k < kScanItems; k++) {
        v[k] = base + k < n ? in[base + k] : 0u;
        acc += v[k];
    }
    s[threadIdx.x] = acc;
    __syncthreads();
    // Hillis-Steele inclusive scan over thread sums
    for (uint32_t st = 1; st < kScanThreads; st <<= 1) {
        const uint32_t x = threadIdx.x >= st ? s[threadIdx.x - st] : 0u;
        __syncthreads();
        s[threadIdx.x] += x;
        __syncthreads();
    }
    uint32_t run = (threadIdx.x ? s[threadIdx.x - 1] : 0u) + (block_offsets ? block_offsets[blockIdx.x] : 0u);
    for (int k = 0; k < kScanItems; k++) {
        if (base + k < n) out[base + k] = run;
        run += v[k];
    }
    if (total && gridDim.x == 1 && threadIdx.x == kScanThreads - 1) *total = s[kScanThreads - 1];
}

// ---- Karras hierarchy -----------------------------------------------------------
__device__ __forceinline__ int delta(const uint32_t* keys, int n, int i, int j)
{
    if (j < 0 || j >= n) return -1;
    const uint32_t a = keys[i], b = keys[j];
    if (a == b) return 32 + __clz(uint32_t(i) ^ uint32_t(j));
    return __clz(a ^ b);
}

// Boxes of the sorted primitives (level 0) and of every aligned group of 8, 64, 512, ... of them.
// A tree node covers a range of sorted primitives, so its box is the union of at most 14 entries per
// level, and every node's boxes are found by its own thread in one launch. (A level-by-level refit
// takes two launches for each of up to 64 levels, most of them empty: with the per-level collapse,
// 440 launches per iteration. Photon trees per iteration, before -> with this and the collapse
// below: small box 1.27 -> 0.58 ms, box 1.77 -> 0.93, guided 2.06 -> 1.09, slab room 3.0 -> 2.0,
// predefined fog room 10.2 -> 9.7, blob grid 10.5 -> 10.1; the blob grid's beam tree, 13.3M sub-beams:
// refit 3.4 -> 1.5 ms in one launch and the pyramid's, collapse 3.3 -> 4.6.)
constexpr int kPyrLevels = 12;
constexpr uint32_t kPyrBlock = 512; // three levels per launch
struct Pyramid {
    float4 *lo, *hi;
    uint32_t off[kPyrLevels]; // first entry of a level
    int levels;               // the last has at most 8 entries
};

// reads level `from` (0: from the unsorted boxes, which it also writes) and writes the next three
__global__ void __launch_bounds__(kPyrBlock) k_pyramid(Pyramid P, int from, const float4* lo, const float4* hi,
                                                       const uint32_t* order, uint32_t cap, const uint32_t* n_dev)
{
    __shared__ float4 slo[kPyrBlock / 64], shi[kPyrBlock / 64];
    const uint32_t n = dev_count(cap, n_dev), m = uint32_t((uint64_t(n) + (uint64_t(1) << (3 * from)) - 1) >> (3 * from));
    if (blockIdx.x * kPyrBlock >= m) return;
    const uint32_t i = blockIdx.x * kPyrBlock + threadIdx.x, lane = threadIdx.x & 63u;
    float4 a = make_float4(INFINITY, INFINITY, INFINITY, 0.f), b = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
    if (i < m) {
        if (from == 0) {
            const uint32_t p = order[i];
            a = lo[p]; // with its tag
            b = hi[p];
            P.lo[i] = a;
            P.hi[i] = b;
        } else {
            a = P.lo[P.off[from] + i];
            b = P.hi[P.off[from] + i];
        }
    }
    const auto join = [&](uint32_t step) {
        for (uint32_t o = step; o < 8u * step; o <<= 1) {
            a = make_float4(fminf(a.x, __shfl_xor(a.x, o)), fminf(a.y, __shfl_xor(a.y, o)),
                            fminf(a.z, __shfl_xor(a.z, o)), 0.f);
            b = make_float4(fmaxf(b.x, __shfl_xor(b.x, o)), fmaxf(b.y, __shfl_xor(b.y, o)),
                            fmaxf(b.z, __shfl_xor(b.z, o)), 0.f);
        }
    };
    const auto put = [&](int level, uint32_t at) {
        if (level >= P.levels) return;
        P.lo[P.off[level] + at] = a;
        P.hi[P.off[level] + at] = b;
    };
    join(1);
    if ((lane & 7u) == 0u && i < m) put(from + 1, i >> 3);
    join(8);
    if (lane == 0u) {
        if (i < m) put(from + 2, i >> 6);
        slo[threadIdx.x >> 6] = a;
        shi[threadIdx.x >> 6] = b;
    }
    __syncthreads();
    if (threadIdx.x < 8u) {
        a = slo[threadIdx.x];
        b = shi[threadIdx.x];
        join(1);
        if (threadIdx.x == 0u) put(from + 3, blockIdx.x);
    }
}

// box of the sorted primitives [first, end)
__device__ __forceinline__ void range_box(const Pyramid& P, uint32_t first, uint32_t end, float4& lo, float4& hi)
{
    lo = make_float4(INFINITY, INFINITY, INFINITY, 0.f);
    hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
    const auto add = [&](uint32_t at) {
        const float4 a = P.lo[at], b = P.hi[at];
        lo = make_float4(fminf(lo.x, a.x), fminf(lo.y, a.y), fminf(lo.z, a.z), 0.f);
        hi = make_float4(fmaxf(hi.x, b.x), fmaxf(hi.y, b.y), fmaxf(hi.z, b.z), 0.f);
    };
    for (int l = 0; first < end; l++) {
        const bool top = l + 1 == P.levels;
        while (first < end && (top || (first & 7u))) add(P.off[l] + first++);
        while (first < end && (end & 7u)) add(P.off[l] + --end);
        first >>= 3;
        end >>= 3;
    }
}

// the hierarchy with its boxes; tags: a leaf child's box tag, an inner child's primitive count
__global__ void k_karras(const uint32_t* keys, uint32_t cap, const uint32_t* n_dev, Pyramid P, BNode* nodes)
{
    const int n = int(dev_count(cap, n_dev));
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    const int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    const int dmin = delta(keys, n, i, i - d);
    int lmax = 2;
    while (delta(keys, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
    const int j = i + l * d;
    const int dnode = delta(keys, n, i, j);
    int s = 0;
    int div = 2;
    int t = (l + div - 1) / div;
    for (;;) {
        if (delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
        if (t == 1) break;
        div <<= 1;
        t = (l + div - 1) / div;
    }
    const int g = i + s * d + (d < 0 ? -1 : 0);
    const int lo = i < j ? i : j, hi = i < j ? j : i;
    const auto child = [&](int first, int end, float4& a, float4& b) {
        if (end - first == 1) {
            a = P.lo[first];
            b = P.hi[first];
        } else {
            range_box(P, uint32_t(first), uint32_t(end), a, b);
            a.w = __uint_as_float(uint32_t(end - first));
        }
    };
    float4 a0, b0, a1, b1;
    child(lo, g + 1, a0, b0);
    child(g + 1, hi + 1, a1, b1);
    float4* f = reinterpret_cast<float4*>(&nodes[i]);
    f[0] = make_float4(a0.x, a0.y, a0.z, b0.x);
    f[1] = make_float4(b0.y, b0.z, a1.x, a1.y);
    f[2] = make_float4(a1.z, b1.x, b1.y, b1.z);
    f[3] = make_float4(__int_as_float((lo == g) ? ~g : g), __int_as_float((hi == g + 1) ? ~(g + 1) : g + 1), a0.w, a1.w);
}

// ---- wide collapse ----------------------------------------------------------------
// Each wide node takes one binary node and opens its largest-area inner child until it
// has kWide children (or only leaves). The nodes over many primitives are opened by one block,
// level by level; the subtrees below them, by one wave each.
constexpr uint32_t kTopNodes = 2048; // frontier of the top: disjoint ranges of more than n / kTopNodes
constexpr uint32_t kTopLeaves = 128; // smallest subtree worth the top's levels
constexpr int kMaxLevels = 64;       // 32-bit codes with index tie-breaks
constexpr uint32_t kRestCap = 512;   // a subtree's frontier up to which 64 nodes are opened per step
constexpr uint32_t kRestAlloc = kRestCap + 7 * kMaxLevels + 8; // + growth of one-node steps
constexpr int kRestWaves = 4;

__device__ __forceinline__ float box_area(float4 a, float4 b)
{
    const float x = b.x - a.x, y = b.y - a.y, z = b.z - a.z;
    return x * y + y * z + z * x;
}

// power-of-two grid step covering [lo, hi] in 255 steps, as a biased exponent
__device__ __forceinline__ uint32_t grid_exponent(float lo, float hi)
{
    const float t = (hi - lo) * (1.f / 255.f);
    int e = (__float_as_int(t) >> 23) & 255;
    if (t > __int_as_float(e << 23)) e++;
    e = e < 1 ? 1 : e;
    for (; e < 254; e++) // the decoded top of the grid must reach hi
        if (wnode_decode(lo, 255u, 0, __int_as_float(e << 23)) >= hi) break;
    return uint32_t(e);
}

__device__ __forceinline__ uint32_t quant_lo(float o, float step, float v)
{
    float f = floorf((v - o) / step);
    uint32_t q = f <= 0.f ? 0u : (f >= 255.f ? 255u : uint32_t(f));
    while (q > 0 && wnode_decode(o, q, 0, step) > v) q--;
    return q;
}

__device__ __forceinline__ uint32_t quant_hi(float o, float step, float v)
{
    float f = ceilf((v - o) / step);
    uint32_t q = f <= 0.f ? 0u : (f >= 255.f ? 255u : uint32_t(f));
    while (q < 255 && wnode_decode(o, q, 0, step) < v) q++;
    return q;
}

// The children of the wide node over a binary node. All indexes are static once unrolled: with the
// boxes in an indexed array the kernel spent its time on 0.5 KB of scratch per lane (blob grid's beam
// tree 6.5 ms, 4.0 so), so a child is named by the binary node and side that hold its box.
struct Opened {
    uint32_t at[kWide]; // node << 1 | side
    int c[kWide];       // its link
    float area[kWide];  // -1 for a leaf
    int n, inner;       // children; those of them that are inner nodes
};
__device__ __forceinline__ void open_node(const BNode* bn, uint32_t node, Opened& o)
{
    const auto area = [](const BNode& x, int side) {
        return side ? (x.c1 < 0 ? -1.f : box_area(make_float4(x.lx1, x.ly1, x.lz1, 0.f), make_float4(x.ux1, x.uy1, x.uz1, 0.f)))
                    : (x.c0 < 0 ? -1.f : box_area(make_float4(x.lx0, x.ly0, x.lz0, 0.f), make_float4(x.ux0, x.uy0, x.uz0, 0.f)));
    };
#pragma unroll
    for (int k = 0; k < kWide; k++) {
        o.at[k] = 0u;
        o.c[k] = -1;
        o.area[k] = -1.f;
    }
    const BNode r = bn[node];
    o.at[0] = node << 1;
    o.at[1] = node << 1 | 1u;
    o.c[0] = r.c0;
    o.c[1] = r.c1;
    o.area[0] = area(r, 0);
    o.area[1] = area(r, 1);
    o.n = 2;
#pragma unroll
    for (int i = 2; i < kWide; i++) {
        int best = -1, link = -1;
        float ba = -1.f;
#pragma unroll
        for (int k = 0; k < i; k++)
            if (o.c[k] >= 0 && o.area[k] > ba) {
                ba = o.area[k];
                best = k;
                link = o.c[k];
            }
        if (best < 0) continue; // only leaves are left, now and after
        const BNode x = bn[link];
        const float a0 = area(x, 0);
#pragma unroll
        for (int k = 0; k < i; k++)
            if (k == best) {
                o.at[k] = uint32_t(link) << 1;
                o.c[k] = x.c0;
                o.area[k] = a0;
            }
        o.at[i] = uint32_t(link) << 1 | 1u;
        o.c[i] = x.c1;
        o.area[i] = area(x, 1);
        o.n = i + 1;
    }
    o.inner = 0;
#pragma unroll
    for (int k = 0; k < kWide; k++) o.inner += o.c[k] >= 0 ? 1 : 0;
}

// writes the wide node over binary node `node`, opened; its inner children are the wide nodes from
// `at` on, in order, and each is handed to next(child's binary node, its wide node, its primitives)
template <class Next>
__device__ __forceinline__ void write_wide(const BNode* bn, uint32_t node, WNode* dst, const Opened& o, uint32_t at,
                                           Next next)
{
    const BNode& r = bn[node];
    const f3 nlo = mk(fminf(r.lx0, r.lx1), fminf(r.ly0, r.ly1), fminf(r.lz0, r.lz1));
    const f3 nhi = mk(fmaxf(r.ux0, r.ux1), fmaxf(r.uy0, r.uy1), fmaxf(r.uz0, r.uz1));
    const uint32_t ex = grid_exponent(nlo.x, nhi.x), ey = grid_exponent(nlo.y, nhi.y), ez = grid_exponent(nlo.z, nhi.z);
    const float sx = __int_as_float(int(ex << 23)), sy = __int_as_float(int(ey << 23)), sz = __int_as_float(int(ez << 23));
    WNode w;
    w.ox = nlo.x;
    w.oy = nlo.y;
    w.oz = nlo.z;
    w.meta = ex | (ey << 8) | (ez << 16) | (uint32_t(o.n) << 24);
#pragma unroll
    for (int k = 0; k < 12; k++) w.q[k] = 0;
#pragma unroll
    for (int k = 0; k < 5; k++) w.pad[k] = 0;
    w.signs = 0u;
    w.grown_lo = INFINITY;
    w.grown_hi = 0.f;
#pragma unroll
    for (int k = 0; k < kWide; k++) {
        w.child[k] = 0;
        if (k >= o.n) continue;
        // a node's floats: low and high corner of side 0, of side 1, two links, two tags
        const uint32_t side = o.at[k] & 1u;
        const float* f = reinterpret_cast<const float*>(bn + (o.at[k] >> 1));
        const uint32_t tag = __float_as_uint(f[14u + side]);
        f += 6u * side;
        if (o.c[k] >= 0) {
            next(uint32_t(o.c[k]), at, tag);
            w.child[k] = int(at++);
        } else {
            w.child[k] = o.c[k];
            w.signs |= (tag & 7u) << (3 * k);
            w.grown_lo = fminf(w.grown_lo, __uint_as_float(tag & ~7u));
            w.grown_hi = fmaxf(w.grown_hi, __uint_as_float(tag | 7u));
        }
        const int sh = 8 * (k & 3), wd = k >> 2; // plane p of child k: byte k & 3 of q[2 p + (k >> 2)]
        w.q[0 + wd] |= quant_lo(w.ox, sx, f[0]) << sh;
        w.q[2 + wd] |= quant_lo(w.oy, sy, f[1]) << sh;
        w.q[4 + wd] |= quant_lo(w.oz, sz, f[2]) << sh;
        w.q[6 + wd] |= quant_hi(w.ox, sx, f[3]) << sh;
        w.q[8 + wd] |= quant_hi(w.oy, sy, f[4]) << sh;
        w.q[10 + wd] |= quant_hi(w.oz, sz, f[5]) << sh;
    }
    *dst = w;
}

// the nodes over many primitives, by one block; items: the subtrees left (binary node, wide node);
// meta: their number, the wide nodes numbered so far, the subtrees taken (by k_wide_rest)
__global__ void __launch_bounds__(1024) k_wide_top(const BNode* bn, WNode* wn, uint2* items, uint32_t* meta, uint32_t cap,
                                                   const uint32_t* n_dev)
{
    __shared__ uint2 front[2][kTopNodes];
    __shared__ uint32_t count[2], n_items, n_wide;
    const uint32_t n = dev_count(cap, n_dev), t = threadIdx.x;
    const uint32_t small = max(kTopLeaves, n / kTopNodes + 1u);
    if (t == 0) {
        const bool one = n >= 2u && n <= small;
        front[0][0] = make_uint2(0u, 0u);
        count[0] = n > small ? 1u : 0u;
        count[1] = 0u;
        n_items = one ? 1u : 0u;
        n_wide = 1u;
        if (one) items[0] = make_uint2(0u, 0u);
    }
    __syncthreads();
    for (int cur = 0;; cur ^= 1) {
        const uint32_t c = count[cur];
        if (c == 0u) break;
        for (uint32_t i = t; i < c; i += blockDim.x) {
            const uint2 e = front[cur][i];
            Opened o;
            open_node(bn, e.x, o);
            const uint32_t at = atomicAdd(&n_wide, uint32_t(o.inner));
            write_wide(bn, e.x, &wn[e.y], o, at, [&](uint32_t b, uint32_t w, uint32_t prims) {
                if (prims > small) front[cur ^ 1][atomicAdd(&count[cur ^ 1], 1u)] = make_uint2(b, w);
                else items[atomicAdd(&n_items, 1u)] = make_uint2(b, w);
            });
        }
        __syncthreads();
        if (t == 0) count[cur] = 0u;
        __syncthreads();
    }
    if (t == 0) {
        meta[0] = n_items;
        meta[1] = n_wide;
        meta[2] = 0u;
    }
}

// a subtree per wave; its frontier is bounded as a depth-first walk's (a subtree's nodes are opened
// one by one once it is full)
__global__ void __launch_bounds__(64 * kRestWaves) k_wide_rest(const BNode* bn, WNode* wn, const uint2* items,
                                                               uint32_t* meta)
{
    __shared__ uint2 front_all[kRestWaves][kRestAlloc];
    uint2* front = front_all[threadIdx.x >> 6];
    const uint32_t lane = __lane_id(), n_items = meta[0];
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    const uint32_t waves = gridDim.x * kRestWaves;
    // the first subtrees are dealt out, the rest taken from the counter
    for (uint32_t item = blockIdx.x * kRestWaves + (threadIdx.x >> 6); item < n_items;) {
        if (lane == 0) front[0] = items[item];
        uint32_t fs = 1; // same value in every lane
        while (fs > 0u) {
            wave_lds_sync();
            const uint32_t take = min(min(64u, fs), max(1u, fs < kRestCap ? (kRestCap - fs) / 7u : 0u));
            if (fs + 7u * take > kRestAlloc) break; // unreachable for trees of at most kMaxLevels levels
            const bool has = lane < take;
            uint2 e = make_uint2(0u, 0u);
            Opened o = {};
            if (has) {
                e = front[fs - 1u - lane];
                open_node(bn, e.x, o);
            }
            fs -= take;
            wave_lds_sync();
            uint32_t pre = 0, tot = 0;
            for (int bit = 0; bit < 4; bit++) { // at most kWide = 8: four bits
                const uint64_t m = __ballot((uint32_t(o.inner) >> bit) & 1u);
                pre += uint32_t(__popcll(m & lt)) << bit;
                tot += uint32_t(__popcll(m)) << bit;
            }
            uint32_t at = 0;
            if (lane == 0 && tot) at = atomicAdd(&meta[1], tot);
            at = __shfl(at, 0) + pre;
            uint32_t put = fs + pre;
            if (has)
                write_wide(bn, e.x, &wn[e.y], o, at, [&](uint32_t b, uint32_t w, uint32_t) { front[put++] = make_uint2(b, w); });
            fs += tot;
        }
        if (waves >= n_items) break;
        if (lane == 0) item = waves + atomicAdd(&meta[2], 1u);
        item = __shfl(item, 0);
    }
}

// one primitive: a wide root with a single leaf child; none: a wide root without children (with
// n_dev, the kernel runs every build and acts only for those two counts)
__global__ void k_wide_single(const BNode* bn, WNode* wn, const uint32_t* n_dev)
{
    if (n_dev && *n_dev >= 2) return;
    WNode w;
    for (int k = 0; k < kWide; k++) w.child[k] = 0;
    for (int k = 0; k < 12; k++) w.q[k] = 0;
    for (int k = 0; k < 5; k++) w.pad[k] = 0;
    w.signs = 0u;
    w.grown_lo = w.grown_hi = 0.f;
    if (n_dev && *n_dev == 0) {
        w.ox = w.oy = w.oz = 0.f;
        w.meta = (127u) | (127u << 8) | (127u << 16);
        wn[0] = w;
        return;
    }
    const BNode& b = bn[0];
    w.ox = b.lx0;
    w.oy = b.ly0;
    w.oz = b.lz0;
    const uint32_t ex = grid_exponent(b.lx0, b.ux0), ey = grid_exponent(b.ly0, b.uy0), ez = grid_exponent(b.lz0, b.uz0);
    w.meta = ex | (ey << 8) | (ez << 16) | (1u << 24);
    w.child[0] = ~0;
    w.signs = __float_as_uint(b.tag0) & 7u;
    w.grown_lo = __uint_as_float(__float_as_uint(b.tag0) & ~7u);
    w.grown_hi = __uint_as_float(__float_as_uint(b.tag0) | 7u);
    // child 0: low planes at the origin (byte 0 of q[0], q[2], q[4] stays 0), high planes in q[6..10]
    w.q[6] = quant_hi(b.lx0, __int_as_float(int(ex << 23)), b.ux0);
    w.q[8] = quant_hi(b.ly0, __int_as_float(int(ey << 23)), b.uy0);
    w.q[10] = quant_hi(b.lz0, __int_as_float(int(ez << 23)), b.uz0);
    wn[0] = w;
}

// single primitive: one inner node with leaf 0 on the left and an empty right box
__global__ void k_single(const float4* lo, const float4* hi, BNode* nodes, uint32_t* order, const uint32_t* n_dev)
{
    if (n_dev && *n_dev != 1) return; // with n_dev the kernel runs every build and acts for one primitive
    BNode nd;
    nd.lx0 = lo[0].x;
    nd.ly0 = lo[0].y;
    nd.lz0 = lo[0].z;
    nd.ux0 = hi[0].x;
    nd.uy0 = hi[0].y;
    nd.uz0 = hi[0].z;
    // the unused right slot gets a point box far outside any scene: an inverted box would pass
    // the slab test, which is symmetric in the two planes of each axis
    nd.lx1 = nd.ly1 = nd.lz1 = 3e38f;
    nd.ux1 = nd.uy1 = nd.uz1 = 3e38f;
    nd.c0 = ~0;
    nd.c1 = ~0;
    nd.tag0 = lo[0].w;
    nd.tag1 = 0.f;
    nodes[0] = nd;
    order[0] = 0;
}

inline uint32_t blocks_for(uint64_t n, uint32_t tpb) { return uint32_t((n + tpb - 1) / tpb); }

} // namespace

namespace upbp_host {

// scan_exclusive uses sc.scan as a stack of block-sum arrays, starting at word `base`
static int scan_rec(const uint32_t* in, uint32_t* out, uint32_t n, uint32_t* total_dev, BvhScratch& sc, size_t base,
                    hipStream_t s)
{
    if (n == 0) {
        if (total_dev) hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(1), 0, s, total_dev, 0u, 1u);
        return int(hipGetLastError());
    }
    const uint32_t nb = blocks_for(n, kScanTile);
    if (nb == 1) {
        hipLaunchKernelGGL(k_scan_tile, dim3(1), dim3(kScanThreads), 0, s, in, out, n, nullptr, total_dev);
        return int(hipGetLastError());
    }
    uint32_t* sums = sc.scan.as<uint32_t>() + base;
    hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(kScanThreads), 0, s, in, n, sums);
    int e = scan_rec(sums, sums, nb, total_dev, sc, base + nb + 1, s);
    if (e) return e;
    hipLaunchKernelGGL(k_scan_tile, dim3(nb), dim3(kScanThreads), 0, s, in, out, n, sums, nullptr);
    return int(hipGetLastError());
}

int scan_exclusive(const uint32_t* in, uint32_t* out, uint32_t n, uint32_t* total_dev, BvhScratch& sc, hipStream_t s)
{
    size_t need = 16;
    for (uint64_t m = n; m > uint64_t(kScanTile); m = blocks_for(m, kScanTile)) need += blocks_for(m, kScanTile) + 1;
    if (sc.scan.ensure(need * 4)) return 1;
    return scan_rec(in, out, n, total_dev, sc, 0, s);
}

int radix_sort_pairs(uint32_t* keys, uint32_t* vals, uint32_t n, int bits, BvhScratch& sc, hipStream_t s,
                     const uint32_t* n_dev)
{
    if (n <= 1) return 0;
    const uint32_t nb = blocks_for(n, kSortTile);
    if (sc.keys2.ensure(size_t(n) * 4) || sc.vals2.ensure(size_t(n) * 4) || sc.hist.ensure(size_t(256) * nb * 4))
        return 1;
    uint32_t* hist = sc.hist.as<uint32_t>();
    uint32_t *ka = keys, *va = vals, *kb = sc.keys2.as<uint32_t>(), *vb = sc.vals2.as<uint32_t>();
    int passes = 0;
    for (int shift = 0; shift < bits; shift += 8) {
        hipLaunchKernelGGL(k_radix_hist, dim3(nb), dim3(kSortThreads), 0, s, ka, n, n_dev, shift, hist, nb);
        const int e = scan_exclusive(hist, hist, 256 * nb, nullptr, sc, s);
        if (e) return e;
        hipLaunchKernelGGL(k_radix_scatter, dim3(nb), dim3(kSortThreads), 0, s, ka, va, kb, vb, n, n_dev, shift, hist,
                           nb);
        std::swap(ka, kb);
        std::swap(va, vb);
        passes++;
    }
    if (passes & 1) {
        if (hipMemcpyAsync(keys, ka, size_t(n) * 4, hipMemcpyDeviceToDevice, s) != hipSuccess) return 1;
        if (hipMemcpyAsync(vals, va, size_t(n) * 4, hipMemcpyDeviceToDevice, s) != hipSuccess) return 1;
    }
    return int(hipGetLastError());
}

int lbvh_build(BvhStore& st, BvhScratch& sc, const float4* lo, const float4* hi, uint32_t n, hipStream_t s,
               const uint32_t* n_dev, float4 region)
{
    st.n = n;
    if (n == 0) return 0;
    const uint32_t inner = n > 1 ? n - 1 : 1;
    if (st.cap < n) {
        lbvh_free(st);
        const uint32_t c = n + n / 4;
        if (hipMalloc(&st.nodes, size_t(std::max<uint32_t>(c - 1, inner)) * sizeof(BNode)) != hipSuccess) return 1;
        if (hipMalloc(&st.order, size_t(c) * sizeof(uint32_t)) != hipSuccess) return 1;
        st.cap = c;
    }
    if (n == 1) {
        hipLaunchKernelGGL(k_single, dim3(1), dim3(1), 0, s, lo, hi, st.nodes, st.order, n_dev);
        return int(hipGetLastError());
    }
    if (sc.keys.ensure(size_t(n) * 4) || sc.bounds.ensure(64))
        return 1;
    uint32_t* bounds = sc.bounds.as<uint32_t>();
    uint32_t* keys = sc.keys.as<uint32_t>();
    const uint32_t tpb = 256;
    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(3), 0, s, bounds, 0xffffffffu, 3u);
    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(3), 0, s, bounds + 3, 0u, 3u);
    hipLaunchKernelGGL(k_centroid_bounds, dim3(std::min<uint32_t>(blocks_for(n, tpb), 1024)), dim3(tpb), 0, s, lo, hi,
                       n, n_dev, bounds);
    hipLaunchKernelGGL(k_morton, dim3(blocks_for(n, tpb)), dim3(tpb), 0, s, lo, hi, n, n_dev, bounds,
                       region, keys, st.order);
    const int e = radix_sort_pairs(keys, st.order, n, region.w > 0.f ? 32 : 30, sc, s, n_dev);
    if (e) return e;
    // with a count in device memory the tree may hold a single primitive (written whole here) or none
    if (n_dev) hipLaunchKernelGGL(k_single, dim3(1), dim3(1), 0, s, lo, hi, st.nodes, st.order, n_dev);
    Pyramid P;
    P.levels = 0;
    size_t total = 0;
    for (uint64_t m = n;; m = (m + 7) / 8) {
        P.off[P.levels++] = uint32_t(total);
        total += m;
        if (m <= 8) break;
    }
    if (sc.pyramid.ensure(2 * total * sizeof(float4))) return 1;
    P.lo = sc.pyramid.as<float4>();
    P.hi = P.lo + total;
    uint64_t m = n;
    for (int l = 0; l == 0 || l + 1 < P.levels; l += 3, m = (m + 511) / 512)
        hipLaunchKernelGGL(k_pyramid, dim3(uint32_t((m + kPyrBlock - 1) / kPyrBlock)), dim3(kPyrBlock), 0, s, P, l, lo, hi,
                           st.order, n, n_dev);
    hipLaunchKernelGGL(k_karras, dim3(blocks_for(n - 1, tpb)), dim3(tpb), 0, s, keys, n, n_dev, P, st.nodes);
    return int(hipGetLastError());
}

int wbvh_build(WBvhStore& w, const BvhStore& bin, BvhScratch& sc, uint32_t n, hipStream_t s, const uint32_t* n_dev)
{
    w.n = n;
    if (n == 0) return 0;
    const uint32_t need = n > 1 ? n - 1 : 1;
    if (w.cap < need) {
        wbvh_free(w);
        const uint32_t c = need + need / 4;
        if (hipMalloc(&w.nodes, size_t(c) * sizeof(WNode)) != hipSuccess) return 1;
        w.cap = c;
    }
    if (n == 1 || n_dev) hipLaunchKernelGGL(k_wide_single, dim3(1), dim3(1), 0, s, bin.nodes, w.nodes, n_dev);
    if (n == 1) return int(hipGetLastError());
    if (sc.meta.ensure(3 * 4) || sc.items.ensure(size_t(n / 2 + 1) * sizeof(uint2))) return 1;
    uint32_t* meta = sc.meta.as<uint32_t>();
    uint2* items = sc.items.as<uint2>(); // subtrees are disjoint and have two primitives or more
    hipLaunchKernelGGL(k_wide_top, dim3(1), dim3(1024), 0, s, bin.nodes, w.nodes, items, meta, n, n_dev);
    hipLaunchKernelGGL(k_wide_rest, dim3(std::min<uint32_t>(blocks_for(n, 64 * kRestWaves), 1024)), dim3(64 * kRestWaves), 0, s,
                       bin.nodes, w.nodes, items, meta);
    return int(hipGetLastError());
}

void wbvh_free(WBvhStore& w)
{
    if (w.nodes) (void)hipFree(w.nodes);
    w.nodes = nullptr;
    w.cap = 0;
}

void lbvh_free(BvhStore& st)
{
    if (st.nodes) (void)hipFree(st.nodes);
    if (st.order) (void)hipFree(st.order);
    st.nodes = nullptr;
    st.order = nullptr;
    st.cap = 0;
}

void lbvh_scratch_free(BvhScratch& sc)
{
    for (DevBuf* b : {&sc.keys, &sc.keys2, &sc.vals2, &sc.hist, &sc.scan, &sc.pyramid, &sc.items, &sc.meta, &sc.bounds})
        b->release();
}

} // namespace upbp_host
