// LBVH traversal on the device and the host-side builder interface.
//
// Replaces the RTX traversals of nolmoonen/gpuupbp (optixTrace in
// gpuupbp/kernel/intersector.cuh:120,214 and gpuupbp/kernel/pde/functs_*.cuh) by
// stack traversal of a binary LBVH whose inner nodes carry both child boxes.
// Leaf boxes are inflated at build time so that box tests are conservative with
// respect to the exact FP32 acceptance predicates evaluated at the leaves.
#pragma once

#include "upbp_device.h"

namespace upbp {

// orders this wave's LDS accesses before the ones that follow (all lanes of one wave)
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

constexpr int kBvhStack = 64;

struct RayBox {
    f3 o, inv;
    float tmin, tmax;
};

UPBP_HD RayBox make_raybox(f3 o, f3 d, float tmin, float tmax)
{
    return {o, mk(1.f / d.x, 1.f / d.y, 1.f / d.z), tmin, tmax};
}

// Slab test; NaNs from 0*inf are ignored by fminf/fmaxf, which keeps the test conservative.
UPBP_HD bool slab(const RayBox& r, float lx, float ly, float lz, float ux, float uy, float uz, float tmax,
                  float& tentry)
{
    const float tx0 = (lx - r.o.x) * r.inv.x, tx1 = (ux - r.o.x) * r.inv.x;
    const float ty0 = (ly - r.o.y) * r.inv.y, ty1 = (uy - r.o.y) * r.inv.y;
    const float tz0 = (lz - r.o.z) * r.inv.z, tz1 = (uz - r.o.z) * r.inv.z;
    const float tn = fmaxf(fmaxf(fminf(tx0, tx1), fminf(ty0, ty1)), fmaxf(fminf(tz0, tz1), r.tmin));
    const float tf = fminf(fminf(fmaxf(tx0, tx1), fmaxf(ty0, ty1)), fminf(fmaxf(tz0, tz1), tmax));
    tentry = tn;
    return tn <= tf;
}

UPBP_HD bool inside(f3 p, float lx, float ly, float lz, float ux, float uy, float uz)
{
    return p.x >= lx && p.y >= ly && p.z >= lz && p.x <= ux && p.y <= uy && p.z <= uz;
}

// Visits every leaf whose box contains p. fn(sorted_leaf) -> void.
template <typename F>
__device__ __forceinline__ bool bvh_point_query(const Bvh& b, f3 p, F&& fn)
{
    if (b.n == 0) return true;
    int stack[kBvhStack];
    int sp = 0;
    int node = 0;
    for (;;) {
        const BNode nd = b.nodes[node];
        const bool h0 = inside(p, nd.lx0, nd.ly0, nd.lz0, nd.ux0, nd.uy0, nd.uz0);
        const bool h1 = inside(p, nd.lx1, nd.ly1, nd.lz1, nd.ux1, nd.uy1, nd.uz1);
        int next = -1;
        if (h0) {
            if (nd.c0 < 0) fn(uint32_t(~nd.c0));
            else next = nd.c0;
        }
        if (h1) {
            if (nd.c1 < 0) fn(uint32_t(~nd.c1));
            else if (next < 0) next = nd.c1;
            else {
                if (sp == kBvhStack) return false;
                stack[sp++] = nd.c1;
            }
        }
        if (next < 0) {
            if (sp == 0) return true;
            next = stack[--sp];
        }
        node = next;
    }
}

// Visits every leaf whose box meets the segment [tmin, tmax] of the ray.
// fn(sorted_leaf, float& tmax) may shrink tmax (closest-hit queries).
template <typename F>
__device__ __forceinline__ bool bvh_ray_query(const Bvh& b, f3 o, f3 d, float tmin, float tmax, F&& fn)
{
    if (b.n == 0) return true;
    const RayBox r = make_raybox(o, d, tmin, tmax);
    float tcur = tmax;
    int stack[kBvhStack];
    int sp = 0;
    int node = 0;
    for (;;) {
        const BNode nd = b.nodes[node];
        float e0, e1;
        const bool h0 = slab(r, nd.lx0, nd.ly0, nd.lz0, nd.ux0, nd.uy0, nd.uz0, tcur, e0);
        const bool h1 = slab(r, nd.lx1, nd.ly1, nd.lz1, nd.ux1, nd.uy1, nd.uz1, tcur, e1);
        int n0 = -1, n1 = -1; // inner children to visit, nearest first
        if (h0) {
            if (nd.c0 < 0) fn(uint32_t(~nd.c0), tcur);
            else n0 = nd.c0;
        }
        if (h1) {
            if (nd.c1 < 0) fn(uint32_t(~nd.c1), tcur);
            else n1 = nd.c1;
        }
        int next;
        if (n0 >= 0 && n1 >= 0) {
            if (e1 < e0) {
                const int t = n0;
                n0 = n1;
                n1 = t;
            }
            if (sp == kBvhStack) return false;
            stack[sp++] = n1;
            next = n0;
        } else {
            next = n0 >= 0 ? n0 : n1;
        }
        if (next < 0) {
            if (sp == 0) return true;
            next = stack[--sp];
        }
        node = next;
    }
}

// Ray for the merge kernels' node step: a plane at origin + q * step (q an 8-bit grid index) is met at
// fma(q, step * inv, (origin - o) * inv), one operation per plane after three per node and axis. A
// direction component below 1e-18 counts as +-1e-18, so that no product is infinite times zero.
struct GridRay {
    f3 o, inv;
    float tmin, tmax;
};
UPBP_HD GridRay make_gridray(f3 o, f3 d, float tmin, float tmax)
{
    const f3 c{fabsf(d.x) < 1e-18f ? copysignf(1e-18f, d.x) : d.x, fabsf(d.y) < 1e-18f ? copysignf(1e-18f, d.y) : d.y,
               fabsf(d.z) < 1e-18f ? copysignf(1e-18f, d.z) : d.z};
    return {o, mk(1.f / c.x, 1.f / c.y, 1.f / c.z), tmin, tmax};
}

UPBP_HD uint32_t f2bits(float x) { return __builtin_bit_cast(uint32_t, x); }

// A wide node in registers (native vectors and no indexed member, or it ends up in scratch memory).
typedef float vf4 __attribute__((ext_vector_type(4)));
typedef int vi4 __attribute__((ext_vector_type(4)));
struct WNodeRegs {
    vf4 h, q0, q1, q2, t; // origin and meta; planes; signs and inflations
    vi4 c0, c1;           // child links
};
__device__ __forceinline__ void load_wnode(const WNode* node, WNodeRegs& n)
{
    const vf4* np = reinterpret_cast<const vf4*>(node);
    const vi4* ni = reinterpret_cast<const vi4*>(node);
    n.h = np[0];
    n.c0 = ni[1];
    n.c1 = ni[2];
    n.q0 = np[3];
    n.q1 = np[4];
    n.q2 = np[5];
    n.t = np[6];
}
__device__ __forceinline__ uint32_t wnode_leaves(const WNodeRegs& n)
{
    return (uint32_t(n.c0.x) >> 31) | ((uint32_t(n.c0.y) >> 31) << 1) | ((uint32_t(n.c0.z) >> 31) << 2) |
           ((uint32_t(n.c0.w) >> 31) << 3) | ((uint32_t(n.c1.x) >> 31) << 4) | ((uint32_t(n.c1.y) >> 31) << 5) |
           ((uint32_t(n.c1.z) >> 31) << 6) | ((uint32_t(n.c1.w) >> 31) << 7);
}
// link of child k (k differs between lanes: selects)
__device__ __forceinline__ int wnode_child(const WNodeRegs& n, uint32_t k)
{
    const bool b0 = k & 1u, b1 = k & 2u, b2 = k & 4u;
    const int x0 = b0 ? n.c0.y : n.c0.x, x1 = b0 ? n.c0.w : n.c0.z, x2 = b0 ? n.c1.y : n.c1.x, x3 = b0 ? n.c1.w : n.c1.z;
    const int y0 = b1 ? x1 : x0, y1 = b1 ? x3 : x2;
    return b2 ? y1 : y0;
}

// The children of a wide node whose boxes, grown by `grow` on every side, meet [tmin, tmax] of the
// ray: a bit per child. The sign of each direction component picks the near and far planes once per
// node, so a child costs six conversions, six FMAs and three-operand minima and maxima; decoding the
// boxes and ordering each plane pair took twice the instructions.
// A plane's t = q s + b is off by at most 5 * 2^-24 |b| and 4 * 2^-24 q |s| (the roundings of the
// difference, the reciprocal, the two products and the sum), whatever cancels in it, so all planes
// move outwards by 2^-21 (|b| + 255 |s|): the boxes met include every box the exact arithmetic meets.
UPBP_HD uint32_t wide_hits(const WNodeRegs& n, const GridRay& r, float grow)
{
    const vf4 h = n.h, q0 = n.q0, q1 = n.q1, q2 = n.q2;
    const uint32_t meta = f2bits(h.w);
    const bool px = r.inv.x >= 0.f, py = r.inv.y >= 0.f, pz = r.inv.z >= 0.f;
    const float sx = wnode_step(meta, 0) * r.inv.x, sy = wnode_step(meta, 1) * r.inv.y,
                sz = wnode_step(meta, 2) * r.inv.z;
    const float bx = (h.x - r.o.x) * r.inv.x, by = (h.y - r.o.y) * r.inv.y, bz = (h.z - r.o.z) * r.inv.z;
    const auto out = [&](float inv, float step, float b) {
        return __builtin_fmaf(0x1p-21f, fabsf(b) + 255.f * fabsf(step), grow * fabsf(inv));
    };
    const float gx = out(r.inv.x, sx, bx), gy = out(r.inv.y, sy, by), gz = out(r.inv.z, sz, bz);
    // planes of children 0-3 and 4-7: low x q0.xy, low y q0.zw, low z q1.xy, high x q1.zw, high y
    // q2.xy, high z q2.zw
    const uint32_t nx[2] = {f2bits(px ? q0.x : q1.z), f2bits(px ? q0.y : q1.w)};
    const uint32_t fx[2] = {f2bits(px ? q1.z : q0.x), f2bits(px ? q1.w : q0.y)};
    const uint32_t ny[2] = {f2bits(py ? q0.z : q2.x), f2bits(py ? q0.w : q2.y)};
    const uint32_t fy[2] = {f2bits(py ? q2.x : q0.z), f2bits(py ? q2.y : q0.w)};
    const uint32_t nz[2] = {f2bits(pz ? q1.x : q2.z), f2bits(pz ? q1.y : q2.w)};
    const uint32_t fz[2] = {f2bits(pz ? q2.z : q1.x), f2bits(pz ? q2.w : q1.y)};
    const float nbx = bx - gx, nby = by - gy, nbz = bz - gz, fbx = bx + gx, fby = by + gy, fbz = bz + gz;
    uint32_t hits = 0;
#pragma unroll
    for (int k = 0; k < kWide; k++) {
        const int w = k >> 2, sh = 8 * (k & 3);
        const auto at = [&](const uint32_t* q, float s, float t0) {
            return __builtin_fmaf(float((q[w] >> sh) & 255u), s, t0);
        };
        const float tn = fmaxf(fmaxf(at(nx, sx, nbx), at(ny, sy, nby)), fmaxf(at(nz, sz, nbz), r.tmin));
        const float tf = fminf(fminf(at(fx, sx, fbx), at(fy, sy, fby)), fminf(at(fz, sz, fbz), r.tmax));
        hits |= tn <= tf ? 1u << k : 0u;
    }
    return hits & ((1u << wnode_count(meta)) - 1u);
}

// Whether leaf child k's segment comes within reach of the line through ro along rd (unit): a cull
// in front of the exact predicate that reads nothing beyond the node. The segment is its box's
// diagonal (the node holds the direction's signs) shrunk by the box's inflation, known to half a grid
// step per axis. `reach`: the predicate's radius (plus what the line stands for); `grown`: the part
// of the inflation that is radius and slack; `slack`: the boxes' allowance for the FP32 error of the
// beam predicate's line parameters, by which a pair can be owned by a sub-beam some way off. That
// error grows as the lines become parallel (at the predicate's cut-off, 0.2 degrees, a tenth of a
// unit along the beam) and as they become perpendicular (it divides by their cosine): below 6 and
// above 87 degrees every segment passes, between them a tenth of the slack is ample. `spread`:
// largest difference of a direction the line stands for from rd. The rest of the inflation (the
// primitive's own rounding allowance) and 1e-6 of the distance are added. NaN passes.
// A candidate's 48-byte record and its query's are most of the per-piece walk's cache misses, and
// one box hit in four is within reach (blob grid: B-B1D 67 -> 58 ms, slab room 98 -> 90, with the
// slabs in fused multiply-adds).
__device__ __forceinline__ bool leaf_near(const WNodeRegs& n, uint32_t k, f3 ro, f3 rd, float reach, float grown,
                                          float slack, float spread)
{
    const uint32_t meta = __float_as_uint(n.h.w), sh = 8u * (k & 3u);
    const bool up = k >= 4u;
    const auto plane = [&](float a, float b) { return float((__float_as_uint(up ? b : a) >> sh) & 255u); };
    const float lx = plane(n.q0.x, n.q0.y), ly = plane(n.q0.z, n.q0.w), lz = plane(n.q1.x, n.q1.y);
    const float ux = plane(n.q1.z, n.q1.w), uy = plane(n.q2.x, n.q2.y), uz = plane(n.q2.z, n.q2.w);
    const float sx = .5f * wnode_step(meta, 0), sy = .5f * wnode_step(meta, 1), sz = .5f * wnode_step(meta, 2);
    const f3 base = mk(n.h.x - ro.x, n.h.y - ro.y, n.h.z - ro.z);
    const float glo = n.t.y, ghi = n.t.z, gmid = .5f * (glo + ghi), gdif = .5f * (ghi - glo);
    // centre and half vector of the segment
    const f3 u{__builtin_fmaf(sx, lx + ux, base.x), __builtin_fmaf(sy, ly + uy, base.y),
               __builtin_fmaf(sz, lz + uz, base.z)};
    const uint32_t sg = __float_as_uint(n.t.x) >> (3u * k);
    const auto flip = [&](float h, uint32_t bit) { return __uint_as_float(__float_as_uint(h) ^ (bit << 31)); };
    const f3 v{flip(__builtin_fmaf(sx, ux - lx, -(sx + gmid)), sg & 1u),
               flip(__builtin_fmaf(sy, uy - ly, -(sy + gmid)), (sg >> 1) & 1u),
               flip(__builtin_fmaf(sz, uz - lz, -(sz + gmid)), (sg >> 2) & 1u)};
    const auto fdot = [](f3 a, f3 b) { return __builtin_fmaf(a.x, b.x, __builtin_fmaf(a.y, b.y, a.z * b.z)); };
    const auto along = [](f3 a, float t, f3 b) { // a + t b
        return f3{__builtin_fmaf(t, b.x, a.x), __builtin_fmaf(t, b.y, a.y), __builtin_fmaf(t, b.z, a.z)};
    };
    const float vd = fdot(v, rd);
    const f3 up_ = along(u, -fdot(u, rd), rd), vp = along(v, -vd, rd); // across the line
    const float vv = fdot(vp, vp);
    const float t = fminf(fmaxf(-fdot(up_, vp) * __builtin_amdgcn_rcpf(fmaxf(vv, 1e-30f)), -1.f), 1.f);
    const f3 w = along(up_, t, vp);
    const float ex = sx + gdif, ey = sy + gdif, ez = sz + gdif;
    const float err = __builtin_amdgcn_sqrtf(__builtin_fmaf(ex, ex, __builtin_fmaf(ey, ey, ez * ez)));
    const float far = fmaxf(fabsf(base.x), fmaxf(fabsf(base.y), fabsf(base.z)));
    float R = reach + fmaxf(ghi - grown, 0.f) + .1f * slack;
    R = __builtin_fmaf(err, 1.0001f, __builtin_fmaf(far, 1e-6f, R));
    const float par = .1f + spread, perp = .05f + spread;
    return vv < par * par * vd * vd || vd * vd < perp * perp * vv || !(fdot(w, w) > R * R * 1.0001f);
}

// Visits every leaf of a photon map's wide LBVH whose box meets the segment [tmin, tmax] of the ray
// (d unit) and whose primitive comes within reach of its line, as the merge kernels walk it.
template <typename F>
__device__ __forceinline__ bool wbvh_ray_query(const WBvh& b, f3 o, f3 d, float tmin, float tmax, float reach,
                                               float grown, float slack, F&& fn)
{
    if (b.n == 0) return true;
    const GridRay r = make_gridray(o, d, tmin, tmax);
    int stack[kBvhStack];
    int sp = 0;
    int node = 0;
    for (;;) {
        WNodeRegs n;
        load_wnode(&b.nodes[node], n);
        uint32_t hits = wide_hits(n, r, 0.f);
        int next = -1;
        for (; hits; hits &= hits - 1u) {
            const uint32_t k = uint32_t(__ffs(int(hits))) - 1u;
            const int c = wnode_child(n, k);
            if (c < 0) {
                if (leaf_near(n, k, o, d, reach, grown, slack, 0.f)) fn(uint32_t(~c));
            } else if (next < 0) {
                next = c;
            } else {
                if (sp == kBvhStack) return false;
                stack[sp++] = c;
            }
        }
        if (next < 0) {
            if (sp == 0) return true;
            next = stack[--sp];
        }
        node = next;
    }
}

// Moller-Trumbore (Moller & Trumbore 1997); replaces OptiX's built-in triangle test.
UPBP_HD bool tri_test(float4 p0, float4 e1, float4 e2, f3 o, f3 d, float tmin, float tmax, float& th, float& bu,
                      float& bv)
{
    const f3 E1 = mk(e1.x, e1.y, e1.z), E2 = mk(e2.x, e2.y, e2.z);
    const f3 pv = cross(d, E2);
    const float det = dot(E1, pv);
    if (det == 0.f) return false;
    const float inv = 1.f / det;
    const f3 tv = o - mk(p0.x, p0.y, p0.z);
    const float u = dot(tv, pv) * inv;
    if (u < 0.f || u > 1.f) return false;
    const f3 qv = cross(tv, E1);
    const float v = dot(d, qv) * inv;
    if (v < 0.f || u + v > 1.f) return false;
    const float t = dot(E2, qv) * inv;
    if (!(t > tmin && t < tmax)) return false;
    th = t;
    bu = u;
    bv = v;
    return true;
}

// Analytic sphere (centre s.xyz, radius s.w) against a ray: the roots of |o + t d - c| = r with
// the near root refined by one more solve from the first estimate when the ray starts more
// than a radius away, which removes the cancellation of b^2 - c for distant spheres
// (gpuupbp/kernel/intersector.cu:35-95). Writes the roots in (tmin, tmax), near first, and the
// outward normals at them; returns how many (0..2). A closest-hit caller takes the first, an
// all-hits caller every one.
UPBP_HD int sphere_test(float4 s, f3 ro, f3 rd, float tmin, float tmax, float* th, f3* nh)
{
#pragma clang fp contract(off)
    const float radius = s.w;
    const f3 o = ro - mk(s.x, s.y, s.z);
    const float l = 1.f / sqrtf(dot(rd, rd));
    const f3 d = rd * l;
    float b = dot(o, d);
    float c = dot(o, o) - radius * radius;
    float disc = b * b - c;
    if (!(disc > 0.f)) return 0;
    float sdisc = sqrtf(disc);
    const float root1 = -b - sdisc;
    float root11 = 0.f;
    const bool refine = fabsf(root1) > radius;
    if (refine) {
        const f3 o1 = o + d * root1;
        b = dot(o1, d);
        c = dot(o1, o1) - radius * radius;
        disc = b * b - c;
        if (disc > 0.f) {
            sdisc = sqrtf(disc);
            root11 = -b - sdisc;
        }
    }
    int n = 0;
    const float near = root1 + root11;
    float t = near * l;
    if (t > tmin && t < tmax) {
        th[n] = t;
        nh[n++] = (o + d * near) / radius;
    }
    const float root2 = (-b + sdisc) + (refine ? root1 : 0.f);
    t = root2 * l;
    if (t > tmin && t < tmax) {
        th[n] = t;
        nh[n++] = (o + d * root2) / radius;
    }
    return n;
}

} // namespace upbp

// ---- host-side builder ---------------------------------------------------------
namespace upbp_host {

// Device storage of one LBVH: max(n-1,1) inner nodes plus the sorted order.
struct BvhStore {
    upbp::BNode* nodes = nullptr;
    uint32_t* order = nullptr;
    uint32_t n = 0, cap = 0;
};

// Scratch shared by all builds of one renderer (grow-only, one capacity per buffer).
struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
    int ensure(size_t need)
    {
        if (need <= bytes && p) return 0;
        if (p) (void)hipFree(p);
        p = nullptr;
        bytes = 0;
        const size_t b = need < 4096 ? 4096 : need + need / 4;
        if (hipMalloc(&p, b) != hipSuccess) return 1;
        bytes = b;
        return 0;
    }
    void release()
    {
        if (p) (void)hipFree(p);
        p = nullptr;
        bytes = 0;
    }
    template <typename T>
    T* as() const
    {
        return static_cast<T*>(p);
    }
};

struct BvhScratch {
    DevBuf keys, keys2, vals2, hist, scan, pyramid, items, meta, bounds;
};

// Device storage of a wide LBVH collapsed from a binary one (at most n-1 nodes).
struct WBvhStore {
    upbp::WNode* nodes = nullptr;
    uint32_t n = 0, cap = 0;
};

// Primitive boxes are given as lo/hi float4 arrays, already inflated (photon trees: lo.w is box_tag).
// Builds into st on stream s; returns 0 or a hipError_t value. With n_dev, the primitive count
// is read from device memory when the kernels run (at most n, which then sizes the buffers and
// launches): no host synchronisation, and zero or one primitive are handled on the device.
// region (centre, radius > 0): where the Morton grid keeps its resolution when primitives lie far
// outside it; radius 0: a linear grid over all of them.
int lbvh_build(BvhStore& st, BvhScratch& sc, const float4* lo, const float4* hi, uint32_t n, hipStream_t s,
               const uint32_t* n_dev = nullptr, float4 region = float4{0.f, 0.f, 0.f, 0.f});
void lbvh_free(BvhStore& st);
// Collapses the binary LBVH `bin` (n leaves) into a kWide-wide one; same leaf order.
int wbvh_build(WBvhStore& w, const BvhStore& bin, BvhScratch& sc, uint32_t n, hipStream_t s,
               const uint32_t* n_dev = nullptr);
void wbvh_free(WBvhStore& w);
void lbvh_scratch_free(BvhScratch& sc);

// Stable LSD radix sort of (key, value) pairs on the low `bits` bits; keys/vals updated in place.
int radix_sort_pairs(uint32_t* keys, uint32_t* vals, uint32_t n, int bits, BvhScratch& sc, hipStream_t s,
                     const uint32_t* n_dev = nullptr);
// Exclusive prefix sum of n u32 values; in and out may alias. Returns the total through *total_dev
// (device pointer, may be null).
int scan_exclusive(const uint32_t* in, uint32_t* out, uint32_t n, uint32_t* total_dev, BvhScratch& sc,
                   hipStream_t s);

} // namespace upbp_host
