// Camera-subpath wavefront. A path segment takes three kernels:
// * k_camera_bounce: the medium-aware intersector, one P-B2D / B-B1D query per scattering medium
//   segment of the ray (evaluated by the segment merge kernels), light hits, and the list of the
//   vertex's occlusion rays: next-event estimation and one vertex connection per vertex of the
//   chosen light path;
// * k_camera_connect: those rays, one per lane, each with its estimator;
// * k_camera_shade: the rays' contributions in list order, surface / P-P3D / B-P2D merges (point
//   queries), scattering and wave-aggregated queue compaction;
// or one, k_camera_whole, whose lanes trace their vertex's rays themselves (IterParams::whole).
// A path makes up to max_len rays per vertex, one after another when one lane traces them all: the
// last bounces' few paths took 0.3 to 0.4 ms each that way, and a wave waited for its longest path.
// Every contribution carries its constant-time MIS weight computed in place.
// Semantics: nolmoonen/gpuupbp gpuupbp/kernel/trace_camera.cu:49-390,
// gpuupbp/kernel/functs_camera.cuh:41-527 and gpuupbp/kernel/pde/functs_*.cuh.
#include "estimators.h"
#include "kernels.h"

#include <algorithm>

namespace upbp {

// kernel/pde/functs_pb2d.cuh:226-342 and functs_bb1d.cuh:273-397: one P-B2D / B-B1D query per
// scattering medium segment of the camera ray, carrying the camera state the merge needs
// (throughput times the attenuation before the segment, the accumulated ray-sampling pdfs
// and the MIS quantities of the segment's start). MODE 0 counts the queries and sums the lengths
// they are cut over, MODE 1 also counts their pieces, MODE 2 writes queries and pieces.
struct SegCount {
    uint32_t recs = 0, pieces = 0;
    float len = 0.f;
};

template <int MODE>
__device__ __forceinline__ SegCount segment_queries(const DScene& sc, const VolSeg* segs, const LiteSeg* lite, int n,
                                                    unsigned flags, uint32_t qbt, float piece_len, float4 ball, const Sub& s,
                                                    uint32_t pix, SegRec* out, uint8_t* npl)
{
    f3 att = mk(1.f);
    float rsf = 1.f, rsr = 1.f;
    SegCount c;
    for (int i = 0; i < n; i++) {
        const float dmin = segs ? segs[i].dmin : lite[i].dmin;
        const float dmax = segs ? segs[i].dmax : lite[i].dmax;
        const int mid = segs ? segs[i].med : lite[i].med;
        if (mid < 0) continue;
        const DMedium& m = sc.media[mid];
        if (m.has_scattering) {
            float c0, c1;
            cut_range(s.origin, s.dir, dmin, dmax, ball, c0, c1);
            const float len = c1 - c0;
            const uint32_t np = MODE == 0 ? 0u : piece_count(len, piece_len);
            if (MODE == 2) {
                const SegQ q{s.origin, s.dir, dmin, dmax, mid, rsf, rsr, kEndInMedium | (i == 0 ? flags : 0u),
                             s.path_length};
                store_segrec(out + c.recs, q, s.sw, s.throughput * att, pix);
                npl[c.recs] = uint8_t(np);
            }
            c.recs++;
            c.pieces += np;
            c.len += len;
        }
        if (segs) {
            if (qbt == T_BEAM_SHORT) att *= segs[i].att / segs[i].pf;
            else att *= segs[i].att;
            if (!positive(att)) break;
            rsf *= segs[i].pf;
            rsr *= segs[i].pr;
        } else {
            att *= eval_attenuation(m, dmax - dmin);
            if (!positive(att)) break;
            float srr;
            const float sff = ray_sample_pdf(m, dmin, dmax, i == 0 ? flags : 0u, &srr);
            rsf *= sff;
            rsr *= srr;
        }
    }
    return c;
}

// Wave-aggregated allocation of c < 2^BITS slots per lane: one atomic per wave.
template <int BITS>
__device__ __forceinline__ uint32_t wave_alloc(uint32_t c, uint32_t* counter)
{
    const uint32_t lane = __lane_id();
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    uint32_t pre = 0, tot = 0;
    for (int bit = 0; bit < BITS; bit++) {
        const uint64_t m = __ballot((c >> bit) & 1u);
        pre += uint32_t(__popcll(m & lt)) << bit;
        tot += uint32_t(__popcll(m)) << bit;
    }
    const int leader = __ffsll((unsigned long long)__ballot(1)) - 1;
    uint32_t base = 0;
    if (int(lane) == leader && tot) base = atomicAdd(counter, tot);
    base = __shfl(base, leader);
    return base + pre;
}

// Wave-aggregated allocation of one block for the whole wave (c < 2^BITS per lane): returns
// the block's first slot and its size (the same in every lane).
template <int BITS>
__device__ __forceinline__ uint32_t wave_alloc_block(uint32_t c, uint32_t* counter, uint32_t& tot)
{
    const uint32_t lane = __lane_id();
    tot = 0;
    for (int bit = 0; bit < BITS; bit++) tot += uint32_t(__popcll(__ballot((c >> bit) & 1u))) << bit;
    const int leader = __ffsll((unsigned long long)__ballot(1)) - 1;
    uint32_t base = 0;
    if (int(lane) == leader && tot) base = atomicAdd(counter, tot);
    return __shfl(base, leader);
}

// kernel/functs_camera.cuh:41-103
__device__ __forceinline__ int generate_camera_sample(const DScene& sc, const IterParams& p, uint32_t pix, Sub& s,
                                                      float& sx, float& sy, Rng& rng)
{
    const DCamera& cam = sc.cam;
    const uint32_t rx = uint32_t(cam.res_x);
    const uint32_t x = pix % rx, y = pix / rx;
    const float j0 = rng.next(), j1 = rng.next();
    sx = float(x) + j0;
    sy = float(y) + j1;
    const f3 dir = raster_dir(cam, sx, sy);
    const float cos_at = dot(cam.forward, dir);
    const float ipd = cam.ipd / cos_at;
    const float cam_pdf_w = (ipd * ipd) / cos_at;
    s.origin = cam.origin;
    s.dir = dir;
    s.throughput = mk(1.f);
    s.path_length = 1;
    s.specular_path = true;
    s.infinite = false;
    s.sw.w.d_shared = float(p.n_light) / cam_pdf_w;
    s.sw.w.d_bpt = 0.f;
    s.sw.w.d_pde = 0.f;
    s.sw.w.for_inv = s.sw.w.rev_inv = s.sw.w.for_ratio = s.sw.w.rev_ratio = 0.f;
    s.sw.w.prev_specular = 0;
    s.sw.w.prev_in_medium = 0;
    s.sw.last_sin = s.sw.d_bpt_a = s.sw.d_bpt_b = s.sw.d_pde_a = s.sw.d_pde_b = 0.f;
    return init_stack(sc, s.stack, cam.mat_id, cam.med_id);
}

// Camera paths start in 8x8-pixel tiles per wave (16x16 per block): the queue of live paths, and
// with it the bounce kernels' waves and the segment-query pieces they write, then hold compact
// pixel tiles, whose rays are more coherent than a 64-pixel row. Only the order changes; every
// pixel keeps its own random streams.
// vb: the block's index within its job (blockIdx.x for a single job)
__device__ __forceinline__ void camera_generate_body(const DScene& sc, const Bufs& b, uint32_t res_x, uint32_t tiles_x,
                                                     uint32_t vb)
{
    const IterParams& p = *b.params;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t x = (vb % tiles_x) * 16u + (wave & 1u) * 8u + (lane & 7u);
    const uint32_t y = (vb / tiles_x) * 16u + (wave >> 1) * 8u + (lane >> 3);
    const uint32_t pix = y * res_x + x;
    if (x >= res_x || pix >= p.n_pixels) return;
    Rng rng(kDomainCamera, pix, p.iter_key, 0, P_JITTER);
    Sub s;
    float sx, sy;
    const int ret = generate_camera_sample(sc, p, pix, s, sx, sy, rng);
    PathState st;
    st.flags = ((p.techniques & (T_PREVIOUS | T_COMPATIBLE)) != 0) ? PF_ONLY_SPEC_SURF : 0u;
    st.color = mk(0.f);
    st.sx = sx;
    st.sy = sy;
    save_sub(st, s);
    b.cstate[pix] = st;
    const bool alive = ret == S_OK;
    if (alive) store_stack(b.cstack, pix, s.stack);
    else stat_add(b.stats, STAT_ERRORS, 1);
    queue_append(alive, pix, b.queue[0], &b.qcount[64]);
}

__global__ void __launch_bounds__(256) k_camera_generate(DScene sc, Bufs b, uint32_t res_x, uint32_t tiles_x)
{
    camera_generate_body(sc, b, res_x, tiles_x, blockIdx.x);
}

__global__ void __launch_bounds__(256) k_camera_generate_batch(const BatchJob* jobs, const uint2* bmap)
{
    const uint2 m = bmap[blockIdx.x];
    const BatchJob& J = jobs[m.x];
    camera_generate_body(J.sc, J.b, J.res_x, J.tiles_x, m.y);
}

struct CamCounters {
    uint32_t conn = 0, pq = 0, sq = 0, acc = 0, pieces = 0;
};

// The contributions to a camera path of its vertex's next-event estimation and of the connection to
// the light vertex in `slot`, with the status (kernel/trace_camera.cu:284-339).
template <bool LOG>
__device__ __forceinline__ f3 vertex_nee(const DScene& sc, const IterParams& p, const Bufs& b, uint32_t pix, const Sub& s,
                                         const Bsdf& bs, int& ret)
{
    const bool logged = LOG && pix % b.mis_stride == 0;
    Rng nrng(kDomainCamera, pix, p.iter_key, s.path_length - 1, P_NEE);
    float wl = -1.f;
    int lid = 0;
    f3 ct;
    ret = direct_illumination(sc, p, ct, s, bs.pos, bs, nrng, logged ? &wl : nullptr, &lid);
    if (ret == S_OK && logged && wl >= 0.f && sc.lights[lid].type == L_AREA)
        mis_log(b, MT_NEE, s.path_length + 1, 1, pix, uint32_t(lid), wl);
    return s.throughput * ct;
}
template <bool LOG>
__device__ __forceinline__ f3 vertex_connection(const DScene& sc, const IterParams& p, const Bufs& b, uint32_t pix,
                                                const Sub& s, const Bsdf& bs, uint32_t slot, int& ret)
{
    const bool logged = LOG && pix % b.mis_stride == 0;
    float wl = -1.f;
    f3 ct;
    LVertex lv;
    load_vertex(&b.verts[slot], lv);
    ret = connect_vertices(sc, p, ct, lv, bs, bs.pos, s, logged ? &wl : nullptr);
    // logged when the light path's vertices before this one were all stored
    if (ret == S_OK && logged && wl >= 0.f && lv.path_length == slot % p.vstride + 1)
        mis_log(b, MT_BPT, lv.path_length + s.path_length + 1, lv.path_length + 1, pix, slot / p.vstride, wl);
    return s.throughput * lv.throughput * ct;
}

// Occlusion rays of a vertex: a run of the bounce's list, the first next-event estimation if nee.
struct VertexRays {
    uint32_t at, n, nee;
};

// The ray of one segment of kernel/trace_camera.cu:79-382 up to its vertex: returns whether there is
// one to shade, with its hit and scattering function. Its occlusion rays are listed in `rays`, or,
// WHOLE, traced here and added to the colour. LOG adds the MIS weight log of the sampled camera paths
// (Bufs::mislog).
template <bool WHOLE, bool LOG>
__device__ __forceinline__ bool camera_step(const DScene& sc, const IterParams& p, const Bufs& b, uint32_t pix, int bounce,
                                            Sub& s, uint32_t& pflags, f3& color, int& ret, CamCounters& cc, Hit& is,
                                            Bsdf& bs, VertexRays& rays)
{
    const bool origin_in_medium = (pflags & PF_ORIGIN_IN_MEDIUM) != 0;
    bool only_spec_surf = (pflags & PF_ONLY_SPEC_SURF) != 0;
    const uint32_t seg = s.path_length - 1;
    Rng mrng(kDomainCamera, pix, p.iter_key, seg, P_MEDIUM);
    hit_reset(is, kInf);
    VolSeg segs[kMaxSegments];
    LiteSeg lite[kMaxSegments];
    int nseg, nlite;
    bool hit;
    const unsigned rf = origin_in_medium ? kOriginInMedium : 0u;
    ret = intersect(sc, hit, s.origin, s.dir, is, s.stack, rf, segs, nseg, lite, nlite, &mrng);
    if (ret != S_OK) return false;
    const bool use_full = is.on_surface() || p.qbt == T_BEAM_SHORT || !hit;
    if ((p.build_pb2d && b.maps->med.n > 0) || (p.build_bb1d && b.maps->beam.n > 0)) {
        const VolSeg* sg = use_full ? segs : nullptr;
        const LiteSeg* lt = use_full ? nullptr : lite;
        const int ns = use_full ? nseg : nlite;
        const SegCount c0 = segment_queries<0>(sc, sg, lt, ns, rf, p.qbt, 0.f, p.piece_ball, s, pix, nullptr, nullptr);
        // piece length: the tuned length, stretched so that one ray makes at most kPiecesPerRay
        // pieces plus one per segment
        const float pl = bounce < p.bundle_bounces ? p.bundle_piece_len : p.piece_len;
        const float plen = pl > 0.f ? fmaxf(pl, c0.len / float(kPiecesPerRay)) : 0.f;
        const SegCount c1 = segment_queries<1>(sc, sg, lt, ns, rf, p.qbt, plen, p.piece_ball, s, pix, nullptr, nullptr);
        const uint32_t at = wave_alloc<4>(c1.recs, &b.qcount[128 + bounce]);
        uint32_t ptot;
        const uint32_t pbase = wave_alloc_block<6>(c1.pieces, &b.qcount[320 + bounce], ptot);
        if (c1.recs) {
            // an overflowing wave writes no pieces at all (the merge kernels skip pieces whose
            // record index is out of range)
            if (__ballot(at + c1.recs > b.seg_cap) || pbase + ptot > b.piece_cap) {
                ret = S_ERR_SEGMENTS;
                return false;
            }
            uint8_t npl[16];
            segment_queries<2>(sc, sg, lt, ns, rf, p.qbt, plen, p.piece_ball, s, pix, b.segq + at, npl);
            // Primary rays' pieces go to the wave's block piece-index-major: first every lane's
            // first piece, then every lane's second, ... so that the merge kernel, which hands 64
            // consecutive pieces to one wave, gives a wave (or bundle) the same stretch of 64
            // neighbouring rays. Scattered rays have no such neighbours: their pieces go ray by
            // ray, so that a wave's lanes walk consecutive stretches of one ray, which share
            // nodes (predefined fog room, B-B1D 77.3 -> 73.7 ms; with few pieces per ray or more
            // than the caches hold, slab room and blob grid, no difference).
            const uint32_t lane = __lane_id();
            const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
            // Bounces walked per bundle also list each j-th run (every lane's j-th piece: 64
            // neighbouring rays at similar depth) as one bundle. Runs are at most the wave's
            // pieces, so the bundle list fits the piece capacity.
            // (Lanes without a query are inactive here: the run count is the largest piece count
            // of the active lanes, found bit by bit with ballots, and the first active lane
            // allocates.)
            uint32_t ubase = 0;
            const bool bundles = b.units != nullptr && bounce < p.bundle_bounces;
            const int uleader = __ffsll((unsigned long long)__ballot(1)) - 1;
            if (bundles) {
                uint32_t ng = 0;
                for (int bit = 5; bit >= 0; bit--)
                    if (__ballot(c1.pieces >= (ng | (1u << bit)))) ng |= 1u << bit;
                if (int(lane) == uleader && ng) ubase = atomicAdd(&b.qcount[384 + bounce], ng);
                ubase = __shfl(ubase, uleader);
            }
            uint32_t start = 0, rec = 0, k = 0;
            const bool by_ray = bounce > 0 && !bundles && bounce >= p.packet_bounces;
            if (by_ray) {
                for (int bit = 0; bit < 6; bit++)
                    start += uint32_t(__popcll(__ballot((c1.pieces >> bit) & 1u) & below)) << bit;
                for (; rec < c1.recs; rec++)
                    for (k = 0; k < npl[rec]; k++)
                        b.pieces[pbase + start++] = make_uint2(at + rec, k | (uint32_t(npl[rec]) << 16));
            }
            for (uint32_t j = 0; !by_ray; j++) {
                const uint64_t mj = __ballot(c1.pieces > j);
                if (!mj) break;
                if (bundles && int(lane) == uleader && ubase + j < b.piece_cap)
                    b.units[ubase + j] = make_uint2(pbase + start, uint32_t(__popcll(mj)));
                if (c1.pieces > j) {
                    b.pieces[pbase + start + uint32_t(__popcll(mj & below))] =
                        make_uint2(at + rec, k | (uint32_t(npl[rec]) << 16));
                    if (++k == npl[rec]) {
                        k = 0;
                        rec++;
                    }
                }
                start += uint32_t(__popcll(mj));
            }
            cc.sq += c1.recs;
            cc.pieces += c1.pieces;
        }
    }
    if (!hit) {
        if (s.path_length < p.min_len) return false;
        if (sc.background_light < 0) return false;
        if (sc.media[sc.global_medium].has_attenuation) return false;
    }
    float rsf = 1.f, rsr = 1.f;
    if (nseg) {
        rsf = acc_for(segs, nseg);
        rsr = acc_rev(segs, nseg);
        s.throughput *= acc_att(segs, nseg) / rsf;
    }
    if (black_or_neg(s.throughput)) return false;
    Weights& w = s.sw.w;
    if (s.path_length > 1u) {
        const float fi = pde_factor(p, w.prev_in_medium, w.prev_specular, 1.f / rsr, w.rev_ratio, w.for_inv,
                                    w.for_ratio, s.sw.last_sin);
        w.d_bpt = s.sw.d_bpt_a * fi + s.sw.d_bpt_b;
        w.d_pde = s.sw.d_pde_a * fi + s.sw.d_pde_b;
    }
    w.d_shared /= rsf;
    w.d_bpt /= rsf;
    w.d_pde /= rsf;
    if (!hit) {
        color += s.throughput * light_radiance_mis(sc, p, sc.lights[sc.background_light], s, rsr);
        return false;
    }
    bsdf_setup(bs, s.dir, is, sc, false, relative_ior(sc, is, s.stack));
    if (!bs.valid()) return false;
    float for_ratio = 0.f, rev_ratio = 0.f;
    if (bs.in_medium()) for_ratio = rev_ratio = 1.f / sc.media[bs.id].min_pos_att;
    const f3 hitp = s.origin + s.dir * is.dist;
    bs.pos = hitp;
    pflags = is.in_medium() ? (pflags | PF_ORIGIN_IN_MEDIUM) : (pflags & ~PF_ORIGIN_IN_MEDIUM);
    {
        const float d = bs.d_factor();
        w.d_shared *= is.dist * is.dist;
        w.d_shared /= d;
        w.d_bpt /= d;
        w.d_pde /= d;
        w.for_inv = 1.f / rsf;
        w.rev_inv = 1.f / rsr;
        w.for_ratio = for_ratio;
        w.rev_ratio = rev_ratio;
    }
    const bool logged = LOG && pix % b.mis_stride == 0;
    if (is.light >= 0) {
        if (s.path_length < p.min_len) return false;
        float wl = -1.f;
        color += s.throughput * light_radiance_mis(sc, p, sc.lights[is.light], s, rsr, logged ? &wl : nullptr);
        if (logged && wl >= 0.f && sc.lights[is.light].type == L_AREA)
            mis_log(b, MT_LIGHT_HIT, s.path_length, 0, pix, uint32_t(is.light), wl);
        return false;
    }
    if (s.path_length >= p.max_len) return false;
    // the vertex's occlusion rays: next-event estimation, then the connections to the chosen light
    // path's vertices (kernel/trace_camera.cu:284-339)
    const bool connects = p.do_bpt && !bs.delta() && (bs.in_medium() || !only_spec_surf);
    const bool nee = connects && s.path_length + 1 >= p.min_len && sc.n_lights > 0;
    uint32_t slot0 = 0, n_light = 0; // the light path's vertices in reach
    bool behind = false;
    const auto skipped = [&](const float4& g) { // too short a path, or two media with a surface between
        const int fl = __float_as_int(g.z);
        const bool small = uint32_t(__float_as_int(g.w)) + 1 + s.path_length < p.min_len;
        return small || ((fl & Bsdf::IN_MEDIUM) && bs.in_medium() && __float_as_int(g.y) != bs.id &&
                         ((fl & VF_BEHIND_SURF) || behind));
    };
    s.origin = hitp; // the arriving direction stays in s.dir
    if (WHOLE && nee) {
        const f3 c = vertex_nee<LOG>(sc, p, b, pix, s, bs, ret);
        if (ret != S_OK) return false;
        color += c;
    }
    rays.nee = nee ? 1u : 0u;
    rays.n = rays.nee;
    if (connects) {
        if (bs.in_medium() && s.stack.n > 0) {
            const int m = s.stack.mat[s.stack.n - 1];
            if (m >= 0 && sc.mats[m].real) behind = true;
        }
        Rng brng(kDomainCamera, pix, p.iter_key, seg, P_BPT_PICK);
        const uint32_t lp = uint32_t(brng.next() * float(p.n_light));
        const uint32_t nv = b.nvert[lp];
        slot0 = lp * p.vstride;
        for (; n_light < nv; n_light++) {
            const float4 g = b.verts[slot0 + n_light].g;
            if (uint32_t(__float_as_int(g.w)) + 1 + s.path_length > p.max_len) break;
            if (skipped(g)) continue;
            rays.n++;
            if (WHOLE) {
                cc.conn++;
                const f3 c = vertex_connection<LOG>(sc, p, b, pix, s, bs, slot0 + n_light, ret);
                if (ret != S_OK) return false;
                color += c;
            }
        }
    }
    rays.at = 0;
    if (!WHOLE && p.do_bpt) {
        rays.at = wave_alloc<7>(rays.n, &b.qcount[512 + bounce]);
        uint32_t k = rays.at;
        if (nee) b.ctask[k++] = make_uint2(pix, kTaskNee);
        for (uint32_t i = 0; i < n_light; i++)
            if (!skipped(b.verts[slot0 + i].g)) b.ctask[k++] = make_uint2(pix, slot0 + i);
    }
    return true;
}

// the hit and scattering function of the vertex a path is at (as camera_step set them up)
__device__ __forceinline__ void load_vertex_hit(const DScene& sc, const CamHit& v, const Sub& s, Hit& is, Bsdf& bs)
{
    hit_reset(is, 0.f);
    is.normal = mk(v.a.x, v.a.y, v.a.z);
    is.mat = __float_as_int(v.a.w);
    is.shading = mk(v.b.x, v.b.y, v.b.z);
    is.med = __float_as_int(v.b.w);
    is.enter = v.c.w != 0u;
    bsdf_setup(bs, s.dir, is, sc, false, relative_ior(sc, is, s.stack));
    bs.pos = s.origin;
}

// One occlusion ray of a camera vertex with its estimator; the contribution to the path and the
// status.
template <bool LOG>
__device__ __forceinline__ f3 camera_connect(const DScene& sc, const IterParams& p, const Bufs& b, uint2 task, int& ret)
{
    const uint32_t pix = task.x;
    const PathState st = b.cstate[pix];
    Sub s;
    load_sub(st, s);
    load_stack(b.cstack, pix, s.stack);
    Hit is;
    Bsdf bs;
    load_vertex_hit(sc, b.chit[pix], s, is, bs);
    if (task.y == kTaskNee) return vertex_nee<LOG>(sc, p, b, pix, s, bs, ret);
    return vertex_connection<LOG>(sc, p, b, pix, s, bs, task.y, ret);
}

// ---- point merges (SURF, P-P3D, B-P2D) at the vertices of one wave's paths -------------------------
// A lane walks its own photon tree, one binary node per trip of a loop the whole wave makes, and the
// photons it accepts go to a queue of the wave; 64 queued pairs at a time are evaluated with full
// lanes, each lane taking the vertex it needs from its owner's registers by shuffles and adding the
// result to the owner's sum in LDS. Evaluated where they were found, two or three lanes at a time
// went through the estimator (a 112-byte record, two scattering functions and the weights) while the
// rest of the wave waited. Lanes without a walk take the oldest pending subtree of a lane that has
// one: a vertex in a dense medium lies in hundreds of sub-beam boxes, and the few such lanes of a
// wave walked them one by one (256x256 box, 27k pairs: 600 us per bounce; 485 with full-lane
// evaluation; 160 with shared walks).
struct PointQueue {
    uint32_t slot[128];  // light vertex or beam slot: < 64 pending + one accept per lane
    uint8_t owner[128];  // lane whose vertex the pair is at
    float x[128], y[128]; // B-P2D: distance along the beam, squared distance from it
    float r[64], g[64], b[64]; // per lane: sum over its pairs
    int given[64];             // subtrees handed to idle lanes, and their owners
    uint8_t given_owner[64];
};

__device__ __forceinline__ f3 shfl3(f3 v, int src) { return mk(__shfl(v.x, src), __shfl(v.y, src), __shfl(v.z, src)); }

// the parts of a path's state and scattering function that the point estimators read, from lane src
__device__ __forceinline__ void vertex_from_lane(const Sub& s, const Bsdf& bs, uint32_t pix, int src, Sub& os, Bsdf& ob,
                                                 uint32_t& opix)
{
    opix = uint32_t(__shfl(int(pix), src));
    os.path_length = uint32_t(__shfl(int(s.path_length), src));
    os.sw.w.d_shared = __shfl(s.sw.w.d_shared, src);
    os.sw.w.d_pde = __shfl(s.sw.w.d_pde, src);
    os.sw.w.for_inv = __shfl(s.sw.w.for_inv, src);
    os.sw.w.rev_inv = __shfl(s.sw.w.rev_inv, src);
    os.sw.w.for_ratio = __shfl(s.sw.w.for_ratio, src);
    os.sw.w.prev_specular = __shfl(s.sw.w.prev_specular, src);
    ob.flags = __shfl(bs.flags, src);
    ob.id = __shfl(bs.id, src);
    ob.frame.x = shfl3(bs.frame.x, src);
    ob.frame.y = shfl3(bs.frame.y, src);
    ob.frame.z = shfl3(bs.frame.z, src);
    ob.cont_prob = __shfl(bs.cont_prob, src);
    ob.local_dir_fix = shfl3(bs.local_dir_fix, src);
    ob.geom_normal = shfl3(bs.geom_normal, src);
    ob.cos_fix_geom = __shfl(bs.cos_fix_geom, src);
    ob.diff_prob = __shfl(bs.diff_prob, src);
    ob.phong_prob = __shfl(bs.phong_prob, src);
    ob.wdir = shfl3(bs.wdir, src);
    ob.pos = shfl3(bs.pos, src);
}

// Every lane of the wave calls this with the same tree, data (its points or sub-beam records) and
// radius; `want` lanes merge at their vertex. BEAM: B-P2D over sub-beams; else SURF or P-P3D over points within r2. Returns
// the sum over the lane's pairs. ok: the lane's walk did not run out of stack.
template <bool BEAM, bool LOG>
__device__ __forceinline__ f3 point_merges(const DScene& sc, const IterParams& p, const Bufs& b, PointQueue& Q, bool want,
                                           const Bvh& tree, const float4* data, float r2, uint32_t pix, const Sub& s,
                                           const Bsdf& bs, uint32_t& n_acc, bool& ok)
{
    const uint32_t lane = __lane_id();
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    Q.r[lane] = Q.g[lane] = Q.b[lane] = 0.f;
    wave_lds_sync();
    f3 hitp = bs.pos;    // the vertex of this lane's walk
    uint32_t own = lane; // and the lane it belongs to
    int stack[kBvhStack];
    int sb = 0, sp = 0, node = want && tree.n > 0 ? 0 : -1; // pending subtrees: stack[sb, sp)
    uint32_t qn = 0; // pairs queued (same value in every lane)
    for (;;) {
        const bool walking = __ballot(node >= 0) != 0;
        const uint64_t idle = __ballot(node < 0), donors = __ballot(node >= 0 && sp > sb);
        if (donors && idle) {
            const uint32_t t = min(uint32_t(__popcll(idle)), uint32_t(__popcll(donors)));
            if ((donors >> lane) & 1u) {
                const uint32_t k = uint32_t(__popcll(donors & below));
                if (k < t) {
                    Q.given[k] = stack[sb++];
                    Q.given_owner[k] = uint8_t(own);
                }
            }
            wave_lds_sync();
            if ((idle >> lane) & 1u) {
                const uint32_t k = uint32_t(__popcll(idle & below));
                if (k < t) {
                    node = Q.given[k];
                    own = Q.given_owner[k];
                    sb = sp = 0;
                }
            }
            wave_lds_sync();
            hitp = shfl3(bs.pos, int(own));
        }
        int leaf[2] = {-1, -1};
        if (node >= 0) {
            const BNode nd = tree.nodes[node];
            const bool h0 = inside(hitp, nd.lx0, nd.ly0, nd.lz0, nd.ux0, nd.uy0, nd.uz0);
            const bool h1 = inside(hitp, nd.lx1, nd.ly1, nd.lz1, nd.ux1, nd.uy1, nd.uz1);
            int next = -1;
            if (h0) {
                if (nd.c0 < 0) leaf[0] = ~nd.c0;
                else next = nd.c0;
            }
            if (h1) {
                if (nd.c1 < 0) leaf[1] = ~nd.c1;
                else if (next < 0) next = nd.c1;
                else if (sp < kBvhStack) stack[sp++] = nd.c1;
                else { // unreachable: a walk keeps at most one subtree per level, and trees have at most 64
                    ok = false;
                    next = -1;
                    sb = sp = 0;
                }
            }
            if (next < 0 && sp > sb) next = stack[--sp];
            if (sp == sb) sb = sp = 0;
            node = next;
        }
#pragma unroll
        for (int c = 0; c < 2; c++) {
            bool acc = false;
            uint32_t slot = 0;
            float x = 0.f, y = 0.f;
            if (leaf[c] >= 0) {
                if (BEAM) { // program_bp2d.cu:31-45, and the sub-beam that owns the point
                    const float4 g0 = data[3 * leaf[c]], g1 = data[3 * leaf[c] + 1];
                    const f3 bo = mk(g0.x, g0.y, g0.z), bd = mk(g1.x, g1.y, g1.z);
                    if (pred_point_beam(bo, bd, g0.w, hitp, r2) && pred_bre(x, y, bo, bd, 0.f, g0.w, hitp, r2)) {
                        const float4 g2 = data[3 * leaf[c] + 2];
                        acc = x >= g2.x && x < g2.y;
                        slot = uint32_t(__float_as_int(g1.w));
                    }
                } else {
                    const float4 pt = data[leaf[c]];
                    acc = pred_point_point(hitp, mk(pt.x, pt.y, pt.z), r2);
                    slot = uint32_t(__float_as_int(pt.w));
                }
            }
            const uint64_t m = __ballot(acc);
            if (acc) {
                const uint32_t at = qn + uint32_t(__popcll(m & below));
                Q.slot[at] = slot;
                Q.owner[at] = uint8_t(own);
                if (BEAM) {
                    Q.x[at] = x;
                    Q.y[at] = y;
                }
                n_acc++;
            }
            qn += uint32_t(__popcll(m));
            if (qn >= 64u || (c == 1 && !walking && qn > 0u)) {
                const uint32_t n = qn < 64u ? qn : 64u;
                qn -= n;
                wave_lds_sync();
                const uint32_t e = qn + (lane < n ? lane : 0u);
                const int src = int(Q.owner[e]);
                Sub os;
                Bsdf ob;
                uint32_t opix;
                vertex_from_lane(s, bs, pix, src, os, ob, opix);
                if (lane < n) {
                    f3 sum = mk(0.f);
                    const uint32_t sl = Q.slot[e];
                    const bool logged = LOG && opix % b.mis_stride == 0;
                    float wl = -1.f;
                    if (BEAM) {
                        LBeam lb;
                        load_beam(&b.beams[sl], lb);
                        eval_bp2d(sc, p, sum, os, ob, lb, Q.x[e], Q.y[e], logged ? &wl : nullptr);
                        if (logged && wl >= 0.f)
                            mis_log(b, MT_BP2D, lb.path_length + os.path_length, lb.path_length, opix, lb.path_idx, wl);
                    } else {
                        LVertex lv;
                        load_vertex(&b.verts[sl], lv);
                        eval_pp(sc, p, sum, os, ob, lv, logged ? &wl : nullptr);
                        if (logged && wl >= 0.f && sl % p.vstride + 1 == lv.path_length)
                            mis_log(b, lv.in_medium ? MT_PP3D : MT_SURF, lv.path_length + os.path_length,
                                    lv.path_length, opix, sl / p.vstride, wl);
                    }
                    if (sum.x != 0.f) atomicAdd(&Q.r[src], sum.x);
                    if (sum.y != 0.f) atomicAdd(&Q.g[src], sum.y);
                    if (sum.z != 0.f) atomicAdd(&Q.b[src], sum.z);
                }
                wave_lds_sync();
            }
        }
        if (!walking) break;
    }
    const f3 sum = mk(Q.r[lane], Q.g[lane], Q.b[lane]);
    wave_lds_sync();
    return sum;
}

// The rest of the segment at its vertex: point merges and scattering. Every lane of the wave calls
// this, `live` ones with a path; returns whether the path continues.
template <bool LOG>
__device__ __forceinline__ bool camera_shade(const DScene& sc, const IterParams& p, const Bufs& b, PointQueue& Q,
                                             bool live, uint32_t pix, const Hit& is, const Bsdf& bs, Sub& s,
                                             uint32_t& pflags, f3& color, int& ret, CamCounters& cc, float& guide_den)
{
    const bool only_spec_surf = (pflags & PF_ONLY_SPEC_SURF) != 0;
    const uint32_t seg = s.path_length - 1;
    const f3 hitp = s.origin;
    const PhotonMaps& M = *b.maps;
    const bool medium = bs.in_medium();
    const bool surf = live && p.build_surf && M.surf.n > 0 && !medium && !bs.delta() && !only_spec_surf;
    const bool pp3d = live && p.build_pp3d && M.med.n > 0 && medium && !bs.delta();
    const bool bp2d = live && p.build_bp2d && M.beam.n > 0 && medium;
    bool ok = true;
    // (a tree per call: a lane may end up with a subtree of any other lane of the wave)
    if (__ballot(surf)) {
        const f3 acc = point_merges<false, LOG>(sc, p, b, Q, surf, M.surf, M.surf_pts, p.r2_surf, pix, s, bs, cc.acc, ok);
        if (surf) {
            cc.pq++;
            color += s.throughput * p.norm_surf * acc;
        }
    }
    if (__ballot(pp3d)) {
        const f3 acc = point_merges<false, LOG>(sc, p, b, Q, pp3d, M.med, M.med_pts, p.r2_pp3d, pix, s, bs, cc.acc, ok);
        if (pp3d) {
            cc.pq++;
            color += s.throughput * p.norm_pp3d * acc;
        }
    }
    if (__ballot(bp2d)) {
        const f3 acc = point_merges<true, LOG>(sc, p, b, Q, bp2d, M.beam, M.beam_geo, p.r2_bp2d, pix, s, bs, cc.acc, ok);
        if (bp2d) {
            cc.pq++;
            color += s.throughput * p.norm_bp2d * acc;
        }
    }
    if (!live) return false;
    if (!ok) {
        ret = S_ERR_STACK;
        return false;
    }
    bool cont;
    Rng srng(kDomainCamera, pix, p.iter_key, seg, P_SCATTER);
    ret = sample_scattering(sc, p, cont, bs, hitp, is, s, srng, b.gsamp ? &guide_den : nullptr);
    if (ret != S_OK) return false;
    if (!cont) return false;
    if (bs.on_surface()) {
        if (!s.sw.w.prev_specular && (only_spec_surf || (p.techniques & T_SPECULAR_ONLY))) return false;
    } else {
        if (p.techniques & T_SPECULAR_ONLY) return false;
        if (only_spec_surf) {
            if (p.techniques & T_COMPATIBLE) pflags &= ~PF_ONLY_SPEC_SURF;
            else return false;
        }
    }
    return true;
}

// Training data of the learned proposal. A scattering of a camera path in a medium or at a
// guidable surface that continues is credited with everything the path collects after it:
// emission, next-event estimation, connections and point merges at later vertices (the path
// colour) and the P-B2D / B-B1D merges along its later segments (the merge colour). With
// throughput T before the scattering, scattering function f, cosine cos, continuation
// probability cp and sampling pdf p, the path carries T f cos / (p cp) onward, so
// lum(collected after) cp / lum(T f cos) estimates L_i / p: the incident radiance along the
// sampled direction (the part the path's later vertices collect under their MIS weights) over
// its pdf, the weight of the KL gradient that fits the proposal's radiance mixture to L_i. The sample is (position, scattered direction) with
// the arrival inputs zero: the mixture depends on the position only.
//
// The scattering at vertex k waits in the path's pending slot until the next bounce, where the
// merges along the segment it sampled have run; it then enters the pool with the snapshot
// lum(path colour after vertex k) + lum(merge colour before segment k + 1's merges).
// k_guide_finalise turns snapshots into weights once the iteration's colours are final.
// Inlined: a call taking the kernel's scene and buffer arguments by reference would copy them
// to scratch memory for the whole bounce kernel.
__device__ __forceinline__ void guide_emit_pending(const Bufs& b, uint32_t pix)
{
    float* pend = b.gpend + size_t(pix) * kGuidePend;
    bool emit = false;
    float rec[kGuideRaw];
    if (pend[9] > 0.f) {
        for (int k = 0; k < 10; k++) rec[k] = pend[k];
        rec[10] = pend[10] + luminance(mk(b.mcolor[3 * pix], b.mcolor[3 * pix + 1], b.mcolor[3 * pix + 2]));
        rec[11] = __uint_as_float(pix);
        emit = true;
        pend[9] = 0.f;
    }
    const uint64_t m = __ballot(emit);
    if (m) { // wave-aggregated append
        const uint32_t lane = __lane_id();
        const int leader = __ffsll((unsigned long long)m) - 1;
        uint32_t base = 0;
        if (int(lane) == leader) base = atomicAdd(b.gcount, uint32_t(__popcll(m)));
        base = __shfl(base, leader);
        const uint32_t at = base + uint32_t(__popcll(m & (lane == 0 ? 0ull : (~0ull >> (64 - lane)))));
        if (emit && at < b.gcap)
            for (int k = 0; k < kGuideRaw; k++) b.graw[size_t(at) * kGuideRaw + k] = rec[k];
    }
}

// a scattering in a medium or at a guidable surface that continues becomes the pending record
__device__ __forceinline__ void guide_pend_sample(const DScene& sc, const Bufs& b, uint32_t pix, f3 color, f3 origin,
                                                  f3 dir, float den)
{
    if (!(den > 0.f)) return;
    float* pend = b.gpend + size_t(pix) * kGuidePend;
    const DGuide& g = sc.guide;
    const float inv_res = 1.f / float(g.res);
    pend[0] = (origin.x - g.lo.x) * g.inv_cell.x * inv_res;
    pend[1] = (origin.y - g.lo.y) * g.inv_cell.y * inv_res;
    pend[2] = (origin.z - g.lo.z) * g.inv_cell.z * inv_res;
    pend[3] = pend[4] = pend[5] = 0.f;
    pend[6] = dir.x;
    pend[7] = dir.y;
    pend[8] = dir.z;
    pend[9] = den;
    pend[10] = luminance(color);
}

// pool of raw records -> training samples (10 floats: position, arrival, scattered, weight) with
// a positive weight, written to the sample ring after the splat, when path and merge colours are
// final. Counters: gcount[1] samples kept this iteration, gcount[2] the ring's write position
// (modulo gring), gcount[3] its fill. At most gring samples are written per iteration, so no ring
// slot is written twice in one launch.
__global__ void __launch_bounds__(256) k_guide_finalise(Bufs b)
{
    const uint32_t n = min(b.gcount[0], b.gcap);
    const uint32_t start = b.gcount[2];
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const float* r = b.graw + size_t(i) * kGuideRaw;
        const uint32_t pix = __float_as_uint(r[11]);
        const float fin = luminance(b.cstate[pix].color) +
                          luminance(mk(b.mcolor[3 * pix], b.mcolor[3 * pix + 1], b.mcolor[3 * pix + 2]));
        const float w = (fin - r[10]) / r[9];
        const bool keep = w > 0.f && isfinite(w);
        const uint64_t m = __ballot(keep);
        if (!m) continue;
        const uint32_t lane = __lane_id();
        const int leader = __ffsll((unsigned long long)m) - 1;
        uint32_t base = 0;
        if (int(lane) == leader) base = atomicAdd(b.gcount + 1, uint32_t(__popcll(m)));
        base = __shfl(base, leader);
        const uint32_t at = base + uint32_t(__popcll(m & (lane == 0 ? 0ull : (~0ull >> (64 - lane)))));
        if (keep && at < b.gring) {
            float* o = b.gsamp + size_t((uint64_t(start) + at) % b.gring) * 10;
            for (int k = 0; k < 9; k++) o[k] = r[k];
            o[9] = w;
        }
    }
}

// advances the ring past this iteration's samples (one thread, after k_guide_finalise)
__global__ void k_guide_ring_advance(Bufs b)
{
    const uint32_t kept = min(b.gcount[1], b.gring);
    b.gcount[2] = uint32_t((uint64_t(b.gcount[2]) + kept) % b.gring);
    b.gcount[3] = min(b.gcount[3] + kept, b.gring);
}

template <bool LOG>
__device__ __forceinline__ void camera_bounce_body(const DScene& sc, const Bufs& b, int bounce, uint32_t vb, uint32_t waves)
{
    const IterParams& p = *b.params;
    const uint32_t i = wave_entry((vb * blockDim.x + threadIdx.x) >> 6, b.qcount[64 + bounce], waves);
    if (i == ~0u) return;
    const uint32_t pix = b.queue[bounce & 1][i];
    PathState st = b.cstate[pix];
    Sub s;
    load_sub(st, s);
    load_stack(b.cstack, pix, s.stack);
    uint32_t pflags = st.flags;
    f3 color = st.color;
    int ret = S_OK;
    CamCounters cc;
    Hit is;
    Bsdf bs;
    VertexRays rays;
    bool shade = camera_step<false, LOG>(sc, p, b, pix, bounce, s, pflags, color, ret, cc, is, bs, rays);
    if (ret != S_OK) {
        shade = false;
        stat_add(b.stats, STAT_ERRORS, 1);
    }
    if (b.gsamp) guide_emit_pending(b, pix);
    stat_add(b.stats, STAT_SEG_Q, cc.sq);
    stat_add(b.stats, STAT_SEG_PIECES, cc.pieces);
    st.color = color;
    if (shade) {
        st.flags = pflags;
        save_sub(st, s);
        store_stack(b.cstack, pix, s.stack);
        CamHit vertex;
        vertex.a = make_float4(is.normal.x, is.normal.y, is.normal.z, __int_as_float(is.mat));
        vertex.b = make_float4(is.shading.x, is.shading.y, is.shading.z, __int_as_float(is.med));
        vertex.c = make_uint4(rays.at, rays.n, rays.nee, is.enter ? 1u : 0u);
        b.chit[pix] = vertex;
    }
    b.cstate[pix] = st;
    queue_append(shade, pix, b.queue_shade, &b.qcount[640 + bounce]);
}

// One job's occlusion rays of one bounce: each wave takes 1 to 64 at a time (wave_share) until none are left.
template <bool LOG>
__device__ __forceinline__ void camera_connect_body(const DScene& sc, const Bufs& b, int bounce, uint32_t wave, uint32_t waves,
                                                    uint32_t share)
{
    const IterParams& p = *b.params;
    const uint32_t lane = __lane_id();
    const uint32_t n = b.qcount[512 + bounce];
    uint32_t* head = &b.qcount[576 + bounce];
    const uint32_t take = wave_share(n, share), given = waves * take;
    // the first entries are dealt out, the rest taken from the counter
    for (uint32_t base = wave * take; base < n;) {
        if (lane < take && base + lane < n) {
            int ret = S_OK;
            const f3 c = camera_connect<LOG>(sc, p, b, b.ctask[base + lane], ret);
            b.ctask_res[base + lane] = make_float4(c.x, c.y, c.z, __int_as_float(ret));
        }
        if (given >= n) break;
        if (lane == 0) base = given + atomicAdd(head, take);
        base = __shfl(base, 0);
    }
}

template <bool LOG>
__device__ __forceinline__ void camera_shade_body(const DScene& sc, const Bufs& b, int bounce, uint32_t vb, PointQueue& Q)
{
    const IterParams& p = *b.params;
    const uint32_t i = vb * blockDim.x + threadIdx.x;
    const uint32_t n = b.qcount[640 + bounce];
    if (i - __lane_id() >= n) return; // the whole wave
    const bool has = i < n;
    const uint32_t pix = has ? b.queue_shade[i] : 0u;
    PathState st;
    Sub s;
    s.stack.n = 0;
    s.path_length = 1;
    s.origin = s.dir = mk(0.f);
    uint32_t pflags = 0;
    f3 color = mk(0.f);
    if (has) {
        st = b.cstate[pix];
        load_sub(st, s);
        load_stack(b.cstack, pix, s.stack);
        pflags = st.flags;
        color = st.color;
    }
    int ret = S_OK;
    CamCounters cc;
    float guide_den = 0.f;
    Hit is;
    Bsdf bs;
    bs.flags = 0;
    bool live = has;
    if (has) { // the occlusion rays' contributions in list order
        const CamHit vertex = b.chit[pix];
        for (uint32_t k = 0; k < vertex.c.y; k++) {
            const float4 r = b.ctask_res[vertex.c.x + k];
            if (k >= vertex.c.z) cc.conn++;
            ret = __float_as_int(r.w);
            if (ret != S_OK) { // as when the ray was traced here: the path ends
                live = false;
                break;
            }
            color += mk(r.x, r.y, r.z);
        }
        load_vertex_hit(sc, vertex, s, is, bs);
    }
    bool cont = camera_shade<LOG>(sc, p, b, Q, live, pix, is, bs, s, pflags, color, ret, cc, guide_den);
    if (ret != S_OK) {
        cont = false;
        stat_add(b.stats, STAT_ERRORS, 1);
    }
    if (b.gsamp && cont) guide_pend_sample(sc, b, pix, color, s.origin, s.dir, guide_den);
    stat_add(b.stats, STAT_BPT_CONN, cc.conn);
    stat_add(b.stats, STAT_POINT_Q, cc.pq);
    stat_add(b.stats, STAT_ACCEPT, cc.acc);
    if (has) {
        st.color = color;
        if (cont) {
            s.path_length++;
            st.flags = pflags;
            save_sub(st, s);
            store_stack(b.cstack, pix, s.stack);
        }
        b.cstate[pix] = st;
    }
    queue_append(cont, pix, b.queue[(bounce + 1) & 1], &b.qcount[64 + bounce + 1]);
}

// All of a segment by one lane; the wave shares its point merges. Two waves per SIMD: at four it spills
// 550 registers a lane, and the predefined scenes' frames took 1.2 to 1.4 times as long.
template <bool LOG>
__device__ __forceinline__ void camera_whole_body(const DScene& sc, const Bufs& b, int bounce, uint32_t wave, uint32_t waves,
                                                  PointQueue& Q)
{
    const IterParams& p = *b.params;
    const uint32_t i = wave_entry(wave, b.qcount[64 + bounce], waves);
    const bool has = i != ~0u;
    if (!__ballot(has)) return;
    uint32_t pix = 0;
    PathState st;
    Sub s;
    s.stack.n = 0;
    s.path_length = 1;
    s.origin = s.dir = mk(0.f);
    uint32_t pflags = 0;
    f3 color = mk(0.f);
    int ret = S_OK;
    CamCounters cc;
    float guide_den = 0.f;
    Hit is;
    Bsdf bs;
    bs.flags = 0;
    bool live = false;
    if (has) {
        pix = b.queue[bounce & 1][i];
        st = b.cstate[pix];
        load_sub(st, s);
        load_stack(b.cstack, pix, s.stack);
        pflags = st.flags;
        color = st.color;
        VertexRays rays;
        live = camera_step<true, LOG>(sc, p, b, pix, bounce, s, pflags, color, ret, cc, is, bs, rays);
        if (b.gsamp) guide_emit_pending(b, pix);
    }
    bool cont = camera_shade<LOG>(sc, p, b, Q, live, pix, is, bs, s, pflags, color, ret, cc, guide_den);
    if (ret != S_OK) {
        cont = false;
        stat_add(b.stats, STAT_ERRORS, 1);
    }
    if (b.gsamp && cont) guide_pend_sample(sc, b, pix, color, s.origin, s.dir, guide_den);
    stat_add(b.stats, STAT_SEG_Q, cc.sq);
    stat_add(b.stats, STAT_SEG_PIECES, cc.pieces);
    stat_add(b.stats, STAT_BPT_CONN, cc.conn);
    stat_add(b.stats, STAT_POINT_Q, cc.pq);
    stat_add(b.stats, STAT_ACCEPT, cc.acc);
    if (has) {
        st.color = color;
        if (cont) {
            s.path_length++;
            st.flags = pflags;
            save_sub(st, s);
            store_stack(b.cstack, pix, s.stack);
        }
        b.cstate[pix] = st;
    }
    queue_append(cont, pix, b.queue[(bounce + 1) & 1], &b.qcount[64 + bounce + 1]);
}

// one wave per block
template <bool LOG>
__global__ void __launch_bounds__(64, 2) k_camera_whole(DScene sc, Bufs b, int bounce, uint32_t waves)
{
    __shared__ PointQueue pq;
    camera_whole_body<LOG>(sc, b, bounce, blockIdx.x, waves, pq);
}

template <bool LOG, int OCC>
__global__ void __launch_bounds__(256, OCC) k_camera_bounce(DScene sc, Bufs b, int bounce, uint32_t waves)
{
    camera_bounce_body<LOG>(sc, b, bounce, blockIdx.x, waves);
}

template <bool LOG, int OCC>
__global__ void __launch_bounds__(256, OCC) k_camera_connect(DScene sc, Bufs b, int bounce, uint32_t share)
{
    camera_connect_body<LOG>(sc, b, bounce, blockIdx.x, gridDim.x, share);
}

// one wave per block
template <bool LOG, int OCC>
__global__ void __launch_bounds__(64, OCC) k_camera_shade(DScene sc, Bufs b, int bounce)
{
    __shared__ PointQueue pq;
    camera_shade_body<LOG>(sc, b, bounce, blockIdx.x, pq);
}

__global__ void __launch_bounds__(256, 4) k_camera_bounce_batch(const BatchJob* jobs, const uint2* bmap, int bounce, uint32_t share)
{
    const uint2 m = bmap[blockIdx.x];
    if (jobs[m.x].b.params->whole) return;
    const uint32_t own = (jobs[m.x].b.params->n_pixels + 255u) / 256u * 4u;
    camera_bounce_body<false>(jobs[m.x].sc, jobs[m.x].b, bounce, m.y, min(share, own));
}

// every job's rays: the blocks walk the jobs in turn from their own, as in the segment merges
__global__ void __launch_bounds__(256, 4) k_camera_connect_batch(const BatchJob* jobs, uint32_t njobs, int bounce)
{
    for (uint32_t t = 0; t < njobs; t++) {
        const uint32_t j = (blockIdx.x + t) % njobs;
        const BatchJob& J = jobs[j];
        if (bounce >= int(J.b.params->max_len) || J.b.params->whole) continue;
        // the jobs' first entries go to different waves
        const uint32_t wave = (blockIdx.x + j * (gridDim.x / njobs)) % gridDim.x;
        camera_connect_body<false>(J.sc, J.b, bounce, wave, gridDim.x, gridDim.x / 2u / njobs);
    }
}

__global__ void __launch_bounds__(256, 4) k_camera_shade_batch(const BatchJob* jobs, const uint2* bmap, int bounce)
{
    __shared__ PointQueue pq[4];
    const uint2 m = bmap[blockIdx.x];
    if (jobs[m.x].b.params->whole) return;
    camera_shade_body<false>(jobs[m.x].sc, jobs[m.x].b, bounce, m.y, pq[threadIdx.x >> 6]);
}

__global__ void __launch_bounds__(256, 2) k_camera_whole_batch(const BatchJob* jobs, const uint2* bmap, int bounce, uint32_t share)
{
    __shared__ PointQueue pq[4];
    const uint2 m = bmap[blockIdx.x];
    if (!jobs[m.x].b.params->whole) return;
    const uint32_t own = (jobs[m.x].b.params->n_pixels + 255u) / 256u * 4u;
    camera_whole_body<false>(jobs[m.x].sc, jobs[m.x].b, bounce, m.y * 4u + (threadIdx.x >> 6), min(share, own),
                             pq[threadIdx.x >> 6]);
}

// adds every camera path's colour at its jittered raster position (frame_buffer.cuh:35-44)
__device__ __forceinline__ void camera_splat_body(const Bufs& b, float res_x, float res_y, uint32_t vb)
{
    const IterParams& p = *b.params;
    const uint32_t pix = vb * 256u + threadIdx.x;
    if (pix >= p.n_pixels) return;
    const PathState& st = b.cstate[pix];
    if (!(st.sx >= 0.f && st.sx < res_x && st.sy >= 0.f && st.sy < res_y)) return;
    const size_t tgt = size_t(int(st.sx)) + size_t(int(st.sy)) * size_t(res_x);
    const f3 c = st.color + mk(b.mcolor[3 * pix], b.mcolor[3 * pix + 1], b.mcolor[3 * pix + 2]);
    atomicAdd(&b.fb32[3 * tgt], c.x);
    atomicAdd(&b.fb32[3 * tgt + 1], c.y);
    atomicAdd(&b.fb32[3 * tgt + 2], c.z);
}

__global__ void __launch_bounds__(256) k_camera_splat(Bufs b, float res_x, float res_y)
{
    camera_splat_body(b, res_x, res_y, blockIdx.x);
}

// folds the FP32 iteration buffer into the FP64 cross-iteration accumulator, unless the iteration
// overflowed a photon list (then it is discarded and rendered again)
__global__ void __launch_bounds__(256) k_accumulate(const float* fb32, double* accum, uint32_t n, const uint32_t* ovf)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && *ovf == 0u) accum[i] += double(fb32[i]);
}

// splat (phase 0, a block per 256 pixels of each job) and accumulate (phase 1, a block per 256
// values of each job) of every job; bmap gives each block its job and its block within the job.
// A job's accumulate must see all of its splat, so the phases are two launches.
__global__ void __launch_bounds__(256) k_finish_batch(const BatchJob* jobs, const uint2* bmap, int phase)
{
    const uint2 m = bmap[blockIdx.x];
    const BatchJob& J = jobs[m.x];
    if (phase == 0) {
        camera_splat_body(J.b, J.fres_x, J.fres_y, m.y);
    } else {
        const uint32_t i = m.y * 256u + threadIdx.x;
        const uint32_t n = 3u * J.b.params->n_pixels;
        if (i < n && *J.ovf == 0u) J.b.accum[i] += double(J.b.fb32[i]);
    }
}

void launch_camera_generate(const DScene& sc, const IterParams& p, const Bufs& b, hipStream_t s)
{
    const uint32_t res_x = uint32_t(sc.cam.res_x);
    const uint32_t res_y = (p.n_pixels + res_x - 1) / res_x;
    const uint32_t tiles_x = (res_x + 15) / 16, tiles_y = (res_y + 15) / 16;
    hipLaunchKernelGGL(k_camera_generate, dim3(tiles_x * tiles_y), dim3(256), 0, s, sc, b, res_x, tiles_x);
}

void launch_camera_generate_batch(const BatchJob* jobs, const uint2* bmap, uint32_t blocks, hipStream_t s)
{
    if (blocks) hipLaunchKernelGGL(k_camera_generate_batch, dim3(blocks), dim3(256), 0, s, jobs, bmap);
}

uint32_t compute_units()
{
    static const uint32_t n = [] {
        int dev = 0, cus = 0;
        (void)hipGetDevice(&dev);
        (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        return uint32_t(cus > 0 ? cus : 1);
    }();
    return n;
}
// waves that share a list of at most cap entries (wave_share), given a kernel's waves per CU
uint32_t share_waves(uint32_t cap, uint32_t per_cu) { return std::min(cap, compute_units() * per_cu); }

void launch_camera_bounce_batch(const BatchJob* jobs, uint32_t njobs, const uint2* bmap, uint32_t blocks, int bounce,
                                bool any_whole, bool any_split, hipStream_t s)
{
    if (!blocks) return;
    const uint32_t share = bounce > 0 ? share_waves(~0u, kBounceShare) * 2u / njobs : 0u;
    if (any_whole) hipLaunchKernelGGL(k_camera_whole_batch, dim3(blocks), dim3(256), 0, s, jobs, bmap, bounce, share);
    if (any_split) {
        hipLaunchKernelGGL(k_camera_bounce_batch, dim3(blocks), dim3(256), 0, s, jobs, bmap, bounce, share);
        hipLaunchKernelGGL(k_camera_connect_batch, dim3(compute_units() * 16u), dim3(64), 0, s, jobs, njobs, bounce);
        hipLaunchKernelGGL(k_camera_shade_batch, dim3(blocks), dim3(256), 0, s, jobs, bmap, bounce);
    }
}

void launch_camera_finish_batch(const BatchJob* jobs, const uint2* bmap_pix, uint32_t blocks_pix, const uint2* bmap_acc,
                                uint32_t blocks_acc, hipStream_t s)
{
    if (blocks_pix) hipLaunchKernelGGL(k_finish_batch, dim3(blocks_pix), dim3(256), 0, s, jobs, bmap_pix, 0);
    if (blocks_acc) hipLaunchKernelGGL(k_finish_batch, dim3(blocks_acc), dim3(256), 0, s, jobs, bmap_acc, 1);
}

// Camera bounces' kernels come at two occupancies: at 4 waves per SIMD (128 registers) they spill, 30 to
// 200 registers a lane; at 2 and 3 none does. A frame that fits the chip at 4 gains nothing from the
// higher one and pays for the spills at every bounce (ms per pass, 4 -> 2: small box 3.84 -> 3.63, box
// 31.9 -> 30.6, plain BPT over 83k triangles at 640x360 16.8 -> 16.4; over 70 small frames of all kinds
// 5%). Larger ones need the waves: blob grid at 1280x720 105 ms, 109 with the second form.
constexpr uint32_t kLooseWaves = 16; // per CU: frames of at most so many waves take the second form

template <bool LOG, int OCC>
static void launch_split(const DScene& sc, const IterParams& p, const Bufs& b, int bounce, uint32_t waves, hipStream_t s)
{
    const dim3 grid((std::max((p.n_pixels + 63) / 64, waves) * 64u + p.block - 1) / p.block), block(p.block);
    hipLaunchKernelGGL((k_camera_bounce<LOG, OCC>), grid, block, 0, s, sc, b, bounce, waves);
    if (p.do_bpt) {
        // a tiny frame has few rays: launching the waves that find none would take longer than the rays
        // (small box, 12 bounces: 4.04 -> 3.84 ms per pass)
        const uint32_t blocks = std::min(std::max(p.n_pixels / 8u, compute_units()), compute_units() * 4u * OCC);
        hipLaunchKernelGGL((k_camera_connect<LOG, OCC>), dim3(blocks), dim3(64), 0, s, sc, b, bounce,
                           std::min(blocks, compute_units() * kConnectShare));
    }
    hipLaunchKernelGGL((k_camera_shade<LOG, OCC>), dim3((p.n_pixels + 63) / 64), dim3(64), 0, s, sc, b, bounce);
}

template <bool LOG>
static void launch_bounce(const DScene& sc, const IterParams& p, const Bufs& b, int bounce, hipStream_t s)
{
    // primary rays stay 64 to a wave: neighbours' segments are bundled by the wave that wrote them
    const auto shared = [&](uint32_t per_cu) { return bounce > 0 ? share_waves(p.n_pixels, per_cu) : 0u; };
    if (p.whole) {
        const uint32_t waves = shared(kWholeShare);
        hipLaunchKernelGGL(k_camera_whole<LOG>, dim3(std::max((p.n_pixels + 63) / 64, waves)), dim3(64), 0, s, sc, b, bounce,
                           waves);
    } else if (LOG || (p.n_pixels + 63) / 64 <= compute_units() * kLooseWaves) {
        launch_split<LOG, 2>(sc, p, b, bounce, shared(kLooseShare), s);
    } else {
        launch_split<false, 4>(sc, p, b, bounce, shared(kBounceShare), s);
    }
}

void launch_camera_bounce(const DScene& sc, const IterParams& p, const Bufs& b, int bounce, hipStream_t s)
{
    if (b.mislog) launch_bounce<true>(sc, p, b, bounce, s);
    else launch_bounce<false>(sc, p, b, bounce, s);
}

void launch_camera_finish(const IterParams& p, const Bufs& b, float res_x, float res_y, const uint32_t* ovf,
                          hipStream_t s)
{
    hipLaunchKernelGGL(k_camera_splat, dim3((p.n_pixels + 255) / 256), dim3(256), 0, s, b, res_x, res_y);
    const uint32_t n = 3 * p.n_pixels;
    hipLaunchKernelGGL(k_accumulate, dim3((n + 255) / 256), dim3(256), 0, s, b.fb32, b.accum, n, ovf);
    if (b.gsamp) {
        hipLaunchKernelGGL(k_guide_finalise, dim3(1024), dim3(256), 0, s, b);
        hipLaunchKernelGGL(k_guide_ring_advance, dim3(1), dim3(1), 0, s, b);
    }
}

} // namespace upbp
