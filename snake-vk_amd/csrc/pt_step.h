// Device side of the wavefront path tracer shared by the single-scene and the
// batched passes: the shade step of one path vertex and the shadow step.
#pragma once

#include "render_modes.h"
#include "snkpt_dev.h"
#include "trace_group.h"

namespace snkpt {

// Scene source of a launch with one scene: the stream id of a path's RNG is
// its path index (the pixel for camera paths).
struct SceneOne {
    SceneDev S;
    __device__ __forceinline__ const SceneDev& at(uint32_t) const { return S; }
    __device__ __forceinline__ uint32_t stream(uint32_t path) const { return path; }
};

// What one path vertex produced.
struct VertexOut {
    bool ext = false, sh = false, q = false;
    bool emit = false;  // c_emit is added to the path's radiance now
    V3 c_emit, ext_o, ext_d, sh_o, sh_d, sh_c;
    float sh_t = 0.0f;
    float4 thr4;        // throughput | pdf after the vertex (unchanged when the path ends here)
    float4 qthr;        // throughput arriving at a cache query vertex
    float qs[13];
};

// The unbiased path tracer at one hit (KIND: see ShadeHooks): emission under
// MIS, cache query or training record, NEE (power-heuristic MIS against BRDF
// sampling), BRDF continuation with Russian roulette.  Eight uniforms are
// drawn at every non-emissive vertex whether used or not, so the wavefront
// and the path kernels consume the stream identically.  rad_now: the
// path's radiance before this vertex (read for training records only).
template <int KIND>
__device__ __forceinline__ void path_vertex_surf(const SceneDev& S, const PtParams& P, const ShadeHooks& H,
                                                 uint32_t path, uint32_t bounce, V3 dir, float t, const Surf& s,
                                                 float4 thr4, Rng& rng, float4 rad_now, VertexOut& o) {
    o.thr4 = thr4;
    const V3 thr{thr4.x, thr4.y, thr4.z};
    if (s.emissive) {
        // MIS against the NEE of the previous vertex; a negative stored pdf
        // marks a vertex whose direct light came from ReSTIR (weight 0 here)
        float w = 1.0f;
        if (bounce > 0) w = thr4.w < 0.0f ? 0.0f : power_heuristic(thr4.w, light_pdf(S, s.gid, s.ng, dir, t));
        o.c_emit = mul(thr, s.le) * w;
        o.emit = true;
        return;
    }
    // the BRDF probe of an indirect query vertex (H.mis) only looks for emission
    if (KIND == 1 && H.mis && bounce == H.query_at + 1) return;
    const V3 wo = dir * -1.0f;
    const bool query = KIND == 1 && bounce == H.query_at;
    if (query) {
        o.q = true;
        o.qthr = thr4;
        float q[13] = {s.p.x, s.p.y, s.p.z, wo.x, wo.y, wo.z, s.ns.x, s.ns.y, s.ns.z, s.m.roughness,
                       s.m.albedo.x, s.m.albedo.y, s.m.albedo.z};
#pragma unroll
        for (int k = 0; k < 13; ++k) o.qs[k] = q[k];
        // terminate into the radiance cache: L_o(x, wo) from the network
        if (!H.indirect) return;
        // indirect split: direct light here by NEE alone (or, with H.mis, NEE and a
        // traced BRDF sample under the power heuristic), the cache answers the rest
    }
    if (KIND == 2 && bounce < H.max_rec) {
        // training record: sample fields, radiance so far, throughput at arrival
        float* r = H.rec + ((size_t)path * H.max_rec + bounce) * kRecFloats;
        float q[kRecFloats] = {s.p.x, s.p.y, s.p.z, wo.x, wo.y, wo.z, s.ns.x, s.ns.y, s.ns.z,
                               s.m.roughness, s.m.albedo.x, s.m.albedo.y, s.m.albedo.z, rad_now.x, rad_now.y,
                               rad_now.z, thr.x, thr.y, thr.z, 0.0f};
#pragma unroll
        for (int k = 0; k < kRecFloats; ++k) r[k] = q[k];
        H.nrec[path] = bounce + 1;
    }
    float u0 = rng.uniform(), u1 = rng.uniform(), u2 = rng.uniform(), u3 = rng.uniform();
    float ul = rng.uniform(), us1 = rng.uniform(), us2 = rng.uniform(), urr = rng.uniform();
    // an indirect query vertex with H.mis continues one BRDF sample as the probe
    const bool probe = KIND == 1 && query && H.mis;
    const bool last = (bounce + 1 >= P.max_depth || query) && !probe;
    // next-event estimation
    LightSample ls = sample_direct(S, s.p, u0, u1, u2, u3);
    if (ls.ok) {
        float cs = dot(s.ns, ls.wi);
        if (cs > 0.0f && dot(s.ng, ls.wi) > 0.0f) {
            const V3 h = brdf_half(s.m, wo, ls.wi);
            V3 f = brdf_eval(s.m, brdf_view(s.m, s.ns, wo), s.ns, wo, ls.wi, h);
            float w = (last || ls.delta) ? 1.0f : power_heuristic(ls.pdf, brdf_pdf(s.m, s.ns, wo, ls.wi, h));
            o.sh_c = mul(mul(thr, f), ls.le) * (cs * w / ls.pdf);
            if (o.sh_c.x > 0.0f || o.sh_c.y > 0.0f || o.sh_c.z > 0.0f) {
                o.sh = true;
                shadow_segment(s.p, s.ng, s.eps, ls.wi, ls.dist, o.sh_o, o.sh_d, o.sh_t);
            }
        }
    }
    // continuation
    V3 wi;
    if (!last && brdf_sample(s.m, s.ns, wo, ul, us1, us2, wi) && dot(s.ng, wi) > 0.0f) {
        const V3 h = brdf_half(s.m, wo, wi);
        float pdf = brdf_pdf(s.m, s.ns, wo, wi, h);
        if (pdf > 0.0f) {
            V3 f = brdf_eval(s.m, brdf_view(s.m, s.ns, wo), s.ns, wo, wi, h);
            V3 nt = mul(thr, f) * (dot(s.ns, wi) / pdf);
            bool alive = nt.x > 0.0f || nt.y > 0.0f || nt.z > 0.0f;
            if (alive && P.rr_start > 0 && bounce + 1 >= P.rr_start) {
                float q = fminf(fmaxf(fmaxf(nt.x, nt.y), nt.z), 0.95f);
                if (urr >= q)
                    alive = false;
                else
                    nt = nt * (1.0f / q);
            }
            if (alive) {
                o.ext = true;
                o.ext_o = s.p + s.ng * s.eps;
                o.ext_d = wi;
                o.thr4 = make_float4(nt.x, nt.y, nt.z, pdf);
            }
        }
    }
}

template <int KIND>
__device__ __forceinline__ void path_vertex(const SceneDev& S, const PtParams& P, const ShadeHooks& H, uint32_t path,
                                            uint32_t bounce, V3 dir, float t, uint32_t inst, uint32_t prim, float hu,
                                            float hv, float4 thr4, Rng& rng, float4 rad_now, VertexOut& o) {
    const Surf s = surface_at(S, dir, inst, prim, hu, hv);
    path_vertex_surf<KIND>(S, P, H, path, bounce, dir, t, s, thr4, rng, rad_now, o);
}

// Queue appends of one path vertex: continuation ray, shadow ray and (KIND 1)
// cache query.  Every thread of the block calls it (block-wide appends).
template <int KIND, int BLOCK>
__device__ __forceinline__ void vertex_appends(const VertexOut& o, uint32_t path, uint32_t bounce, const Rng& rng,
                                               const Queue& out, const ShadowQueue& sq, const PathState& ps,
                                               uint32_t* __restrict__ counts, uint32_t nxt, const ShadeHooks& H,
                                               uint32_t* lds_app) {
    uint32_t slot = block_append<BLOCK>(o.ext, &counts[nxt], lds_app);
    if (o.ext) {
        out.org[slot] = make_float4(o.ext_o.x, o.ext_o.y, o.ext_o.z, 0.0f);
        out.dir[slot] = make_float4(o.ext_d.x, o.ext_d.y, o.ext_d.z, 1e30f);
        out.path[slot] = path;
        ps.thr[path] = o.thr4;
        ps.rng[path] = make_uint2((uint32_t)rng.state, (uint32_t)(rng.state >> 32));
        ps.bounce[path] = bounce + 1;
    }
    uint32_t sslot = block_append<BLOCK>(o.sh, &counts[2], lds_app);
    if (o.sh) {
        sq.org[sslot] = make_float4(o.sh_o.x, o.sh_o.y, o.sh_o.z, 0.0f);
        sq.dir[sslot] = make_float4(o.sh_d.x, o.sh_d.y, o.sh_d.z, o.sh_t);
        sq.contrib[sslot] = make_float4(o.sh_c.x, o.sh_c.y, o.sh_c.z, __uint_as_float(path));
    }
    if (KIND == 1) {
        uint32_t qslot = block_append<BLOCK>(o.q, H.q_count, lds_app);
        if (o.q) {
            float* q = H.q_samples + (size_t)qslot * 16;
#pragma unroll
            for (int k = 0; k < 13; ++k) q[k] = o.qs[k];
            q[13] = q[14] = q[15] = 0.0f;
            H.q_meta[qslot] = make_float4(o.qthr.x, o.qthr.y, o.qthr.z, __uint_as_float(path));
        }
    }
}

// One path vertex of the wavefront path tracer for queue entry i.  Every
// thread of the block calls it (the queue appends are block-wide); `valid`
// marks threads with an entry.
template <int KIND, int BLOCK, class SS>
__device__ __forceinline__ void shade_step(const SS& ss, const PtParams& P, const Queue& in, const HitArrays& hit,
                                           const Queue& out, const ShadowQueue& sq, const PathState& ps,
                                           float4* __restrict__ rad, uint32_t* __restrict__ counts, uint32_t nxt,
                                           const ShadeHooks& H, uint32_t i, bool valid, uint32_t* lds_app) {
    VertexOut o;
    uint32_t path = 0, bounce = 0;
    Rng rng{0, 0};
    if (valid) {
        path = in.path[i];
        const SceneDev& S = ss.at(path);
        const float4 thr4 = ps.thr[path];
        uint2 rs = ps.rng[path];
        rng.state = (uint64_t)rs.x | ((uint64_t)rs.y << 32);
        rng.inc = ((uint64_t)ss.stream(path) << 1u) | 1u;
        bounce = ps.bounce[path];
        const float t = hit.t[i];
        if (t >= 0.0f) {
            const float4 dq = in.dir[i];
            const float4 rn = KIND == 2 ? rad[path] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            path_vertex<KIND>(S, P, H, path, bounce, V3{dq.x, dq.y, dq.z}, t, hit.inst[i], hit.prim[i], hit.u[i],
                              hit.v[i], thr4, rng, rn, o);
            if (o.emit) {
                float4 r = rad[path];
                rad[path] = make_float4(r.x + o.c_emit.x, r.y + o.c_emit.y, r.z + o.c_emit.z, r.w);
            }
        }
    }
    vertex_appends<KIND, BLOCK>(o, path, bounce, rng, out, sq, ps, counts, nxt, H, lds_app);
}

// The rest of one path, traced in place: bounces bounce0..max_depth-1 from the
// ray r of bounce bounce0, with the path's throughput and random stream at that
// bounce.  Every contribution is added to L in the wavefront's order (emission,
// then the unoccluded shadow ray, vertex by vertex).  n_ext counts the rays after
// the first, n_sh the shadow rays.
template <int KIND, int STACK>
__device__ __forceinline__ float4 path_rest(const SceneDev& S, const PtParams& P, const ShadeHooks& H, uint32_t path,
                                            uint32_t bounce0, Ray r, float4 thr4, Rng rng, uint2* stk, int sstride,
                                            float4 L, uint32_t& n_ext, uint32_t& n_sh) {
    uint32_t nv = 0, tv = 0;
    for (uint32_t bounce = bounce0; bounce < P.max_depth; ++bounce) {
        if (bounce > bounce0) ++n_ext;
        TraceResult res = traverse<false, false, STACK>(S.nodes, S.leaf, r, stk, sstride, nv, tv);
        if (res.rec == 0xFFFFFFFFu) break;
        const float4 r2 = S.leaf[(size_t)res.rec * kTriWords + 2];
        float hu, hv;
        hit_uv(S.leaf, res.rec, r, hu, hv);
        VertexOut o;
        path_vertex<KIND>(S, P, H, path, bounce, V3{r.dx, r.dy, r.dz}, res.t, __float_as_uint(r2.y),
                          __float_as_uint(r2.z), hu, hv, thr4, rng, L, o);
        if (o.emit) L = make_float4(L.x + o.c_emit.x, L.y + o.c_emit.y, L.z + o.c_emit.z, L.w);
        if (o.sh) {
            ++n_sh;
            Ray sr{o.sh_o.x, o.sh_o.y, o.sh_o.z, 0.0f, o.sh_d.x, o.sh_d.y, o.sh_d.z, o.sh_t};
            TraceResult vis = traverse<true, false, STACK>(S.nodes, S.leaf, sr, stk, sstride, nv, tv);
            if (vis.rec == 0xFFFFFFFFu) L = make_float4(L.x + o.sh_c.x, L.y + o.sh_c.y, L.z + o.sh_c.z, L.w);
        }
        if (!o.ext) break;
        r = Ray{o.ext_o.x, o.ext_o.y, o.ext_o.z, 0.0f, o.ext_d.x, o.ext_d.y, o.ext_d.z, 1e30f};
        thr4 = o.thr4;
    }
    return L;
}

// The path kernel below: four waves per SIMD (the shading needs up to 128 VGPRs),
// fewer where the stacks' LDS is short.
__host__ __device__ constexpr int tail_waves(int stack) { return cu_waves(stack) < 16 ? cu_waves(stack) / 2 : 8; }
template <int STACK>
struct TailLds {
    uint2 stk[STACK * 64 * tail_waves(STACK)];
    uint32_t cursor, n_ext, n_sh;
};
inline TraceGrid tail_grid(int stack, uint32_t cus, uint32_t n) {
    return TraceGrid{std::min(cus * 2u, std::max(1u, (n + 7) / 8)), (uint32_t)tail_waves(stack) * 64u, 0u};
}
// Lanes of a wave with a hit to shade at which the wave stops traversing and shades
// them: it costs about as much as three traversal steps, whatever the number of
// lanes.  A quarter of the lanes where a lane sees few paths (frames of 1.02M
// triangles and of the room at 1080p, tail from bounce 1, 16 / 32 lanes: 1.597 /
// 1.595 and 0.986 / 0.961 ms; room at 256 x 256 and 400 x 300, measured before a thread
// per path took such frames: 356 / 370 and 394 / 409 us).  Lanes that only need their next ray started (a settled shadow ray, a
// path from the queue) are served from an eighth of the lanes on: waiting for the
// shading with them took 395 us on the 256 x 256 frame, 0.99 ms on the 1080p room.
constexpr uint32_t kServeLanes = 32;
// Groups waiting for any service at which a wave of eight-lane groups serves them.
constexpr uint32_t kServeGroups = 2;

// The late bounces of every path queued in `in` (n of them), each from its stored
// throughput, random stream and bounce to its end.  After Russian roulette has
// thinned the queue, a launch per bounce leaves most lanes idle; here a lane
// carries one path and all lanes of a wave traverse together, extension rays
// beside shadow rays.  A lane whose ray is finished waits until enough lanes do;
// then the wave shades their hits, settles their shadow rays, hands out the
// next queued paths to lanes whose path ended, and traverses on.  (Running each
// path's trace, shade and shadow in its own loop had 8.5 of 64 lanes active per
// VALU instruction: 774 us for the 367k paths of the 1.02M-triangle frame.)
// What a path holds between rays stays in its queue slot and path state
// (in.org / in.dir: its next ray; ps: throughput and random stream).  The traversal
// state of lanes still under way stays live across the shading of the others, though:
// at 128 VGPRs (four waves per SIMD) 13 to 20 of them spill, 40 to 52 B a lane; with
// eight lanes per path 21 (56 B).  Contributions are added to rad[path] in
// the wavefront's order (emission, then the unoccluded shadow ray, vertex by
// vertex), so the radiance is bit-identical.  The first ray of each entry was
// counted when it was queued; stats[1] / stats[2] get the rest.
template <int STACK, class SS>
__device__ __forceinline__ void tail_paths(const SS& ss, const PtParams& P, const ShadeHooks& H, const Queue& in,
                                           uint32_t n, const PathState& ps, float4* __restrict__ rad,
                                           TailLds<STACK>& lds, unsigned long long* __restrict__ stats) {
    enum { kNone = 0u, kExt = 1u, kShadow = 2u, kShadowThenExt = 3u };
    const RayShare share(n, blockIdx.x, gridDim.x);
    const uint32_t lane = __lane_id();
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    const uint32_t lanes = share.lanes();
    const bool usable = lane < lanes;
    const uint32_t serve = share.end > 2u * blockDim.x ? kServeLanes : max(1u, lanes / 4u);
    const uint32_t restart = max(1u, lanes / 8u);
    uint2* stk = lds.stk + (threadIdx.x >> 6) * (STACK * 64u) + lane;
    if (threadIdx.x == 0) lds.cursor = lds.n_ext = lds.n_sh = 0u;
    __syncthreads();
    uint32_t n_ext = 0, n_sh = 0, nv = 0, tv = 0;
    uint32_t what = kNone, slot = 0, path = 0, bounce = 0;
    bool active = false, drained = false;
    V3 sh_c{0.0f, 0.0f, 0.0f};
    const uint4* nodes = nullptr;
    const float4* tris = nullptr;
    TravState st;
    while (true) {
        const bool none = __ballot(active) == 0ull;
        const bool shade = none || (uint32_t)__popcll(__ballot(!active && what == kExt)) >= serve;
        const bool light = shade || (uint32_t)__popcll(__ballot(usable && !active && what != kExt &&
                                                                 !(drained && what == kNone))) >= restart;
        if (light) {
            Ray r;
            bool start = false;
            if (!active && what >= kShadow) {
                if (st.res.rec == 0xFFFFFFFFu) {
                    const float4 L = rad[path];
                    rad[path] = make_float4(L.x + sh_c.x, L.y + sh_c.y, L.z + sh_c.z, L.w);
                }
                start = what == kShadowThenExt;
                what = start ? kExt : kNone;
                if (start) {
                    const float4 o = in.org[slot], d = in.dir[slot];
                    r = Ray{o.x, o.y, o.z, o.w, d.x, d.y, d.z, d.w};
                }
            } else if (shade && !active && what == kExt) {
                what = kNone;
                if (st.res.rec != 0xFFFFFFFFu) {
                    const SceneDev& S = ss.at(path);
                    const float4 r2 = S.leaf[(size_t)st.res.rec * kTriWords + 2];
                    float hu, hv;
                    hit_uv(S.leaf, st.res.rec, st.p, hu, hv);
                    const float4 d = in.dir[slot];
                    const uint2 rs = ps.rng[path];
                    Rng rng{(uint64_t)rs.x | ((uint64_t)rs.y << 32), ((uint64_t)ss.stream(path) << 1u) | 1u};
                    VertexOut o;
                    path_vertex<0>(S, P, H, path, bounce, V3{d.x, d.y, d.z}, st.res.t, __float_as_uint(r2.y),
                                   __float_as_uint(r2.z), hu, hv, ps.thr[path], rng, make_float4(0.0f, 0.0f, 0.0f, 0.0f),
                                   o);
                    if (o.emit) {
                        const float4 L = rad[path];
                        rad[path] = make_float4(L.x + o.c_emit.x, L.y + o.c_emit.y, L.z + o.c_emit.z, L.w);
                    }
                    if (o.ext) {
                        ++n_ext;
                        ++bounce;
                        in.org[slot] = make_float4(o.ext_o.x, o.ext_o.y, o.ext_o.z, 0.0f);
                        in.dir[slot] = make_float4(o.ext_d.x, o.ext_d.y, o.ext_d.z, 1e30f);
                        ps.thr[path] = o.thr4;
                        ps.rng[path] = make_uint2((uint32_t)rng.state, (uint32_t)(rng.state >> 32));
                        r = Ray{o.ext_o.x, o.ext_o.y, o.ext_o.z, 0.0f, o.ext_d.x, o.ext_d.y, o.ext_d.z, 1e30f};
                        what = kExt;
                    }
                    if (o.sh) {
                        ++n_sh;
                        sh_c = o.sh_c;
                        r = Ray{o.sh_o.x, o.sh_o.y, o.sh_o.z, 0.0f, o.sh_d.x, o.sh_d.y, o.sh_d.z, o.sh_t};
                        what = o.ext ? kShadowThenExt : kShadow;
                    }
                    start = what != kNone;
                }
            }
            if (!drained) {
                const uint64_t free = __ballot(usable && !active && what == kNone);
                const uint32_t nfree = (uint32_t)__popcll(free);
                uint32_t at = 0;
                if (lane == 0) at = atomicAdd(&lds.cursor, nfree);
                at = __builtin_amdgcn_readfirstlane(at);
                const uint32_t k = at + (uint32_t)__popcll(free & below);
                if (usable && !active && what == kNone && k < share.end) {
                    slot = share.id(k);
                    path = in.path[slot];
                    bounce = ps.bounce[path];
                    const float4 o = in.org[slot], d = in.dir[slot];
                    r = Ray{o.x, o.y, o.z, o.w, d.x, d.y, d.z, d.w};
                    const SceneDev& S = ss.at(path);
                    nodes = S.nodes;
                    tris = S.leaf;
                    what = kExt;
                    start = true;
                }
                drained = at + nfree >= share.end;
            }
            if (start) active = trav_init(r, st);
            if (drained && __ballot(what != kNone) == 0ull) break;
        }
        if (active && trav_steps<false, kStepsPerRefill>(nodes, tris, st, stk, 64, what >= kShadow, nv, tv))
            active = false;
    }
    for (int o = 32; o > 0; o >>= 1) {
        n_ext += __shfl_xor(n_ext, o, 64);
        n_sh += __shfl_xor(n_sh, o, 64);
    }
    if (lane == 0) {
        atomicAdd(&lds.n_ext, n_ext);
        atomicAdd(&lds.n_sh, n_sh);
    }
    __syncthreads();
    if (threadIdx.x == 0 && (lds.n_ext | lds.n_sh)) {
        atomicAdd(&stats[1], (unsigned long long)lds.n_ext);
        atomicAdd(&stats[2], (unsigned long long)lds.n_sh);
    }
}

// tail_paths with each path's loop in a thread of its own, for queues that give a lane
// about one path: no lane has another path to go on with, and the loop keeps a path's
// state in registers (119 VGPRs, no spill) where tail_paths keeps it in memory between
// rays.  Frames of max_depth 4, this / tail_paths, us: room at 256 x 256, 480 x 360, 512
// x 512: 309 / 353, 371 / 419, 454 / 492; 10,000 emitters 476 / 485, 501 / 562, 636 /
// 657; two contexts on streams of their own at 512 x 512 658 / 825 and 927 / 1,133.
template <int STACK, int BLOCK, class SS>
__device__ __forceinline__ void tail_paths_thread(const SS& ss, const PtParams& P, const ShadeHooks& H, const Queue& in,
                                                  uint32_t n, const PathState& ps, float4* __restrict__ rad, uint2* stk,
                                                  unsigned long long* __restrict__ stats, uint32_t* red) {
    if (threadIdx.x == 0) red[0] = red[1] = 0u;
    __syncthreads();
    uint32_t n_ext = 0, n_sh = 0;
    for (uint32_t i = blockIdx.x * BLOCK + threadIdx.x; i < n; i += gridDim.x * BLOCK) {
        const uint32_t path = in.path[i];
        const float4 o = in.org[i], d = in.dir[i];
        const uint2 rs = ps.rng[path];
        const Rng rng{(uint64_t)rs.x | ((uint64_t)rs.y << 32), ((uint64_t)ss.stream(path) << 1u) | 1u};
        rad[path] = path_rest<0, STACK>(ss.at(path), P, H, path, ps.bounce[path],
                                        Ray{o.x, o.y, o.z, o.w, d.x, d.y, d.z, d.w}, ps.thr[path], rng, stk, BLOCK,
                                        rad[path], n_ext, n_sh);
    }
    for (int o = 32; o > 0; o >>= 1) {
        n_ext += __shfl_xor(n_ext, o, 64);
        n_sh += __shfl_xor(n_sh, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&red[0], n_ext);
        atomicAdd(&red[1], n_sh);
    }
    __syncthreads();
    if (threadIdx.x == 0 && (red[0] | red[1])) {
        atomicAdd(&stats[1], (unsigned long long)red[0]);
        atomicAdd(&stats[2], (unsigned long long)red[1]);
    }
}

// tail_paths with eight lanes per path (trace_group.h), for small queues: a path's
// rays are traced by its group, its vertices shaded by every lane of the group
// alike; one lane adds to the radiance and counts.  Same order of contributions.
template <int STACK, class SS>
__device__ __forceinline__ void tail_paths_group(const SS& ss, const PtParams& P, const ShadeHooks& H, const Queue& in,
                                                 uint32_t n, const PathState& ps, float4* __restrict__ rad,
                                                 GroupLds<STACK>& lds, unsigned long long* __restrict__ stats) {
    enum { kNone = 0u, kExt = 1u, kShadow = 2u, kShadowThenExt = 3u };
    const RayShare share(n, blockIdx.x, gridDim.x);
    const uint32_t lane = __lane_id(), group = lane >> 3;
    const bool first = (lane & 7u) == 0u;
    const uint32_t groups = min(8u, max(1u, (share.end + kGroupWaves - 1u) / kGroupWaves));
    const bool usable = group < groups;
    const uint64_t below = (1ull << (group * 8u)) - 1ull;
    uint2* stk = lds.group_stack();
    if (threadIdx.x == 0) lds.cursor = lds.n_ext = lds.n_sh = 0u;
    __syncthreads();
    uint32_t n_ext = 0, n_sh = 0;
    uint32_t what = kNone, slot = 0, path = 0, bounce = 0;
    bool active = false, drained = false;
    V3 sh_c{0.0f, 0.0f, 0.0f};
    const uint4* nodes = nullptr;
    const float4* tris = nullptr;
    TravState st;
    while (true) {
        const uint32_t waiting = (uint32_t)__popcll(__ballot(usable && !active && !(drained && what == kNone))) >> 3;
        const bool none = __ballot(active) == 0ull;
        if (none || waiting >= kServeGroups) {
            Ray r;
            bool start = false;
            if (!active && what >= kShadow) {
                if (first && st.res.rec == 0xFFFFFFFFu) {
                    const float4 L = rad[path];
                    rad[path] = make_float4(L.x + sh_c.x, L.y + sh_c.y, L.z + sh_c.z, L.w);
                }
                start = what == kShadowThenExt;
                what = start ? kExt : kNone;
                if (start) {
                    const float4 o = in.org[slot], d = in.dir[slot];
                    r = Ray{o.x, o.y, o.z, o.w, d.x, d.y, d.z, d.w};
                }
            } else if (!active && what == kExt) {
                what = kNone;
                if (st.res.rec != 0xFFFFFFFFu) {
                    const SceneDev& S = ss.at(path);
                    const float4 r2 = S.leaf[(size_t)st.res.rec * kTriWords + 2];
                    float hu, hv;
                    hit_uv(S.leaf, st.res.rec, st.p, hu, hv);
                    const float4 d = in.dir[slot];
                    const uint2 rs = ps.rng[path];
                    Rng rng{(uint64_t)rs.x | ((uint64_t)rs.y << 32), ((uint64_t)ss.stream(path) << 1u) | 1u};
                    VertexOut o;
                    path_vertex<0>(S, P, H, path, bounce, V3{d.x, d.y, d.z}, st.res.t, __float_as_uint(r2.y),
                                   __float_as_uint(r2.z), hu, hv, ps.thr[path], rng, make_float4(0.0f, 0.0f, 0.0f, 0.0f),
                                   o);
                    if (first && o.emit) {
                        const float4 L = rad[path];
                        rad[path] = make_float4(L.x + o.c_emit.x, L.y + o.c_emit.y, L.z + o.c_emit.z, L.w);
                    }
                    if (o.ext) {  // every lane stores the same values, so each reads back its own
                        if (first) ++n_ext;
                        ++bounce;
                        in.org[slot] = make_float4(o.ext_o.x, o.ext_o.y, o.ext_o.z, 0.0f);
                        in.dir[slot] = make_float4(o.ext_d.x, o.ext_d.y, o.ext_d.z, 1e30f);
                        ps.thr[path] = o.thr4;
                        ps.rng[path] = make_uint2((uint32_t)rng.state, (uint32_t)(rng.state >> 32));
                        r = Ray{o.ext_o.x, o.ext_o.y, o.ext_o.z, 0.0f, o.ext_d.x, o.ext_d.y, o.ext_d.z, 1e30f};
                        what = kExt;
                    }
                    if (o.sh) {
                        if (first) ++n_sh;
                        sh_c = o.sh_c;
                        r = Ray{o.sh_o.x, o.sh_o.y, o.sh_o.z, 0.0f, o.sh_d.x, o.sh_d.y, o.sh_d.z, o.sh_t};
                        what = o.ext ? kShadowThenExt : kShadow;
                    }
                    start = what != kNone;
                }
            }
            if (!drained) {
                const uint64_t free = __ballot(usable && !active && what == kNone);
                const uint32_t nfree = (uint32_t)__popcll(free) >> 3;
                uint32_t at = 0;
                if (lane == 0) at = atomicAdd(&lds.cursor, nfree);
                at = __builtin_amdgcn_readfirstlane(at);
                const uint32_t j = at + ((uint32_t)__popcll(free & below) >> 3);
                if (usable && !active && what == kNone && j < share.end) {
                    slot = share.id(j);
                    path = in.path[slot];
                    bounce = ps.bounce[path];
                    const float4 o = in.org[slot], d = in.dir[slot];
                    r = Ray{o.x, o.y, o.z, o.w, d.x, d.y, d.z, d.w};
                    const SceneDev& S = ss.at(path);
                    nodes = S.nodes;
                    tris = S.leaf;
                    what = kExt;
                    start = true;
                }
                drained = at + nfree >= share.end;
            }
            if (start) active = trav_init(r, st);
            if (drained && __ballot(what != kNone) == 0ull) break;
        }
        if (active) {
            const bool any = what >= kShadow;
            bool fin = group_step(nodes, tris, st, stk, any);
            if (!fin) fin = group_step(nodes, tris, st, stk, any);
            if (fin) active = false;
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        n_ext += __shfl_xor(n_ext, o, 64);
        n_sh += __shfl_xor(n_sh, o, 64);
    }
    if (lane == 0) {
        atomicAdd(&lds.n_ext, n_ext);
        atomicAdd(&lds.n_sh, n_sh);
    }
    __syncthreads();
    if (threadIdx.x == 0 && (lds.n_ext | lds.n_sh)) {
        atomicAdd(&stats[1], (unsigned long long)lds.n_ext);
        atomicAdd(&stats[2], (unsigned long long)lds.n_sh);
    }
}

// A whole path per thread (no queues): camera ray of path i through pixel
// (start + i * stride) mod (w h), closest hits and shadow rays traced in place.
// Same vertex logic, random stream and order of radiance additions as the
// wavefront kernels, so the radiance is bit-identical.
// L: the path's radiance so far (the pixel's sum of earlier passes); every
// contribution is added to it in the wavefront's order.
template <int KIND, int STACK>
__device__ __forceinline__ float4 whole_path(const SceneDev& S, const CamDev& cam, uint32_t w, uint32_t h,
                                             uint32_t i, uint32_t start, uint32_t stride, uint64_t initstate,
                                             const PtParams& P, const ShadeHooks& H, uint2* stk, int sstride,
                                             float4 L, uint32_t& n_ext, uint32_t& n_sh) {
    const uint32_t px = (uint32_t)(((uint64_t)start + (uint64_t)i * stride) % ((uint64_t)w * h));
    if (KIND == 2) H.nrec[i] = 0;
    const V3 d0 = camera_dir(cam, px % w, px / w, w, h);
    const Ray r{cam.pos.x, cam.pos.y, cam.pos.z, 0.0f, d0.x, d0.y, d0.z, 1e30f};
    return path_rest<KIND, STACK>(S, P, H, i, 0u, r, make_float4(1.0f, 1.0f, 1.0f, 0.0f), rng_seed(initstate, i),
                                  stk, sstride, L, n_ext, n_sh);
}

// Lanes a persistent traversal wave waits for before refilling idle lanes.
constexpr uint32_t kRefillLanes = 16;

// Shadow-queue entry i as a ray; its contribution, added when unoccluded.
__device__ __forceinline__ Ray shadow_ray(const ShadowQueue& sq, uint32_t i) {
    float4 a = sq.org[i], d = sq.dir[i];
    return Ray{a.x, a.y, a.z, a.w, d.x, d.y, d.z, d.w};
}
__device__ __forceinline__ void shadow_done(const ShadowQueue& sq, uint32_t i, const TraceResult& res,
                                            float4* __restrict__ rad) {
    if (res.rec == 0xFFFFFFFFu) {
        float4 c = sq.contrib[i];
        uint32_t px = __float_as_uint(c.w);
        float4 o = rad[px];
        rad[px] = make_float4(o.x + c.x, o.y + c.y, o.z + c.z, o.w);
    }
}

}  // namespace snkpt
