// Device-side layouts and inline routines shared by the snkpt kernels.
//
// BVH8 node (80 B, five 16 B words), after Ylitie, Karras & Laine 2017
// ("Efficient incoherent ray traversal on GPUs through compressed wide BVHs"):
//   w0 = p.x, p.y, p.z, (e.x | e.y << 8 | e.z << 16 | imask << 24)
//   w1 = child_base, tri_base, meta[0..3], meta[4..7]
//   w2 = qlo_x[0..3], qlo_x[4..7], qlo_y[0..3], qlo_y[4..7]
//   w3 = qlo_z[0..3], qlo_z[4..7], qhi_x[0..3], qhi_x[4..7]
//   w4 = qhi_y[0..3], qhi_y[4..7], qhi_z[0..3], qhi_z[4..7]
// Child box of slot s on axis a: [p_a + qlo_a[s] * 2^(e_a-127), p_a + qhi_a[s] * 2^(e_a-127)].
// meta[s] == 0: empty slot.  Internal child (imask bit s): meta = 0x20 | (24 + s);
// its node index is child_base + popcount(imask & ((1 << s) - 1)).  Leaf child:
// meta = (unary triangle count 1/3/7) << 5 | offset, its triangles are leaf
// records tri_base + offset ... + count - 1.
// Slot s holds the child lying towards octant s (bit a set = positive side of
// axis a), so a ray visits slots in order k = 0, 1, ... with s = k ^ octant(ray).
//
// Leaf triangle record (48 B, three 16 B words):
//   r0 = v0.x, v0.y, v0.z, v1.x   r1 = v1.y, v1.z, v2.x, v2.y   r2 = v2.z, inst, prim, gid
// gid is the global triangle id (instances in record order, triangles in
// submesh order); equal-t hits are resolved to the smaller gid so the closest
// hit does not depend on traversal order.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "exact_math.h"

namespace snkpt {

constexpr int kNodeWords = 5;  // uint4 per BVH8 node
constexpr int kTriWords = 3;   // float4 per leaf triangle
// 1 + 2^-16: box exits (and the current closest t they are clipped to) are
// widened by this factor so rounding never culls a box holding a closer hit.
constexpr float kBoxRobust = 1.0000152587890625f;

struct Ray {
    float ox, oy, oz, tmin;
    float dx, dy, dz, tmax;
};

// Per-ray constants of the watertight test (Woop, Benthin & Wald 2013) and of
// the box test.
struct RayPre {
    float ox, oy, oz;
    float ix, iy, iz;  // 1/d, NaN on a parallel axis
    float Sx, Sy, Sz;
    // the axis permutation, octant and parallel axes in one register: the traversal
    // loop keeps all of RayPre live, and as five registers they made the 64-VGPR
    // closest-hit loop spill one register to scratch on every step.  Bits 0-5: kx
    // is 0, kx is 1, ky is 0, ky is 1, kz is 0, kz is 1; oct << 6 | par << 9.
    uint32_t bits;
    // all ones where bit b is set
    __device__ __forceinline__ uint32_t mask(int b) const { return (uint32_t)((int32_t)(bits << (31 - b)) >> 31); }
    // bit a set: the ray runs towards -a
    __device__ __forceinline__ uint32_t oct() const { return (bits >> 6) & 7u; }
    // bit a set: axis a is parallel
    __device__ __forceinline__ uint32_t par() const { return (bits >> 9) & 7u; }
};

// x, y or z by the masks of "is x" and "is y".
__device__ __forceinline__ float sel3(float x, float y, float z, uint32_t mx, uint32_t my) {
    return __uint_as_float(bit_sel(__float_as_uint(x), bit_sel(__float_as_uint(y), __float_as_uint(z), my), mx));
}
__device__ __forceinline__ float ubyte_f(uint32_t w, int b) { return (float)((w >> (8 * b)) & 0xFFu); }

// 0xFF in byte i for every set bit i of a 4-bit mask.
__device__ __forceinline__ uint32_t byte_mask4(uint32_t m4) {
    return ((m4 & 1u) | (m4 & 2u) << 7 | (m4 & 4u) << 14 | (m4 & 8u) << 21) * 0xFFu;
}

// 1/d; an axis with |d| < 1e-20 is "parallel" and gets NaN: every fused slab
// term of that axis is then NaN, which fminf/fmaxf drop, and the axis is
// instead tested exactly (origin inside the child's decoded [lo, hi]).  A huge
// or infinite inverse would make the fused terms cancel or turn into NaN in
// the wrong places (a vertical ray would then visit most of the tree).
constexpr float kParallelEps = 1e-20f;
__device__ __forceinline__ float safe_inv(float d) {
    return fabsf(d) < kParallelEps ? __builtin_nanf("") : 1.0f / d;
}

__device__ __forceinline__ RayPre ray_setup(const Ray& r) {
    RayPre p;
    p.ox = r.ox;
    p.oy = r.oy;
    p.oz = r.oz;
    const float ax = fabsf(r.dx), ay = fabsf(r.dy), az = fabsf(r.dz);
    const int kz = (ax >= ay && ax >= az) ? 0 : (ay >= az ? 1 : 2);
    int kx = kz == 2 ? 0 : kz + 1;
    int ky = kx == 2 ? 0 : kx + 1;
    const float dkz = kz == 0 ? r.dx : (kz == 1 ? r.dy : r.dz);
    if (dkz < 0.0f) {
        int t = kx;
        kx = ky;
        ky = t;
    }
    const float dkx = kx == 0 ? r.dx : (kx == 1 ? r.dy : r.dz);
    const float dky = ky == 0 ? r.dx : (ky == 1 ? r.dy : r.dz);
    // quotients of at most 1 and at least 2^-120: inside what div_exact asks for
    constexpr float kLo = 0x1p-60f, kHi = 0x1p60f;
    if (fminf(fminf(ax, ay), az) >= kLo && fmaxf(fmaxf(ax, ay), az) <= kHi) {
        p.ix = rcp_exact(r.dx);
        p.iy = rcp_exact(r.dy);
        p.iz = rcp_exact(r.dz);
        p.Sz = kz == 0 ? p.ix : (kz == 1 ? p.iy : p.iz);
        p.Sx = div_exact(dkx, dkz, p.Sz);
        p.Sy = div_exact(dky, dkz, p.Sz);
    } else {
        p.ix = safe_inv(r.dx);
        p.iy = safe_inv(r.dy);
        p.iz = safe_inv(r.dz);
        p.Sx = dkx / dkz;
        p.Sy = dky / dkz;
        p.Sz = 1.0f / dkz;
    }
    const uint32_t oct = (p.ix < 0.0f ? 1u : 0u) | (p.iy < 0.0f ? 2u : 0u) | (p.iz < 0.0f ? 4u : 0u);
    const uint32_t par = (ax < kParallelEps ? 1u : 0u) | (ay < kParallelEps ? 2u : 0u) | (az < kParallelEps ? 4u : 0u);
    p.bits = (kx == 0 ? 1u : 0u) | (kx == 1 ? 2u : 0u) | (ky == 0 ? 4u : 0u) | (ky == 1 ? 8u : 0u) |
             (kz == 0 ? 16u : 0u) | (kz == 1 ? 32u : 0u) | oct << 6 | par << 9;
    return p;
}

// Watertight ray/triangle test, both faces, FP32 only.  On a hit writes
// t = T/det and returns true; U/V/W/det are kept for the barycentrics.
// The operation order is fixed (the library is built without FP contraction)
// so the CPU restatement reproduces every bit.
__device__ __forceinline__ bool intersect_tri(const RayPre& p, float v0x, float v0y, float v0z, float v1x, float v1y,
                                              float v1z, float v2x, float v2y, float v2z, float& t, float& U,
                                              float& V, float& W, float& det) {
    float Ax_ = v0x - p.ox, Ay_ = v0y - p.oy, Az_ = v0z - p.oz;
    float Bx_ = v1x - p.ox, By_ = v1y - p.oy, Bz_ = v1z - p.oz;
    float Cx_ = v2x - p.ox, Cy_ = v2y - p.oy, Cz_ = v2z - p.oz;
    const uint32_t x0 = p.mask(0), x1 = p.mask(1), y0 = p.mask(2), y1 = p.mask(3), z0 = p.mask(4), z1 = p.mask(5);
    float Akz = sel3(Ax_, Ay_, Az_, z0, z1), Bkz = sel3(Bx_, By_, Bz_, z0, z1), Ckz = sel3(Cx_, Cy_, Cz_, z0, z1);
    float Ax = sel3(Ax_, Ay_, Az_, x0, x1) - p.Sx * Akz;
    float Ay = sel3(Ax_, Ay_, Az_, y0, y1) - p.Sy * Akz;
    float Bx = sel3(Bx_, By_, Bz_, x0, x1) - p.Sx * Bkz;
    float By = sel3(Bx_, By_, Bz_, y0, y1) - p.Sy * Bkz;
    float Cx = sel3(Cx_, Cy_, Cz_, x0, x1) - p.Sx * Ckz;
    float Cy = sel3(Cx_, Cy_, Cz_, y0, y1) - p.Sy * Ckz;
    U = Cx * By - Cy * Bx;
    V = Ax * Cy - Ay * Cx;
    W = Bx * Ay - By * Ax;
    if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f)) return false;
    det = U + V + W;
    if (det == 0.0f) return false;
    float Az = p.Sz * Akz, Bz = p.Sz * Bkz, Cz = p.Sz * Ckz;
    float T = U * Az + V * Bz + W * Cz;
    t = T / det;
    return true;
}

struct TraceResult {
    float t;
    uint32_t gid;
    uint32_t rec;  // leaf record of the closest hit, ~0u if none
};

// Children (bit s) whose decoded box does not contain the ray origin on some
// parallel axis.  fmaf rounds once and monotonically, so the decoded planes
// still enclose the child.
__device__ __forceinline__ uint32_t parallel_miss_axis(float o, float pa, uint32_t ebyte, uint32_t lo0, uint32_t lo1,
                                                       uint32_t hi0, uint32_t hi1) {
    float sc = __uint_as_float(ebyte << 23);
    uint32_t miss = 0;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        float lo = fmaf(ubyte_f(s < 4 ? lo0 : lo1, s & 3), sc, pa);
        float hi = fmaf(ubyte_f(s < 4 ? hi0 : hi1, s & 3), sc, pa);
        if (!(lo <= o && o <= hi)) miss |= 1u << s;
    }
    return miss;
}
__device__ __forceinline__ uint32_t parallel_miss(const RayPre& p, uint4 w0, uint4 w2, uint4 w3, uint4 w4) {
    uint32_t miss = 0;
    if (p.par() & 1u)
        miss |= parallel_miss_axis(p.ox, __uint_as_float(w0.x), w0.w & 0xFFu, w2.x, w2.y, w3.z, w3.w);
    if (p.par() & 2u)
        miss |= parallel_miss_axis(p.oy, __uint_as_float(w0.y), (w0.w >> 8) & 0xFFu, w2.z, w2.w, w4.x, w4.y);
    if (p.par() & 4u)
        miss |= parallel_miss_axis(p.oz, __uint_as_float(w0.z), (w0.w >> 16) & 0xFFu, w3.x, w3.y, w4.z, w4.w);
    return miss;
}

// BVH8 traversal state of one ray.  Stack entries are node groups:
// (child_base, hit bits << 24 | imask); the stack never holds more than depth-1
// entries, so STACK >= depth-1 is checked by the launcher.
struct TravState {
    RayPre p;
    float tmin;
    uint32_t ng_base, ng_hits;
    uint32_t tg_base, tg_hits;  // leaf triangles of the last node still to test
    int sp;
    TraceResult res;
};

// Sets up the traversal of `ray`; false when the ray is invalid (it misses):
// non-finite rays, a zero direction or an empty [tmin, tmax] miss at once, as a
// NaN would otherwise pass every box test and walk the whole tree.
__device__ __forceinline__ bool trav_init(const Ray& ray, TravState& s) {
    s.res = TraceResult{ray.tmax, 0xFFFFFFFFu, 0xFFFFFFFFu};
    const bool valid = __builtin_isfinite(ray.ox) && __builtin_isfinite(ray.oy) && __builtin_isfinite(ray.oz) &&
                       __builtin_isfinite(ray.dx) && __builtin_isfinite(ray.dy) && __builtin_isfinite(ray.dz) &&
                       (ray.dx != 0.0f || ray.dy != 0.0f || ray.dz != 0.0f) && ray.tmin <= ray.tmax &&
                       !__builtin_isnan(ray.tmin) && !__builtin_isnan(ray.tmax);
    if (!valid) return false;
    s.p = ray_setup(ray);
    s.tmin = ray.tmin;
    s.sp = 0;
    // start with a node group holding the root in slot 0
    s.ng_base = 0;
    s.ng_hits = (1u << (24 + (0u ^ s.p.oct()))) | 1u;
    s.tg_base = 0;
    s.tg_hits = 0;
    return true;
}

// Tests the next pending leaf triangle of the ray (st.tg_hits must be non-zero);
// true when `any` and it is a hit.
template <bool COUNT>
__device__ __forceinline__ bool trav_tri(const float4* __restrict__ tris, TravState& st, bool any, uint32_t& tvis) {
    const uint32_t j = __builtin_ctz(st.tg_hits);
    st.tg_hits &= st.tg_hits - 1u;
    const uint32_t rec = st.tg_base + j;
    const float4* tp = tris + (size_t)rec * kTriWords;
    float4 r0 = tp[0], r1 = tp[1], r2 = tp[2];
    if (COUNT) ++tvis;
    float t, U, V, W, det;
    if (intersect_tri(st.p, r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w, r2.x, t, U, V, W, det)) {
        const uint32_t gid = __float_as_uint(r2.w);
        if (t >= st.tmin && (t < st.res.t || (t == st.res.t && gid < st.res.gid))) {
            st.res.t = t;
            st.res.gid = gid;
            st.res.rec = rec;
            if (any) return true;
        }
    }
    return false;
}

// Leaf triangles a lane may test in one traversal step before it goes on to the
// next node.  Every triangle of a node is still tested before the next node, so
// a ray's sequence of tests (and its culling) does not depend on this; it only
// bounds how long the other lanes of the wave wait for a lane with a full leaf.
// 1.29M incoherent rays, Grays/s: with leaves of up to three triangles (SAH
// triangle cost 0.3) all of a node's triangles per step 2.82, one 3.09, two
// 3.22, three 3.19, four 3.09; with leaves of mostly one triangle (cost 2.0)
// two 3.57, one 3.72.
constexpr int kTrisPerStep = 1;

// One traversal step: up to kTrisPerStep pending leaf triangles, then, when
// none is left, the next node of the current group (its 8 child boxes, which
// sets the pending triangles of its hit leaves); pops the stack when the group
// is empty.  Returns true when the ray is finished.  `stk` points to this lane's
// first stack entry in LDS; consecutive entries are `stride` uint2 apart.  `any`:
// the first hit found ends the ray (a constant, or per lane in the path kernels).
template <bool COUNT>
__device__ __forceinline__ bool trav_step(const uint4* __restrict__ nodes, const float4* __restrict__ tris,
                                          TravState& st, uint2* stk, int stride, bool any, uint32_t& nvis,
                                          uint32_t& tvis) {
    const RayPre& p = st.p;
    const float tmin = st.tmin;
#pragma unroll
    for (int i = 0; i < kTrisPerStep; ++i)
        if (st.tg_hits && trav_tri<COUNT>(tris, st, any, tvis)) return true;
    if (!st.tg_hits && (st.ng_hits & 0xFF000000u)) {
        uint32_t k = __builtin_ctz(st.ng_hits >> 24);
        st.ng_hits &= ~(1u << (24 + k));
        uint32_t s = k ^ p.oct();
        uint32_t node = st.ng_base + __builtin_popcount(st.ng_hits & 0xFFu & ((1u << s) - 1u));
        if (st.ng_hits & 0xFF000000u) {
            stk[st.sp * stride] = make_uint2(st.ng_base, st.ng_hits);
            ++st.sp;
        }
        const uint4* np = nodes + (size_t)node * kNodeWords;
        uint4 w0 = np[0], w1 = np[1], w2 = np[2], w3 = np[3], w4 = np[4];
        if (COUNT) ++nvis;
        float sx = __uint_as_float((w0.w & 0xFFu) << 23) * p.ix;
        float sy = __uint_as_float(((w0.w >> 8) & 0xFFu) << 23) * p.iy;
        float sz = __uint_as_float(((w0.w >> 16) & 0xFFu) << 23) * p.iz;
        float ax = (__uint_as_float(w0.x) - p.ox) * p.ix;
        float ay = (__uint_as_float(w0.y) - p.oy) * p.iy;
        float az = (__uint_as_float(w0.z) - p.oz) * p.iz;
        uint32_t imask = w0.w >> 24;
        // near / far plane bytes per axis (qlo first for a positive direction)
        const uint32_t nx = (uint32_t)((int32_t)__float_as_uint(p.ix) >> 31);  // all ones: the ray runs towards -x
        const uint32_t ny = (uint32_t)((int32_t)__float_as_uint(p.iy) >> 31);
        const uint32_t nz = (uint32_t)((int32_t)__float_as_uint(p.iz) >> 31);
        const uint32_t nx0 = bit_sel(w3.z, w2.x, nx), nx1 = bit_sel(w3.w, w2.y, nx);
        const uint32_t fx0 = bit_sel(w2.x, w3.z, nx), fx1 = bit_sel(w2.y, w3.w, nx);
        const uint32_t ny0 = bit_sel(w4.x, w2.z, ny), ny1 = bit_sel(w4.y, w2.w, ny);
        const uint32_t fy0 = bit_sel(w2.z, w4.x, ny), fy1 = bit_sel(w2.w, w4.y, ny);
        const uint32_t nz0 = bit_sel(w4.z, w3.x, nz), nz1 = bit_sel(w4.w, w3.y, nz);
        const uint32_t fz0 = bit_sel(w3.x, w4.z, nz), fz1 = bit_sel(w3.y, w4.w, nz);
        // meta bytes of slots 0-3 and 4-7; a parallel-axis miss clears the slot's
        // byte, so it reads as empty below
        uint32_t m0 = w1.z, m1 = w1.w;
        if (p.par()) {
            const uint32_t pmiss = parallel_miss(p, w0, w2, w3, w4);
            m0 &= ~byte_mask4(pmiss & 15u);
            m1 &= ~byte_mask4(pmiss >> 4);
        }
        // One hit word for both kinds of child, four slots at a time (Ylitie et al.
        // 2017, sec. 4): an internal child's meta byte is 0x20 | (24 + s), the only
        // bytes with bits 4 and 3 both set (leaf offsets stay below 24), and XOR-ing
        // its low three bits with the octant turns its bit index into 24 + (s ^ oct),
        // the visiting-order bit of the node group.  A leaf child keeps its index,
        // the offset of its first triangle, and its unary count.  An empty slot's
        // byte is 0 and sets nothing.
        const uint32_t oct4 = __builtin_amdgcn_perm(0u, p.oct(), 0u);  // octant in every byte
        const uint32_t in0 = (m0 & (m0 << 1)) & 0x10101010u, in1 = (m1 & (m1 << 1)) & 0x10101010u;
        // (in >> 1) - (in >> 4): 0x07 in the bytes of internal children, no borrow between bytes
        const uint32_t bi0 = (m0 ^ (oct4 & ((in0 >> 1) - (in0 >> 4)))) & 0x1F1F1F1Fu;
        const uint32_t bi1 = (m1 ^ (oct4 & ((in1 >> 1) - (in1 >> 4)))) & 0x1F1F1F1Fu;
        uint32_t hits = 0;
#pragma unroll
        for (int s2 = 0; s2 < 8; ++s2) {
            const int b = s2 & 3;
            uint32_t nxw = s2 < 4 ? nx0 : nx1, fxw = s2 < 4 ? fx0 : fx1;
            uint32_t nyw = s2 < 4 ? ny0 : ny1, fyw = s2 < 4 ? fy0 : fy1;
            uint32_t nzw = s2 < 4 ? nz0 : nz1, fzw = s2 < 4 ? fz0 : fz1;
            float tnx = fmaf(ubyte_f(nxw, b), sx, ax);
            float tny = fmaf(ubyte_f(nyw, b), sy, ay);
            float tnz = fmaf(ubyte_f(nzw, b), sz, az);
            float tfx = fmaf(ubyte_f(fxw, b), sx, ax);
            float tfy = fmaf(ubyte_f(fyw, b), sy, ay);
            float tfz = fmaf(ubyte_f(fzw, b), sz, az);
            float tn = fmaxf(fmaxf(fmaxf(tnx, tny), tnz), tmin);
            float tf = fminf(fminf(fminf(tfx, tfy), tfz), st.res.t) * kBoxRobust;
            const uint32_t bits = (((s2 < 4 ? m0 : m1) >> (8 * b + 5)) & 7u) << (((s2 < 4 ? bi0 : bi1) >> (8 * b)) & 31u);
            hits |= tn <= tf ? bits : 0u;
        }
        const uint32_t int_hits = hits & 0xFF000000u, tri_hits = hits & 0x00FFFFFFu;
        st.ng_base = w1.x;
        st.ng_hits = int_hits | imask;
        st.tg_base = w1.y;
        st.tg_hits = tri_hits;
    }
    if (!(st.ng_hits & 0xFF000000u)) {
        if (st.sp == 0) return st.tg_hits == 0u;
        --st.sp;
        uint2 e = stk[st.sp * stride];
        st.ng_base = e.x;
        st.ng_hits = e.y;
    }
    return false;
}

// BVH8 traversal of one ray to completion (closest hit, or any hit with ANY).
template <bool ANY, bool COUNT, int STACK>
__device__ __forceinline__ TraceResult traverse(const uint4* __restrict__ nodes, const float4* __restrict__ tris,
                                                const Ray& ray, uint2* stk, int stride, uint32_t& nvis,
                                                uint32_t& tvis) {
    TravState st;
    if (!trav_init(ray, st)) return st.res;
    while (!trav_step<COUNT>(nodes, tris, st, stk, stride, ANY, nvis, tvis)) {
    }
    return st.res;
}

// Waves of a persistent traversal kernel that reside on a CU: the LDS of the
// stacks (a wave's take STACK x 512 B of the 160 KB), and at most the waves whose
// VGPRs fit.
__host__ __device__ constexpr int cu_waves(int stack) {
    return stack <= 8 ? 32 : stack <= 10 ? 28 : stack <= 12 ? 24 : stack <= 16 ? 18 : stack <= 32 ? 8 : 4;
}
// Most waves per block, which share one ray cursor: half a CU's, so that few rays are
// left when a block's waves drain (1.24M bounce rays of 1.02M triangles: 12 waves
// 221 us, 6: 233, 4: 243, 2: 250; trace_grid says when it takes fewer).  Batches take
// one or two (their tuning): frames of several batches on streams of their own share a
// CU with finer blocks (64 views, three batches at once / alone: pairs 9.41 / 11.55 ms
// per frame, 4 waves 9.48 / 11.58, 12 waves 10.24 / 11.13).
__host__ __device__ constexpr int trace_waves(int stack) {
    return stack <= 8 ? 16 : stack <= 10 ? 14 : stack <= 12 ? 12 : stack <= 16 ? 9 : stack <= 32 ? 4 : 2;
}
constexpr uint32_t kFewWaves = 4;
constexpr uint32_t kFewLanes = 22 * 64;
__host__ __device__ constexpr int trace_waves_per_simd(int stack) { return stack <= 12 ? cu_waves(stack) / 4 : 1; }
// (the LDS, which is given at the launch, bounds the waves that the compiler may plan for)
__host__ __device__ constexpr int trace_waves_most(int stack) { return (cu_waves(stack) + 3) / 4; }

// Calls f(integral_constant<int, STACK>) with the smallest stack variant that holds
// `need` entries; false when none does.
template <class F>
bool with_stack(uint32_t need, F f) {
    if (need <= 8)
        f(std::integral_constant<int, 8>{});
    else if (need <= 10)
        f(std::integral_constant<int, 10>{});
    else if (need <= 12)
        f(std::integral_constant<int, 12>{});
    else if (need <= 16)
        f(std::integral_constant<int, 16>{});
    else if (need <= 32)
        f(std::integral_constant<int, 32>{});
    else if (need <= 64)
        f(std::integral_constant<int, 64>{});
    else
        return false;
    return true;
}

// Grid and LDS of a persistent traversal launch with `waves_per_cu` waves on each of
// `cus` CUs (capped by what resides), in blocks of w waves, for at most n rays.
// While every lane gets one ray at most, there is no cursor worth sharing: blocks of
// up to kFewWaves waves then, no more than the rays fill, so that a launch on another
// stream finds room beside this one (a block's LDS comes free when its last wave ends).
// One launch / two at once, us, large blocks -> four waves: 1.02M triangles 150k rays
// 87 / 125 -> 82 / 97, 250k 104 / 150 -> 97 / 121, 350k 119 / 169 -> 119 / 145; room 250k
// 66 / 96 -> 61 / 76, 350k 79 / 110 -> 75 / 95, but 390k 81 / 114 -> 87 / 109: hence
// kFewLanes.
struct TraceGrid {
    uint32_t blocks, threads, lds;
};
inline TraceGrid trace_grid(int stack, int w, uint32_t waves_per_cu, uint32_t cus, uint32_t n) {
    const uint32_t most = std::min((uint32_t)cu_waves(stack), std::max(1u, waves_per_cu));
    // large blocks: two on a CU, narrower when fewer waves are asked for
    uint32_t waves = std::min((uint32_t)w, (most + 1) / 2);
    // not more blocks than groups of 8 rays
    uint32_t blocks = std::max(1u, (n + 7) / 8);
    if (n <= cus * std::min(most * 64u, kFewLanes)) {
        waves = std::min(waves, kFewWaves);
        blocks = std::max((n + 64u * waves - 1) / (64u * waves), std::min(cus, blocks));
    }
    blocks = std::min(blocks, cus * std::max(1u, most / waves));
    return TraceGrid{blocks, waves * 64u, 16u + (uint32_t)stack * 512u * waves};
}

// The same for a batch: blocks of `lanes` (64 or 128) lanes, blocks_per_cu on each CU,
// capped by what resides and by what n rays fill.
inline uint32_t batch_blocks_per_cu(int stack, uint32_t lanes, uint32_t blocks_per_cu) {
    return std::min(std::max(1u, blocks_per_cu), (uint32_t)cu_waves(stack) * 64u / lanes);
}
inline TraceGrid batch_grid(int stack, uint32_t lanes, uint32_t blocks_per_cu, uint32_t cus, uint32_t n) {
    const uint32_t fill = std::max(n / lanes + 1u, std::min(cus, std::max(1u, n / 8u)));
    return TraceGrid{std::min(cus * batch_blocks_per_cu(stack, lanes, blocks_per_cu), fill), lanes,
                     16u + (uint32_t)stack * 8u * lanes};
}

// LDS of a persistent traversal block (TraceGrid::lds bytes, given at the launch): the
// block's ray cursor and each wave's stacks (entries 64 lanes apart, so lanes at equal
// depth hit distinct banks).
template <int STACK>
struct TraceLds {
    uint32_t& cursor;
    uint2* stk;
    __device__ __forceinline__ explicit TraceLds(uint4* mem) : cursor(mem->x), stk((uint2*)(mem + 1)) {}
    __device__ __forceinline__ uint2* lane_stack() const {
        return stk + (threadIdx.x >> 6) * (STACK * 64u) + (threadIdx.x & 63u);
    }
};

constexpr uint32_t kSpreadWaves = 3;

// Rays handed out by one block: of the rays [0, n), block b of nb owns the
// 64-ray chunk b of every whole band of nb x 64 rays (so the blocks in flight
// trace one band of neighbouring rays at a time and share its BVH nodes in L2)
// and the [b rest / nb, (b + 1) rest / nb) slice of the last, partial band.
struct RayShare {
    uint32_t block, nblocks, full64, base, end;  // end: rays of this block
    __device__ __forceinline__ RayShare(uint32_t n, uint32_t b, uint32_t nb) : block(b), nblocks(nb) {
        const uint32_t band = nb * 64u, full = n / band;
        base = full * band;
        full64 = full * 64u;
        const uint32_t rest = n - base;
        const uint32_t lo = (uint32_t)(((uint64_t)b * rest) / nb);
        end = full64 + (uint32_t)(((uint64_t)(b + 1u) * rest) / nb) - lo;
        base += lo;
    }
    // the block's k-th ray
    __device__ __forceinline__ uint32_t id(uint32_t k) const {
        return k < full64 ? ((k >> 6) * nblocks + block) * 64u + (k & 63u) : base + (k - full64);
    }
    // Lanes of a wave that take rays: all of them, or, when the block's rays do not
    // fill kSpreadWaves waves, an even part of them (at least 8): a small call then
    // uses more SIMDs, and a wave waits for fewer rays.  Waves per block, 65k paths of
    // a 256 x 256 room frame / 16k collision rays (while a lane carried each; such calls
    // take other kernels now, queues shorter than the host's bound and counted calls
    // still come here): 2: 455 / 33.6 us, 3: 457 / 35.7, 4: 471 / 32.9, 6: 500 / 31.4;
    // one 64-ray chunk per wave over the chip 478 / 39.5.
    __device__ __forceinline__ uint32_t lanes() const {
        const uint32_t waves = min(kSpreadWaves, blockDim.x >> 6);
        return min(64u, max(8u, (end + waves - 1u) / waves));
    }
};

// Up to N traversal steps; true as soon as one finishes the ray.
template <bool COUNT, int N>
__device__ __forceinline__ bool trav_steps(const uint4* __restrict__ nodes, const float4* __restrict__ tris,
                                           TravState& st, uint2* stk, int stride, bool any, uint32_t& nvis,
                                           uint32_t& tvis) {
    if (trav_step<COUNT>(nodes, tris, st, stk, stride, any, nvis, tvis)) return true;
    if constexpr (N > 1) return trav_steps<COUNT, N - 1>(nodes, tris, st, stk, stride, any, nvis, tvis);
    return false;
}

// Persistent traversal with ray refill (after Aila & Laine 2009, "Understanding
// the efficiency of ray traversal on GPUs").  The waves of a block take the
// block's rays (RayShare) in order from one cursor in LDS, whenever at least
// `refill` of a wave's lanes are idle (or all are), so a wave does not wait for
// its slowest ray with the other lanes masked off, and the waves of a block end
// together: with a fixed slice per wave, waves of the same launch were busy for
// 76 to 257 us (161 on average; 1.24M bounce rays, 1.02M triangles), since a slice
// of a few chunks does not average out.  Between two such checks a lane takes up
// to STEPS traversal steps.  load(id, ray, nodes, tris) fetches ray `id` and the
// BVH it is traced against; done(id, state, nvis, tvis) is called once per ray
// with its finished state, also for invalid rays (which miss), when the wave
// hands out rays again: the lanes that finished in between deliver together (a
// call per finished lane ran the hit's stores and barycentrics at 1-3 of 64
// lanes).  Every ray's traversal is the one of traverse(), so results are
// identical.  All threads of the block must call it.
template <bool ANY, bool COUNT, int STACK, int STEPS, class Load, class Done>
__device__ __forceinline__ void refill_trace(uint32_t n, const TraceLds<STACK>& lds, uint32_t refill, Load load, Done done) {
    const RayShare share(n, blockIdx.x, gridDim.x);
    const uint32_t lane = __lane_id();
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    const uint32_t lanes = share.lanes();
    const bool usable = lane < lanes;
    if (lanes < 64u) refill = min(refill, lanes / 4u);
    uint2* stk = lds.lane_stack();
    if (threadIdx.x == 0) lds.cursor = 0u;
    __syncthreads();
    bool drained = false;
    bool active = false, pending = false;  // pending: the lane's ray is finished, done() not yet called
    uint32_t id = 0, nv = 0, tv = 0;
    const uint4* nodes = nullptr;
    const float4* tris = nullptr;
    TravState st;
    while (true) {
        const uint64_t idle = __ballot(usable && !active);
        const uint32_t nidle = (uint32_t)__popcll(idle);
        if (nidle == lanes || (!drained && nidle >= refill)) {
            if (pending) done(id, st, nv, tv);
            if (drained) break;
            uint32_t at = 0;
            if (lane == 0) at = atomicAdd(&lds.cursor, nidle);
            at = __builtin_amdgcn_readfirstlane(at);
            if (usable && !active) {
                pending = false;
                const uint32_t k = at + (uint32_t)__popcll(idle & below);
                if (k < share.end) {
                    id = share.id(k);
                    Ray ray;
                    load(id, ray, nodes, tris);
                    nv = tv = 0;
                    active = trav_init(ray, st);
                    pending = !active;
                }
            }
            drained = at + nidle >= share.end;
        }
        if (active && trav_steps<COUNT, STEPS>(nodes, tris, st, stk, 64, ANY, nv, tv)) {
            active = false;
            pending = true;
        }
    }
}

// Traversal steps between two refill checks where they are not tuned: the check
// (a ballot and the ray hand-out) costs as much as a light step.  C2 incoherent
// rays, Grays/s: 1 step 3.21, 2: 3.33, 3: 3.37, 4: 3.35, 6: 3.31; the config-5
// batch frame 15.6, 14.4, 13.9, 13.6, 13.7 ms.
constexpr int kStepsPerRefill = 4;

// Barycentrics (u, v) of a leaf record hit; bary = (1-u-v, u, v).
__device__ __forceinline__ void hit_uv(const float4* __restrict__ tris, uint32_t rec, const RayPre& p, float& u,
                                       float& v) {
    const float4* tp = tris + (size_t)rec * kTriWords;
    float4 r0 = tp[0], r1 = tp[1], r2 = tp[2];
    float t, U, V, W, det;
    intersect_tri(p, r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w, r2.x, t, U, V, W, det);
    u = V / det;
    v = W / det;
}
__device__ __forceinline__ void hit_uv(const float4* __restrict__ tris, uint32_t rec, const Ray& ray, float& u,
                                       float& v) {
    hit_uv(tris, rec, ray_setup(ray), u, v);
}

// Block-level queue append: every thread of the block calls it (convergent:
// no thread may have returned before); threads with `want` get consecutive
// slots from one atomicAdd per block, in wave-then-lane order.  Same-address
// atomics are serialised by the memory system, so one per block instead of one
// per wave matters for the big early bounces.  `lds` holds BLOCK / 64 + 1 words
// and may be reused right after the call.
template <int BLOCK>
__device__ __forceinline__ uint32_t block_append(bool want, uint32_t* counter, uint32_t* lds) {
    constexpr int kWaves = BLOCK / 64;
    const uint64_t m = __ballot(want);
    const uint32_t lane = __lane_id(), wave = threadIdx.x >> 6;
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    if (lane == 0) lds[wave] = (uint32_t)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t run = 0;
        for (int w = 0; w < kWaves; ++w) {
            uint32_t c = lds[w];
            lds[w] = run;
            run += c;
        }
        lds[kWaves] = run ? atomicAdd(counter, run) : 0u;
    }
    __syncthreads();
    const uint32_t slot = lds[kWaves] + lds[wave] + (uint32_t)__popcll(m & lt);
    __syncthreads();
    return want ? slot : 0xFFFFFFFFu;
}

}  // namespace snkpt
