// BVH8 traversal with eight lanes per ray, for calls too small to fill the chip
// with a lane per ray.
//
// A lane alone needs about 250 instructions for a node (eight child boxes) and
// 100 for a triangle, and with one or two waves on a SIMD it is their latency, not
// the issue rate, that a small call waits for: its longest ray times that.  Here a
// group of eight lanes carries one ray, each lane tests one child box (lane k the
// child visited k-th) or one of the node's triangles, and the group's state is the
// same in all of its lanes.  The sequence of nodes, the culling and the hits are
// those of trav_step, bit for bit.
#pragma once

#include "snkpt_dev.h"

namespace snkpt {

// Bits of the group's lanes for which `x` holds (all eight lanes must be active).
__device__ __forceinline__ uint32_t group_ballot(bool x) {
    return (uint32_t)(__ballot(x) >> (__lane_id() & 56u)) & 0xFFu;
}
// The partner's value: lane ^ 1, lane ^ 2, 7 - lane of the group.
template <int STAGE>
__device__ __forceinline__ uint32_t group_swap(uint32_t x) {
    constexpr int ctrl = STAGE == 0 ? 0xB1 : STAGE == 1 ? 0x4E : 0x141;  // quad_perm 1,0,3,2 / 2,3,0,1, row_half_mirror
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, ctrl, 0xF, 0xF, true);
}
template <int STAGE>
__device__ __forceinline__ void group_closer(float& t, uint32_t& gid, uint32_t& rec) {
    const float ot = __uint_as_float(group_swap<STAGE>(__float_as_uint(t)));
    const uint32_t og = group_swap<STAGE>(gid), orec = group_swap<STAGE>(rec);
    const bool take = ot < t || (ot == t && og < gid);
    t = take ? ot : t;
    gid = take ? og : gid;
    rec = take ? orec : rec;
}

// One step of the group's ray: up to eight of its pending triangles, then, when none
// is left, the next node.  stk: the group's stack (entries 8 uint2 apart).
__device__ __forceinline__ bool group_step(const uint4* __restrict__ nodes, const float4* __restrict__ tris,
                                           TravState& st, uint2* stk, bool any) {
    const RayPre& p = st.p;
    const uint32_t k = __lane_id() & 7u;
    if (st.tg_hits) {
        const uint32_t first = __builtin_ctz(st.tg_hits) & 24u;
        const uint32_t rec = st.tg_base + first + k;
        bool hit = false;
        float t = __builtin_inff();
        uint32_t gid = 0xFFFFFFFFu;
        if ((st.tg_hits >> (first + k)) & 1u) {
            const float4* tp = tris + (size_t)rec * kTriWords;
            const float4 r0 = tp[0], r1 = tp[1], r2 = tp[2];
            float tt, U, V, W, det;
            if (intersect_tri(p, r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w, r2.x, tt, U, V, W, det)) {
                const uint32_t g = __float_as_uint(r2.w);
                hit = tt >= st.tmin && (tt < st.res.t || (tt == st.res.t && g < st.res.gid));
                if (hit) t = tt, gid = g;
            }
        }
        const uint32_t hits = group_ballot(hit);
        if (hits) {
            uint32_t r = rec;
            if (any) {  // the first of them in the order of the triangles
                const int src = (int)((__lane_id() & 56u) + __builtin_ctz(hits));
                st.res.t = __shfl(t, src, 64);
                st.res.gid = (uint32_t)__shfl((int)gid, src, 64);
                st.res.rec = (uint32_t)__shfl((int)rec, src, 64);
                return true;
            }
            group_closer<0>(t, gid, r);
            group_closer<1>(t, gid, r);
            group_closer<2>(t, gid, r);
            st.res = TraceResult{t, gid, r};
        }
        st.tg_hits &= ~(0xFFu << first);
    }
    if (!st.tg_hits && (st.ng_hits & 0xFF000000u)) {
        const uint32_t k0 = __builtin_ctz(st.ng_hits >> 24);
        st.ng_hits &= ~(1u << (24 + k0));
        const uint32_t node = st.ng_base + __builtin_popcount(st.ng_hits & 0xFFu & ((1u << (k0 ^ p.oct())) - 1u));
        if (st.ng_hits & 0xFF000000u) {
            stk[st.sp * 8] = make_uint2(st.ng_base, st.ng_hits);
            ++st.sp;
        }
        // the lane's child: slot s, visited k-th
        const uint32_t s = k ^ p.oct();
        const uint8_t* np = (const uint8_t*)(nodes + (size_t)node * kNodeWords);
        const uint4 w0 = *(const uint4*)np;
        const uint2 base = *(const uint2*)(np + 16);
        const uint8_t* q = np + 32 + s;  // qlo x, y, z at 0, 8, 16; qhi at 24, 32, 40
        const uint32_t meta = np[24 + s];
        const uint32_t nx = p.ix < 0.0f ? 24u : 0u, ny = p.iy < 0.0f ? 24u : 0u, nz = p.iz < 0.0f ? 24u : 0u;
        const float qnx = (float)q[nx], qfx = (float)q[24u - nx];
        const float qny = (float)q[8u + ny], qfy = (float)q[32u - ny];
        const float qnz = (float)q[16u + nz], qfz = (float)q[40u - nz];
        const float cx = __uint_as_float((w0.w & 0xFFu) << 23), cy = __uint_as_float(((w0.w >> 8) & 0xFFu) << 23),
                    cz = __uint_as_float(((w0.w >> 16) & 0xFFu) << 23);
        const float px = __uint_as_float(w0.x), py = __uint_as_float(w0.y), pz = __uint_as_float(w0.z);
        const float sx = cx * p.ix, sy = cy * p.iy, sz = cz * p.iz;
        const float ax = (px - p.ox) * p.ix, ay = (py - p.oy) * p.iy, az = (pz - p.oz) * p.iz;
        const float tn = fmaxf(fmaxf(fmaxf(fmaf(qnx, sx, ax), fmaf(qny, sy, ay)), fmaf(qnz, sz, az)), st.tmin);
        const float tf = fminf(fminf(fminf(fmaf(qfx, sx, ax), fmaf(qfy, sy, ay)), fmaf(qfz, sz, az)), st.res.t) *
                         kBoxRobust;
        bool hit = tn <= tf && meta != 0u;
        if (p.par()) {  // the inverse of a parallel axis is NaN (near plane = lower plane)
            if (p.par() & 1u) hit = hit && fmaf(qnx, cx, px) <= p.ox && p.ox <= fmaf(qfx, cx, px);
            if (p.par() & 2u) hit = hit && fmaf(qny, cy, py) <= p.oy && p.oy <= fmaf(qfy, cy, py);
            if (p.par() & 4u) hit = hit && fmaf(qnz, cz, pz) <= p.oz && p.oz <= fmaf(qfz, cz, pz);
        }
        const uint32_t imask = w0.w >> 24;
        const bool inner = (imask >> s) & 1u;
        uint32_t tri = hit && !inner ? (meta >> 5) << (meta & 31u) : 0u;
        tri |= group_swap<0>(tri);
        tri |= group_swap<1>(tri);
        tri |= group_swap<2>(tri);
        st.ng_hits = group_ballot(hit && inner) << 24 | imask;
        st.ng_base = base.x;
        st.tg_base = base.y;
        st.tg_hits = tri;
    }
    if (!(st.ng_hits & 0xFF000000u)) {
        if (st.sp == 0) return st.tg_hits == 0u;
        --st.sp;
        const uint2 e = stk[st.sp * 8];
        st.ng_base = e.x;
        st.ng_hits = e.y;
    }
    return false;
}

// Waves per block; a small call gives each wave few rays (down to one).
constexpr int kGroupWaves = 4;
constexpr uint32_t kGroupCuWaves = 24;
// Largest call with a group per ray, by the tree's depth.  A group / a lane per ray, us
// (closest hit; contacts): depth 7 82k 41 / 45 and 43 / 45, 98k 43 / 45 and 47 / 44, 131k
// 51 / 45 and 56 / 43, two calls at once 72 / 56 and 79 / 54; depth 8 131k 56 / 62 and 60 /
// 63, 197k 77 / 72 and 87 / 63; depth 10 131k 72 / 98 and 78 / 77; depth 12 131k 69 / 87
// and 73 / 74, 164k 75 / 99 and 87 / 87, two at once 101 / 116 and 116 / 98.
inline uint32_t group_rays(uint32_t depth) { return depth < 8u ? 81920u : 1u << 17; }
// Largest queue whose paths run a group each, by the tree's depth (deeper trees take
// more steps per ray, and their latency is what a group shortens).  Frames with a group
// / a thread per path, us, on both sides of the line: depth 7 (line 35,840 paths) 32k 256 /
// 267, 50k 344 / 289; depth 8 (40,960) 32k 299 / 353, 50k 398 / 389; depth 10 (52,000)
// 50k 458 / 459, 65k 581 / 490; depth 12 (89,856), on two scenes, 77k 555 / 624 and 592 /
// 596, 101k 659 / 652 and 689 / 654.  Deeper trees, not measured, share depth 12's line.
inline uint32_t group_paths(uint32_t depth) {
    const uint32_t d = std::min(depth, 12u);
    return std::max(5120u * d, 52u * d * d * d);
}
template <int STACK>
struct GroupLds {
    uint2 stk[kGroupWaves * STACK * 64 / 8];
    uint32_t cursor, n_ext, n_sh;
    __device__ __forceinline__ uint2* group_stack() {
        const uint32_t lane = threadIdx.x & 63u;
        return stk + (threadIdx.x >> 6) * (STACK * 8u) + (lane >> 3);
    }
};
inline TraceGrid group_grid(uint32_t waves_per_cu, uint32_t cus, uint32_t n) {
    return TraceGrid{std::min(cus * (waves_per_cu / kGroupWaves), std::max(1u, (n + kGroupWaves - 1) / kGroupWaves)),
                     64u * kGroupWaves, 0u};
}

// refill_trace with a group per ray.  load(id, ray, nodes, tris) and done(id, state)
// run in all lanes of the group; done's writes must be the same from each.
template <bool ANY, int STACK, class Load, class Done>
__device__ __forceinline__ void group_trace(uint32_t n, GroupLds<STACK>& lds, Load load, Done done) {
    const RayShare share(n, blockIdx.x, gridDim.x);
    const uint32_t group = __lane_id() >> 3;
    const uint32_t groups = min(8u, max(1u, (share.end + kGroupWaves - 1u) / kGroupWaves));
    const bool usable = group < groups;
    const uint64_t below = (1ull << (group * 8u)) - 1ull;
    uint2* stk = lds.group_stack();
    if (threadIdx.x == 0) lds.cursor = 0u;
    __syncthreads();
    bool drained = false, active = false, pending = false;
    uint32_t id = 0;
    const uint4* nodes = nullptr;
    const float4* tris = nullptr;
    TravState st;
    while (true) {
        const uint64_t idle = __ballot(usable && !active);
        const uint32_t nidle = (uint32_t)__popcll(idle) >> 3;
        if (nidle == groups || (!drained && nidle >= 2u)) {
            if (pending) done(id, st);
            if (drained) break;
            uint32_t at = 0;
            if (__lane_id() == 0) at = atomicAdd(&lds.cursor, nidle);
            at = __builtin_amdgcn_readfirstlane(at);
            if (usable && !active) {
                pending = false;
                const uint32_t j = at + ((uint32_t)__popcll(idle & below) >> 3);
                if (j < share.end) {
                    id = share.id(j);
                    Ray ray;
                    load(id, ray, nodes, tris);
                    active = trav_init(ray, st);
                    pending = !active;
                }
            }
            drained = at + nidle >= share.end;
        }
        if (active) {
            bool fin = group_step(nodes, tris, st, stk, ANY);
            if (!fin) fin = group_step(nodes, tris, st, stk, ANY);
            if (fin) {
                active = false;
                pending = true;
            }
        }
    }
}

}  // namespace snkpt
