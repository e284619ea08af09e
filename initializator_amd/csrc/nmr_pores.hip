// nmr_pores.hip -- the sweeps over a list of the pores (gfx950).
//
// Only pores change in a step, and in a porous medium they are a fifth to a
// third of the voxels.  The tile sweeps (nmr_kernels.hip) stream the grid and
// skip what is all solid, but a 4-voxel chunk or 128-byte brick with one pore
// costs as much as a full one.  Here the state of the pores is kept as a
// list: 64 slots to a group, in the grid's order, so that the wavefront of a
// group has a pore in every lane.  A slot's x neighbours are the slots next
// to it; its y and z neighbours are given as 16-bit offsets from a base of
// the group; which neighbours are pores, and which lanes count in the signal,
// are 64-bit lane masks of the group's descriptor, read into scalar registers
// and used as lane conditions directly.  A group never spans two planes, so
// z and the precession angle of a z gradient are uniform in a wavefront.
//
// A step moves 38 bytes a pore -- two components read and written (16), the
// velocity sums (12), the offsets (8), the descriptor (2) -- less than half of
// the tile sweep's traffic a voxel at 20 % porosity; a workgroup's groups are
// consecutive and each XCD takes a contiguous run of workgroups, so the
// planes above and below are in that XCD's L2.  256^3, porosity 0.2, flow and
// gradient: 20.6 us a step (the tile sweep on bricks: 58.0).  What bounds it
// there is not those bytes but the vector memory path: 200 L1 accesses a group
// (16 for a 64-lane load of 8 bytes, ten such accesses a slot), 17 us at one
// a cycle and CU; leaving out the gathers' spread or a third of the vector
// instructions changed nothing.  On 512x512x130 (259 MB a step, past the
// memory-side cache) it is the bytes: 39 us, 6.6 TB/s.
//
// The arithmetic of a voxel is that of the tile sweeps (update_chunk,
// gupdate_chunk) and of general_kernel, operation by operation, so the fields
// are the same bits.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "nmr_device.h"
#include "nmr_kernels.h"

namespace nmr {

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
// Codes among the offsets.  y: the signed distance to the neighbour's slot, 0
// where the slot's own value is read; z (and x, where it has offsets): the
// distance from the group's base.
constexpr uint32_t kOwn = 0xffffu;   // x: the own value is read
constexpr uint32_t kZero = 0xfffeu;  // x, z: 0 is read (slot 0, which stays 0)
constexpr uint32_t kZeroY = 0x8000u; // y: 0 is read

// Group descriptors are read through the constant address space: uniform
// loads from it go to scalar registers, also in a loop that stores.
typedef const __attribute__((address_space(4))) PoreGroup* GroupPtr;
typedef const __attribute__((address_space(4))) PoreGhost* GhostPtr;
__device__ __forceinline__ GroupPtr group_at(const PoreGroup* g, int i) { return (GroupPtr)(uintptr_t)(g + i); }

// Values that the compiler must have at this point: it would otherwise sink
// the load behind a select (of a base, of the neighbours' values) into a
// branch, one dependent wait each.
template <typename T>
__device__ __forceinline__ void have_s(T& x)
{
    asm volatile("" : "+s"(x));
}
__device__ __forceinline__ void have_v(float& x) { asm volatile("" : "+v"(x)); }

__device__ __forceinline__ bool lane_in(uint64_t mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }

// State of slot i, NC floats per slot.  Byte offsets stay below 4 GiB, so an
// access is a scalar base plus a 32-bit offset.
template <int NC>
struct VecOf;
template <>
struct VecOf<1> {
    typedef float type __attribute__((ext_vector_type(1)));
};
template <>
struct VecOf<2> {
    typedef float type __attribute__((ext_vector_type(2)));
};
template <>
struct VecOf<3> {
    typedef float type __attribute__((ext_vector_type(3), aligned(4)));
};
template <int NC>
using Vec = typename VecOf<NC>::type;

template <int NC>
__device__ __forceinline__ Vec<NC> ldm(const float* base, uint32_t i)
{
    return *reinterpret_cast<const Vec<NC>*>(reinterpret_cast<const char*>(base) + i * (uint32_t)(4 * NC));
}
template <int NC>
__device__ __forceinline__ void stm(float* base, uint32_t i, const Vec<NC>& v)
{
    *reinterpret_cast<Vec<NC>*>(reinterpret_cast<char*>(base) + i * (uint32_t)(4 * NC)) = v;
}
template <typename T>
__device__ __forceinline__ T ldw(const T* base, uint32_t i)
{
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + i * (uint32_t)sizeof(T));
}

// A value at byte offset o of an array.
template <typename T>
__device__ __forceinline__ T at_byte(const void* base, uint32_t o)
{
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + o);
}
// v of another lane by a DPP move of both halves (0 where the move has no source).
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v)
{
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROWS, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, ROWS, 0xf, false);
    return v + __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Sum over the wavefront, in lane 63: within rows of 16 lanes by shifts,
// then across the rows by broadcasts -- register moves, where a shuffle
// through LDS costs a round trip each.
__device__ __forceinline__ double wave_sum(double v)
{
    v = dpp_add<0x111, 0xf>(v); // row_shr:1
    v = dpp_add<0x112, 0xf>(v); // row_shr:2
    v = dpp_add<0x114, 0xf>(v); // row_shr:4
    v = dpp_add<0x118, 0xf>(v); // row_shr:8
    v = dpp_add<0x142, 0xa>(v); // row_bcast:15 into rows 1 and 3
    v = dpp_add<0x143, 0xc>(v); // row_bcast:31 into rows 2 and 3
    return v;
}

// Workgroup sum of acc into dst[q] (fixed order): lane by lane over the
// wavefronts through LDS first, so that only one wavefront runs the sum over
// the lanes (about 35 instructions a sum).
template <int NS>
__device__ __forceinline__ void group_reduce(double (&acc)[NS], double (*sred)[NS][64], double* dst)
{
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (wave > 0) {
#pragma unroll
        for (int q = 0; q < NS; q++) sred[wave - 1][q][lane] = acc[q];
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int q = 0; q < NS; q++) {
        double v = acc[q];
#pragma unroll
        for (int w = 0; w < kWaves - 1; w++) v += sred[w][q][lane];
        v = wave_sum(v);
        if (lane == 63) dst[q] = v;
    }
}

// The descriptor of a group, in scalar registers.
struct GroupRegs {
    uint32_t base[6];
    float zc;
    uint64_t pore[6], active, window, xm, xp, zm, zp;
    template <bool GEN>
    __device__ __forceinline__ void load(GroupPtr G)
    {
#pragma unroll
        for (int s = GEN ? 0 : 4; s < 6; s++) base[s] = (uint32_t)G->base[s];
        zc = G->zc;
#pragma unroll
        for (int s = 0; s < 6; s++) pore[s] = G->pore[s];
        active = G->active;
        window = G->window;
        xm = G->xm;
        xp = G->xp;
        zm = G->zm;
        zp = G->zp;
#pragma unroll
        for (int s = GEN ? 0 : 4; s < 6; s++) have_s(base[s]);
        have_s(xm);
        have_s(xp);
        have_s(zm);
        have_s(zp);
    }
};

// A 16-bit half of x times K plus a, one instruction each.
template <int K, bool HI>
__device__ __forceinline__ uint32_t mad_i16(uint32_t x, uint32_t a)
{
    uint32_t r;
    if constexpr (HI) asm("v_mad_i32_i16 %0, %1, %2, %3 op_sel:[1,0,0,0]" : "=v"(r) : "v"(x), "n"(K), "v"(a));
    else asm("v_mad_i32_i16 %0, %1, %2, %3" : "=v"(r) : "v"(x), "n"(K), "v"(a));
    return r;
}
template <int K, bool HI>
__device__ __forceinline__ uint32_t mad_u16(uint32_t x, uint32_t a)
{
    uint32_t r;
    if constexpr (HI) asm("v_mad_u32_u16 %0, %1, %2, %3 op_sel:[1,0,0,0]" : "=v"(r) : "v"(x), "n"(K), "s"(a));
    else asm("v_mad_u32_u16 %0, %1, %2, %3" : "=v"(r) : "v"(x), "n"(K), "s"(a));
    return r;
}
// max(v, 0) and min(v, 0) (0 for a NaN) without the canonicalisation that
// fmaxf adds for signalling NaNs, which no loaded sum is.
__device__ __forceinline__ float pos(float v)
{
    float r;
    asm("v_max_f32 %0, 0, %1" : "=v"(r) : "v"(v));
    return r;
}
__device__ __forceinline__ float neg(float v)
{
    float r;
    asm("v_min_f32 %0, 0, %1" : "=v"(r) : "v"(v));
    return r;
}

// Offsets of the neighbours x-, x+, y-, y+, z-, z+ of a slot, in units of K
// bytes a slot; a missing neighbour gives the slot itself.
template <int K, bool GEN>
__device__ __forceinline__ void neighbours(const PoreArgs& a, const GroupRegs& G, uint2 off, uint32_t slot,
                                           uint32_t (&nb)[6])
{
    const uint32_t own = slot * (uint32_t)K;
    nb[0] = lane_in(G.xm) ? own - (uint32_t)K : own;
    nb[1] = lane_in(G.xp) ? own + (uint32_t)K : own;
    nb[2] = mad_i16<K, false>(off.x, own);
    nb[3] = mad_i16<K, true>(off.x, own);
    const uint32_t zm = mad_u16<K, false>(off.y, G.base[4] * (uint32_t)K);
    const uint32_t zp = mad_u16<K, true>(off.y, G.base[5] * (uint32_t)K);
    nb[4] = lane_in(G.zm) ? zm : own;
    nb[5] = lane_in(G.zp) ? zp : own;
    if constexpr (GEN) {
        if ((off.x & 0xffffu) == kZeroY) nb[2] = 0u;
        if ((off.x >> 16) == kZeroY) nb[3] = 0u;
        if ((off.y & 0xffffu) == kZero) nb[4] = 0u;
        if ((off.y >> 16) == kZero) nb[5] = 0u;
        if (a.xoff) {
            const uint32_t xo = ldw(a.xoff, slot);
            const uint32_t m = xo & 0xffffu, p = xo >> 16;
            nb[0] = m == kOwn ? own : (m == kZero ? 0u : (G.base[0] + m) * (uint32_t)K);
            nb[1] = p == kOwn ? own : (p == kZero ? 0u : (G.base[1] + p) * (uint32_t)K);
        }
    }
}

// r + s0*(faces to solids on the axis of sides m and m+1): fmaf(s, n, r) with n
// 0, 1 or 2 from the lane masks.
__device__ __forceinline__ float solid_faces(const GroupRegs& G, int m)
{
    const uint64_t any = ~(G.pore[m] & G.pore[m + 1]), both = ~(G.pore[m] | G.pore[m + 1]);
    const float n = lane_in(any) ? 1.f : 0.f;
    return lane_in(both) ? 2.f : n;
}

// One step (or MacCormack stage ST) of the 64 slots of group g, lane by lane.
// GEN: per-voxel field, masked advection, non-zero-derivative ghosts and
// phase weights may be present (null pointers and flags say which); COEF:
// per-voxel diffusivity and rates.
template <int NC, bool VEL, int ST, bool EXACT, bool GEN, bool COEF, int NS>
__device__ __forceinline__ void pore_step(const PoreArgs& a, const Coef& cf, const int g, double (&acc)[NS])
{
    constexpr int K = 4 * NC;
    const uint32_t slot = (uint32_t)g * 64u + (threadIdx.x & 63u);
    const uint2 off = ldw(a.off, slot);
    const Vec<NC> mc = ldm<NC>(a.f, slot);
    GroupRegs G;
    G.load<GEN>(group_at(a.groups, g));
    Vec<3> adv = {0.f, 0.f, 0.f};
    if constexpr (VEL) adv = ldm<3>(a.vel, slot);
    uint32_t nb[6];
    neighbours<K, GEN>(a, G, off, slot, nb);
    Vec<NC> fn[6];
#pragma unroll
    for (int s = 0; s < 6; s++) fn[s] = at_byte<Vec<NC>>(a.f, nb[s]);

    bool kn[6];
#pragma unroll
    for (int s = 0; s < 6; s++) kn[s] = lane_in(G.pore[s]);

    // face weights on (neighbour - centre), as update_chunk and
    // gupdate_chunk form them (a product with the 0/1 pore flag is a select)
    float w[6];
    if constexpr (COEF) {
        uint32_t nd[6];
        neighbours<4, GEN>(a, G, off, slot, nd);
        const float dc = ldw(a.dn, slot);
        const float cd[3] = {cf.cdx, cf.cdy, cf.cdz};
#pragma unroll
        for (int s = 0; s < 6; s++) {
            float dnb = at_byte<float>(a.dn, nd[s]);
            // ghosts carry the diffusivity of the voxel they border
            if (a.ghost && lane_in(((GhostPtr)(uintptr_t)(a.ghost + g))->side[s])) dnb = dc;
            const float hm = hmean(dc, dnb);
            w[s] = cd[s / 2] * hm * (kn[s] ? 1.f : 0.f);
        }
    } else {
        w[0] = kn[0] ? cf.cdx : 0.f;
        w[1] = kn[1] ? cf.cdx : 0.f;
        w[2] = kn[2] ? cf.cdy : 0.f;
        w[3] = kn[3] ? cf.cdy : 0.f;
        w[4] = kn[4] ? cf.cdz : 0.f;
        w[5] = kn[5] ? cf.cdz : 0.f;
    }
    if constexpr (VEL) {
        const float h[3] = {0.5f * cf.hx, 0.5f * cf.hy, 0.5f * cf.hz};
#pragma unroll
        for (int ax = 0; ax < 3; ax++) {
            const int m = 2 * ax, p = m + 1;
            const float v = adv[ax];
            if constexpr (ST == GEN_UPWIND) {
                const float wm = fmaf(h[ax], pos(v), w[m]);
                const float wp = fmaf(-h[ax], neg(v), w[p]);
                w[m] = (!GEN || !a.amask || kn[m]) ? wm : w[m];
                w[p] = (!GEN || !a.amask || kn[p]) ? wp : w[p];
            } else if constexpr (ST == GEN_PREDICT) {
                w[m] = fmaf(kn[m] ? h[ax] : 0.f, v, w[m]);
            } else {
                w[p] = fmaf(kn[p] ? -h[ax] : 0.f, v, w[p]);
            }
        }
    }
    const float nsx = solid_faces(G, 0), nsy = solid_faces(G, 2), nsz = solid_faces(G, 4);
    float rate2;
    if constexpr (COEF) rate2 = ldw(a.r2v, slot);
    else rate2 = fmaf(cf.s2z, nsz, fmaf(cf.s2y, nsy, fmaf(cf.s2x, nsx, cf.r2)));

    float d[NC];
#pragma unroll
    for (int q = 0; q < NC; q++) {
        const float m = mc[q];
        float t = w[0] * (fn[0][q] - m);
        t = fmaf(w[1], fn[1][q] - m, t);
        t = fmaf(w[2], fn[2][q] - m, t);
        t = fmaf(w[3], fn[3][q] - m, t);
        t = fmaf(w[4], fn[4][q] - m, t);
        d[q] = fmaf(w[5], fn[5][q] - m, t);
    }
    float thz = cf.bgz * G.zc;
    if constexpr (NC == 3) {
        const uint32_t xy = ldw(a.xy, slot);
        float thx = cf.bgx * ((float)(xy & 0xffffu) + 0.5f);
        float thy = cf.bgy * ((float)(xy >> 16) + 0.5f);
        if (GEN && a.bn) {
            const float tb = cf.dtg * ldw(a.bn, slot);
            thx = a.bnax == 0 ? tb : thx;
            thy = a.bnax == 1 ? tb : thy;
            thz = a.bnax == 2 ? tb : thz;
        }
        float rate1;
        if (COEF && a.r1v) rate1 = ldw(a.r1v, slot);
        else rate1 = fmaf(cf.s1z, nsz, fmaf(cf.s1y, nsy, fmaf(cf.s1x, nsx, cf.r1)));
        const float par = fmaf(cf.n2, mc[2], fmaf(cf.n1, mc[1], cf.n0 * mc[0]));
        const float nn[3] = {cf.n0, cf.n1, cf.n2};
#pragma unroll
        for (int q = 0; q < 3; q++) {
            const float mpar = nn[q] * par;
            d[q] = fmaf(rate1, fmaf(cf.peq, nn[q], -mpar), d[q]);
            d[q] = fmaf(rate2, mpar - mc[q], d[q]);
        }
        d[0] = fmaf(thz, mc[1], fmaf(-thy, mc[2], d[0]));
        d[1] = fmaf(-thz, mc[0], fmaf(thx, mc[2], d[1]));
        d[2] = fmaf(thy, mc[0], fmaf(-thx, mc[1], d[2]));
    } else {
#pragma unroll
        for (int q = 0; q < NC; q++) d[q] = fmaf(-rate2, mc[q], d[q]);
        if constexpr (NC == 2) {
            if constexpr (EXACT) {
                // plane_rotation: the angle is uniform in the group, and 0
                // between the gradient's lobes, where sinf is not needed
                float sn = thz, h = 0.5f * thz;
                if (thz != 0.f) {
                    sn = sinf(thz);
                    h = sinf(h);
                }
                const float cm1 = -2.f * h * h;
                d[0] = fmaf(mc[1], sn, fmaf(mc[0], cm1, d[0]));
                d[1] = fmaf(-mc[0], sn, fmaf(mc[1], cm1, d[1]));
            } else {
                if (GEN && a.bn && a.bnax == 2) thz = cf.dtg * ldw(a.bn, slot);
                d[0] = fmaf(thz, mc[1], d[0]);
                d[1] = fmaf(-thz, mc[0], d[1]);
            }
        }
    }
    const bool act = lane_in(G.active);
    Vec<NC> out;
    if constexpr (ST == GEN_CORRECT) {
        const Vec<NC> mav = ldm<NC>(a.mavg, slot);
#pragma unroll
        for (int q = 0; q < NC; q++) {
            float v = 0.5f * (mav[q] + (mc[q] + d[q]));
            have_v(v);
            out[q] = act ? v : 0.f;
        }
    } else {
#pragma unroll
        for (int q = 0; q < NC; q++) {
            float v = mc[q] + d[q];
            have_v(v);
            out[q] = act ? v : (ST == GEN_PREDICT ? 0.f : mc[q]);
        }
    }
    stm<NC>(a.out, slot, out);
    if constexpr (ST != GEN_PREDICT) {
        const bool win = lane_in(G.window);
        if constexpr (NS == 2 * NC) {
            const double w1 = (double)ldw(a.w[0], slot), w2 = (double)ldw(a.w[1], slot);
#pragma unroll
            for (int q = 0; q < NC; q++) {
                const double v = (double)(win ? out[q] : 0.f);
                acc[q] += v * w1;
                acc[NC + q] += v * w2;
            }
        } else {
#pragma unroll
            for (int q = 0; q < NC; q++) acc[q] += (double)(win ? out[q] : 0.f);
        }
    }
}

// One domain: workgroup t takes groups [first + t*gpt, first + (t+1)*gpt),
// its four wavefronts in turn.
template <int NC, bool VEL, int ST, bool EXACT, bool GEN, bool COEF, bool W>
__global__ void __launch_bounds__(kThreads) pore_kernel(PoreArgs a)
{
    constexpr int NS = W ? 2 * NC : NC;
    __shared__ double sred[ST == GEN_PREDICT ? 1 : kWaves - 1][NS][64];
    const int t = xcd_tile(blockIdx.x, a.ntiles);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int g0 = 1 + t * a.gpt, g1 = min(g0 + a.gpt, a.ngroups);
    double acc[NS];
#pragma unroll
    for (int q = 0; q < NS; q++) acc[q] = 0.0;
    for (int g = g0 + wave; g < g1; g += kWaves) pore_step<NC, VEL, ST, EXACT, GEN, COEF, NS>(a, a.c, g, acc);
    if constexpr (ST != GEN_PREDICT) group_reduce<NS>(acc, sred, a.partials + (size_t)t * NS);
}

// Pore sums of the state over the signal window (weights: phase-weighted).
template <int NC, bool W>
__global__ void __launch_bounds__(kThreads) pore_sum_kernel(PoreArgs a)
{
    constexpr int NS = W ? 2 * NC : NC;
    __shared__ double sred[kWaves - 1][NS][64];
    const int t = blockIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int g0 = 1 + t * a.gpt, g1 = min(g0 + a.gpt, a.ngroups);
    double acc[NS];
#pragma unroll
    for (int q = 0; q < NS; q++) acc[q] = 0.0;
    for (int g = g0 + wave; g < g1; g += kWaves) {
        if (!lane_in(group_at(a.groups, g)->window)) continue;
        const uint32_t slot = (uint32_t)g * 64u + (threadIdx.x & 63u);
        const Vec<NC> m = ldm<NC>(a.f, slot);
        if constexpr (W) {
            const double w1 = (double)ldw(a.w[0], slot), w2 = (double)ldw(a.w[1], slot);
#pragma unroll
            for (int q = 0; q < NC; q++) {
                acc[q] += (double)m[q] * w1;
                acc[NC + q] += (double)m[q] * w2;
            }
        } else {
#pragma unroll
            for (int q = 0; q < NC; q++) acc[q] += (double)m[q];
        }
    }
    group_reduce<NS>(acc, sred, a.partials + (size_t)t * NS);
}

// ---- building the list ----

// Whether voxel (x, y, z) gets a slot: a pore, or a solid whose value a pore
// can read -- across a face when solids are read (upwind with velocity on
// pore-solid faces), or as a periodic ghost (the opposite voxel of an edge
// pore, solid or not).
__device__ __forceinline__ bool has_slot(const PoreBuild& b, int x, int y, int z)
{
    const int c[3] = {x, y, z}, n[3] = {b.nx, b.ny, b.nz};
    const size_t st[3] = {1, (size_t)b.pitch, (size_t)b.ny * (size_t)b.pitch};
    const size_t o = (size_t)z * st[2] + (size_t)y * st[1] + (size_t)x;
    if (b.mask[o]) return true;
    for (int ax = 0; ax < 3; ax++) {
        if (b.read_solids) {
            if (c[ax] > 0 && b.mask[o - st[ax]]) return true;
            if (c[ax] < n[ax] - 1 && b.mask[o + st[ax]]) return true;
        }
        if (b.bc[ax] == BC_PERIODIC) {
            if (c[ax] == 0 && b.mask[o + (size_t)(n[ax] - 1) * st[ax]]) return true;
            if (c[ax] == n[ax] - 1 && b.mask[o - (size_t)(n[ax] - 1) * st[ax]]) return true;
        }
    }
    return false;
}

// Slots per row (y, z): one wavefront a row.
__global__ void __launch_bounds__(kThreads) pore_count_kernel(PoreBuild b)
{
    const int64_t row = (int64_t)blockIdx.x * kWaves + (threadIdx.x >> 6);
    if (row >= (int64_t)b.ny * b.nz) return;
    const int lane = threadIdx.x & 63;
    const int y = (int)(row % b.ny), z = (int)(row / b.ny);
    int n = 0;
    for (int x0 = 0; x0 < b.nx; x0 += 64) {
        const int x = x0 + lane;
        n += __popcll(__ballot(x < b.nx && has_slot(b, x, y, z)));
    }
    if (lane == 0) b.rows[row] = (uint32_t)n;
}

// rows[] of each plane -> exclusive prefix within the plane; planes[z] =
// its slots rounded up to whole groups.  One workgroup a plane.
__global__ void __launch_bounds__(kThreads) pore_plane_kernel(PoreBuild b)
{
    __shared__ uint32_t sh[kThreads];
    const int z = blockIdx.x, t = threadIdx.x;
    uint32_t* r = b.rows + (size_t)z * b.ny;
    uint32_t carry = 0;
    for (int y0 = 0; y0 < b.ny; y0 += kThreads) {
        const int y = y0 + t;
        const uint32_t v = y < b.ny ? r[y] : 0u;
        sh[t] = v;
        __syncthreads();
        for (int h = 1; h < kThreads; h <<= 1) {
            const uint32_t u = t >= h ? sh[t - h] : 0u;
            __syncthreads();
            sh[t] += u;
            __syncthreads();
        }
        if (y < b.ny) r[y] = carry + sh[t] - v;
        carry += sh[kThreads - 1];
        __syncthreads();
    }
    if (t == 0) b.planes[z] = ((uint64_t)carry + 63u) & ~(uint64_t)63u;
}

// planes[] -> exclusive prefix starting at `first`; planes[nz] = the end.
// One workgroup.
__global__ void __launch_bounds__(kThreads) pore_base_kernel(PoreBuild b)
{
    __shared__ uint64_t sh[kThreads];
    const int t = threadIdx.x;
    uint64_t carry = b.first;
    for (int z0 = 0; z0 < b.nz; z0 += kThreads) {
        const int z = z0 + t;
        const uint64_t v = z < b.nz ? b.planes[z] : 0u;
        sh[t] = v;
        __syncthreads();
        for (int h = 1; h < kThreads; h <<= 1) {
            const uint64_t u = t >= h ? sh[t - h] : 0u;
            __syncthreads();
            sh[t] += u;
            __syncthreads();
        }
        if (z < b.nz) b.planes[z] = carry + sh[t] - v;
        carry += sh[kThreads - 1];
        __syncthreads();
    }
    if (t == 0) b.planes[b.nz] = carry;
}

// Slot of every voxel (slotmap, 0: none) and voxel of every slot (vox).
__global__ void __launch_bounds__(kThreads) pore_assign_kernel(PoreBuild b)
{
    const int64_t row = (int64_t)blockIdx.x * kWaves + (threadIdx.x >> 6);
    if (row >= (int64_t)b.ny * b.nz) return;
    const int lane = threadIdx.x & 63;
    const int y = (int)(row % b.ny), z = (int)(row / b.ny);
    uint32_t s0 = (uint32_t)b.planes[z] + b.rows[row];
    for (int x0 = 0; x0 < b.nx; x0 += 64) {
        const int x = x0 + lane;
        const bool in = x < b.nx && has_slot(b, x, y, z);
        const uint64_t m = __ballot(in);
        const uint32_t s = s0 + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
        const size_t o = (size_t)row * (size_t)b.pitch + (size_t)x;
        if (x < b.nx) b.slotmap[o] = in ? s : 0u;
        if (in) b.vox[s] = (uint32_t)o;
        s0 += (uint32_t)__popcll(m);
    }
}

// Descriptor and neighbour offsets of the group of every wavefront.
__global__ void __launch_bounds__(kThreads) pore_link_kernel(PoreBuild b)
{
    const int64_t gi = (int64_t)blockIdx.x * kWaves + (threadIdx.x >> 6);
    const int64_t g = (int64_t)(b.first / 64) + gi;
    if (gi >= b.count) return;
    const int lane = threadIdx.x & 63;
    const uint32_t slot = (uint32_t)g * 64u + (uint32_t)lane;
    const uint32_t o = b.vox[slot];
    const bool used = o != 0xffffffffu;
    const uint32_t P = (uint32_t)b.pitch, plane = (uint32_t)b.ny * P;
    const int z = used ? (int)(o / plane) : 0;
    const uint32_t in = used ? o % plane : 0u;
    const int y = (int)(in / P), x = (int)(in % P);
    const bool act = used && b.mask[o] != 0;
    const int c[3] = {x, y, z}, n[3] = {b.nx, b.ny, b.nz};
    const uint32_t st[3] = {1u, P, plane};

    // neighbour slots: kOwn / kZero codes, else a slot number
    uint32_t nbs[6];
    bool own[6], zero[6], pore[6], ghost[6];
#pragma unroll
    for (int s = 0; s < 6; s++) {
        const int ax = s >> 1, up = s & 1;
        own[s] = true;
        zero[s] = pore[s] = ghost[s] = false;
        nbs[s] = 0;
        if (!act) continue;
        const bool edge = up ? c[ax] == n[ax] - 1 : c[ax] == 0;
        if (!edge) {
            const uint32_t v = up ? o + st[ax] : o - st[ax];
            pore[s] = b.mask[v] != 0;
            if (pore[s] || b.read_solids) {
                nbs[s] = b.slotmap[v];
                own[s] = nbs[s] == 0;
            }
        } else {
            pore[s] = ghost[s] = true;
            if (b.bc[ax] == BC_PERIODIC) {
                const uint32_t d = (uint32_t)(n[ax] - 1) * st[ax];
                nbs[s] = b.slotmap[up ? o - d : o + d];
                own[s] = false;
            } else if (b.bc[ax] == BC_DIRICHLET) {
                zero[s] = true;
                own[s] = false;
            }
        }
    }
    uint32_t base[6], off[6];
    bool over = false;
#pragma unroll
    for (int s = 0; s < 6; s++) {
        const bool at = !own[s] && !zero[s];
        uint32_t lo = at ? nbs[s] : 0xffffffffu;
        for (int h = 32; h > 0; h >>= 1) lo = min(lo, (uint32_t)__shfl_xor((int)lo, h, 64));
        base[s] = lo == 0xffffffffu ? 0u : lo;
        if (s == 2 || s == 3) { // signed distance
            const int64_t d = at ? (int64_t)nbs[s] - (int64_t)slot : 0;
            if (d < -32767 || d > 32767) over = true;
            off[s] = zero[s] ? kZeroY : ((uint32_t)(int32_t)d & 0xffffu);
        } else {
            const uint32_t d = at ? nbs[s] - base[s] : 0u;
            const bool x_next = s < 2 && !b.xoff; // the slot next to this one
            if (at && !x_next && d >= kZero) over = true;
            off[s] = own[s] ? kOwn : (zero[s] ? kZero : (d & 0xffffu));
        }
    }
    if (over) *b.overflow = 1;
    b.off[slot] = make_uint2(off[2] | (off[3] << 16), off[4] | (off[5] << 16));
    if (b.xoff) b.xoff[slot] = off[0] | (off[1] << 16);
    if (b.xy) b.xy[slot] = (uint32_t)x | ((uint32_t)y << 16);
    const bool win = act && x >= b.w[0] && x < b.w[1] && y >= b.w[2] && y < b.w[3] && z >= b.w[4] && z < b.w[5];
    const uint64_t any = __ballot(used);
    const int first = any ? (int)__ffsll((unsigned long long)any) - 1 : 0;
    const int gz = __shfl(z, first, 64);
    uint64_t pm[6], gm[6];
#pragma unroll
    for (int s = 0; s < 6; s++) {
        pm[s] = __ballot(pore[s]);
        gm[s] = __ballot(ghost[s]);
    }
    const uint64_t am = __ballot(act), wm = __ballot(win), xm = __ballot(!own[0]), xp = __ballot(!own[1]);
    const uint64_t zm = __ballot(!own[4]), zp = __ballot(!own[5]);
    if (lane == 0) {
        PoreGroup G{};
        for (int s = 0; s < 6; s++) {
            G.base[s] = (int32_t)base[s];
            G.pore[s] = pm[s];
        }
        G.zc = (float)gz + 0.5f;
        G.active = am;
        G.window = wm;
        G.xm = xm;
        G.xp = xp;
        G.zm = zm;
        G.zp = zp;
        b.groups[g] = G;
        if (b.ghost)
            for (int s = 0; s < 6; s++) b.ghost[g].side[s] = gm[s];
    }
}

// Words of the row arrays at the slots: out[stride*slot + at] = row[vox[slot]], 0 at empty slots.
__global__ void __launch_bounds__(kThreads) pore_gather_kernel(const float* __restrict__ row,
                                                               const uint32_t* __restrict__ vox, uint32_t s0,
                                                               uint32_t s1, int stride, int at,
                                                               float* __restrict__ out)
{
    const uint32_t s = s0 + blockIdx.x * (uint32_t)kThreads + threadIdx.x;
    if (s >= s1) return;
    const uint32_t o = vox[s];
    out[(size_t)s * stride + at] = o != 0xffffffffu ? row[o] : 0.f;
}

// The state of the slots (nc components) back into one row array.
__global__ void __launch_bounds__(kThreads) pore_scatter_kernel(const float* __restrict__ f,
                                                                const uint32_t* __restrict__ vox, uint32_t s0,
                                                                uint32_t s1, int stride, int at,
                                                                float* __restrict__ row, float* __restrict__ row2)
{
    const uint32_t s = s0 + blockIdx.x * (uint32_t)kThreads + threadIdx.x;
    if (s >= s1) return;
    const uint32_t o = vox[s];
    if (o == 0xffffffffu) return;
    const float v = f[(size_t)s * stride + at];
    row[o] = v;
    if (row2) row2[o] = v;
}

// *flag = 1 when a solid holds a value that is not finite.
__global__ void __launch_bounds__(kThreads) solids_finite_kernel(const float* __restrict__ row,
                                                                 const uint8_t* __restrict__ mask, size_t n,
                                                                 int* flag)
{
    bool bad = false;
    for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (size_t)gridDim.x * kThreads)
        bad |= mask[i] == 0 && !isfinite(row[i]);
    if (bad) *flag = 1;
}

} // namespace

// Rotation of the state of every pore in the list (pulse_kernel's angles and
// arithmetic, nmr_kernels.hip).
__global__ void __launch_bounds__(kThreads) pore_pulse_kernel(PulseArgs a, float* __restrict__ f, int nc,
                                                              const uint32_t* __restrict__ vox, uint32_t s0,
                                                              uint32_t s1)
{
    const uint32_t s = s0 + blockIdx.x * (uint32_t)kThreads + threadIdx.x;
    if (s >= s1) return;
    const uint32_t o = vox[s];
    if (o == 0xffffffffu || a.mask[o] == 0) return;
    const uint32_t plane = (uint32_t)a.ny * (uint32_t)a.pitch;
    const int z = (int)(o / plane), y = (int)(o % plane / (uint32_t)a.pitch), x = (int)(o % (uint32_t)a.pitch);
    pulse_voxel(a, x, y, z, f + (size_t)s * nc, f + (size_t)s * nc + 1, nc == 3 ? f + (size_t)s * nc + 2 : nullptr);
}

hipError_t launch_pore_pulse(const PulseArgs& a, float* f, int nc, const uint32_t* vox, uint32_t s0, uint32_t s1,
                             hipStream_t s)
{
    if (s1 <= s0) return hipSuccess;
    hipLaunchKernelGGL(pore_pulse_kernel, dim3((s1 - s0 + kThreads - 1) / kThreads), dim3(kThreads), 0, s, a, f, nc, vox,
                       s0, s1);
    return hipGetLastError();
}

hipError_t launch_pore_count(const PoreBuild& b, hipStream_t s)
{
    const int64_t nrows = (int64_t)b.ny * b.nz;
    hipLaunchKernelGGL(pore_count_kernel, dim3((unsigned)((nrows + kWaves - 1) / kWaves)), dim3(kThreads), 0, s, b);
    hipLaunchKernelGGL(pore_plane_kernel, dim3((unsigned)b.nz), dim3(kThreads), 0, s, b);
    hipLaunchKernelGGL(pore_base_kernel, dim3(1), dim3(kThreads), 0, s, b);
    return hipGetLastError();
}

hipError_t launch_pore_link(const PoreBuild& b, hipStream_t s)
{
    const int64_t nrows = (int64_t)b.ny * b.nz;
    hipLaunchKernelGGL(pore_assign_kernel, dim3((unsigned)((nrows + kWaves - 1) / kWaves)), dim3(kThreads), 0, s, b);
    if (b.count > 0)
        hipLaunchKernelGGL(pore_link_kernel, dim3((unsigned)((b.count + kWaves - 1) / kWaves)), dim3(kThreads), 0, s,
                           b);
    return hipGetLastError();
}

hipError_t launch_pore_gather(const float* row, const uint32_t* vox, uint32_t s0, uint32_t s1, int stride, int at,
                              float* out, hipStream_t s)
{
    if (s1 <= s0) return hipSuccess;
    hipLaunchKernelGGL(pore_gather_kernel, dim3((s1 - s0 + kThreads - 1) / kThreads), dim3(kThreads), 0, s, row, vox, s0,
                       s1, stride, at, out);
    return hipGetLastError();
}

hipError_t launch_pore_scatter(const float* f, const uint32_t* vox, uint32_t s0, uint32_t s1, int stride, int at,
                               float* row, float* row2, hipStream_t s)
{
    if (s1 <= s0) return hipSuccess;
    hipLaunchKernelGGL(pore_scatter_kernel, dim3((s1 - s0 + kThreads - 1) / kThreads), dim3(kThreads), 0, s, f, vox, s0,
                       s1, stride, at, row, row2);
    return hipGetLastError();
}

hipError_t launch_solids_finite(const float* row, const uint8_t* mask, size_t n, int* flag, hipStream_t s)
{
    const unsigned grid = (unsigned)std::min<size_t>(4096, (n + kThreads - 1) / kThreads);
    hipLaunchKernelGGL(solids_finite_kernel, dim3(std::max(1u, grid)), dim3(kThreads), 0, s, row, mask, n, flag);
    return hipGetLastError();
}

hipError_t launch_pore_sum(int nc, const PoreArgs& a, hipStream_t s)
{
    const dim3 grid((unsigned)a.ntiles), block(kThreads);
    const bool w = a.w[0] != nullptr;
#define SUM(N)                                                                           \
    case N:                                                                              \
        if (w) hipLaunchKernelGGL((pore_sum_kernel<N, true>), grid, block, 0, s, a);     \
        else hipLaunchKernelGGL((pore_sum_kernel<N, false>), grid, block, 0, s, a);      \
        break
    switch (nc) {
        SUM(1);
        SUM(2);
        SUM(3);
    default: return hipErrorInvalidValue;
    }
#undef SUM
    return hipGetLastError();
}

namespace {

template <int NC, bool VEL, int ST, bool EXACT>
void launch_pores_st(bool gen, bool coef, const PoreArgs& a, hipStream_t s)
{
    const dim3 grid((unsigned)a.ntiles), block(kThreads);
    if constexpr (EXACT) {
        hipLaunchKernelGGL((pore_kernel<NC, VEL, ST, true, false, false, false>), grid, block, 0, s, a);
    } else {
        const bool w = a.w[0] != nullptr && ST != GEN_PREDICT;
        if (!gen) hipLaunchKernelGGL((pore_kernel<NC, VEL, ST, false, false, false, false>), grid, block, 0, s, a);
        else if (coef && w) hipLaunchKernelGGL((pore_kernel<NC, VEL, ST, false, true, true, ST != GEN_PREDICT>), grid, block, 0, s, a);
        else if (coef) hipLaunchKernelGGL((pore_kernel<NC, VEL, ST, false, true, true, false>), grid, block, 0, s, a);
        else if (w) hipLaunchKernelGGL((pore_kernel<NC, VEL, ST, false, true, false, ST != GEN_PREDICT>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((pore_kernel<NC, VEL, ST, false, true, false, false>), grid, block, 0, s, a);
    }
}

template <int NC, bool VEL>
hipError_t launch_pores_nc(int st, bool exact, bool gen, bool coef, const PoreArgs& a, hipStream_t s)
{
    if (exact) {
        if constexpr (NC == 2) launch_pores_st<NC, VEL, GEN_UPWIND, true>(gen, coef, a, s);
        else return hipErrorInvalidValue;
    } else if (st == GEN_UPWIND) {
        launch_pores_st<NC, VEL, GEN_UPWIND, false>(gen, coef, a, s);
    } else if (st == GEN_PREDICT) {
        launch_pores_st<NC, VEL, GEN_PREDICT, false>(gen, coef, a, s);
    } else {
        launch_pores_st<NC, VEL, GEN_CORRECT, false>(gen, coef, a, s);
    }
    return hipGetLastError();
}

} // namespace

hipError_t launch_pores(int nc, bool vel, int st, bool exact, bool gen, bool coef, const PoreArgs& a, hipStream_t s)
{
    if (a.ntiles < 1 || a.gpt < 1) return hipErrorInvalidValue;
#define GO(N, V) \
    case 2 * N + V: return launch_pores_nc<N, (V) != 0>(st, exact, gen, coef, a, s)
    switch (nc * 2 + (vel ? 1 : 0)) {
        GO(1, 0);
        GO(1, 1);
        GO(2, 0);
        GO(2, 1);
        GO(3, 0);
        GO(3, 1);
    default: return hipErrorInvalidValue;
    }
#undef GO
}

} // namespace nmr
