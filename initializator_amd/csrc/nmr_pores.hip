// nmr_pores.hip -- the sweeps over a list of the pores (gfx950).
//
// Only pores change in a step, and in a porous medium they are a fifth to a
// third of the voxels.  The tile sweeps (nmr_kernels.hip) stream the grid and
// skip what is all solid, but a 4-voxel chunk or 128-byte brick with one pore
// costs as much as a full one.  Here the state of the pores is kept as a
// list: 64 slots to a group, in the grid's order, so that the wavefront of a
// group has a pore in every lane.  A slot's x neighbours are the slots next
// to it; its y and z neighbours are given as 8-bit offsets from four bases of
// the group (16-bit ones where a group needs them), packed with the three
// velocity sums into one 16-byte record; which neighbours are pores, and
// which lanes count in the signal, are 64-bit lane masks of the group's
// descriptor, read into scalar registers and used as lane conditions
// directly.  A group never spans two planes, so z and the precession angle of
// a z gradient are uniform in a wavefront.
//
// What bounds it: bytes past the L2.  A step moves 34 a pore -- two
// components read and written (16), the record (16), the descriptor (2) --
// less than half of the tile sweep's a voxel at 20 % porosity; the neighbours
// are L1 and L2 hits (each XCD takes a contiguous run of workgroups).  256^3,
// porosity 0.2, flow and gradient: 19.9 us a step (the tile sweep on bricks:
// 57.9; this list with 16-bit offsets and a separate 12-byte velocity: 20.6),
// of which about 4 are the launch's ramp and tail; 123 MB past the L2 in the
// rest, 7.6 TB/s, what a copy inside the memory-side cache reaches (7.7-8.3).
// 512x512x130 (231 MB a step): 35.3 us, 6.5 TB/s.  Not what bounds it: the
// gathers (left out: the same time), the vector instructions (131 or 85 a
// group: the same), L1 accesses (halved by staging the neighbourhood in LDS:
// the same, and slower with three components or periodic rows).
//
// The arithmetic of a voxel is that of the tile sweeps (update_chunk,
// gupdate_chunk) and of general_kernel, operation by operation, so the fields
// are the same bits.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "nmr_device.h"
#include "nmr_kernels.h"
#include "nmr_pore_device.h"

namespace nmr {

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
// Group descriptors are read through the constant address space: uniform
// loads from it go to scalar registers, also in a loop that stores.
typedef const __attribute__((address_space(4))) PoreGroup* GroupPtr;
typedef const __attribute__((address_space(4))) PoreAux* AuxPtr;
typedef const __attribute__((address_space(4))) PoreTile* TilePtr;
typedef const __attribute__((address_space(4))) PoreInst* InstPtr;
__device__ __forceinline__ GroupPtr group_at(const PoreGroup* g, int i) { return (GroupPtr)(uintptr_t)(g + i); }

__device__ __forceinline__ bool lane_in(uint64_t mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }

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
    uint32_t base[6], wide;
    float zc;
    uint64_t pore[6], active, window, xm, xp;
    __device__ __forceinline__ void load(GroupPtr G)
    {
#pragma unroll
        for (int s = 0; s < 6; s++) base[s] = G->base[s];
        wide = G->wide;
        zc = G->zc;
#pragma unroll
        for (int s = 0; s < 6; s++) pore[s] = G->pore[s];
        active = G->active;
        window = G->window;
        xm = G->xm;
        xp = G->xp;
        // the compiler would sink these loads into branches around the
        // selects that use them, one dependent wait each
#pragma unroll
        for (int s = 2; s < 6; s++) have_s(base[s]);
        have_s(xm);
        have_s(xp);
    }
};

// Byte offsets, K bytes a slot, of the neighbours x-, x+, y-, y+, z-, z+ of a
// slot.  A side with nothing to read gives the slot itself.
template <int K, bool GEN, bool WIDE>
__device__ __forceinline__ void neighbours(const PoreArgs& a, const GroupRegs& G, int g, uint32_t off8, uint32_t slot,
                                           uint32_t (&nb)[6])
{
    const uint32_t own = slot * (uint32_t)K;
    nb[0] = lane_in(G.xm) ? own - (uint32_t)K : own;
    nb[1] = lane_in(G.xp) ? own + (uint32_t)K : own;
    uint32_t o[4] = {off8 & 0xffu, (off8 >> 8) & 0xffu, (off8 >> 16) & 0xffu, off8 >> 24};
    if (WIDE && G.wide) { // some neighbour lies more than 255 slots from its base
        const uint2 o16 = ldw(a.off16, slot);
        o[0] = o16.x & 0xffffu;
        o[1] = o16.x >> 16;
        o[2] = o16.y & 0xffffu;
        o[3] = o16.y >> 16;
    }
    uint32_t v[6];
#pragma unroll
    for (int s = 2; s < 6; s++) {
        v[s] = o[s - 2] * (uint32_t)K + G.base[s] * (uint32_t)K;
        nb[s] = lane_in(G.pore[s]) ? v[s] : own; // pores and ghosts are read, solids are not
    }
    if constexpr (GEN) {
        if (a.xoff) {
            const uint32_t xo = ldw(a.xoff, slot);
            v[0] = ((xo & 0xffffu) + G.base[0]) * (uint32_t)K;
            v[1] = ((xo >> 16) + G.base[1]) * (uint32_t)K;
            nb[0] = lane_in(G.pore[0]) ? v[0] : own;
            nb[1] = lane_in(G.pore[1]) ? v[1] : own;
        }
        if (a.aux) { // solids that are read, ghosts that read as 0 (slot 0 stays 0)
            const AuxPtr A = (AuxPtr)(uintptr_t)(a.aux + g);
#pragma unroll
            for (int s = 0; s < 6; s++) {
                if (s >= 2 || a.xoff) nb[s] = lane_in(A->has[s]) ? v[s] : own;
                nb[s] = lane_in(A->zero[s]) ? 0u : nb[s];
            }
        }
    }
}

// Faces to solids on the axis of sides m and m+1: 0, 1 or 2 from the lane masks.
__device__ __forceinline__ float solid_faces(const GroupRegs& G, int m)
{
    const uint64_t any = ~(G.pore[m] & G.pore[m + 1]), both = ~(G.pore[m] | G.pore[m + 1]);
    const float n = lane_in(any) ? 1.f : 0.f;
    return lane_in(both) ? 2.f : n;
}

// One step (or MacCormack stage ST) of the 64 slots of group g, lane by lane.
// GEN: per-voxel field, masked advection, non-zero-derivative ghosts and
// phase weights may be present (null pointers and flags say which); COEF:
// per-voxel diffusivity and rates; WIDE: some group needs its 16-bit offsets.
template <int NC, bool VEL, int ST, bool EXACT, bool GEN, bool COEF, bool WIDE, int NS>
__device__ __forceinline__ void pore_step(const PoreArgs& a, const Coef& cf, const int g, double (&acc)[NS])
{
    constexpr int K = 4 * NC;
    const uint32_t slot = (uint32_t)g * 64u + (threadIdx.x & 63u);
    uint32_t off8;
    float adv[3] = {0.f, 0.f, 0.f};
    if constexpr (VEL) {
        const uint4 r = ldw(a.rec, slot);
        off8 = r.x;
        adv[0] = __uint_as_float(r.y);
        adv[1] = __uint_as_float(r.z);
        adv[2] = __uint_as_float(r.w);
    } else {
        off8 = ldw(a.off8, slot);
    }
    const Vec<NC> mc = at_byte<Vec<NC>>(a.f, slot * (uint32_t)K);
    GroupRegs G;
    G.load(group_at(a.groups, g));
    uint32_t nb[6];
    neighbours<K, GEN, WIDE>(a, G, g, off8, slot, nb);
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
        neighbours<4, GEN, WIDE>(a, G, g, off8, slot, nd);
        const float dc = ldw(a.dn, slot);
        const float cd[3] = {cf.cdx, cf.cdy, cf.cdz};
#pragma unroll
        for (int s = 0; s < 6; s++) {
            float dnb = at_byte<float>(a.dn, nd[s]);
            // ghosts carry the diffusivity of the voxel they border
            if (a.ghost && lane_in(((AuxPtr)(uintptr_t)(a.ghost + g))->ghost[s])) dnb = dc;
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
        const Vec<NC> mav = at_byte<Vec<NC>>(a.mavg, slot * (uint32_t)K);
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

template <bool BATCH>
__device__ __forceinline__ void tile_range(const PoreArgs& a, int t, int& g0, int& g1, uint32_t& inst)
{
    inst = 0;
    if constexpr (BATCH) {
        const TilePtr T = (TilePtr)(uintptr_t)(a.tiles + t);
        g0 = (int)T->first;
        g1 = g0 + (int)T->count;
        inst = T->inst;
    } else {
        g0 = 1 + t * a.gpt;
        g1 = min(g0 + a.gpt, a.ngroups);
    }
}

// Coefficients of the step: the launch's, or in a batch the instance's with
// the gradient of its pulsed-gradient pair at this step (+G on steps [0, nd),
// -G on [nD, nD + nd), the second lobe where they overlap).
template <bool BATCH>
__device__ __forceinline__ Coef step_coef(const PoreArgs& a, uint32_t inst)
{
    if constexpr (!BATCH) return a.c;
    const InstPtr I = (InstPtr)(uintptr_t)(a.inst + inst);
    Coef c;
    const __attribute__((address_space(4))) float* s = (const __attribute__((address_space(4))) float*)&I->c;
    float* d = reinterpret_cast<float*>(&c);
#pragma unroll
    for (unsigned k = 0; k < sizeof(Coef) / 4; k++) d[k] = s[k];
    const int step = *a.step_base + a.local_step;
    c.bgz = (step >= I->nD && step < I->nD + I->nd) ? -I->bgz : (step < I->nd ? I->bgz : 0.f);
    return c;
}

// Workgroup t takes tile t's groups, its wavefronts in turn: of one domain
// gpt consecutive groups, of a batch what the tile list says.
template <int NC, bool VEL, int ST, bool EXACT, bool GEN, bool COEF, bool W, bool BATCH, bool WIDE>
__global__ void __launch_bounds__(kThreads) pore_kernel(PoreArgs a)
{
    constexpr int NS = W ? 2 * NC : NC;
    __shared__ double sred[ST == GEN_PREDICT ? 1 : kWaves - 1][NS][64];
    const int t = xcd_tile(blockIdx.x, a.ntiles);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    int g0, g1;
    uint32_t inst;
    tile_range<BATCH>(a, t, g0, g1, inst);
    const Coef cf = step_coef<BATCH>(a, inst);
    double acc[NS];
#pragma unroll
    for (int q = 0; q < NS; q++) acc[q] = 0.0;
    for (int g = g0 + wave; g < g1; g += kWaves) pore_step<NC, VEL, ST, EXACT, GEN, COEF, WIDE, NS>(a, cf, g, acc);
    if constexpr (ST != GEN_PREDICT) group_reduce<NS>(acc, sred, a.partials + (size_t)t * NS);
}

// Pore sums of the state over the signal window (weights: phase-weighted),
// one partial a tile.
template <int NC, bool W, bool BATCH>
__global__ void __launch_bounds__(kThreads) pore_sum_kernel(PoreArgs a)
{
    constexpr int NS = W ? 2 * NC : NC;
    __shared__ double sred[kWaves - 1][NS][64];
    const int t = blockIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    int g0, g1;
    uint32_t inst;
    tile_range<BATCH>(a, t, g0, g1, inst);
    double acc[NS];
#pragma unroll
    for (int q = 0; q < NS; q++) acc[q] = 0.0;
    for (int g = g0 + wave; g < g1; g += kWaves) {
        if (!lane_in(group_at(a.groups, g)->window)) continue;
        const uint32_t slot = (uint32_t)g * 64u + (threadIdx.x & 63u);
        const Vec<NC> m = at_byte<Vec<NC>>(a.f, slot * (uint32_t)(4 * NC));
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

// Slots per row (y, z): one wavefront a row, rows in turn where there are more
// than a launch may have threads for.
__global__ void __launch_bounds__(kThreads) pore_count_kernel(PoreBuild b)
{
    const int64_t nrows = (int64_t)b.ny * b.nz;
    const int lane = threadIdx.x & 63;
    for (int64_t row = (int64_t)blockIdx.x * kWaves + (threadIdx.x >> 6); row < nrows; row += (int64_t)gridDim.x * kWaves) {
        const int y = (int)(row % b.ny), z = (int)(row / b.ny);
        int n = 0;
        for (int x0 = 0; x0 < b.nx; x0 += 64) {
            const int x = x0 + lane;
            n += __popcll(__ballot(x < b.nx && has_slot(b, x, y, z)));
        }
        if (lane == 0) b.rows[row] = (uint32_t)n;
    }
}

// rows[] of each plane -> exclusive prefix within the plane; planes[z] =
// its slots rounded up to whole groups.  One workgroup a plane (planes in turn).
__global__ void __launch_bounds__(kThreads) pore_plane_kernel(PoreBuild b)
{
    __shared__ uint32_t sh[kThreads];
    const int t = threadIdx.x;
    for (int z = blockIdx.x; z < b.nz; z += (int)gridDim.x) {
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
    const int64_t nrows = (int64_t)b.ny * b.nz;
    const int lane = threadIdx.x & 63;
    for (int64_t row = (int64_t)blockIdx.x * kWaves + (threadIdx.x >> 6); row < nrows; row += (int64_t)gridDim.x * kWaves) {
        const int y = (int)(row % b.ny), z = (int)(row / b.ny);
        uint32_t s0 = (uint32_t)(b.planes[z] + b.shift) + b.rows[row];
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

    // neighbour slots; a zero-derivative ghost reads the slot itself
    uint32_t nbs[6];
    bool has[6], zero[6], pore[6], ghost[6];
#pragma unroll
    for (int s = 0; s < 6; s++) {
        const int ax = s >> 1, up = s & 1;
        has[s] = zero[s] = pore[s] = ghost[s] = false;
        nbs[s] = 0;
        if (!act) continue;
        const bool edge = up ? c[ax] == n[ax] - 1 : c[ax] == 0;
        if (!edge) {
            const uint32_t v = up ? o + st[ax] : o - st[ax];
            pore[s] = b.mask[v] != 0;
            if (pore[s] || b.read_solids) {
                nbs[s] = b.slotmap[v];
                has[s] = nbs[s] != 0;
            }
        } else {
            pore[s] = ghost[s] = true;
            has[s] = b.bc[ax] != BC_DIRICHLET;
            zero[s] = !has[s];
            nbs[s] = slot;
            if (b.bc[ax] == BC_PERIODIC) {
                const uint32_t d = (uint32_t)(n[ax] - 1) * st[ax];
                nbs[s] = b.slotmap[up ? o - d : o + d];
            }
        }
    }
    // the lowest slot read on each side, and the offsets from it
    uint32_t lo[6];
#pragma unroll
    for (int s = 0; s < 6; s++) {
        lo[s] = has[s] ? nbs[s] : 0xffffffffu;
        for (int h = 32; h > 0; h >>= 1) lo[s] = min(lo[s], (uint32_t)__shfl_xor((int)lo[s], h, 64));
    }
    uint32_t off[6];
    bool wide = false, over = false;
#pragma unroll
    for (int s = 0; s < 6; s++) {
        off[s] = has[s] ? nbs[s] - lo[s] : 0u;
        if (s >= 2 && off[s] > 0xffu) wide = true;
        if ((s >= 2 || b.xoff) && off[s] > 0xffffu) over = true;
    }
    if (over) b.found[0] = 1;
    if (wide) b.found[1] = 1;
    const uint32_t off8 = (off[2] & 0xffu) | (off[3] & 0xffu) << 8 | (off[4] & 0xffu) << 16 | (off[5] & 0xffu) << 24;
    b.off8[slot] = off8;
    if (b.vel[0]) {
        uint4 r = make_uint4(off8, 0u, 0u, 0u);
        if (used) {
            r.y = __float_as_uint(b.vel[0][o]);
            r.z = __float_as_uint(b.vel[1][o]);
            r.w = __float_as_uint(b.vel[2][o]);
        }
        b.rec[slot] = r;
    }
    b.off16[slot] = make_uint2((off[2] & 0xffffu) | off[3] << 16, (off[4] & 0xffffu) | off[5] << 16);
    if (b.xoff) b.xoff[slot] = (off[0] & 0xffffu) | off[1] << 16;
    if (b.xy) b.xy[slot] = (uint32_t)x | ((uint32_t)y << 16);
    const bool win = act && x >= b.w[0] && x < b.w[1] && y >= b.w[2] && y < b.w[3] && z >= b.w[4] && z < b.w[5];
    const uint64_t any = __ballot(used);
    const int first = any ? (int)__ffsll((unsigned long long)any) - 1 : 0;
    const int gz = __shfl(z, first, 64);
    uint64_t pm[6], hm[6], zm[6], gm[6];
#pragma unroll
    for (int s = 0; s < 6; s++) {
        pm[s] = __ballot(pore[s]);
        hm[s] = __ballot(has[s]);
        zm[s] = __ballot(zero[s]);
        gm[s] = __ballot(ghost[s]);
    }
    const uint64_t am = __ballot(act), wm = __ballot(win), wd = __ballot(wide);
    const uint64_t xm = __ballot(has[0] && nbs[0] != slot), xp = __ballot(has[1] && nbs[1] != slot);
    if (lane == 0) {
        PoreGroup G{};
        for (int s = 0; s < 6; s++) {
            G.base[s] = lo[s] == 0xffffffffu ? 0u : lo[s];
            G.pore[s] = pm[s];
        }
        G.zc = (float)gz + 0.5f;
        G.wide = wd != 0;
        G.active = am;
        G.window = wm;
        G.xm = xm;
        G.xp = xp;
        b.groups[g] = G;
        if (b.aux)
            for (int s = 0; s < 6; s++) {
                b.aux[g].has[s] = hm[s];
                b.aux[g].zero[s] = zm[s];
                b.aux[g].ghost[s] = gm[s];
            }
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

// The first word of every record: the packed offsets.
__global__ void __launch_bounds__(kThreads) pore_record_kernel(const uint32_t* __restrict__ off8, uint32_t n,
                                                               uint4* __restrict__ rec)
{
    const uint32_t s = blockIdx.x * (uint32_t)kThreads + threadIdx.x;
    if (s < n) rec[s].x = off8[s];
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

// Workgroups that take a wavefront a row: a launch's threads number below 2^32,
// and a grid within the 4 GiB of its arrays may have 2^28 rows.
constexpr int64_t kMostGroups = (int64_t)1 << 22;
static unsigned row_groups(const PoreBuild& b)
{
    return (unsigned)std::min(kMostGroups, ((int64_t)b.ny * b.nz + kWaves - 1) / kWaves);
}

hipError_t launch_pore_count(const PoreBuild& b, hipStream_t s)
{
    hipLaunchKernelGGL(pore_count_kernel, dim3(row_groups(b)), dim3(kThreads), 0, s, b);
    hipLaunchKernelGGL(pore_plane_kernel, dim3((unsigned)std::min<int64_t>(kMostGroups, b.nz)), dim3(kThreads), 0, s, b);
    hipLaunchKernelGGL(pore_base_kernel, dim3(1), dim3(kThreads), 0, s, b);
    return hipGetLastError();
}

hipError_t launch_pore_link(const PoreBuild& b, hipStream_t s)
{
    hipLaunchKernelGGL(pore_assign_kernel, dim3(row_groups(b)), dim3(kThreads), 0, s, b);
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

hipError_t launch_pore_record(const uint32_t* off8, uint32_t n, uint4* rec, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(pore_record_kernel, dim3((n + kThreads - 1) / kThreads), dim3(kThreads), 0, s, off8, n, rec);
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
#define SUM(N)                                                                                     \
    case N:                                                                                        \
        if (a.inst) hipLaunchKernelGGL((pore_sum_kernel<N, false, true>), grid, block, 0, s, a);   \
        else if (w) hipLaunchKernelGGL((pore_sum_kernel<N, true, false>), grid, block, 0, s, a);   \
        else hipLaunchKernelGGL((pore_sum_kernel<N, false, false>), grid, block, 0, s, a);         \
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

template <int NC, bool VEL, int ST, bool EXACT, bool GEN, bool COEF, bool W, bool BATCH>
hipError_t launch_one(const PoreArgs& a, hipStream_t s)
{
    const dim3 grid((unsigned)a.ntiles), block(kThreads);
    if (a.wide) hipLaunchKernelGGL((pore_kernel<NC, VEL, ST, EXACT, GEN, COEF, W, BATCH, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((pore_kernel<NC, VEL, ST, EXACT, GEN, COEF, W, BATCH, false>), grid, block, 0, s, a);
    return hipGetLastError();
}

template <int NC, bool VEL, int ST>
hipError_t launch_st(bool exact, bool gen, bool coef, const PoreArgs& a, hipStream_t s)
{
    if (exact) {
        if constexpr (NC == 2 && ST == GEN_UPWIND) {
            if (gen) return launch_one<NC, VEL, ST, true, true, false, false, false>(a, s);
            return launch_one<NC, VEL, ST, true, false, false, false, false>(a, s);
        }
        return hipErrorInvalidValue;
    }
    constexpr bool SUMS = ST != GEN_PREDICT; // the predictor has no signal
    const bool w = SUMS && a.w[0] != nullptr;
    if (!gen) return launch_one<NC, VEL, ST, false, false, false, false, false>(a, s);
    if (coef && w) return launch_one<NC, VEL, ST, false, true, true, SUMS, false>(a, s);
    if (coef) return launch_one<NC, VEL, ST, false, true, true, false, false>(a, s);
    if (w) return launch_one<NC, VEL, ST, false, true, false, SUMS, false>(a, s);
    return launch_one<NC, VEL, ST, false, true, false, false, false>(a, s);
}

template <int NC, bool VEL>
hipError_t launch_nc(int st, bool exact, bool gen, bool coef, const PoreArgs& a, hipStream_t s)
{
    if (a.inst) { // a batch: the plain upwind step, solids read or not
        if constexpr (NC == 2) {
            if (exact && gen) return launch_one<NC, VEL, GEN_UPWIND, true, true, false, false, true>(a, s);
            if (exact) return launch_one<NC, VEL, GEN_UPWIND, true, false, false, false, true>(a, s);
        }
        if (exact || coef || st != GEN_UPWIND) return hipErrorInvalidValue;
        if (gen) return launch_one<NC, VEL, GEN_UPWIND, false, true, false, false, true>(a, s);
        return launch_one<NC, VEL, GEN_UPWIND, false, false, false, false, true>(a, s);
    }
    switch (st) {
    case GEN_UPWIND: return launch_st<NC, VEL, GEN_UPWIND>(exact, gen, coef, a, s);
    case GEN_PREDICT: return launch_st<NC, VEL, GEN_PREDICT>(exact, gen, coef, a, s);
    case GEN_CORRECT: return launch_st<NC, VEL, GEN_CORRECT>(exact, gen, coef, a, s);
    default: return hipErrorInvalidValue;
    }
}

} // namespace

hipError_t launch_pores(int nc, bool vel, int st, bool exact, bool gen, bool coef, const PoreArgs& a, hipStream_t s)
{
    if (a.ntiles < 1 || (!a.inst && a.gpt < 1)) return hipErrorInvalidValue;
    switch (nc * 2 + (vel ? 1 : 0)) {
    case 2: return launch_nc<1, false>(st, exact, gen, coef, a, s);
    case 3: return launch_nc<1, true>(st, exact, gen, coef, a, s);
    case 4: return launch_nc<2, false>(st, exact, gen, coef, a, s);
    case 5: return launch_nc<2, true>(st, exact, gen, coef, a, s);
    case 6: return launch_nc<3, false>(st, exact, gen, coef, a, s);
    case 7: return launch_nc<3, true>(st, exact, gen, coef, a, s);
    default: return hipErrorInvalidValue;
    }
}

} // namespace nmr
