// nmr_pore_blocks.hip -- several steps in one launch, for grids whose step is
// bound by its launch (gfx950).
//
// A step over the list of a small grid takes 2.9-3.3 us however few its pores
// are: the launch, three dependent trips to memory (descriptor, state,
// neighbours) and the end.  Here a workgroup takes the pores of a box of
// 8 x 8 x 8 voxels and all those within four faces of it, and advances them
// four steps in LDS without a word from its neighbours: step s brings forward
// the pores within 4 - s faces, so that the box itself is right after the
// last.  A box's pores are listed by distance, so that each step works on the
// first so many.  The halo is computed more than once -- 2.3 times the work
// for a box inside -- which is nothing while the launch is what takes the time.
// 64^3, one component, porosity 0.3: 3.9 -> 2.2 us a step; 48^3, three
// components: 3.8 -> 2.2.  Of the 5.6 us of such a launch about 4 are the launch
// and the trips to memory; a step takes 0.4, the instructions of one wavefront
// in a row.  (512 threads with twice the slots each: 10-20 % slower, but for one
// component at 64^3.)
//
// Only plain upwind problems whose solids are not read (the kernels over the
// list take the others).  The arithmetic of a voxel is pore_step's
// (nmr_pores.hip), operation by operation, so the fields are the same bits.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "nmr_device.h"
#include "nmr_kernels.h"
#include "nmr_pore_device.h"

namespace nmr {

namespace {

constexpr int kThreads = kBlockThreads, kWaves = kThreads / 64;
constexpr int kExt = kBlockEdge + 2 * kBlockSteps; // edge of a box with its surroundings
// Voxels within kBlockSteps faces of a box: over its faces, edges and corners.
constexpr int ball(int r)
{
    const int e = kBlockEdge;
    return e * e * e + 6 * e * e * r + 12 * e * (r * (r - 1) / 2) + 8 * (r * (r - 1) * (r - 2) / 6);
}
constexpr int kCap = ball(kBlockSteps), kPer = (kCap + kThreads - 1) / kThreads; // slots of a block, of a thread
static_assert(kExt == 16 && kCap <= 4096, "4-bit positions, 12-bit slots");
static_assert(kBlockEdge * kBlockEdge * kBlockEdge <= kThreads, "the box's own pores are every thread's first slot");

// One slot of a block: the slot in the list, then a 16-bit word for each of
// the six sides: the neighbour's slot in the block (12 bits; the own one for a
// solid or past the grid), 3 spare bits, and in bit 15 that it counts as a
// pore.  The spare bits hold the position in the surroundings -- z in side 0's,
// x in side 2's, y in side 3's, their fourth bits in side 1's -- and in side
// 4's that the voxel is in the signal window.
__device__ __forceinline__ uint32_t side(const u32x4& r, int s) { return (s & 1) ? r[1 + s / 2] >> 16 : r[1 + s / 2] & 0xffffu; }
__device__ __forceinline__ uint32_t spare(const u32x4& r, int s) { return (side(r, s) >> 12) & 7u; }

// Faces between a voxel of the surroundings and the box.
__device__ __forceinline__ int away(int l) { return max(max(kBlockSteps - l, l - (kBlockSteps + kBlockEdge - 1)), 0); }

struct Box {
    int x0, y0, z0; // first voxel of the surroundings
    __device__ __forceinline__ Box(int b, int nbx, int nby)
    {
        x0 = b % nbx * kBlockEdge - kBlockSteps;
        y0 = b / nbx % nby * kBlockEdge - kBlockSteps;
        z0 = b / (nbx * nby) * kBlockEdge - kBlockSteps;
    }
    // Voxel c of the surroundings: whether it is a pore, and where.
    __device__ __forceinline__ bool voxel(const PoreBuild& b, int c, int& x, int& y, int& z, size_t& o) const
    {
        x = x0 + (c & 15);
        y = y0 + ((c >> 4) & 15);
        z = z0 + (c >> 8);
        if (x < 0 || y < 0 || z < 0 || x >= b.nx || y >= b.ny || z >= b.nz) return false;
        o = ((size_t)z * b.ny + y) * b.pitch + x;
        return b.mask[o] != 0;
    }
};

// Pores by distance, and a place for them.
__global__ void __launch_bounds__(kThreads) block_count_kernel(PoreBuild b)
{
    __shared__ uint32_t n[kBlockSteps + 1];
    const Box box(blockIdx.x, b.nbx, b.nby);
    if (threadIdx.x <= kBlockSteps) n[threadIdx.x] = 0;
    __syncthreads();
    for (int c = threadIdx.x; c < kExt * kExt * kExt; c += kThreads) {
        int x, y, z;
        size_t o;
        const int d = away(c & 15) + away((c >> 4) & 15) + away(c >> 8);
        if (d <= kBlockSteps && box.voxel(b, c, x, y, z, o)) atomicAdd(&n[d], 1u);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t* out = b.bcount + (size_t)blockIdx.x * 8;
        uint32_t sum = 0;
        for (int d = 0; d <= kBlockSteps; d++) out[d] = sum += n[d];
        out[kBlockSteps + 1] = (uint32_t)atomicAdd(&b.found[2], (int)sum);
    }
}

// The slots of a block, by distance and then by position.  Built with every
// mask upload, so its barriers count: one pass over the surroundings finds the
// pores of all distances (64^3: 14 us; a pass a distance, with two barriers for
// every 256 voxels: 52).
__global__ void __launch_bounds__(kThreads) block_build_kernel(PoreBuild b)
{
    constexpr int kVox = kExt * kExt * kExt, kRuns = kVox / 64; // runs of 64 voxels: a wavefront's
    constexpr uint16_t kNone = 0xffffu;
    __shared__ uint16_t at[kVox];                    // slot in the block of a voxel
    __shared__ uint32_t runs[(kBlockSteps + 1) * kRuns]; // pores of a run at a distance, then the slots before them
    static_assert(kVox % kThreads == 0 && kRuns == 64 && kThreads >= 64 * (kBlockSteps + 1));
    constexpr int kEach = kVox / kThreads;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const Box box(blockIdx.x, b.nbx, b.nby);
    const uint32_t* cnt = b.bcount + (size_t)blockIdx.x * 8;
    u32x4* out = b.blocks + cnt[kBlockSteps + 1];
    if (t < 8) b.bcount_to[(size_t)blockIdx.x * 8 + t] = cnt[t];
    int dist[kEach];
    uint32_t lower[kEach]; // pores of its distance before a voxel in its run
#pragma unroll
    for (int k = 0; k < kEach; k++) {
        const int c = t + k * kThreads;
        int x, y, z;
        size_t o;
        const int d = away(c & 15) + away((c >> 4) & 15) + away(c >> 8);
        dist[k] = d <= kBlockSteps && box.voxel(b, c, x, y, z, o) ? d : -1;
        lower[k] = 0;
        for (int q = 0; q <= kBlockSteps; q++) {
            const uint64_t m = __ballot(dist[k] == q);
            if (dist[k] == q) lower[k] = (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
            if (lane == 0) runs[q * kRuns + k * kWaves + wave] = (uint32_t)__popcll(m);
        }
    }
    __syncthreads();
    if (wave <= kBlockSteps) { // a wavefront takes the runs of a distance
        const uint32_t own = runs[t];
        uint32_t sum = own;
        for (int h = 1; h < 64; h <<= 1) {
            const uint32_t u = (uint32_t)__shfl_up((int)sum, h, 64);
            if (lane >= h) sum += u;
        }
        runs[t] = sum - own + (wave > 0 ? cnt[wave - 1] : 0u);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kEach; k++)
        at[t + k * kThreads] =
            dist[k] < 0 ? kNone : (uint16_t)(runs[dist[k] * kRuns + k * kWaves + wave] + lower[k]);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kEach; k++) {
        const int c = t + k * kThreads, d = dist[k];
        if (d < 0) continue;
        const int lx = c & 15, ly = (c >> 4) & 15, lz = c >> 8;
        const int x = box.x0 + lx, y = box.y0 + ly, z = box.z0 + lz;
        const size_t o = ((size_t)z * b.ny + y) * b.pitch + x;
        const uint32_t own = at[c];
        const int p[3] = {x, y, z}, size[3] = {b.nx, b.ny, b.nz}, step[3] = {1, 16, 256};
        uint32_t w[6];
#pragma unroll
        for (int s = 0; s < 6; s++) {
            const int ax = s >> 1, up = s & 1;
            w[s] = own;
            if (d == kBlockSteps) continue; // never brought forward
            if (up ? p[ax] == size[ax] - 1 : p[ax] == 0) { // a zero-derivative ghost: the own value
                w[s] = own | 0x8000u;
                continue;
            }
            const uint16_t nb = at[up ? c + step[ax] : c - step[ax]]; // (at most one face further)
            if (nb != kNone) w[s] = nb | 0x8000u;
        }
        const bool win = x >= b.w[0] && x < b.w[1] && y >= b.w[2] && y < b.w[3] && z >= b.w[4] && z < b.w[5];
        w[0] |= (uint32_t)(lz & 7) << 12;
        w[1] |= (uint32_t)((lz >> 3) | (lx >> 3) << 1 | (ly >> 3) << 2) << 12;
        w[2] |= (uint32_t)(lx & 7) << 12;
        w[3] |= (uint32_t)(ly & 7) << 12;
        w[4] |= win ? 0x1000u : 0u;
        out[own] = u32x4{b.slotmap[o], w[0] | w[1] << 16, w[2] | w[3] << 16, w[4] | w[5] << 16};
    }
}

// pore_step's arithmetic for a plain upwind problem: the new value of a voxel
// from its own, its neighbours' (fn), which of them are pores (kn), its
// velocity sums and its position (voxel centres in voxels).
template <int NC, bool VEL, bool EXACT>
__device__ __forceinline__ Vec<NC> plain_update(const Coef& cf, const Vec<NC>& mc, const Vec<NC> (&fn)[6],
                                                const bool (&kn)[6], const float (&adv)[3], float xc, float yc,
                                                float zc)
{
    float w[6];
    w[0] = kn[0] ? cf.cdx : 0.f;
    w[1] = kn[1] ? cf.cdx : 0.f;
    w[2] = kn[2] ? cf.cdy : 0.f;
    w[3] = kn[3] ? cf.cdy : 0.f;
    w[4] = kn[4] ? cf.cdz : 0.f;
    w[5] = kn[5] ? cf.cdz : 0.f;
    if constexpr (VEL) {
        const float h[3] = {0.5f * cf.hx, 0.5f * cf.hy, 0.5f * cf.hz};
#pragma unroll
        for (int ax = 0; ax < 3; ax++) {
            w[2 * ax] = fmaf(h[ax], pos(adv[ax]), w[2 * ax]);
            w[2 * ax + 1] = fmaf(-h[ax], neg(adv[ax]), w[2 * ax + 1]);
        }
    }
    const float nsx = (kn[0] ? 0.f : 1.f) + (kn[1] ? 0.f : 1.f), nsy = (kn[2] ? 0.f : 1.f) + (kn[3] ? 0.f : 1.f),
                nsz = (kn[4] ? 0.f : 1.f) + (kn[5] ? 0.f : 1.f);
    const float rate2 = fmaf(cf.s2z, nsz, fmaf(cf.s2y, nsy, fmaf(cf.s2x, nsx, cf.r2)));
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
    const float thz = cf.bgz * zc;
    if constexpr (NC == 3) {
        const float thx = cf.bgx * xc, thy = cf.bgy * yc;
        const float rate1 = fmaf(cf.s1z, nsz, fmaf(cf.s1y, nsy, fmaf(cf.s1x, nsx, cf.r1)));
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
        if constexpr (NC == 2 && EXACT) {
            float sn = thz, h = 0.5f * thz;
            if (cf.bgz != 0.f) {
                sn = sinf(thz);
                h = sinf(h);
            }
            const float cm1 = -2.f * h * h;
            d[0] = fmaf(mc[1], sn, fmaf(mc[0], cm1, d[0]));
            d[1] = fmaf(-mc[0], sn, fmaf(mc[1], cm1, d[1]));
        } else if constexpr (NC == 2) {
            d[0] = fmaf(thz, mc[1], d[0]);
            d[1] = fmaf(-thz, mc[0], d[1]);
        }
    }
    Vec<NC> out;
#pragma unroll
    for (int q = 0; q < NC; q++) out[q] = mc[q] + d[q];
    return out;
}

template <int NC, bool VEL, bool EXACT>
__global__ void __launch_bounds__(kThreads) block_kernel(BlockArgs a)
{
    __shared__ float st[2][kCap * NC];
    __shared__ double red[kBlockSteps][NC][kWaves];
    const int b = xcd_tile(blockIdx.x, a.nblocks), t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    typedef const __attribute__((address_space(4))) uint32_t* CountPtr; // (uniform loads to scalar registers)
    const CountPtr cnt = (CountPtr)(uintptr_t)(a.bcount + (size_t)b * 8);
    const u32x4* mine = a.blocks + cnt[kBlockSteps + 1];
    u32x4 r[kPer];
    r[0] = mine[t]; // (past the block's last slot: not used; the array is a workgroup longer than its slots)
    static_assert(kBlockSteps == 4);
    const int n0 = (int)cnt[0], n1 = (int)cnt[1], n2 = (int)cnt[2], n3 = (int)cnt[3], n4 = (int)cnt[4];
    auto within = [&](int d) { return d == 0 ? n0 : d == 1 ? n1 : d == 2 ? n2 : d == 3 ? n3 : n4; };
    const int box = n0, all = within(a.steps), moved = within(a.steps - 1);
    if (box == 0) { // nothing to bring forward
        for (int i = t; i < a.steps * NC; i += kThreads)
            a.partials[((size_t)(i / NC) * a.nblocks + b) * NC + i % NC] = 0.0;
        return;
    }
#pragma unroll
    for (int k = 1; k < kPer; k++) r[k] = t + k * kThreads < all ? mine[t + k * kThreads] : u32x4{0u, 0u, 0u, 0u};
    Vec<NC> m[kPer];
    float adv[kPer][3];
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        m[k] = Vec<NC>{};
        const int i = t + k * kThreads;
        if (i < all) m[k] = at_byte<Vec<NC>>(a.f, r[k][0] * (uint32_t)(4 * NC));
#pragma unroll
        for (int q = 0; q < 3; q++) adv[k][q] = 0.f;
        if constexpr (VEL) {
            if (i < moved) {
                const u32x4 v = at_byte<u32x4>(a.rec, r[k][0] * 16u);
#pragma unroll
                for (int q = 0; q < 3; q++) adv[k][q] = __uint_as_float(v[1 + q]);
            }
        }
        if (i < all)
#pragma unroll
            for (int q = 0; q < NC; q++) st[0][i * NC + q] = m[k][q];
    }
    __syncthreads();
    const Box at(b, a.nbx, a.nby);
    const bool win = t < box && (spare(r[0], 4) & 1u) != 0;
    for (int s = 1; s <= a.steps; s++) {
        const Coef& cf = a.c[s - 1];
        const float* in = st[(s - 1) & 1];
        float* nx = st[s & 1];
        const int lim = within(a.steps - s);
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const int i = t + k * kThreads;
            if (i >= lim) continue;
            Vec<NC> fn[6];
            bool kn[6];
#pragma unroll
            for (int q = 0; q < 6; q++) {
                const uint32_t w = side(r[k], q);
                kn[q] = (w & 0x8000u) != 0;
#pragma unroll
                for (int c = 0; c < NC; c++) fn[q][c] = in[(w & 0xfffu) * NC + c];
            }
            const uint32_t hi = spare(r[k], 1);
            const float xc = (float)(at.x0 + (int)(spare(r[k], 2) | (hi & 2u) << 2)) + 0.5f;
            const float yc = (float)(at.y0 + (int)(spare(r[k], 3) | (hi & 4u) << 1)) + 0.5f;
            const float zc = (float)(at.z0 + (int)(spare(r[k], 0) | (hi & 1u) << 3)) + 0.5f;
            m[k] = plain_update<NC, VEL, EXACT>(cf, m[k], fn, kn, adv[k], xc, yc, zc);
            if (s < a.steps) {
#pragma unroll
                for (int c = 0; c < NC; c++) nx[i * NC + c] = m[k][c];
            } else if (i < box) {
                stm<NC>(a.out, r[k][0], m[k]);
            }
        }
        if (wave * 64 < box) { // the box's own pores are the threads' first slots
#pragma unroll
            for (int q = 0; q < NC; q++) {
                const double v = wave_sum((double)(win ? m[0][q] : 0.f));
                if (lane == 63) red[s - 1][q][wave] = v;
            }
        }
        __syncthreads();
    }
    if (t < a.steps * NC) {
        const int s = t / NC, q = t % NC;
        double v = 0.0;
        for (int w = 0; w * 64 < box; w++) v += red[s][q][w];
        a.partials[((size_t)s * a.nblocks + b) * NC + q] = v;
    }
}

} // namespace

hipError_t launch_block_count(const PoreBuild& b, hipStream_t s)
{
    hipLaunchKernelGGL(block_count_kernel, dim3((unsigned)(b.nbx * b.nby * b.nbz)), dim3(kThreads), 0, s, b);
    return hipGetLastError();
}

hipError_t launch_block_build(const PoreBuild& b, hipStream_t s)
{
    hipLaunchKernelGGL(block_build_kernel, dim3((unsigned)(b.nbx * b.nby * b.nbz)), dim3(kThreads), 0, s, b);
    return hipGetLastError();
}

hipError_t launch_blocks(int nc, bool vel, bool exact, const BlockArgs& a, hipStream_t s)
{
    if (a.steps < 1 || a.steps > kBlockSteps || a.nblocks < 1 || (exact && nc != 2)) return hipErrorInvalidValue;
    const dim3 grid((unsigned)a.nblocks), block(kThreads);
    switch (nc * 2 + (vel ? 1 : 0)) {
    case 2: hipLaunchKernelGGL((block_kernel<1, false, false>), grid, block, 0, s, a); break;
    case 3: hipLaunchKernelGGL((block_kernel<1, true, false>), grid, block, 0, s, a); break;
    case 4:
        if (exact) hipLaunchKernelGGL((block_kernel<2, false, true>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((block_kernel<2, false, false>), grid, block, 0, s, a);
        break;
    case 5:
        if (exact) hipLaunchKernelGGL((block_kernel<2, true, true>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((block_kernel<2, true, false>), grid, block, 0, s, a);
        break;
    case 6: hipLaunchKernelGGL((block_kernel<3, false, false>), grid, block, 0, s, a); break;
    case 7: hipLaunchKernelGGL((block_kernel<3, true, false>), grid, block, 0, s, a); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

} // namespace nmr
