// nmr_learn_kernels.hip -- device kernels of the learned corrector: a 3-layer
// 3-D convolution net (6 -> 16 -> 16 -> 2 channels, 3x3x3 kernels, "same"
// zero padding, ReLU between layers) with BF16 weights and activations and
// FP32 accumulation on the gfx950 matrix cores
// (v_mfma_f32_16x16x32_bf16), its backward pass (input and weight
// gradients), Adam, and the glue between the solver's FP32 fields and the
// net's tensors.
//
// Tensors live on the grid padded by one zero voxel per side, channels last:
// element (x, y, z, c) of an nx*ny*nz grid with C channels is at
// (((z+1)*(ny+2) + y+1)*(nx+2) + x+1)*C + c.  The halo stays zero, which is
// the zero padding of the convolution.
//
// Convolution as an implicit GEMM: out[v][co] = sum_{t,ci} W[co][ci][t] *
// in[v + off(t)][ci].  One wavefront computes a row of 16 x-consecutive
// voxels for all 16 output channels: the MFMA's A operand is the weight
// matrix (16 output channels x 32 reduction indices), its B operand the
// input (32 reduction indices x 16 voxels), and the reduction index k of a
// 32-chunk covers 32/CIN taps of CIN channels.  The A fragments of all
// chunks stay in registers for the whole kernel.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "nmr_device.h"
#include "nmr_kernels.h"

namespace nmr {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float fl4 __attribute__((ext_vector_type(4)));

// Round to nearest even (NaN kept quiet), and back.
__device__ __forceinline__ uint16_t f2bf(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
// The same of two values, b in the upper half (one v_cvt_pk_bf16_f32; the same
// bits as f2bf for every value).
__device__ __forceinline__ uint32_t f2bf2(float a, float b)
{
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const bf16x2 v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ bool bf_pos(uint16_t h) { return h != 0 && (h & 0x8000u) == 0; }

__device__ __forceinline__ bf16x8 as_bf8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

// A barrier that orders LDS accesses only: global loads stay in flight across it.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// tap t = kz*9 + ky*3 + kx, offsets -1..1 on each axis
__device__ __forceinline__ long tap_off(int t, long px, long plane)
{
    const int kz = t / 9, ky = (t / 3) % 3, kx = t % 3;
    return (long)(kz - 1) * plane + (long)(ky - 1) * px + (long)(kx - 1);
}

// MODE 0: + bias, ReLU, BF16 out (16 ch); 1: + bias, FP32 out (2 ch);
// 2: gated by ref > 0, BF16 out (16 ch) -- the input gradient through ReLU.
template <int CIN, int MODE>
__global__ void __launch_bounds__(256) conv_kernel(ConvArgs a)
{
    constexpr int TPC = 32 / CIN;               // taps per reduction chunk
    constexpr int NCH = (27 + TPC - 1) / TPC;   // chunks
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, n = lane & 15;
    bf16x8 A[NCH];
    const uint4* wa4 = reinterpret_cast<const uint4*>(a.wa);
#pragma unroll
    for (int c = 0; c < NCH; c++) A[c] = as_bf8(wa4[c * 64 + lane]);
    const long px = a.nx + 2, plane = px * (long)(a.ny + 2);
    const int cin0 = (8 * g) % CIN;
    const int wave = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int nwaves = gridDim.x * 4;
    for (int r = wave; r < a.nrows; r += nwaves) {
        const int row = a.rows ? a.rows[r] : r;
        const int seg = row % a.nseg, yz = row / a.nseg;
        const int y = yz % a.ny, z = yz / a.ny;
        const int x = seg * 16 + n;
        const int xv = x < a.nx ? x : a.nx - 1;
        const long base = ((long)(z + 1) * (a.ny + 2) + (y + 1)) * px + (xv + 1);
        uint4 B[NCH];
#pragma unroll
        for (int c = 0; c < NCH; c++) {
            const int t = c * TPC + (8 * g) / CIN;
            B[c] = make_uint4(0u, 0u, 0u, 0u);
            if (t < 27)
                B[c] = *reinterpret_cast<const uint4*>(a.in + (base + tap_off(t, px, plane)) * CIN + cin0);
        }
        fl4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < NCH; c++) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[c], as_bf8(B[c]), acc, 0, 0, 0);
        if (x >= a.nx) continue;
        // lane holds output channels 4g..4g+3 of voxel n
        if constexpr (MODE == 1) {
            if (g == 0) {
                a.outf[base * 2 + 0] = acc[0] + a.bias[0];
                a.outf[base * 2 + 1] = acc[1] + a.bias[1];
            }
        } else {
            uint16_t h[4];
            if constexpr (MODE == 0) {
#pragma unroll
                for (int j = 0; j < 4; j++) h[j] = f2bf(fmaxf(acc[j] + a.bias[4 * g + j], 0.f));
            } else {
                const uint2 rv = *reinterpret_cast<const uint2*>(a.ref + base * 16 + 4 * g);
                const uint16_t rr[4] = {(uint16_t)(rv.x & 0xffffu), (uint16_t)(rv.x >> 16),
                                        (uint16_t)(rv.y & 0xffffu), (uint16_t)(rv.y >> 16)};
#pragma unroll
                for (int j = 0; j < 4; j++) h[j] = bf_pos(rr[j]) ? f2bf(acc[j]) : (uint16_t)0;
            }
            *reinterpret_cast<uint2*>(a.out + base * 16 + 4 * g) =
                make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
        }
    }
}

// The same convolution over tiles of 16 x 8 x 4 output voxels: the tile's
// input region (18 x 10 x 6 voxels, all channels) is staged in LDS once and
// every B operand is read from there, instead of 27 gathers per voxel from
// L1/L2.  Each wavefront computes 8 of the tile's 32 output rows with the
// row kernel's MFMA sequence (same operands, same chunk order), so the two
// kernels produce the same bits.  Persistent: workgroup b takes tiles b,
// b + gridDim.x, ...; every row of the grid is computed (no row list).
constexpr int kTileY = 8, kTileZ = 4;
template <int CIN, int MODE>
__global__ void __launch_bounds__(256) conv_tile_kernel(ConvArgs a)
{
    constexpr int TPC = 32 / CIN;
    constexpr int NCH = (27 + TPC - 1) / TPC;
    constexpr int HX = 18, HY = kTileY + 2, HZ = kTileZ + 2;
    constexpr int NV = HX * HY * HZ;
    constexpr int V16 = CIN / 8; // 16-byte parts per voxel
    __shared__ uint4 sin[NV * V16];
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, n = lane & 15;
    const int wave = threadIdx.x >> 6;
    bf16x8 A[NCH];
    const uint4* wa4 = reinterpret_cast<const uint4*>(a.wa);
#pragma unroll
    for (int c = 0; c < NCH; c++) A[c] = as_bf8(wa4[c * 64 + lane]);
    const long px = a.nx + 2;
    const int nty = (a.ny + kTileY - 1) / kTileY, ntz = (a.nz + kTileZ - 1) / kTileZ;
    const int ntiles = a.nseg * nty * ntz;
    const int part0 = ((8 * g) % CIN) / 8;
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int seg = tile % a.nseg, r2 = tile / a.nseg;
        const int x0 = seg * 16, y0 = (r2 % nty) * kTileY, z0 = (r2 / nty) * kTileZ;
        // staged voxel (xx, yy, zz) = padded voxel (x0 + xx, y0 + yy, z0 + zz),
        // clamped to the padded grid (clamped ones feed only outputs that are
        // not stored)
        for (int i = threadIdx.x; i < NV * V16; i += 256) {
            const int v = i / V16, pt = i % V16;
            const int xx = v % HX, yy = (v / HX) % HY, zz = v / (HX * HY);
            const long gx = min(x0 + xx, a.nx + 1), gy = min(y0 + yy, a.ny + 1), gz = min(z0 + zz, a.nz + 1);
            sin[i] = *reinterpret_cast<const uint4*>(a.in + ((gz * (a.ny + 2) + gy) * px + gx) * CIN + pt * 8);
        }
        __syncthreads();
        for (int rr = wave; rr < kTileY * kTileZ; rr += 4) {
            const int ly = rr % kTileY, lz = rr / kTileY;
            fl4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < NCH; c++) {
                const int t = c * TPC + (8 * g) / CIN;
                uint4 B = make_uint4(0u, 0u, 0u, 0u);
                if (t < 27) {
                    const int kz = t / 9, ky = (t / 3) % 3, kx = t % 3;
                    B = sin[(((lz + kz) * HY + (ly + ky)) * HX + (n + kx)) * V16 + part0];
                }
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[c], as_bf8(B), acc, 0, 0, 0);
            }
            const int x = x0 + n, y = y0 + ly, z = z0 + lz;
            if (x >= a.nx || y >= a.ny || z >= a.nz) continue;
            const long base = ((long)(z + 1) * (a.ny + 2) + (y + 1)) * px + (x + 1);
            // lane holds output channels 4g..4g+3 of voxel n
            if constexpr (MODE == 1) {
                if (g == 0) {
                    a.outf[base * 2 + 0] = acc[0] + a.bias[0];
                    a.outf[base * 2 + 1] = acc[1] + a.bias[1];
                }
            } else {
                uint16_t h[4];
                if constexpr (MODE == 0) {
#pragma unroll
                    for (int j = 0; j < 4; j++) h[j] = f2bf(fmaxf(acc[j] + a.bias[4 * g + j], 0.f));
                } else {
                    const uint2 rv = *reinterpret_cast<const uint2*>(a.ref + base * 16 + 4 * g);
                    const uint16_t rr4[4] = {(uint16_t)(rv.x & 0xffffu), (uint16_t)(rv.x >> 16),
                                             (uint16_t)(rv.y & 0xffffu), (uint16_t)(rv.y >> 16)};
#pragma unroll
                    for (int j = 0; j < 4; j++) h[j] = bf_pos(rr4[j]) ? f2bf(acc[j]) : (uint16_t)0;
                }
                *reinterpret_cast<uint2*>(a.out + base * 16 + 4 * g) =
                    make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
            }
        }
        __syncthreads();
    }
}

// The same convolution marching along z through columns of 16 x 16 output
// rows: the input planes of the column (18 x 18 voxels, all channels) pass
// through a ring of three LDS slots, so that each is loaded once per column
// instead of once per 16 x 8 x 4 tile (1.27 input reads per output voxel
// instead of 2.1).  A plane is used for all three output planes that read it
// while it is there: output z takes its taps of plane z, then of z + 1, then
// of z + 2, which is the order of the reduction, so three planes of
// accumulators are open at a time and the bits equal those of conv_kernel and
// conv_tile_kernel (same operands, same chunk order).
//
// Bound by LDS reads where every chunk reads its own operand (56 of 16 bytes a
// lane for the 56 MFMAs of four rows at 16 channels: 1800 cycles a plane of
// one workgroup, against 900 of the matrix cores).  A wavefront therefore
// takes four consecutive rows, whose chunks share operands: those of one plane
// are runs of taps that recur at another row offset (kx 0,1 | kx 1,2 | kx 2 and
// the next row's 0), so 22 reads serve the 56 MFMAs (22 for 28 at 8 channels).
// The channel halves of a plane lie apart in LDS, so that 16 lanes read 256
// consecutive bytes.  Two planes of global loads are in flight behind the one
// that is computed (the barrier orders LDS only), and BF16 results are rounded
// two at a time in one instruction (a branch on NaN for each value cost 15 %).
// What is left is the chain of a plane -- reads, MFMAs, store, barrier -- with
// two workgroups a CU.  96x80x64, with one read an MFMA and columns of 16
// planes before: 34.4 -> 14.2 us at 16 -> 16, 26.7 -> 11.3 at 16 -> 2, 39.5 ->
// 14.8 the input gradient, 25.9 -> 10.1 at 8 -> 16.  128^3: 41.6 -> 33.2, 31.6 ->
// 28.5 (the MFMAs of 18 planes take 13.4 a SIMD's wavefront, two of them 27 us
// at 2.4 GHz), 45.2 the gradient, 23.2 at 8 -> 16.
//
// Persistent: workgroup b takes columns b, b + gridDim.x, ...; a column is
// a.zc output planes (the last one what is left).
constexpr int kZmY = 16;
template <int CIN, int MODE>
__global__ void __launch_bounds__(256, 2) conv_zm_kernel(ConvArgs a)
{
    constexpr int TPC = 32 / CIN;
    constexpr int NCH = (27 + TPC - 1) / TPC;
    constexpr int HX = 18, HY = kZmY + 2, HV = HX * HY;
    constexpr int V16 = CIN / 8;
    constexpr int PV = HV * V16;               // uint4 per staged plane
    constexpr int NLD = (PV + 255) / 256;
    constexpr int ROWB = HX * 16, SLOTB = PV * 16; // bytes per staged row and per slot
    __shared__ u32x4 sin[3 * PV + HX + 16];    // (the zeroed half of the last row's last chunk reads past the plane)
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, n = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    bf16x8 A[NCH];
    const uint4* wa4 = reinterpret_cast<const uint4*>(a.wa);
#pragma unroll
    for (int c = 0; c < NCH; c++) A[c] = as_bf8(wa4[c * 64 + lane]);
    // Byte offset of this lane's part of an operand within a plane: (row, x)
    // of the lane's tap from the operand's row of this wavefront.
    auto at = [&](int row, int dx) {
        return ((CIN == 16 ? (g & 1) * HV : 0) + (wave * 4 + row) * HX + n + dx) * 16;
    };
    const int tg = CIN == 16 ? g >> 1 : g; // the lane's tap in a chunk
    // operands of one plane: 16 channels: kx 0,1 | kx 1,2 | kx 2 and the next
    // row's kx 0; 8 channels: kx 0,1,2 and the next row's 0 | kx 1,2 and the
    // next row's 0,1 | kx 2 and the next row's 0,1,2
    int o0, o1, o2;
    if constexpr (CIN == 16) {
        o0 = at(0, tg);
        o1 = at(0, 1 + tg);
        o2 = tg ? at(1, 0) : at(0, 2);
    } else {
        o0 = tg < 3 ? at(0, tg) : at(1, 0);
        o1 = tg < 2 ? at(0, 1 + tg) : at(1, tg - 2);
        o2 = tg ? at(1, tg - 1) : at(0, 2);
    }
    // operands that span two planes: ky 2, kx 2 (8 channels: or kx 1,2) of the
    // plane before and the first taps of this one; by slot of this plane
    int m0[3], m1[3];
#pragma unroll
    for (int s = 0; s < 3; s++) {
        const int before = (s + 2) % 3 * SLOTB, here = s * SLOTB;
        m0[s] = tg == 0 ? before + at(2, 2) : here + at(0, tg - 1);
        m1[s] = tg < 2 ? before + at(2, 1 + tg) : here + at(0, tg - 2);
    }
    const bool last = (NCH - 1) * TPC + tg < 27; // the lane's tap of the last chunk exists
    float bias[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (MODE == 0) {
#pragma unroll
        for (int j = 0; j < 4; j++) bias[j] = a.bias[4 * g + j];
    } else if constexpr (MODE == 1) {
        bias[0] = a.bias[0];
        bias[1] = a.bias[1];
    }
    const int px = a.nx + 2, plane = (a.ny + 2) * px; // (the padded grid has fewer than 2^31 voxels)
    const int zc = a.zc;
    const int nyb = (a.ny + kZmY - 1) / kZmY, nzb = (a.nz + zc - 1) / zc;
    const int ncol = a.nseg * nyb * nzb;
    char* lds = reinterpret_cast<char*>(sin);
    auto read = [&](int o) { return *reinterpret_cast<const u32x4*>(lds + o); };
    auto mfma = [&](int c, const u32x4& b, fl4& d) {
        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[c], __builtin_bit_cast(bf16x8, b), d, 0, 0, 0);
    };
    for (int col = xcd_tile(blockIdx.x, (int)gridDim.x); col < ncol; col += gridDim.x) {
        const int seg = col % a.nseg, r2 = col / a.nseg;
        const int x0 = seg * 16, y0 = (r2 % nyb) * kZmY, zs = (r2 / nyb) * zc;
        const int ze = min(zs + zc, a.nz);
        // staged element i = threadIdx.x + 256 j of a plane: voxel (xx, yy) =
        // padded (x0 + xx, y0 + yy), clamped to the padded grid (clamped ones
        // feed only outputs that are not stored); a thread's element past the
        // plane loads element 0 again and is not stored
        uint32_t goff[NLD]; // bytes in a plane (below 4 GiB)
#pragma unroll
        for (int j = 0; j < NLD; j++) {
            const int i = threadIdx.x + 256 * j < PV ? threadIdx.x + 256 * j : 0;
            const int v = i / V16;
            const int gx = min(x0 + v % HX, a.nx + 1), gy = min(y0 + v / HX, a.ny + 1);
            goff[j] = (uint32_t)(gy * px + gx) * (uint32_t)(2 * CIN) + (uint32_t)(i % V16) * 16u;
        }
        auto load = [&](int pz, u32x4 (&r)[NLD]) {
            const char* in = reinterpret_cast<const char*>(a.in + (size_t)pz * plane * CIN);
#pragma unroll
            for (int j = 0; j < NLD; j++) r[j] = *reinterpret_cast<const u32x4*>(in + goff[j]);
        };
        auto stash = [&](int slot, const u32x4 (&r)[NLD]) {
#pragma unroll
            for (int j = 0; j < NLD; j++) {
                const int i = threadIdx.x + 256 * j;
                if (i < PV) sin[slot * PV + (i % V16) * HV + i / V16] = r[j];
            }
        };
        const int x = x0 + n, yw = y0 + wave * 4;
        const bool live = yw < a.ny; // this wavefront has rows
        // this lane's first output in its plane, in bytes
        const uint32_t oo = (uint32_t)((yw + 1) * px + x + 1) * (MODE == 1 ? 8u : 32u) + (MODE == 1 ? 0u : 8u * g);
        u32x4 l0[NLD], l1[NLD], l2[NLD];
        // Plane p in slot s (p - zs modulo 3): opens output plane p in `first`,
        // goes on with p - 1 in `mid` and completes p - 2 in `fin`; plane p + 1 is
        // on its way in `next`, and p + 2 sets out into `ahead`.
        auto step = [&](const int p, auto S, const u32x4 (&next)[NLD], u32x4 (&ahead)[NLD], fl4 (&first)[4], fl4 (&mid)[4],
                        fl4 (&fin)[4]) {
            constexpr int s = decltype(S)::value;
            constexpr int sb = s * SLOTB;
            const int z = p - 2;
            const bool out = z >= zs;
            load(min(p + 2, ze + 1), ahead); // (without a branch, whose join would wait for the loads)
            const size_t zb = (size_t)(z + 1) * plane; // (z + 1 = p - 1 < 0 only where nothing is stored)
            uint2 gate[4];
            if (live) {
                u32x4 P[6], Q[6], X[6];
#pragma unroll
                for (int r = 0; r < 6; r++) {
                    P[r] = read(o0 + sb + r * ROWB);
                    if (CIN == 16 || (r >= 1 && r < 5)) Q[r] = read(o1 + sb + r * ROWB);
                    if (CIN == 16 || r < 4) X[r] = read(o2 + sb + r * ROWB);
                }
                if (p < ze) {
#pragma unroll
                    for (int i = 0; i < 4; i++) first[i] = fl4{0.f, 0.f, 0.f, 0.f};
                    if constexpr (CIN == 16) {
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(0, P[i], first[i]);
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(1, X[i], first[i]);
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(2, Q[i + 1], first[i]);
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(3, P[i + 2], first[i]);
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(0, P[i], first[i]);
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(1, Q[i + 1], first[i]);
                    }
                }
                if (p - 1 >= zs && p - 1 < ze) {
                    u32x4 M[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) M[i] = read(m0[s] + i * ROWB);
                    if constexpr (CIN == 16) {
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(4, M[i], mid[i]);
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(5, Q[i], mid[i]);
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(6, P[i + 1], mid[i]);
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(7, X[i + 1], mid[i]);
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(8, Q[i + 2], mid[i]);
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(2, M[i], mid[i]);
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(3, P[i + 1], mid[i]);
                    }
                }
                if (out) {
                    const u32x4 none = {0u, 0u, 0u, 0u};
                    if constexpr (MODE == 2) {
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            gate[i] = make_uint2(0u, 0u);
                            if (x < a.nx && yw + i < a.ny)
                                gate[i] = *reinterpret_cast<const uint2*>(
                                    reinterpret_cast<const char*>(a.ref + (zb + (size_t)i * px) * 16) + oo);
                        }
                    }
                    if constexpr (CIN == 16) {
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(9, P[i], fin[i]);
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(10, X[i], fin[i]);
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(11, Q[i + 1], fin[i]);
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(12, P[i + 2], fin[i]);
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(13, last ? X[i + 2] : none, fin[i]);
                    } else {
                        u32x4 M[4];
#pragma unroll
                        for (int i = 0; i < 4; i++) M[i] = read(m1[s] + i * ROWB);
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(4, M[i], fin[i]);
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(5, X[i], fin[i]);
#pragma unroll
                        for (int i = 0; i < 4; i++) mfma(6, last ? P[i + 2] : none, fin[i]);
                    }
                }
            }
            // the next plane goes into the slot of plane p - 2, last read in the step before
            stash((s + 1) % 3, next);
            if (live && out) {
                // lane holds output channels 4g..4g+3 of voxel n
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (x >= a.nx || yw + i >= a.ny) continue;
                    if constexpr (MODE == 1) {
                        if (g == 0)
                            *reinterpret_cast<float2*>(reinterpret_cast<char*>(a.outf + (zb + (size_t)i * px) * 2) + oo) =
                                make_float2(fin[i][0] + bias[0], fin[i][1] + bias[1]);
                    } else {
                        uint32_t h[2];
                        if constexpr (MODE == 0) {
                            float v[4];
#pragma unroll
                            for (int j = 0; j < 4; j++) v[j] = fmaxf(fin[i][j] + bias[j], 0.f);
                            h[0] = f2bf2(v[0], v[1]);
                            h[1] = f2bf2(v[2], v[3]);
                        } else {
                            const uint32_t gt[2] = {gate[i].x, gate[i].y};
#pragma unroll
                            for (int j = 0; j < 2; j++) {
                                const uint32_t lo = bf_pos((uint16_t)(gt[j] & 0xffffu)) ? 0xffffu : 0u;
                                const uint32_t hi = bf_pos((uint16_t)(gt[j] >> 16)) ? 0xffff0000u : 0u;
                                h[j] = f2bf2(fin[i][2 * j], fin[i][2 * j + 1]) & (lo | hi);
                            }
                        }
                        *reinterpret_cast<uint2*>(reinterpret_cast<char*>(a.out + (zb + (size_t)i * px) * 16) + oo) =
                            make_uint2(h[0], h[1]);
                    }
                }
            }
            lds_barrier();
        };
        load(zs, l0);
        load(zs + 1, l1);
        stash(0, l0);
        lds_barrier();
        fl4 acc[3][4];
#pragma unroll
        for (int k = 0; k < 3; k++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[k][i] = fl4{0.f, 0.f, 0.f, 0.f};
        for (int p = zs; p <= ze + 1; p += 3) {
            step(p, std::integral_constant<int, 0>{}, l1, l2, acc[0], acc[2], acc[1]);
            if (p + 1 > ze + 1) break;
            step(p + 1, std::integral_constant<int, 1>{}, l2, l0, acc[1], acc[0], acc[2]);
            if (p + 2 > ze + 1) break;
            step(p + 2, std::integral_constant<int, 2>{}, l0, l1, acc[2], acc[1], acc[0]);
        }
    }
}

// Weight gradient dW[t][ci][co] = sum_v in[v + off(t)][ci] * gout[v][co] and
// bias gradient sum_v gout[v][co], as partials over 32-voxel x segments:
// partial w takes segments w, w + npart, ..., into part[w][27*256 + 16].
// MFMA: A = input (16 ci x 32 voxels), B = output gradient (32 voxels x 16
// co): eight voxels of one channel a lane, from channels-last tensors.
//
// A workgroup takes a partial, its nine wavefronts the nine (dz, dy) of the
// taps.  The segment's nine input rows and its gradient are loaded 16 bytes a
// thread in the tensors' order and turned into channel-major rows in LDS,
// where a lane's eight voxels are 16 bytes and the taps of kx 0 and 2 the same
// shifted by half a word; two segments are on their way meanwhile.  Rows of 56
// halfwords (28 words): 16 lanes' 16-byte reads and a wavefront's writes cover
// all banks.  What bounds it is the instructions around three MFMAs: gathering
// the operands from the tensors takes 18 two-byte loads for them (31.9 us at
// 96x80x64 and 16 channels, 38.1 at 8; this: 27.1 and 22.5; 32^3 to 96^3 in turns,
// where the gathers miss the caches, 47.5 -> 27.3 and 71.0 -> 21.6).  Tried: two
// voxels' pieces a thread in voxel order (each 16 bytes from a line of its own):
// 38; partials of neighbouring segments on one L2: no different; four segments
// on their way: 68 (their registers leave one workgroup a CU).
// Each tap's sum runs over the same voxels in the same order as a gather's, so
// the gradients keep their bits.
constexpr int kWgradThreads = 9 * 64, kWgradPitch = 56;
template <int CIN>
__global__ void __launch_bounds__(kWgradThreads) wgrad_kernel(WgradArgs a, int npart)
{
    // pieces of a segment: eight channels of a voxel, loaded in the tensors'
    // order; of two voxels that share a word in LDS each thread writes four channels
    constexpr int V16 = CIN / 8, NIN = 9 * V16 * 36, NP = NIN + 64;
    constexpr int NLD = (NP + kWgradThreads - 1) / kWgradThreads;
    constexpr int kSwap = V16 == 2 ? 0x4e : 0xb1; // quad_perm to the other voxel's thread
    constexpr int ROWS = 9 * CIN + 16;
    __shared__ __align__(16) uint16_t sh[2][(ROWS + 1) * kWgradPitch]; // the last row: zeros, for lanes past 8 channels
    const int t = threadIdx.x, lane = t & 63;
    const int g = lane >> 4, n = lane & 15;
    const int d = __builtin_amdgcn_readfirstlane(t >> 6); // (dz, dy) = (d / 3 - 1, d % 3 - 1)
    const int px = a.nx + 2, plane = px * (a.ny + 2); // (the padded grid has fewer than 2^31 voxels)
    const int w = blockIdx.x;
    const int nseg32 = (a.nx + 31) / 32;
    const int nrows = nseg32 * a.ny * a.nz;
    const uint32_t second = (t & V16) != 0 ? 0xffffffffu : 0u; // of its two voxels
    // this thread's pieces: voxel xv of input row (dz, dy), counted from the
    // segment's first (two that only fill their words repeat -1 and 32), or of
    // the gradient
    const char* from[NLD]; // of the segment of the grid's first padded voxel
    int xv[NLD], dst[NLD];
    bool grad[NLD];
#pragma unroll
    for (int k = 0; k < NLD; k++) {
        const int p = min(t + k * kWgradThreads, NP - 1); // (threads past the last piece load it too: no branch, whose
                                                          // join would wait for every load on its way)
        grad[k] = p >= NIN;
        if (!grad[k]) {
            const int row = p / (36 * V16), part = p % V16;
            xv[k] = min(max(p / V16 % 36 - 2, -1), 32);
            from[k] = reinterpret_cast<const char*>(a.in) +
                      ((long)((row / 3 - 1) * plane + (row % 3 - 1) * px + xv[k]) * V16 + part) * 16;
            dst[k] = (row * CIN + part * 8) * kWgradPitch + p / V16 % 36 + 6;
        } else {
            const int q = p - NIN, part = V16 == 2 ? q % 2 : q / 32;
            xv[k] = V16 == 2 ? q / 2 : q % 32;
            from[k] = reinterpret_cast<const char*>(a.gout) + (xv[k] * 2 + part) * 16;
            dst[k] = (9 * CIN + part * 8) * kWgradPitch + xv[k] + 8;
        }
        if (second) dst[k] += 4 * kWgradPitch - 1;
    }
    // Position of the segment to load next, and how far npart segments on is.
    int ls = w % nseg32, ly = w / nseg32 % a.ny, lz = w / nseg32 / a.ny;
    const int ds = npart % nseg32, dy = npart / nseg32 % a.ny, dz = npart / nseg32 / a.ny;
    auto load = [&](u32x4 (&v)[NLD]) { // (past the last segment: some voxel of the last plane)
        const int x0 = ls * 32;
        const int vox = (min(lz, a.nz - 1) + 1) * plane + (ly + 1) * px + x0 + 1;
#pragma unroll
        for (int k = 0; k < NLD; k++) { // (past the padded row's end: its last voxel)
            const int bytes = V16 == 2 || grad[k] ? 32 : 16;
            const int at = vox - max(x0 + xv[k] - a.nx, 0); // (below 0 on the smallest grids; from[k] adds xv back)
            v[k] = *reinterpret_cast<const u32x4*>(from[k] + (long)at * bytes);
        }
        const int was = x0;
        ls += ds;
        ly += dy;
        lz += dz;
        if (ls >= nseg32) {
            ls -= nseg32;
            ly++;
        }
        if (ly >= a.ny) {
            ly -= a.ny;
            lz++;
        }
        return was;
    };
    auto stash = [&](uint16_t* to, u32x4 (&v)[NLD], int x0) {
        if (x0 + 32 > a.nx) // past the row's end: no gradient
#pragma unroll
            for (int k = 0; k < NLD; k++)
                if (grad[k] && x0 + xv[k] >= a.nx) v[k] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
        for (int k = 0; k < NLD; k++) {
            if (t + k * kWgradThreads >= NP) continue;
            uint32_t own[2], other[2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                // (masks: a select of two elements becomes an indexed one)
                own[h] = (second & v[k][2 + h]) | (~second & v[k][h]);
                const uint32_t give = (second & v[k][h]) | (~second & v[k][2 + h]);
                other[h] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)give, kSwap, 0xf, 0xf, false);
                const uint32_t lo = (second & other[h]) | (~second & own[h]), hi = (second & own[h]) | (~second & other[h]);
                uint32_t* w = reinterpret_cast<uint32_t*>(to + dst[k] + 2 * h * kWgradPitch);
                w[0] = (lo & 0xffffu) | (hi << 16);
                w[kWgradPitch / 2] = (lo >> 16) | (hi & 0xffff0000u);
            }
        }
    };
    fl4 acc[3];
#pragma unroll
    for (int k = 0; k < 3; k++) acc[k] = fl4{0.f, 0.f, 0.f, 0.f};
    float bsum = 0.f;
    const bool chan = n < CIN;
    auto segment = [&](const int b) {
        const uint16_t* in = sh[b] + (chan ? d * CIN + n : ROWS) * kWgradPitch + 8 + 8 * g;
        const u32x4 B = *reinterpret_cast<const u32x4*>(sh[b] + (9 * CIN + n) * kWgradPitch + 8 + 8 * g);
        const u32x4 c = *reinterpret_cast<const u32x4*>(in);
        const uint32_t before = *reinterpret_cast<const uint32_t*>(in - 2), after = *reinterpret_cast<const uint32_t*>(in + 8);
        if (d == 0) {
#pragma unroll
            for (int j = 0; j < 8; j++) bsum += bf2f((uint16_t)(B[j / 2] >> (16 * (j & 1))));
        }
        uint32_t m[5]; // voxels -1 0, 1 2, 3 4, 5 6, 7 8 of the lane's eight
        m[0] = __builtin_amdgcn_alignbit(c[0], before, 16);
        m[1] = __builtin_amdgcn_alignbit(c[1], c[0], 16);
        m[2] = __builtin_amdgcn_alignbit(c[2], c[1], 16);
        m[3] = __builtin_amdgcn_alignbit(c[3], c[2], 16);
        m[4] = __builtin_amdgcn_alignbit(after, c[3], 16);
        const u32x4 av[3] = {u32x4{m[0], m[1], m[2], m[3]}, c, u32x4{m[1], m[2], m[3], m[4]}};
#pragma unroll
        for (int k = 0; k < 3; k++)
            acc[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av[k]),
                                                             __builtin_bit_cast(bf16x8, B), acc[k], 0, 0, 0);
    };
    // two segments on their way
    if (t < kWgradPitch) sh[0][ROWS * kWgradPitch + t] = sh[1][ROWS * kWgradPitch + t] = 0;
    u32x4 n0[NLD], n1[NLD];
    int x0 = 0, x1 = 0;
    if (w < nrows) {
        x0 = load(n0);
        x1 = load(n1);
    }
    for (int r = w; r < nrows; r += 2 * npart) {
        stash(sh[0], n0, x0); // (read two segments ago)
        x0 = load(n0);
        lds_barrier();
        segment(0);
        if (r + npart >= nrows) break;
        stash(sh[1], n1, x1);
        x1 = load(n1);
        lds_barrier();
        segment(1);
    }
    float* to = a.part + (size_t)w * kWgradPart;
    // D[i = ci = 4g + j][col = co = n]
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
        for (int j = 0; j < 4; j++) to[(3 * d + k) * 256 + (4 * g + j) * 16 + n] = acc[k][j];
    // bias: lanes n, n+16, n+32, n+48 hold the same co
    bsum += __shfl_xor(bsum, 16);
    bsum += __shfl_xor(bsum, 32);
    if (d == 0 && g == 0) to[27 * 256 + n] = bsum;
}

// Sums of the partials (FP64), scattered to the canonical gradient layout
// W[co][ci][t] (cout_real x cin_real x 27) followed by the bias; blockIdx.y is
// the layer.  A workgroup takes 16 elements, 16 threads each: a thread adds
// every sixteenth partial, so that its loads are all on their way at once and
// the chain of additions is 32 long instead of 512: 13.4 us for the three
// layers in one launch, 10.7 a layer with one thread an element.
constexpr int kRedEl = 16, kRedSlices = 16;
__global__ void __launch_bounds__(256) wreduce_kernel(WreduceArgs a)
{
    __shared__ double sh[kRedSlices][kRedEl];
    const int l = blockIdx.y, col = threadIdx.x % kRedEl, slice = threadIdx.x / kRedEl;
    const int e = blockIdx.x * kRedEl + col;
    const float* part = a.part[l];
    double s = 0.0;
    if (e < kWgradPart) {
#pragma unroll 8
        for (int w = slice; w < a.npart; w += kRedSlices) s += (double)part[(size_t)w * kWgradPart + e];
    }
    sh[slice][col] = s;
    __syncthreads();
    if (slice != 0 || e >= kWgradPart) return;
    for (int k = 1; k < kRedSlices; k++) s += sh[k][col];
    float* grad = a.grad[l];
    const int cin = a.cin[l], cout = a.cout[l];
    if (e < 27 * 256) {
        const int t = e / 256, ci = (e / 16) % 16, co = e % 16;
        if (ci < cin && co < cout) grad[((size_t)co * cin + ci) * 27 + t] = (float)s;
    } else {
        const int co = e - 27 * 256;
        if (co < cout) grad[(size_t)cout * cin * 27 + co] = (float)s;
    }
}

// Zeroes the halo of a grid's tensors (x of 8 channels, the others of 16 or
// null): what another grid left there.
__global__ void __launch_bounds__(256) halo_kernel(HaloArgs a)
{
    const int px = a.nx + 2, py = a.ny + 2, plane = px * py;
    const uint32_t v = blockIdx.x * 256u + threadIdx.x;
    if (v >= (uint32_t)plane * (uint32_t)(a.nz + 2)) return;
    const int x = (int)(v % (uint32_t)px), y = (int)(v / (uint32_t)px % (uint32_t)py), z = (int)(v / (uint32_t)plane);
    if (x >= 1 && x <= a.nx && y >= 1 && y <= a.ny && z >= 1 && z <= a.nz) return;
    const uint4 none = make_uint4(0u, 0u, 0u, 0u);
    reinterpret_cast<uint4*>(a.x)[v] = none;
#pragma unroll
    for (int k = 0; k < 5; k++)
        if (a.t[k]) {
            uint4* p = reinterpret_cast<uint4*>(a.t[k]) + (size_t)v * 2;
            p[0] = none;
            p[1] = none;
        }
}

// Packs the canonical FP32 weights of one layer, W[co][ci][t], into the A
// fragments of conv_kernel: forward (rows = output channels co, reduction
// (t, ci) with cin_store channels per tap) or input gradient (rows = ci,
// reduction (t', co) over 16 stored channels, W'[t'][co][ci] = W[26-t'][ci][co]).
// blockIdx.y is the set of fragments.
__global__ void __launch_bounds__(256) pack_kernel(PackArgs a)
{
    const PackJob& p = a.job[blockIdx.y];
    const int cin = p.backward ? 16 : p.cin_store;
    const int tpc = 32 / cin, nch = (27 + tpc - 1) / tpc;
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nch * 64 * 8) return;
    const int c = e / 512, lane = (e / 8) % 64, j = e % 8;
    const int g = lane / 16, row = lane % 16;
    const int k = 8 * g + j;
    const int t = c * tpc + k / cin, ch = k % cin;
    float v = 0.f;
    if (t < 27) {
        if (!p.backward) {
            if (ch < p.cin_real && row < p.cout_real) v = p.w[((size_t)row * p.cin_real + ch) * 27 + t];
        } else {
            if (ch < p.cout_real && row < p.cin_real) v = p.w[((size_t)ch * p.cin_real + row) * 27 + (26 - t)];
        }
    }
    p.frag[e] = f2bf(v);
}

// Input tensor of the net: (Mx, My) * pore, pore, cell-centred velocity /
// vscale, two zero channels, BF16, 8 channels per voxel.
__global__ void __launch_bounds__(256) feature_kernel(FeatureArgs a)
{
    const long n = (long)a.nx * a.ny * a.nz;
    const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n) return;
    const int x = (int)(v % a.nx), y = (int)((v / a.nx) % a.ny), z = (int)(v / ((long)a.nx * a.ny));
    const size_t c = ((size_t)z * a.ny + y) * a.pitch + x;
    const float pore = a.mask[c] ? 1.f : 0.f;
    float f[8] = {a.mx[c] * pore, a.my ? a.my[c] * pore : 0.f, pore, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (a.vx) {
        const size_t cx = ((size_t)z * a.ny + y) * a.pitch1 + x;
        const size_t cy = ((size_t)z * (a.ny + 1) + y) * a.pitch + x;
        const size_t plane = (size_t)a.ny * a.pitch;
        f[3] = 0.5f * (a.vx[cx] + a.vx[cx + 1]) * a.vinv;
        f[4] = 0.5f * (a.vy[cy] + a.vy[cy + a.pitch]) * a.vinv;
        f[5] = 0.5f * (a.vz[c] + a.vz[c + plane]) * a.vinv;
    }
    const long pv = ((long)(z + 1) * (a.ny + 2) + (y + 1)) * (a.nx + 2) + (x + 1);
    uint32_t w[4];
#pragma unroll
    for (int q = 0; q < 4; q++) w[q] = (uint32_t)f2bf(f[2 * q]) | ((uint32_t)f2bf(f[2 * q + 1]) << 16);
    *reinterpret_cast<uint4*>(a.out + pv * 8) = make_uint4(w[0], w[1], w[2], w[3]);
}

// Same tensor from host-given FP32 features [nz][ny][nx][6] (test entry).
__global__ void __launch_bounds__(256) feature_copy_kernel(const float* __restrict__ f6, int nx, int ny, int nz,
                                                           uint16_t* __restrict__ out)
{
    const long n = (long)nx * ny * nz;
    const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n) return;
    const int x = (int)(v % nx), y = (int)((v / nx) % ny), z = (int)(v / ((long)nx * ny));
    const long pv = ((long)(z + 1) * (ny + 2) + (y + 1)) * (nx + 2) + (x + 1);
    uint32_t w[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const float lo = 2 * q < 6 ? f6[v * 6 + 2 * q] : 0.f, hi = 2 * q + 1 < 6 ? f6[v * 6 + 2 * q + 1] : 0.f;
        w[q] = (uint32_t)f2bf(lo) | ((uint32_t)f2bf(hi) << 16);
    }
    *reinterpret_cast<uint4*>(out + pv * 8) = make_uint4(w[0], w[1], w[2], w[3]);
}

// Output gradient of the last layer as a BF16 16-channel tensor from
// host-given FP32 values [nz][ny][nx][2] (test entry).
__global__ void __launch_bounds__(256) gout_copy_kernel(const float* __restrict__ g2, int nx, int ny, int nz,
                                                        uint16_t* __restrict__ out)
{
    const long n = (long)nx * ny * nz;
    const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n) return;
    const int x = (int)(v % nx), y = (int)((v / nx) % ny), z = (int)(v / ((long)nx * ny));
    const long pv = ((long)(z + 1) * (ny + 2) + (y + 1)) * (nx + 2) + (x + 1);
    uint4* o = reinterpret_cast<uint4*>(out + pv * 16);
    o[0] = make_uint4((uint32_t)f2bf(g2[v * 2]) | ((uint32_t)f2bf(g2[v * 2 + 1]) << 16), 0u, 0u, 0u);
    o[1] = make_uint4(0u, 0u, 0u, 0u);
}

// Squared-error loss over pores of (pred - target/scale), the target being the
// plain steps' result less the coarse step's, and its gradient
// 2 (pred - t) / npore as the BF16 16-channel output gradient; per-block
// partial loss sums.
__global__ void __launch_bounds__(256) loss_kernel(LossArgs a)
{
    __shared__ double sh[256];
    const long n = (long)a.nx * a.ny * a.nz;
    const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    double l = 0.0;
    if (v < n) {
        const int x = (int)(v % a.nx), y = (int)((v / a.nx) % a.ny), z = (int)(v / ((long)a.nx * a.ny));
        const size_t c = ((size_t)z * a.ny + y) * a.pitch + x;
        const long pv = ((long)(z + 1) * (a.ny + 2) + (y + 1)) * (a.nx + 2) + (x + 1);
        float g0 = 0.f, g1 = 0.f;
        if (a.mask[c]) {
            const float d0 = a.pred[pv * 2] - (a.ax[c] - a.bx[c]) * a.tinv;
            const float d1 = a.pred[pv * 2 + 1] - (a.ay[c] - a.by[c]) * a.tinv;
            l = (double)d0 * d0 + (double)d1 * d1;
            g0 = 2.f * d0 * a.winv;
            g1 = 2.f * d1 * a.winv;
        }
        uint4* o = reinterpret_cast<uint4*>(a.gout + pv * 16);
        o[0] = make_uint4((uint32_t)f2bf(g0) | ((uint32_t)f2bf(g1) << 16), 0u, 0u, 0u);
        o[1] = make_uint4(0u, 0u, 0u, 0u);
    }
    sh[threadIdx.x] = l;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) sh[threadIdx.x] += sh[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) a.lpart[blockIdx.x] = sh[0];
}

// Adam on the FP32 master parameters (bias-corrected moments).
__global__ void __launch_bounds__(256) adam_kernel(float* __restrict__ p, float* __restrict__ m, float* __restrict__ v,
                                                   const float* __restrict__ g, int n, float lr, float b1, float b2,
                                                   float eps, float c1, float c2)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// Adds scale * pred to the pores of the state, brings the result into the
// net's input (channels 0 and 1, what feature_kernel writes there: the other
// channels do not change during a run, and solids hold 0), and reduces, per
// block, the state's pore energy sum(Mx^2 + My^2), the largest |correction|,
// the largest |M| of the state before the correction, a non-finite count, and
// the signal sums over the trim window: part[block][6].  LIST: the state is
// in the list of the pores.  128^3, porosity 0.2: 9.8 us on the list, 16.2 over
// the rows (every voxel's mask, 64-bit indices).
constexpr int kApplyBlocks = 1024; // workgroups (= partials) of the apply pass
template <bool LIST>
__global__ void __launch_bounds__(256) apply_kernel(ApplyArgs a)
{
    __shared__ double sh[4][6];
    // (the padded grid has fewer than 2^31 voxels)
    const uint32_t n = LIST ? a.s1 - a.s0 : (uint32_t)a.nx * (uint32_t)a.ny * (uint32_t)a.nz;
    double st[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0}; // energy, max |d|, max |M|, non-finite, sum Mx, sum My
    for (uint32_t v = blockIdx.x * 256u + threadIdx.x; v < n; v += gridDim.x * 256u) {
        const uint32_t row = LIST ? (uint32_t)a.pitch : (uint32_t)a.nx, plane = (uint32_t)a.ny * row;
        const uint32_t o = LIST ? a.vox[a.s0 + v] : v;
        if (LIST && o == 0xffffffffu) continue;
        const int x = (int)(o % plane % row), y = (int)(o % plane / row), z = (int)(o / plane);
        const size_t c = ((size_t)z * a.ny + y) * a.pitch + x;
        if (!a.mask[c]) continue;
        const size_t pv = ((size_t)(z + 1) * (a.ny + 2) + (y + 1)) * (a.nx + 2) + (x + 1);
        float mx, my;
        if constexpr (LIST) {
            const float2 m = *reinterpret_cast<const float2*>(a.slots + 2 * (size_t)(a.s0 + v));
            mx = m.x;
            my = m.y;
        } else {
            mx = a.mx[c];
            my = a.my[c];
        }
        st[2] = fmax(st[2], (double)fmaxf(fabsf(mx), fabsf(my)));
        if (a.pred) {
            const float2 p = *reinterpret_cast<const float2*>(a.pred + pv * 2);
            const float d0 = a.scale * p.x, d1 = a.scale * p.y;
            mx += d0;
            my += d1;
            if constexpr (LIST) {
                *reinterpret_cast<float2*>(a.slots + 2 * (size_t)(a.s0 + v)) = make_float2(mx, my);
            } else {
                a.mx[c] = mx;
                a.my[c] = my;
            }
            st[1] = fmax(st[1], (double)fmaxf(fabsf(d0), fabsf(d1)));
            if (!(fabsf(d0) <= 3.0e38f) || !(fabsf(d1) <= 3.0e38f)) st[3] += 1.0;
        }
        *reinterpret_cast<uint32_t*>(a.x + pv * 8) = f2bf2(mx, my);
        if (!(fabsf(mx) <= 3.0e38f) || !(fabsf(my) <= 3.0e38f)) st[3] += 1.0;
        st[0] += (double)mx * mx + (double)my * my;
        if (x >= a.bx0 && x < a.bx1 && y >= a.by0 && y < a.by1 && z >= a.bz0 && z < a.bz1) {
            st[4] += mx;
            st[5] += my;
        }
    }
    // wavefront, then workgroup (fixed order)
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
        for (int k = 0; k < 6; k++) {
            const double o = __shfl_xor(st[k], off);
            st[k] = (k == 1 || k == 2) ? fmax(st[k], o) : st[k] + o;
        }
    }
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int k = 0; k < 6; k++) sh[wave][k] = st[k];
    __syncthreads();
    if (threadIdx.x < 6) {
        const int k = threadIdx.x;
        double r = sh[0][k];
        for (int w = 1; w < 4; w++) r = (k == 1 || k == 2) ? fmax(r, sh[w][k]) : r + sh[w][k];
        a.part[(size_t)blockIdx.x * 6 + k] = r;
    }
}

__global__ void __launch_bounds__(256) stats_reduce_kernel(const double* __restrict__ part, int nblocks,
                                                           double* __restrict__ out)
{
    __shared__ double sh[6][256];
    double v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int b = threadIdx.x; b < nblocks; b += 256) {
        const double* q = part + (size_t)b * 6;
        v[0] += q[0];
        v[1] = fmax(v[1], q[1]);
        v[2] = fmax(v[2], q[2]);
        v[3] += q[3];
        v[4] += q[4];
        v[5] += q[5];
    }
#pragma unroll
    for (int k = 0; k < 6; k++) sh[k][threadIdx.x] = v[k];
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) {
            sh[0][threadIdx.x] += sh[0][threadIdx.x + h];
            sh[1][threadIdx.x] = fmax(sh[1][threadIdx.x], sh[1][threadIdx.x + h]);
            sh[2][threadIdx.x] = fmax(sh[2][threadIdx.x], sh[2][threadIdx.x + h]);
            sh[3][threadIdx.x] += sh[3][threadIdx.x + h];
            sh[4][threadIdx.x] += sh[4][threadIdx.x + h];
            sh[5][threadIdx.x] += sh[5][threadIdx.x + h];
        }
        __syncthreads();
    }
    if (threadIdx.x < 6) out[threadIdx.x] = sh[threadIdx.x][0];
}

// flag[row] = 1 when the 16-voxel x segment `row` holds a pore.
__global__ void __launch_bounds__(256) row_flag_kernel(const uint8_t* __restrict__ mask, int nx, int ny, int nz,
                                                       int pitch, int nseg, uint8_t* __restrict__ flag)
{
    const long r = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= (long)nseg * ny * nz) return;
    const int seg = (int)(r % nseg);
    const long yz = r / nseg;
    const uint8_t* m = mask + (size_t)yz * pitch;
    uint8_t f = 0;
    for (int x = seg * 16; x < min(seg * 16 + 16, nx); x++) f |= m[x];
    flag[r] = f ? 1 : 0;
}

} // namespace

// ---- launchers ----

hipError_t launch_conv(int cin, int mode, const ConvArgs& a, int grid, hipStream_t s)
{
    const dim3 g(grid), b(256);
    if (cin == 8 && mode == 0) hipLaunchKernelGGL((conv_kernel<8, 0>), g, b, 0, s, a);
    else if (cin == 16 && mode == 0) hipLaunchKernelGGL((conv_kernel<16, 0>), g, b, 0, s, a);
    else if (cin == 16 && mode == 1) hipLaunchKernelGGL((conv_kernel<16, 1>), g, b, 0, s, a);
    else if (cin == 16 && mode == 2) hipLaunchKernelGGL((conv_kernel<16, 2>), g, b, 0, s, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

int conv_tiles(int nx, int ny, int nz)
{
    return ((nx + 15) / 16) * ((ny + kTileY - 1) / kTileY) * ((nz + kTileZ - 1) / kTileZ);
}

hipError_t launch_conv_tiled(int cin, int mode, const ConvArgs& a, int grid, hipStream_t s)
{
    const dim3 g(grid), b(256);
    if (cin == 8 && mode == 0) hipLaunchKernelGGL((conv_tile_kernel<8, 0>), g, b, 0, s, a);
    else if (cin == 16 && mode == 0) hipLaunchKernelGGL((conv_tile_kernel<16, 0>), g, b, 0, s, a);
    else if (cin == 16 && mode == 1) hipLaunchKernelGGL((conv_tile_kernel<16, 1>), g, b, 0, s, a);
    else if (cin == 16 && mode == 2) hipLaunchKernelGGL((conv_tile_kernel<16, 2>), g, b, 0, s, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

int conv_columns(int nx, int ny, int nz, int zc)
{
    return ((nx + 15) / 16) * ((ny + kZmY - 1) / kZmY) * ((nz + zc - 1) / zc);
}

hipError_t launch_conv_zm(int cin, int mode, const ConvArgs& a, int grid, hipStream_t s)
{
    const dim3 g(grid), b(256);
    if (cin == 8 && mode == 0) hipLaunchKernelGGL((conv_zm_kernel<8, 0>), g, b, 0, s, a);
    else if (cin == 16 && mode == 0) hipLaunchKernelGGL((conv_zm_kernel<16, 0>), g, b, 0, s, a);
    else if (cin == 16 && mode == 1) hipLaunchKernelGGL((conv_zm_kernel<16, 1>), g, b, 0, s, a);
    else if (cin == 16 && mode == 2) hipLaunchKernelGGL((conv_zm_kernel<16, 2>), g, b, 0, s, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_wgrad(int cin, const WgradArgs& a, int npart, hipStream_t s)
{
    const dim3 grid((unsigned)npart), block(kWgradThreads);
    if (cin == 8) hipLaunchKernelGGL((wgrad_kernel<8>), grid, block, 0, s, a, npart);
    else if (cin == 16) hipLaunchKernelGGL((wgrad_kernel<16>), grid, block, 0, s, a, npart);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_wreduce(const WreduceArgs& a, hipStream_t s)
{
    hipLaunchKernelGGL(wreduce_kernel, dim3((kWgradPart + kRedEl - 1) / kRedEl, 3), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_pack(const PackArgs& a, hipStream_t s)
{
    constexpr int n = 14 * 64 * 8; // of the largest set
    hipLaunchKernelGGL(pack_kernel, dim3((n + 255) / 256, kPackJobs), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_halo(const HaloArgs& a, hipStream_t s)
{
    const uint64_t n = (uint64_t)(a.nx + 2) * (a.ny + 2) * (a.nz + 2);
    hipLaunchKernelGGL(halo_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

static int blocks_for(long n) { return (int)((n + 255) / 256); }

hipError_t launch_features(const FeatureArgs& a, hipStream_t s)
{
    hipLaunchKernelGGL(feature_kernel, dim3(blocks_for((long)a.nx * a.ny * a.nz)), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_feature_copy(const float* f6, int nx, int ny, int nz, uint16_t* out, hipStream_t s)
{
    hipLaunchKernelGGL(feature_copy_kernel, dim3(blocks_for((long)nx * ny * nz)), dim3(256), 0, s, f6, nx, ny, nz,
                       out);
    return hipGetLastError();
}

hipError_t launch_gout_copy(const float* g2, int nx, int ny, int nz, uint16_t* out, hipStream_t s)
{
    hipLaunchKernelGGL(gout_copy_kernel, dim3(blocks_for((long)nx * ny * nz)), dim3(256), 0, s, g2, nx, ny, nz,
                       out);
    return hipGetLastError();
}

int loss_blocks(int nx, int ny, int nz) { return blocks_for((long)nx * ny * nz); }

hipError_t launch_loss(const LossArgs& a, hipStream_t s)
{
    hipLaunchKernelGGL(loss_kernel, dim3(loss_blocks(a.nx, a.ny, a.nz)), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_adam(float* p, float* m, float* v, const float* g, int n, float lr, float b1, float b2, float eps,
                       float c1, float c2, hipStream_t s)
{
    hipLaunchKernelGGL(adam_kernel, dim3(blocks_for(n)), dim3(256), 0, s, p, m, v, g, n, lr, b1, b2, eps, c1, c2);
    return hipGetLastError();
}

int apply_blocks(uint64_t n) { return (int)std::max<uint64_t>(1, std::min<uint64_t>(kApplyBlocks, (n + 255) / 256)); }

hipError_t launch_apply(const ApplyArgs& a, int blocks, hipStream_t s)
{
    if (a.vox) hipLaunchKernelGGL(apply_kernel<true>, dim3(blocks), dim3(256), 0, s, a);
    else hipLaunchKernelGGL(apply_kernel<false>, dim3(blocks), dim3(256), 0, s, a);
    return hipGetLastError();
}

} // namespace nmr

namespace nmr {

hipError_t launch_stats_reduce(const double* part, int nblocks, double* out, hipStream_t s)
{
    hipLaunchKernelGGL(stats_reduce_kernel, dim3(1), dim3(256), 0, s, part, nblocks, out);
    return hipGetLastError();
}

hipError_t launch_row_flags(const uint8_t* mask, int nx, int ny, int nz, int pitch, uint8_t* flag, hipStream_t s)
{
    const int nseg = (nx + 15) / 16;
    const long n = (long)nseg * ny * nz;
    hipLaunchKernelGGL(row_flag_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, mask, nx, ny, nz, pitch,
                       nseg, flag);
    return hipGetLastError();
}

} // namespace nmr
