// nmr_kernels.h -- internal interface between the C ABI (nmr_abi.hip) and
// the gfx950 kernels (nmr_kernels.hip).  Not part of the public ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nmr {

// (local arrays of uint4 end up in scratch memory where those of this type do not)
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Per-step coefficients of the update, all pre-multiplied by dt (FP32).
struct Coef {
    float cdx, cdy, cdz;    // dt*D/d^2 per axis (0 when diffusion is off)
    float hx, hy, hz;       // dt/d per axis
    float r1, r2;           // dt/T1_bulk, dt/T2_bulk
    float s1x, s1y, s1z;    // dt*rho1/d per solid face
    float s2x, s2y, s2z;    // dt*rho2/d per solid face
    float peq;              // equilibrium magnetization
    float n0, n1, n2;       // unit main-field direction
    float bgx, bgy, bgz;    // dt*g*G_a*d_a: precession angle per index unit
    float dtg;              // dt*g (0 without precession): angle per tesla of a per-voxel field
};

struct SweepArgs {
    const float* min[3];
    float* mout[3];
    const uint8_t* mask;
    const float* adv[3];    // upwind velocity sums per axis (adv_kernel), laid out as the state
    double* partials;       // [nblocks][nc] signal partials of this step
    int nx, ny, nz;
    int pitch, pitch1;
    int ntx, nty, ntz, lz, nblocks;
    int bx0, bx1, by0, by1, bz0, bz1; // signal window [b0, b1) per axis
    int inert;              // no pore-solid face carries velocity
    int nby;                // brick layout: brick rows per plane
    Coef c;
};

// One instance of a batch (device memory).
struct BatchInst {
    float* m[2][3];         // ping-pong magnetization buffers (rows, or bricks with the velocity sums in bricks too)
    const uint8_t* mask;
    const float* adv[3];    // upwind velocity sums, laid out as the state
    int nx, ny, nz, pitch, pitch1;
    int ntx, nty, ntz, lz;
    int bx0, bx1, by0, by1, bz0, bz1;
    int inert;
    int nby;                // brick layout: brick rows per plane
    int nd, nD;             // PGSE lobe length and start of the second lobe (steps)
    float bgz;              // dt*g*G*dz of the +G lobe, rounded once on the host
                            // (the -G lobe negates it, which is exact)
    Coef c;                 // coefficients without the gradient
};

struct BatchArgs {
    const BatchInst* inst;
    const int2* tiles;      // (instance, tile index within the instance)
    int ntiles;
    int parity;             // which ping-pong buffer holds the current state
    int local_step;         // step within the captured chunk
    const int* step_base;   // device step counter (first step of the chunk)
    double* partials;       // [ntiles][nc] of this step
};

// Per-voxel sums of the two face velocities of each axis from the face
// velocities (row layout: vx [nz][ny][pitch1], vy [nz][ny+1][pitch], vz
// [nz+1][ny][pitch]), written as the state's rows [nz][ny][pitch]: the
// upwind sums of the plain sweep (0 where the inflow face carries no
// velocity) or, with centred, the plain sums of the MacCormack stages.
struct AdvArgs {
    const float* vx;
    const float* vy;
    const float* vz;
    float* out[3];
    int nx, ny, nz, pitch, pitch1;
    int centred;
};

struct InertArgs {
    const uint8_t* mask;
    const float* vx;
    const float* vy;
    const float* vz;
    int* flag;
    int nx, ny, nz, pitch, pitch1;
};

// Two-step (temporally blocked) sweep: one x tile (nx <= 4*LX), TY = 512/LX - 2
// rows per tile, z-chunks of lz planes.
struct Sweep2Args {
    const float* min[3];
    float* mout[3];
    const uint8_t* mask;
    const float* adv[3];    // upwind velocity sums (row layout)
    double* partials1;      // [nblocks][nc] signal after the first step
    double* partials2;      // [nblocks][nc] signal after the second step
    int nx, ny, nz;
    int pitch, pitch1;
    int nty, ntz, lz, nblocks;
    int bx0, bx1, by0, by1, bz0, bz1;
    Coef c1, c2;            // coefficients of the two steps
};

// Per-voxel step for the schemes and boundary conditions the z-sweep does
// not cover (MacCormack, periodic and zero-value ghosts).
enum { GEN_UPWIND = 0, GEN_PREDICT = 1, GEN_CORRECT = 2 };
enum { BC_NEUMANN = 0, BC_PERIODIC = 1, BC_DIRICHLET = 2 };
struct GenArgs {
    const float* m[3];      // state at the start of the step
    const float* p[3];      // predictor (corrector stage)
    float* out[3];          // result of the stage
    const uint8_t* mask;
    const float* vx;
    const float* vy;
    const float* vz;
    int nx, ny, nz, pitch, pitch1;
    int bc[3];              // BC_* per axis
    int vel;                // face velocities present
    int amask;              // upwind advection only across faces to pores (NMR_F_ADVECT_MASK)
    const float* dn;        // per-voxel diffusivity / reference (null: uniform, from the mask)
    const float* r1v;       // per-voxel dt/T1 with surface terms (null: from the mask)
    const float* r2v;       // per-voxel dt/T2 with surface terms
    const float* bn;        // per-voxel field (T) along axis bnax, in place of that axis's gradient field; or null
    int bnax;
    Coef c;
};

// General z-sweep: the sweep's tile march (planes in registers, plane k
// with its halo in LDS) for what the plain sweep does not cover -- the
// MacCormack stages, periodic and zero-value ghosts, per-voxel
// coefficients -- with the per-voxel kernel's arithmetic, so that the two
// agree bit for bit.
struct GSweepArgs {
    const float* f[3];      // field the stage differentiates (the state, or the predictor)
    const float* mavg[3];   // corrector stage: the state at the start of the step
    float* out[3];          // result of the stage
    const uint8_t* mask;
    const float* dn;        // per-voxel diffusivity / reference (coefficient variant)
    const float* r1v;       // per-voxel dt/T1
    const float* r2v;       // per-voxel dt/T2
    const float* bn;        // per-voxel field (T) along axis bnax, in place of that axis's gradient field; or null
    int bnax;
    double* partials;       // [nblocks][nc] pore sums of the result, or null
    const float* w[2];      // brick sweep: phase weights (row layout) of fused weighted sums,
                            // partials then [nblocks][2*nc]; or null
    const float* cs[3];     // face-velocity sums per voxel, laid out as the state: centred
                            // (MacCormack stages) or upwind (the upwind stage), AdvArgs
    int nx, ny, nz, pitch, pitch1;
    int ntx, nty, ntz, lz, nblocks;
    int bx0, bx1, by0, by1, bz0, bz1; // signal window [b0, b1) per axis
    int bc[3];              // BC_* per axis
    int skip_m;             // all-solid chunks are never read by a pore: not loaded
    int amask;              // upwind advection only across faces to pores (NMR_F_ADVECT_MASK)
    int nby;                // brick layout (lanes 16): brick rows per plane
    Coef c;
};

struct PulseArgs {
    float* m[3];            // row layout, or bricks when nb8 > 0
    const uint8_t* mask;
    int nx, ny, nz, pitch, nc;
    int nby, nb8;           // brick layout: brick rows per plane, bricks per brick row (0: rows)
    int flag;
    double param, ax, ay, az;
    double dx, dy, dz, gamma;
};

struct FieldSumArgs {
    const float* f[3];      // row layout, or bricks when nb8 > 0
    const uint8_t* mask;
    const float* w[2];      // phase weights (null: plain sums)
    double* part;           // [field_sum_blocks][nc] or, with weights, [..][2*nc]
    int nx, ny, nz, pitch;
    int bx0, bx1, by0, by1, bz0, bz1;
    int nby, nb8;           // brick layout of f (0: rows)
};

// ---- list of pores (nmr_pores.hip) ----
// 64 slots of the list, in the grid's order and of one plane: the lowest slot
// that its lanes read per side (x-, x+, y-, y+, z-, z+), which the offsets
// count from, and 64-bit lane masks.
struct PoreGroup {
    uint32_t base[6];
    float zc;               // plane + 1/2
    uint32_t wide;          // an offset needs more than 8 bits: the 16-bit ones are read
    uint64_t pore[6];       // the neighbour on this side counts as a pore
    uint64_t active;        // the slot holds a pore (else a solid that pores read, or nothing)
    uint64_t window;        // a pore inside the signal window
    uint64_t xm, xp;        // the x neighbour is the slot before / after (else the own value is read)
    uint64_t pad[2];
};
static_assert(sizeof(PoreGroup) == 128, "group descriptor");

// Lane masks for ghosts other than zero-derivative ones and for solids that
// are read: the side is read through its offset, reads as 0, is a ghost.
struct PoreAux {
    uint64_t has[6], zero[6], ghost[6];
};

// Consecutive groups of one workgroup of a batch, all of one instance.
struct PoreTile {
    uint32_t first, count;
    uint32_t inst;
};

// One instance of a batch: coefficients without the gradient, and its
// pulsed-gradient pair (as BatchInst).
struct PoreInst {
    Coef c;
    float bgz;
    int nd, nD;
};

struct PoreArgs {
    const float* f;         // field the stage differentiates, nc floats per slot
    const float* mavg;      // corrector stage: the state at the start of the step
    float* out;
    const PoreGroup* groups;
    const PoreAux* aux;     // where solids are read or a ghost reads as 0; or null
    const PoreAux* ghost;   // the same array, for per-voxel diffusivities behind ghosts; or null
    const uint4* rec;       // with velocity: 8-bit y-, y+, z-, z+ offsets, 3 velocity sums (upwind or centred)
    const uint32_t* off8;   // without: the offsets
    const uint2* off16;     // the same in 16 bits
    const uint32_t* xoff;   // 16-bit x-, x+ offsets where they are not the slots next to it; or null
    const uint32_t* xy;     // x | y << 16 (three components)
    const float* dn;        // per-voxel diffusivity / reference, dt/T1, dt/T2, field: or null
    const float* r1v;
    const float* r2v;
    const float* bn;
    const float* w[2];      // phase weights, or null
    double* partials;       // [ntiles][sums] of this step
    int ntiles;             // workgroups
    int ngroups, gpt;       // one domain: past its last group (group 0 is empty), groups per workgroup
    int wide;               // some group needs its 16-bit offsets
    int bnax, amask;
    const PoreTile* tiles;  // a batch: the workgroups' groups, its instances, the device step counter and
    const PoreInst* inst;   //   the step within the chunk
    const int* step_base;
    int local_step;
    Coef c;
};

// Building the list of one domain; slots [first, ...), whole groups.
struct PoreBuild {
    const uint8_t* mask;
    int nx, ny, nz, pitch;
    int bc[3];
    int read_solids;        // upwind velocity on pore-solid faces: solids next to pores get slots
    int w[6];               // signal window
    uint64_t first;         // first slot (a multiple of 64)
    uint64_t shift;         // to add to planes, where they were counted from another slot
    int64_t count;          // groups of this domain (linking)
    uint32_t* rows;         // [nz*ny] slots before the row in its plane
    uint64_t* planes;       // [nz + 1] first slot of each plane
    uint32_t* slotmap;      // [nz][ny][pitch] slot of a voxel, 0: none
    uint32_t* vox;          // voxel (row layout) of a slot, ~0: empty
    PoreGroup* groups;
    PoreAux* aux;           // or null
    uint32_t* off8;
    uint2* off16;
    uint32_t* xoff;         // or null
    uint32_t* xy;           // or null
    uint4* rec;             // records, to be written here from
    const float* vel[3];    //   the velocity sums (row layout) unless they are null
    int* found;             // what is found on the way: [0] an offset that does not fit, [1] a group that needs
                            // 16-bit offsets, [2] slots of all blocks, [3] a solid that is not finite
    void* temp;             // what rows, planes, slotmap, bcount and found lie in, where that is their own
    u32x4* blocks;          // the blocks' slots, or null
    uint32_t* bcount;       // [nblocks][8]: slots within 0 .. kBlockSteps faces of the box, the first one's place
    uint32_t* bcount_to;    // the same in the list
    int nbx, nby, nbz;      // boxes per axis
};

// Several steps of the pores of one box of kBlockEdge^3 voxels in one
// workgroup (nmr_pore_blocks.hip): its pores and those within kBlockSteps
// faces of it, by distance.
constexpr int kBlockEdge = 8, kBlockSteps = 4, kBlockThreads = 1024;
struct BlockArgs {
    const float* f;         // the list's state, nc floats per slot
    float* out;
    const uint4* rec;       // with velocity: the list's records
    const u32x4* blocks;
    const uint32_t* bcount;
    double* partials;       // [steps][nblocks][nc]
    int nblocks, nbx, nby;
    int steps;              // 1 .. kBlockSteps
    Coef c[kBlockSteps];
};

hipError_t launch_pore_count(const PoreBuild& b, hipStream_t s);
hipError_t launch_pore_link(const PoreBuild& b, hipStream_t s);
hipError_t launch_block_count(const PoreBuild& b, hipStream_t s);
hipError_t launch_block_build(const PoreBuild& b, hipStream_t s);
// a.steps plain upwind steps (exact: with the exact phase)
hipError_t launch_blocks(int nc, bool vel, bool exact, const BlockArgs& a, hipStream_t s);
// out[stride*slot + at] = row[vox[slot]] for slots [s0, s1), 0 at empty ones
hipError_t launch_pore_gather(const float* row, const uint32_t* vox, uint32_t s0, uint32_t s1, int stride, int at,
                              float* out, hipStream_t s);
// rec[s].x = off8[s], s < n
hipError_t launch_pore_record(const uint32_t* off8, uint32_t n, uint4* rec, hipStream_t s);
// row[vox[slot]] (and row2, unless null) = f[stride*slot + at]
hipError_t launch_pore_scatter(const float* f, const uint32_t* vox, uint32_t s0, uint32_t s1, int stride, int at,
                               float* row, float* row2, hipStream_t s);
// *flag = 1 when row is not finite at a solid
hipError_t launch_solids_finite(const float* row, const uint8_t* mask, size_t n, int* flag, hipStream_t s);
hipError_t launch_pore_sum(int nc, const PoreArgs& a, hipStream_t s);
// a step (stage st) of the whole list; gen: anything but the plain problem
// (per-voxel data, ghosts other than zero-derivative ones, solids that are
// read, masked advection)
hipError_t launch_pores(int nc, bool vel, int st, bool exact, bool gen, bool coef, const PoreArgs& a, hipStream_t s);
hipError_t launch_pore_pulse(const PulseArgs& a, float* f, int nc, const uint32_t* vox, uint32_t s0, uint32_t s1,
                             hipStream_t s);

// ---- learned corrector (nmr_learn_kernels.hip) ----
// Tensors: BF16 channels-last on the grid padded by one zero voxel per side.
constexpr int kWgradPart = 27 * 256 + 16; // floats per partial of wgrad

struct ConvArgs {
    const uint16_t* in;     // [(nz+2)(ny+2)(nx+2)][cin]
    const uint16_t* wa;     // packed A fragments [chunks][64][8]
    const float* bias;      // [16] (forward modes)
    const uint16_t* ref;    // gate tensor [..][16] (input-gradient mode)
    uint16_t* out;          // [..][16]
    float* outf;            // [..][2] (linear mode)
    const int* rows;        // row list, row = (z*ny + y)*nseg + seg; null = all rows
    int nrows;
    int nx, ny, nz, nseg;   // nseg = ceil(nx/16)
    int zc;                 // output planes per column of the z-marching kernel
};

struct WgradArgs {
    const uint16_t* in;     // layer input [..][cin]
    const uint16_t* gout;   // output gradient [..][16]
    float* part;            // [npart][kWgradPart]
    int nx, ny, nz;
};

struct FeatureArgs {
    const float* mx;
    const float* my;        // nullable
    const uint8_t* mask;
    const float* vx;        // nullable (no velocity)
    const float* vy;
    const float* vz;
    uint16_t* out;          // [..][8]
    int nx, ny, nz, pitch, pitch1;
    float vinv;             // 1 / velocity scale
};

struct WreduceArgs {
    const float* part[3];   // [npart][kWgradPart] of each layer
    float* grad[3];
    int cin[3], cout[3];    // real channels
    int npart;
};

// A layer's weights, and the fragments to make of them.
struct PackJob {
    const float* w;
    uint16_t* frag;
    int cin_real, cout_real, cin_store, backward;
};
constexpr int kPackJobs = 5;
struct PackArgs {
    PackJob job[kPackJobs];
};

struct HaloArgs {
    uint16_t* x;            // [..][8]
    uint16_t* t[5];         // [..][16], or null
    int nx, ny, nz;
};

struct LossArgs {
    const float* pred;      // [..][2]
    const float *ax, *ay;   // target: a - b, compact with pitch
    const float *bx, *by;
    const uint8_t* mask;
    uint16_t* gout;         // [..][16]
    double* lpart;          // [blocks]
    int nx, ny, nz, pitch;
    float tinv;             // 1 / output scale
    float winv;             // 1 / number of pores
};

struct ApplyArgs {
    float* mx;              // the state in rows, or
    float* my;
    float* slots;           //   in the list of the pores: (Mx, My) of the slots [s0, s1), whose voxels
    const uint32_t* vox;    //   vox[] gives; null: rows
    uint32_t s0, s1;
    uint16_t* x;            // the net's input, whose channels 0 and 1 take the state at the pores
    const uint8_t* mask;
    const float* pred;      // [..][2] or null (statistics only)
    double* part;           // [blocks][6]
    int nx, ny, nz, pitch;
    int bx0, bx1, by0, by1, bz0, bz1;
    float scale;
};

hipError_t launch_conv(int cin, int mode, const ConvArgs& a, int grid, hipStream_t s);
// tiles of 16 x 8 x 4 output voxels of the LDS-staged convolution (all rows)
int conv_tiles(int nx, int ny, int nz);
hipError_t launch_conv_tiled(int cin, int mode, const ConvArgs& a, int grid, hipStream_t s);
// columns of 16 x 16 output rows by zc planes of the z-marching convolution
int conv_columns(int nx, int ny, int nz, int zc);
hipError_t launch_conv_zm(int cin, int mode, const ConvArgs& a, int grid, hipStream_t s);
// npart partial sums
hipError_t launch_wgrad(int cin, const WgradArgs& a, int npart, hipStream_t s);
hipError_t launch_wreduce(const WreduceArgs& a, hipStream_t s);
hipError_t launch_pack(const PackArgs& a, hipStream_t s);
hipError_t launch_halo(const HaloArgs& a, hipStream_t s);
hipError_t launch_features(const FeatureArgs& a, hipStream_t s);
hipError_t launch_feature_copy(const float* f6, int nx, int ny, int nz, uint16_t* out, hipStream_t s);
hipError_t launch_gout_copy(const float* g2, int nx, int ny, int nz, uint16_t* out, hipStream_t s);
int loss_blocks(int nx, int ny, int nz);
hipError_t launch_loss(const LossArgs& a, hipStream_t s);
hipError_t launch_adam(float* p, float* m, float* v, const float* g, int n, float lr, float b1, float b2, float eps,
                       float c1, float c2, hipStream_t s);
// workgroups for n voxels or slots
int apply_blocks(uint64_t n);
hipError_t launch_apply(const ApplyArgs& a, int blocks, hipStream_t s);
// out: six doubles, in host memory that the device sees
hipError_t launch_stats_reduce(const double* part, int nblocks, double* out, hipStream_t s);
hipError_t launch_row_flags(const uint8_t* mask, int nx, int ny, int nz, int pitch, uint8_t* flag, hipStream_t s);
// grid workgroups of 256 threads, each wave `iters` x 8 MFMA 16x16x32 BF16; out: grid*256 floats
hipError_t launch_mfma_rate(int iters, int grid, float* out, hipStream_t s);

int num_variants();
// the compacted brick sweep's variant index (the last one)
int compact_variant();
// steps: time steps per pass (1, or 2 for the temporally blocked sweep)
bool variant_shape(int v, int* lx, int* rpt, int* tx, int* ty, int* steps);
// keep: the state's loads and stores go without the non-temporal hint (the
// brick 64 x 16 tile, variant 4; other tiles ignore it)
hipError_t launch_sweep(int nc, bool vel, bool exact, int variant, const SweepArgs& a, hipStream_t s,
                        bool brick = false, bool keep = false);
// whether tile variant v has a brick-layout sweep, and the automatic one
bool brick_variant(int v);
int brick_auto_variant(int nx);
// floats of a field of nc4 4-voxel chunks per row, Y rows, Z planes in
// bricks of 8 x-voxels by 4 rows
size_t brick_floats(int nc4, int Y, int Z);
// row layout [Z][Y][4*nc4] <-> bricks (to_brick: row -> brick)
hipError_t launch_brick(const float* src, float* dst, int nc4, int Y, int Z, bool to_brick, hipStream_t s);
hipError_t launch_sweep2(int nc, bool vel, bool exact, int lx, const Sweep2Args& a, hipStream_t s);
hipError_t launch_batch(int nc, bool vel, bool exact, int variant, int grid, const BatchArgs& b, hipStream_t s,
                        bool brick = false);
int batch_resident_blocks(int nc, bool vel, bool exact, int variant, bool brick = false);
// Workgroups of the one-step sweep (variant 0..6, row or brick layout) and of
// the general sweep's upwind kernel (upwind) or MacCormack corrector (on
// bricks with fused phase-weighted sums: its weighted instantiation)
// resident on the device at once (CUs x occupancy); -1 if the query fails.
int sweep_resident_blocks(int nc, bool vel, bool exact, int variant, bool brick, bool keep = false);
int gsweep_resident_blocks(int nc, bool vel, bool coef, int lanes, bool brick, bool weighted, bool upwind);
hipError_t launch_batch_reduce(const double* part, int ntiles, int nc, const int* off, const int* ids,
                               const int* step_base, int row0, int64_t rows, double* signal, int nsteps, int ninst,
                               hipStream_t s);
hipError_t launch_step_advance(int* step_base, int n, hipStream_t s);
hipError_t launch_reduce_partials(const double* part, int nsteps, int nwg, int nc, double* out, hipStream_t s);
hipError_t launch_inert_check(const InertArgs& a, hipStream_t s);
hipError_t launch_adv(const AdvArgs& a, hipStream_t s);
hipError_t launch_pulse(const PulseArgs& a, hipStream_t s);
hipError_t launch_general(int nc, int stage, const GenArgs& a, hipStream_t s);
// lanes per tile row of the general sweep for a grid of width nx (tile 4*lanes wide)
int gsweep_lanes(int nx);
// keep: as for launch_sweep (the brick sweeps)
hipError_t launch_gsweep(int nc, bool vel, int stage, bool coef, int lanes, const GSweepArgs& a, hipStream_t s,
                         bool brick = false, bool keep = false);
// m[q][i] = 0 where mask[i] == 0, i < n, for q < nc
hipError_t launch_zero_solids(float* const* m, int nc, const uint8_t* mask, size_t n, hipStream_t s);
// the same for fields in bricks (nz planes of ny rows of pitch voxels)
// dst = src over nchunks 16-byte chunks (16-byte aligned) by copy kernel
// shape `kind` (0 .. copy_kinds() - 1) on a device of `cus` compute units
int copy_kinds();
hipError_t launch_copy(int kind, const float* src, float* dst, size_t nchunks, int cus, hipStream_t s);
hipError_t launch_zero_solids_brick(float* const* m, int nc, const uint8_t* mask, int ny, int nz, int pitch,
                                    hipStream_t s);
// workgroups (= partials) of a field sum over the signal window
int field_sum_blocks(const FieldSumArgs& a);
hipError_t launch_field_sum(int nc, const FieldSumArgs& a, hipStream_t s);

} // namespace nmr
