// nmr_pore_list.hip -- host side of the pore list (nmr_pores.hip): its
// buffers, and building it from a mask on the device.
#include "nmr_internal.h"

using nmri::fail;

namespace nmri {

namespace {

template <typename T>
int grow(T** p, size_t count, int fill, hipStream_t s, int64_t* bytes, size_t old_count)
{
    const size_t n = std::max<size_t>(count * sizeof(T), 256);
    if (*p) {
        HIP_TRY(hipStreamSynchronize(s));
        HIP_TRY(hipFree(*p));
        *p = nullptr;
        *bytes -= (int64_t)std::max<size_t>(old_count * sizeof(T), 256);
    }
    HIP_TRY(hipMalloc((void**)p, n));
    *bytes += (int64_t)n;
    HIP_TRY(hipMemsetAsync(*p, fill, n, s));
    return NMR_OK;
}

} // namespace

bool pores_fit(uint64_t nslots, bool vel)
{
    constexpr uint64_t state = 3 * sizeof(float), rec = sizeof(*PoreList::rec);
    static_assert(rec >= state && state >= sizeof(*PoreList::off16) && state >= sizeof(*PoreList::vox), "widest arrays");
    return nslots > 64 && (nslots + 64) * (vel ? rec : state) < ((uint64_t)1 << 32) - 256;
}

double pores_padded(int nx, int ny, int nz)
{
    return (((int64_t)nx + 63) / 64 * 64) * (double)(((int64_t)ny + 15) / 16 * 16) * nz;
}

bool pores_pay(double slots, const PoreProblem& p)
{
    // The plain problem: where at most 0.6 of the voxels are pores, or the
    // list's data stay well inside the memory-side cache.  Measured per step,
    // list against tiles on bricks: 256^3 flow, two components, porosity 0.2 /
    // 0.35 / 0.5 / 0.65 / 0.8 / 1: 19.9 / 31.2 / 61.2 / 81.9 / 101 / 124 against
    // 57.9 / 66.2 / 74.1 / 80.1 / 84.0 / 84.2 us; 256^3, one component without
    // flow, 0.5 / 0.8 (188 MB) / 1: 29.3 / 41.0 / 47.8 against 36.4 / 39.0 / 39.2;
    // 160^3 MacCormack, 1 (172 MB): 47.9 against 54.1; 512x512x256, 1: 511
    // against 388; 64^3, one component, 1: 2.9 against 9.4.
    if (slots > 0.6 * p.voxels && 4.0 * ((p.mak ? 3 : 2) * p.nc + (p.vel ? 3 : 0) + 1.5) * slots > 180e6) return false;
    // Ghosts, per-voxel data and solids that are read cost the list, which
    // loads offsets and masks for them, more than the tiles, and the less the
    // more components share them.  So the voxels that the tiles work on (whole
    // 64 x 16 tiles) are compared with the slots weighed by what they load more;
    // the factors are fitted to 36 kinds of problem on 128^3 to 320^3 at
    // porosities 0.3 to 1.  Time of a step on tiles over that on the list: one
    // component, zero-value ghosts, 200^3, porosity 0.4 / 0.6 / 1: 1.14 / 0.87 /
    // 0.58; periodic, 256^3, 0.3 / 0.5 / 0.7: 1.28 / 0.90 / 0.65; two components
    // with flow, periodic, 200^3, 0.8 / 1: 1.32 / 0.82; MacCormack, periodic,
    // per-voxel coefficients and weights, 160^3, 0.6 / 0.8 / 1: 1.13 / 0.87 / 0.71.
    // (On seven other grids, 612 problems, the choice costs more than 5 % in
    // five, 14 % at most.)
    const bool ghosts = p.ghost_x || p.zeros || p.wraps > 0;
    const double more = (p.ghost_x ? 0.6 : 0.0) + (p.zeros ? 0.55 : 0.0) + 0.15 * p.wraps +
                        (p.coef && ghosts ? 0.5 : 0.0) + (p.weights ? 0.12 : 0.0) + (p.solids ? 0.17 : 0.0);
    // words a slot: state (predictor), record or offsets, descriptor, lane
    // masks, x and 16-bit offsets, positions, per-voxel data
    const double words = (p.mak ? 3 : 2) * p.nc + (p.vel ? 4 : 1) + 0.5 +
                         (p.zeros || p.solids || (p.coef && ghosts) ? 0.56 : 0.0) + (p.ghost_x ? 1 : 0) +
                         (p.wraps > 0 ? 2 : 0) + (p.nc == 3 ? 1 : 0) + (p.coef ? 2 + (p.nc == 3) : 0) + (p.field ? 1 : 0) +
                         (p.weights ? 2 : 0);
    static const double in_cache[3] = {0.85, 1.05, 1.25}, past[3] = {0.65, 0.75, 1.0}; // by components
    double most = 4.0 * words * slots <= 225e6 ? in_cache[p.nc - 1] : past[p.nc - 1];
    if (p.voxels <= 2.2e6) most *= 2.0; // (up to 128^3: the tiles do not fill the chip; 128^3 all pores 0.9-1.5)
    return slots * (1.0 + more / (p.nc * p.nc)) <= most * p.padded;
}

int pores_alloc(PoreList* L, uint32_t nslots, const PoreNeeds& n, hipStream_t s, int64_t* bytes)
{
    const bool more = nslots > L->cap || n.nc != L->nc;
    const size_t old = L->cap, cap = more ? (size_t)nslots : L->cap;
    const size_t all = cap + 64, was = old + 64; // a spare group past the end: the last slot reads the one after it
    int rc = NMR_OK;
    auto need = [&](auto** p, size_t per, int fill) {
        if (rc) return;
        if (more || !*p) rc = grow(p, all * per, fill, s, bytes, was * per);
        else if (hipMemsetAsync(*p, fill, all * per * sizeof(**p), s) != hipSuccess)
            rc = fail(NMR_ERR_DEVICE, "pore list: clearing a buffer failed");
    };
    auto groups = [&](auto** p) {
        if (rc) return;
        if (more || !*p) rc = grow(p, all / 64, 0, s, bytes, was / 64);
        else if (hipMemsetAsync(*p, 0, all / 64 * sizeof(**p), s) != hipSuccess)
            rc = fail(NMR_ERR_DEVICE, "pore list: clearing a buffer failed");
    };
    if (L->nc != n.nc) { // sizes below are in slots of nc words
        for (float** p : {&L->state[0], &L->state[1], &L->pred})
            if (*p) {
                HIP_TRY(hipStreamSynchronize(s));
                HIP_TRY(hipFree(*p));
                *p = nullptr;
                *bytes -= (int64_t)(was * 4 * (size_t)L->nc);
            }
        L->nc = n.nc;
    }
    groups(&L->groups);
    if (n.aux || L->aux) groups(&L->aux);
    need(&L->off8, 1, 0);
    need(&L->off16, 1, 0);
    if (n.xoff || L->xoff) need(&L->xoff, 1, 0);
    need(&L->vox, 1, 0xff);
    if (n.nc == 3 || L->xy) need(&L->xy, 1, 0);
    need(&L->state[0], (size_t)n.nc, 0);
    need(&L->state[1], (size_t)n.nc, 0);
    if (n.pred || L->pred) need(&L->pred, (size_t)n.nc, 0);
    if (n.vel || L->rec) need(&L->rec, 1, 0);
    if (more)
        for (float*& p : L->pv)
            if (p && !rc) {
                if (hipStreamSynchronize(s) != hipSuccess || hipFree(p) != hipSuccess)
                    rc = fail(NMR_ERR_DEVICE, "pore list: freeing a buffer failed");
                p = nullptr;
                *bytes -= (int64_t)(was * 4);
            }
    if (rc) return rc;
    L->cap = cap;
    L->nslots = nslots;
    L->wide = false;
    L->nbx = L->nby = L->nbz = 0;
    L->blocks_ok = false;
    return NMR_OK;
}

void pores_free(PoreList* L)
{
    for (void* p : {(void*)L->groups, (void*)L->aux, (void*)L->off8, (void*)L->off16, (void*)L->xoff, (void*)L->vox,
                    (void*)L->xy, (void*)L->state[0], (void*)L->state[1], (void*)L->pred,
                    (void*)L->rec, (void*)L->blocks, (void*)L->bcount, (void*)L->pv[0],
                    (void*)L->pv[1], (void*)L->pv[2], (void*)L->pv[3], (void*)L->pv[4], (void*)L->pv[5]})
        if (p) (void)hipFree(p);
    *L = PoreList{};
}

void pores_drop_temp(nmr::PoreBuild* b)
{
    for (void* p : {(void*)b->rows, (void*)b->planes, (void*)b->slotmap, (void*)b->overflow})
        if (p) (void)hipFree(p);
    b->rows = nullptr;
    b->planes = nullptr;
    b->slotmap = nullptr;
    b->overflow = nullptr;
}

int pores_temp(nmr::PoreBuild* b, size_t rows, size_t planes, size_t voxels, hipStream_t s)
{
    b->rows = nullptr;
    b->planes = nullptr;
    b->slotmap = nullptr;
    b->overflow = nullptr;
    int rc = NMR_OK;
    auto check = [&](hipError_t e) {
        if (!rc && e != hipSuccess)
            rc = fail(e == hipErrorOutOfMemory ? NMR_ERR_NOMEM : NMR_ERR_DEVICE, "pore list: %s", hipGetErrorString(e));
        return !rc;
    };
    if (check(hipMalloc((void**)&b->rows, rows * sizeof(uint32_t))) &&
        check(hipMalloc((void**)&b->planes, (planes + 1) * sizeof(uint64_t))) &&
        check(hipMalloc((void**)&b->slotmap, voxels * sizeof(uint32_t))) &&
        check(hipMalloc((void**)&b->overflow, 256)))
        check(hipMemsetAsync(b->overflow, 0, 256, s));
    if (rc) pores_drop_temp(b);
    return rc;
}

void pores_into(const PoreList& L, nmr::PoreBuild* b, uint64_t end)
{
    b->vox = L.vox;
    b->groups = L.groups;
    b->aux = L.aux;
    b->off8 = L.off8;
    b->off16 = L.off16;
    b->xoff = L.xoff;
    b->xy = L.xy;
    b->count = (int64_t)((end - b->first) / 64);
}

int pores_finish(PoreList* L, const nmr::PoreBuild& b, hipStream_t s, bool* ok)
{
    int over[2] = {0, 0};
    HIP_TRY(hipMemcpyAsync(over, b.overflow, sizeof(over), hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    *ok = over[0] == 0;
    L->wide = over[1] != 0;
    L->blocks_ok = *ok && b.blocks;
    return NMR_OK;
}

int pores_blocks(PoreList* L, nmr::PoreBuild* b, hipStream_t s, int64_t* bytes)
{
    // up to two boxes a CU: past one a CU they run in turns.  us a step, blocks
    // against single steps, at 1 component / 2 with velocity / 3 / 3 with
    // velocity: 20^3 (27 boxes) 1.4 1.7 1.9 2.0 against 3.7 3.7 3.7 3.9; 48^3
    // (216) 1.4 1.8 2.2 2.4 against 3.7 3.9 3.8 4.0; 64^3 (512) 2.2 2.9 3.6 3.9
    // against 4.0 4.0 4.0 4.2; 80^3 (1000) 3.7 5.3 6.5 7.2 against 3.8 4.3 4.4
    // 4.5; the porosity (0.15, 0.3, 0.5 at 64^3) hardly matters.
    constexpr uint64_t kMost = 512;
    constexpr int e = nmr::kBlockEdge;
    const uint64_t nx = (b->nx + e - 1) / e, ny = (b->ny + e - 1) / e, nz = (b->nz + e - 1) / e, n = nx * ny * nz;
    if (n > kMost) return NMR_OK;
    int rc = NMR_OK;
    if (n > L->ncap) {
        if ((rc = grow(&L->bcount, n * 8, 0, s, bytes, L->ncap * 8))) return rc;
        L->ncap = n;
    }
    b->bcount = L->bcount;
    b->nbx = (int)nx;
    b->nby = (int)ny;
    b->nbz = (int)nz;
    HIP_TRY(nmr::launch_block_count(*b, s));
    int total = 0;
    HIP_TRY(hipMemcpyAsync(&total, b->overflow + 2, sizeof(total), hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    const size_t all = (size_t)total + nmr::kBlockThreads; // (a block's first load is a whole workgroup's)
    if (all > L->bcap) {
        if ((rc = grow(&L->blocks, all, 0, s, bytes, L->bcap))) return rc;
        L->bcap = all;
    }
    b->blocks = L->blocks;
    L->nbx = b->nbx;
    L->nby = b->nby;
    L->nbz = b->nbz;
    return NMR_OK;
}

int pores_per_tile(int64_t groups)
{
    // one group a wavefront: 256^3, porosity 0.2 (52 K groups) 19.8 / 20.2 /
    // 20.3 us a step at 4 / 8 / 12 groups a workgroup, 512x512x130 35.3 / 36.1
    // at 4 / 8, 64^3 2.8 / 3.3; more where a step's partial sums, one a
    // workgroup, would pass 64 K
    int per = 4;
    while (groups / per > 65536) per *= 2;
    return per;
}

} // namespace nmri
