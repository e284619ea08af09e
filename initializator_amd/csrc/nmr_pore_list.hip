// nmr_pore_list.hip -- host side of the pore list (nmr_pores.hip): its
// buffers, and building it from a mask on the device.
#include "nmr_internal.h"

using nmri::fail;

namespace nmri {

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

namespace {

// Consecutive arrays of one allocation, each on its own 256 bytes.
struct Carver {
    char* base;
    size_t used = 0;
    template <typename T>
    void take(T** p, size_t count)
    {
        *p = base && count ? reinterpret_cast<T*>(base + used) : nullptr;
        used += (count * sizeof(T) + 255) / 256 * 256;
    }
};

} // namespace

void pores_free(PoreList* L, int64_t* bytes)
{
    if (L->mem) (void)hipFree(L->mem);
    *bytes -= (int64_t)L->mem_bytes;
    for (float* p : L->pv)
        if (p) {
            (void)hipFree(p);
            *bytes -= (int64_t)((L->cap + 64) * sizeof(float));
        }
    *L = PoreList{};
}

int pores_alloc(PoreList* L, uint32_t nslots, const PoreNeeds& n, hipStream_t s, int64_t* bytes)
{
    const size_t all = (size_t)nslots + 64; // a spare group past the end: the last slot reads the one after it
    auto carve = [&](char* base) {
        Carver c{base};
        c.take(&L->groups, all / 64);
        c.take(&L->aux, n.aux ? all / 64 : 0);
        c.take(&L->off8, all);
        c.take(&L->off16, all);
        c.take(&L->xoff, n.xoff ? all : 0);
        c.take(&L->xy, n.nc == 3 ? all : 0);
        for (float*& f : L->state) c.take(&f, all * n.nc);
        c.take(&L->pred, n.pred ? all * n.nc : 0);
        c.take(&L->rec, n.vel ? all : 0);
        c.take(&L->bcount, (size_t)n.boxes * 8);
        // (a block's first load is a whole workgroup's)
        c.take(&L->blocks, n.boxes ? (size_t)n.block_slots + nmr::kBlockThreads : 0);
        c.take(&L->vox, all); // last: the others are cleared in one go
        return c.used;
    };
    const size_t need = carve(nullptr);
    if (need > L->mem_bytes) {
        if (L->mem) {
            HIP_TRY(hipStreamSynchronize(s));
            HIP_TRY(hipFree(L->mem));
            *bytes -= (int64_t)L->mem_bytes;
            L->mem = nullptr;
            L->mem_bytes = 0;
        }
        HIP_TRY(hipMalloc((void**)&L->mem, need));
        L->mem_bytes = need;
        *bytes += (int64_t)need;
    }
    carve(L->mem);
    HIP_TRY(hipMemsetAsync(L->mem, 0, (size_t)(reinterpret_cast<char*>(L->vox) - L->mem), s));
    HIP_TRY(hipMemsetAsync(L->vox, 0xff, all * sizeof(*L->vox), s));
    if (nslots > L->cap) { // the per-voxel arrays have become too small
        for (float*& p : L->pv) {
            if (!p) continue;
            HIP_TRY(hipStreamSynchronize(s));
            HIP_TRY(hipFree(p));
            p = nullptr;
            *bytes -= (int64_t)((L->cap + 64) * sizeof(float));
        }
        L->cap = nslots;
    }
    L->nslots = nslots;
    L->wide = false;
    L->nbx = L->nby = L->nbz = 0;
    L->blocks_ok = false;
    return NMR_OK;
}

void pores_drop_temp(nmr::PoreBuild* b)
{
    if (b->temp) (void)hipFree(b->temp);
    b->temp = nullptr;
}

int pores_temp(nmr::PoreBuild* b, size_t rows, size_t planes, size_t voxels, hipStream_t s, void* mem, size_t bytes)
{
    const int boxes = b->nbx * b->nby * b->nbz;
    auto carve = [&](char* base) {
        Carver c{base};
        c.take(&b->rows, rows);
        c.take(&b->slotmap, voxels);
        c.take(&b->bcount, (size_t)boxes * 8);
        // the domain's end and what the kernels found lie side by side, for one copy
        c.take(&b->planes, planes + 1 + sizeof(PoreFound) / sizeof(*b->planes));
        return c.used;
    };
    const size_t need = carve(nullptr);
    b->temp = nullptr;
    if (need > bytes) {
        HIP_TRY(hipMalloc(&b->temp, need));
        mem = b->temp;
    }
    carve(static_cast<char*>(mem));
    b->found = reinterpret_cast<int*>(b->planes + planes + 1);
    const hipError_t e = hipMemsetAsync(b->found, 0, sizeof(PoreFound), s);
    if (e != hipSuccess) pores_drop_temp(b);
    HIP_TRY(e);
    return NMR_OK;
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
    b->rec = L.rec;
    b->blocks = L.blocks;
    b->bcount_to = L.bcount;
    b->count = (int64_t)((end - b->first) / 64);
}

int pores_finish(PoreList* L, const nmr::PoreBuild& b, hipStream_t s, PoreFound* found)
{
    HIP_TRY(hipMemcpyAsync(found, b.found, sizeof(*found), hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    L->wide = found->wide != 0;
    L->nbx = b.nbx;
    L->nby = b.nby;
    L->nbz = b.nbz;
    L->blocks_ok = !found->overflow && b.blocks;
    return NMR_OK;
}

void pores_boxes(nmr::PoreBuild* b)
{
    // up to two boxes a CU: past one a CU they run in turns.  us a step, blocks
    // against single steps, at 1 component / 2 with velocity / 3 / 3 with
    // velocity: 20^3 (27 boxes) 1.4 1.7 1.9 2.0 against 3.7 3.7 3.7 3.9; 48^3
    // (216) 1.4 1.8 2.2 2.4 against 3.7 3.9 3.8 4.0; 64^3 (512) 2.2 2.9 3.6 3.9
    // against 4.0 4.0 4.0 4.2; 80^3 (1000) 3.7 5.3 6.5 7.2 against 3.8 4.3 4.4
    // 4.5.  With the porosity a thread's slots grow from one to three: 64^3, 0.3 /
    // 0.6 / 1: one component 2.2 / 2.4 / 2.6 against 3.6 / 3.6 / 3.7, two with
    // velocity 2.9 / 3.4 / 4.0 against 3.7 / 4.0 / 4.4, three 3.7 / 4.4 / 5.3
    // against 4.1 / 4.4 / 4.9: the same or behind only for three with velocity
    // at 0.6 and more.
    constexpr uint64_t kMost = 512;
    constexpr int e = nmr::kBlockEdge;
    const uint64_t nx = (b->nx + e - 1) / e, ny = (b->ny + e - 1) / e, nz = (b->nz + e - 1) / e;
    if (nx * ny * nz > kMost) return;
    b->nbx = (int)nx;
    b->nby = (int)ny;
    b->nbz = (int)nz;
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
