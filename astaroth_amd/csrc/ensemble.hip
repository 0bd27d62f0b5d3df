// Batched ensembles: many independent periodic boxes of uneven sizes advanced together.
//
// There is no counterpart in the reference, which runs one box per Device; this is the batching
// pattern of the single-device path. Each box keeps the reference's layout (8 `in` and 8 `out`
// fields of m_x m_y m_z cells, x fastest) and its own AcMeshInfo (grid spacing, viscosity, ...).
// One RK3 substep is
//   * one periodic-fill launch over the ghost shells of all boxes (a flat list of ghost cells),
//   * one persistent solve launch (solve_ring_batch) over a (box, tile column, z range) work
//     list, dealt out beforehand: the items by decreasing cost, each to the resident block with
//     the least work so far,
// and a step ends with per-box FP64 diagnostics (max and sum of squares of |u| and |A|, max, min
// and sum of squares of lnrho) in two launches. acEnsembleIntegrateStepGraph records the whole
// step once per (dt, buffer parity) into a HIP graph and replays it.
#include "ghost.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <queue>
#include <vector>

using namespace ac;

namespace {

constexpr int NDIAG     = 7;  // per-box diagnostics, see acEnsembleDiagnostics
constexpr int DIAG_CELLS  = 16384; // interior cells per block of the diagnostics launch
constexpr int DIAG_UNROLL = 4;     // cells per lane whose loads are in flight together
constexpr int FILL_BLOCK  = 256; // threads per block of the batched fill

// The field pointers of a box come from a device array, so the compiler cannot tell their
// address space and would use flat loads and stores; they are global memory.
typedef __attribute__((address_space(1))) AcReal GlobalReal;
__device__ __forceinline__ GlobalReal*
global(AcReal* p)
{
    return (GlobalReal*)p;
}
__device__ __forceinline__ const GlobalReal*
global(const AcReal* p)
{
    return (const GlobalReal*)p;
}

struct FillBox {
    AcReal* f[NF];
    GhostShell g;
    long first; // thread index of the box's first ghost cell, a multiple of FILL_BLOCK
};

// Each box's ghost cells start on a block boundary, so a block serves one box and finds it with
// a search keyed by its block index alone (uniform, scalar loads).
__global__ void __launch_bounds__(FILL_BLOCK)
periodic_fill_batch(const FillBox* __restrict__ boxes, const int nboxes)
{
    const long t0 = (long)blockIdx.x * FILL_BLOCK;
    int lo = 0, hi = nboxes - 1; // last box whose first cell is <= t0
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (boxes[mid].first <= t0)
            lo = mid;
        else
            hi = mid - 1;
    }
    const FillBox& b = boxes[lo];
    const long u     = t0 - b.first + threadIdx.x;
    if (u >= b.g.cells()) // the padding up to the next box's first block
        return;
    int i, j, k;
    b.g.cell((unsigned)u, i, j, k);
    long dst, src;
    b.g.indices(i, j, k, dst, src);
    // all eight loads in flight before the first store (the field pointers may alias as far as
    // the compiler knows, which would otherwise make each load wait for the store before it)
    AcReal v[NF];
#pragma unroll
    for (int q = 0; q < NF; ++q)
        v[q] = global(b.f[q])[src];
#pragma unroll
    for (int q = 0; q < NF; ++q)
        global(b.f[q])[dst] = v[q];
}

struct DiagBox {
    const AcReal* f[NF];
    int nx, ny, nz, mx;
    long mxy;
    int first_blk; // the box's first block of the diagnostics launch (ceil(cells / DIAG_CELLS) each)
};

__device__ __forceinline__ double
dmax(double a, double b)
{
    return a > b ? a : b;
}
__device__ __forceinline__ double
dmin(double a, double b)
{
    return a < b ? a : b;
}

// Quantity q of the diagnostics: 0 max |u|^2, 1 sum |u|^2, 2 max |A|^2, 3 sum |A|^2,
// 4 max lnrho, 5 min lnrho, 6 sum lnrho^2 (square roots taken when finalising).
__device__ __forceinline__ bool
is_max(int q)
{
    return q == 0 || q == 2 || q == 4;
}

// Every block takes DIAG_CELLS cells of one box's interior, walked as one flat list (x fastest,
// rows back to back), so that short rows leave no lane idle and every block does the same work
// whatever the box's size; the block finds its box by a search keyed by its index alone
// (uniform). Each lane has the loads of DIAG_UNROLL cells in flight before it accumulates them.
__global__ void __launch_bounds__(256)
diagnostics_batch(const DiagBox* __restrict__ boxes, const int nboxes, double* __restrict__ partials)
{
    __shared__ double lds[4][NDIAG];
    int lo = 0, hi = nboxes - 1; // last box whose first block is <= blockIdx.x
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (boxes[mid].first_blk <= (int)blockIdx.x)
            lo = mid;
        else
            hi = mid - 1;
    }
    const DiagBox& b = boxes[lo];
    double v[NDIAG]  = {0.0, 0.0, 0.0, 0.0, -INFINITY, INFINITY, 0.0};
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned nx = (unsigned)b.nx, nxy = (unsigned)b.nx * (unsigned)b.ny;
    const unsigned cbeg   = (blockIdx.x - (unsigned)b.first_blk) * (unsigned)DIAG_CELLS;
    const unsigned ncell  = min(nxy * (unsigned)b.nz, cbeg + (unsigned)DIAG_CELLS);
    const unsigned stride = 256u;
    for (unsigned c0 = cbeg + threadIdx.x; c0 < ncell; c0 += DIAG_UNROLL * stride) {
        AcReal f[DIAG_UNROLL][7];
        bool ok[DIAG_UNROLL];
#pragma unroll
        for (int uu = 0; uu < DIAG_UNROLL; ++uu) {
            const unsigned c = c0 + uu * stride;
            ok[uu]           = c < ncell;
            const unsigned k = (ok[uu] ? c : 0u) / nxy, rem = (ok[uu] ? c : 0u) - k * nxy;
            const unsigned j = rem / nx, i = rem - j * nx;
            const long m = (long)(i + 3) + (long)(j + 3) * b.mx + (long)(k + 3) * b.mxy;
            f[uu][0] = global(b.f[VTXBUF_UUX])[m];
            f[uu][1] = global(b.f[VTXBUF_UUY])[m];
            f[uu][2] = global(b.f[VTXBUF_UUZ])[m];
            f[uu][3] = global(b.f[VTXBUF_AX])[m];
            f[uu][4] = global(b.f[VTXBUF_AY])[m];
            f[uu][5] = global(b.f[VTXBUF_AZ])[m];
            f[uu][6] = global(b.f[VTXBUF_LNRHO])[m];
        }
#pragma unroll
        for (int uu = 0; uu < DIAG_UNROLL; ++uu) {
            if (!ok[uu])
                continue;
            const double ux = f[uu][0], uy = f[uu][1], uz = f[uu][2];
            const double ax = f[uu][3], ay = f[uu][4], az = f[uu][5], lr = f[uu][6];
            const double u2 = ux * ux + uy * uy + uz * uz, a2 = ax * ax + ay * ay + az * az;
            v[0] = dmax(v[0], u2);
            v[1] += u2;
            v[2] = dmax(v[2], a2);
            v[3] += a2;
            v[4] = dmax(v[4], lr);
            v[5] = dmin(v[5], lr);
            v[6] += lr * lr;
        }
    }
#pragma unroll
    for (int q = 0; q < NDIAG; ++q) {
        double x = v[q];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const double y = __shfl_xor(x, off, 64);
            x              = q == 5 ? dmin(x, y) : is_max(q) ? dmax(x, y) : x + y;
        }
        if (lane == 0)
            lds[wave][q] = x;
    }
    __syncthreads();
    if (threadIdx.x < NDIAG) {
        const int q = threadIdx.x;
        double x    = lds[0][q];
        for (int w = 1; w < 4; ++w)
            x = q == 5 ? dmin(x, lds[w][q]) : is_max(q) ? dmax(x, lds[w][q]) : x + lds[w][q];
        partials[(long)blockIdx.x * NDIAG + q] = x;
    }
}

// Per box and quantity, the box's block partials folded in block order.
__global__ void
diagnostics_finalize(const double* __restrict__ partials, const DiagBox* __restrict__ boxes,
                     const int nboxes, const int nblk, double* __restrict__ results)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nboxes * NDIAG)
        return;
    const int box = t / NDIAG, q = t % NDIAG;
    const int b0 = boxes[box].first_blk, b1 = box + 1 < nboxes ? boxes[box + 1].first_blk : nblk;
    double x = partials[(long)b0 * NDIAG + q];
    for (int i = b0 + 1; i < b1; ++i) {
        const double y = partials[(long)i * NDIAG + q];
        x              = q == 5 ? dmin(x, y) : is_max(q) ? dmax(x, y) : x + y;
    }
    results[t] = x;
}

} // namespace

struct ensemble_s {
    int id;
    int nboxes;
    std::vector<AcMeshInfo> info;
    std::vector<AcReal*> fields[2][NF]; // [set][field][box]; set 0/1 = in/out at parity 0
    AcReal* base;
    size_t base_bytes;
    hipStream_t stream;
    int parity; // number of swaps mod 2: set `parity` holds the current state
    // batched solve: one tile shape per launch, 64 x 8 for 512-thread blocks (see wide_tiling); the
    // z-depth of a box's work items is that of its size class (its column length n_z) when the ensemble
    // chose it, else z_depth (0: whole columns)
    int tile_x, tile_y, z_depth, nblocks;
    std::map<int, int> class_depth;
    BatchItem* d_items;
    int nitems;
    SubstepArgs* d_args[3][2]; // per (substep, parity), for dt_args
    AcReal dt_args;
    bool args_valid;
    // batched fill and diagnostics, per parity
    FillBox* d_fill[2];
    long fill_total;
    DiagBox* d_diag[2];
    int diag_blocks; // blocks of the diagnostics launch, DIAG_CELLS interior cells each
    double* d_partials;
    double* d_results;
    double* h_results; // pinned
    std::map<unsigned long long, hipGraphExec_t> graphs[2];
};

namespace {

int3
dims_of(const AcMeshInfo& i)
{
    return make_int3(i.int_params[AC_nx], i.int_params[AC_ny], i.int_params[AC_nz]);
}

size_t
cells_of(const AcMeshInfo& i)
{
    const int3 n = dims_of(i);
    return (size_t)(n.x + 6) * (n.y + 6) * (n.z + 6);
}

bool
ens_ok(const Ensemble e, int box)
{
    return e && box >= 0 && box < e->nboxes;
}

void
drop_graphs(Ensemble e)
{
    for (int p = 0; p < 2; ++p) {
        for (auto& kv : e->graphs[p])
            (void)hipGraphExecDestroy(kv.second);
        e->graphs[p].clear();
    }
}

// Output planes per work item of a box whose columns are nz planes long.
int
box_depth(const Ensemble e, int nz)
{
    const auto it = e->class_depth.find(nz);
    const int zd  = it != e->class_depth.end() ? it->second : e->z_depth;
    return (zd <= 0 || zd >= nz) ? nz : zd;
}

// Planes a work item costs besides its outputs: it stages six planes and scatters three of them.
constexpr int PROLOGUE = 3;

// Tiles of one box for a launch: their shape, and the time of a plane of one relative to the others.
struct Tiling {
    int tx, ty, tall, weight;
};

int
tiles(int n, int t)
{
    return (n + t - 1) / t;
}

// Cost of a plane of the box in whole tiles.
long
plane_cost(const Tiling& t, int3 n)
{
    return (long)tiles(n.x, t.tx) * tiles(n.y, t.ty) * t.weight;
}

// 512-thread blocks (FP32) take 64 x 8 tiles, or 32 x 16 ones in a box where those cover enough
// fewer cells beyond it. A plane of either, and two of 16 x 16 (as many cells), take 81, 92 and 98:
// 32 boxes of 64^3 0.82 ms per step in 64 x 8 tiles and 0.92 in 16 x 16 (0.11 of it fill and
// diagnostics), 8 of 128^3 1.64 and 1.72; 16 of 96^3, of which 64 x 8 tiles cover 128, 1.58 in 32 x 16
// and 1.76 in 16 x 16. The wide tiles read fewer halo cells and fewer parts of cache lines, which is
// what bounds a full chip here.
Tiling
wide_tiling(int3 n)
{
    const Tiling flat{64, 8, 0, 81}, tall{32, 16, 1, 92};
    return plane_cost(flat, n) <= plane_cost(tall, n) ? flat : tall;
}

// Tiles of one shape in every box. A plane of a 16 x 8 or 32 x 4 tile, half of the blocks' threads, takes
// 27 and 26 in FP32 (32 boxes of 64^3 in 16 x 8 tiles 1.02 ms per step, in 32 x 4 ones 1.04) and 62 in
// FP64, where 16 x 16 takes 100 (1.61 / 1.98 / 1.99 ms).
Tiling
narrow_tiling(int tx, int ty)
{
    const int weight = tx * ty == 256 ? (AC_DOUBLE_PRECISION ? 100 : 49) : AC_DOUBLE_PRECISION ? 62 : tx == 16 ? 27 : 26;
    return {tx, ty, 0, weight};
}

// Tile shape of the launch of a configuration. In FP32 a 16 x 16 one runs 512-thread blocks if their
// tiles cost less over the whole ensemble (100 boxes of 48^3, which they cover with a third to spare, take
// 1.43 ms per step in 16 x 16 tiles and 1.52 in 64 x 8).
int2
launch_shape(const Ensemble e, int tile_x, int tile_y)
{
    if (!AC_DOUBLE_PRECISION && tile_x == 16 && tile_y == 16) {
        long wide = 0, narrow = 0;
        for (const AcMeshInfo& i : e->info) {
            const int3 n = dims_of(i);
            wide += plane_cost(wide_tiling(n), n) * n.z;
            narrow += plane_cost(narrow_tiling(16, 16), n) * n.z;
        }
        if (wide < narrow)
            return make_int2(64, 8);
    }
    return make_int2(tile_x, tile_y);
}

Tiling
box_tiling(int2 launch, int3 n)
{
    return launch.x == 64 ? wide_tiling(n) : narrow_tiling(launch.x, launch.y);
}

struct Deal {
    std::vector<BatchItem> items; // slot s has items s, s + slots, ..., up to an empty one
    int slots;
    long makespan; // cost of the slot with the most work
};

// Work items at the current tile shape and z-depths, dealt to `slots` blocks: by decreasing cost,
// each to the block with the least work so far (the lowest numbered of equals, which keeps
// neighbouring tile columns in neighbouring slots).
Deal
deal_items(const Ensemble e, int2 launch, int slots)
{
    struct Item {
        BatchItem w;
        long cost;
    };
    std::vector<Item> items;
    for (int b = 0; b < e->nboxes; ++b) {
        const int3 n   = dims_of(e->info[b]);
        const Tiling t = box_tiling(launch, n);
        const int zd   = box_depth(e, n.z);
        for (int zs = 0; zs < n.z; zs += zd)
            for (int ty = 0; ty < tiles(n.y, t.ty); ++ty)
                for (int tx = 0; tx < tiles(n.x, t.tx); ++tx)
                    items.push_back({{b, tx, ty, NGHOST + zs, zd, t.tall},
                                     (long)(PROLOGUE + std::min(zd, n.z - zs)) * t.weight});
    }
    std::stable_sort(items.begin(), items.end(),
                     [](const Item& a, const Item& b) { return a.cost > b.cost; });
    Deal d;
    d.slots    = (int)std::min<size_t>(slots, items.size());
    d.makespan = 0;
    typedef std::pair<long, int> Load; // work so far, slot
    std::priority_queue<Load, std::vector<Load>, std::greater<Load>> least;
    for (int s = 0; s < d.slots; ++s)
        least.push({0, s});
    std::vector<int> rounds(d.slots, 0);
    const BatchItem none{-1, 0, 0, 0, 0, 0};
    for (const Item& i : items) {
        const Load l = least.top();
        least.pop();
        const size_t at = (size_t)rounds[l.second]++ * d.slots + l.second;
        if (at >= d.items.size())
            d.items.resize((at / d.slots + 1) * d.slots, none);
        d.items[at] = i.w;
        d.makespan  = std::max(d.makespan, l.first + i.cost);
        least.push({l.first + i.cost, l.second});
    }
    return d;
}

AcResult
build_items(Ensemble e)
{
    AC_HIP_CHECK(hipSetDevice(e->id));
    const int2 launch = make_int2(e->tile_x, e->tile_y);
    // the persistent grid: one block per resident block slot of the batched kernel
    const int slots = batch_resident_blocks(launch.x, launch.y);
    if (slots < 1)
        return AC_FAILURE;
    const Deal d = deal_items(e, launch, slots);
    if (d.items.size() > 0x7fffffffUL)
        return AC_FAILURE;
    if (e->d_items)
        AC_HIP_CHECK(hipFree(e->d_items));
    e->d_items = nullptr;
    AC_HIP_CHECK(hipMalloc((void**)&e->d_items, d.items.size() * sizeof(BatchItem)));
    AC_HIP_CHECK(hipMemcpy(e->d_items, d.items.data(), d.items.size() * sizeof(BatchItem),
                           hipMemcpyHostToDevice));
    e->nitems  = (int)d.items.size();
    e->nblocks = d.slots;
    return AC_SUCCESS;
}

// Every box's columns in equal parts of at most `depth` planes.
std::map<int, int>
equal_parts(const Ensemble e, int depth)
{
    std::map<int, int> d;
    for (const AcMeshInfo& i : e->info) {
        const int nz = dims_of(i).z;
        d[nz]        = tiles(nz, tiles(nz, depth));
    }
    return d;
}

// A configuration of the batched launch, and its expected time (of a plane of all blocks that a CU holds).
struct Candidate {
    int tile_x, tile_y;
    std::map<int, int> class_depth;
    double time;
};

void
apply(Ensemble e, const Candidate& c)
{
    e->tile_x      = c.tile_x;
    e->tile_y      = c.tile_y;
    e->z_depth     = 0;
    e->class_depth = c.class_depth;
}

// The z-depths of a tile shape by decreasing promise: the work of the busiest block after the dealing,
// for columns cut at 2 to 128 planes and whole ones. Fewer, longer items save prologues; more, shorter
// ones fill the chip and leave less of a tail. A depth is not dealt where even an equal share of its work
// takes over MARGIN times `least` or the best so far: the tuner would not time it (with all of them dealt
// seven ensembles of 12 mixed boxes took 79 ms to create, without 47). Leaves the ensemble at the first, where
// there is one.
constexpr double MARGIN = 1.1;

AcResult
rank_depths(Ensemble e, int2 launch, double least, std::vector<Candidate>* ranked)
{
    AC_HIP_CHECK(hipSetDevice(e->id));
    e->tile_x       = launch.x;
    e->tile_y       = launch.y;
    e->z_depth      = 0;
    const int slots = batch_resident_blocks(launch.x, launch.y);
    if (slots < 1)
        return AC_FAILURE;
    int cus = 0;
    AC_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, e->id));
    const double per_cu = (double)slots / cus;
    ranked->clear();
    std::map<int, int> last;
    for (const int depth : {1 << 30, 128, 96, 64, 48, 32, 24, 16, 12, 8, 6, 4, 2}) {
        const std::map<int, int> cut = equal_parts(e, depth);
        if (cut == last)
            continue;
        last        = cut;
        double even = 0;
        for (const AcMeshInfo& i : e->info) {
            const int3 n = dims_of(i);
            even += (double)plane_cost(box_tiling(launch, n), n) * (PROLOGUE * tiles(n.z, cut.at(n.z)) + n.z) / cus;
        }
        if (even > MARGIN * least)
            continue;
        e->class_depth = cut;
        const Deal d   = deal_items(e, launch, slots);
        ranked->push_back({launch.x, launch.y, cut, d.makespan * per_cu});
        least = std::min(least, d.makespan * per_cu);
        if (d.items.size() > 32 * (size_t)slots)
            break; // shorter items only cost more
    }
    if (ranked->empty())
        return AC_SUCCESS;
    std::stable_sort(ranked->begin(), ranked->end(), [](const Candidate& a, const Candidate& b) { return a.time < b.time; });
    apply(e, ranked->front());
    return AC_SUCCESS;
}

AcResult
build_args(Ensemble e, AcReal dt)
{
    drop_graphs(e); // recorded graphs read these argument arrays
    AC_HIP_CHECK(hipStreamSynchronize(e->stream));
    // (a plain array: std::vector cannot relocate a struct of __restrict__ pointer arrays)
    std::unique_ptr<SubstepArgs[]> a(new SubstepArgs[e->nboxes]);
    for (int s = 0; s < 3; ++s)
        for (int par = 0; par < 2; ++par) {
            // substep s at buffer parity `par` reads set `par` and writes the other set
            for (int b = 0; b < e->nboxes; ++b) {
                const int3 n    = dims_of(e->info[b]);
                SubstepArgs& x  = a[b];
                for (int q = 0; q < NF; ++q) {
                    x.in[q]   = e->fields[par][q][b];
                    x.out[q]  = e->fields[1 - par][q][b];
                    x.cin[q]  = nullptr;
                    x.cout[q] = nullptr;
                }
                x.mx    = n.x + 6;
                x.my    = n.y + 6;
                x.mz    = n.z + 6;
                x.mxy    = x.mx * x.my;
                x.stride = x.in[1] - x.in[0];
                x.start = make_int3(NGHOST, NGHOST, NGHOST);
                x.end   = make_int3(n.x + NGHOST, n.y + NGHOST, n.z + NGHOST);
                x.wrap  = 1;
                x.phys  = make_phys_params(e->info[b]);
                x.rk    = make_rk3_coeffs(s, dt);
            }
            AC_HIP_CHECK(hipMemcpy(e->d_args[s][par], a.get(), e->nboxes * sizeof(SubstepArgs),
                                   hipMemcpyHostToDevice));
        }
    e->dt_args    = dt;
    e->args_valid = true;
    return AC_SUCCESS;
}

AcResult
ensure_args(Ensemble e, AcReal dt)
{
    if (e->args_valid && e->dt_args == dt)
        return AC_SUCCESS;
    return build_args(e, dt);
}

hipError_t
enqueue_fill(Ensemble e, int par)
{
    if (e->fill_total == 0)
        return hipSuccess;
    const long blocks = e->fill_total / FILL_BLOCK;
    if (blocks > 0x7fffffffL)
        return hipErrorInvalidConfiguration;
    periodic_fill_batch<<<dim3((unsigned)blocks), dim3(FILL_BLOCK), 0, e->stream>>>(e->d_fill[par],
                                                                                    e->nboxes);
    return hipGetLastError();
}

hipError_t
enqueue_diagnostics(Ensemble e, int par)
{
    diagnostics_batch<<<dim3((unsigned)e->diag_blocks), dim3(256), 0, e->stream>>>(
        e->d_diag[par], e->nboxes, e->d_partials);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess)
        return err;
    const int n = e->nboxes * NDIAG;
    diagnostics_finalize<<<dim3((n + 255) / 256), dim3(256), 0, e->stream>>>(
        e->d_partials, e->d_diag[par], e->nboxes, e->diag_blocks, e->d_results);
    return hipGetLastError();
}

// The step at the current parity, enqueued on the ensemble stream (also what a graph records).
AcResult
enqueue_step(Ensemble e, int par0)
{
    // The batched solve reads periodic images instead of ghost cells, so the substeps need no
    // fill; one fill after the last substep leaves every box's ghosts current.
    int par = par0;
    for (int s = 0; s < 3; ++s) {
        AC_HIP_CHECK(launch_substep_batch(e->tile_x, e->tile_y, s, e->d_args[s][par], e->d_items,
                                          e->nitems, e->nblocks, e->stream));
        par = 1 - par;
    }
    AC_HIP_CHECK(enqueue_fill(e, par));
    AC_HIP_CHECK(enqueue_diagnostics(e, par));
    return AC_SUCCESS;
}

bool
valid_dt(AcReal dt)
{
    return std::isfinite((double)dt) && dt > 0;
}

// Time of a step's three launches of the batched solve over the current work list. All read the current
// set and write the other one, which holds no state between steps. The three differ: substep 0 has no
// previous stage to read, and 16 x 16 blocks gain more by that than 512-thread ones (2 boxes of 200^3: substep 1
// 0.59 and 0.60 ms, substep 0 0.46 and 0.56).
float
time_solves(Ensemble e)
{
    hipEvent_t t0, t1;
    AC_HIP_CHECK(hipEventCreate(&t0));
    AC_HIP_CHECK(hipEventCreate(&t1));
    AC_HIP_CHECK(hipEventRecord(t0, e->stream));
    for (int s = 0; s < 3; ++s)
        AC_HIP_CHECK(launch_substep_batch(e->tile_x, e->tile_y, s, e->d_args[s][e->parity], e->d_items,
                                          e->nitems, e->nblocks, e->stream));
    AC_HIP_CHECK(hipEventRecord(t1, e->stream));
    AC_HIP_CHECK(hipEventSynchronize(t1));
    float ms = 0;
    AC_HIP_CHECK(hipEventElapsedTime(&ms, t0, t1));
    AC_HIP_CHECK(hipEventDestroy(t0));
    AC_HIP_CHECK(hipEventDestroy(t1));
    return ms;
}

// Tuned choices per ensemble composition (device, box sizes in order), kept for the process.
std::map<std::vector<int>, Candidate>&
tuning_cache()
{
    static std::map<std::vector<int>, Candidate> cache;
    return cache;
}

std::mutex&
tuning_mutex()
{
    static std::mutex m;
    return m;
}

} // namespace

extern "C" {

AcResult
acEnsembleCreate(const int device_id, const int nboxes, const AcMeshInfo* configs,
                 Ensemble* ensemble)
{
    if (!ensemble || !configs || nboxes < 1)
        return AC_FAILURE;
    *ensemble = nullptr;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || device_id < 0 || device_id >= count) {
        fprintf(stderr, "acEnsembleCreate: no HIP device %d\n", device_id);
        return AC_FAILURE;
    }
    for (int b = 0; b < nboxes; ++b) {
        const int3 n = dims_of(configs[b]);
        // The batched solve reads the periodic images of the ghost cells instead of filled
        // ghosts; an image lies in the interior only if every axis holds NGHOST cells or more.
        if (n.x < NGHOST || n.y < NGHOST || n.z < NGHOST) {
            fprintf(stderr, "acEnsembleCreate: box %d is %d x %d x %d; every axis needs at least %d cells\n",
                    b, n.x, n.y, n.z, NGHOST);
            return AC_FAILURE;
        }
    }
    AC_HIP_CHECK(hipSetDevice(device_id));
    Ensemble e   = new ensemble_s();
    e->id        = device_id;
    e->nboxes    = nboxes;
    e->info.assign(configs, configs + nboxes);
    for (auto& i : e->info)
        acHostUpdateBuiltinParams(&i);
    e->parity   = 0;
    e->tile_x   = 16; // (and chosen below)
    e->tile_y   = 16;
    e->z_depth  = 0;
    e->d_items  = nullptr;
    e->args_valid = false;
    e->dt_args  = 0;
    // one allocation: box after box, 16 fields each (8 per set), 256-byte aligned
    size_t bytes = 0;
    std::vector<size_t> offs(nboxes);
    for (int b = 0; b < nboxes; ++b) {
        offs[b] = bytes;
        const size_t fb = (cells_of(e->info[b]) * sizeof(AcReal) + 255) / 256 * 256;
        bytes += 2 * NF * fb;
    }
    e->base_bytes = bytes;
    AC_HIP_CHECK(hipMalloc((void**)&e->base, bytes));
    AC_HIP_CHECK(hipMemset(e->base, 0, bytes));
    for (int set = 0; set < 2; ++set)
        for (int q = 0; q < NF; ++q)
            e->fields[set][q].resize(nboxes);
    for (int b = 0; b < nboxes; ++b) {
        const size_t fb = (cells_of(e->info[b]) * sizeof(AcReal) + 255) / 256 * 256;
        for (int set = 0; set < 2; ++set)
            for (int q = 0; q < NF; ++q)
                e->fields[set][q][b] = (AcReal*)((char*)e->base + offs[b] + (set * NF + q) * fb);
    }
    AC_HIP_CHECK(hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking));
    for (int s = 0; s < 3; ++s)
        for (int p = 0; p < 2; ++p)
            AC_HIP_CHECK(hipMalloc((void**)&e->d_args[s][p], nboxes * sizeof(SubstepArgs)));
    // fill and diagnostics descriptors per parity
    std::vector<FillBox> fb(nboxes);
    std::vector<DiagBox> db(nboxes);
    int diag_blocks = 0;
    for (int p = 0; p < 2; ++p) {
        AC_HIP_CHECK(hipMalloc((void**)&e->d_fill[p], nboxes * sizeof(FillBox)));
        AC_HIP_CHECK(hipMalloc((void**)&e->d_diag[p], nboxes * sizeof(DiagBox)));
        long first  = 0;
        diag_blocks = 0; // the same for both parities
        for (int b = 0; b < nboxes; ++b) {
            const int3 n = dims_of(e->info[b]);
            for (int q = 0; q < NF; ++q) {
                fb[b].f[q] = e->fields[p][q][b];
                db[b].f[q] = e->fields[p][q][b];
            }
            fb[b].g     = GhostShell::of(n.x, n.y, n.z);
            if (!fb[b].g.fits_32bit()) {
                fprintf(stderr, "acEnsembleCreate: box %d is too large for the batched fill\n", b);
                return AC_FAILURE;
            }
            if ((long)n.x * n.y * n.z >= (1L << 31)) { // the diagnostics' 32-bit cell index
                fprintf(stderr, "acEnsembleCreate: box %d is too large for the batched diagnostics\n", b);
                return AC_FAILURE;
            }
            fb[b].first = first;
            first += (fb[b].g.cells() + FILL_BLOCK - 1) / FILL_BLOCK * FILL_BLOCK;
            db[b].nx  = n.x;
            db[b].ny  = n.y;
            db[b].nz  = n.z;
            db[b].mx  = n.x + 6;
            db[b].mxy = (long)(n.x + 6) * (n.y + 6);
            db[b].first_blk = diag_blocks;
            diag_blocks += (int)(((long)n.x * n.y * n.z + DIAG_CELLS - 1) / DIAG_CELLS);
        }
        e->fill_total = first;
        AC_HIP_CHECK(hipMemcpy(e->d_fill[p], fb.data(), nboxes * sizeof(FillBox),
                               hipMemcpyHostToDevice));
        AC_HIP_CHECK(hipMemcpy(e->d_diag[p], db.data(), nboxes * sizeof(DiagBox),
                               hipMemcpyHostToDevice));
    }
    e->diag_blocks = diag_blocks;
    AC_HIP_CHECK(hipMalloc((void**)&e->d_partials, (size_t)diag_blocks * NDIAG * sizeof(double)));
    AC_HIP_CHECK(hipMalloc((void**)&e->d_results, (size_t)nboxes * NDIAG * sizeof(double)));
    AC_HIP_CHECK(hipMemset(e->d_results, 0, (size_t)nboxes * NDIAG * sizeof(double)));
    AC_HIP_CHECK(hipHostMalloc((void**)&e->h_results, (size_t)nboxes * NDIAG * sizeof(double)));
    // Tile shape and z-depths measured on this composition, as Devices tune at creation; with
    // AC_AUTOTUNE=0 16 x 16 tiles (or the wide ones of launch_shape) at the depths ranked first.
    const char* tune = getenv("AC_AUTOTUNE");
    if (tune && tune[0] == '0') {
        std::vector<Candidate> ranked;
        if (rank_depths(e, launch_shape(e, 16, 16), INFINITY, &ranked) != AC_SUCCESS || build_items(e) != AC_SUCCESS)
            return AC_FAILURE;
    }
    else if (acEnsembleAutoOptimize(e) != AC_SUCCESS)
        return AC_FAILURE;
    AC_HIP_CHECK(hipDeviceSynchronize());
    *ensemble = e;
    return AC_SUCCESS;
}

AcResult
acEnsembleDestroy(Ensemble e)
{
    if (!e)
        return AC_FAILURE;
    AC_HIP_CHECK(hipSetDevice(e->id));
    AC_HIP_CHECK(hipStreamSynchronize(e->stream));
    drop_graphs(e);
    AC_HIP_CHECK(hipFree(e->base));
    for (int s = 0; s < 3; ++s)
        for (int p = 0; p < 2; ++p)
            AC_HIP_CHECK(hipFree(e->d_args[s][p]));
    for (int p = 0; p < 2; ++p) {
        AC_HIP_CHECK(hipFree(e->d_fill[p]));
        AC_HIP_CHECK(hipFree(e->d_diag[p]));
    }
    if (e->d_items)
        AC_HIP_CHECK(hipFree(e->d_items));
    AC_HIP_CHECK(hipFree(e->d_partials));
    AC_HIP_CHECK(hipFree(e->d_results));
    AC_HIP_CHECK(hipHostFree(e->h_results));
    AC_HIP_CHECK(hipStreamDestroy(e->stream));
    delete e;
    return AC_SUCCESS;
}

int
acEnsembleBoxCount(const Ensemble e)
{
    return e ? e->nboxes : 0;
}

AcResult
acEnsembleSetKernelConfig(Ensemble e, const AcKernelConfig config)
{
    if (!e || config.variant != 3 || !batch_tile_supported(config.tile_x, config.tile_y) ||
        config.z_depth < 0)
        return AC_FAILURE;
    AC_HIP_CHECK(hipSetDevice(e->id));
    AC_HIP_CHECK(hipStreamSynchronize(e->stream));
    const int2 launch = launch_shape(e, config.tile_x, config.tile_y);
    e->tile_x         = launch.x;
    e->tile_y         = launch.y;
    e->z_depth        = config.z_depth;
    e->class_depth.clear(); // one z-depth for every box
    drop_graphs(e);
    return build_items(e);
}

AcResult
acEnsembleAutoOptimize(Ensemble e)
{
    if (!e)
        return AC_FAILURE;
    AC_HIP_CHECK(hipSetDevice(e->id));
    AC_HIP_CHECK(hipStreamSynchronize(e->stream));
    drop_graphs(e);
    std::vector<int> key{e->id};
    for (const AcMeshInfo& i : e->info) {
        const int3 n = dims_of(i);
        key.insert(key.end(), {n.x, n.y, n.z});
    }
    {
        std::lock_guard<std::mutex> lock(tuning_mutex());
        const auto it = tuning_cache().find(key);
        if (it != tuning_cache().end()) {
            apply(e, it->second);
            return build_items(e);
        }
    }
    // the timed launches need argument arrays; any dt times the same
    if (!e->args_valid && build_args(e, AcReal(1e-3)) != AC_SUCCESS)
        return AC_FAILURE;
    // Of every tile shape the four most promising depths, unless they are expected to take more than
    // 1.1 times the best: thin boxes fill a tile of one shape and a part of another's (256 boxes of
    // 32 x 4 x 64 in FP32: 0.70 ms per step in 16 x 16 tiles, 0.42 in 16 x 8, 0.33 in 32 x 4). Between
    // shapes the expectation is 10 to 20 % off (500 boxes of 20^3, where 32 x 4 is expected to be 4 %
    // faster than 16 x 8: 0.94 ms against 0.81), but a wider margin times shapes that do not win: 12
    // boxes of 32 to 128 cells an edge took 9 ms longer to create with 1.2.
    std::vector<Candidate> candidates;
    double least = INFINITY;
    // The 512-thread blocks and 16 x 16 ones are both in the choice (FP32; the one that covers the boxes at
    // less cost first): with few boxes the rounds of blocks decide (2 boxes of 200^3 1.95 ms per step in 16 x
    // 16 tiles and 2.07 in 64 x 8, which cover them at 2 % less).
    std::vector<int2> shapes{launch_shape(e, 16, 16)};
    if (!AC_DOUBLE_PRECISION)
        shapes.push_back(shapes[0].x == 64 ? make_int2(16, 16) : make_int2(64, 8));
    shapes.push_back(make_int2(16, 8));
    shapes.push_back(make_int2(32, 4));
    for (const int2 launch : shapes) {
        std::vector<Candidate> ranked;
        if (rank_depths(e, launch, least, &ranked) != AC_SUCCESS)
            return AC_FAILURE;
        if (ranked.empty())
            continue;
        least = std::min(least, ranked.front().time);
        candidates.insert(candidates.end(), ranked.begin(), ranked.begin() + std::min<size_t>(ranked.size(), 4));
    }
    candidates.erase(std::remove_if(candidates.begin(), candidates.end(),
                                    [=](const Candidate& c) { return c.time > MARGIN * least; }),
                     candidates.end());
    float best  = INFINITY;
    size_t keep = 0;
    for (int round = 0; round < 3; ++round) // the clocks still rise during the first
        for (size_t i = 0; i < candidates.size(); ++i) {
            apply(e, candidates[i]);
            if (build_items(e) != AC_SUCCESS)
                return AC_FAILURE;
            const float ms   = time_solves(e);
            const bool other = candidates[i].tile_x != candidates[keep].tile_x || candidates[i].tile_y != candidates[keep].tile_y;
            if (round > 0 && ms < (other ? 0.98f : 1.f) * best) { // (the timings scatter by 1 to 2 %)
                best = ms;
                keep = i;
            }
        }
    apply(e, candidates[keep]);
    if (build_items(e) != AC_SUCCESS)
        return AC_FAILURE;
    std::lock_guard<std::mutex> lock(tuning_mutex());
    tuning_cache()[key] = candidates[keep];
    return AC_SUCCESS;
}

int
acEnsembleBoxZDepth(const Ensemble e, const int box)
{
    if (!ens_ok(e, box))
        return -1;
    const int nz = dims_of(e->info[box]).z;
    const int zd = box_depth(e, nz);
    return zd >= nz ? 0 : zd;
}

AcResult
acEnsembleGetKernelConfig(const Ensemble e, AcKernelConfig* config)
{
    if (!e || !config)
        return AC_FAILURE;
    config->variant = 3;
    const bool wide = e->tile_x == 64; // not a configuration of its own: 16 x 16 stands for it
    config->tile_x  = wide ? 16 : e->tile_x;
    config->tile_y  = wide ? 16 : e->tile_y;
    config->z_depth = e->z_depth;
    return AC_SUCCESS;
}

AcResult
acEnsembleRandomizeUniform(Ensemble e, const int box, const VertexBufferHandle handle,
                           const double lo, const double hi, const unsigned long long seed)
{
    if (!ens_ok(e, box) || handle < 0 || handle >= NF)
        return AC_FAILURE;
    AC_HIP_CHECK(hipSetDevice(e->id));
    AC_HIP_CHECK(launch_fill_uniform(e->fields[e->parity][handle][box], e->info[box], lo, hi,
                                     seed, e->stream));
    return AC_SUCCESS;
}

AcResult
acEnsembleSetVertexBuffer(Ensemble e, const int box, const VertexBufferHandle handle,
                          const AcReal value)
{
    if (!ens_ok(e, box) || handle < 0 || handle >= NF || !std::isfinite((double)value))
        return AC_FAILURE;
    AC_HIP_CHECK(hipSetDevice(e->id));
    const long n = (long)cells_of(e->info[box]);
    for (int set = 0; set < 2; ++set)
        AC_HIP_CHECK(launch_fill_constant(e->fields[set][handle][box], n, value, e->stream));
    return AC_SUCCESS;
}

AcResult
acEnsembleLoadMesh(Ensemble e, const int box, const AcMesh host)
{
    if (!ens_ok(e, box))
        return AC_FAILURE;
    const int3 n = dims_of(host.info);
    if (n.x != dims_of(e->info[box]).x || n.y != dims_of(e->info[box]).y ||
        n.z != dims_of(e->info[box]).z)
        return AC_FAILURE;
    AC_HIP_CHECK(hipSetDevice(e->id));
    const size_t bytes = cells_of(e->info[box]) * sizeof(AcReal);
    for (int q = 0; q < NF; ++q)
        AC_HIP_CHECK(hipMemcpyAsync(e->fields[e->parity][q][box], host.vertex_buffer[q], bytes,
                                    hipMemcpyHostToDevice, e->stream));
    AC_HIP_CHECK(hipStreamSynchronize(e->stream));
    return AC_SUCCESS;
}

AcResult
acEnsembleStoreMesh(Ensemble e, const int box, AcMesh* host)
{
    if (!ens_ok(e, box) || !host)
        return AC_FAILURE;
    const int3 n = dims_of(host->info);
    if (n.x != dims_of(e->info[box]).x || n.y != dims_of(e->info[box]).y ||
        n.z != dims_of(e->info[box]).z)
        return AC_FAILURE;
    AC_HIP_CHECK(hipSetDevice(e->id));
    const size_t bytes = cells_of(e->info[box]) * sizeof(AcReal);
    for (int q = 0; q < NF; ++q)
        AC_HIP_CHECK(hipMemcpyAsync(host->vertex_buffer[q], e->fields[e->parity][q][box], bytes,
                                    hipMemcpyDeviceToHost, e->stream));
    AC_HIP_CHECK(hipStreamSynchronize(e->stream));
    return AC_SUCCESS;
}

AcResult
acEnsemblePeriodicBoundconds(Ensemble e)
{
    if (!e)
        return AC_FAILURE;
    AC_HIP_CHECK(hipSetDevice(e->id));
    AC_HIP_CHECK(enqueue_fill(e, e->parity));
    return AC_SUCCESS;
}

AcResult
acEnsembleIntegrateStep(Ensemble e, const AcReal dt)
{
    if (!e || !valid_dt(dt))
        return AC_FAILURE;
    AC_HIP_CHECK(hipSetDevice(e->id));
    if (ensure_args(e, dt) != AC_SUCCESS || enqueue_step(e, e->parity) != AC_SUCCESS)
        return AC_FAILURE;
    e->parity = 1 - e->parity;
    return AC_SUCCESS;
}

AcResult
acEnsembleIntegrateStepGraph(Ensemble e, const AcReal dt)
{
    if (!e || !valid_dt(dt))
        return AC_FAILURE;
    AC_HIP_CHECK(hipSetDevice(e->id));
    if (ensure_args(e, dt) != AC_SUCCESS) // a new dt rebuilds the arguments and drops the graphs
        return AC_FAILURE;
    unsigned long long key = 0;
    memcpy(&key, &dt, sizeof(dt));
    auto& cache = e->graphs[e->parity];
    auto it     = cache.find(key);
    if (it == cache.end()) {
        AC_HIP_CHECK(hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal));
        const AcResult r = enqueue_step(e, e->parity);
        hipGraph_t graph;
        AC_HIP_CHECK(hipStreamEndCapture(e->stream, &graph));
        if (r != AC_SUCCESS)
            return AC_FAILURE;
        hipGraphExec_t exec;
        AC_HIP_CHECK(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
        AC_HIP_CHECK(hipGraphDestroy(graph));
        it = cache.emplace(key, exec).first;
    }
    AC_HIP_CHECK(hipGraphLaunch(it->second, e->stream));
    e->parity = 1 - e->parity;
    return AC_SUCCESS;
}

AcResult
acEnsembleIntegrateStepLooped(Ensemble e, const AcReal dt)
{
    if (!e || !valid_dt(dt))
        return AC_FAILURE;
    AC_HIP_CHECK(hipSetDevice(e->id));
    int par = e->parity;
    for (int s = 0; s < 3; ++s) {
        for (int b = 0; b < e->nboxes; ++b) {
            const int3 n = dims_of(e->info[b]);
            AcReal* cin[NF];
            AcReal* cout[NF];
            for (int q = 0; q < NF; ++q) {
                cin[q]  = e->fields[par][q][b];
                cout[q] = e->fields[1 - par][q][b];
            }
            // each box as a single-box Device steps it: its default configuration, reading the
            // ghost cells' periodic images where that is the default form, else fill + launch
            const AcKernelConfig cfg = default_kernel_config(n.x, n.y, n.z);
            const bool images        = kernel_config_reads_images(cfg) &&
                                default_reads_images(n.x, n.y, n.z) && n.x >= NGHOST &&
                                n.y >= NGHOST && n.z >= NGHOST;
            const int3 zero = make_int3(0, 0, 0), m = make_int3(n.x + 6, n.y + 6, n.z + 6);
            if (!images)
                AC_HIP_CHECK(launch_periodic_fill(cin, NF, n.x, n.y, n.z, zero, m, e->stream));
            SubstepArgs a;
            for (int q = 0; q < NF; ++q) {
                a.in[q]   = cin[q];
                a.out[q]  = cout[q];
                a.cin[q]  = nullptr;
                a.cout[q] = nullptr;
            }
            a.mx    = n.x + 6;
            a.my    = n.y + 6;
            a.mz    = n.z + 6;
            a.mxy    = a.mx * a.my;
            a.stride = a.in[1] - a.in[0];
            a.start = make_int3(NGHOST, NGHOST, NGHOST);
            a.end   = make_int3(n.x + NGHOST, n.y + NGHOST, n.z + NGHOST);
            a.wrap  = images;
            a.phys  = make_phys_params(e->info[b]);
            a.rk    = make_rk3_coeffs(s, dt);
            AC_HIP_CHECK(launch_substep(cfg, a, e->stream));
        }
        par = 1 - par;
    }
    AC_HIP_CHECK(enqueue_diagnostics(e, par));
    e->parity = par;
    return AC_SUCCESS;
}

AcResult
acEnsembleDiagnostics(Ensemble e, double* results)
{
    if (!e || !results)
        return AC_FAILURE;
    AC_HIP_CHECK(hipSetDevice(e->id));
    const size_t n = (size_t)e->nboxes * NDIAG;
    AC_HIP_CHECK(hipMemcpyAsync(e->h_results, e->d_results, n * sizeof(double),
                                hipMemcpyDeviceToHost, e->stream));
    AC_HIP_CHECK(hipStreamSynchronize(e->stream));
    for (int b = 0; b < e->nboxes; ++b) {
        const int3 nn   = dims_of(e->info[b]);
        const double N  = (double)nn.x * nn.y * nn.z;
        const double* r = e->h_results + (size_t)b * NDIAG;
        double* o       = results + (size_t)b * NDIAG;
        o[0] = std::sqrt(r[0]);     // max |u|
        o[1] = std::sqrt(r[1] / N); // rms |u|
        o[2] = std::sqrt(r[2]);     // max |A|
        o[3] = std::sqrt(r[3] / N); // rms |A|
        o[4] = r[4];                // max lnrho
        o[5] = r[5];                // min lnrho
        o[6] = std::sqrt(r[6] / N); // rms lnrho
    }
    return AC_SUCCESS;
}

AcResult
acEnsembleTimestepCFL(Ensemble e, double* dts)
{
    if (!e || !dts)
        return AC_FAILURE;
    std::vector<double> d((size_t)e->nboxes * NDIAG);
    if (acEnsembleDiagnostics(e, d.data()) != AC_SUCCESS)
        return AC_FAILURE;
    for (int b = 0; b < e->nboxes; ++b)
        dts[b] = cfl_timestep(d[(size_t)b * NDIAG], 0.0, e->info[b]);
    return AC_SUCCESS;
}

AcResult
acEnsembleSynchronize(const Ensemble e)
{
    if (!e)
        return AC_FAILURE;
    AC_HIP_CHECK(hipSetDevice(e->id));
    AC_HIP_CHECK(hipStreamSynchronize(e->stream));
    return AC_SUCCESS;
}

void*
acEnsembleGetStreamHandle(const Ensemble e)
{
    return e ? (void*)e->stream : nullptr;
}

} // extern "C"
