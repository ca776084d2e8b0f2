// batch.hip -- many FD shots on uneven grids, one launch per time step
// (phc_batch_* C ABI).
//
// No reference counterpart: the reference runs one shot per process (its FD
// driver, src/fd/FDTDmain.cpp:9-108).  Each shot here is exactly that FD
// problem -- same setup, same step (FDTDkernels.hpp:8-34, 108-128), same
// sponge -- on its own grid size, source and model.  One launch advances every
// shot by one step: one block per (shot, tile column, plane range) work item,
// dealt to the XCDs by a host-built table, each block marching its item with
// the same tile body as the single-grid kernel (fd_tile).  The run is captured
// in one hipGraph; the autotuner picks block shape and chunk length.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <vector>

#include "fd_kernels.hpp"
#include "fd_quad.hpp"
#include "fd_tile.hpp"
#include "xcd_sched.hpp"
#include "march.hpp"
#include "phc_common.hpp"

namespace phc {

// One shot: its layout and device arrays (inside the batch's pool).
struct ShotDesc {
    FdLayout L;
    float *lev[2];
    const float *vp;  // vp^2 dt^2
    const float *fy, *fz;
    const float *rhs;
    int64_t src_off;
    int krem;         // first k of the shot's remainder slab (0: none)
    int tiles_k;      // k tiles of the shot's tile columns
};

// One block's work, an int4 (shot, w, i0, i1): w >= 0: tile column w (k tile
// w % tiles_k, j tile w / tiles_k) of the shot marched over planes [i0, i1);
// w < 0: part -1 - w of the shot's k-remainder slab, BATCH_SLAB_PASSES x the
// block's threads points in slab order; i0 >= i1: nothing (padding).
constexpr int BATCH_SLAB_PASSES = 4;

// The per-grid fields fd_tile reads, for one work item (scalar registers).
struct FdGrid {
    FdLayout L;
    const float *pn;
    float *pnm1;
    const float *vp, *fy, *fz;
    int64_t src_off;
    int inj;
    float *trace;
    int ilo, ihi, jlo, jhi, klo, khi;  // every point of the shot
    int krem;
    int jrem;  // no j-remainder slab in the batch (0)
};

constexpr int BATCH_XCDS = 8;

// Receivers of the level a launch reads as current (the previous step's
// result), sampled by extra blocks after the others, one receiver per thread.
struct BatchSample {
    const int64_t *off;
    float *out;
    int n, nrec, stride, step;  // n = shots x nrec (0: no sampling blocks)
};

// out[t * stride + step] = the level's value at receiver t.  A receiver on the
// source point reads the value recorded before the fused injection of the
// next step.
__device__ __forceinline__ void batch_sample(const BatchSample &r, const ShotDesc *shots, const float *traces,
                                             int level, int t)
{
    if (t >= r.n) return;
    const int s = t / r.nrec;
    const ShotDesc &d = shots[s];
    const int64_t o = r.off[t];
    r.out[(int64_t)t * r.stride + r.step] =
        (o == d.src_off) ? traces[(int64_t)s * r.stride + r.step] : d.lev[level][o];
}

// One time step of every shot.  `c` holds what the shots share (coefficients,
// sponge table, deferred damping flag).  The hardware deals block b to XCD
// b % 8 and starts an XCD's blocks in order as slots on its CUs free up; the
// table gives each XCD a contiguous run of items in spatial order and of
// about equal cost, so neighbouring tiles that run side by side share their
// halo rows in that XCD's L2.  A block holds one item and several blocks are
// resident per CU, so one block's first loads (9 planes of ring, about 3 us
// with the descriptor reads) run beside the others' marches; resident blocks
// that claimed their items from a queue one after the other left that
// latency and the claim's open: 12 shots of U[96,224]^3, best one-point shape
// of each, 200 us per step against 240 (47.7 M points: 3.8 against 3.2 TB/s;
// 189 with four points per lane, 4.0 TB/s).
//
// fd_batch_item fills the grid of the block's item; false: nothing to march
// (a sampling block, padding, or slab points, which it has updated).
template <int R, int TY, int ARITH, typename IT>
__device__ __forceinline__ bool fd_batch_item(const FdStepArgs &c, const ShotDesc *__restrict__ shots,
                                              const int4 *__restrict__ items, int nitems, int cur, const int *it0,
                                              int inj, float *traces, int trace_stride, int step,
                                              const BatchSample &rec, FdGrid &g, float &rhs_next, int4 &tile)
{
    constexpr int T = FD_TK * TY;
    if ((int)blockIdx.x >= nitems) {
        batch_sample(rec, shots, traces, cur,
                     ((int)blockIdx.x - nitems) * T + (int)(threadIdx.y * FD_TK + threadIdx.x));
        return false;
    }
    const int it = uniform_value(it0) + step;
    const int4 wi = items[blockIdx.x];
    if (wi.z >= wi.w) return false;  // padding of a shorter XCD list (whole block)
    const ShotDesc &sd = shots[wi.x];
    g.L = sd.L;
    g.pn = sd.lev[cur];
    g.pnm1 = sd.lev[1 - cur];
    g.vp = sd.vp;
    g.fy = sd.fy;
    g.fz = sd.fz;
    g.src_off = sd.src_off;
    g.inj = inj;
    rhs_next = uniform_value(inj ? sd.rhs + it + 1 : nullptr);
    g.trace = traces + (int64_t)wi.x * trace_stride + step;
    g.ilo = 0; g.ihi = sd.L.nx;
    g.jlo = 0; g.jhi = sd.L.ny;
    g.klo = 0; g.khi = sd.L.nz;
    g.krem = sd.krem;
    g.jrem = 0;
    if (wi.y < 0) {
        const int64_t part = -1 - wi.y;
        for (int m = 0; m < BATCH_SLAB_PASSES; ++m)
            fd_rem_points<R, ARITH, IT>(c, g, rhs_next, (part * BATCH_SLAB_PASSES + m) * T);
        return false;
    }
    tile = make_int4(wi.y % sd.tiles_k, wi.y / sd.tiles_k, wi.z, wi.w);
    return true;
}

template <int R, int TY, int NJ, int ARITH, typename IT>
__global__ void __launch_bounds__(FD_TK *TY)
fd_batch_kernel(FdStepArgs c, const ShotDesc *__restrict__ shots, const int4 *__restrict__ items, int nitems,
                int cur, const int *it0, int inj, float *traces, int trace_stride, int step, BatchSample rec)
{
    using SH = FdTileShape<R, TY, NJ>;
    __shared__ float tile[2][SH::LH][SH::LW];
    FdGrid g;
    float rhs_next;
    int4 w;
    if (fd_batch_item<R, TY, ARITH, IT>(c, shots, items, nitems, cur, it0, inj, traces, trace_stride, step, rec, g,
                                        rhs_next, w))
        fd_tile<R, TY, NJ, ARITH, IT>(c, g, rhs_next, w.x, w.y, w.z, w.w, tile);
}

// The shapes with 4 rows per wavefront: four points per lane (fd_quad.hpp).
template <int TY, int ARITH, bool NT>
__global__ void __launch_bounds__(FD_TK *TY) __attribute__((amdgpu_waves_per_eu(3)))
fd_batch_quad_kernel(FdStepArgs c, const ShotDesc *__restrict__ shots, const int4 *__restrict__ items, int nitems,
                     int cur, const int *it0, int inj, float *traces, int trace_stride, int step, BatchSample rec)
{
    using SH = FdQuadShape<TY>;
    __shared__ quad_f4 tile[2][SH::LH][SH::LQ];
    FdGrid g;
    float rhs_next;
    int4 w;
    if (fd_batch_item<4, TY, ARITH, uint32_t>(c, shots, items, nitems, cur, it0, inj, traces, trace_stride, step,
                                              rec, g, rhs_next, w))
        fd_quad<TY, ARITH, uint32_t, false, NT>(c, g, rhs_next, w.x, w.y, w.z, w.w, tile);
}

// Start of a run at sample it: rhs[it] into every shot's current level at its
// source (FDTDkernels.hpp:121-128), and it where the run's steps read it.
__global__ void fd_batch_inject_kernel(const ShotDesc *shots, int nshots, int cur, int it, int *it0)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s == 0) *it0 = it;
    if (s >= nshots) return;
    const ShotDesc &d = shots[s];
    float *p = d.lev[cur];
    p[d.src_off] = add_nc(p[d.src_off], mul_nc(d.vp[d.src_off], d.rhs[it]));
}

// Receivers of the last step of a run (the others are sampled by the step launches).
__global__ void fd_batch_sample_kernel(BatchSample rec, const ShotDesc *shots, const float *traces, int level)
{
    batch_sample(rec, shots, traces, level, blockIdx.x * blockDim.x + threadIdx.x);
}

using BatchFn = void (*)(FdStepArgs, const ShotDesc *, const int4 *, int, int, const int *, int, float *, int, int,
                         BatchSample);

template <int R, int TY, int NJ>
static BatchFn batch_arith(int arith)
{
    return arith == PHC_FD_ARITH_REF ? fd_batch_kernel<R, TY, NJ, PHC_FD_ARITH_REF, uint32_t>
                                     : fd_batch_kernel<R, TY, NJ, PHC_FD_ARITH_FP32, uint32_t>;
}

template <int TY>
static BatchFn batch_quad(int arith, bool nt)
{
    if (arith == PHC_FD_ARITH_REF)
        return nt ? fd_batch_quad_kernel<TY, PHC_FD_ARITH_REF, true> : fd_batch_quad_kernel<TY, PHC_FD_ARITH_REF, false>;
    return nt ? fd_batch_quad_kernel<TY, PHC_FD_ARITH_FP32, true> : fd_batch_quad_kernel<TY, PHC_FD_ARITH_FP32, false>;
}

// nt: non-temporal accesses to the streamed arrays (the four-points-per-lane
// shapes; the others always have them).
static BatchFn batch_pick(int R, int ty, int nj, int arith, bool nt = true)
{
    if (R != 4) return nullptr;
    if (ty == 16 && nj == 1) return batch_arith<4, 16, 1>(arith);
    if (ty == 8 && nj == 1) return batch_arith<4, 8, 1>(arith);
    if (ty == 8 && nj == 2) return batch_arith<4, 8, 2>(arith);
    if (ty == 4 && nj == 2) return batch_arith<4, 4, 2>(arith);
    if (ty == 4 && nj == 4) return batch_quad<4>(arith, nt);
    if (ty == 8 && nj == 4) return batch_quad<8>(arith, nt);
    return nullptr;
}

void fd_axis_damping(int n, int W, float alpha, std::vector<float> &f);

} // namespace phc

using namespace phc;

struct phc_batch {
    int nshots = 0, R = 4, nsamples = 0, arith = 0, sw = 0;
    float alpha = 0.f;
    float coef[FD_MAX_R + 1];
    double coef0 = 0.0;
    std::vector<FdLayout> L;
    std::vector<int> src;
    std::vector<ShotDesc> hdesc;
    DevBuf pool, shots, items, it0, traces, rec, recoff;
    int cur = 1;      // level holding the current field (the reference's i2)
    int pending = 0;  // the previous level still owes its sponge product
    hipStream_t stream = nullptr;
    int ty = 16, nj = 1, chunk_i = 64, blocks_per_cu = 1, cus = 256;
    int krem_mode = 0;  // phc_batch_params.k_remainder
    int nitems = 0;  // entries of the work table, padding included
    int nrec = 0;  // receivers per shot
    int timing = 0;
    double last_ms = 0.0;
    int last_n = 0, last_nrec = 0;
    RunGraphs graph[2];  // of phc_batch_run, by the level it starts from
};

static void batch_drop_graph(phc_batch *h)
{
    for (RunGraphs &g : h->graph) g.drop();
}

// Planes per work item when the caller gives none: 24, fewer where a resident
// block then gets less than a few items' worth of planes.  Items of c planes
// waste about (2R+1)/c of the time on ring lead-ins (loads without a stencil)
// and c/2x on the part-empty last round, x = planes of tile columns per
// resident block.  Measured (4 waves x 16 rows; x = 13, 15, 44, 75, 214): 24
// planes 34.1, 29.2, 88.8, 188, 612 us per step, the best of 8-128 planes
// 31.7, 29.2, 88.8, 186, 609; at x = 1.1, 8 planes 9.6, 24 planes 16.1.
static int batch_default_chunk(const phc_batch *h, const int *dims)
{
    const int TJ = h->ty * h->nj;
    double planes = 0.0;
    for (int s = 0; s < h->nshots; ++s)
        planes += (double)((dims[3 * s + 2] + FD_TK - 1) / FD_TK) * ((dims[3 * s + 1] + TJ - 1) / TJ) * dims[3 * s];
    const double slots = (double)h->cus * (h->nj == 4 ? 12 / h->ty : std::max(32 / (h->ty * h->nj), 1));
    return std::clamp((int)std::lround(7.0 * planes / slots), 8, 24);
}

// Work items of every shot for the current shape, one list per XCD,
// interleaved into the table (entry 8 l + x = entry l of XCD x's list, shorter
// lists padded).  With k_remainder 1 a shot's partial last k tile becomes
// point-by-point items instead (as a tile it was faster on every survey
// measured: 200 against 228 us per step on 12 shots of U[96,224]^3, 40
// against 50 on 14 of U[60,100]^3, 642 against 686 on 24 of U[128,256]^3).
// * chunk_i > 0: items in spatial order (shot, i-chunk, j-tile, k-tile,
//   then the slab parts), cut into contiguous runs of about equal cost
//   (planes incl. the 2R lead-in x rows; a slab point costs a few tile
//   points: it reads its stencil from memory).
// * chunk_i = -m: each shot's per-XCD schedule (xcd_sched.hpp, split m, one
//   round = blocks_per_cu blocks on each of the XCD's CUs): list x takes the
//   entries of XCD x, shot after shot; slab parts go to the list with the
//   least work so far.
static phc_status batch_build_items(phc_batch *h)
{
    std::vector<std::vector<int4>> lists(BATCH_XCDS);
    std::vector<double> lcost(BATCH_XCDS, 0.0);
    std::vector<int4> items;
    std::vector<double> cost;
    const int TJ = h->ty * h->nj;
    const int T = FD_TK * h->ty;
    const bool sched = h->chunk_i < 0;
    const int slots = std::max(h->cus / BATCH_XCDS, 1) * h->blocks_per_cu;
    std::vector<int4> tab;
    for (int s = 0; s < h->nshots; ++s) {
        const FdLayout &L = h->L[s];
        const int full = L.nz / FD_TK, rem = L.nz - full * FD_TK;
        const bool slab = h->krem_mode == 1 && full > 0 && rem > 0;
        h->hdesc[s].krem = slab ? FD_TK * full : 0;
        const int tk = slab ? full : (L.nz + FD_TK - 1) / FD_TK, tj = (L.ny + TJ - 1) / TJ;
        h->hdesc[s].tiles_k = tk;
        auto tile_cost = [&](int jt, int planes) {
            return (double)(planes + 2 * h->R) * std::min(TJ, L.ny - jt * TJ);
        };
        if (sched) {
            build_xcd_schedule(L.nx, 0, tk * tj, slots, -h->chunk_i, 1, tab);
            for (size_t b = 0; b < tab.size(); ++b) {
                const int4 e = tab[b];
                if (e.y >= e.z) continue;
                const int x = (int)(b % BATCH_XCDS);
                lists[x].push_back(make_int4(s, e.x, e.y, e.z));
                lcost[x] += tile_cost(e.x / tk, e.z - e.y);
            }
        } else {
            const int nc = (L.nx + h->chunk_i - 1) / h->chunk_i;
            for (int ic = 0; ic < nc; ++ic) {
                const int i0 = (int)((int64_t)L.nx * ic / nc), i1 = (int)((int64_t)L.nx * (ic + 1) / nc);
                for (int w = 0; w < tk * tj; ++w) {
                    items.push_back(make_int4(s, w, i0, i1));
                    cost.push_back(tile_cost(w / tk, i1 - i0));
                }
            }
        }
        if (slab) {
            const int64_t pts = (int64_t)rem * L.ny * L.nx, per = (int64_t)BATCH_SLAB_PASSES * T;
            for (int64_t q = 0; q * per < pts; ++q) {
                const double c = 3.0 * (double)std::min(per, pts - q * per) / FD_TK;
                const int4 it = make_int4(s, -1 - (int)q, 0, 1);
                if (sched) {
                    const int x = (int)(std::min_element(lcost.begin(), lcost.end()) - lcost.begin());
                    lists[x].push_back(it);
                    lcost[x] += c;
                } else {
                    items.push_back(it);
                    cost.push_back(c);
                }
            }
        }
    }
    // the descriptors carry each shot's slab start and tile count
    PHC_HIP(hipMemcpy(h->shots.ptr, h->hdesc.data(), sizeof(ShotDesc) * h->nshots, hipMemcpyHostToDevice));
    if (!sched) {
        const double total = std::accumulate(cost.begin(), cost.end(), 0.0);
        double acc = 0.0;
        for (size_t i = 0; i < items.size(); ++i) {
            // the list whose share of the cost holds the item's middle
            const int x = (int)((acc + 0.5 * cost[i]) / total * BATCH_XCDS);
            lists[std::min(x, BATCH_XCDS - 1)].push_back(items[i]);
            acc += cost[i];
        }
    }
    size_t longest = 0;
    for (const auto &l : lists) longest = std::max(longest, l.size());
    std::vector<int4> table(BATCH_XCDS * longest, make_int4(0, 0, 0, 0));
    for (int x = 0; x < BATCH_XCDS; ++x)
        for (size_t l = 0; l < lists[x].size(); ++l) table[BATCH_XCDS * l + x] = lists[x][l];
    h->nitems = (int)table.size();
    PHC_TRY(h->items.alloc(sizeof(int4) * table.size()));
    PHC_HIP(hipMemcpy(h->items.ptr, table.data(), sizeof(int4) * table.size(), hipMemcpyHostToDevice));
    return PHC_OK;
}

static void batch_common(const phc_batch *h, FdStepArgs &c, int damp)
{
    std::memset(&c, 0, sizeof(c));
    for (int l = 0; l <= FD_MAX_R; ++l) c.cx[l] = c.cy[l] = c.cz[l] = h->coef[l];
    c.coef0 = h->coef0;
    c.c0f = (float)h->coef0;
    c.sw = h->sw;
    for (int d = 0; d <= h->sw && d <= FD_MAX_SW; ++d)
        c.stab[d] = (float)std::exp((double)h->alpha * std::pow((double)d, 2.0));
    c.damp_prev = damp;
    c.chunk_i = h->chunk_i;
}

// One batched step: every shot from level `cur` (current) and 1-cur
// (previous, overwritten by the new level).  traces[shot*stride + step] gets
// each shot's new source value before the fused injection of rhs[it+1]; `rec`
// samples the receivers of level `cur`.
static phc_status batch_launch(phc_batch *h, int cur, int inj, int damp, float *traces, int stride, int step,
                               const BatchSample &rec)
{
    // a pool past what the 256 MB memory-side cache keeps streams past it
    BatchFn fn = batch_pick(h->R, h->ty, h->nj, h->arith, h->pool.bytes > (size_t)300e6);
    if (!fn) return fail(PHC_ERR_INVALID, "no batched kernel for %d waves x %d rows", h->ty, h->nj);
    FdStepArgs c;
    batch_common(h, c, damp);
    const int T = FD_TK * h->ty;
    hipLaunchKernelGGL(fn, dim3(h->nitems + (rec.n + T - 1) / T), dim3(FD_TK, h->ty), 0, h->stream, c,
                       h->shots.as<ShotDesc>(), h->items.as<int4>(), h->nitems, cur, h->it0.as<int>(), inj, traces, stride, step,
                       rec);
    PHC_HIP(hipGetLastError());
    return PHC_OK;
}

// A run's steps on h->stream (fd_batch_inject_kernel has gone before): one
// batched step per sample; a step's receivers are sampled by the next step's
// launch, the last step's by a launch of their own.  Names no time sample, so
// that a captured run serves every chunk.  With `ev`, events bracket every
// batched launch.
static phc_status batch_enqueue(phc_batch *h, int nsteps, hipEvent_t *ev)
{
    int cur = h->cur;
    BatchSample rec{h->recoff.as<int64_t>(), h->rec.as<float>(), 0, h->nrec, nsteps, 0};
    for (int s = 0; s < nsteps; ++s) {
        const int damp = (s == 0) ? h->pending : (h->sw > 0 ? 1 : 0);
        rec.n = s > 0 ? h->nshots * h->nrec : 0;
        rec.step = s - 1;
        if (ev) PHC_HIP(hipEventRecord(ev[2 * s], h->stream));
        PHC_TRY(batch_launch(h, cur, s + 1 < nsteps ? 1 : 0, damp, h->traces.as<float>(), nsteps, s, rec));
        if (ev) PHC_HIP(hipEventRecord(ev[2 * s + 1], h->stream));
        cur = 1 - cur;
    }
    if (h->nrec > 0) {
        rec.n = h->nshots * h->nrec;
        rec.step = nsteps - 1;
        hipLaunchKernelGGL(fd_batch_sample_kernel, dim3((rec.n + 255) / 256), dim3(256), 0, h->stream, rec,
                           h->shots.as<ShotDesc>(), h->traces.as<float>(), cur);
        PHC_HIP(hipGetLastError());
    }
    return PHC_OK;
}

static phc_status batch_upload(const std::vector<float> &buf, float *dev)
{
    PHC_HIP(hipMemcpy(dev, buf.data(), sizeof(float) * buf.size(), hipMemcpyHostToDevice));
    return PHC_OK;
}

extern "C" {

phc_status phc_batch_create(const phc_batch_params *p, phc_batch **out)
{
    if (!out) return fail(PHC_ERR_INVALID, "out is NULL");
    *out = nullptr;
    if (!p) return fail(PHC_ERR_INVALID, "params is NULL");
    if (p->nshots < 1) return fail(PHC_ERR_INVALID, "no shots (nshots = %d)", p->nshots);
    if (!p->dims || !p->src || !p->vp || !p->rhs || !p->coef)
        return fail(PHC_ERR_INVALID, "dims, src, vp, rhs or coef is NULL");
    if (p->half_width != 4) return fail(PHC_ERR_INVALID, "batched shots need half width 4 (got %d)", p->half_width);
    if (p->sponge_width < 0 || p->sponge_width > FD_MAX_SW)
        return fail(PHC_ERR_INVALID, "sponge width %d outside 0..%d", p->sponge_width, FD_MAX_SW);
    if (p->arith != PHC_FD_ARITH_REF && p->arith != PHC_FD_ARITH_FP32)
        return fail(PHC_ERR_INVALID, "unknown arithmetic mode %d", p->arith);
    if (p->nsamples < 1) return fail(PHC_ERR_INVALID, "nsamples must be >= 1 (got %d)", p->nsamples);
    if (p->chunk_i < -4 || p->blocks_per_cu < 0 || p->blocks_per_cu > 8)
        return fail(PHC_ERR_INVALID, "bad chunk_i (planes per item, or -1..-4) or blocks_per_cu");
    if (p->k_remainder < -1 || p->k_remainder > 1)
        return fail(PHC_ERR_INVALID, "k_remainder must be -1, 0 or 1 (got %d)", p->k_remainder);
    // default: 4 waves x 16 rows, four points per lane, the fastest shape on
    // every survey measured (12 shots of U[96,224]^3 / 8 of U[106,190]^3 / 14
    // of U[60,100]^3 / 24 of U[128,256]^3, best chunk of each: 188 / 88 / 31 /
    // 649 us per step; 8 waves x 32 rows 202 / 102 / 34 / 672; 8 waves x 1 row
    // 200 / 102 / 45 / 685; 4 waves x 2 rows 217 / 112 / 53 / 728)
    const bool shape = p->block_waves || p->tile_j;
    const int ty = p->block_waves ? p->block_waves : shape ? 16 : 4;
    const int tj = p->tile_j ? p->tile_j : shape ? ty : 16;
    if (ty <= 0 || tj % ty != 0 || !batch_pick(p->half_width, ty, tj / ty, p->arith))
        return fail(PHC_ERR_INVALID, "no batched kernel for tile_j %d, %d waves per block", tj, ty);
    for (int s = 0; s < p->nshots; ++s) {
        const int nx = p->dims[3 * s], ny = p->dims[3 * s + 1], nz = p->dims[3 * s + 2];
        const int xs = p->src[3 * s], ys = p->src[3 * s + 1], zs = p->src[3 * s + 2];
        if (nx < 1 || ny < 1 || nz < 1) return fail(PHC_ERR_INVALID, "shot %d: empty grid", s);
        if (xs < 0 || xs >= nx || ys < 0 || ys >= ny || zs < 0 || zs >= nz)
            return fail(PHC_ERR_INVALID, "shot %d: source (%d,%d,%d) outside the grid", s, xs, ys, zs);
        if (!p->vp[s] || !p->rhs[s]) return fail(PHC_ERR_INVALID, "shot %d: vp or rhs is NULL", s);
        if (make_fd_layout(nx, ny, nz, p->half_width).total * 4 >= ((int64_t)1 << 32))
            return fail(PHC_ERR_INVALID, "shot %d: arrays exceed 4 GiB", s);
    }
    phc_batch *h = new phc_batch();
    auto bail = [&](phc_status st) { phc_batch_destroy(h); return st; };
    h->nshots = p->nshots;
    h->R = p->half_width;
    h->nsamples = p->nsamples;
    h->arith = p->arith;
    h->sw = p->sponge_width;
    h->alpha = p->sponge_alpha;
    std::memset(h->coef, 0, sizeof(h->coef));
    for (int l = 0; l <= h->R; ++l) h->coef[l] = p->coef[l];
    h->coef0 = p->coef0;
    h->src.assign(p->src, p->src + 3 * h->nshots);
    h->ty = ty;
    h->nj = tj / ty;
    h->chunk_i = p->chunk_i;
    h->blocks_per_cu = p->blocks_per_cu ? p->blocks_per_cu : 1;
    h->krem_mode = p->k_remainder;
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
        h->cus = prop.multiProcessorCount;
    if (h->chunk_i == 0) h->chunk_i = batch_default_chunk(h, p->dims);
    if (hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking) != hipSuccess)
        return bail(fail(PHC_ERR_HIP, "hipStreamCreate failed"));
    // one pool: per shot two levels, vp^2dt^2, fy, fz, rhs; each shot 256-byte aligned
    std::vector<int64_t> off(h->nshots);
    int64_t total = 0;
    h->L.resize(h->nshots);
    for (int s = 0; s < h->nshots; ++s) {
        h->L[s] = make_fd_layout(p->dims[3 * s], p->dims[3 * s + 1], p->dims[3 * s + 2], h->R);
        off[s] = total;
        total += 3 * h->L[s].total + h->L[s].ny + h->L[s].nz + h->nsamples;
        total = round_up(total, 64);
    }
    phc_status st;
    if ((st = h->pool.alloc(sizeof(float) * total)) || (st = h->shots.alloc(sizeof(ShotDesc) * h->nshots)) ||
        (st = h->it0.alloc(sizeof(int))))
        return bail(st);
    h->hdesc.resize(h->nshots);
    for (int s = 0; s < h->nshots; ++s) {
        const FdLayout &L = h->L[s];
        float *base = h->pool.as<float>() + off[s];
        ShotDesc &d = h->hdesc[s];
        d.L = L;
        d.lev[0] = base;
        d.lev[1] = base + L.total;
        float *vp = base + 2 * L.total, *fy = vp + L.total, *fz = fy + L.ny, *rhs = fz + L.nz;
        d.vp = vp;
        d.fy = fy;
        d.fz = fz;
        d.rhs = rhs;
        d.src_off = fd_off(L, h->src[3 * s], h->src[3 * s + 1], h->src[3 * s + 2]);
        std::vector<float> buf((size_t)L.total, p->init_value);
        if ((st = batch_upload(buf, d.lev[0])) || (st = batch_upload(buf, d.lev[1]))) return bail(st);
        std::fill(buf.begin(), buf.end(), 0.f);
        const float *v = p->vp[s];
        for (int64_t n = 0; n < (int64_t)L.nx * L.ny * L.nz; ++n)
            if (!(v[n] >= 0.f) || !std::isfinite(v[n]))
                return bail(fail(PHC_ERR_INVALID, "shot %d: vp^2 dt^2 at %lld is negative or not finite", s,
                                 (long long)n));
        for (int i = 0; i < L.nx; ++i)
            for (int j = 0; j < L.ny; ++j)
                std::memcpy(&buf[(size_t)fd_off(L, i, j, 0)], v + ((int64_t)i * L.ny + j) * L.nz,
                            sizeof(float) * L.nz);
        if ((st = batch_upload(buf, vp))) return bail(st);
        std::vector<float> f;
        fd_axis_damping(L.ny, h->sw, h->alpha, f);
        if ((st = batch_upload(f, fy))) return bail(st);
        fd_axis_damping(L.nz, h->sw, h->alpha, f);
        if ((st = batch_upload(f, fz))) return bail(st);
        if ((st = batch_upload(std::vector<float>(p->rhs[s], p->rhs[s] + h->nsamples), rhs))) return bail(st);
    }
    if (hipMemcpy(h->shots.ptr, h->hdesc.data(), sizeof(ShotDesc) * h->nshots, hipMemcpyHostToDevice) !=
        hipSuccess)
        return bail(fail(PHC_ERR_HIP, "descriptor upload failed"));
    if ((st = batch_build_items(h))) return bail(st);
    *out = h;
    return PHC_OK;
}

phc_status phc_batch_destroy(phc_batch *h)
{
    if (!h) return PHC_OK;
    if (h->stream) (void)hipStreamSynchronize(h->stream);
    batch_drop_graph(h);
    for (DevBuf *b : {&h->pool, &h->shots, &h->items, &h->it0, &h->traces, &h->rec, &h->recoff})
        b->release();
    if (h->stream) (void)hipStreamDestroy(h->stream);
    delete h;
    return PHC_OK;
}

phc_status phc_batch_set_receivers(phc_batch *h, int nrec, const int *ijk)
{
    if (!h) return fail(PHC_ERR_INVALID, "handle is NULL");
    if (nrec < 0 || (nrec > 0 && !ijk)) return fail(PHC_ERR_INVALID, "bad receiver list");
    std::vector<int64_t> offs((size_t)h->nshots * nrec);
    for (int s = 0; s < h->nshots; ++s)
        for (int r = 0; r < nrec; ++r) {
            const int *q = ijk + 3 * ((size_t)s * nrec + r);
            const FdLayout &L = h->L[s];
            if (q[0] < 0 || q[0] >= L.nx || q[1] < 0 || q[1] >= L.ny || q[2] < 0 || q[2] >= L.nz)
                return fail(PHC_ERR_INVALID, "shot %d receiver %d at (%d,%d,%d) is outside the grid", s, r, q[0],
                            q[1], q[2]);
            offs[(size_t)s * nrec + r] = fd_off(L, q[0], q[1], q[2]);
        }
    PHC_HIP(hipStreamSynchronize(h->stream));
    batch_drop_graph(h);
    h->nrec = nrec;
    if (nrec > 0) {
        PHC_TRY(h->recoff.alloc(sizeof(int64_t) * offs.size()));
        PHC_HIP(hipMemcpy(h->recoff.ptr, offs.data(), sizeof(int64_t) * offs.size(), hipMemcpyHostToDevice));
    }
    return PHC_OK;
}

phc_status phc_batch_run(phc_batch *h, int it0, int nsteps)
{
    RoctxRange rr_("phc_batch_run");
    if (!h) return fail(PHC_ERR_INVALID, "handle is NULL");
    if (nsteps < 0) return fail(PHC_ERR_INVALID, "negative step count");
    if (nsteps == 0) return PHC_OK;
    if (it0 < 0 || it0 + nsteps > h->nsamples)
        return fail(PHC_ERR_INVALID, "steps %d..%d outside the %d source samples", it0, it0 + nsteps - 1,
                    h->nsamples);
    const size_t tbytes = sizeof(float) * (size_t)nsteps * h->nshots;
    const size_t rbytes = tbytes * h->nrec;
    if (h->traces.bytes < tbytes || (h->nrec > 0 && h->rec.bytes < rbytes)) {
        PHC_HIP(hipStreamSynchronize(h->stream));
        batch_drop_graph(h);
        if (h->traces.bytes < tbytes) PHC_TRY(h->traces.alloc(tbytes));
        if (h->nrec > 0 && h->rec.bytes < rbytes) PHC_TRY(h->rec.alloc(rbytes));
    }
    // changes the current level: launched once nothing but launches can fail
    auto begin = [&]() -> phc_status {
        hipLaunchKernelGGL(fd_batch_inject_kernel, dim3((h->nshots + 63) / 64), dim3(64), 0, h->stream,
                           h->shots.as<ShotDesc>(), h->nshots, h->cur, it0, h->it0.as<int>());
        PHC_HIP(hipGetLastError());
        return PHC_OK;
    };
    if (h->timing) {
        std::vector<hipEvent_t> ev(2 * (size_t)nsteps);
        for (auto &e : ev) PHC_HIP(hipEventCreate(&e));
        phc_status st = begin();
        if (st == PHC_OK) st = batch_enqueue(h, nsteps, ev.data());
        if (st == PHC_OK) {
            PHC_HIP(hipStreamSynchronize(h->stream));
            double tot = 0.0;
            for (int s = 0; s < nsteps; ++s) {
                float ms = 0.f;
                PHC_HIP(hipEventElapsedTime(&ms, ev[2 * s], ev[2 * s + 1]));
                tot += ms;
            }
            h->last_ms = tot / nsteps;
        }
        for (auto &e : ev) (void)hipEventDestroy(e);
        PHC_TRY(st);
    } else {
        PHC_TRY(prepare_captured(h->stream, h->graph[h->cur], nsteps, h->pending, h->nrec,
                                 [&] { return batch_enqueue(h, nsteps, nullptr); }));
        PHC_TRY(begin());
        PHC_HIP(hipGraphLaunch(h->graph[h->cur].exec(), h->stream));
    }
    if (nsteps % 2) h->cur = 1 - h->cur;
    h->pending = h->sw > 0 ? 1 : 0;
    h->last_n = nsteps;
    h->last_nrec = h->nrec;
    return PHC_OK;
}

phc_status phc_batch_get_traces(phc_batch *h, float *src, float *rec)
{
    if (!h) return fail(PHC_ERR_INVALID, "handle is NULL");
    PHC_HIP(hipStreamSynchronize(h->stream));
    const size_t n = (size_t)h->last_n * h->nshots;
    if (src && n > 0) PHC_HIP(hipMemcpy(src, h->traces.ptr, sizeof(float) * n, hipMemcpyDeviceToHost));
    if (rec && n > 0 && h->last_nrec > 0)
        PHC_HIP(hipMemcpy(rec, h->rec.ptr, sizeof(float) * n * h->last_nrec, hipMemcpyDeviceToHost));
    return PHC_OK;
}

phc_status phc_batch_get_field(phc_batch *h, int shot, int current, float *host)
{
    if (!h || !host) return fail(PHC_ERR_INVALID, "handle or host buffer is NULL");
    if (shot < 0 || shot >= h->nshots) return fail(PHC_ERR_INVALID, "shot %d outside 0..%d", shot, h->nshots - 1);
    PHC_HIP(hipStreamSynchronize(h->stream));
    const FdLayout &L = h->L[shot];
    const int level = current ? h->cur : 1 - h->cur;
    std::vector<float> buf((size_t)L.total);
    PHC_HIP(hipMemcpy(buf.data(), h->hdesc[shot].lev[level], sizeof(float) * L.total, hipMemcpyDeviceToHost));
    const int R = L.R, NYe = L.ny + 2 * R, NZe = L.nz + 2 * R, W = h->sw;
    const bool damp = !current && h->pending;
    std::vector<float> fx, fy, fz;
    fd_axis_damping(L.nx, W, h->alpha, fx);
    fd_axis_damping(L.ny, W, h->alpha, fy);
    fd_axis_damping(L.nz, W, h->alpha, fz);
    for (int i = -R; i < L.nx + R; ++i)
        for (int j = -R; j < L.ny + R; ++j) {
            float *dst = host + ((int64_t)(i + R) * NYe + (j + R)) * NZe;
            std::memcpy(dst, &buf[(size_t)fd_off(L, i, j, -R)], sizeof(float) * NZe);
            if (!damp || i < 0 || i >= L.nx || j < 0 || j >= L.ny) continue;
            const bool inI = i >= W && i < L.nx - W, inJ = j >= W && j < L.ny - W;
            for (int k = 0; k < L.nz; ++k) {
                const bool inK = k >= W && k < L.nz - W;
                float s = 1.f;
                if (inJ && inK && !inI) s = fx[i];
                if (inK && inI && !inJ) s = fy[j];
                if (inJ && inI && !inK) s = fz[k];
                dst[k + R] = dst[k + R] * s;
            }
        }
    return PHC_OK;
}

phc_status phc_batch_set_timing(phc_batch *h, int enable)
{
    if (!h) return fail(PHC_ERR_INVALID, "handle is NULL");
    h->timing = enable ? 1 : 0;
    return PHC_OK;
}

phc_status phc_batch_last_run_kernel_ms(phc_batch *h, double *ms)
{
    if (!h || !ms) return fail(PHC_ERR_INVALID, "handle or ms is NULL");
    *ms = h->last_ms;
    return PHC_OK;
}

phc_status phc_batch_synchronize(phc_batch *h)
{
    if (!h) return fail(PHC_ERR_INVALID, "handle is NULL");
    PHC_HIP(hipStreamSynchronize(h->stream));
    return PHC_OK;
}

phc_status phc_batch_autotune(phc_batch *h, int steps_per_trial, int *tile_j, int *block_waves, int *chunk_i,
                              int *blocks_per_cu)
{
    RoctxRange rr_("phc_batch_autotune");
    if (!h) return fail(PHC_ERR_INVALID, "handle is NULL");
    if (steps_per_trial < 1 || steps_per_trial > 1000)
        return fail(PHC_ERR_INVALID, "steps_per_trial %d outside 1..1000", steps_per_trial);
    PHC_HIP(hipStreamSynchronize(h->stream));
    batch_drop_graph(h);
    // trials run on a copy of the pool; the shots' state is restored after
    DevBuf save, tr;
    PHC_TRY(save.alloc(h->pool.bytes));
    PHC_TRY(tr.alloc(sizeof(float) * h->nshots));
    PHC_HIP(hipMemcpy(save.ptr, h->pool.ptr, h->pool.bytes, hipMemcpyDeviceToDevice));
    hipEvent_t e0 = nullptr, e1 = nullptr;
    PHC_HIP(hipEventCreate(&e0));
    PHC_HIP(hipEventCreate(&e1));
    static const int shapes[][2] = {{16, 1}, {8, 1}, {8, 2}, {8, 4}, {4, 2}, {4, 4}};
    static const int chunks[] = {8, 16, 24, 32, 48, 64, 128, -1, -2, -3, -4};
    static const int bpcs[] = {1, 2, 4};
    double best = 1e30;
    int bty = h->ty, bnj = h->nj, bci = h->chunk_i, bbp = h->blocks_per_cu;
    phc_status st = PHC_OK;
    for (const auto &sh : shapes)
        for (int ci : chunks)
            for (int bp : bpcs) {
                if (st != PHC_OK) break;
                if (sh[0] * bp > 32) continue;  // at most 32 waves of one shape per CU
                if (ci > 0 && bp > bpcs[0]) continue;  // only the per-XCD schedules depend on it
                h->ty = sh[0];
                h->nj = sh[1];
                h->chunk_i = ci;
                h->blocks_per_cu = bp;
                if ((st = batch_build_items(h))) break;
                float ms = 0.f;
                for (int rep = 0; rep < 2 && st == PHC_OK; ++rep) {  // first pass warms up
                    if (hipEventRecord(e0, h->stream) != hipSuccess) st = fail(PHC_ERR_HIP, "event record failed");
                    for (int s = 0; s < steps_per_trial && st == PHC_OK; ++s)
                        st = batch_launch(h, (h->cur + s) & 1, 0, h->sw > 0, tr.as<float>(), 1, 0, BatchSample{});
                    if (st == PHC_OK && (hipEventRecord(e1, h->stream) != hipSuccess ||
                                         hipEventSynchronize(e1) != hipSuccess ||
                                         hipEventElapsedTime(&ms, e0, e1) != hipSuccess))
                        st = fail(PHC_ERR_HIP, "trial timing failed");
                }
                if (st == PHC_OK && ms < best) {
                    best = ms;
                    bty = h->ty; bnj = h->nj; bci = h->chunk_i; bbp = h->blocks_per_cu;
                }
            }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipStreamSynchronize(h->stream);
    if (hipMemcpy(h->pool.ptr, save.ptr, h->pool.bytes, hipMemcpyDeviceToDevice) != hipSuccess && st == PHC_OK)
        st = fail(PHC_ERR_HIP, "restoring the shots after tuning failed");
    save.release();
    tr.release();
    h->ty = bty; h->nj = bnj; h->chunk_i = bci; h->blocks_per_cu = bbp;
    PHC_TRY(st);
    PHC_TRY(batch_build_items(h));
    if (tile_j) *tile_j = bty * bnj;
    if (block_waves) *block_waves = bty;
    if (chunk_i) *chunk_i = bci;
    if (blocks_per_cu) *blocks_per_cu = bbp;
    return PHC_OK;
}

} // extern "C"
