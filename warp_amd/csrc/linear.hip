// Conjugate gradient on gfx950.
//
// Replaces the reference CG iteration (warp/_src/optim/linear.py:893-1121)
// and its JIT kernels: TiledDot (linear.py:309-612), _initialize_tolerance
// (2051-2083), _diag_mv_kernel (2271-2287), _cg_kernel_1/2 (2332-2373) and
// the host loop _run_solver_loop (2182-2243).
//
// Precision policy: vectors stay in the system scalar type S (fp32 or fp64);
// every dot product is accumulated in FP64 with a deterministic two-level
// reduction, and alpha/beta are formed in FP64.
//
// One iteration = three fused kernels on a device-resident state and no
// one-workgroup finalize kernel: each reduction leaves one FP64 partial per
// workgroup, and every workgroup of the next kernel sums all of them in the
// same fixed order in its prologue (bit-identical in every workgroup; the
// grids are capped so that these sums stay a few KB of L2 reads):
//   spmv     : Ap = A p, partials of p.Ap
//   update   : alpha = rz / pAp (0 once converged); x += alpha p,
//              r -= alpha Ap, z = M r, partials of r.r and r.z
//   direction: beta = rz_new / rz_old, done; p = z + beta p
// A field of the state is never written by a kernel whose workgroups read
// it: workgroup 0 of each kernel records what the next one needs (r.z of the
// previous iterate, `done` as the update saw it, the iteration count).
// Small systems (launch-bound: every kernel costs a few microseconds however
// little it does) fold the direction pass into the next SpMV: its prologue
// sums the update's partials into beta, and it evaluates p' = z + beta p
// entry by entry where the product gathers it (the same fma, so the iterates
// are bit-identical) and writes p' to the other of two direction buffers,
// since workgroups still gather p while others write p'.  r.z of the
// previous iterate is +inf after (re)initialisation, which makes beta 0 and
// p' = z.  Large systems keep the separate pass: gathering two vectors costs
// the HBM-bound SpMV more than the pass it saves.
// The convergence flag `done` (r.r <= atol^2) makes later kernels no-ops, the
// device-side equivalent of the reference's frozen alpha/beta.
#include "bsr_core.h"

#include <cmath>
#include <condition_variable>
#include <mutex>
#include <vector>

namespace wa {
namespace {

constexpr int kBlock = 256;
constexpr int kMaxGrid = 2048;  // generic vector kernels

struct CgState {
    double bb;
    double rr;       // r.r of the current iterate (host-visible)
    double rz;       // r.z of the current iterate
    double rz_prev;  // r.z of the previous iterate; +inf after (re)initialisation, so beta = 0
    double pAp;
    double atol_sq;
    double alpha;
    double beta;
    double rtol;
    double atol;
    int iter;       // iterations done (host-visible)
    int iter_copy;  // the SpMV's copy of iter (fused direction buffers), read by the update
    int done;       // r.r <= atol^2 for the current iterate
    int done_prev;  // `done` as the update saw it, read by the direction pass
    // small systems (cg_small_kernel): largest column window and block count of
    // a workgroup's rows, workgroups that finished
    int small_window;
    int small_blocks;
    int small_done;
};

enum PrecKind { kPrecNone = 0, kPrecDiag = 1, kPrecBlock = 2 };

// Grid caps.  Every reduction of an iteration leaves one FP64 partial per
// workgroup, and the next kernel's workgroups each sum all of them in the
// same fixed order in their prologue (so no one-workgroup finalize kernel
// sits between two work kernels): the SpMV walks its row tiles with at most
// kMaxSpmvGrid workgroups, the update and direction passes grid-stride with
// at most kMaxVecGrid.
constexpr int kMaxSpmvGrid = 2048;
constexpr int kSmallMaxGroups = 128;  // workgroups of cg_small_kernel
constexpr int kSmallReplicas = 8;     // copies of its exchange slots
constexpr int kMaxVecGrid = 1024;

struct CgWs {
    CgState* state;
    double* init_partials;  // 3 * max_init_blocks (b.b, r.r, r.z of the initial residual)
    double* spmv_partials;  // kMaxSpmvGrid (p.Ap)
    double* upd_partials;   // 2 * kMaxVecGrid (r.r, r.z)
    unsigned long long* small_slots;  // exchange slots of cg_small_kernel
    int max_init_blocks;
    void* r;
    void* z;
    void* p;   // direction buffers: iterations alternate which one holds p (fused path)
    void* p2;
    void* Ap;
};

// Largest row grid (the initial residual): one workgroup per 256/G block rows, G <= 64.
int cg_max_blocks(int64_t nrow) { return (int)std::max<int64_t>(1, ceil_div(nrow, 4)); }

CgWs carve_cg(void* base, size_t bytes, int64_t nrow, int64_t n, size_t scalar_bytes, size_t* needed)
{
    Carve c(base, bytes);
    CgWs w;
    w.max_init_blocks = cg_max_blocks(nrow);
    w.state = c.take<CgState>(1);
    w.init_partials = c.take<double>((size_t)3 * w.max_init_blocks);
    w.spmv_partials = c.take<double>((size_t)kMaxSpmvGrid);
    w.upd_partials = c.take<double>((size_t)2 * kMaxVecGrid);
    w.small_slots = c.take<unsigned long long>((size_t)kSmallReplicas * 6 * kSmallMaxGroups);
    w.r = c.take<char>((size_t)n * scalar_bytes);
    w.z = c.take<char>((size_t)n * scalar_bytes);
    w.p = c.take<char>((size_t)n * scalar_bytes);
    w.p2 = c.take<char>((size_t)n * scalar_bytes);
    w.Ap = c.take<char>((size_t)n * scalar_bytes);
    *needed = c.used;
    return w;
}

constexpr int kFinalizeBlock = 1024;

// Fixed-order sum of NV rows of `count` <= MAXP partials (row v at parts + v *
// stride) by one workgroup of kBlock threads, result in every thread.  Every
// workgroup of a kernel that calls it gets bit-identical sums: thread t adds
// parts[t], parts[t + kBlock], ... in order, then the same block reduction.
template <int NV, int MAXP>
__device__ __forceinline__ void sum_parts(const double* __restrict__ parts, size_t stride, int count, double* lds,
                                          double (&out)[NV])
{
    constexpr int kPer = MAXP / kBlock;
    static_assert(MAXP % kBlock == 0, "partial capacity is a multiple of the block");
    double t[NV][kPer];
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const int k = (int)threadIdx.x + u * kBlock;
            t[v][u] = k < count ? parts[(size_t)v * stride + k] : 0.0;
        }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        double a = 0.0;
#pragma unroll
        for (int u = 0; u < kPer; ++u)
            a += t[v][u];
        out[v] = block_sum<kBlock>(a, lds);
    }
}

// Direction buffers.  Unfused, p stays in ws.p.  Fused, iteration k reads
// buffer k & 1 and writes the other: the choice is made on the device, so a
// captured iteration replays correctly any number of times.
template <typename S> __device__ __forceinline__ S* dir_buffer(const CgWs& ws, int which)
{
    return static_cast<S*>(which ? ws.p2 : ws.p);
}

// Vectors up to this size fold the direction pass into the SpMV (measured on
// MI355X: 2D Poisson, 16,129 dofs, 18 -> 15 us per iteration; 823,875-dof
// elasticity and 2M-dof FP64 systems slower by 2-12 us per iteration).
constexpr size_t kFusedDirectionMaxBytes = (size_t)1 << 20;

// z = M r for one block row.
template <typename S, int BR, int PREC>
__device__ __forceinline__ void apply_prec(const S* __restrict__ prec, int row, const S (&r)[BR], S (&z)[BR])
{
    if (PREC == kPrecDiag) {
#pragma unroll
        for (int s = 0; s < BR; ++s)
            z[s] = prec[(size_t)row * BR + s] * r[s];
    } else if (PREC == kPrecBlock) {
        const S* m = prec + (size_t)row * BR * BR;
#pragma unroll
        for (int s = 0; s < BR; ++s) {
            S v = S(0);
#pragma unroll
            for (int c = 0; c < BR; ++c)
                v = fma(m[s * BR + c], r[c], v);
            z[s] = v;
        }
    } else {
#pragma unroll
        for (int s = 0; s < BR; ++s)
            z[s] = r[s];
    }
}

// r = b - A x ; z = M r ; p = z ; partials of (b.b, r.r, r.z).  The grid
// covers the matrix: kCgRpg consecutive block rows per group of G lanes.
template <typename S, int BR, int G, int PREC, int kCgRpg = rows_per_group_for(BR, BR)>
__global__ __launch_bounds__(kBlock) void cg_init_kernel(
    int nrow, const int* __restrict__ offsets, const int* __restrict__ columns, const S* __restrict__ values,
    const S* __restrict__ prec, const S* __restrict__ b, const S* __restrict__ x, S* __restrict__ r, S* __restrict__ z,
    int fused, CgWs ws
)
{
    __shared__ double lds[kBlock / kWave];
    S* __restrict__ p = dir_buffer<S>(ws, fused ? (ws.state->iter & 1) : 0);
    const int row0 = (blockIdx.x * (kBlock / G) + threadIdx.x / G) * kCgRpg;
    const int lane = threadIdx.x % G;
    double acc3[3] = {0.0, 0.0, 0.0};
    if (row0 < nrow) {
        const RowAcc<S, BR * kCgRpg> ax =
            group_rows_product<S, BR, BR, G, kCgRpg>(row0, nrow, lane, offsets, nullptr, columns, values, x);
        for (int j = lane; j < kCgRpg && row0 + j < nrow; j += G) {
            const int row = row0 + j;
            S rv[BR], zv[BR];
#pragma unroll
            for (int s = 0; s < BR; ++s) {
                const S bv = b[(size_t)row * BR + s];
                rv[s] = bv - pick(ax, j * BR + s);
                acc3[0] += (double)bv * (double)bv;
            }
            apply_prec<S, BR, PREC>(prec, row, rv, zv);
#pragma unroll
            for (int s = 0; s < BR; ++s) {
                const size_t i = (size_t)row * BR + s;
                r[i] = rv[s];
                if (PREC != kPrecNone)
                    z[i] = zv[s];
                p[i] = zv[s];
                acc3[1] += (double)rv[s] * (double)rv[s];
                acc3[2] += (double)rv[s] * (double)zv[s];
            }
        }
    }
    write_block_partials<kBlock, 3>(acc3, ws.init_partials, lds);
}

// One workgroup: sums the initial residual's partials and (re)initialises
// the state; on the fused path also leaves r.r and r.z as the update's
// partials (first entry, zeros after it), which the first SpMV sums back
// exactly.
__global__ __launch_bounds__(kFinalizeBlock) void cg_init_finalize_kernel(CgWs ws, int nparts, int upd_parts,
                                                                          int has_prec, int first, int fused)
{
    __shared__ double lds[kFinalizeBlock / kWave];
    CgState* state = ws.state;
    double tot[3];
    sum_partials_rows<kFinalizeBlock, 3>(ws.init_partials, (size_t)nparts, nparts, lds, tot);
    const double rz = has_prec ? tot[2] : tot[1];
    if (fused) {
        for (int k = threadIdx.x; k < upd_parts; k += kFinalizeBlock) {
            ws.upd_partials[k] = k == 0 ? tot[1] : 0.0;
            ws.upd_partials[upd_parts + k] = k == 0 ? rz : 0.0;
        }
    }
    if (threadIdx.x != 0)
        return;
    if (first) {
        state->bb = tot[0];
        const double a = fmax(state->rtol * sqrt(tot[0]), state->atol);
        state->atol_sq = a * a;
        state->iter = 0;
    }
    state->rr = tot[1];
    state->rz = rz;
    state->rz_prev = __builtin_inf();
    state->done = !(tot[1] > state->atol_sq);
    state->done_prev = state->done;
    state->alpha = 0.0;
    state->beta = 0.0;
}

// p' = z + beta p, entry i.
template <typename S> struct NextDirection {
    const S* __restrict__ z;
    const S* __restrict__ p;
    S beta;
    __device__ __forceinline__ S operator()(size_t i) const { return fma(beta, p[i], z[i]); }
};

// Ap = A p and p.Ap partials, the grid walking tiles of kBlock / G * kCgRpg
// block rows.  FUSED: the prologue first sums the update's partials into
// r.r and r.z of the current iterate, hence beta and `done` (workgroup 0
// records them), and the product is A p' with p' = z + beta p evaluated
// where it is gathered and written to the other direction buffer.
// Unfused: `done` and p come from the direction pass.
template <typename S, int BR, int G, bool FUSED, int kCgRpg = rows_per_group_for(BR, BR)>
__global__ __launch_bounds__(kBlock) void cg_spmv_kernel(
    int nrow, const int* __restrict__ offsets, const int* __restrict__ columns, const S* __restrict__ values,
    const S* __restrict__ z, S* __restrict__ Ap, int upd_parts, CgWs ws, double* __restrict__ parts
)
{
    __shared__ double lds[kBlock / kWave];
    CgState* state = ws.state;
    S beta = S(0);
    int par = 0;
    if constexpr (FUSED) {
        double t[2];
        sum_parts<2, kMaxVecGrid>(ws.upd_partials, (size_t)upd_parts, upd_parts, lds, t);
        const bool live = t[0] > state->atol_sq;
        const double bt = live ? t[1] / state->rz_prev : 0.0;
        par = state->iter & 1;
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            state->rr = t[0];
            state->rz = t[1];
            state->beta = bt;
            state->done = !live;
            state->iter_copy = state->iter;
        }
        if (!live)
            return;
        beta = (S)bt;
    } else {
        if (state->done)
            return;
    }
    const S* __restrict__ p = dir_buffer<S>(ws, par);
    S* __restrict__ p_next = dir_buffer<S>(ws, par ^ 1);
    const NextDirection<S> dir{z, p, beta};
    constexpr int kTileRows = (kBlock / G) * kCgRpg;
    const int ntiles = (nrow + kTileRows - 1) / kTileRows;
    const int lane = threadIdx.x % G;
    // odd iterations walk the tiles from the last: each product starts with
    // the rows the previous one read last, still in the memory-side cache
    const bool reverse = state->iter & 1;
    double acc[1] = {0.0};
    for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const int tile = reverse ? ntiles - 1 - t : t;
        const int row0 = (tile * (kBlock / G) + (int)threadIdx.x / G) * kCgRpg;
        if (row0 >= nrow)
            continue;
        if constexpr (FUSED) {
            const RowAcc<S, BR * kCgRpg> ap = group_rows_product_f<S, BR, BR, G, kCgRpg, S>(
                row0, nrow, lane, offsets, nullptr, columns, values, dir
            );
            for (int e = lane; e < BR * kCgRpg && row0 + e / BR < nrow; e += G) {
                const size_t i = (size_t)row0 * BR + e;
                const S v = pick(ap, e);
                const S pn = dir(i);
                p_next[i] = pn;
                Ap[i] = v;
                acc[0] += (double)pn * (double)v;
            }
        } else {
            const RowAcc<S, BR * kCgRpg> ap =
                group_rows_product<S, BR, BR, G, kCgRpg>(row0, nrow, lane, offsets, nullptr, columns, values, p);
            for (int e = lane; e < BR * kCgRpg && row0 + e / BR < nrow; e += G) {
                const size_t i = (size_t)row0 * BR + e;
                const S v = pick(ap, e);
                Ap[i] = v;
                acc[0] += (double)p[i] * (double)v;
            }
        }
    }
    write_block_partials<kBlock, 1>(acc, parts, lds);
}

// The unfused SpMV of large scalar systems by wave tiles (see
// wave_rows_product; each row's sum as above), one workgroup of four tiles
// each, their partials reduced as the wide grid's.  256^3 FP32: 250-261 ->
// 220 us.
template <typename S, int G, int RW, int CH, bool STREAM>
__global__ __launch_bounds__(kBlock) void cg_spmv_wave_kernel(
    int nrow, const int* __restrict__ offsets, const int* __restrict__ columns, const S* __restrict__ values,
    S* __restrict__ Ap, CgWs ws, double* __restrict__ parts
)
{
    __shared__ __attribute__((aligned(16))) WaveTile<S, S, CH> tiles[kBlock / kWave];
    __shared__ double lds[kBlock / kWave];
    const CgState* state = ws.state;
    if (state->done)
        return;
    const S* __restrict__ p = static_cast<const S*>(ws.p);
    int b = xcd_run_block((int)blockIdx.x, (int)gridDim.x);
    if (state->iter & 1)  // odd iterations from the last tile, as above
        b = (int)gridDim.x - 1 - b;
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int64_t first = ((int64_t)b * (kBlock / kWave) + wave) * RW;
    double acc[1] = {0.0};
    if (first < nrow) {
        const int row0 = (int)first;
        const S v =
            wave_rows_product<S, G, RW, CH, STREAM>(row0, nrow, lane, offsets, columns, values, LoadX<S>{p}, tiles[wave]);
        if (lane < RW && row0 + lane < nrow) {
            Ap[row0 + lane] = v;
            acc[0] = (double)p[row0 + lane] * (double)v;
        }
    }
    write_block_partials<kBlock, 1>(acc, parts, lds);
}

// Wide SpMV grids (one workgroup per tile, more than kMaxSpmvGrid): their
// partials reduced to kWideParts, workgroup b summing the b-th contiguous
// range in a fixed order into spmv_partials[b]; the update sums those.
constexpr int kWideParts = 64;
__global__ __launch_bounds__(kFinalizeBlock) void cg_wide_spmv_finalize_kernel(const double* __restrict__ parts,
                                                                              int nparts, CgWs ws)
{
    __shared__ double lds[kFinalizeBlock / kWave];
    if (ws.state->done)
        return;
    const int chunk = (nparts + kWideParts - 1) / kWideParts;
    const int lo = min((int)blockIdx.x * chunk, nparts);
    const int hi = min(lo + chunk, nparts);
    const double t = sum_partials<kFinalizeBlock>(parts + lo, hi - lo, lds);
    if (threadIdx.x == 0)
        ws.spmv_partials[blockIdx.x] = t;
}

// x += alpha p, r -= alpha Ap, z = M r, partials of (r.r, r.z).  The
// prologue sums the SpMV's partials into p.Ap and forms alpha; workgroup 0
// records alpha and the values the next kernel must read unchanged (r.z of
// this iterate, `done`, the iteration count).  Each thread loads its first
// rows before that sum, so the L2 round trips of the prologue overlap the
// HBM loads.
template <typename S, int BR, int PREC>
__global__ __launch_bounds__(kBlock) void cg_update_kernel(
    int nrow, const S* __restrict__ prec, S* __restrict__ x, S* __restrict__ r, S* __restrict__ z,
    const S* __restrict__ Ap, int fused, int spmv_parts, CgWs ws
)
{
    __shared__ double lds[kBlock / kWave];
    CgState* state = ws.state;
    const int done = state->done;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        state->rz_prev = state->rz;
        state->done_prev = done;
        if (!done)
            state->iter = (fused ? state->iter_copy : state->iter) + 1;
    }
    if (done)
        return;
    // the direction this iteration's SpMV used (fused: the buffer it wrote)
    const S* __restrict__ p = dir_buffer<S>(ws, fused ? ((state->iter_copy & 1) ^ 1) : 0);
    const int stride = (int)gridDim.x * kBlock;
    int row = (int)(blockIdx.x * kBlock + threadIdx.x);
    S pv[BR], apv[BR], xv[BR], rv0[BR];
    if (row < nrow) {
#pragma unroll
        for (int s = 0; s < BR; ++s) {
            const size_t i = (size_t)row * BR + s;
            pv[s] = p[i];
            apv[s] = Ap[i];
            xv[s] = x[i];
            rv0[s] = r[i];
        }
    }
    double t[1];
    sum_parts<1, kMaxSpmvGrid>(ws.spmv_partials, 0, spmv_parts, lds, t);
    const double a = state->rr > state->atol_sq ? state->rz / t[0] : 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        state->pAp = t[0];
        state->alpha = a;
    }
    const S alpha = (S)a;
    double acc[2] = {0.0, 0.0};
    for (bool first = true; row < nrow; row += stride, first = false) {
        if (!first) {
#pragma unroll
            for (int s = 0; s < BR; ++s) {
                const size_t i = (size_t)row * BR + s;
                pv[s] = p[i];
                apv[s] = Ap[i];
                xv[s] = x[i];
                rv0[s] = r[i];
            }
        }
        S rv[BR], zv[BR];
#pragma unroll
        for (int s = 0; s < BR; ++s) {
            const size_t i = (size_t)row * BR + s;
            x[i] = fma(alpha, pv[s], xv[s]);
            rv[s] = fma(-alpha, apv[s], rv0[s]);
            r[i] = rv[s];
        }
        apply_prec<S, BR, PREC>(prec, row, rv, zv);
#pragma unroll
        for (int s = 0; s < BR; ++s) {
            if (PREC != kPrecNone)
                z[(size_t)row * BR + s] = zv[s];
            acc[0] += (double)rv[s] * (double)rv[s];
            acc[1] += (double)rv[s] * (double)zv[s];
        }
    }
    write_block_partials<kBlock, 2>(acc, ws.upd_partials, lds);
}

// The same pass over scalars in 16-byte vectors, for a point preconditioner (or
// none): each thread loads its next vectors while it stores the current ones.
// Bound by its eight streams (5.5 TB/s at 256^3 FP32); 100^3 FP32 33.4 -> 32.0
// us per iteration against one row per thread.  2048 workgroups, and vectors
// skewed against each other in the workspace, measured the same.
template <typename S, int PREC, bool STREAM>
__global__ __launch_bounds__(kBlock) void cg_update_vec_kernel(
    int64_t n, const S* __restrict__ prec, S* __restrict__ x, S* __restrict__ r, S* __restrict__ z,
    const S* __restrict__ Ap, int spmv_parts, CgWs ws
)
{
    constexpr int kV = 16 / (int)sizeof(S);
    typedef S V __attribute__((ext_vector_type(kV)));
    __shared__ double lds[kBlock / kWave];
    CgState* state = ws.state;
    const int done = state->done;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        state->rz_prev = state->rz;
        state->done_prev = done;
        if (!done)
            state->iter = state->iter + 1;
    }
    if (done)
        return;
    const S* __restrict__ p = dir_buffer<S>(ws, 0);
    const V* __restrict__ pv = reinterpret_cast<const V*>(p);
    const V* __restrict__ av = reinterpret_cast<const V*>(Ap);
    const V* __restrict__ mv = reinterpret_cast<const V*>(prec);
    V* __restrict__ xv = reinterpret_cast<V*>(x);
    V* __restrict__ rv = reinterpret_cast<V*>(r);
    V* __restrict__ zv = reinterpret_cast<V*>(z);
    const int64_t nv = n / kV;
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    V pc = {}, ac = {}, xc = {}, rc = {}, mc = {};
    auto load = [&](int64_t k) {
        pc = pv[k];
        ac = stream_load<STREAM>(av + k);
        xc = stream_load<STREAM>(xv + k);
        rc = stream_load<STREAM>(rv + k);
        if (PREC == kPrecDiag)
            mc = stream_load<STREAM>(mv + k);
    };
    if (i < nv)
        load(i);
    double t[1];
    sum_parts<1, kMaxSpmvGrid>(ws.spmv_partials, 0, spmv_parts, lds, t);
    const double a = state->rr > state->atol_sq ? state->rz / t[0] : 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        state->pAp = t[0];
        state->alpha = a;
    }
    const S alpha = (S)a;
    double acc[2] = {0.0, 0.0};
    for (; i < nv; i += stride) {
        V xn, rn, zn;
#pragma unroll
        for (int k = 0; k < kV; ++k) {
            xn[k] = fma(alpha, pc[k], xc[k]);
            rn[k] = fma(-alpha, ac[k], rc[k]);
            zn[k] = PREC == kPrecDiag ? mc[k] * rn[k] : rn[k];
        }
        if (i + stride < nv)
            load(i + stride);
        stream_store<STREAM>(xn, xv + i);
        stream_store<STREAM && PREC != kPrecNone>(rn, rv + i);  // r is the next direction without one
        if (PREC != kPrecNone)
            zv[i] = zn;
#pragma unroll
        for (int k = 0; k < kV; ++k) {
            acc[0] += (double)rn[k] * (double)rn[k];
            acc[1] += (double)rn[k] * (double)zn[k];
        }
    }
    // the last n % kV entries
    const int64_t j = nv * kV + threadIdx.x;
    if (blockIdx.x == 0 && j < n) {
        x[j] = fma(alpha, p[j], x[j]);
        const S rj = fma(-alpha, Ap[j], r[j]);
        r[j] = rj;
        const S zj = PREC == kPrecDiag ? prec[j] * rj : rj;
        if (PREC != kPrecNone)
            z[j] = zj;
        acc[0] += (double)rj * (double)rj;
        acc[1] += (double)rj * (double)zj;
    }
    write_block_partials<kBlock, 2>(acc, ws.upd_partials, lds);
}

// p = z + beta p (unfused path).  The prologue sums the update's partials
// into r.r and r.z of the new iterate, forms beta and `done`; workgroup 0
// records them.  z and p are 256-byte aligned workspace slices, moved in
// 16-byte vectors (the first ones loaded before the prologue, the next ones
// while the current are stored); one fma per entry, as a scalar loop.
template <typename S, bool STREAM>
__global__ __launch_bounds__(kBlock) void cg_direction_kernel(int64_t n, const S* __restrict__ z, S* __restrict__ p,
                                                              int upd_parts, CgWs ws)
{
    constexpr int kV = 16 / (int)sizeof(S);
    typedef S V __attribute__((ext_vector_type(kV)));
    __shared__ double lds[kBlock / kWave];
    CgState* state = ws.state;
    if (state->done_prev)
        return;
    const V* __restrict__ zv = reinterpret_cast<const V*>(z);
    V* __restrict__ pv = reinterpret_cast<V*>(p);
    const int64_t nv = n / kV;
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    V zc = {}, pc = {};
    if (i < nv) {
        zc = stream_load<STREAM>(zv + i);
        pc = pv[i];
    }
    double t[2];
    sum_parts<2, kMaxVecGrid>(ws.upd_partials, (size_t)upd_parts, upd_parts, lds, t);
    const bool live = t[0] > state->atol_sq;
    const double bt = live ? t[1] / state->rz_prev : 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        state->rr = t[0];
        state->rz = t[1];
        state->beta = bt;
        state->done = !live;
    }
    const S beta = (S)bt;
    for (; i < nv; i += stride) {
        V zn = {}, pn = {};
        if (i + stride < nv) {
            zn = stream_load<STREAM>(zv + i + stride);
            pn = pv[i + stride];
        }
        V o;
#pragma unroll
        for (int k = 0; k < kV; ++k)
            o[k] = fma(beta, pc[k], zc[k]);
        pv[i] = o;
        zc = zn;
        pc = pn;
    }
    // the last n % kV entries
    const int64_t j = nv * kV + threadIdx.x;
    if (blockIdx.x == 0 && j < n)
        p[j] = fma(beta, p[j], z[j]);
}

// Fused path at a residual check: r.r, r.z and `done` of the current iterate
// from the update's partials (the next SpMV recomputes the same sums).
__global__ __launch_bounds__(kBlock) void cg_check_kernel(int upd_parts, CgWs ws)
{
    __shared__ double lds[kBlock / kWave];
    CgState* state = ws.state;
    double t[2];
    sum_parts<2, kMaxVecGrid>(ws.upd_partials, (size_t)upd_parts, upd_parts, lds, t);
    if (threadIdx.x == 0) {
        state->rr = t[0];
        state->rz = t[1];
        state->done = !(t[0] > state->atol_sq);
    }
}

__global__ void cg_state_init_kernel(CgWs ws, double rtol, double atol)
{
    CgState* state = ws.state;
    state->rtol = rtol;
    state->atol = atol;
    state->atol_sq = 0.0;
    state->done = 0;
    state->done_prev = 0;
    state->iter = 0;
    state->iter_copy = 0;
    state->small_window = 0;
    state->small_blocks = 0;
    state->small_done = 0;
}

// ---------------------------------------------------------------------------
// Small systems: all iterations of a solve in one launch
// ---------------------------------------------------------------------------
//
// What bounds a small solve is the latency of two kernels per iteration (2D
// Poisson, 16 K unknowns: 6.1 + 3.8 us and two gaps for 1.2 MB of data).  Here
// N workgroups stay for the whole solve: each keeps its rows' matrix, the p
// entries of the columns they touch (a window of the numbering), x, r and the
// preconditioner in LDS and registers, and an iteration is two all-reductions
// over the workgroups (p.Ap; r.r and r.z) and one exchange of z.  p = z + beta p
// is evaluated by every workgroup for its whole window, so only z travels.  us
// per iteration, two kernels (replayed as graphs) / this: 2D Poisson 128^2 11.3 /
// 6.2, 250^2 12.1 / 8.6, elasticity 12^3 11.1 / 7.1, 7-point 40^3 12.1 / 9.5; what a
// solve costs besides its iterations 230 / 83 us.  The two all-reductions are
// most of what is left.
//
// All-reduction: each workgroup stores its FP64 partial in its own slot with a
// device-scope store; one wave of every workgroup polls all slots until none
// holds the sentinel and adds them in the same order, so all workgroups form
// bit-identical alpha, beta and `done`.  Slots alternate between two sets by the
// iteration's parity.  A workgroup clears its slots of the other set right after
// the p.Ap reduction: there every workgroup has arrived, hence has read that set
// for the last time, and the clear is ordered before the workgroup's r.r / r.z
// partials by the release fence, hence before anyone polls that set again.  z is
// overwritten only after the p.Ap reduction, by when all have read the old one.
//
// All workgroups are resident (SmallShare), and every wait is bounded: a
// workgroup that polls kSmallPolls times leaves without finishing, x is only
// written by cg_small_commit_kernel once all have finished, and the host then
// solves by the kernels above.
constexpr int kSmallThreads = 512;
constexpr int kSmallPer = 2;       // scalars per thread
constexpr int kSmallLds = 144 * 1024;
constexpr int kSmallPolls = 1 << 21;
// Scalars of p that a workgroup's columns may span: it reads z for all of them
// once an iteration.  Random numbering, us per iteration, two kernels / one
// launch: 96^2 FP32 11.5 / 10.3, FP64 12.2 / 10.6; 112^2 12.2 / 12.2, 12.7 / 12.5;
// 128^2 12.2 / 13.9, 12.8 / 12.9.  Systems numbered along their axes span half
// of this at most.
constexpr int kSmallMaxWindow = 12 * 1024;
constexpr unsigned long long kSlotEmpty = 0x7ff8dead00c0ffeeull;  // a NaN no sum stores

// Slot set of quantity q (0 p.Ap, 1 r.r, 2 r.z) and parity.  Every partial is
// stored in kSmallReplicas copies and workgroup w polls copy w % kSmallReplicas:
// polls of one line by every workgroup queue at its memory channel.
__device__ __forceinline__ unsigned long long* small_slots(const CgWs& ws, int replica, int q, int parity)
{
    return ws.small_slots + ((size_t)replica * 6 + q * 2 + parity) * kSmallMaxGroups;
}

// A sum's bits, any NaN as one NaN (never the sentinel).
__device__ __forceinline__ unsigned long long slot_bits(double v)
{
    return v == v ? (unsigned long long)__double_as_longlong(v) : 0x7ff8000000000000ull;
}

// Column window and block count of each workgroup's rows (their maxima go to the
// state, for the LDS the solve needs), and empty slots.  Bound by the latency of
// its column loads, hence 1024 threads with four in flight each.
constexpr int kPlanThreads = 1024;

__global__ __launch_bounds__(kPlanThreads) void cg_small_plan_kernel(int nrow, int rows, const int* __restrict__ offsets,
                                                              const int* __restrict__ columns, CgWs ws)
{
    __shared__ int s_lo, s_hi;
    const int w = blockIdx.x;
    if (threadIdx.x < 6 * kSmallReplicas)
        small_slots(ws, threadIdx.x / 6, threadIdx.x % 6 / 2, threadIdx.x % 2)[w] = kSlotEmpty;
    const int r0 = min(w * rows, nrow), r1 = min(r0 + rows, nrow);
    if (threadIdx.x == 0) {
        s_lo = r0;
        s_hi = r1 - 1;  // the last column
    }
    __syncthreads();
    const int b0 = offsets[r0], b1 = offsets[r1];
    int lo = r0, hi = r1 - 1;
    for (int k = threadIdx.x; k < b1 - b0; k += 4 * kPlanThreads) {
        int c[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            c[u] = k + u * kPlanThreads < b1 - b0 ? columns[b0 + k + u * kPlanThreads] : lo;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            lo = min(lo, c[u]);
            hi = max(hi, c[u]);
        }
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
        lo = min(lo, __shfl_xor(lo, off));
        hi = max(hi, __shfl_xor(hi, off));
    }
    if (threadIdx.x % kWave == 0) {
        atomicMin(&s_lo, lo);
        atomicMax(&s_hi, hi);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        // columns outside the matrix: no window fits (the general kernels take the system as before)
        const bool bad = s_lo < 0 || s_hi >= nrow;
        atomicMax(&ws.state->small_window, bad ? 0x7fffffff : s_hi + 1 - s_lo);
        atomicMax(&ws.state->small_blocks, b1 - b0);
    }
}

// Dynamic LDS of cg_small_kernel, in bytes: offsets, columns, values, p window,
// Ap, r, reductions.
template <typename S, int BR> struct SmallLds {
    size_t off, col, val, p, ap, r, red, bytes;
    __host__ __device__ SmallLds(int rows, int blocks, int window)
    {
        size_t at = 0;
        const auto take = [&](size_t n) {
            const size_t here = at;
            at += (n + 15) / 16 * 16;
            return here;
        };
        off = take(sizeof(int) * (size_t)(rows + 1));
        col = take(sizeof(int) * (size_t)(blocks + 1));
        val = take(sizeof(S) * (size_t)(blocks + 1) * BR * BR);
        p = take(sizeof(S) * (size_t)window * BR);
        ap = take(sizeof(S) * (size_t)rows * BR);
        r = take(sizeof(S) * (size_t)rows * BR);
        red = take(sizeof(double) * 2 * (kSmallThreads / kWave + 1));
        bytes = at;
    }
};

// Sum of each of NV values over all threads of all `n` workgroups, bit-identical
// everywhere; false where `polls` looks at the others' slots did not find them
// all.  ORDER: what the workgroup has stored
// for others is visible to them once they return.
template <int NV, bool ORDER>
__device__ __forceinline__ bool small_all_reduce(double (&v)[NV], int q0, int parity, int n, int polls, const CgWs& ws,
                                                 double* red)
{
    constexpr int kWaves = kSmallThreads / kWave;
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        v[q] = wave_sum(v[q]);
        if (lane == 0)
            red[q * kWaves + wave] = v[q];
    }
    if (ORDER)
        __builtin_amdgcn_s_waitcnt(0);  // this wave's exchanged stores have arrived
    __syncthreads();
    bool ok = true;
    if (wave == 0) {
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            double t = 0.0;
#pragma unroll
            for (int w = 0; w < kWaves; ++w)
                t += red[q * kWaves + w];
            v[q] = t;
        }
        if (n > 1) {
            if (ORDER)
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            if (lane < kSmallReplicas) {
#pragma unroll
                for (int q = 0; q < NV; ++q)
                    store_agent(small_slots(ws, lane, q0 + q, parity) + blockIdx.x, slot_bits(v[q]));
            }
            const int replica = (int)blockIdx.x % kSmallReplicas;
            constexpr int kPer = kSmallMaxGroups / kWave;
            unsigned long long got[NV][kPer] = {};
            for (int look = 0;; ++look) {
                if (look >= polls) {
                    ok = false;
                    break;
                }
                bool ready = true;
#pragma unroll
                for (int q = 0; q < NV; ++q)
#pragma unroll
                    for (int u = 0; u < kPer; ++u) {
                        const int w = lane + u * kWave;
                        got[q][u] = w < n ? load_agent(small_slots(ws, replica, q0 + q, parity) + w) : 0ull;
                        ready = ready && got[q][u] != kSlotEmpty;
                    }
                if (__all(ready))
                    break;
            }
            if (ORDER)
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                double t = 0.0;
#pragma unroll
                for (int u = 0; u < kPer; ++u)
                    t += lane + u * kWave < n ? __longlong_as_double((long long)got[q][u]) : 0.0;
                v[q] = wave_sum(t);
            }
        }
        if (lane == 0) {
#pragma unroll
            for (int q = 0; q < NV; ++q)
                red[NV * kWaves + q] = __longlong_as_double((long long)(ok ? slot_bits(v[q]) : kSlotEmpty));
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        v[q] = red[NV * kWaves + q];
        ok = (unsigned long long)__double_as_longlong(v[q]) != kSlotEmpty;
    }
    __syncthreads();
    return ok;
}

template <typename S, int BR, int G, int PREC>
__global__ __launch_bounds__(kSmallThreads) void cg_small_kernel(
    int nrow, int rows, int max_blocks, int max_window, int maxiter, int polls, const int* __restrict__ offsets,
    const int* __restrict__ columns, const S* __restrict__ values, const S* __restrict__ prec,
    const S* __restrict__ x_in, CgWs ws
)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char small_smem[];
    const SmallLds<S, BR> lay(rows, max_blocks, max_window);
    int* l_off = reinterpret_cast<int*>(small_smem + lay.off);
    int* l_col = reinterpret_cast<int*>(small_smem + lay.col);
    S* l_val = reinterpret_cast<S*>(small_smem + lay.val);
    S* l_p = reinterpret_cast<S*>(small_smem + lay.p);
    S* l_ap = reinterpret_cast<S*>(small_smem + lay.ap);
    S* l_r = reinterpret_cast<S*>(small_smem + lay.r);
    double* red = reinterpret_cast<double*>(small_smem + lay.red);
    const int n = (int)gridDim.x, w = (int)blockIdx.x, tid = (int)threadIdx.x;
    const int r0 = min(w * rows, nrow), r1 = min(r0 + rows, nrow), mine = r1 - r0;
    const int b0 = offsets[r0], nb = offsets[r1] - b0;
    S* zx = static_cast<S*>(ws.p2);  // z, exchanged

    // the window of columns
    int lo = r0, hi = r1;
    for (int b = tid; b < nb; b += kSmallThreads) {
        const int c = columns[b0 + b];
        l_col[b] = c;
        lo = min(lo, c);
        hi = max(hi, c + 1);
    }
    int* span = reinterpret_cast<int*>(red);
    if (tid == 0) {
        span[0] = r0;
        span[1] = r1;
        l_off[0] = 0;
        if (nb == 0) {  // inactive slots of the product read block 0
            l_col[0] = r0;
            for (int e = 0; e < BR * BR; ++e)
                l_val[e] = S(0);
        }
    }
    __syncthreads();
    atomicMin(&span[0], lo);
    atomicMax(&span[1], hi);
    for (int i = tid; i < mine; i += kSmallThreads)
        l_off[i + 1] = offsets[r0 + i + 1] - b0;
    for (int i = tid; i < nb * BR * BR; i += kSmallThreads)
        l_val[i] = values[(size_t)b0 * BR * BR + i];
    __syncthreads();
    lo = span[0];
    const int window = (span[1] - lo) * BR;
    for (int b = tid; b < max(nb, 1); b += kSmallThreads)
        l_col[b] -= lo;
    const S* p_in = static_cast<const S*>(ws.p);
    for (int i = tid; i < window; i += kSmallThreads)
        l_p[i] = p_in[(size_t)lo * BR + i];

    // own scalars i = tid + u * kSmallThreads of rows r0 .. r1 - 1
    const int own = mine * BR;
    const S* r_in = static_cast<const S*>(ws.r);
    S x[kSmallPer], r[kSmallPer], m[kSmallPer][PREC == kPrecBlock ? BR : 1];
#pragma unroll
    for (int u = 0; u < kSmallPer; ++u) {
        const int i = tid + u * kSmallThreads;
        const size_t g = (size_t)r0 * BR + i;
        x[u] = i < own ? x_in[g] : S(0);
        r[u] = i < own ? r_in[g] : S(0);
        if (PREC == kPrecDiag)
            m[u][0] = i < own ? prec[g] : S(0);
        if constexpr (PREC == kPrecBlock)
#pragma unroll
            for (int c = 0; c < BR; ++c)
                m[u][c] = i < own ? prec[g * BR + c] : S(0);
    }
    const double atol_sq = ws.state->atol_sq;
    double rr = ws.state->rr, rz = ws.state->rz, alpha = 0.0, beta = 0.0, pap = 0.0;
    const S* l_pown = l_p + (size_t)(r0 - lo) * BR;
    int it = 0;
    bool ok = true;
    __syncthreads();
    while (rr > atol_sq && it < maxiter) {
        const int parity = it & 1;
        // Ap
        constexpr int RPG = rows_per_group_for(BR, BR);
        for (int row = tid / G * RPG; row < mine; row += kSmallThreads / G * RPG) {
            const RowAcc<S, BR * RPG> a = group_rows_product_f<S, BR, BR, G, RPG, S>(
                row, mine, tid % G, l_off, nullptr, l_col, l_val, LoadX<S>{l_p});
            for (int e = tid % G; e < BR * RPG && row + e / BR < mine; e += G)
                l_ap[row * BR + e] = pick(a, e);
        }
        __syncthreads();
        double s1[1] = {0.0};
#pragma unroll
        for (int u = 0; u < kSmallPer; ++u) {
            const int i = tid + u * kSmallThreads;
            if (i < own)
                s1[0] += (double)l_pown[i] * (double)l_ap[i];
        }
        ok = small_all_reduce<1, false>(s1, 0, parity, n, polls, ws, red);
        if (!ok)
            return;
        if (tid < 3 * kSmallReplicas && n > 1)  // everyone has read the other set for the last time
            store_agent(small_slots(ws, tid / 3, tid % 3, parity ^ 1) + w, kSlotEmpty);
        pap = s1[0];
        alpha = rz / pap;
        const S al = (S)alpha;
#pragma unroll
        for (int u = 0; u < kSmallPer; ++u) {
            const int i = tid + u * kSmallThreads;
            if (i < own) {
                x[u] = fma(al, l_pown[i], x[u]);
                r[u] = fma(-al, l_ap[i], r[u]);
                if constexpr (PREC == kPrecBlock)
                    l_r[i] = r[u];
            }
        }
        if constexpr (PREC == kPrecBlock)
            __syncthreads();
        double s2[2] = {0.0, 0.0};
#pragma unroll
        for (int u = 0; u < kSmallPer; ++u) {
            const int i = tid + u * kSmallThreads;
            if (i < own) {
                S z = r[u];
                if (PREC == kPrecDiag)
                    z = m[u][0] * r[u];
                if constexpr (PREC == kPrecBlock) {
                    z = S(0);
#pragma unroll
                    for (int c = 0; c < BR; ++c)
                        z = fma(m[u][c], l_r[i - i % BR + c], z);
                }
                store_agent(zx + (size_t)r0 * BR + i, z);
                s2[0] += (double)r[u] * (double)r[u];
                s2[1] += (double)r[u] * (double)z;
            }
        }
        ok = small_all_reduce<2, true>(s2, 1, parity, n, polls, ws, red);
        if (!ok)
            return;
        rr = s2[0];
        ++it;
        if (!(rr > atol_sq) || it >= maxiter) {
            rz = s2[1];
            break;
        }
        beta = s2[1] / rz;
        rz = s2[1];
        const S be = (S)beta;
        for (int i = tid; i < window; i += kSmallThreads)
            l_p[i] = fma(be, l_p[i], load_agent(zx + (size_t)lo * BR + i));
        __syncthreads();
    }
    S* out = static_cast<S*>(ws.Ap);
#pragma unroll
    for (int u = 0; u < kSmallPer; ++u) {
        const int i = tid + u * kSmallThreads;
        if (i < own)
            out[(size_t)r0 * BR + i] = x[u];
    }
    if (tid == 0) {
        if (w == 0) {
            CgState* state = ws.state;
            state->rr = rr;
            state->rz = rz;
            state->alpha = alpha;
            state->beta = beta;
            state->pAp = pap;
            state->iter = it;
            state->iter_copy = it;
            state->done = !(rr > atol_sq);
        }
        atomicAdd(&ws.state->small_done, 1);
    }
}

// x = the solution, if every workgroup of cg_small_kernel finished
template <typename S>
__global__ __launch_bounds__(kBlock) void cg_small_commit_kernel(int n, int groups, S* __restrict__ x, CgWs ws)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n && ws.state->small_done == groups)
        x[i] = static_cast<const S*>(ws.Ap)[i];
}

// ---------------------------------------------------------------------------
// Host driver
// ---------------------------------------------------------------------------

// Tolerance defaults (linear.py:2010-2032); NaN stands for None.
void get_tolerances(bool is_f64, double tol, double atol, double* rtol_out, double* atol_out)
{
    const double eps = is_f64 ? 1.0e-16 : 1.0e-8;
    const double default_tol = std::pow(eps, 0.75);
    const double min_tol = std::pow(eps, 2.25);
    if (std::isnan(tol) && std::isnan(atol)) {
        tol = atol = default_tol;
    } else if (std::isnan(tol)) {
        tol = atol;
    } else if (std::isnan(atol)) {
        atol = tol;
    }
    *rtol_out = tol;
    *atol_out = std::max(atol, min_tol);
}

// Pinned staging for state read-backs; one per host thread, kept for the
// life of the process (freeing it at thread exit could race runtime teardown).
struct PinnedState {
    CgState* host = nullptr;
};

int read_state(const CgState* dev, CgState* out, hipStream_t stream)
{
    static thread_local PinnedState pinned;
    if (!pinned.host)
        WA_HIP(hipHostMalloc((void**)&pinned.host, sizeof(CgState), hipHostMallocDefault));
    WA_HIP(hipMemcpyAsync(pinned.host, dev, sizeof(CgState), hipMemcpyDeviceToHost, stream));
    WA_HIP(hipStreamSynchronize(stream));
    *out = *pinned.host;
    return kOk;
}

int group_for_square(int64_t nnz_hint, int nrow, int br) { return bsr_mv_lanes(nrow, br, br, nnz_hint); }

typedef int (*CgCallback)(int iteration, double err, double atol, void* user);

struct CgProblem {
    int nrow;
    int br;
    const int* offsets;
    const int* columns;
    const void* values;
    int64_t nnz_hint;
    int prec_kind;
    const void* prec;
    const void* b;
    void* x;
};

template <typename S> struct CgLauncher {
    CgProblem pb;
    CgWs ws;
    hipStream_t stream;
    // Direction pass folded into the SpMV (small systems).
    bool fused = false;

    const S* z_vec() const { return pb.prec_kind != kPrecNone ? (const S*)ws.z : (const S*)ws.r; }

    template <int BR, int G> unsigned rows_grid() const
    {
        return (unsigned)ceil_div(pb.nrow, (kBlock / G) * rows_per_group_for(BR, BR));
    }
    // Very large unfused systems: one workgroup per tile, the partials then
    // reduced to kWideParts by a small kernel (256^3 7-point operator, 65,536 tiles:
    // FP32 inner CG iteration 423 -> 391 us); otherwise at most kMaxSpmvGrid
    // persistent workgroups whose partials the update sums in its prologue
    // (64^3 3x3 elasticity, 17,164 tiles: 66 us per iteration, 71 with the wide grid).
    static constexpr unsigned kWideSpmvTiles = 16u * kMaxSpmvGrid;
    template <int BR, int G> bool wide_spmv() const
    {
        return !fused && (rows_grid<BR, G>() > kWideSpmvTiles || wave_spmv<BR, G>());
    }
    static constexpr int kWaveRW = sizeof(S) == 4 ? 64 : 32, kWaveCH = sizeof(S) == 4 ? 2 : 1;
    template <int BR, int G> bool wave_spmv() const
    {
        // 65^3 FP64 23.9 us per iteration, 24.9 by wave tiles (their partials take a
        // launch more), 100^3 45.1 / 42.7, 128^3 84.9 / 70
        return !fused && BR == 1 && G == 4 && pb.nrow >= (1 << 19) &&
               wave_rows_supported(G, pb.nrow, pb.nnz_hint, sizeof(S) == 8, nullptr, pb.columns, pb.values);
    }
    // What bypasses the caches (256 MB memory-side).  The matrix, where it is
    // twice that: a product cannot start on what the last one left, and p, Ap
    // and z stay for the next pass (256^3 FP32 348 -> 337 us per iteration; a
    // 420 MB FP64 matrix 194 -> 207, so not below).  x, r and the
    // preconditioner, touched once per iteration, where an iteration's matrix
    // and vectors exceed it and a vector its L2 (256^3 FP32 366 -> 337 us,
    // 160^3 90 -> 84, 128^3 FP64 77 -> 73; 128^3 FP32, 167 MB in all, 49 -> 55,
    // so not below).
    int64_t matrix_bytes() const { return pb.nnz_hint * (int64_t)(sizeof(int) + pb.br * pb.br * sizeof(S)); }
    int64_t vector_bytes() const { return (int64_t)pb.nrow * pb.br * (int64_t)sizeof(S); }
    bool stream_matrix() const { return matrix_bytes() > ((int64_t)512 << 20); }
    bool stream_vectors() const
    {
        return vector_bytes() > ((int64_t)8 << 20) && matrix_bytes() + 6 * vector_bytes() > ((int64_t)256 << 20);
    }
    template <int BR, int G> unsigned spmv_grid() const
    {
        if (wave_spmv<BR, G>())
            return (unsigned)ceil_div(pb.nrow, (kBlock / kWave) * kWaveRW);
        return wide_spmv<BR, G>() ? rows_grid<BR, G>() : std::min<unsigned>(rows_grid<BR, G>(), (unsigned)kMaxSpmvGrid);
    }
    // partials the update reads
    template <int BR, int G> unsigned spmv_parts() const
    {
        return wide_spmv<BR, G>() ? (unsigned)kWideParts : spmv_grid<BR, G>();
    }
    static unsigned vec_grid(int64_t count)
    {
        return (unsigned)std::max<int64_t>(1, std::min<int64_t>(ceil_div(count, kBlock), kMaxVecGrid));
    }
    // The update in 16-byte vectors: unfused, point preconditioner, x and the
    // preconditioner aligned (the workspace vectors are).
    bool vec_update() const
    {
        return !fused && pb.prec_kind != kPrecBlock && (((uintptr_t)pb.x | (uintptr_t)pb.prec) & 15) == 0;
    }
    // workgroups (= partials) of the update pass: one thread per vector or block row
    unsigned upd_grid() const
    {
        return vec_update() ? vec_grid(ceil_div((int64_t)pb.nrow * pb.br, 16 / (int)sizeof(S))) : vec_grid(pb.nrow);
    }

    template <int BR, int G, int PREC> int init_t(int first)
    {
        const unsigned grid = rows_grid<BR, G>();
        cg_init_kernel<S, BR, G, PREC><<<grid, kBlock, 0, stream>>>(
            pb.nrow, pb.offsets, pb.columns, (const S*)pb.values, (const S*)pb.prec, (const S*)pb.b,
            (const S*)pb.x, (S*)ws.r, (S*)ws.z, fused ? 1 : 0, ws
        );
        WA_LAUNCH_CHECK();
        cg_init_finalize_kernel<<<1, kFinalizeBlock, 0, stream>>>(
            ws, (int)grid, (int)upd_grid(), pb.prec_kind != kPrecNone ? 1 : 0, first, fused ? 1 : 0
        );
        WA_LAUNCH_CHECK();
        return kOk;
    }
    template <int BR, int G> int spmv_t()
    {
        const unsigned grid = spmv_grid<BR, G>();
        if (fused) {
            cg_spmv_kernel<S, BR, G, true><<<grid, kBlock, 0, stream>>>(
                pb.nrow, pb.offsets, pb.columns, (const S*)pb.values, z_vec(), (S*)ws.Ap, (int)upd_grid(), ws,
                ws.spmv_partials
            );
            WA_LAUNCH_CHECK();
            return kOk;
        }
        // the wide grid's partials go to the initial residual's partial buffer
        // (unused between restarts; it holds one per workgroup of any row grid)
        double* parts = wide_spmv<BR, G>() ? ws.init_partials : ws.spmv_partials;
        if constexpr (BR == 1 && G == 4) {
            if (wave_spmv<BR, G>()) {
                if (stream_matrix())
                    cg_spmv_wave_kernel<S, G, kWaveRW, kWaveCH, true><<<grid, kBlock, 0, stream>>>(
                        pb.nrow, pb.offsets, pb.columns, (const S*)pb.values, (S*)ws.Ap, ws, parts);
                else
                    cg_spmv_wave_kernel<S, G, kWaveRW, kWaveCH, false><<<grid, kBlock, 0, stream>>>(
                        pb.nrow, pb.offsets, pb.columns, (const S*)pb.values, (S*)ws.Ap, ws, parts);
                WA_LAUNCH_CHECK();
                cg_wide_spmv_finalize_kernel<<<kWideParts, kFinalizeBlock, 0, stream>>>(parts, (int)grid, ws);
                WA_LAUNCH_CHECK();
                return kOk;
            }
        }
        cg_spmv_kernel<S, BR, G, false><<<grid, kBlock, 0, stream>>>(
            pb.nrow, pb.offsets, pb.columns, (const S*)pb.values, nullptr, (S*)ws.Ap, (int)upd_grid(), ws, parts
        );
        WA_LAUNCH_CHECK();
        if (wide_spmv<BR, G>()) {
            cg_wide_spmv_finalize_kernel<<<kWideParts, kFinalizeBlock, 0, stream>>>(parts, (int)grid, ws);
            WA_LAUNCH_CHECK();
        }
        return kOk;
    }
    template <int BR, int PREC> int update_t()
    {
        unsigned spmv_parts = 0;
#define WA_SPMV_PARTS(BR_, G) spmv_parts = this->template spmv_parts<BR_, G>(); break;
        switch (g()) {
        case 1: WA_SPMV_PARTS(BR, 1)
        case 2: WA_SPMV_PARTS(BR, 2)
        case 4: WA_SPMV_PARTS(BR, 4)
        case 8: WA_SPMV_PARTS(BR, 8)
        case 16: WA_SPMV_PARTS(BR, 16)
        case 32: WA_SPMV_PARTS(BR, 32)
        default: WA_SPMV_PARTS(BR, 64)
        }
#undef WA_SPMV_PARTS
        if constexpr (PREC != kPrecBlock) {
            if (vec_update()) {
                const int64_t n = (int64_t)pb.nrow * BR;
                if (stream_vectors())
                    cg_update_vec_kernel<S, PREC, true><<<upd_grid(), kBlock, 0, stream>>>(
                        n, (const S*)pb.prec, (S*)pb.x, (S*)ws.r, (S*)ws.z, (const S*)ws.Ap, (int)spmv_parts, ws);
                else
                    cg_update_vec_kernel<S, PREC, false><<<upd_grid(), kBlock, 0, stream>>>(
                        n, (const S*)pb.prec, (S*)pb.x, (S*)ws.r, (S*)ws.z, (const S*)ws.Ap, (int)spmv_parts, ws);
                WA_LAUNCH_CHECK();
                return kOk;
            }
        }
        cg_update_kernel<S, BR, PREC><<<upd_grid(), kBlock, 0, stream>>>(
            pb.nrow, (const S*)pb.prec, (S*)pb.x, (S*)ws.r, (S*)ws.z, (const S*)ws.Ap, fused ? 1 : 0, (int)spmv_parts,
            ws
        );
        WA_LAUNCH_CHECK();
        return kOk;
    }

    int g() const { return group_for_square(pb.nnz_hint, pb.nrow, pb.br); }

#define WA_CG_DISPATCH_G(BR, CALL)                                                                                    \
    switch (g()) {                                                                                                    \
    case 1: return CALL(BR, 1);                                                                                       \
    case 2: return CALL(BR, 2);                                                                                       \
    case 4: return CALL(BR, 4);                                                                                       \
    case 8: return CALL(BR, 8);                                                                                       \
    case 16: return CALL(BR, 16);                                                                                     \
    case 32: return CALL(BR, 32);                                                                                     \
    default: return CALL(BR, 64);                                                                                     \
    }

    int init(int first)
    {
#define WA_INIT_CALL(BR, G) init_prec<BR, G>(first)
        if (pb.br == 1) {
            WA_CG_DISPATCH_G(1, WA_INIT_CALL)
        }
        WA_CG_DISPATCH_G(3, WA_INIT_CALL)
#undef WA_INIT_CALL
    }
    template <int BR, int G> int init_prec(int first)
    {
        switch (pb.prec_kind) {
        case kPrecDiag: return init_t<BR, G, kPrecDiag>(first);
        case kPrecBlock: return init_t<BR, G, kPrecBlock>(first);
        default: return init_t<BR, G, kPrecNone>(first);
        }
    }
    int spmv()
    {
#define WA_SPMV_CALL(BR, G) spmv_t<BR, G>()
        if (pb.br == 1) {
            WA_CG_DISPATCH_G(1, WA_SPMV_CALL)
        }
        WA_CG_DISPATCH_G(3, WA_SPMV_CALL)
#undef WA_SPMV_CALL
    }
    int update()
    {
        if (pb.br == 1) {
            switch (pb.prec_kind) {
            case kPrecDiag: return update_t<1, kPrecDiag>();
            case kPrecBlock: return update_t<1, kPrecBlock>();
            default: return update_t<1, kPrecNone>();
            }
        }
        switch (pb.prec_kind) {
        case kPrecDiag: return update_t<3, kPrecDiag>();
        case kPrecBlock: return update_t<3, kPrecBlock>();
        default: return update_t<3, kPrecNone>();
        }
    }
#undef WA_CG_DISPATCH_G

    int direction()
    {
        const int64_t n = (int64_t)pb.nrow * pb.br;
        if (stream_vectors() && pb.prec_kind != kPrecNone)
            cg_direction_kernel<S, true><<<vec_grid(n), kBlock, 0, stream>>>(n, z_vec(), (S*)ws.p, (int)upd_grid(), ws);
        else
            cg_direction_kernel<S, false><<<vec_grid(n), kBlock, 0, stream>>>(n, z_vec(), (S*)ws.p, (int)upd_grid(), ws);
        WA_LAUNCH_CHECK();
        return kOk;
    }

    // Makes the state's r.r and `done` current before the host reads them
    // (the fused path leaves the last update's sums in its partials).
    int check()
    {
        if (!fused)
            return kOk;
        cg_check_kernel<<<1, kBlock, 0, stream>>>((int)upd_grid(), ws);
        WA_LAUNCH_CHECK();
        return kOk;
    }

    // last_in_cycle: a restart follows, which sets p = z itself.
    int iteration(bool last_in_cycle)
    {
        WA_TRY(spmv());
        WA_TRY(update());
        if (!fused && !last_in_cycle)
            WA_TRY(direction());
        return kOk;
    }
};

// Runs the solver's cycles on a private stream and, with graphs on, replays
// each group of cycles between two residual checks as one HIP graph (the
// reference captures its iterations in CUDA graphs, linear.py:2205-2215).  The caller's stream may be the legacy
// default stream, which cannot be captured, hence the private stream; it
// starts after the caller's pending work and the caller's stream waits for
// it at the end.  A failed capture falls back to eager launches.
struct CycleRunner {
    hipStream_t caller;
    hipStream_t ps = nullptr;
    hipEvent_t ev = nullptr;
    hipGraphExec_t exec = nullptr;
    bool graph_ok = false;

    CycleRunner(hipStream_t s, bool use_graph) : caller(s)
    {
        if (!use_graph)
            return;
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(s, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) {
            (void)hipGetLastError();
            return;  // already inside the caller's capture: launch into it
        }
        if (hipStreamCreateWithFlags(&ps, hipStreamNonBlocking) != hipSuccess ||
            hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess ||
            hipEventRecord(ev, caller) != hipSuccess || hipStreamWaitEvent(ps, ev, 0) != hipSuccess) {
            (void)hipGetLastError();
            release();
            return;
        }
        graph_ok = true;
    }
    ~CycleRunner()
    {
        if (ps) {
            // everything enqueued here precedes the caller's later work; the
            // graph is destroyed only once it has run
            if (hipEventRecord(ev, ps) == hipSuccess)
                (void)hipStreamWaitEvent(caller, ev, 0);
            (void)hipStreamSynchronize(ps);
        }
        release();
    }
    void release()
    {
        if (exec)
            (void)hipGraphExecDestroy(exec);
        if (ps)
            (void)hipStreamDestroy(ps);
        if (ev)
            (void)hipEventDestroy(ev);
        exec = nullptr;
        ps = nullptr;
        ev = nullptr;
    }
    hipStream_t stream() const { return ps ? ps : caller; }

    // `count` cycles of `body`; with graph = true they are one replayable
    // graph (always the same count: the group between two residual checks).
    template <typename F> int run(F&& body, int count, bool graph)
    {
        auto eager = [&]() -> int {
            for (int c = 0; c < count; ++c)
                WA_TRY(body());
            return kOk;
        };
        if (!graph || !graph_ok)
            return eager();
        if (exec) {
            WA_HIP(hipGraphLaunch(exec, ps));
            return kOk;
        }
        hipGraph_t g = nullptr;
        if (hipStreamBeginCapture(ps, hipStreamCaptureModeRelaxed) != hipSuccess) {
            (void)hipGetLastError();
            graph_ok = false;
            return eager();
        }
        const int st = eager();
        const hipError_t e = hipStreamEndCapture(ps, &g);
        if (st != kOk) {
            if (g)
                (void)hipGraphDestroy(g);
            return st;
        }
        hipError_t ie = e;
        if (e == hipSuccess && g)
            ie = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
        if (g)
            (void)hipGraphDestroy(g);
        if (e != hipSuccess || !g || ie != hipSuccess) {
            (void)hipGetLastError();
            exec = nullptr;
            graph_ok = false;
            return eager();  // nothing of the capture ran: run the cycles eagerly
        }
        WA_HIP(hipGraphLaunch(exec, ps));
        return kOk;
    }
};

// Number of workgroups of cg_small_kernel for a system (a power of two; 0: not
// small): 32 KB of matrix each until there are 128, then up to 96 KB.  us per
// iteration at 24 / 32 / 48 KB: 2D Poisson 128^2 6.20 / 6.18 / 6.76, 64^2 5.4 / 5.4 /
// 6.2, 12^3 elasticity 7.9 / 7.1 / 7.2; 128 workgroups against 256: 2D Poisson
// 250^2 8.6 / 10.8, 18^3 elasticity 9.7 / 11.6 (the all-reductions grow with their
// number).
template <typename S> int small_groups(const CgProblem& pb)
{
    const int64_t n = (int64_t)pb.nrow * pb.br;
    const int64_t matrix = pb.nnz_hint * (int64_t)(sizeof(int) + pb.br * pb.br * sizeof(S));
    if (n * (int64_t)sizeof(S) > (int64_t)kFusedDirectionMaxBytes || matrix > (int64_t)kSmallMaxGroups * 96 * 1024)
        return 0;
    int g = 1;
    while (g < kSmallMaxGroups && ((int64_t)g * 32 * 1024 < matrix || (int64_t)g * kSmallThreads < n))
        g *= 2;
    return ceil_div(pb.nrow, g) * pb.br <= kSmallThreads * kSmallPer ? g : 0;
}

// The kernel of a block size, lanes per row and preconditioner; null where it is
// not compiled: each form is a kernel of its own, so only the rows that grids and
// meshes give have one (means above 2 and up to 32 entries of scalar rows, above 4
// and up to 32 blocks of 3x3 rows); nearly diagonal and nearly dense systems stay
// with the general kernels.
template <typename S> const void* small_kernel(int br, int lanes, int prec)
{
#define WA_SMALL_PREC(BR, G)                                                                                          \
    if (br == BR && lanes == G) {                                                                                     \
        if (prec == kPrecNone)                                                                                        \
            return (const void*)cg_small_kernel<S, BR, G, kPrecNone>;                                                 \
        if (prec == kPrecDiag || BR == 1) /* a 1x1 block is a point */                                                \
            return (const void*)cg_small_kernel<S, BR, G, kPrecDiag>;                                                 \
        return (const void*)cg_small_kernel<S, BR, G, BR == 1 ? kPrecDiag : kPrecBlock>;                              \
    }
    WA_SMALL_PREC(1, 2)
    WA_SMALL_PREC(1, 4)
    WA_SMALL_PREC(1, 8)
    WA_SMALL_PREC(1, 16)
    WA_SMALL_PREC(3, 8)
    WA_SMALL_PREC(3, 16)
    WA_SMALL_PREC(3, 32)
#undef WA_SMALL_PREC
    return nullptr;
}

// What the one-launch solves in flight hold of a device.  Cooperative launches
// of one process run one after another, whatever their streams (2D Poisson 128^2,
// 80 iterations, eight threads: 511 us a solve, 332 by the general kernels, whose
// launches overlap).  So only a solve with no other in flight is launched
// cooperatively; the others are ordinary launches, resident all the same because
// of what may be in flight at once: one workgroup for each compute unit, or two
// where every workgroup in flight is one of which three fit (a unit that holds
// one of them has room for another, wherever in its LDS and registers the first
// lies).  Launches are dealt evenly to the XCDs, and any other kernel on the
// device ends by itself, after which its units are free.  Further solves wait
// here, in order of arrival; those inside entered with their streams drained, so
// they always end.  us a solve of 80 iterations with 1 / 2 / 4 / 8 threads, by the
// general kernels: 64^2 1113 / 667 / 381 / 310, 128^2 1108 / 656 / 381 / 321,
// 250^2 1236 / 704 / 441 / 398; all cooperative: 535 / 454 / 444 / 440, 593 / 520 /
// 511 / 511, 799 / 721 / 712 / 711; so: 570 / 287 / 193 / 179, 577 / 432 / 256 /
// 250, 801 / 489 / 395 / 393.
class SmallShare {
    struct Device {
        std::mutex lock;
        std::condition_variable left;
        uint64_t arrived = 0, entered = 0;
        int held = 0;   // workgroups in flight
        int whole = 0;  // those of which fewer than three fit a compute unit
    };
    static constexpr int kMaxDevices = 64;
    static Device& device(int id)
    {
        static Device* devices = new Device[kMaxDevices];  // never freed: threads may still solve at exit
        return devices[id];
    }
    Device* dev = nullptr;
    int share = 0, whole = 0;

public:
    bool alone = false;

    // false: not on this device (the caller takes the general kernels)
    bool enter(int groups, const void* kernel, size_t lds)
    {
        int id = 0, units = 0, per_unit = 0;
        if (hipGetDevice(&id) != hipSuccess || id < 0 || id >= kMaxDevices ||
            hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, id) != hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_unit, kernel, kSmallThreads, lds) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        // whole eighths: the workgroups of a launch are dealt to 8 XCDs
        const int need = (groups + 7) / 8 * 8;
        if (need > units || per_unit < 1)
            return false;
        Device& d = device(id);
        std::unique_lock<std::mutex> hold(d.lock);
        const uint64_t ticket = d.arrived++;
        d.left.wait(hold, [&] {
            return ticket == d.entered && d.held + need <= (per_unit > 2 && d.whole == 0 ? 2 * units : units);
        });
        ++d.entered;
        alone = d.held == 0;
        dev = &d;
        share = need;
        whole = per_unit > 2 ? 0 : need;
        d.held += share;
        d.whole += whole;
        d.left.notify_all();
        return true;
    }
    SmallShare() = default;
    SmallShare(const SmallShare&) = delete;
    SmallShare& operator=(const SmallShare&) = delete;
    ~SmallShare()
    {
        if (!dev)
            return;
        std::lock_guard<std::mutex> hold(dev->lock);
        dev->held -= share;
        dev->whole -= whole;
        dev->left.notify_all();
    }
};

// Solves by cg_small_kernel where the system fits; *solved = 0 with x untouched
// otherwise.  *initial then says whether the workspace holds the solve's initial
// state (read back into *h) for the general kernels to go on from: so it is
// where only the columns' window did not fit, and the one thing such a solve
// pays is cg_small_plan_kernel (2D Poisson 250^2 in random numbering, 10
// iterations: 383 us by the general kernels alone, 386 now; 412 against 347
// when they began again).  The caller's stream is not capturing (the state is
// read back).
template <typename S>
int cg_solve_small(CgLauncher<S>& L, double rtol, double atol, int maxiter, int check_every, int polls, CgState* h,
                   int* cur_iter, int* solved, int* initial)
{
    *solved = *initial = 0;
    const CgProblem& pb = L.pb;
    const int groups = small_groups<S>(pb);
    const void* kernel = groups ? small_kernel<S>(pb.br, L.g(), pb.prec_kind) : nullptr;
    if (!kernel)
        return kOk;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(L.stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return kOk;
    }
    int rows = (int)ceil_div(pb.nrow, groups);
    cg_state_init_kernel<<<1, 1, 0, L.stream>>>(L.ws, rtol, atol);
    WA_LAUNCH_CHECK();
    WA_TRY(L.init(1));
    cg_small_plan_kernel<<<groups, kPlanThreads, 0, L.stream>>>(pb.nrow, rows, pb.offsets, pb.columns, L.ws);
    WA_LAUNCH_CHECK();
    WA_TRY(read_state(L.ws.state, h, L.stream));
    *initial = 1;
    *cur_iter = 0;
    if (h->rr <= h->atol_sq) {
        *solved = 1;
        return kOk;
    }
    if ((int64_t)h->small_window * pb.br > kSmallMaxWindow)
        return kOk;
    const size_t lds = pb.br == 1 ? SmallLds<S, 1>(rows, h->small_blocks, h->small_window).bytes
                                  : SmallLds<S, 3>(rows, h->small_blocks, h->small_window).bytes;
    if (lds > (size_t)kSmallLds)
        return kOk;
    const int n = pb.nrow * pb.br;
    int nrow = pb.nrow, blocks = h->small_blocks, window = h->small_window;
    const S *values = (const S*)pb.values, *prec = (const S*)pb.prec, *x = (const S*)pb.x;
    const int *offsets = pb.offsets, *columns = pb.columns;
    void* args[] = {&nrow, &rows, &blocks, &window, &maxiter, &polls, &offsets, &columns, &values, &prec, &x, &L.ws};
    SmallShare share;  // until the solve has ended (read_state below)
    const dim3 grid((unsigned)groups), block(kSmallThreads);
    if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kSmallLds) != hipSuccess ||
        !share.enter(groups, kernel, lds) ||
        (share.alone ? hipLaunchCooperativeKernel(kernel, grid, block, args, (unsigned)lds, L.stream)
                     : hipLaunchKernel(kernel, grid, block, args, lds, L.stream)) != hipSuccess) {
        (void)hipGetLastError();  // does not fit this device: the general kernels
        return kOk;
    }
    *initial = 0;  // z, Ap and the state are written from here on
    cg_small_commit_kernel<S><<<(unsigned)ceil_div(n, kBlock), kBlock, 0, L.stream>>>(n, groups, (S*)pb.x, L.ws);
    WA_LAUNCH_CHECK();
    WA_TRY(read_state(L.ws.state, h, L.stream));
    if (h->small_done != groups)
        return kOk;
    // as the host loop counts: whole groups of check_every, and to the end on NaN
    *cur_iter = h->rr <= h->atol_sq ? (int)std::min<int64_t>(maxiter, ceil_div(h->iter, check_every) * check_every) : maxiter;
    *solved = 1;
    return kOk;
}

template <typename S>
int cg_solve_impl(
    const CgProblem& pb, double tol, double atol, int maxiter, int check_every, int restart, int use_graph,
    CgCallback cb, void* cb_user, void* workspace, size_t workspace_bytes, int* iters_out, double* rnorm_out,
    double* atol_out, hipStream_t caller_stream, int polls = kSmallPolls
)
{
    WA_REQUIRE(pb.br == 1 || pb.br == 3, "cg_solve: block size must be 1 or 3, got %d", pb.br);
    WA_REQUIRE(pb.prec_kind >= 0 && pb.prec_kind <= 2, "cg_solve: invalid preconditioner kind %d", pb.prec_kind);
    WA_REQUIRE(pb.prec_kind == kPrecNone || pb.prec, "cg_solve: null preconditioner data");
    const int64_t n = (int64_t)pb.nrow * pb.br;
    WA_REQUIRE(pb.nrow > 0, "cg_solve: empty system");
    size_t needed = 0;
    CgWs ws = carve_cg(workspace, workspace_bytes, pb.nrow, n, sizeof(S), &needed);
    WA_REQUIRE(workspace && needed <= workspace_bytes, "cg_solve: workspace too small (%zu < %zu bytes)",
               workspace_bytes, needed);
    // the vector passes move workspace slices in 16-byte vectors
    WA_REQUIRE((uintptr_t)workspace % 16 == 0, "cg_solve: workspace must be 16-byte aligned");
    if (maxiter <= 0)
        maxiter = (int)n;

    double rtol_v, atol_v;
    get_tolerances(sizeof(S) == 8, tol, atol, &rtol_v, &atol_v);
    CgState h;
    int initial = 0;  // the state, r, z and p of the initial residual are there, and h holds the state
    if (check_every > 0 && restart <= 0 && !cb) {
        CgLauncher<S> small{pb, ws, caller_stream};
        small.fused = true;
        int cur_iter = 0, solved = 0;
        WA_TRY(cg_solve_small(small, rtol_v, atol_v, maxiter, check_every, polls, &h, &cur_iter, &solved, &initial));
        if (solved) {
            if (iters_out)
                *iters_out = cur_iter;
            if (rnorm_out)
                *rnorm_out = std::sqrt(h.rr);
            if (atol_out)
                *atol_out = std::sqrt(h.atol_sq);
            return kOk;
        }
    }

    // graphs only where launches bound the iteration: measured on MI355X,
    // replaying the cycles between two checks as one graph gave 2D Poisson
    // (16 K dofs) 19 -> 17 us per iteration but the 3x3 elasticity system
    // (824 K dofs) 78.6 -> 79.6 us, and one graph per iteration was slower for both
    CycleRunner runner(caller_stream, use_graph != 0 && (size_t)n * sizeof(S) <= kFusedDirectionMaxBytes);
    const hipStream_t stream = runner.stream();
    CgLauncher<S> L{pb, ws, stream};
    L.fused = (size_t)n * sizeof(S) <= kFusedDirectionMaxBytes;

    int cycle = 1;
    if (restart > 0) {
        cycle = std::max(1, std::min(restart, maxiter));
        if (check_every > 0)
            check_every = std::max(check_every, cycle);
    }

    if (!initial) {
        cg_state_init_kernel<<<1, 1, 0, stream>>>(ws, rtol_v, atol_v);
        WA_LAUNCH_CHECK();
        WA_TRY(L.init(1));
    }

    auto cycle_body = [&]() -> int {
        for (int k = 0; k < cycle; ++k)
            WA_TRY(L.iteration(restart > 0 && k == cycle - 1));
        if (restart > 0)
            WA_TRY(L.init(0));
        return kOk;
    };
    // k cycles, then the state made current for the host's read-back
    auto group_of = [&](int k) {
        return [&, k]() -> int {
            for (int c = 0; c < k; ++c)
                WA_TRY(cycle_body());
            return L.check();
        };
    };
    auto run_cycle = [&]() -> int { return runner.run(group_of(1), 1, false); };

    if (check_every <= 0) {
        // Device-side convergence only: enqueue every cycle, no host read-back
        // (groups of kDeviceGroup cycles, one graph replay each).
        constexpr int kDeviceGroup = 16;
        const int total = (int)ceil_div(maxiter, cycle);
        for (int c = 0; c < total; c += kDeviceGroup) {
            const int k = std::min(kDeviceGroup, total - c);
            WA_TRY(runner.run(group_of(k), 1, k == kDeviceGroup));
        }
        if (iters_out || rnorm_out || atol_out) {
            WA_TRY(read_state(ws.state, &h, stream));
            if (iters_out)
                *iters_out = h.iter;
            if (rnorm_out)
                *rnorm_out = std::sqrt(h.rr);
            if (atol_out)
                *atol_out = std::sqrt(h.atol_sq);
        }
        return kOk;
    }

    if (!initial)
        WA_TRY(read_state(ws.state, &h, stream));
    const double atol_out_v = std::sqrt(h.atol_sq);
    int cur_iter = 0;
    if (cb)
        cb(cur_iter, std::sqrt(h.rr), atol_out_v, cb_user);
    if (!(h.rr <= h.atol_sq) && check_every % cycle == 0) {
        // the cycles between two checks run as one group (one graph replay)
        const int per_check = check_every / cycle;
        for (;;) {
            const int left = (int)ceil_div(maxiter - cur_iter, cycle);
            const int k = std::min(per_check, left);
            WA_TRY(runner.run(group_of(k), 1, k == per_check));
            cur_iter += k * cycle;
            if (cur_iter >= maxiter)
                break;
            WA_TRY(read_state(ws.state, &h, stream));
            if (h.rr <= h.atol_sq)
                break;
            if (cb)
                cb(cur_iter, std::sqrt(h.rr), atol_out_v, cb_user);
        }
        WA_TRY(read_state(ws.state, &h, stream));
        if (cb)
            cb(cur_iter, std::sqrt(h.rr), atol_out_v, cb_user);
    } else if (!(h.rr <= h.atol_sq)) {
        for (;;) {
            WA_TRY(run_cycle());
            cur_iter += cycle;
            if (cur_iter >= maxiter)
                break;
            if ((cur_iter % check_every) < cycle) {
                WA_TRY(read_state(ws.state, &h, stream));
                if (h.rr <= h.atol_sq)
                    break;
                if (cb)
                    cb(cur_iter, std::sqrt(h.rr), atol_out_v, cb_user);
            }
        }
        WA_TRY(read_state(ws.state, &h, stream));
        if (cb)
            cb(cur_iter, std::sqrt(h.rr), atol_out_v, cb_user);
    }
    if (iters_out)
        *iters_out = cur_iter;
    if (rnorm_out)
        *rnorm_out = std::sqrt(h.rr);
    if (atol_out)
        *atol_out = atol_out_v;
    return kOk;
}

// ---------------------------------------------------------------------------
// Generic primitives (operators supplied by the caller)
// ---------------------------------------------------------------------------

template <typename S>
__global__ __launch_bounds__(kBlock) void dot_partials_kernel(
    int64_t n, const S* __restrict__ a, const S* __restrict__ b, double* partials
)
{
    __shared__ double lds[kBlock / kWave];
    double acc[1] = {0.0};
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock)
        acc[0] += (double)a[i] * (double)b[i];
    write_block_partials<kBlock, 1>(acc, partials, lds);
}

__global__ __launch_bounds__(kFinalizeBlock) void dot_finalize_kernel(const double* partials, int nparts, double* out)
{
    __shared__ double lds[kFinalizeBlock / kWave];
    const double t = sum_partials<kFinalizeBlock>(partials, nparts, lds);
    if (threadIdx.x == 0)
        *out = t;
}

// x += alpha p ; r -= alpha Ap with alpha = rr > atol_sq ? rz / pAp : 0
template <typename S>
__global__ __launch_bounds__(kBlock) void step_xr_kernel(
    int64_t n, S* __restrict__ x, S* __restrict__ r, const S* __restrict__ p, const S* __restrict__ Ap,
    const double* rr, const double* atol_sq, const double* rz, const double* pAp
)
{
    const double a = *rr > *atol_sq ? *rz / *pAp : 0.0;
    const S alpha = (S)a;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        x[i] = fma(alpha, p[i], x[i]);
        r[i] = fma(-alpha, Ap[i], r[i]);
    }
}

// p = z + beta p with beta = rr > atol_sq ? rz_new / rz_old : 0
template <typename S>
__global__ __launch_bounds__(kBlock) void step_p_kernel(
    int64_t n, const S* __restrict__ z, S* __restrict__ p, const double* rr, const double* atol_sq,
    const double* rz_new, const double* rz_old
)
{
    const double bt = *rr > *atol_sq ? *rz_new / *rz_old : 0.0;
    const S beta = (S)bt;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock)
        p[i] = fma(beta, p[i], z[i]);
}

// atol_sq = max(rtol * sqrt(bb), atol)^2 (linear.py:2051-2060)
__global__ void tolerance_kernel(const double* bb, double rtol, double atol, double* atol_sq)
{
    const double a = fmax(rtol * sqrt(*bb), atol);
    *atol_sq = a * a;
}

// ---------------------------------------------------------------------------
// Batched solves (linear.py:33-131, 2010-2373 with batch_offsets): scalar dofs
// [off[b], off[b + 1]) form subproblem b < nb; dofs below off[0] or at or
// beyond off[nb] are inactive.  Dots are per subproblem; alpha / beta and
// the convergence test are per subproblem too.
// ---------------------------------------------------------------------------

// Dofs per workgroup of a segmented dot.  Chunks never cross a subproblem
// boundary, so each subproblem's partials are contiguous and summed in a
// fixed order: the results do not depend on timing.
constexpr int kSegChunk = 4 * kBlock;

__global__ __launch_bounds__(kBlock) void seg_chunk_counts_kernel(int nb, const int* __restrict__ off,
                                                                 int* __restrict__ counts)
{
    const int b = blockIdx.x * kBlock + threadIdx.x;
    if (b < nb) {
        const int len = off[b + 1] - off[b];
        counts[b] = len > 0 ? (len + kSegChunk - 1) / kSegChunk : 0;
    }
}

// Subproblem of chunk w: the last b with chunk_start[b] <= w.
__device__ __forceinline__ int chunk_batch(int w, int nb, const int* chunk_start)
{
    int lo = 0, hi = nb - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (chunk_start[mid] <= w)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

template <typename S>
__global__ __launch_bounds__(kBlock) void seg_dot_partials_kernel(int nb, const int* __restrict__ off,
                                                                 const int* __restrict__ chunk_start,
                                                                 const S* __restrict__ a, const S* __restrict__ c,
                                                                 double* __restrict__ partials)
{
    __shared__ double lds[kBlock / kWave];
    const int w = blockIdx.x;
    if (w >= chunk_start[nb])
        return;  // workgroup-uniform
    const int bt = chunk_batch(w, nb, chunk_start);
    const int64_t beg = off[bt] + (int64_t)(w - chunk_start[bt]) * kSegChunk;
    const int64_t end = min(beg + (int64_t)kSegChunk, (int64_t)off[bt + 1]);
    double acc = 0.0;
    for (int64_t i = beg + threadIdx.x; i < end; i += kBlock)
        acc += (double)a[i] * (double)c[i];
    const double sum = block_sum<kBlock>(acc, lds);
    if (threadIdx.x == 0)
        partials[w] = sum;
}

// out[b] = sum of subproblem b's partials, one workgroup per subproblem.
__global__ __launch_bounds__(kBlock) void seg_dot_finalize_kernel(const int* __restrict__ chunk_start,
                                                                 const double* __restrict__ partials,
                                                                 double* __restrict__ out)
{
    __shared__ double lds[kBlock / kWave];
    const int bt = blockIdx.x;
    const int c0 = chunk_start[bt], c1 = chunk_start[bt + 1];
    double acc = 0.0;
    for (int k = c0 + (int)threadIdx.x; k < c1; k += kBlock)
        acc += partials[k];
    const double sum = block_sum<kBlock>(acc, lds);
    if (threadIdx.x == 0)
        out[bt] = sum;
}

// Subproblem of entry e (dpe scalars; the entry's first dof decides, as the
// reference's _find_entry_batch does), -1 when inactive.
__device__ __forceinline__ int entry_batch(int64_t e, int dpe, int nb, const int* off)
{
    const int64_t dof = e * dpe;
    if (dof < off[0] || dof >= off[nb])
        return -1;
    int lo = 0, hi = nb - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (off[mid] <= dof)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

template <typename S>
__global__ __launch_bounds__(kBlock) void step_xr_batched_kernel(
    int64_t nent, int dpe, int nb, const int* __restrict__ off, S* __restrict__ x, S* __restrict__ r,
    const S* __restrict__ p, const S* __restrict__ Ap, const double* rr, const double* atol_sq, const double* rz,
    const double* pAp
)
{
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < nent; e += (int64_t)gridDim.x * kBlock) {
        const int bt = entry_batch(e, dpe, nb, off);
        if (bt < 0)
            continue;
        const S alpha = (S)(rr[bt] > atol_sq[bt] ? rz[bt] / pAp[bt] : 0.0);
        for (int k = 0; k < dpe; ++k) {
            const int64_t i = e * dpe + k;
            x[i] = fma(alpha, p[i], x[i]);
            r[i] = fma(-alpha, Ap[i], r[i]);
        }
    }
}

template <typename S>
__global__ __launch_bounds__(kBlock) void step_p_batched_kernel(
    int64_t nent, int dpe, int nb, const int* __restrict__ off, const S* __restrict__ z, S* __restrict__ p,
    const double* rr, const double* atol_sq, const double* rz_new, const double* rz_old
)
{
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < nent; e += (int64_t)gridDim.x * kBlock) {
        const int bt = entry_batch(e, dpe, nb, off);
        if (bt < 0)
            continue;
        const S beta = (S)(rr[bt] > atol_sq[bt] ? rz_new[bt] / rz_old[bt] : 0.0);
        for (int k = 0; k < dpe; ++k) {
            const int64_t i = e * dpe + k;
            p[i] = fma(beta, p[i], z[i]);
        }
    }
}

__global__ __launch_bounds__(kBlock) void tolerance_batched_kernel(int nb, const double* bb, double rtol,
                                                                  double atol, double* atol_sq)
{
    const int b = blockIdx.x * kBlock + threadIdx.x;
    if (b < nb) {
        const double a = fmax(rtol * sqrt(bb[b]), atol);
        atol_sq[b] = a * a;
    }
}

// z = alpha * (d o x) + beta * y (linear.py:2271-2287)
template <typename S>
__global__ __launch_bounds__(kBlock) void diag_mv_kernel(
    int64_t n, const S* __restrict__ d, const S* __restrict__ x, const S* __restrict__ y, S* __restrict__ z, S alpha,
    S beta
)
{
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        S s = S(0);
        if (alpha != S(0))
            s += alpha * (d[i] * x[i]);
        if (beta != S(0))
            s += beta * y[i];
        z[i] = s;
    }
}

// z = alpha * A x + beta * y for a dense row-major m x k matrix, one wave per
// row (linear.py:2246-2268).
template <typename S>
__global__ __launch_bounds__(kBlock) void dense_mv_kernel(
    int m, int k, const S* __restrict__ A, const S* __restrict__ x, const S* __restrict__ y, S* __restrict__ z,
    S alpha, S beta
)
{
    const int row = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    const int lane = threadIdx.x % kWave;
    if (row >= m)
        return;
    S s = S(0);
    if (alpha != S(0))
        for (int c = lane; c < k; c += kWave)
            s += A[(size_t)row * k + c] * x[c];
    s = wave_sum(s) * alpha;
    if (lane == 0) {
        if (beta != S(0))
            s += beta * y[row];
        z[row] = s;
    }
}

int vec_grid(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>(kMaxGrid, ceil_div(n, kBlock))); }

}  // namespace
}  // namespace wa

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------

// n scalar unknowns; the reduction scratch is sized for n block rows, an
// upper bound for every block size.
WA_API size_t warp_amd_cg_workspace_size(int64_t n, int scalar_size)
{
    size_t needed = 0;
    wa::carve_cg(nullptr, 0, n, n, (size_t)scalar_size, &needed);
    return needed + 256;
}

// Byte offsets of the device-resident scalars inside the CG workspace, so
// callers can read them without a host copy of the layout:
// 0 iterations (int32), 1 r.r (double), 2 atol^2 (double); and what says which
// kernels solved (int32): 3 the largest column window of the one-launch solve's
// plan (0: no plan since the state was last initialised), 4 its workgroups that
// finished (0: the general kernels solved).
WA_API size_t warp_amd_cg_state_offset(int which)
{
    switch (which) {
    case 0: return offsetof(wa::CgState, iter);
    case 1: return offsetof(wa::CgState, rr);
    case 2: return offsetof(wa::CgState, atol_sq);
    case 3: return offsetof(wa::CgState, small_window);
    case 4: return offsetof(wa::CgState, small_done);
    default: return 0;
    }
}

#define WA_DEFINE_CG(SUFFIX, S)                                                                                       \
    WA_API int warp_amd_cg_solve_##SUFFIX(                                                                            \
        int nrow, int block_size, const int* offsets, const int* columns, const S* values, int64_t nnz_hint,          \
        int prec_kind, const S* prec, const S* b, S* x, double tol, double atol, int maxiter, int check_every,        \
        int restart, int use_graph, wa::CgCallback callback, void* callback_user, void* workspace,                    \
        size_t workspace_bytes,                                                                                       \
        int* iterations, double* residual_norm, double* abs_tolerance, void* stream                                   \
    )                                                                                                                 \
    {                                                                                                                 \
        wa::CgProblem pb{nrow, block_size, offsets, columns, values, nnz_hint, prec_kind, prec, b, x};                \
        return wa::cg_solve_impl<S>(                                                                                  \
            pb, tol, atol, maxiter, check_every, restart, use_graph, callback, callback_user, workspace,              \
            workspace_bytes, iterations, residual_norm, abs_tolerance, wa::as_stream(stream)                          \
        );                                                                                                            \
    }                                                                                                                 \
    WA_API int warp_amd_cg_solve_polls_##SUFFIX(                                                                      \
        int nrow, int block_size, const int* offsets, const int* columns, const S* values, int64_t nnz_hint,          \
        int prec_kind, const S* prec, const S* b, S* x, double tol, double atol, int maxiter, int check_every,        \
        int polls, void* workspace, size_t workspace_bytes, int* iterations, double* residual_norm,                   \
        double* abs_tolerance, void* stream                                                                           \
    )                                                                                                                 \
    {                                                                                                                 \
        wa::CgProblem pb{nrow, block_size, offsets, columns, values, nnz_hint, prec_kind, prec, b, x};                \
        return wa::cg_solve_impl<S>(pb, tol, atol, maxiter, check_every, 0, 0, nullptr, nullptr, workspace,           \
                                    workspace_bytes, iterations, residual_norm, abs_tolerance,                        \
                                    wa::as_stream(stream), polls);                                                    \
    }                                                                                                                 \
    WA_API int warp_amd_dot_##SUFFIX(                                                                                 \
        int64_t n, const S* a, const S* b, double* out, void* workspace, size_t workspace_bytes, void* stream         \
    )                                                                                                                 \
    {                                                                                                                 \
        const int grid = wa::vec_grid(n);                                                                             \
        WA_REQUIRE(workspace && workspace_bytes >= sizeof(double) * grid,                                            \
                   "dot: workspace too small (need %zu bytes)", sizeof(double) * grid);                               \
        double* partials = (double*)workspace;                                                                        \
        wa::dot_partials_kernel<S><<<grid, wa::kBlock, 0, wa::as_stream(stream)>>>(n, a, b, partials);               \
        WA_LAUNCH_CHECK();                                                                                            \
        wa::dot_finalize_kernel<<<1, wa::kFinalizeBlock, 0, wa::as_stream(stream)>>>(partials, grid, out);           \
        WA_LAUNCH_CHECK();                                                                                            \
        return wa::kOk;                                                                                               \
    }                                                                                                                 \
    WA_API int warp_amd_cg_step_xr_##SUFFIX(                                                                          \
        int64_t n, S* x, S* r, const S* p, const S* Ap, const double* rr, const double* atol_sq, const double* rz,    \
        const double* pAp, void* stream                                                                               \
    )                                                                                                                 \
    {                                                                                                                 \
        wa::step_xr_kernel<S><<<wa::vec_grid(n), wa::kBlock, 0, wa::as_stream(stream)>>>(                             \
            n, x, r, p, Ap, rr, atol_sq, rz, pAp                                                                      \
        );                                                                                                            \
        WA_LAUNCH_CHECK();                                                                                            \
        return wa::kOk;                                                                                               \
    }                                                                                                                 \
    WA_API int warp_amd_cg_step_p_##SUFFIX(                                                                           \
        int64_t n, const S* z, S* p, const double* rr, const double* atol_sq, const double* rz_new,                   \
        const double* rz_old, void* stream                                                                            \
    )                                                                                                                 \
    {                                                                                                                 \
        wa::step_p_kernel<S><<<wa::vec_grid(n), wa::kBlock, 0, wa::as_stream(stream)>>>(                              \
            n, z, p, rr, atol_sq, rz_new, rz_old                                                                      \
        );                                                                                                            \
        WA_LAUNCH_CHECK();                                                                                            \
        return wa::kOk;                                                                                               \
    }                                                                                                                 \
    WA_API int warp_amd_seg_dot_##SUFFIX(                                                                             \
        int64_t n, int nb, const int* batch_offsets, const int* chunk_start, int max_chunks, const S* a, const S* b,  \
        double* partials, double* out, void* stream                                                                   \
    )                                                                                                                 \
    {                                                                                                                 \
        WA_REQUIRE(nb > 0 && max_chunks >= 0 && batch_offsets && chunk_start && partials && out,                      \
                   "seg_dot: invalid arguments");                                                                     \
        hipStream_t s = wa::as_stream(stream);                                                                        \
        if (max_chunks > 0) {                                                                                         \
            wa::seg_dot_partials_kernel<S><<<(unsigned)max_chunks, wa::kBlock, 0, s>>>(nb, batch_offsets,            \
                                                                                      chunk_start, a, b, partials);   \
            WA_LAUNCH_CHECK();                                                                                        \
        }                                                                                                             \
        wa::seg_dot_finalize_kernel<<<(unsigned)nb, wa::kBlock, 0, s>>>(chunk_start, partials, out);                  \
        WA_LAUNCH_CHECK();                                                                                            \
        return wa::kOk;                                                                                               \
    }                                                                                                                 \
    WA_API int warp_amd_cg_step_xr_batched_##SUFFIX(                                                                  \
        int64_t nent, int dpe, int nb, const int* batch_offsets, S* x, S* r, const S* p, const S* Ap,                 \
        const double* rr, const double* atol_sq, const double* rz, const double* pAp, void* stream                    \
    )                                                                                                                 \
    {                                                                                                                 \
        WA_REQUIRE(nb > 0 && dpe > 0 && batch_offsets, "cg_step_xr_batched: invalid arguments");                     \
        if (nent <= 0)                                                                                                \
            return wa::kOk;                                                                                           \
        wa::step_xr_batched_kernel<S><<<wa::vec_grid(nent), wa::kBlock, 0, wa::as_stream(stream)>>>(                 \
            nent, dpe, nb, batch_offsets, x, r, p, Ap, rr, atol_sq, rz, pAp                                          \
        );                                                                                                            \
        WA_LAUNCH_CHECK();                                                                                            \
        return wa::kOk;                                                                                               \
    }                                                                                                                 \
    WA_API int warp_amd_cg_step_p_batched_##SUFFIX(                                                                   \
        int64_t nent, int dpe, int nb, const int* batch_offsets, const S* z, S* p, const double* rr,                  \
        const double* atol_sq, const double* rz_new, const double* rz_old, void* stream                               \
    )                                                                                                                 \
    {                                                                                                                 \
        WA_REQUIRE(nb > 0 && dpe > 0 && batch_offsets, "cg_step_p_batched: invalid arguments");                      \
        if (nent <= 0)                                                                                                \
            return wa::kOk;                                                                                           \
        wa::step_p_batched_kernel<S><<<wa::vec_grid(nent), wa::kBlock, 0, wa::as_stream(stream)>>>(                  \
            nent, dpe, nb, batch_offsets, z, p, rr, atol_sq, rz_new, rz_old                                           \
        );                                                                                                            \
        WA_LAUNCH_CHECK();                                                                                            \
        return wa::kOk;                                                                                               \
    }                                                                                                                 \
    WA_API int warp_amd_diag_mv_##SUFFIX(                                                                             \
        int64_t n, const S* d, const S* x, const S* y, S* z, S alpha, S beta, void* stream                            \
    )                                                                                                                 \
    {                                                                                                                 \
        if (n <= 0)                                                                                                   \
            return wa::kOk;                                                                                           \
        wa::diag_mv_kernel<S><<<wa::vec_grid(n), wa::kBlock, 0, wa::as_stream(stream)>>>(n, d, x, y, z, alpha, beta); \
        WA_LAUNCH_CHECK();                                                                                            \
        return wa::kOk;                                                                                               \
    }                                                                                                                 \
    WA_API int warp_amd_dense_mv_##SUFFIX(                                                                            \
        int m, int k, const S* A, const S* x, const S* y, S* z, S alpha, S beta, void* stream                         \
    )                                                                                                                 \
    {                                                                                                                 \
        if (m <= 0)                                                                                                   \
            return wa::kOk;                                                                                           \
        const int rows_per_block = wa::kBlock / wa::kWave;                                                            \
        wa::dense_mv_kernel<S><<<(unsigned)wa::ceil_div(m, rows_per_block), wa::kBlock, 0, wa::as_stream(stream)>>>(  \
            m, k, A, x, y, z, alpha, beta                                                                             \
        );                                                                                                            \
        WA_LAUNCH_CHECK();                                                                                            \
        return wa::kOk;                                                                                               \
    }

WA_DEFINE_CG(f32, float)
WA_DEFINE_CG(f64, double)

WA_API size_t warp_amd_dot_workspace_size(int64_t n) { return sizeof(double) * wa::vec_grid(n); }

// Chunks a segmented dot over n active dofs in nb subproblems can use.
WA_API int warp_amd_seg_dot_max_chunks(int64_t n, int nb)
{
    return (int)(wa::ceil_div(n, wa::kSegChunk) + nb);
}

WA_API size_t warp_amd_seg_dot_plan_workspace_size(int nb)
{
    return wa::align_up(sizeof(int) * (size_t)(nb + 1), 256) + wa::scan_workspace_bytes((int64_t)nb + 1);
}

// chunk_start[0..nb] = exclusive scan of the chunks per subproblem
// (chunk_start[nb] = total); computed once per batch layout.
WA_API int warp_amd_seg_dot_plan(int nb, const int* batch_offsets, int* chunk_start, void* workspace,
                                 size_t workspace_bytes, void* stream)
{
    WA_REQUIRE(nb > 0 && batch_offsets && chunk_start, "seg_dot_plan: invalid arguments");
    WA_REQUIRE(workspace && workspace_bytes >= warp_amd_seg_dot_plan_workspace_size(nb),
               "seg_dot_plan: workspace too small");
    hipStream_t s = wa::as_stream(stream);
    int* counts = static_cast<int*>(workspace);
    void* scan_ws = static_cast<char*>(workspace) + wa::align_up(sizeof(int) * (size_t)(nb + 1), 256);
    wa::seg_chunk_counts_kernel<<<(unsigned)wa::ceil_div(nb, wa::kBlock), wa::kBlock, 0, s>>>(nb, batch_offsets,
                                                                                            counts);
    WA_LAUNCH_CHECK();
    return wa::exclusive_scan_i32(counts, chunk_start, nb, scan_ws, s);
}

WA_API int warp_amd_cg_tolerance_batched(int nb, const double* bb, double tol, double atol, int is_f64,
                                         double* atol_sq, void* stream)
{
    WA_REQUIRE(nb > 0 && bb && atol_sq, "cg_tolerance_batched: invalid arguments");
    double rtol_v, atol_v;
    wa::get_tolerances(is_f64 != 0, tol, atol, &rtol_v, &atol_v);
    wa::tolerance_batched_kernel<<<(unsigned)wa::ceil_div(nb, wa::kBlock), wa::kBlock, 0, wa::as_stream(stream)>>>(
        nb, bb, rtol_v, atol_v, atol_sq);
    WA_LAUNCH_CHECK();
    return wa::kOk;
}

WA_API int warp_amd_cg_tolerance(const double* bb, double tol, double atol, int is_f64, double* atol_sq, void* stream)
{
    double rtol_v, atol_v;
    wa::get_tolerances(is_f64 != 0, tol, atol, &rtol_v, &atol_v);
    wa::tolerance_kernel<<<1, 1, 0, wa::as_stream(stream)>>>(bb, rtol_v, atol_v, atol_sq);
    WA_LAUNCH_CHECK();
    return wa::kOk;
}
