// Device-side building blocks for block-sparse row (BSR) products.
//
// Storage is the compact / padded BSR layout of the reference
// (warp/_src/sparse.py:103-131): offsets[nrow+1], optional row_counts[nrow]
// (active blocks of row r are offsets[r] .. offsets[r]+row_counts[r]),
// columns[], and values[] holding BR x BC row-major scalars per block.
#pragma once

#include "common.h"

namespace wa {

__device__ __forceinline__ int row_end(const int* offsets, const int* row_counts, int row)
{
    return row_counts ? offsets[row] + row_counts[row] : offsets[row + 1];
}

// Per-lane partial sums of one block row (kept in registers: only ever
// indexed with compile-time indices).
template <typename S, int BR> struct RowAcc {
    S v[BR];
};

// One block row handled by an aligned group of G lanes (vector-BSR): lane g
// takes blocks beg+g, beg+g+G, ..., accumulates its BR partial row sums with
// explicit FMAs (block columns in order), and the group then reduces them with
// an xor butterfly (lane g adds lane g^off for off = G/2 .. 1).  On return every
// lane of the group holds the BR sums of (A x)[row*BR + s].  The order is
// fixed by G alone, so a CPU restatement can reproduce the bits.
template <typename S, int BR, int BC, int G>
__device__ __forceinline__ RowAcc<S, BR> group_row_product(
    int row, int lane, const int* __restrict__ offsets, const int* __restrict__ row_counts,
    const int* __restrict__ columns, const S* __restrict__ values, const S* __restrict__ x
)
{
    RowAcc<S, BR> acc;
#pragma unroll
    for (int s = 0; s < BR; ++s)
        acc.v[s] = S(0);
    const int beg = offsets[row];
    const int end = row_end(offsets, row_counts, row);
    for (int b = beg + lane; b < end; b += G) {
        const int col = columns[b];
        const S* blk = values + (size_t)b * (BR * BC);
        S m[BR * BC];
#pragma unroll
        for (int k = 0; k < BR * BC; ++k)
            m[k] = blk[k];
        S xv[BC];
#pragma unroll
        for (int c = 0; c < BC; ++c)
            xv[c] = x[(size_t)col * BC + c];
#pragma unroll
        for (int s = 0; s < BR; ++s)
#pragma unroll
            for (int c = 0; c < BC; ++c)
                acc.v[s] = fma(m[s * BC + c], xv[c], acc.v[s]);
    }
#pragma unroll
    for (int s = 0; s < BR; ++s)
        acc.v[s] = group_sum<G>(acc.v[s]);
    return acc;
}

// Several consecutive block rows per lane group: lane g takes block g, g+G, ...
// of each of the RPG rows row0 .. row0+RPG-1, issuing the loads of all rows
// before the FMAs (more bytes in flight per wave).  Each row is summed in the
// same order as group_row_product, so results are identical to it.  On return
// acc.v[j*BR + s] holds (A x)[(row0+j*rstride)*BR + s] in every lane of the
// group; rows at or beyond nrow contribute zeros.
//
// V is the stored value type and S the vector / accumulation type (V = float,
// S = double gives the FP64 residual of an FP32 matrix).
//
// XF: x(i) returns entry i of the vector being multiplied (a plain load, or
// a value computed from several arrays by fused kernels).
template <typename S, int BR, int BC, int G, int RPG, typename V, typename XF>
__device__ __forceinline__ RowAcc<S, BR * RPG> group_rows_product_f(
    int row0, int nrow, int lane, const int* __restrict__ offsets, const int* __restrict__ row_counts,
    const int* __restrict__ columns, const V* __restrict__ values, XF x, int rstride = 1
)
{
    RowAcc<S, BR * RPG> acc;
#pragma unroll
    for (int s = 0; s < BR * RPG; ++s)
        acc.v[s] = S(0);
    int beg[RPG], cnt[RPG];
    int nmax = 0;
#pragma unroll
    for (int j = 0; j < RPG; ++j) {
        const int r = row0 + j * rstride;
        beg[j] = 0;
        cnt[j] = 0;
        if (r < nrow) {
            beg[j] = offsets[r];
            cnt[j] = row_end(offsets, row_counts, r) - beg[j];
        }
        nmax = cnt[j] > nmax ? cnt[j] : nmax;
    }
    for (int k = lane; k < nmax; k += G) {
        bool ok[RPG];
        int col[RPG];
        V m[RPG][BR * BC];
#pragma unroll
        for (int j = 0; j < RPG; ++j) {
            ok[j] = k < cnt[j];
            // Inactive slots read storage slot 0 (in bounds whenever any row
            // has blocks) and gather x at column 0: slot 0 of a padded matrix
            // may be an unused slot whose column is -1.
            const int b = ok[j] ? beg[j] + k : 0;
            const int cb = columns[b];
            col[j] = ok[j] ? cb : 0;
            const V* blk = values + (size_t)b * (BR * BC);
#pragma unroll
            for (int q = 0; q < BR * BC; ++q)
                m[j][q] = blk[q];
        }
#pragma unroll
        for (int j = 0; j < RPG; ++j) {
            S xv[BC];
#pragma unroll
            for (int c = 0; c < BC; ++c)
                xv[c] = x((size_t)col[j] * BC + c);
#pragma unroll
            for (int s = 0; s < BR; ++s) {
                S a = acc.v[j * BR + s];
#pragma unroll
                for (int c = 0; c < BC; ++c)
                    a = fma((S)m[j][s * BC + c], xv[c], a);
                acc.v[j * BR + s] = ok[j] ? a : acc.v[j * BR + s];
            }
        }
    }
#pragma unroll
    for (int s = 0; s < BR * RPG; ++s)
        acc.v[s] = group_sum<G>(acc.v[s]);
    return acc;
}

template <typename S> struct LoadX {
    const S* __restrict__ p;
    __device__ __forceinline__ S operator()(size_t i) const { return p[i]; }
};

template <typename S, int BR, int BC, int G, int RPG, typename V = S>
__device__ __forceinline__ RowAcc<S, BR * RPG> group_rows_product(
    int row0, int nrow, int lane, const int* __restrict__ offsets, const int* __restrict__ row_counts,
    const int* __restrict__ columns, const V* __restrict__ values, const S* __restrict__ x, int rstride = 1
)
{
    return group_rows_product_f<S, BR, BC, G, RPG, V>(row0, nrow, lane, offsets, row_counts, columns, values,
                                                      LoadX<S>{x}, rstride);
}

// acc.v[i] for a lane-dependent i.  Written as an explicit select chain on
// named values: a loop of selects gets turned back into a dynamic index,
// which moves the accumulators to LDS.
template <typename S, int N> __device__ __forceinline__ S pick(const RowAcc<S, N>& acc, int i)
{
    static_assert(N >= 1 && N <= 16, "pick supports up to 16 values");
    S v = acc.v[0];
#define WA_PICK_STEP(K)                                                                                               \
    if constexpr (N > K) {                                                                                            \
        const S t = acc.v[K];                                                                                         \
        v = i == K ? t : v;                                                                                           \
    }
    WA_PICK_STEP(1) WA_PICK_STEP(2) WA_PICK_STEP(3) WA_PICK_STEP(4) WA_PICK_STEP(5) WA_PICK_STEP(6) WA_PICK_STEP(7)
    WA_PICK_STEP(8) WA_PICK_STEP(9) WA_PICK_STEP(10) WA_PICK_STEP(11) WA_PICK_STEP(12) WA_PICK_STEP(13)
    WA_PICK_STEP(14) WA_PICK_STEP(15)
#undef WA_PICK_STEP
    return v;
}

// Rows per lane group of the vector-BSR kernels (measured on MI355X: two
// 3x3 rows, four scalar rows).
constexpr int rows_per_group_for(int br, int bc) { return (br == 1 && bc == 1) ? 4 : 2; }

// Lanes per block row and rows per lane group for a matrix with `nnz_hint`
// blocks over `nrow` rows: about one block per lane for block rows, two
// entries per lane for scalar rows (lanes = the power of two covering that).
struct BsrShape {
    int lanes;
    int rows_per_group;
};

inline BsrShape default_bsr_shape(int nrow, int br, int bc, int64_t nnz_hint)
{
    const double mean = nrow > 0 && nnz_hint > 0 ? (double)nnz_hint / nrow : 8.0;
    const double per_lane = (br == 1 && bc == 1) ? 2.0 : 1.0;
    int g = 1;
    while (g * per_lane < mean && g < 64)
        g <<= 1;
    return BsrShape{g, rows_per_group_for(br, bc)};
}

// ---------------------------------------------------------------------------
// Scalar rows by wave tiles
// ---------------------------------------------------------------------------
//
// A wavefront takes RW consecutive scalar rows: it loads their columns and
// values in 16-byte pieces (four entries per lane, CH times), gathers x for
// them, lays (value, x) out in LDS, and each lane adds one row from there, in
// the order of group_row_product with G lanes (entry k into partial k % G, then
// the butterfly), so the bits are the same.  What limits the lane-group kernel
// on 7- and 9-entry rows is the rate of 4-byte requests (a plain copy at 4
// bytes per lane reaches 3.7 TB/s here, at 16 bytes 6.5); no barrier is needed,
// since a wave reads only what it wrote.  7-point rows, us per product with
// alternating direction, lane groups / wave tiles: FP32 128^3 26.6 / 24.5,
// 200^3 105 / 95, 256^3 241 / 200 (5.7 TB/s); FP64 128^3 41 / 33, 161^3 92 / 73,
// 195^3 155 / 130.  FP64 tiles are half as long (RW = 32, CH = 1: their LDS
// image is twice as large; 64 rows took 87 us at 161^3).  A tile whose entries
// exceed the LDS image (rows far above the mean) is added by lane groups: FP32,
// 2^21 rows, one eighth of them of 36 entries 80 / 68 us, by one lane a row 338.
// Persistent workgroups that load the next tile ahead were slower (262 us at
// 256^3), as were non-temporal matrix loads wherever consecutive products meet
// in the memory-side cache (30 us at 128^3).
//
// The tiles are dealt to the XCDs in runs (xcd_run_block), so that the rows of
// neighbouring tiles find their x in one L2 (FP32 256^3 214 -> 203 us; runs of
// 32 or 64 gain 1 % more there and lose 4 % at 128^3).
constexpr int kWaveTileEntries = 256;  // entries of one 16-byte piece per lane

template <typename S, typename V, int CH> struct WaveTile {
    V v[CH * kWaveTileEntries];
    S x[CH * kWaveTileEntries];
};

// Workgroup b of `grid`, renumbered so that XCD b % 8 gets runs of consecutive
// workgroups; a bijection for any grid.
template <int kRun = 8> __device__ __forceinline__ int xcd_run_block(int b, int grid)
{
    constexpr int kXcd = 8;
    const int full = grid - grid % (kXcd * kRun);
    if (b >= full)
        return b;
    const int i = b / kXcd;
    return ((i / kRun) * kXcd + b % kXcd) * kRun + i % kRun;
}

// Sum of row row0 + lane (lane < RW and row < nrow, else 0).  STREAM: columns
// and values are loaded past the caches.
template <typename S, int G, int RW, int CH, bool STREAM = false, typename V, typename XF>
__device__ __forceinline__ S wave_rows_product(int row0, int nrow, int lane, const int* __restrict__ offsets,
                                               const int* __restrict__ columns, const V* __restrict__ values, XF x,
                                               WaveTile<S, V, CH>& tile)
{
    typedef int I4 __attribute__((ext_vector_type(4)));
    typedef V V4 __attribute__((ext_vector_type(4)));
    typedef S S4 __attribute__((ext_vector_type(4)));
    const int row = row0 + lane;
    const bool on = lane < RW && row < nrow;
    const int beg = on ? offsets[row] : 0;
    const int end = on ? offsets[row + 1] : 0;
    const int len = end - beg;
    const int nnz = offsets[nrow];
    const int last = (nrow - row0 < RW ? nrow - row0 : RW) - 1;
    const int b0 = __builtin_amdgcn_readfirstlane(beg);
    const int e0 = __builtin_amdgcn_readlane(end, last);
    const int base = b0 & ~3;
    S a[G];
#pragma unroll
    for (int g = 0; g < G; ++g)
        a[g] = S(0);
    if (e0 - base <= CH * kWaveTileEntries) {  // wave-uniform
        I4 c[CH];
        V4 v[CH];
#pragma unroll
        for (int u = 0; u < CH; ++u) {
            // unsigned: a piece of the last tile may start past the largest int
            const unsigned k = (unsigned)base + (u * kWave + lane) * 4;
            if (k < (unsigned)e0) {
                if (k + 3 < (unsigned)nnz) {
                    c[u] = stream_load<STREAM>(reinterpret_cast<const I4*>(columns + k));
                    v[u] = stream_load<STREAM>(reinterpret_cast<const V4*>(values + k));
                } else {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        c[u][q] = k + q < (unsigned)nnz ? columns[k + q] : 0;
                        v[u][q] = k + q < (unsigned)nnz ? values[k + q] : V(0);
                    }
                }
            }
        }
        S4 xv[CH];
#pragma unroll
        for (int u = 0; u < CH; ++u) {
            const unsigned k = (unsigned)base + (u * kWave + lane) * 4;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                xv[u][q] = (k + q >= (unsigned)b0 && k + q < (unsigned)e0) ? x((size_t)c[u][q]) : S(0);
        }
#pragma unroll
        for (int u = 0; u < CH; ++u) {
            const int k = (u * kWave + lane) * 4;
            if (k < e0 - base) {
                *reinterpret_cast<V4*>(tile.v + k) = v[u];
                *reinterpret_cast<S4*>(tile.x + k) = xv[u];
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (int k = 0; k < len; k += G) {
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const bool in = k + g < len;
                const int i = beg - base + (in ? k + g : 0);
                const S t = fma((S)tile.v[i], tile.x[i], a[g]);
                a[g] = in ? t : a[g];
            }
        }
    } else {
        constexpr int RPG = RW * G / kWave;
        const RowAcc<S, RPG> acc = group_rows_product_f<S, 1, 1, G, RPG, V>(row0 + lane / G * RPG, nrow, lane % G,
                                                                          offsets, nullptr, columns, values, x);
        S v = S(0);
#pragma unroll
        for (int e = 0; e < RPG; ++e) {
            const S t = __shfl(acc.v[e], lane / RPG * G);
            v = lane % RPG == e ? t : v;
        }
        return on ? v : S(0);
    }
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1)
#pragma unroll
        for (int g = 0; g < off; ++g)
            a[g] = a[g] + a[g + off];
    return a[0];
}

// Wave tiles take compact scalar matrices with 16-byte aligned columns and
// values, 4 lanes per row (more than 4 entries per row on average) and at most
// 7.25, so that nearly every tile of 32 or 64 rows fits its image of 8 entries
// per row (9-entry rows, 24 to 48 of them per tile, were slower: FP64 60
// against 48 us on 1400^2 nodes).  The smallest systems stay with the lane
// groups, which have more waves in flight there: FP32 values and x below 2M
// rows (100^3 15.5 / 16.3 us), otherwise below 2^18 (64^3 FP64 6.9 / 6.1 us,
// 41^3 even).
inline bool wave_rows_supported(int lanes, int nrow, int64_t nnz_hint, bool wide_x, const int* row_counts,
                                const void* columns, const void* values)
{
    return lanes == 4 && nrow >= (wide_x ? 1 << 18 : 1 << 21) && 4 * nnz_hint <= (int64_t)29 * nrow && !row_counts &&
           (((uintptr_t)columns | (uintptr_t)values) & 15) == 0;
}

}  // namespace wa
