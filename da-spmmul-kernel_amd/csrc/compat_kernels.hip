// compat_kernels.hip -- the reference's 12-kernel SpMV/SpMM family,
// redesigned for gfx950 wave64, behind the reference's launcher names.
//
// Algorithm classes and output semantics follow the reference
// (spmvspmm.h:72-197): CSR = row-balanced, overwrite; COO = nnz-balanced,
// atomic accumulate.  What changes is the mapping onto CDNA4:
//   * lane groups of L lanes x VW floats cover a dense row slab (float4
//     along N) instead of one lane per column;
//   * the sparse operand of a workgroup is staged through LDS with
//     coalesced loads, then read as LDS broadcasts;
//   * parallel reductions are wave64 butterflies / segmented scans on
//     DPP, ds_swizzle and permlane32 (wave64.hpp);
//   * blocks are renumbered so each XCD walks a contiguous row range.
// Sequential (SR) kernels sum every output in nonzero order with a
// separately rounded multiply and add (the library is built with
// -ffp-contract=off), so the row-balanced SR kernels reproduce the
// reference host loop (spmvspmm_benchmark.cu:11-39) bit for bit.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "common.hpp"
#include "internal.hpp"
#include "native.hpp"

namespace dspmm {

constexpr int kWin = 2048;   // LDS staging window (nonzeros) of the row-balanced kernels

// Per-lane in-order accumulation of a window of nonzeros [p0, p1) staged
// in LDS at s_col/s_val (offset w), gathering VW floats of B per nonzero.
// Gathers are issued UNR at a time before they are summed, in order.
template <typename TB, int VW, int UNR>
__device__ __forceinline__ void seq_accumulate(float (&acc)[VW], int p0, int p1, int w,
                                               const int *s_col, const float *s_val,
                                               const TB *__restrict__ B, int64_t ldb,
                                               int col0) {
    int p = p0;
    for (; p1 - p >= UNR; p += UNR) {
        float b[UNR][VW];
#pragma unroll
        for (int u = 0; u < UNR; u++)
            load_g<TB, VW>(b[u], B + (int64_t)s_col[p + u - w] * ldb + col0);
#pragma unroll
        for (int u = 0; u < UNR; u++) {
            const float a = s_val[p + u - w];
#pragma unroll
            for (int k = 0; k < VW; k++) acc[k] = acc[k] + a * b[u][k];
        }
    }
    if (p < p1) {                               // the rest, loaded together
        float b[UNR - 1][VW];
#pragma unroll
        for (int u = 0; u < UNR - 1; u++)
            if (p + u < p1) load_g<TB, VW>(b[u], B + (int64_t)s_col[p + u - w] * ldb + col0);
#pragma unroll
        for (int u = 0; u < UNR - 1; u++) {
            if (p + u < p1) {
                const float a = s_val[p + u - w];
#pragma unroll
                for (int k = 0; k < VW; k++) acc[k] = acc[k] + a * b[u][k];
            }
        }
    }
}

// Cooperative staging of nonzeros [w, w+cnt) into LDS by a whole block.
__device__ __forceinline__ void stage_window(int *s_col, float *s_val, const int *__restrict__ colIdx,
                                             const float *__restrict__ values, int w, int cnt) {
    for (int i = threadIdx.x; i < cnt; i += kBlock) {
        s_col[i] = colIdx[w + i];
        s_val[i] = values[w + i];
    }
}

// Rows that a block of k_csr_scalar_rm sums together, all its groups
// gathering: at least kLongRow nonzeros and twice the block's mean row, so
// that the row's own group would otherwise work on alone.
constexpr int kLongRow = 96;
// The longest rows (kScoutRow nonzeros or more, and kScoutMean times the mean,
// so that most blocks have none) are found and summed by the first blocks of
// the launch, the scouts, each of which looks at up to kScoutRows rows and sums
// kScoutCols of their columns: begun last, or with the gathers of one block
// only, one of them would set the kernel's time.  On a power-law matrix
// (262144 rows, the longest 4900, nv = 64): 32 columns 160 us, 16
// (64-byte gathers) 192, without these blocks 203, with a lane group alone on
// each row 660.  A scout's rows lie far apart, since long rows may be neighbours:
// 65536 such rows sorted by length, nv = 32, csr_vector 73 us, with consecutive
// rows to a scout 2300.  128 rows each instead of 512 are faster there (65536 rows,
// nv = 32, csr_vector 39 and 54 us) and slower on rows of like lengths, for whose
// blocks so many scouts leave less room (65536 rows of 12 to 24, nv = 16: 5 to 10%).
constexpr int kScoutRow = 1024;
constexpr int kScoutMean = 8;
constexpr int kScoutRows = 512;
constexpr int kScoutCols = 32;

// The scouts of a launch: their number and the length from which rows are theirs.
struct Scouts {
    int blocks = 0, row = INT_MAX;
};

// One of the rows that scout `i` of `n` looks at: its k-th.  Many rows go in
// fours, since one by one their lines of rowPtr are read 32 times (power law of
// 262144 rows, nv = 1, csr_vector: 27.3 us, in fours 24.5).
__device__ __forceinline__ int64_t scout_at(int i, int n, int nr, int k) {
    const int w = nr / n >= 128 ? 4 : 1;
    return ((int64_t)(k / w) * n + i) * w + k % w;
}
constexpr int kScoutList = kScoutRows + 4;     // rows that one scout may look at

// Collects the scout's long rows (their k's) in s_scout; *s_n is their number.
// Every thread calls it (barriers inside).
__device__ __forceinline__ void scout_look(int i, int n, int nr, const int *__restrict__ rowPtr,
                                           int scout_row, uint16_t *s_scout, int *s_n) {
    if (threadIdx.x == 0) *s_n = 0;
    __syncthreads();
    for (int k = threadIdx.x; scout_at(i, n, nr, k) < nr; k += kBlock) {   // k < kScoutList
        const int64_t q = scout_at(i, n, nr, k);
        const auto p = *reinterpret_cast<const VecAt<int, 2, 4>::type *>(rowPtr + q);
        if (p[1] - p[0] >= scout_row) s_scout[atomicAdd(s_n, 1)] = (uint16_t)k;
    }
    __syncthreads();
}

__device__ __forceinline__ bool is_long_row(int len, int block_nnz, int block_rows) {
    return len >= kLongRow && (int64_t)len * block_rows >= 2 * (int64_t)block_nnz;
}

// One row [p0, p1) summed by the whole block in nonzero order.  Per step the
// groups multiply P nonzeros into LDS (P products of L * VW columns, two
// steps' gathers in flight) and thread t < L * VW adds column t's products in
// order; the (column, value) pairs go through LDS in chunks, loaded a chunk
// ahead.  `base` is the first of the L * VW columns.  Returns column t's sum.
// Every thread calls it (barriers inside).
template <int VW, int L, int U>
struct LongRow {
    static constexpr int W = L * VW;
    static constexpr int P = kBlock / L * U;
    static constexpr int PPT = P > kBlock / 4 ? 4 * P / kBlock : 1;   // pairs per thread and chunk
    static constexpr int CHK = PPT * kBlock;                // pairs per chunk
    static constexpr int kFloats = P * W + 4 * CHK;         // products, two chunks of pairs
    static constexpr int S = CHK / P;                       // steps per chunk
    static_assert(U >= 1 && S >= 4 && P % 16 == 0, "steps of 16 products, four to a chunk");

    static __device__ __forceinline__ float sum(int p0, int p1, const int *__restrict__ colIdx,
                                                const float *__restrict__ values,
                                                const float *__restrict__ B, int64_t ldb, int base,
                                                int nv_, float *mem) {
        const int t = threadIdx.x, g = t / L, l = t % L;
        const int col0 = slab_col<VW>(base + l * VW, nv_), at = col0 - base;
        const bool colok = col0 < nv_, whole = nv_ % VW == 0;
        float *prod = mem;
        int *s_c = reinterpret_cast<int *>(mem + P * W);
        float *s_v = mem + P * W + 2 * CHK;
        const float *__restrict__ Bc = B + (colok ? col0 : 0);
        const int n = p1 - p0;
        const int steps = (n + 2 * P - 1) / (2 * P) * 2;    // even: two register sets in turn
        int nc[PPT];                                        // this thread's pairs of the next chunk
        float nv[PPT];
        auto load_pairs = [&](int j) {
#pragma unroll
            for (int x = 0; x < PPT; x++) {
                const int q = p0 + min(j * CHK + x * kBlock + t, n - 1);
                nc[x] = colIdx[q];
                nv[x] = values[q];
            }
        };
        auto put_pairs = [&](int j) {
#pragma unroll
            for (int x = 0; x < PPT; x++) {
                s_c[(j & 1) * CHK + x * kBlock + t] = nc[x];
                s_v[(j & 1) * CHK + x * kBlock + t] = nv[x];
            }
        };
        float b[2][U][VW];
        auto gather = [&](int k, float (&d)[U][VW]) {
#pragma unroll
            for (int u = 0; u < U; u++)
                load_g<float, VW>(d[u], Bc + (int64_t)s_c[(k * P + g * U + u) % (2 * CHK)] * ldb);
        };
        float sum = 0.f;
        auto step = [&](int k, float (&d)[U][VW]) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = k * P + g * U + u;
                const float v = s_v[i % (2 * CHK)];
                float m[VW];
#pragma unroll
                for (int q = 0; q < VW; q++)   // +0 past the end: a sum that began at +0 keeps its bits
                    m[q] = i < n ? v * d[u][q] : 0.f;
                float *to = prod + (g * U + u) * W + at;
                if (whole) {
                    store_vec<VW>(to, m);
                } else {                       // the row's last columns, some of them a neighbour's
#pragma unroll
                    for (int q = 0; q < VW; q++)
                        if (at + q >= 0) to[q] = m[q];
                }
            }
            gather(k + 2, d);
            if ((k + 3) % S == 0) {            // the chunk that step k + 3 begins, read from step k + 1 on
                put_pairs((k + 3) / S);
                load_pairs((k + 3) / S + 1);
            }
            __syncthreads();
            const int m = min(P, n - k * P);
            if (t < W) {                       // H products read ahead of the H being added
                constexpr int H = 8;
                const float *pr = prod + t;
                float x[H], y[H];
#pragma unroll
                for (int j = 0; j < H; j++) x[j] = pr[j * W];
                for (int i = 0; i < m; i += 2 * H) {
#pragma unroll
                    for (int j = 0; j < H; j++) y[j] = pr[(i + H + j) * W];
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int j = 0; j < H; j++) sum = sum + x[j];
                    __builtin_amdgcn_sched_barrier(0);
                    const int nx = min(i + 2 * H, P - H);
#pragma unroll
                    for (int j = 0; j < H; j++) x[j] = pr[(nx + j) * W];
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int j = 0; j < H; j++) sum = sum + y[j];
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            __syncthreads();
        };
        load_pairs(0);
        __syncthreads();                       // `mem` is free
        put_pairs(0);
        load_pairs(1);
        __syncthreads();
        gather(0, b[0]);
        gather(1, b[1]);
        for (int k = 0; k < steps; k += 2) {
            step(k, b[0]);
            step(k + 1, b[1]);
        }
        return sum;
    }
};

// ===========================================================================
// Row-balanced, sequential reduction, row-major, for few columns
// (spmv_csr_scalar; spmm_csr_scalar_row with L * VW <= 8 and few rows, or with
// 4).  A wavefront owns G consecutive rows, at most 64 / (L * VW).  In windows
// of PW of their pairs (counted from the window's start: nnz may be close to
// INT_MAX), every lane gathers B for its share of the window at once, the next window's
// while this one is added, and the products go to the wavefront's LDS region,
// one column after another; then lane (row, column) adds its row's products
// in nonzero order.  However long a row is, all 64 lanes gather for it.
//
// What bounds it: gather latency for short rows, the chain of additions for
// long ones.  nv = 1, lanes that gathered their own rows before and now:
// stencil 64^3 28.7 -> 15.9 us, 20000 rows of 100 82 -> 12 us, power law
// (262144 rows, the longest 4900) 320 -> 61 us.
// ===========================================================================
// Pairs per window at W columns.
constexpr int stream_pairs(int W) { return W == 1 ? 512 : W == 8 ? 128 : 256; }
// COL: column-major operands, W = L columns (from W * blockIdx.y on) at a time,
// one per lane.
template <int VW, int L, bool COL>
__global__ __launch_bounds__(kBlock) void k_csr_stream(int nr, int nv, int64_t ldb, int64_t ldc,
                                                           const int *__restrict__ rowPtr,
                                                           const int *__restrict__ colIdx,
                                                           const float *__restrict__ values,
                                                           const float *__restrict__ B,
                                                           float *__restrict__ C, int G) {
    constexpr int W = L * VW, WPB = kBlock / kWave;
    constexpr int PW = stream_pairs(W);
    constexpr int E = PW * L / kWave;                             // gathers per lane and window
    constexpr int LD = PW + 8;                                    // floats per column of products
    __shared__ float s_prod[WPB][W * LD];
    const int ln = lane_id(), wv = (int)threadIdx.x / kWave;
    const int64_t rw = ((int64_t)xcd_remap(blockIdx.x, gridDim.x) * WPB + wv) * G;
    if (rw >= nr) return;                      // the whole wavefront leaves; no barrier follows
    const int c = ln % W;
    const bool mine = ln / W < G && rw + ln / W < nr;
    const int r = (int)min(rw + ln / W, (int64_t)nr);
    const int start = rowPtr[r], end = mine ? rowPtr[r + 1] : start;
    const int e0 = rowPtr[rw], e1 = rowPtr[min(rw + G, (int64_t)nr)];
    static_assert(!COL || VW == 1, "a column per lane");
    if constexpr (COL) {
        B += (int64_t)blockIdx.y * W * ldb;
        C += (int64_t)blockIdx.y * W * ldc;
        nv -= (int)blockIdx.y * W;
    }
    const int gl = slab_col<VW>((ln % L) * VW, nv);   // first column that this lane gathers
    const float *__restrict__ Bc = B + (gl < nv ? (COL ? gl * ldb : (int64_t)gl) : 0);
    float *sp = s_prod[wv];
    int cc[E];
    float vv[E], b[E][VW];
    auto gather = [&](int w) {
#pragma unroll
        for (int k = 0; k < E; k++) {
            const int p = w + min(ln / L + k * (kWave / L), e1 - 1 - w);
            cc[k] = colIdx[p];
            vv[k] = values[p];
        }
#pragma unroll
        for (int k = 0; k < E; k++) load_g<float, VW>(b[k], Bc + (COL ? (int64_t)cc[k] : (int64_t)cc[k] * ldb));
    };
    float acc = 0.f;
    if (e0 < e1) gather(e0);
    for (int w = e0; w < e1; w = e1 - w > PW ? w + PW : e1) {
        const int left = e1 - w;
        wave_lds_sync();                       // the last window's products have been read
#pragma unroll
        for (int k = 0; k < E; k++) {
            const int i = ln / L + k * (kWave / L);
#pragma unroll
            for (int q = 0; q < VW; q++)       // +0 past the end: a sum that began at +0 keeps its bits
                sp[(gl + q) * LD + i] = i < left ? vv[k] * b[k][q] : 0.f;
        }
        if (left > PW) gather(w + PW);
        wave_lds_sync();
        const int p0 = max(start, w) - w;
        int n = min(end - w, PW) - p0;
        // Long rows (of this window): 64 products at a time in the lanes of one
        // register per column, and each lane adds its product to the sum that
        // its lower neighbour hands up: 63 steps put the row's sum in order in
        // lane 63.  (A lane that reads one product after the other from LDS
        // took 66 cycles each.)
        uint64_t longs = __ballot(c == 0 && n >= kWave);
        if (__popcll(longs) > 4) longs = 0;    // as many lanes add their rows side by side
        for (; longs; longs &= longs - 1) {
            const int o = __builtin_ctzll(longs);          // the row's lane of column 0
            const int q0 = read_lane(p0, o), qn = read_lane(n, o);
            float sum[W];
#pragma unroll
            for (int q = 0; q < W; q++)
                sum[q] = __int_as_float(read_lane(__float_as_int(acc), o + q));
            for (int i = 0; i < qn; i += kWave) {
                float x[W], y[W];
#pragma unroll
                for (int q = 0; q < W; q++) {
                    const float v = sp[q * LD + min(q0 + i + ln, PW)];
                    x[q] = i + ln < qn ? v : 0.f;
                    if (ln == 0) x[q] = sum[q] + x[q];
                    y[q] = x[q];
                }
#pragma unroll 9
                for (int k = 0; k < kWave - 1; k++) {
#pragma unroll
                    for (int q = 0; q < W; q++) y[q] = dpp0_f<kDppWaveShr1>(y[q]) + x[q];
                }
#pragma unroll
                for (int q = 0; q < W; q++)
                    sum[q] = __int_as_float(read_lane(__float_as_int(y[q]), kWave - 1));
            }
#pragma unroll
            for (int q = 0; q < W; q++)
                if (ln == o + q) acc = sum[q];
            if (ln / W == o / W) n = 0;
        }
        const float *pr = sp + c * LD + p0;
        for (; n > 0; n -= 8, pr += 8) {       // reads past the row stay in the window's LDS
            float x[8];
#pragma unroll
            for (int u = 0; u < 8; u++) x[u] = pr[u];
#pragma unroll
            for (int u = 0; u < 8; u++) acc = acc + (u < n ? x[u] : 0.f);
        }
    }
    if (mine && c < nv)
        __builtin_nontemporal_store(acc, C + (COL ? (int64_t)c * ldc + r : (int64_t)r * ldc + c));
}

// ===========================================================================
// Row-balanced, sequential reduction, row-major (spmm_csr_scalar_row with more
// than 8 columns, or more than 4 and many rows).  A group of L lanes owns one row; each lane
// owns VW consecutive columns of the slab.  The block's rows' nonzeros are
// staged through LDS in windows; every lane reads its row's (col, val) as an
// LDS broadcast within its group.  Overwrites every row (empty rows -> 0).
// Rows far longer than the block's others are summed by the whole block, the
// longest ones by blocks of their own at the front of the grid (LongRow).
// PARTS: a row's sum in parts (add_parts), by its own group however long it is.
// SLICED: a block whose rows overflow one window, and one of whose rows is
// at least 4 shares of a window long (kWin / rows per block), splits each
// window into one slice per row that still has nonzeros (kWin / n for n
// such rows, rounded down to a power of two), staged by the whole block, so
// that no row waits while windows cover only other rows; a long row gets
// the whole window once the others are done.  Both forms add each row's
// products in nonzero order.
// ===========================================================================
template <int VW, int L, bool SLICED, bool PARTS = false>
__global__ __launch_bounds__(kBlock) void k_csr_scalar_rm(int nr, int nv, int64_t ldb, int64_t ldc,
                                                           const int *__restrict__ rowPtr,
                                                           const int *__restrict__ colIdx,
                                                           const float *__restrict__ values,
                                                           const float *__restrict__ B,
                                                           float *__restrict__ C, int slab_w,
                                                           int scouts, int scout_row) {
    constexpr int RPB = kBlock / L;
    constexpr int NW = kBlock / kWave;
    using Long = LongRow<VW, L, (L >= 32 ? 4 : L >= 16 ? 2 : 1)>;
    constexpr int SW = L * VW < kScoutCols ? L * VW : kScoutCols;
    constexpr int SL = SW / VW;                // lanes of a scout's group
    using Scout = LongRow<VW, SL, (SL >= 8 ? SL / 4 : SL / 2)>;
    constexpr int kLds = Long::kFloats > 2 * kWin ? Long::kFloats : 2 * kWin;
    static_assert(Scout::kFloats <= kLds, "LDS");
    __shared__ __align__(16) float s_mem[kLds];
    int *s_col = reinterpret_cast<int *>(s_mem);
    float *s_val = s_mem + kWin;
    __shared__ int s_long[RPB];                // rows that the block sums together
    __shared__ uint16_t s_scout[kScoutList];
    __shared__ int s_nlong;
    __shared__ int s_tab[SLICED ? 2 * RPB + NW : 1];   // slice start, count per rank; per-wave counts
    if ((int)blockIdx.x < scouts) {            // the longest rows first
        const int parts = (min(slab_w, nv - (int)blockIdx.y * slab_w) + SW - 1) / SW;
        const int me = (int)blockIdx.x / parts, all = scouts / parts;
        if (me >= all) return;
        scout_look(me, all, nr, rowPtr, scout_row, s_scout, &s_nlong);
        const int cb = blockIdx.y * slab_w + (int)blockIdx.x % parts * SW;
        for (int i = 0; i < s_nlong; i++) {
            const int q = (int)scout_at(me, all, nr, s_scout[i]);
            const float sum = Scout::sum(rowPtr[q], rowPtr[q + 1], colIdx, values, B, ldb, cb,
                                         nv, s_mem);
            if ((int)threadIdx.x < SW && cb + (int)threadIdx.x < nv)
                C[(int64_t)q * ldc + cb + (int)threadIdx.x] = sum;
        }
        return;
    }
    const int b = xcd_remap(blockIdx.x - scouts, gridDim.x - scouts);
    const int r0 = b * RPB;
    const int r = r0 + (int)threadIdx.x / L;
    const int col0 = slab_col<VW>(blockIdx.y * slab_w + ((int)threadIdx.x % L) * VW, nv);
    const bool colok = col0 < nv;
    const int rlast = min(r0 + RPB, nr);
    const int bs = rowPtr[r0], be = rowPtr[rlast];
    int start = 0, end = 0;
    if (r < nr) { start = rowPtr[r]; end = rowPtr[r + 1]; }
    float acc[VW];
#pragma unroll
    for (int k = 0; k < VW; k++) acc[k] = 0.f;
    // Rows that this block's groups sum together, or the scouts do.
    auto apart = [&](int len) {
        return is_long_row(len, be - bs, rlast - r0) || len >= scout_row;
    };
    float odd[VW];
#pragma unroll
    for (int k = 0; k < VW; k++) odd[k] = 0.f;
    auto add = [&](int p0, int p1, int w) {
        if constexpr (PARTS) {
            for (int p = p0 - w; p < p1 - w; p += 8) {
                float b8[8][VW];
#pragma unroll
                for (int u = 0; u < 8; u++)
                    load_g<float, VW>(b8[u], B + (int64_t)s_col[min(p + u, p1 - w - 1)] * ldb + col0);
                add_parts<VW>(acc, odd, b8, s_val, p, p1 - w);
            }
        } else {
            seq_accumulate<float, VW, 4>(acc, p0, p1, w, s_col, s_val, B, ldb, col0);
        }
    };
    int nlong = 0;
    if (!PARTS && be - bs >= kLongRow) {       // the same in every thread
        if (threadIdx.x == 0) s_nlong = 0;
        __syncthreads();
        if (threadIdx.x % L == 0 && apart(end - start)) s_long[atomicAdd(&s_nlong, 1)] = r;
        __syncthreads();
        nlong = s_nlong;
        for (int i = 0; i < nlong; i++) {
            const int q = s_long[i], p0 = rowPtr[q], p1 = rowPtr[q + 1];
            if (p1 - p0 >= scout_row) continue;
            const float sum = Long::sum(p0, p1, colIdx, values, B, ldb, blockIdx.y * slab_w, nv, s_mem);
            const int c = blockIdx.y * slab_w + (int)threadIdx.x;
            if ((int)threadIdx.x < L * VW && c < nv)
                __builtin_nontemporal_store(sum, C + (int64_t)q * ldc + c);
        }
    }
    const bool mine = nlong == 0 || !apart(end - start);
    if (!mine) end = start;                    // done
    bool slice = false;
    if constexpr (SLICED) {
        // slices pay where a row is long against its share of a window (kWin /
        // RPB pairs): then windows of contiguous pairs cover few rows each and
        // the others wait.  Rows shorter than 4 shares run in plain windows.
        if (be - bs > kWin) {
            int mx = end - start;
#pragma unroll
            for (int o = kWave / 2; o >= 1; o >>= 1) mx = max(mx, __shfl_xor(mx, o));
            if ((int)threadIdx.x % kWave == 0) s_tab[2 * RPB + (int)threadIdx.x / kWave] = mx;
            __syncthreads();
            for (int k = 0; k < NW; k++) mx = max(mx, s_tab[2 * RPB + k]);
            slice = mx >= 4 * (kWin / RPB);
            __syncthreads();
        }
    }
    if (!slice) {
        for (int w = bs; w < be; w = be - w > kWin ? w + kWin : be) {
            for (int i = 0; i < nlong; i++) {  // no window starts inside a row that is done
                const int q = s_long[i];
                if (w >= rowPtr[q] && w < rowPtr[q + 1]) { w = rowPtr[q + 1]; i = -1; }
            }
            if (w >= be) break;
            const int cnt = min(kWin, be - w);
            __syncthreads();
            stage_window(s_col, s_val, colIdx, values, w, cnt);
            __syncthreads();
            const int p0 = max(start, w), p1 = min(end, w + cnt);
            if (colok) add(p0, p1, w);
        }
    } else if constexpr (SLICED) {
        const int lane = (int)threadIdx.x % kWave, wv = (int)threadIdx.x / kWave;
        const bool leader = (threadIdx.x % L) == 0;
        const uint64_t below = (1ull << (lane & ~(L - 1))) - 1;   // lanes before this group's leader
        int *tab_s = s_tab, *tab_c = s_tab + RPB, *wcnt = s_tab + 2 * RPB;
        const int len = end - start;
        int done = 0;
        for (;;) {
            const int rem = len - done;
            const uint64_t m = __ballot(leader && rem > 0);
            if (lane == 0) wcnt[wv] = __popcll(m);
            __syncthreads();
            int nact = 0, base = 0;
#pragma unroll
            for (int k = 0; k < NW; k++) {
                const int c = wcnt[k];
                nact += c;
                if (k < wv) base += c;
            }
            if (nact == 0) break;                         // the same in every thread
            int lsl = 0;
            while ((2 << lsl) * nact <= kWin) lsl++;      // largest power of two with nact * 2^lsl <= kWin
            const int rank = base + __popcll(m & below);
            const int cnt = rem > 0 ? min(1 << lsl, rem) : 0;
            if (leader && rem > 0) {
                tab_s[rank] = start + done;
                tab_c[rank] = cnt;
            }
            __syncthreads();
            for (int i = threadIdx.x; i < (nact << lsl); i += kBlock) {
                const int q = i >> lsl, o = i & ((1 << lsl) - 1);
                if (o < tab_c[q]) {
                    s_col[i] = colIdx[tab_s[q] + o];
                    s_val[i] = values[tab_s[q] + o];
                }
            }
            __syncthreads();
            if (colok && cnt > 0)
                add(rank << lsl, (rank << lsl) + cnt, 0);
            done += cnt;
            __syncthreads();                              // before the next window's tables
        }
    }
    if constexpr (PARTS) {
#pragma unroll
        for (int k = 0; k < VW; k++) acc[k] += odd[k];
    }
    if (r < nr && colok && mine) store_g<true, VW>(C + (int64_t)r * ldc + col0, acc);
}

// ===========================================================================
// Row-balanced, parallel reduction, row-major (spmv_csr_vector,
// spmm_csr_vector_row).  A team of GT groups x L lanes owns one row; group
// g takes nonzeros start+g, start+g+GT, ..., U gathers in flight; the GT
// partial vectors are combined with a butterfly over stride L..GT*L/2.
// Overwrites.  Rows that a team would work on long after the others (a gather's
// latency per nonzero and group is what bounds them):
//   * beyond kTeamSteps nonzeros per group the team's whole wavefront sums the row;
//   * rows of `scout_row` or more nonzeros (kVecScoutRow, and kScoutMean times the
//     mean) are found and summed by the first `scouts` blocks of the launch,
//     kScoutCols columns and up to kScoutRows rows each.
// Power law (262144 rows, the longest 4900): nv = 1 165 -> 28 us, nv = 8 288 -> 61,
// nv = 64 600 -> 153; 2567 rows, the longest 346, nv = 8: 16 -> 5.6.  The common path's
// code is contiguous, the rare ones out of its way: the other order, or a real call
// for the scouts, cost regular matrices 10 to 70%.
// ===========================================================================
constexpr int kTeamSteps = 16;
constexpr int kVecScoutRow = 256;
// Work (nonzeros times lanes per group) below which no scouts are launched: a
// wavefront takes the longest row that there can be in a few steps.
constexpr int64_t kVecScoutWork = 1000000;

// acc += the nonzeros p0, p0 + stride, ... < e.  PARTS sums each U of them first,
// which shortens the chains (256 nonzeros to four groups: error 9.5e-8 of the
// result's norm, else 1.5e-7) and costs time (15000 rows of 100, nv = 64: 36.8 and 31.6 us).
template <int VW, int U, bool PARTS = false>
__device__ __forceinline__ void strided_accumulate(float (&acc)[VW], int p0, int e, int stride,
                                                   const int *__restrict__ colIdx,
                                                   const float *__restrict__ values,
                                                   const float *__restrict__ Bc, int64_t ldb) {
    if constexpr (U == 1) {
        for (unsigned p = p0; p < (unsigned)e; p += stride) {
            const int c = colIdx[p];
            const float a = values[p];
            float b[VW];
            load_g<float, VW>(b, Bc + (int64_t)c * ldb);
#pragma unroll
            for (int k = 0; k < VW; k++) acc[k] = __builtin_fmaf(a, b[k], acc[k]);
        }
        return;
    }
    const int n = e - p0;
    for (int i = 0; i < n; i += U * stride) {
        int c[U];
        float a[U], b[U][VW];
#pragma unroll
        for (int u = 0; u < U; u++) {          // padded with the last nonzero
            const int q = p0 + min(i + u * stride, n - 1);
            c[u] = colIdx[q];
            a[u] = values[q];
        }
#pragma unroll
        for (int u = 0; u < U; u++) load_g<float, VW>(b[u], Bc + (int64_t)c[u] * ldb);
        if constexpr (PARTS) {
            float part[VW];
#pragma unroll
            for (int k = 0; k < VW; k++) part[k] = a[0] * b[0][k];
#pragma unroll
            for (int u = 1; u < U; u++) {
                if (i + u * stride < n) {
#pragma unroll
                    for (int k = 0; k < VW; k++) part[k] = __builtin_fmaf(a[u], b[u][k], part[k]);
                }
            }
#pragma unroll
            for (int k = 0; k < VW; k++) acc[k] += part[k];
        } else {
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (i + u * stride < n) {
#pragma unroll
                    for (int k = 0; k < VW; k++) acc[k] = __builtin_fmaf(a[u], b[u][k], acc[k]);
                }
            }
        }
    }
}

// A scout block's share: the rows of scout_row or more nonzeros among its own
// (scout `me` of `all`), SW columns from `base` on.
template <int VW, int SW>
__device__ __forceinline__ void scout_rows(int me, int all, int nr, int base, int nv, int64_t ldb, int64_t ldc,
                                        const int *__restrict__ rowPtr, const int *__restrict__ colIdx,
                                        const float *__restrict__ values, const float *__restrict__ B,
                                        float *__restrict__ C, int scout_row) {
    constexpr int SL = SW / VW;                // lanes of a group
    constexpr int NW = kBlock / kWave;
    __shared__ uint16_t s_scout[kScoutList];
    __shared__ int s_n;
    __shared__ float s_part[NW][SW];
    const int t = threadIdx.x, ln = lane_id();
    scout_look(me, all, nr, rowPtr, scout_row, s_scout, &s_n);
    const int col0 = slab_col<VW>(base + (t % SL) * VW, nv);
    for (int i = 0; i < s_n; i++) {
        const int q = (int)scout_at(me, all, nr, s_scout[i]);
        float acc[VW];
#pragma unroll
        for (int k = 0; k < VW; k++) acc[k] = 0.f;
        if (col0 < nv)
            strided_accumulate<VW, 8>(acc, rowPtr[q] + t / SL, rowPtr[q + 1], kBlock / SL, colIdx, values,
                                      B + col0, ldb);
#pragma unroll
        for (int k = 0; k < VW; k++) acc[k] = butterfly_sum<SL, kWave>(acc[k]);
        if (ln < SL && col0 < nv) {
#pragma unroll
            for (int k = 0; k < VW; k++)       // the last lane may share its neighbour's columns
                if (col0 + k >= base) s_part[t / kWave][col0 - base + k] = acc[k];
        }
        __syncthreads();
        if (t < SW && base + t < nv) {
            float sum = s_part[0][t];
#pragma unroll
            for (int w = 1; w < NW; w++) sum += s_part[w][t];
            C[(int64_t)q * ldc + base + t] = sum;
        }
        __syncthreads();                       // before the next row's parts
    }
}

template <int VW, int L, int GT, int U, bool PARTS>
__global__ __launch_bounds__(kBlock) void k_csr_vector_rm(int nr, int nv, int64_t ldb, int64_t ldc,
                                                           const int *__restrict__ rowPtr,
                                                           const int *__restrict__ colIdx,
                                                           const float *__restrict__ values,
                                                           const float *__restrict__ B,
                                                           float *__restrict__ C, int slab_w,
                                                           int scouts, int scout_row) {
    constexpr int T = GT * L;                  // lanes per row
    constexpr int RPB = kBlock / T;
    static_assert(T <= kWave, "team larger than a wavefront");
    const int t = threadIdx.x;
    if (__builtin_expect((int)blockIdx.x < scouts, 0)) {
        constexpr int SW = L * VW < kScoutCols ? L * VW : kScoutCols;
        const int parts = (min(slab_w, nv - (int)blockIdx.y * slab_w) + SW - 1) / SW;
        const int me = (int)blockIdx.x / parts, all = scouts / parts;
        if (me < all)
            scout_rows<VW, SW>(me, all, nr, blockIdx.y * slab_w + (int)blockIdx.x % parts * SW, nv, ldb,
                               ldc, rowPtr, colIdx, values, B, C, scout_row);
        return;
    }
    const int b = xcd_remap(blockIdx.x - scouts, gridDim.x - scouts);
    const int r = b * RPB + t / T;
    const int g = (t % T) / L;
    const int col0 = slab_col<VW>(blockIdx.y * slab_w + (t % L) * VW, nv);
    const bool colok = col0 < nv;
    const float *__restrict__ Bc = B + (colok ? col0 : 0);
    float acc[VW];
#pragma unroll
    for (int k = 0; k < VW; k++) acc[k] = 0.f;
    int s = 0, e = 0;
    if (r < nr) { s = rowPtr[r]; e = rowPtr[r + 1]; }
    const bool apart = e - s >= scout_row;
    const bool wide = T < kWave && !apart && e - s > kTeamSteps * GT;
    const bool mine = r < nr && !apart && !wide;
    if (mine && colok) strided_accumulate<VW, U, PARTS>(acc, s + g, e, GT, colIdx, values, Bc, ldb);
#pragma unroll
    for (int k = 0; k < VW; k++) acc[k] = butterfly_sum<L, T>(acc[k]);
    if (mine && colok && g == 0) store_g<true, VW>(C + (int64_t)r * ldc + col0, acc);
    if constexpr (T < kWave) {
        uint64_t m = __ballot(wide && t % T == 0);
        if (__builtin_expect(m != 0, 0)) {
            const int ln = lane_id();
            for (; m; m &= m - 1) {
                const int o = __builtin_ctzll(m);
                const int q = read_lane(r, o), ps = read_lane(s, o), pe = read_lane(e, o);
#pragma unroll
                for (int k = 0; k < VW; k++) acc[k] = 0.f;
                if (colok)
                    strided_accumulate<VW, 4, PARTS>(acc, ps + ln / L, pe, kWave / L, colIdx, values, Bc, ldb);
#pragma unroll
                for (int k = 0; k < VW; k++) acc[k] = butterfly_sum<L, kWave>(acc[k]);
                if (ln < L && colok) store_g<true, VW>(C + (int64_t)q * ldc + col0, acc);
            }
        }
    }
}

// ===========================================================================
// Nnz-balanced, row-major, nv > 1 (spmm_coo_scalar_row, spmm_coo_vector_row,
// spmv_coo_vector with nv 2 or 4).  A wavefront owns G * NE consecutive
// nonzeros, G = 64 / L, and stages their (row, col, val) in its own LDS
// region with coalesced loads (one pad word per group, so that groups reading
// their k-th element hit distinct banks).  A group of L lanes sums NE
// consecutive ones in order, UNR gathers in flight, and adds every finished
// run of equal row to C with atomics.  Runs that cross group borders are
// joined first by a wave64 segmented scan over the groups' last runs, so that
// a row costs one atomic addition per wavefront it lies in.
//
// What bounds it: the atomics, then the gathers.  L2 takes about 19 G
// atomic accesses a second, one per 64-byte line that an instruction touches,
// so finished runs are added by the whole wavefront with their columns contiguous
// over the lanes (through LDS where a lane holds several columns), and runs are as
// long as the nonzeros of a wavefront allow.  Both reference algorithms run this kernel: without
// the join a row costs an atomic per group (64^3 27-point stencil, nv = 64:
// 395 us against 279 with it, before the contiguous additions; 133 with both;
// an atomic per eight nonzeros and four strided ones per float4 took 947 and
// 1902 us).
// ===========================================================================
template <int VW, int L, int NE>
__global__ __launch_bounds__(kBlock) void k_coo_rm(int nnz, int nv, int64_t ldb, int64_t ldc,
                                                    const int *__restrict__ rowIdx,
                                                    const int *__restrict__ colIdx,
                                                    const float *__restrict__ values,
                                                    const float *__restrict__ B,
                                                    float *__restrict__ C, int slab_w) {
    constexpr int G = kWave / L;               // groups per wavefront
    constexpr int CH = G * NE;                 // nonzeros per wavefront
    constexpr int PADN = CH + G;
    constexpr int WPB = kBlock / kWave;
    constexpr int UNR = NE < 8 ? NE : 8;
    __shared__ int s_row[WPB][PADN];
    __shared__ int s_col[WPB][PADN];
    __shared__ float s_val[WPB][PADN];
    __shared__ __align__(16) float s_flush[WPB][VW > 1 ? kWave * VW : 1];   // a group's columns in order
    const int wv = (int)threadIdx.x / kWave, ln = lane_id();
    const int64_t base = ((int64_t)xcd_remap(blockIdx.x, gridDim.x) * WPB + wv) * CH;
    if (base >= nnz) return;                   // the whole wavefront leaves; no barrier follows
    const int cnt = (int)min<int64_t>(CH, (int64_t)nnz - base);
    // Non-temporal where the gathered rows of B want the caches (64^3 stencil,
    // nv = 64: 132 us, plain loads 142); plain where the sparse operand is most
    // of the traffic and may be resident (nv = 4: 34.8 us, 39.6).
    constexpr bool NT = L >= 16;
    for (int i = ln; i < cnt; i += kWave) {
        const int j = i + i / NE;
        const int64_t p = base + i;
        s_row[wv][j] = NT ? ld_stream(rowIdx + p) : rowIdx[p];
        s_col[wv][j] = NT ? ld_stream(colIdx + p) : colIdx[p];
        s_val[wv][j] = NT ? ld_stream(values + p) : values[p];
    }
    wave_lds_sync();
    constexpr int W = L * VW;                  // columns of a group
    const int g = ln / L;
    const int col0 = blockIdx.y * slab_w + (ln % L) * VW;
    const bool colok = col0 < nv;
    const int n = max(0, min(NE, cnt - g * NE));   // nonzeros of this group
    const int at = n > 0 ? g * (NE + 1) : 0;       // (without any: the first group's, not added)
    const int *sr = s_row[wv] + at, *sc = s_col[wv] + at;
    const float *sv = s_val[wv] + at;
    const float *__restrict__ Bc = B + (colok ? col0 : 0);
    float *__restrict__ Cs = C + blockIdx.y * slab_w;
    const int ncol = nv - (int)blockIdx.y * slab_w;
    // Adds v to row r of C for the groups with `mine`.  An atomic instruction
    // costs one L2 access per 64-byte line it touches, so the wavefront's lanes
    // take the groups' columns in order, from LDS: 64 / W groups to an instruction.
    auto flush = [&](bool mine, int r, const float (&v)[VW]) {
        if constexpr (VW == 1) {
            if (mine && colok) unsafeAtomicAdd(Cs + (int64_t)r * ldc + ln % L, v[0]);
        } else {
            uint64_t m = __ballot(mine && ln % L == 0);
            if (m == 0) return;
            wave_lds_sync();                   // the previous flush has been read
            if (mine) store_vec<VW>(s_flush[wv] + ln * VW, v);
            wave_lds_sync();
            constexpr int P = W < kWave ? kWave / W : 1;
            while (m) {
                int o = -1;                    // first lane of the group whose columns this lane adds
#pragma unroll
                for (int k = 0; k < P; k++) {
                    if (m && ln / W % P == k) o = __builtin_ctzll(m);
                    m &= m - 1;                // (no bit left: stays 0)
                }
                const int row = __shfl(r, max(o, 0));
                if (o >= 0) {
#pragma unroll
                    for (int k = 0; k < W; k += kWave) {
                        const int c = k + ln % (W < kWave ? W : kWave);
                        if (c < ncol) unsafeAtomicAdd(Cs + (int64_t)row * ldc + c, s_flush[wv][o * VW + c]);
                    }
                }
            }
        }
    };
    int cur = INT_MAX, first = INT_MAX;        // rows of the running and of the first run
    bool one = true;                           // a single run so far
    float acc[VW], head[VW];
#pragma unroll
    for (int k = 0; k < VW; k++) acc[k] = head[k] = 0.f;
    if (n > 0) cur = first = sr[0];
    for (int e = 0; e < min(NE, cnt); e += UNR) {  // the same in every group
        float bv[UNR][VW];
#pragma unroll
        for (int u = 0; u < UNR; u++)          // padded with the last entry: no branch around loads
            load_vec<VW>(bv[u], Bc + (int64_t)sc[max(0, min(e + u, n - 1))] * ldb);
        // summed per block of UNR, the blocks' sums then in order: a run of 32
        // rounds no worse than the scan over eight lanes that it replaces
        float part[VW];
#pragma unroll
        for (int k = 0; k < VW; k++) part[k] = 0.f;
#pragma unroll
        for (int u = 0; u < UNR; u++) {
            const bool in = e + u < n;
            const int r = in ? sr[e + u] : cur;
            const float a = in ? sv[e + u] : 0.f;
            const bool ends = r != cur;
            if (__ballot(ends)) {
                if (ends) {
#pragma unroll
                    for (int k = 0; k < VW; k++) acc[k] += part[k];
                    if (one) {                 // the first run may continue the previous group's
#pragma unroll
                        for (int k = 0; k < VW; k++) head[k] = acc[k];
                    }
                }
                flush(ends && !one, cur, acc);
                if (ends) {
                    one = false;
                    cur = r;
#pragma unroll
                    for (int k = 0; k < VW; k++) acc[k] = part[k] = 0.f;
                }
            }
            if (in) {
#pragma unroll
                for (int k = 0; k < VW; k++) part[k] = __builtin_fmaf(a, bv[u][k], part[k]);
            }
        }
#pragma unroll
        for (int k = 0; k < VW; k++) acc[k] += part[k];
    }
    bool ends = n > 0;
    if constexpr (L < kWave) {
        // acc becomes the sum of a row's last runs up to this group, as long as
        // the groups between hold nothing else
        const int prow = __shfl_up(cur, L);
        const bool joins = ln >= L && prow == first;
        segmented_scan<L, VW>(acc, segment_id(ln % L == 0 && !(joins && one)));
#pragma unroll
        for (int k = 0; k < VW; k++) {
            const float p = __shfl_up(acc[k], L);
            if (joins && !one) head[k] += p;
        }
        // the last group of a row's runs adds it (the next group's head takes it otherwise)
        const int nfirst = __shfl_down(first, L);
        ends = ends && (ln >= kWave - L || nfirst != cur);
    }
    flush(n > 0 && !one, first, head);
    flush(ends, cur, acc);
}

// ===========================================================================
// Nnz-balanced, nv = 1 (spmv_coo_scalar, spmv_coo_vector).  A wavefront owns U
// chunks of 64 consecutive nonzeros, one per lane: all U * 64 gathers of x are
// issued, then each chunk is combined by row with the wave64 segmented scan
// (or a butterfly when it is one row), the sum of a row that goes on in the
// next chunk enters that chunk's first lane, and the last lane of each row
// adds it to y.  Rows are adjacent in y, so one instruction's additions fall
// in few lines.
// ===========================================================================
template <int U>
__global__ __launch_bounds__(kBlock) void k_coo_spmv(int nnz, const int *__restrict__ rowIdx,
                                                      const int *__restrict__ colIdx,
                                                      const float *__restrict__ values,
                                                      const float *__restrict__ x, int64_t ldx,
                                                      float *__restrict__ y, int64_t ldy) {
    const int ln = lane_id();
    const int64_t wave = (int64_t)xcd_remap(blockIdx.x, gridDim.x) * (kBlock / kWave) +
                         (int)threadIdx.x / kWave;
    const int64_t base = wave * (U * kWave);   // plain loads below: non-temporal ones cost 4 us
    if (base >= nnz) return;                   // the whole wavefront leaves
    int key[U], c[U];
    float v[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int64_t p = base + u * kWave + ln;
        key[u] = INT_MAX;
        c[u] = 0;
        v[u] = 0.f;
        if (p < nnz) {
            key[u] = rowIdx[p];
            c[u] = colIdx[p];
            v[u] = values[p];
        }
    }
#pragma unroll
    for (int u = 0; u < U; u++)
        if (key[u] != INT_MAX) v[u] *= x[(int64_t)c[u] * ldx];
    float carry = 0.f;                         // of a row that goes on into this chunk
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int klast = read_lane(key[u], kWave - 1);
        const int before = __shfl_up(key[u], 1);
        const bool begins = ln > 0 && before != key[u];
        const uint64_t heads = __ballot(begins);
        const bool single = heads == 0;        // one row in the whole chunk
        float s[1] = {v[u]};
        if (single) s[0] = butterfly_sum<1, kWave>(s[0]);
        else segmented_scan<1, 1>(s, segment_id(begins));
        // added to the chunk's sum, not to its first product: rows of 64 and more
        // round like chunks added one by one
        if (u > 0 && (single || ln < __builtin_ctzll(heads))) s[0] += carry;
        int next = __shfl_down(key[u], 1);
        if (ln == kWave - 1) next = INT_MAX;
        if (u + 1 < U) {                       // a row that goes on: its sum joins the next chunk's
            const int nk = read_lane(key[u + 1 < U ? u + 1 : u], 0);
            const float t = __shfl(s[0], kWave - 1);
            carry = nk == klast ? t : 0.f;
            if (ln == kWave - 1) next = nk;
        }
        if (key[u] != INT_MAX && next != key[u] &&
            !(single && ln != kWave - 1))
            unsafeAtomicAdd(y + (int64_t)key[u] * ldy, s[0]);
    }
}

// ===========================================================================
// Column-major variants.  B(:,j) is contiguous (ld >= nc), C(:,j) too
// (ld >= nr).  The reference re-reads A once per column (grid.y = nv);
// here a lane carries T columns so A is read ceil(nv/T) times.
// ===========================================================================

// Row-balanced, sequential (spmm_csr_scalar_col): one lane per row,
// for products too large for k_csr_stream that find no scratch for row-major copies.
template <int T>
__global__ __launch_bounds__(kBlock) void k_csr_scalar_cm(int nr, int nv, int64_t ldb, int64_t ldc,
                                                           const int *__restrict__ rowPtr,
                                                           const int *__restrict__ colIdx,
                                                           const float *__restrict__ values,
                                                           const float *__restrict__ B,
                                                           float *__restrict__ C) {
    __shared__ int s_col[kWin];
    __shared__ float s_val[kWin];
    const int b = xcd_remap(blockIdx.x, gridDim.x);
    const int r0 = b * kBlock;
    const int r = r0 + (int)threadIdx.x;
    const int j0 = blockIdx.y * T;
    const int nt = min(T, nv - j0);
    const int rlast = min(r0 + kBlock, nr);
    const int bs = rowPtr[r0], be = rowPtr[rlast];
    int start = 0, end = 0;
    if (r < nr) { start = rowPtr[r]; end = rowPtr[r + 1]; }
    float acc[T];
#pragma unroll
    for (int t = 0; t < T; t++) acc[t] = 0.f;
    const float *Bj = B + (int64_t)j0 * ldb;
    for (int w = bs; w < be; w = be - w > kWin ? w + kWin : be) {
        const int cnt = min(kWin, be - w);
        __syncthreads();
        stage_window(s_col, s_val, colIdx, values, w, cnt);
        __syncthreads();
        const int p0 = max(start, w), p1 = min(end, w + cnt);
        for (int p = p0; p < p1; p++) {
            const int c = s_col[p - w];
            const float a = s_val[p - w];
            float bv[T];
#pragma unroll
            for (int t = 0; t < T; t++) bv[t] = (t < nt) ? Bj[(int64_t)t * ldb + c] : 0.f;
#pragma unroll
            for (int t = 0; t < T; t++) acc[t] = acc[t] + a * bv[t];
        }
    }
    if (r < nr) {
#pragma unroll
        for (int t = 0; t < T; t++)
            if (t < nt) C[(int64_t)(j0 + t) * ldc + r] = acc[t];
    }
}

// Row-balanced, parallel (spmm_csr_vector_col, and spmv_csr_vector for
// column-major nv=1): L consecutive lanes per row stride its nonzeros.
template <int T, int L>
__global__ __launch_bounds__(kBlock) void k_csr_vector_cm(int nr, int nv, int64_t ldb, int64_t ldc,
                                                           const int *__restrict__ rowPtr,
                                                           const int *__restrict__ colIdx,
                                                           const float *__restrict__ values,
                                                           const float *__restrict__ B,
                                                           float *__restrict__ C) {
    constexpr int RPB = kBlock / L;
    const int b = xcd_remap(blockIdx.x, gridDim.x);
    const int r = b * RPB + (int)threadIdx.x / L;
    const int l = (int)threadIdx.x % L;
    const int j0 = blockIdx.y * T;
    const int nt = min(T, nv - j0);
    const float *Bj = B + (int64_t)j0 * ldb;
    float acc[T];
#pragma unroll
    for (int t = 0; t < T; t++) acc[t] = 0.f;
    int s = 0, e = 0;
    if (r < nr) { s = rowPtr[r]; e = rowPtr[r + 1]; }
    auto add = [&](int p0, int pe, int stride) {
        for (unsigned p = p0; p < (unsigned)pe; p += stride) {
            const int c = colIdx[p];
            const float a = values[p];
#pragma unroll
            for (int t = 0; t < T; t++)
                if (t < nt) acc[t] = __builtin_fmaf(a, Bj[(int64_t)t * ldb + c], acc[t]);
        }
    };
    const bool wide = L < kWave && e - s > kTeamSteps * L;
    if (!wide) add(s + l, e, L);
#pragma unroll
    for (int t = 0; t < T; t++) acc[t] = group_sum<L>(acc[t]);
    if (r < nr && !wide) {
        // Spread the T stores over the group's lanes.
#pragma unroll
        for (int t = 0; t < T; t++)
            if (t < nt && (t % L) == l) C[(int64_t)(j0 + t) * ldc + r] = acc[t];
    }
    if constexpr (L < kWave) {
        // rows beyond kTeamSteps nonzeros per lane: by the whole wavefront
        const int ln = lane_id();
        for (uint64_t m = __ballot(wide && l == 0); __builtin_expect(m != 0, 0); m &= m - 1) {
            const int o = __builtin_ctzll(m);
            const int q = read_lane(r, o);
#pragma unroll
            for (int t = 0; t < T; t++) acc[t] = 0.f;
            add(read_lane(s, o) + ln, read_lane(e, o), kWave);
#pragma unroll
            for (int t = 0; t < T; t++) acc[t] = group_sum<kWave>(acc[t]);
#pragma unroll
            for (int t = 0; t < T; t++)
                if (t < nt && t == ln) C[(int64_t)(j0 + t) * ldc + q] = acc[t];
        }
    }
}

// Nnz-balanced, parallel (spmm_coo_vector_col, and spmv_coo_vector for
// column-major nv=1): a wavefront takes 64 consecutive nonzeros per step,
// T columns per lane, segmented scan per column.
template <int T>
__global__ __launch_bounds__(kBlock) void k_coo_cm(int nnz, int nv, int64_t ldb, int64_t ldc,
                                                           const int *__restrict__ rowIdx,
                                                           const int *__restrict__ colIdx,
                                                           const float *__restrict__ values,
                                                           const float *__restrict__ B,
                                                           float *__restrict__ C) {
    const int ln = lane_id();
    const int wave = (xcd_remap(blockIdx.x, gridDim.x) * kBlock + (int)threadIdx.x) / kWave;
    const int64_t nwaves = (int64_t)gridDim.x * (kBlock / kWave);
    const int j0 = blockIdx.y * T;
    const int nt = min(T, nv - j0);
    const float *Bj = B + (int64_t)j0 * ldb;
    float *Cj = C + (int64_t)j0 * ldc;
    for (int64_t base = (int64_t)wave * kWave; base < nnz; base += nwaves * kWave) {
        const int64_t p = base + ln;
        const bool valid = p < nnz;
        int key = INT_MAX;
        float v[T];
#pragma unroll
        for (int t = 0; t < T; t++) v[t] = 0.f;
        if (valid) {
            key = rowIdx[p];
            const int c = colIdx[p];
            const float a = values[p];
#pragma unroll
            for (int t = 0; t < T; t++)
                if (t < nt) v[t] = a * Bj[(int64_t)t * ldb + c];
        }
        const int before = __shfl_up(key, 1);
        const bool begins = ln > 0 && before != key;
        if (__ballot(begins) == 0) {           // one row in the whole chunk
#pragma unroll
            for (int t = 0; t < T; t++) v[t] = group_sum<kWave>(v[t]);
            // Lane t adds column t: one atomic per column, spread over lanes.
#pragma unroll
            for (int t = 0; t < T; t++)
                if (ln == t && t < nt) unsafeAtomicAdd(Cj + (int64_t)t * ldc + key, v[t]);
        } else {
            segmented_scan<1, T>(v, segment_id(begins));
            const int next = __shfl_down(key, 1);
            const bool tail = valid && (ln == kWave - 1 || next != key);
            if (tail) {
#pragma unroll
                for (int t = 0; t < T; t++)
                    if (t < nt) unsafeAtomicAdd(Cj + (int64_t)t * ldc + key, v[t]);
            }
        }
    }
}

// ===========================================================================
// Row-major copies of column-major operands: src(j, i) = src[j * lds + i], i in
// [0, n), to dst[i * ldd + j] (TO_ROWS), or back; ADD adds to the destination
// atomically, as the accumulating algorithms do.  A block takes W columns of
// kFlipWords / W rows through LDS, so that both sides are read and written in
// runs: bound by the copy (131072 rows of 32 columns: 33 MB in 7.0 us, 4.8 TB/s).
// ===========================================================================
constexpr int kFlipWords = 2048;

template <int W, bool TO_ROWS, bool ADD>
__global__ __launch_bounds__(kBlock) void k_flip(const float *__restrict__ src, int64_t lds, int n,
                                                 int cols, float *__restrict__ dst, int64_t ldd) {
    constexpr int R = kFlipWords / W;          // rows of a tile
    constexpr int S = R + (W < 32 ? 64 / W : 1);   // stride that spreads a row's W words over the banks
    constexpr int N = kFlipWords / kBlock;     // words per thread
    __shared__ float tile[W * S];
    const int64_t i0 = (int64_t)blockIdx.x * R;
    const int j0 = (int)blockIdx.y * W, t = (int)threadIdx.x;
    const int ni = (int)min<int64_t>(R, (int64_t)n - i0), nj = min(W, cols - j0);
    float v[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int q = k * kBlock + t;
        const int i = TO_ROWS ? q % R : q / W, j = TO_ROWS ? q / R : q % W;
        v[k] = 0.f;
        if (i < ni && j < nj)
            v[k] = TO_ROWS ? src[(int64_t)(j0 + j) * lds + i0 + i] : src[(i0 + i) * lds + j0 + j];
    }
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int q = k * kBlock + t;
        const int i = TO_ROWS ? q % R : q / W, j = TO_ROWS ? q / R : q % W;
        tile[j * S + i] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int q = k * kBlock + t;
        const int i = TO_ROWS ? q / W : q % R, j = TO_ROWS ? q % W : q / R;
        if (i < ni && j < nj) {
            const float x = tile[j * S + i];
            float *d = dst + (TO_ROWS ? (i0 + i) * ldd + j0 + j : (int64_t)(j0 + j) * ldd + i0 + i);
            if constexpr (ADD) {
                if (x != 0.f) unsafeAtomicAdd(d, x);   // rows without a nonzero cost nothing
            } else {
                *d = x;
            }
        }
    }
}

// ===========================================================================
// Host side: template selection and launch.
// ===========================================================================
namespace {

constexpr int kCmCols = 8;      // columns per lane in the column-major kernels

int grid_for_waves(int64_t waves_needed) {
    // Persistent-ish grid for the grid-strided COO vector kernels: enough
    // workgroups to fill MI355X many times over, capped by the work.
    const int64_t blocks = (waves_needed + 3) / 4;
    const int64_t cap = 256 * 64;
    return (int)std::max<int64_t>(1, std::min<int64_t>(blocks, cap));
}

// Lanes per row for the parallel-reduction row-balanced kernels, from the
// mean row length (same thresholds as classic CSR-vector sub-wave sizing).
int lanes_for_mean(double mean, int cap) {
    int g = 2;
    if (mean > 4) g = 4;
    if (mean > 8) g = 8;
    if (mean > 16) g = 16;
    if (mean > 32) g = 32;
    if (mean > 64) g = 64;
    return std::min(g, cap);
}

template <typename F>
void with_lanes(int lanes, F &&f) {
    switch (lanes) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 16: f(std::integral_constant<int, 16>{}); break;
    case 32: f(std::integral_constant<int, 32>{}); break;
    default: f(std::integral_constant<int, 64>{}); break;
    }
}
template <typename F>
void with_vw(int vw, F &&f) {
    switch (vw) {
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    default: f(std::integral_constant<int, 1>{}); break;
    }
}

// Scouts beside `blocks` other blocks, for rows of at least `least` nonzeros:
// enough that each looks at no more than kScoutRows rows, and where the others
// leave the GPU room, more of them, up to kScoutBlocks, since all nonzeros may lie
// in a few hundred rows; a whole number per XCD, which leaves xcd_remap its
// meaning.  4096 rows, 512 neighbours of 2000 nonzeros, the others of 4, nv = 32,
// csr_scalar: 8 scouts 11400 us, 31 369, 62 176, 249 67.  Beside many blocks they cost: 30000
// rows of 128, nv = 1, csr_vector: 59 scouts 7.5 us, 234 8.6.
// `all`: scouts take every row of `least` nonzeros, however long the others are.
constexpr int kScoutBlocks = 256;
constexpr int kScoutWork = 4096;

Scouts scouts_for(int nr, int nnz, int nv, int slab_w, int least, int64_t blocks, bool all) {
    Scouts s;
    const int parts = div_up(std::min(nv, slab_w), std::min(slab_w, kScoutCols));
    const int room = blocks < kScoutBlocks ? kScoutBlocks : blocks <= 4 * kScoutBlocks ? kScoutBlocks / 2 : 0;
    const int rows = std::max(div_up(nr, kScoutRows), std::min({nr, nnz / kScoutWork, room}));
    s.blocks = div_up((int64_t)rows * parts, kNumXcd) * kNumXcd;
    s.row = all ? least
                : (int)std::min<int64_t>(INT_MAX, std::max<int64_t>(least, kScoutMean * (int64_t)nnz / std::max(1, nr)));
    return s;
}

// Rows per wavefront of k_csr_stream: most of a window of pairs, at most one
// row per lane and column.  Fewer pairs leave gathers unused (64^3 stencil,
// nv = 4: half a window 26.6 us, 3/4 18.6, one 16.1), more make a long row's
// wavefront later (power law, nv = 1: 60, 61, 83).
int stream_rows(int W, int nnz, int nr) {
    const double mean = std::max(1.0, (double)nnz / nr);
    return std::max(1, std::min(kWave / W, (int)(0.75 * stream_pairs(W) / mean)));
}

// Rows from which 5 to 8 columns run with a lane group per row (k_csr_scalar_rm):
// below, too few wavefronts of 32 rows hide their gathers.  nv = 8, stream / groups:
// 64^3 stencil 37.6 / 19.9 us, power law of 262144 rows 197 / 116, 131072 rows of 6
// 9.9 / 8.7, 100000 of 20 12.4 / 12.5; power law of 60916 27 / 42, 16384 rows of 32 6.2 / 14.8.
constexpr int kGroupRows8 = 98304;

// The slabs that make_slab gives to vectors as wide as the columns allow.
template <int VW, int L>
constexpr bool kSlabShape = VW == 4 || (VW == 2 && L <= 2) || (VW == 1 && L == 1);

dspmm_status_t csr_scalar_rm(int nr, int nnz, int nv, int64_t ldb, int64_t ldc, const int *rowPtr,
                             const int *colIdx, const float *values, const float *B, float *C,
                             hipStream_t st) {
    const Slab s = make_slab(nv, choose_vw_any(nv, 4));
    if (s.width <= (nr >= kGroupRows8 ? 4 : 8)) {
        with_vw(s.vw, [&](auto vw_c) {
            with_lanes(s.lanes, [&](auto l_c) {
                constexpr int VW_ = decltype(vw_c)::value, L_ = decltype(l_c)::value;
                if constexpr (VW_ * L_ <= 8 && kSlabShape<VW_, L_>) {
                    const int g = stream_rows(VW_ * L_, nnz, nr);
                    hipLaunchKernelGGL((k_csr_stream<VW_, L_, false>), dim3(div_up(nr, (int64_t)g * (kBlock / kWave))),
                                       dim3(kBlock), 0, st, nr, nv, ldb, ldc, rowPtr, colIdx, values,
                                       B, C, g);
                }
            });
        });
        return launch_status();
    }
    // sliced windows where a block's rows typically fill more than half a
    // window (the mean row length decides; a block that fits one window
    // runs the same code in both forms)
    const bool sliced = (double)nnz / std::max(1, nr) * (kBlock / s.lanes) > kWin / 2;
    with_vw(s.vw, [&](auto vw_c) {
        with_lanes(s.lanes, [&](auto l_c) {
            constexpr int VW_ = decltype(vw_c)::value, L_ = decltype(l_c)::value;
            if constexpr (VW_ * L_ >= 8 && kSlabShape<VW_, L_>) {
                const int blocks = div_up(nr, kBlock / L_);
                const int64_t others = (int64_t)blocks * s.count;
                const Scouts sc = scouts_for(nr, nnz, nv, s.width, kScoutRow, others, others < kScoutBlocks);
                dim3 grid(sc.blocks + blocks, s.count);
                if (sliced)
                    hipLaunchKernelGGL((k_csr_scalar_rm<VW_, L_, true>), grid, dim3(kBlock), 0, st, nr,
                                       nv, ldb, ldc, rowPtr, colIdx, values, B, C, s.width, sc.blocks,
                                       sc.row);
                else
                    hipLaunchKernelGGL((k_csr_scalar_rm<VW_, L_, false>), grid, dim3(kBlock), 0, st, nr,
                                       nv, ldb, ldc, rowPtr, colIdx, values, B, C, s.width, sc.blocks,
                                       sc.row);
            }
        });
    });
    return launch_status();
}

// Sums in parts, 5 to 32 columns (the native API's CSR_PARTS on FP32): rows of like
// lengths, so without scouts.
dspmm_status_t csr_parts_rm(int nr, int nnz, int nv, int64_t ldb, int64_t ldc, const int *rowPtr,
                            const int *colIdx, const float *values, const float *B, float *C,
                            hipStream_t st) {
    const Slab s = make_slab(nv, 4);
    if (nv < 5 || s.lanes > 8) return DSPMM_STATUS_NOT_SUPPORTED;
    const bool sliced = (double)nnz / std::max(1, nr) * (kBlock / s.lanes) > kWin / 2;
    with_lanes(s.lanes, [&](auto l_c) {
        constexpr int L_ = decltype(l_c)::value;
        if constexpr (L_ >= 2 && L_ <= 8) {
            auto launch = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3(div_up(nr, kBlock / L_)), dim3(kBlock), 0, st, nr, nv, ldb,
                                   ldc, rowPtr, colIdx, values, B, C, s.width, 0, INT_MAX);
            };
            if (sliced) launch(k_csr_scalar_rm<4, L_, true, true>);
            else launch(k_csr_scalar_rm<4, L_, false, true>);
        }
    });
    return launch_status();
}

constexpr int kVecFewWaves = 2048;     // of launch_csr_vector_rm: 8 per CU

template <int VW, int L, int GT>
void launch_csr_vector_rm(int nr, int nc, int nnz, int nv, int64_t ldb, int64_t ldc, const int *rowPtr,
                          const int *colIdx, const float *values, const float *B, float *C,
                          hipStream_t st, const Slab &s, bool parts) {
    if constexpr (GT * L <= kWave && kSlabShape<VW, L>) {
        // Scouts where a long row's wavefront would set the kernel's time.
        Scouts sc;
        const int blocks = div_up(nr, kBlock / (GT * L));
        if ((int64_t)nnz * L >= kVecScoutWork)
            sc = scouts_for(nr, nnz, nv, s.width, kVecScoutRow, (int64_t)blocks * s.count, false);
        dim3 grid(sc.blocks + blocks, s.count);
        // Four gathers in flight where a group has that many to make: with a B
        // that the L2s hold, only rows of more than 7 nonzeros per group gain (16384
        // rows of 32, nv = 64: 15.7 -> 13.4 us; 64^3 stencil, nv = 32: 98.7 -> 83.7;
        // 32^3 stencil, nv = 64, 6.3 per group: 15.0, with four 16.5).  One lane to
        // a row of B reaches a line per lane and gather, and enough wavefronts to hide
        // them want one at a time (rows of 600, nv = 2: 4800 rows 11.1 with four, 6.9;
        // rows of 1000: 2400 rows 7.8, 6.3; 1200 rows 5.2, 6.1).
        const double per = (double)nnz / ((double)GT * std::max(1, nr));
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(kBlock), 0, st, nr, nv, ldb, ldc, rowPtr, colIdx,
                               values, B, C, s.width, sc.blocks, sc.row);
        };
        if (parts)
            launch(k_csr_vector_rm<VW, L, GT, 4, true>);
        else if ((per > 7 && (L > 1 || (int64_t)blocks * (kBlock / kWave) < kVecFewWaves)) || (per > 2.5 && (int64_t)nc * nv >= (4 << 20)))
            launch(k_csr_vector_rm<VW, L, GT, 4, false>);
        else
            launch(k_csr_vector_rm<VW, L, GT, 1, false>);
    }
}

dspmm_status_t csr_vector_rm(int nr, int nc, int nnz, int nv, int64_t ldb, int64_t ldc, const int *rowPtr,
                             const int *colIdx, const float *values, const float *B, float *C,
                             hipStream_t st, int hint, int min_groups = 0) {
    Slab s = make_slab(nv, choose_vw_any(nv, 4));
    if (min_groups > 0 && s.lanes > 64 / min_groups) {
        s.lanes = 64 / min_groups;
        s.width = s.lanes * s.vw;
        s.count = div_up(nv, s.width);
    }
    const double mean = nr ? (double)nnz / nr : 0.0;
    int gt = hint > 0 ? pow2_floor(hint) : lanes_for_mean(mean, 64);
    gt = std::max(1, std::min(gt, 64 / s.lanes));
    const bool parts = min_groups > 0 && mean > 4.0 * gt;   // chains of more than four
    with_vw(s.vw, [&](auto vw_c) {
        with_lanes(s.lanes, [&](auto l_c) {
            constexpr int VW_ = decltype(vw_c)::value, L_ = decltype(l_c)::value;
            with_lanes(gt, [&](auto gt_c) {
                constexpr int GT_ = decltype(gt_c)::value;
                launch_csr_vector_rm<VW_, L_, GT_>(nr, nc, nnz, nv, ldb, ldc, rowPtr, colIdx, values, B, C,
                                                   st, s, parts);
            });
        });
    });
    return launch_status();
}

// Nonzeros per group of k_coo_rm (chunks per wavefront of k_coo_spmv): as many
// as leave the launch at least kCooWaves wavefronts, 32 per CU, since fewer
// runs are then cut; at most kCooPairs per wavefront, which its LDS holds.
constexpr int64_t kCooWaves = 8192;
constexpr int kCooPairs = 512;
constexpr int kCooRun = 16;      // nonzeros per row from which runs are long

template <int VW, int L, int NE>
void launch_coo_rm(int nnz, int nv, int64_t ldb, int64_t ldc, const int *rowIdx, const int *colIdx,
                   const float *values, const float *B, float *C, hipStream_t st, const Slab &s) {
    if constexpr (NE * (kWave / L) <= kCooPairs) {
        dim3 grid(div_up(nnz, (int64_t)(kBlock / L) * NE), s.count);
        hipLaunchKernelGGL((k_coo_rm<VW, L, NE>), grid, dim3(kBlock), 0, st, nnz, nv, ldb, ldc,
                           rowIdx, colIdx, values, B, C, s.width);
    }
}

template <int U>
void launch_coo_spmv(int nnz, const int *rowIdx, const int *colIdx, const float *values,
                     const float *x, int64_t ldx, float *y, int64_t ldy, hipStream_t st) {
    hipLaunchKernelGGL((k_coo_spmv<U>), dim3(div_up(nnz, kBlock * U)), dim3(kBlock), 0, st, nnz,
                       rowIdx, colIdx, values, x, ldx, y, ldy);
}

dspmm_status_t coo_spmv(int nnz, int64_t ldx, int64_t ldy, const int *rowIdx, const int *colIdx,
                        const float *values, const float *x, float *y, hipStream_t st) {
    // two chunks where that leaves kCooWaves wavefronts (power law, 3.2 M
    // nonzeros: one 20.9, two 20.8, four 22.0 us; stencil, 6.9 M: 26.4, 22.9, 24.3)
    if (nnz >= kCooWaves * kWave * 2)
        launch_coo_spmv<2>(nnz, rowIdx, colIdx, values, x, ldx, y, ldy, st);
    else
        launch_coo_spmv<1>(nnz, rowIdx, colIdx, values, x, ldx, y, ldy, st);
    return launch_status();
}

// ALG_COO_SCALAR and ALG_COO_VECTOR, row-major.
dspmm_status_t coo_rm(int nr, int nnz, int nv, int64_t ldb, int64_t ldc, const int *rowIdx,
                      const int *colIdx, const float *values, const float *B, float *C,
                      hipStream_t st) {
    if (nv == 1) return coo_spmv(nnz, ldb, ldc, rowIdx, colIdx, values, B, C, st);
    // Wide vectors gather more rows of B per instruction, narrow ones leave
    // fewer groups to share a flush: four floats where runs are long, else the
    // widest that leaves a group 16 lanes.  nv = 32, four / two floats: 64^3 stencil 57.8 /
    // 82.2 us, 16384 rows of 32 7.7 / 10.5, 100000 of 20 20.1 / 26.6, power law of mean 12 73.1 /
    // 70.1; nv = 16, four / one: 45.0 / 65.3, 6.5 / 8.7, 15.7 / 21.3, 59.1 / 56.2.
    const bool runs = nnz >= (int64_t)kCooRun * nr && (nv >= 16 || (nv >= 8 && nnz >= 800000));
    const int widest = nv >= 64 || runs ? 4 : nv >= 32 ? 2 : 1;
    const Slab s = make_slab(nv, choose_vw(nv, ldb, ldc, B, C, 4, widest));
    int ne = 32;
    while (ne > 8 && (ne * (kWave / s.lanes) > kCooPairs ||
                      (int64_t)nnz * s.lanes * s.count < kCooWaves * kWave * ne))
        ne /= 2;
    with_vw(s.vw, [&](auto vw_c) {
        with_lanes(s.lanes, [&](auto l_c) {
            constexpr int VW_ = decltype(vw_c)::value, L_ = decltype(l_c)::value;
            if constexpr (VW_ * L_ >= 2) {
                switch (ne) {
                case 32: launch_coo_rm<VW_, L_, 32>(nnz, nv, ldb, ldc, rowIdx, colIdx, values, B, C, st, s); break;
                case 16: launch_coo_rm<VW_, L_, 16>(nnz, nv, ldb, ldc, rowIdx, colIdx, values, B, C, st, s); break;
                default: launch_coo_rm<VW_, L_, 8>(nnz, nv, ldb, ldc, rowIdx, colIdx, values, B, C, st, s); break;
                }
            }
        });
    });
    return launch_status();
}

// Products up to which k_csr_stream, which gathers for long rows with all
// lanes, is the faster kernel (16384 rows of 32, nv = 2: 52 -> 7 us; power law of
// 16806 rows, nv = 16: 336 -> 25; 131072 rows of 6, nv = 8, 6.3 M: 33 against 41).
constexpr int64_t kStreamProducts = 6000000;

dspmm_status_t csr_scalar_cm(int nr, int nnz, int nv, int64_t ldb, int64_t ldc, const int *rowPtr,
                             const int *colIdx, const float *values, const float *B, float *C,
                             hipStream_t st) {
    if ((int64_t)nnz * nv >= kStreamProducts) {
        dim3 grid(div_up(nr, kBlock), div_up(nv, kCmCols));
        hipLaunchKernelGGL((k_csr_scalar_cm<kCmCols>), grid, dim3(kBlock), 0, st, nr, nv, ldb, ldc,
                           rowPtr, colIdx, values, B, C);
        return launch_status();
    }
    with_lanes(std::min(pow2_ceil(nv), kCmCols), [&](auto l_c) {
        constexpr int L_ = decltype(l_c)::value;
        if constexpr (L_ <= kCmCols) {
            const int g = stream_rows(L_, nnz, nr);
            dim3 grid(div_up(nr, (int64_t)g * (kBlock / kWave)), div_up(nv, L_));
            hipLaunchKernelGGL((k_csr_stream<1, L_, true>), grid, dim3(kBlock), 0, st, nr, nv, ldb, ldc,
                               rowPtr, colIdx, values, B, C, g);
        }
    });
    return launch_status();
}

dspmm_status_t csr_vector_cm(int nr, int nnz, int nv, int64_t ldb, int64_t ldc, const int *rowPtr,
                             const int *colIdx, const float *values, const float *B, float *C,
                             hipStream_t st, int hint) {
    const double mean = nr ? (double)nnz / nr : 0.0;
    const int L = hint > 0 ? std::min(64, pow2_floor(hint)) : lanes_for_mean(mean, 64);
    const int T = std::min(pow2_ceil(nv), kCmCols);
    with_lanes(L, [&](auto l_c) {
        constexpr int L_ = decltype(l_c)::value;
        with_lanes(T, [&](auto t_c) {
            constexpr int T_ = decltype(t_c)::value;
            if constexpr (T_ <= kCmCols) {
                dim3 grid(div_up(nr, kBlock / L_), div_up(nv, T_));
                hipLaunchKernelGGL((k_csr_vector_cm<T_, L_>), grid, dim3(kBlock), 0, st, nr, nv, ldb,
                                   ldc, rowPtr, colIdx, values, B, C);
            }
        });
    });
    return launch_status();
}

// ALG_COO_SCALAR and ALG_COO_VECTOR, column-major.
dspmm_status_t coo_cm(int nnz, int nv, int64_t ldb, int64_t ldc, const int *rowIdx,
                             const int *colIdx, const float *values, const float *B, float *C,
                             hipStream_t st) {
    with_lanes(std::min(pow2_ceil(nv), kCmCols), [&](auto t_c) {
        constexpr int T_ = decltype(t_c)::value;
        if constexpr (T_ <= kCmCols) {
            dim3 grid(grid_for_waves(((int64_t)nnz + kWave - 1) / kWave), div_up(nv, T_));
            hipLaunchKernelGGL((k_coo_cm<T_>), grid, dim3(kBlock), 0, st, nnz, nv, ldb, ldc, rowIdx,
                               colIdx, values, B, C);
        }
    });
    return launch_status();
}

// C's copy starts on a line of its own.
size_t align_words(int64_t words) { return ((size_t)words + 63) / 64 * 64; }

template <int W>
void launch_flip(bool to_rows, bool add, const float *src, int64_t lds, int n, int cols, float *dst,
                 int64_t ldd, hipStream_t st) {
    const dim3 grid(div_up(n, kFlipWords / W), div_up(cols, W));
    if (to_rows)
        hipLaunchKernelGGL((k_flip<W, true, false>), grid, dim3(kBlock), 0, st, src, lds, n, cols, dst, ldd);
    else if (add)
        hipLaunchKernelGGL((k_flip<W, false, true>), grid, dim3(kBlock), 0, st, src, lds, n, cols, dst, ldd);
    else
        hipLaunchKernelGGL((k_flip<W, false, false>), grid, dim3(kBlock), 0, st, src, lds, n, cols, dst, ldd);
}

dspmm_status_t flip(bool to_rows, bool add, const float *src, int64_t lds, int n, int cols, float *dst,
                    int64_t ldd, hipStream_t st) {
    if (cols <= 2) launch_flip<2>(to_rows, add, src, lds, n, cols, dst, ldd, st);
    else if (cols <= 4) launch_flip<4>(to_rows, add, src, lds, n, cols, dst, ldd, st);
    else if (cols <= 8) launch_flip<8>(to_rows, add, src, lds, n, cols, dst, ldd, st);
    else if (cols <= 16) launch_flip<16>(to_rows, add, src, lds, n, cols, dst, ldd, st);
    else launch_flip<32>(to_rows, add, src, lds, n, cols, dst, ldd, st);
    return launch_status();
}

}  // namespace

constexpr int kFlipChain = 16;

// Column-major operands on row-major copies of B and C in `scratch`, `cols`
// columns at a time, with the row-major kernel of the same algorithm.
size_t compat_flipped_bytes(int nr, int nc, int nv) {
    return (align_words((int64_t)nc * nv) + (size_t)nr * (size_t)nv) * sizeof(float);
}

dspmm_status_t launch_compat_flipped(int which, int nr, int nc, int nnz, int nv, const int *rowPtr,
                                     const int *rowIdx, const int *colIdx, const float *values,
                                     const float *B, float *C, float *scratch, int cols,
                                     hipStream_t st) {
    const bool coo = which == K_SPMM_COO_SCALAR_COL || which == K_SPMM_COO_VECTOR_COL;
    dspmm_status_t s = DSPMM_STATUS_SUCCESS;
    // k_csr_vector_cm gives a row up to 64 lanes; the few groups that many columns
    // leave would add longer chains, which round worse: at least one for each
    // kFlipChain nonzeros of the mean row.  Error of the result's norm, in place / here
    // / with as few groups as columns allow: 2048 rows of 256, nv = 128 7.8e-8 / 7.9e-8
    // / 2.0e-7 (40 / 25 / 32 us); 7500 of 200, nv = 64 7.6e-8 / 7.8e-8 / 1.3e-7 (335 / 59
    // / 37); 15000 of 100, nv = 64 7.3e-8 / 7.3e-8 / 9.9e-8 (354 / 44 / 42).
    int groups = 1;
    while (groups < 64 && (int64_t)groups * kFlipChain * nr < nnz) groups *= 2;
    for (int j = 0; j < nv && s == DSPMM_STATUS_SUCCESS; j += cols) {
        const int w = std::min(cols, nv - j);
        float *Bt = scratch, *Ct = scratch + align_words((int64_t)nc * w);
        s = flip(true, false, B + (int64_t)j * nc, nc, nc, w, Bt, w, st);
        if (s == DSPMM_STATUS_SUCCESS && coo)
            s = launch_fill_zero(Ct, (size_t)nr * (size_t)w * sizeof(float), st);
        if (s != DSPMM_STATUS_SUCCESS) break;
        if (coo) s = coo_rm(nr, nnz, w, w, w, rowIdx, colIdx, values, Bt, Ct, st);
        else if (which == K_SPMM_CSR_SCALAR_COL)
            s = csr_scalar_rm(nr, nnz, w, w, w, rowPtr, colIdx, values, Bt, Ct, st);
        else s = csr_vector_rm(nr, nc, nnz, w, w, w, rowPtr, colIdx, values, Bt, Ct, st, 0, groups);
        if (s == DSPMM_STATUS_SUCCESS) s = flip(false, coo, Ct, w, nr, w, C + (int64_t)j * nr, nr, st);
    }
    return s;
}

// Shared entry for the 12 launchers, the dispatcher and the native API.
dspmm_status_t launch_compat(int which, int nr, int nc, int nnz, int nv, int64_t ldb, int64_t ldc,
                             const int *rowPtr, const int *rowIdx, const int *colIdx,
                             const float *values, const float *B, float *C, hipStream_t st,
                             int hint) {
    const bool coo = which == K_SPMV_COO_SCALAR || which == K_SPMV_COO_VECTOR ||
                     which == K_SPMM_COO_SCALAR_ROW || which == K_SPMM_COO_VECTOR_ROW ||
                     which == K_SPMM_COO_SCALAR_COL || which == K_SPMM_COO_VECTOR_COL;
    if (nr == 0 || nv == 0) return DSPMM_STATUS_SUCCESS;
    if (coo && nnz == 0) return DSPMM_STATUS_SUCCESS;   // nothing to accumulate
    switch (which) {
    case K_SPMV_CSR_SCALAR:
    case K_SPMM_CSR_SCALAR_ROW:
        return csr_scalar_rm(nr, nnz, nv, ldb, ldc, rowPtr, colIdx, values, B, C, st);
    case K_CSR_PARTS_ROW:
        return csr_parts_rm(nr, nnz, nv, ldb, ldc, rowPtr, colIdx, values, B, C, st);
    case K_SPMV_CSR_VECTOR:
    case K_SPMM_CSR_VECTOR_ROW:
        return csr_vector_rm(nr, nc, nnz, nv, ldb, ldc, rowPtr, colIdx, values, B, C, st, hint);
    case K_SPMV_COO_SCALAR:
    case K_SPMM_COO_SCALAR_ROW:
    case K_SPMV_COO_VECTOR:
    case K_SPMM_COO_VECTOR_ROW:
        return coo_rm(nr, nnz, nv, ldb, ldc, rowIdx, colIdx, values, B, C, st);
    case K_SPMM_CSR_SCALAR_COL:
        return csr_scalar_cm(nr, nnz, nv, ldb, ldc, rowPtr, colIdx, values, B, C, st);
    case K_SPMM_CSR_VECTOR_COL:
        return csr_vector_cm(nr, nnz, nv, ldb, ldc, rowPtr, colIdx, values, B, C, st, hint);
    case K_SPMM_COO_SCALAR_COL:
    case K_SPMM_COO_VECTOR_COL:
        return coo_cm(nnz, nv, ldb, ldc, rowIdx, colIdx, values, B, C, st);
    }
    return DSPMM_STATUS_INVALID_VALUE;
}

}  // namespace dspmm
