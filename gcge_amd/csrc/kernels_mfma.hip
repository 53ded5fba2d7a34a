// FP64 matrix-core (MFMA) kernels for the dense contractions of GCG:
// the Gram blocks of MultiVecInnerProd / MultiVecQtAP (X^T Y) and the
// tall-skinny products of MultiVecLinearComb (X C).
//
// v_mfma_f64_16x16x4_f64 computes D(16x16) += A(16x4) B(4x16) on one
// wavefront.  Lane l supplies A[l%16][l/16] and B[l/16][l%16] and holds
// D[l/16 + 4v][l%16] in element v of its 4-double accumulator (a layout
// any slip in which fails the Gram and LinearComb parity tests of
// tests/test_gpu_slots.py).
#include <hip/hip_runtime.h>
#include <cstdint>
#include <utility>

#include "app_hip_internal.h"
#include "kernels.h"
#include "sell_rows.h"
#include "tuner.h"

namespace gcge {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kWG = 256;
constexpr int kXCD = 8;

__device__ __forceinline__ int64_t xcd_swizzle(int64_t bid, int64_t nblk)
{
    const int64_t q = nblk / kXCD, r = nblk % kXCD;
    const int64_t x = bid % kXCD, k = bid / kXCD;
    return (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + k;
}

__device__ __forceinline__ d4 mfma(double a, double b, d4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// ---------------------------------------------------------------------
// Gram: G (m x n) = X^T Y, over one chunk of rows per workgroup, 16 rows a
// stage through LDS; the partial tiles of the chunks are summed by sum_chunks
// in a fixed order (deterministic, no atomics).
//
// Blocks of more than 64 columns on both sides: a workgroup owns a 128 x 128
// tile of G, its four waves 64 x 64 quadrants (4 x 4 MFMA tiles).  Rows are
// stored column-major (row index fastest, padded to 17) so each 16-lane MFMA
// operand read covers the banks once.  Each thread fetches 4 consecutive rows
// (one 32-byte load) of its columns of each operand, and the next stage's
// loads are issued into registers before the current stage's MFMAs, so HBM
// latency overlaps the matrix-core work; 98 VGPRs + 128 AGPRs, two waves per
// SIMD, the matrix cores busy 80 % (460 x 120 at 2 M rows: 4.3 ms).  The
// layout of the narrow kernel below, double buffered with one barrier, and
// 160-wide tiles where they pad less (75 % busy) measured no faster.
// ---------------------------------------------------------------------
constexpr int kGK = 16;        // rows per stage
constexpr int kGKP = kGK + 1;
constexpr int kGRG = kGK / 4;  // 4-row groups per stage

__global__ __launch_bounds__(kWG) void k_gram_wide(
    int64_t nrows, int m, int n, const double *__restrict__ X, int64_t ldx,
    const double *__restrict__ Y, int64_t ldy, int tm, int tn, int64_t rows_per_chunk,
    int lower_only, double *__restrict__ partial)
{
    constexpr int WN = 2, NB = 4;
    constexpr int TM = 128, TN = 128;
    constexpr int XC = TM * kGRG / kWG;  // X columns per thread
    constexpr int YC = TN * kGRG / kWG;  // Y columns per thread
    __shared__ double sx[TM * kGKP];
    __shared__ double sy[TN * kGKP];
    const int64_t lb = xcd_swizzle(blockIdx.x, gridDim.x);
    const int tiles = tm * tn;
    const int chunk = (int)(lb / tiles);
    const int t = (int)(lb % tiles);
    const int bi = t / tn, bj = t % tn;
    double *out = partial + ((int64_t)chunk * tiles + t) * (TM * TN);
    const int i0 = bi * TM, j0 = bj * TN;
    if (lower_only && i0 + TM - 1 < j0) {  // wholly above the diagonal
        for (int e = threadIdx.x; e < TM * TN; e += kWG) out[e] = 0.0;
        return;
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int wm = wave / WN, wn = wave % WN;
    const int li = lane & 15, lk = lane >> 4;
    const int64_t rbeg = (int64_t)chunk * rows_per_chunk;
    int64_t rend = rbeg + rows_per_chunk;
    if (rend > nrows) rend = nrows;
    // this thread's slots in a stage: rows 4*rg .. 4*rg+3 of its columns
    // (one 32-byte load per column; kGRG lanes cover the stage's rows of a
    // column, so a wave instruction reads whole row segments of 64/kGRG
    // columns, and only the thread's column addresses stay live)
    const int rg = threadIdx.x % kGRG;
    const int cg = threadIdx.x / kGRG;
    const double *xc[XC], *yc[YC];
    bool xok[XC], yok[YC];
#pragma unroll
    for (int c = 0; c < XC; ++c) {
        const int cc = cg * XC + c;
        xok[c] = i0 + cc < m;
        xc[c] = X + (int64_t)(xok[c] ? i0 + cc : 0) * ldx + 4 * rg;
    }
#pragma unroll
    for (int c = 0; c < YC; ++c) {
        const int cc = cg * YC + c;
        yok[c] = j0 + cc < n;
        yc[c] = Y + (int64_t)(yok[c] ? j0 + cc : 0) * ldy + 4 * rg;
    }
    double px[XC][4], py[YC][4];
    auto fetch = [&](int64_t r0) {
        const int64_t r = r0 + 4 * rg;
        if (r + 4 <= rend) {
#pragma unroll
            for (int c = 0; c < XC; ++c) {
                const d4 v = xok[c] ? *reinterpret_cast<const d4 *>(xc[c] + r0)
                                    : d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int q = 0; q < 4; ++q) px[c][q] = v[q];
            }
#pragma unroll
            for (int c = 0; c < YC; ++c) {
                const d4 v = yok[c] ? *reinterpret_cast<const d4 *>(yc[c] + r0)
                                    : d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int q = 0; q < 4; ++q) py[c][q] = v[q];
            }
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const bool rok = r + q < rend;
#pragma unroll
                for (int c = 0; c < XC; ++c) px[c][q] = (rok && xok[c]) ? xc[c][r0 + q] : 0.0;
#pragma unroll
                for (int c = 0; c < YC; ++c) py[c][q] = (rok && yok[c]) ? yc[c][r0 + q] : 0.0;
            }
        }
    };
    d4 acc[4][NB];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = d4{0.0, 0.0, 0.0, 0.0};
    if (rbeg < rend) fetch(rbeg);
    for (int64_t r0 = rbeg; r0 < rend; r0 += kGK) {
#pragma unroll
        for (int c = 0; c < XC; ++c)
#pragma unroll
            for (int q = 0; q < 4; ++q) sx[(cg * XC + c) * kGKP + 4 * rg + q] = px[c][q];
#pragma unroll
        for (int c = 0; c < YC; ++c) {
            // (always so; without the test the compiler's code is 5-10 % slower
            // where a tile has few columns: 300 x 65 at 2 M rows 3.23 -> 3.55
            // ms, 340 x 220 6.42 -> 6.71)
            if (cg * YC + c < TN) {
#pragma unroll
                for (int q = 0; q < 4; ++q) sy[(cg * YC + c) * kGKP + 4 * rg + q] = py[c][q];
            }
        }
        __syncthreads();
        if (r0 + kGK < rend) fetch(r0 + kGK);
#pragma unroll 2
        for (int kk = 0; kk < kGK / 4; ++kk) {
            const int row = kk * 4 + lk;
            double av[4], bv[NB];
#pragma unroll
            for (int a = 0; a < 4; ++a) av[a] = sx[(wm * 64 + a * 16 + li) * kGKP + row];
#pragma unroll
            for (int b = 0; b < NB; ++b) bv[b] = sy[(wn * 16 * NB + b * 16 + li) * kGKP + row];
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < NB; ++b) acc[a][b] = mfma(av[a], bv[b], acc[a][b]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int ii = wm * 64 + a * 16 + lk + 4 * v;
                const int jj = wn * 16 * NB + b * 16 + li;
                out[ii * TN + jj] = acc[a][b][v];
            }
}

// ---------------------------------------------------------------------
// A side of at most 64 columns (the block width of most orthogonalization
// Grams): a workgroup owns a 16 MA x 16 NB tile as wide as that side, with
// MA chosen to pad the other least, and each of its four waves computes the
// whole tile over 4 of a stage's 16 rows; the four sums are added through LDS
// at the end, in order.
//
// 8 lanes load the 16 rows of a column, two rows each (whole 128-byte lines),
// one stage ahead into registers and from there into the other of two LDS
// buffers (one barrier per stage).  The row pairs of a column are permuted by
// bits 1-3 of its index, so that 16 columns' operand reads cover the banks
// once, without padding.
//
// Bound by HBM, and by the matrix cores for the padding of the narrow side to
// 16 columns; small ones by their launches.  Waves side by side over 256 x 16
// NB and 64 x 64 tiles, as before, multiplied zeros for up to three of four
// waves: 60 x 12 at 17 K rows 12.7 us, now 7.0; 200 x 40 at 2.1 M rows 1.25
// ms, now 1.12; 40 x 40 there 0.44, now 0.34 (projections of 110,592 rows, 100
// x 10: 77 -> 50 us, 300 x 60: 228 -> 159 us, whole calls).  Loads two stages
// further ahead measured the same.
// ---------------------------------------------------------------------
typedef double d2 __attribute__((ext_vector_type(2)));
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

template <int MA, int NB>
__global__ __launch_bounds__(kWG, 2) void k_gram_narrow(
    int64_t nrows, int m, int n, const double *__restrict__ X, int64_t ldx,
    const double *__restrict__ Y, int64_t ldy, int tm, int64_t rows_per_chunk,
    double *__restrict__ partial)
{
    constexpr int TM = 16 * MA, TN = 16 * NB;
    constexpr int kLoads = (TM + TN + 31) / 32;  // of 8 columns, per wave
    __shared__ double stage[2][kLoads * 32 * kGK];
    const int64_t lb = xcd_swizzle(blockIdx.x, gridDim.x);
    const int chunk = (int)(lb / tm), t = (int)(lb % tm);
    const int i0 = t * TM;
    double *out = partial + lb * (TM * TN);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int li = lane & 15, lk = lane >> 4;
    const int64_t rbeg = (int64_t)chunk * rows_per_chunk;
    int64_t rend = rbeg + rows_per_chunk;
    if (rend > nrows) rend = nrows;
    const int nstages = rend > rbeg ? (int)((rend - rbeg + kGK - 1) / kGK) : 0;
    // load u of the wave: columns 8 q .. 8 q + 7 of the tile's X and Y
    // columns, q = 4 u + wave; columns past m or n read the last one (their
    // results are not used)
    const int pair = (lane & 7) ^ ((wave & 1) * 4 + (lane >> 4));
    const double *src[kLoads];
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
        const int cc = (4 * u + wave) * 8 + (lane >> 3);
        const int ic = i0 + cc < m ? i0 + cc : m - 1;
        const int jc = cc - TM < n ? cc - TM : n - 1;
        src[u] = cc < TM ? X + (int64_t)ic * ldx : Y + (int64_t)jc * ldy;
        src[u] += rbeg + 2 * pair;
    }
    d2 reg[kLoads];
    auto load = [&](int s) {
        if (s >= nstages) return;  // uniform
        const int64_t row = (int64_t)s * kGK, left = rend - rbeg - row;
        // (the rows' test around all loads: one around each would end in a
        // wait for it)
        if (left >= kGK) {
#pragma unroll
            for (int u = 0; u < kLoads; ++u)
                reg[u] = *reinterpret_cast<const d2u *>(src[u] + row);
        } else {
#pragma unroll
            for (int u = 0; u < kLoads; ++u) {
                reg[u][0] = 2 * pair < left ? src[u][row] : 0.0;
                reg[u][1] = 2 * pair + 1 < left ? src[u][row + 1] : 0.0;
            }
        }
    };
    auto store = [&](double *to) {
#pragma unroll
        for (int u = 0; u < kLoads; ++u)
            *reinterpret_cast<d2 *>(to + (4 * u + wave) * 128 + lane * 2) = reg[u];
    };
    d4 acc[MA][NB];
#pragma unroll
    for (int a = 0; a < MA; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = d4{0.0, 0.0, 0.0, 0.0};
    // row 4 wave + lk of column li of a 16-column tile
    const int at = li * kGK + ((2 * wave + (lk >> 1)) ^ (li >> 1)) * 2 + (lk & 1);
    if (nstages > 0) {
        load(0);
        store(stage[0]);
        load(1);
    }
    for (int s = 0; s < nstages; ++s) {
        __syncthreads();
        // the other buffer was last read before this barrier
        if (s + 1 < nstages) store(stage[(s + 1) & 1]);
        load(s + 2);
        const double *from = stage[s & 1] + at;
        double av[MA], bv[NB];
#pragma unroll
        for (int a = 0; a < MA; ++a) av[a] = from[a * 256];
#pragma unroll
        for (int b = 0; b < NB; ++b) bv[b] = from[(MA + b) * 256];
#pragma unroll
        for (int a = 0; a < MA; ++a)
#pragma unroll
            for (int b = 0; b < NB; ++b) acc[a][b] = mfma(av[a], bv[b], acc[a][b]);
    }
    // the waves' sums in order, a column of tiles at a time: waves 1 and 2
    // leave theirs in the two buffers, then wave 3 in the first
    auto put = [&](double *to, int b) {
#pragma unroll
        for (int a = 0; a < MA; ++a)
#pragma unroll
            for (int v = 0; v < 4; ++v) to[(a * 4 + v) * 64 + lane] = acc[a][b][v];
    };
    auto add = [&](const double *from, int b) {
#pragma unroll
        for (int a = 0; a < MA; ++a)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[a][b][v] += from[(a * 4 + v) * 64 + lane];
    };
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        __syncthreads();
        if (wave == 1) put(stage[0], b);
        if (wave == 2) put(stage[1], b);
        __syncthreads();
        if (wave == 0) {
            add(stage[0], b);
            add(stage[1], b);
        }
        __syncthreads();
        if (wave == 3) put(stage[0], b);
        __syncthreads();
        if (wave == 0) {
            add(stage[0], b);
#pragma unroll
            for (int a = 0; a < MA; ++a)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    out[(a * 16 + lk + 4 * v) * TN + b * 16 + li] = acc[a][b][v];
        }
    }
}

// Tile shape of a Gram of m x n: 128 x 128, or 16 ma x 16 nb with a side of
// at most 64 columns, computed as its transpose (swap) when that is X's.
struct GramShape {
    int ma, nb;
    bool wide, swap;
    int rows() const { return wide ? 128 : 16 * ma; }
    int cols() const { return wide ? 128 : 16 * nb; }
};

GramShape gram_shape(int m, int n)
{
    if (n > 64 && m > 64) return GramShape{0, 0, true, false};
    const bool swap = n > 64;
    const int t = ((swap ? n : m) + 15) / 16, nb = ((swap ? m : n) + 15) / 16;
    // accumulators of at most 21 tiles
    const int most = nb <= 2 ? 8 : nb == 3 ? 7 : 5;
    const int tm = (t + most - 1) / most;
    return GramShape{(t + tm - 1) / tm, nb, false, swap};
}

struct GramPlanM {
    GramShape sh;
    int tm, tn, nchunk;
    int64_t rows_per_chunk;
    int64_t tile_doubles() const { return (int64_t)sh.rows() * sh.cols(); }
};

int64_t gram_tiles(int m, int n)
{
    const GramShape sh = gram_shape(m, n);
    if (sh.swap) std::swap(m, n);
    return (int64_t)((m + sh.rows() - 1) / sh.rows()) * ((n + sh.cols() - 1) / sh.cols());
}

// Row chunking: at most max_wg workgroups in total (256 CUs, two resident
// each, at the default 512: one more than that runs alone in a second
// round and doubles the time) and at least min_rows rows (min_rows / 16
// stages) per chunk, so small problems still spread over many workgroups
// instead of a few walking all their rows.
GramPlanM plan_with(int64_t nrows, int m, int n, int64_t min_rows, int64_t max_wg)
{
    GramPlanM p;
    p.sh = gram_shape(m, n);
    if (p.sh.swap) std::swap(m, n);
    p.tm = (m + p.sh.rows() - 1) / p.sh.rows();
    p.tn = (n + p.sh.cols() - 1) / p.sh.cols();
    const int64_t tiles = (int64_t)p.tm * p.tn;
    int64_t want = max_wg / tiles;
    int64_t cap = (nrows + min_rows - 1) / min_rows;
    int64_t nc = want < cap ? want : cap;
    if (nc < 1) nc = 1;
    int64_t rpc = (nrows + nc - 1) / nc;
    rpc = (rpc + kGK - 1) / kGK * kGK;
    p.rows_per_chunk = rpc;
    p.nchunk = (int)((nrows + rpc - 1) / rpc);
    if (p.nchunk < 1) p.nchunk = 1;
    return p;
}

// Tuner candidates (min_rows, max_wg); the default is index kGramDefault.
constexpr int64_t kGramMinRows[5] = {64, 128, 256, 512, 1024};
constexpr int64_t kGramMaxWg[2] = {512, 1024};
constexpr int kGramCands = kGramMfmaCands;
constexpr int kGramDefault = 3 * 2 + 0;  // 512 rows, 512 workgroups

GramPlanM plan_cand(int64_t nrows, int m, int n, int i)
{
    return plan_with(nrows, m, n, kGramMinRows[i / 2], kGramMaxWg[i % 2]);
}

TuneKey gram_key(int64_t nrows, int m, int n, bool lower_only)
{
    const int64_t tiles = gram_tiles(m, n);
    return TuneKey{kTuneGram, ilog2_floor(nrows), tiles < 64 ? (int)tiles : 64,
                   lower_only ? 1 : 0};
}


// ---------------------------------------------------------------------
// LinearComb: Y (nrows x n) = X (nrows x m) C (m x n) + Y diag(beta),
// evaluated as Y^T = C^T X^T.  A workgroup of four waves owns 128 R2 rows by
// 16 NB columns of Y, a wave 32 R2 rows of it (2 R2 x NB MFMA tiles).  Ct is
// C^T packed k-major: Ct[k * ldct + j].
//
// X is streamed from HBM into the MFMA operand registers: a lane reads two
// consecutive rows of a column at once, the even row for one MFMA tile and
// the odd one for another, so a step of 4 k takes R2 16-byte loads per lane;
// they are issued 4 steps ahead (a ring of 4).  C goes through LDS, 16 k at a
// time and double buffered, shared by the four waves (one barrier per 16 k;
// rows padded so that the operand reads cover the banks once).
//
// Bound by the matrix cores for wide blocks, by HBM for narrow ones.  Streaming
// both operands from HBM and L2 with 8-byte loads (64 x 64 tiles per wave, as
// before) kept the vector L1 busy more than half the time, and tiles of 64
// columns, like the 128-wide ones of the library's GEMM, multiply padding:
// 300 -> 141 columns at 1.03 M rows took the library 2.59 ms and the old
// kernel 1.84 at best, now 1.54 (58 TF/s); 460 -> 220 at 2 M rows 7.35 and
// 7.81, now 6.70; 200 -> 100 at 531 K rows 0.64 and 0.59, now 0.455; at 216 K
// rows 0.255 before, now 0.200; 200 -> 40 at 1.4 M rows 0.66, now 0.57.
// ---------------------------------------------------------------------
constexpr int kLcK = 16;            // k per LDS chunk
constexpr int kLcSteps = kLcK / 4;  // its steps, all of whose X loads are in flight
constexpr int kLcMaxNB = 9;         // 144 accumulator registers (with beta 8: no room to spare)
// Narrow tiles take 64 rows per wave from this many workgroups on: half the
// reads of C per row (200 -> 40 columns at 1.4 M rows: 0.61 -> 0.57 ms).
constexpr int64_t kLcTallWg = 512;
// Up to this many 16-column tiles at most kLcK source columns take a form of
// their own, in which nothing is read ahead of the one chunk of C: what the
// general form reads past m costs as much as the work there (1 -> 8 columns
// with beta per column at 4.1 M rows 167 against 142 us, 4 -> 17 with beta at
// 2 M rows 151 against 141).
constexpr int kLcOneNB = 2;

// BIG: offsets of X or C past the 32 bits of a buffer load; ONE: m <= kLcK
template <int BM, int R2, int NB, bool BIG, bool ONE>
__global__ __launch_bounds__(kWG, 2) void k_lincomb(
    int64_t nrows, int m, int n, const double *__restrict__ X, int64_t ldx,
    const double *__restrict__ Ct, int ldct, double beta_scalar,
    const double *__restrict__ beta, double *__restrict__ Y, int64_t ldy, int ntj)
{
    constexpr int kCols = 16 * NB;
    constexpr int kLd = NB % 2 == 0 ? kCols + 16 : kCols;
    __shared__ double sc[ONE ? 1 : 2][kLcK * kLd];
    const int64_t lb = xcd_swizzle(blockIdx.x, gridDim.x);
    const int j0 = (int)(lb % ntj) * kCols;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int li = lane & 15, lk = lane >> 4;
    const int64_t i0 = lb / ntj * (128 * R2) + wave * (32 * R2);
    // the lane's row pairs (pr, pr + 1), read from rs: a pair that would pass
    // the last row reads the one before instead
    int64_t rs[R2];
    bool ok0[R2], ok1[R2];
    uint32_t xo[R2];
#pragma unroll
    for (int g = 0; g < R2; ++g) {
        const int64_t pr = i0 + g * 32 + 2 * li;
        int64_t r = pr < nrows - 2 ? pr : nrows - 2;
        if (r < 0) r = 0;
        rs[g] = r;
        ok0[g] = pr < nrows && r == pr;
        ok1[g] = pr < nrows && r + 1 < nrows;
        xo[g] = (uint32_t)((r + (int64_t)lk * ldx) * 8);
    }
    d4 acc[2 * R2][NB];
#pragma unroll
    for (int g = 0; g < R2; ++g) {
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            if (BM == 0) {
                acc[2 * g][q] = acc[2 * g + 1][q] = d4{0.0, 0.0, 0.0, 0.0};
                continue;
            }
            // Y diag(beta) first, read 8 values at a time; D = 0 * 0 + init
            // moves them into the accumulator registers
            d4 e, o;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int j = j0 + q * 16 + lk + 4 * v;
                const int jc = j < n ? j : n - 1;
                const double bb = BM == 2 ? beta[jc] : beta_scalar;
                const double *y = Y + rs[g] + (int64_t)jc * ldy;
                const bool use = j < n && bb != 0.0;
                const double y0 = y[0], y1 = y[ok1[g] ? 1 : 0];
                e[v] = use ? bb * y0 : 0.0;
                o[v] = use ? bb * y1 : 0.0;
            }
            acc[2 * g][q] = mfma(0.0, 0.0, e);
            acc[2 * g + 1][q] = mfma(0.0, 0.0, o);
            asm volatile("" ::: "memory");
        }
    }
    const int nchunks = ONE ? 1 : (m + kLcK - 1) / kLcK;
    d2 ring[kLcSteps][R2];
    // the next step's columns of X: those from m on lie past the buffer's end
    // and read as zero, so no load is conditional and none is waited for early
    const double *xk = X;
    int64_t left = ((int64_t)(m - 1) * ldx + nrows) * 8;
    int64_t xl[BIG ? R2 : 1];
    if (BIG)
        for (int g = 0; g < R2; ++g) xl[g] = rs[g] + (int64_t)lk * ldx;
    int kl = lk;
    auto load_x = [&](d2 (&to)[R2]) {
        if constexpr (BIG) {
#pragma unroll
            for (int g = 0; g < R2; ++g) {
                const double *p = X + (kl < m ? xl[g] : rs[g]);
                to[g] = kl < m ? d2{p[0], p[ok1[g] ? 1 : 0]} : d2{0.0, 0.0};
                xl[g] += 4 * ldx;
            }
            kl += 4;
            return;
        }
        const auto rsrc = buffer_rsrc(
            xk, left <= 0 ? 0u : left > (int64_t)UINT32_MAX ? UINT32_MAX : (uint32_t)left);
#pragma unroll
        for (int g = 0; g < R2; ++g)
            to[g] = __builtin_bit_cast(d2, __builtin_amdgcn_raw_buffer_load_b128(rsrc, xo[g], 0, 0));
        left -= 32 * ldx;
        xk += left > 0 ? 4 * ldx : 0;
    };
    // C: rows from m on read as zero; a column past n holds what follows it
    // in memory, for results that are not stored
    const auto crsrc = buffer_rsrc(Ct, (uint32_t)(((int64_t)(m - 1) * ldct + n) * 8));
    double cst[NB];
    auto load_c = [&](int chunk) {
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const int e = threadIdx.x + kWG * u;
            const int k = chunk * kLcK + e / kCols, j = j0 + e % kCols;
            if constexpr (BIG)
                cst[u] = k < m && j < n ? Ct[(int64_t)k * ldct + j] : 0.0;
            else
                cst[u] = buffer_load<double>(crsrc, (uint32_t)((k * ldct + j) * 8));
        }
    };
    auto store_c = [&](double *to) {
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const int e = threadIdx.x + kWG * u;
            to[e / kCols * kLd + e % kCols] = cst[u];
        }
    };
    load_c(0);
#pragma unroll
    for (int b = 0; b < kLcSteps; ++b) load_x(ring[b]);
    store_c(sc[0]);
    if constexpr (!ONE) load_c(1);
    for (int c = 0; c < nchunks; ++c) {
        __syncthreads();
        if constexpr (!ONE) {
            // the other buffer was last read before this barrier
            store_c(sc[(c + 1) & 1]);
            load_c(c + 2);
        }
        const double *cb = sc[ONE ? 0 : c & 1] + lk * kLd + li;
#pragma unroll
        for (int u = 0; u < kLcSteps; ++u) {
            double ac[NB];
#pragma unroll
            for (int q = 0; q < NB; ++q) ac[q] = cb[u * 4 * kLd + q * 16];
#pragma unroll
            for (int g = 0; g < R2; ++g)
#pragma unroll
                for (int q = 0; q < NB; ++q) {
                    acc[2 * g][q] = mfma(ac[q], ring[u][g][0], acc[2 * g][q]);
                    acc[2 * g + 1][q] = mfma(ac[q], ring[u][g][1], acc[2 * g + 1][q]);
                }
            if constexpr (!ONE) load_x(ring[u]);
        }
    }
    // lane l holds (Y^T)[j0 + q*16 + l/16 + 4v][the row of its pair]
#pragma unroll
    for (int g = 0; g < R2; ++g)
#pragma unroll
        for (int q = 0; q < NB; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int j = j0 + q * 16 + lk + 4 * v;
                double *y = Y + rs[g] + (int64_t)(j < n ? j : 0) * ldy;
                if (j >= n) continue;
                if (ok0[g] && ok1[g])
                    *reinterpret_cast<d2u *>(y) = d2u{acc[2 * g][q][v], acc[2 * g + 1][q][v]};
                else if (ok0[g])
                    y[0] = acc[2 * g][q][v];
                else if (ok1[g])
                    y[1] = acc[2 * g + 1][q][v];
            }
}

// Column tiles of 16 nb columns: as few of at most 9 x 16 (8 x 16 with beta)
// as cover n, evenly wide.
struct LcTiles {
    int nb, ntj;
};

LcTiles lc_tiles(int n, int beta_mode)
{
    const int t16 = (n + 15) / 16, most = beta_mode == 0 ? kLcMaxNB : kLcMaxNB - 1;
    const int ntj = (t16 + most - 1) / most;
    return LcTiles{(t16 + ntj - 1) / ntj, ntj};
}

}  // namespace

int lincomb_cols(int n, int beta_mode)
{
    const LcTiles t = lc_tiles(n, beta_mode);
    return 16 * t.nb * t.ntj;
}

int gram_mfma_choice(int64_t nrows, int m, int n, bool lower_only, bool *tune)
{
    const int ch = tune_lookup(gram_key(nrows, m, n, lower_only));
    if (tune) *tune = ch < 0 && tune_enabled();
    return (ch < 0 || ch >= kGramCands) ? kGramDefault : ch;
}

// choice -1: at most max_chunks row chunks of at least kGramMinRows[0] rows
static GramPlanM plan_of(int64_t nrows, int m, int n, int choice, int64_t max_chunks)
{
    if (choice >= 0) return plan_cand(nrows, m, n, choice);
    return plan_with(nrows, m, n, kGramMinRows[0],
                     (max_chunks < 1 ? 1 : max_chunks) * gram_tiles(m, n));
}

int64_t gram_mfma_chunk_doubles(int m, int n)
{
    const GramShape sh = gram_shape(m, n);
    return gram_tiles(m, n) * sh.rows() * sh.cols();
}

int64_t gram_mfma_scratch(int64_t nrows, int m, int n, int choice, int64_t max_chunks)
{
    const GramPlanM p = plan_of(nrows, m, n, choice, max_chunks);
    return (int64_t)p.nchunk * p.tm * p.tn * p.tile_doubles();
}

namespace {

void launch_gram(const GramPlanM &p, int64_t nrows, int m, int n, const double *X, int64_t ldx,
                 const double *Y, int64_t ldy, double *G, int ldg, bool rowmajor, bool lower_only,
                 double *partial, hipStream_t s)
{
    if (p.sh.swap) {
        std::swap(m, n);
        std::swap(X, Y);
        std::swap(ldx, ldy);
        rowmajor = !rowmajor;
    }
    const int64_t nblk = (int64_t)p.nchunk * p.tm * p.tn;
#define GCGE_GRAM_MA(MA, NB)                                                                  \
    case MA:                                                                                  \
        k_gram_narrow<MA, NB><<<(unsigned)nblk, kWG, 0, s>>>(nrows, m, n, X, ldx, Y, ldy, p.tm, \
                                                             p.rows_per_chunk, partial);      \
        break
    if (p.sh.wide) {
        k_gram_wide<<<(unsigned)nblk, kWG, 0, s>>>(nrows, m, n, X, ldx, Y, ldy, p.tm, p.tn,
                                                   p.rows_per_chunk, lower_only ? 1 : 0, partial);
    } else if (p.sh.nb == 1) {
        switch (p.sh.ma) {
            GCGE_GRAM_MA(1, 1);
            GCGE_GRAM_MA(2, 1);
            GCGE_GRAM_MA(3, 1);
            GCGE_GRAM_MA(4, 1);
            GCGE_GRAM_MA(5, 1);
            GCGE_GRAM_MA(6, 1);
            GCGE_GRAM_MA(7, 1);
            GCGE_GRAM_MA(8, 1);
        }
    } else if (p.sh.nb == 2) {
        switch (p.sh.ma) {
            GCGE_GRAM_MA(1, 2);
            GCGE_GRAM_MA(2, 2);
            GCGE_GRAM_MA(3, 2);
            GCGE_GRAM_MA(4, 2);
            GCGE_GRAM_MA(5, 2);
            GCGE_GRAM_MA(6, 2);
            GCGE_GRAM_MA(7, 2);
            GCGE_GRAM_MA(8, 2);
        }
    } else if (p.sh.nb == 3) {
        switch (p.sh.ma) {
            GCGE_GRAM_MA(1, 3);
            GCGE_GRAM_MA(2, 3);
            GCGE_GRAM_MA(3, 3);
            GCGE_GRAM_MA(4, 3);
            GCGE_GRAM_MA(5, 3);
            GCGE_GRAM_MA(6, 3);
            GCGE_GRAM_MA(7, 3);
        }
    } else {
        switch (p.sh.ma) {
            GCGE_GRAM_MA(1, 4);
            GCGE_GRAM_MA(2, 4);
            GCGE_GRAM_MA(3, 4);
            GCGE_GRAM_MA(4, 4);
            GCGE_GRAM_MA(5, 4);
        }
    }
#undef GCGE_GRAM_MA
    sum_chunks(m, n, p.tm, p.tn, p.sh.rows(), p.sh.cols(), p.nchunk, partial, G, ldg, rowmajor, s);
}

}  // namespace

void gram_mfma(int64_t nrows, int m, int n, const double *X, int64_t ldx, const double *Y,
               int64_t ldy, double *G, int ldg, bool rowmajor, bool lower_only, int choice,
               int64_t max_chunks, bool tune, double *partial, hipStream_t s)
{
    if (m <= 0 || n <= 0) return;
    if (tune) {
        // time every chunking on a private partial buffer large enough for
        // all of them (the caller sized its buffer for the default plan)
        const TuneKey key = gram_key(nrows, m, n, lower_only);
        int64_t need = 0;
        for (int i = 0; i < kGramCands; ++i) {
            const GramPlanM q = plan_cand(nrows, m, n, i);
            const int64_t e = (int64_t)q.nchunk * q.tm * q.tn * q.tile_doubles();
            if (e > need) need = e;
        }
        double *buf = nullptr;
        HIPCHECK(hipMalloc(reinterpret_cast<void **>(&buf), sizeof(double) * (size_t)need));
        tune_run(key, kGramCands, kGramDefault,
                 [&](int i) {
                     launch_gram(plan_cand(nrows, m, n, i), nrows, m, n, X, ldx, Y, ldy, G, ldg,
                                 rowmajor, lower_only, buf, s);
                 },
                 s);
        HIPCHECK(hipStreamSynchronize(s));
        HIPCHECK(hipFree(buf));
        return;
    }
    launch_gram(plan_of(nrows, m, n, choice, max_chunks), nrows, m, n, X, ldx, Y, ldy, G, ldg,
                rowmajor, lower_only, partial, s);
}

void lincomb_mfma(int64_t nrows, int m, int n, const double *X, int64_t ldx, const double *Ct,
                  int ldct, int beta_mode, double beta_scalar, const double *beta, double *Y,
                  int64_t ldy, hipStream_t s)
{
    if (nrows <= 0 || n <= 0) return;
    const bool big = 3 * ldx + nrows >= (int64_t(1) << 29) || (int64_t)m * ldct >= (int64_t(1) << 28);
    const LcTiles t = big ? LcTiles{4, (n + 63) / 64} : lc_tiles(n, beta_mode);
    const int nb = t.nb, ntj = t.ntj;
    // 64 rows per wave for narrow tiles, while that leaves enough workgroups
    const bool tall = !big && nb <= 4 && (nrows + 255) / 256 * ntj >= kLcTallWg;
    const int64_t rows = tall ? 256 : 128;
    const unsigned g = (unsigned)((nrows + rows - 1) / rows * ntj);
#define GCGE_LC_GO(BM, R2, NB, BIG, ONE)                                                      \
    k_lincomb<BM, R2, NB, BIG, ONE><<<g, kWG, 0, s>>>(nrows, m, n, X, ldx, Ct, ldct,          \
                                                      beta_scalar, beta, Y, ldy, ntj)
#define GCGE_LC(BM, R2, NB)                                                                   \
    do {                                                                                      \
        if (NB == 4 && R2 == 1 && big)                                                        \
            GCGE_LC_GO(BM, 1, 4, true, false);                                                \
        else if (NB <= kLcOneNB && m <= kLcK)                                                 \
            GCGE_LC_GO(BM, R2, (NB <= kLcOneNB ? NB : 1), false, true);                       \
        else                                                                                  \
            GCGE_LC_GO(BM, R2, NB, false, false);                                             \
    } while (0)
#define GCGE_LC_BM(R2, NB)         \
    do {                           \
        if (beta_mode == 0)        \
            GCGE_LC(0, R2, NB);    \
        else if (beta_mode == 1)   \
            GCGE_LC(1, R2, NB);    \
        else                       \
            GCGE_LC(2, R2, NB);    \
    } while (0)
#define GCGE_LC_CASE(NB)           \
    case NB:                       \
        if (tall)                  \
            GCGE_LC_BM(2, NB);     \
        else                       \
            GCGE_LC_BM(1, NB);     \
        break
#define GCGE_LC_WIDE(NB)           \
    case NB: GCGE_LC_BM(1, NB); break
    switch (nb) {
        GCGE_LC_CASE(1);
        GCGE_LC_CASE(2);
        GCGE_LC_CASE(3);
        GCGE_LC_CASE(4);
        GCGE_LC_WIDE(5);
        GCGE_LC_WIDE(6);
        GCGE_LC_WIDE(7);
        GCGE_LC_WIDE(8);
        case 9: GCGE_LC(0, 1, 9); break;  // without beta (kLcMaxNB)
    }
#undef GCGE_LC_WIDE
#undef GCGE_LC_CASE
#undef GCGE_LC_BM
#undef GCGE_LC
#undef GCGE_LC_GO
}

}  // namespace gcge
