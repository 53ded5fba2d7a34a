// Products with 27-point operators on n^3 grids (any values; point
// x + n y + n^2 z, row entries the in-grid neighbours in ascending order, as
// the variable-coefficient diffusion problems store them).
//
// The SELL row kernels gather 27 values per row and column.  A gather of 64
// 8-byte values takes the vector L1 about 20 cycles, which bounds them
// (counted at 160^3: 541 L1 accesses per wavefront and column, the L1 90 %
// busy, with 15.5 GB fetched for 2.2): 2.62 ms for 40 FP64 columns, 1.22 ms
// for an FP32 BlockPCG product over 5 tiles.  On a grid a row's neighbours
// lie in 9 lines, one per (y, z) offset, and the x - 1 and x + 1 neighbours
// are the line's values one lane over: 9 loads and lane shifts (DPP, no LDS)
// instead of 27 gathers, and no column index is read.
//
// Entries that a boundary row lacks have a zero coefficient and take a zero
// value (a load past its buffer's end gives zero, a shift past the
// wavefront's end too), so each sum is that of the SELL kernel: entries in
// ascending order, one fused multiply-add each, the same bits.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "app_hip_internal.h"
#include "kernels.h"
#include "sell_rows.h"
#include "tile8.h"

namespace gcge {
namespace {

constexpr int kWG = 256;
constexpr uint32_t kOff = 0x80000000u;  // past every buffer's end

typedef double d2v __attribute__((ext_vector_type(2)));
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

// v of the lane before (UP) or after; `end` in the first or last lane
template <bool UP>
__device__ __forceinline__ uint32_t shift32(uint32_t v, uint32_t end)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)end, (int)v, UP ? 0x138 : 0x130, 0xf, 0xf,
                                                 false);
}

template <bool UP>
__device__ __forceinline__ float shift(float v, float end)
{
    return __builtin_bit_cast(float, shift32<UP>(__builtin_bit_cast(uint32_t, v),
                                                 __builtin_bit_cast(uint32_t, end)));
}

template <bool UP>
__device__ __forceinline__ double shift(double v, double end)
{
    const uint2 a = __builtin_bit_cast(uint2, v), e = __builtin_bit_cast(uint2, end);
    return __builtin_bit_cast(double, make_uint2(shift32<UP>(a.x, e.x), shift32<UP>(a.y, e.y)));
}

// the same with 0 in the first or last lane
template <bool UP>
__device__ __forceinline__ double shift0(double v)
{
    constexpr int ctrl = UP ? 0x138 : 0x130;
    const uint2 a = __builtin_bit_cast(uint2, v);
    uint2 r;
    r.x = (uint32_t)__builtin_amdgcn_mov_dpp((int)a.x, ctrl, 0xf, 0xf, true);
    r.y = (uint32_t)__builtin_amdgcn_mov_dpp((int)a.y, ctrl, 0xf, 0xf, true);
    return __builtin_bit_cast(double, r);
}

// ---------------------------------------------------------------------
// Y = A X in FP64.  A lane holds two neighbouring points of an x-line, so a
// line's load is one 16-byte access per lane (the L1 takes a 16-byte access
// of 64 lanes in the time of an 8-byte one) and the two points share their
// shifts: 54 multiply-adds and 36 moves per wavefront and column of 128
// points.  A wavefront takes a whole line up to 128 points; longer lines are
// cut into chunks with a lane of neighbours at each end.  Each line's
// register is reloaded for the next column as soon as it has been used, so
// nine loads of a wavefront stay in flight with one set of registers (162,
// three wavefronts per SIMD; two sets at two per SIMD measured 2 % slower,
// one point per lane 15 %).  Workgroups (four y-lines) are ordered in blocks
// of 8 lines by 8 planes, so the planes that neighbouring workgroups share
// meet in an XCD's L2: 3.4 GB are fetched, against 5.8 in plane order.
// 40 columns: 160^3 2.62 -> 1.28 ms, 128^3 1.39 -> 0.61 ms, 101^3 0.66 ->
// 0.33 ms; up to 33^3 launch latency decides.
// ---------------------------------------------------------------------
constexpr int kPairWaves = 4, kPairBy = 2, kPairBz = 8;

// ODD: n odd, so that a line ends with half a pair
template <bool ODD>
__global__ __launch_bounds__(64 * kPairWaves, 3) void k_grid27_spmm(
    int n, int64_t nrows, int chunks, int xlen, int nby, const int64_t *__restrict__ slice_ptr,
    const double *__restrict__ val, const double *__restrict__ X, int64_t ldx,
    double *__restrict__ Y, int64_t ldy, int ncols)
{
    int L = (int)row_block<true>();
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = (int)(threadIdx.x & 63);
    const int xc = L % chunks;
    L /= chunks;
    int g = L % kPairBy;
    L /= kPairBy;
    int z = L % kPairBz;
    L /= kPairBz;
    g += L % nby * kPairBy;
    z += L / nby * kPairBz;
    const int y = g * kPairWaves + wv;
    if (y >= n || z >= n) return;  // wave-uniform; no barriers
    const int halo = chunks > 1 ? 1 : 0;
    const int x = xc * xlen + 2 * (lane - halo);
    const bool loads = x >= 0 && x < n && 2 * (lane - 2 * halo) < xlen;
    const bool live = loads && lane >= halo && 2 * (lane - halo) < xlen;
    const bool tail = ODD && x == n - 1;  // the second point is past the line
    const int64_t row = (int64_t)z * n * n + (int64_t)y * n + x;
    // the wavefront's rows lie in at most three slices: their entries through
    // one buffer, kOff for an entry off the grid
    double c[2][27];
    uint32_t lo[9];
    const int64_t s0 = ((int64_t)z * n * n + (int64_t)y * n + xc * xlen) >> 6;
    const int64_t s1 = s0 + 3 < (nrows + 63) / 64 ? s0 + 3 : (nrows + 63) / 64;
    const int64_t base = slice_ptr[s0];
    const auto vr = buffer_rsrc(val + base, (uint32_t)(slice_ptr[s1] - base) * 8u);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const bool on = live && x + p < n;
        const int64_t r = on ? row + p : s0 << 6;
        uint32_t at = (uint32_t)(slice_ptr[r >> 6] - base + (r & 63)) * 8u;
#pragma unroll
        for (int k = 0; k < 27; ++k) {
            const int dz = k / 9 - 1, dy = k / 3 % 3 - 1, dx = k % 3 - 1;
            const bool in = (unsigned)(y + dy) < (unsigned)n && (unsigned)(z + dz) < (unsigned)n;
            const bool ok = on && in && (unsigned)(x + p + dx) < (unsigned)n;
            c[p][k] = buffer_load<double>(vr, ok ? at : kOff);
            at += ok ? 512u : 0u;
            if (p == 0 && dx == 0)
                lo[k / 3] = in && loads
                                ? (uint32_t)(row - (tail ? 1 : 0) + dy * n + dz * n * n) * 8u
                                : kOff;
        }
    }
    const uint32_t colbytes = (uint32_t)(nrows * 8);
    auto load = [&](__amdgpu_buffer_rsrc_t rs, int l) {
        return __builtin_bit_cast(d2v, __builtin_amdgcn_raw_buffer_load_b128(rs, lo[l], 0, 0));
    };
    d2v v[9];
    const auto r0 = buffer_rsrc(X, colbytes);
#pragma unroll
    for (int l = 0; l < 9; ++l) v[l] = load(r0, l);
    for (int q = 0; q < ncols; ++q) {
        const auto rs = buffer_rsrc(X + (int64_t)(q + 1) * ldx, q + 1 < ncols ? colbytes : 0u);
        double a0 = 0.0, a1 = 0.0;
#pragma unroll
        for (int l = 0; l < 9; ++l) {
            double a = v[l][0], b = v[l][1];
            if constexpr (ODD) {
                a = tail ? b : a;
                b = tail ? 0.0 : b;
            }
            a0 = fma(c[0][3 * l], shift0<true>(b), a0);
            a0 = fma(c[0][3 * l + 1], a, a0);
            a0 = fma(c[0][3 * l + 2], b, a0);
            a1 = fma(c[1][3 * l], a, a1);
            a1 = fma(c[1][3 * l + 1], b, a1);
            a1 = fma(c[1][3 * l + 2], shift0<false>(a), a1);
            // (keeps the line's terms here rather than sunk into the store's
            // branch, where they would hold the line past its reload)
            asm volatile("" : "+v"(a0), "+v"(a1));
            __builtin_amdgcn_sched_barrier(0);
            v[l] = load(rs, l);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (live) {
            double *yp = Y + row + (int64_t)q * ldy;
            if (tail)
                *yp = a0;
            else
                *reinterpret_cast<d2u *>(yp) = d2u{a0, a1};
        }
    }
}

// ---------------------------------------------------------------------
// The BlockPCG's forms keep the rows of the SELL kernels, 64 consecutive
// rows per wavefront and 256 per workgroup, because their partial sums
// follow them.  A wavefront's rows may span two x-lines or more: a run of 64
// rows stands for the line, the first and last lane load their outer
// neighbour, and wavefronts with an x boundary among their rows mask the
// values shifted across it.
// ---------------------------------------------------------------------
template <typename V>
struct Row27 {
    V c[27];
    uint32_t line[9];  // byte offset of the row's value in each run (kOff: off the grid)
    uint32_t step;     // from line[l] to the outer neighbour (kOff but in the end lanes)
    bool first, last;  // x == 0, x == n - 1
    bool cut;          // some row of the wavefront is at an x boundary (uniform)
    bool live;
    int64_t row;

    // size: bytes per row of the vectors
    __device__ __forceinline__ void init(int64_t rb, int n, int64_t nrows,
                                         const int64_t *__restrict__ slice_ptr,
                                         const V *__restrict__ val, uint32_t size)
    {
        constexpr uint32_t kAway = 0x40000000u;  // past the end from any line, kOff included
        const int64_t s = wave_slice<kWG>(rb);
        const int lane = (int)(threadIdx.x & 63);
        row = s * 64 + lane;
        live = row < nrows;
        const uint32_t r = (uint32_t)row, un = (uint32_t)n;
        const uint32_t x = r % un, y = r / un % un, z = r / un / un;
        first = x == 0;
        last = x == un - 1;
        cut = __any(live && (first || last));
        step = lane == 0 ? (first ? kAway : 0u - size) : (lane < 63 || last) ? kAway : size;
        uint32_t bytes = 0;
        int64_t base = 0;
        if (s * 64 < nrows) {  // wave-uniform
            base = slice_ptr[s];
            bytes = (uint32_t)(slice_ptr[s + 1] - base) * (uint32_t)sizeof(V);
        }
        const auto rs = buffer_rsrc(val + base, (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes));
        uint32_t at = (uint32_t)lane * (uint32_t)sizeof(V);
#pragma unroll
        for (int l = 0; l < 9; ++l) {
            const int dz = l / 3 - 1, dy = l % 3 - 1;
            const bool in = live && y + (uint32_t)dy < un && z + (uint32_t)dz < un;
            line[l] = in ? (r + (uint32_t)(dy * n) + (uint32_t)(dz * n * n)) * size : kOff;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const bool on = in && (k != 0 || !first) && (k != 2 || !last);
                c[3 * l + k] = buffer_load<V>(rs, on ? at : kOff);
                at += on ? 64u * (uint32_t)sizeof(V) : 0u;
            }
        }
    }

    // the three terms of run l: its value v, the outer neighbour e (read in
    // the end lanes)
    template <bool CUT>
    __device__ __forceinline__ V terms(int l, V v, V e, V acc) const
    {
        V a = shift<true>(v, e), b = shift<false>(v, e);
        if constexpr (CUT) {
            a = first ? V(0) : a;
            b = last ? V(0) : b;
        }
        acc = fma(c[3 * l], a, acc);
        acc = fma(c[3 * l + 1], v, acc);
        return fma(c[3 * l + 2], b, acc);
    }
};

// Calls f with cut as a compile-time value.  (The marks keep loads that both
// forms share from being hoisted above the branch, all at once.)
template <typename F>
__device__ __forceinline__ void for_cut(bool cut, F &&f)
{
    if (cut) {
        asm volatile("; rows at an x boundary" ::: "memory");
        f(std::integral_constant<bool, true>{});
    } else {
        asm volatile("; interior rows" ::: "memory");
        f(std::integral_constant<bool, false>{});
    }
}

// w = A p over the listed 8-column tiles with the partial p.w sums, the rows
// and sums of k_spmm_pw (pcg32.hip).  The coefficients are read once and stay
// in registers over the tiles.  Bound by its vector instructions (216
// multiply-adds and 144 shifts per wavefront and tile, 810 with the moves,
// masks and sums, which occupy the SIMDs 66 % of the time at 160^3) and by
// HBM (3.0 GB there, 4.5 TB/s: p is read 2.9 times).  160^3, 5 tiles: 1.22
// -> 0.66 ms; a whole BlockPCG call at 50^3 with 33 columns 3.22 -> 2.15 ms.
// One run ahead (a ring of 2) with four wavefronts per SIMD, and
// plane-blocked workgroup orders, measured 1-2 % slower; loading the outer
// neighbours under a lane mask 1 % slower.
__global__ __launch_bounds__(kWG, 3) void k_grid27_pw(int n, int64_t nrows,
                                                      const int64_t *__restrict__ slice_ptr,
                                                      const float *__restrict__ val,
                                                      const int *__restrict__ tiles,
                                                      const int *__restrict__ ntact_p,
                                                      const float *__restrict__ P,
                                                      float *__restrict__ Wv,
                                                      float *__restrict__ partial)
{
    constexpr int kRing = 3;  // run l is used while runs l + 1 and l + 2 are in flight
    __shared__ float wsum[2][kTileWaves][kC];
    const int64_t rb = row_block<true>(), nblk = gridDim.x;
    const int ntact = *ntact_p;
    Row27<float> g;
    g.init(rb, n, nrows, slice_ptr, val, (uint32_t)(kC * sizeof(float)));
    const uint32_t tbytes = (uint32_t)(nrows * kC * (int64_t)sizeof(float));
    for (int k = 0; k < ntact; ++k) {
        const int tile = tiles[k];
        const int64_t o = (int64_t)tile * nrows * kC;
        const auto rs = buffer_rsrc(P + o, tbytes);
        f8 acc, own;
        float dot[kC];
#pragma unroll
        for (int t = 0; t < kC; ++t) acc.v[t] = dot[t] = 0.f;
        for_cut(g.cut, [&](auto cut) {
            constexpr bool CUT = decltype(cut)::value;
            f8 v[kRing], e[kRing];
            auto fetch = [&](int l) {
                v[l % kRing] = buffer_load8(rs, g.line[l]);
                e[l % kRing] = buffer_load8(rs, g.line[l] + g.step);
            };
#pragma unroll
            for (int l = 0; l < kRing - 1; ++l) fetch(l);
#pragma unroll
            for (int l = 0; l < 9; ++l) {
                if (l + kRing - 1 < 9) fetch(l + kRing - 1);
                __builtin_amdgcn_sched_barrier(0);
                if (l == 4) own = v[l % kRing];
#pragma unroll
                for (int t = 0; t < kC; ++t)
                    acc.v[t] = g.terms<CUT>(l, v[l % kRing].v[t], e[l % kRing].v[t], acc.v[t]);
                // (keeps the run's terms here)
#pragma unroll
                for (int t = 0; t < kC; ++t) asm volatile("" : "+v"(acc.v[t]));
                __builtin_amdgcn_sched_barrier(0);
            }
        });
        if (g.live) {
            store8(Wv + o + g.row * kC, acc);
#pragma unroll
            for (int t = 0; t < kC; ++t) dot[t] = acc.v[t] * own.v[t];
        }
        // one barrier per tile: the sums alternate between two arrays
        int which;
        const float s = wave_sums<kC>(dot, which);
        if ((threadIdx.x & (64 / kC - 1)) == 0) wsum[k & 1][threadIdx.x >> 6][which] = s;
        __syncthreads();
        if (threadIdx.x < kC) {
            float t = 0.f;
#pragma unroll
            for (int w = 0; w < kTileWaves; ++w) t += wsum[k & 1][w][threadIdx.x];
            partial[(int64_t)(tile * kC + threadIdx.x) * nblk + rb] = t;
        }
    }
}

// R = fl32(b - A x) in tiles with the partial R.R sums, the rows and sums of
// k_resid64 (pcg32.hip), which takes 7.1 ms for 40 columns at 160^3 (its 8
// columns' gathers of a tile were unrolled together into 256 registers and
// more); here 2.25 ms.
__global__ __launch_bounds__(kWG, 3) void k_grid27_resid(int n, int64_t nrows,
                                                         const int64_t *__restrict__ slice_ptr,
                                                         const double *__restrict__ val, int nc,
                                                         const double *__restrict__ Bv,
                                                         int64_t ldb,
                                                         const double *__restrict__ Xv,
                                                         int64_t ldx, float *__restrict__ R,
                                                         float *__restrict__ partial)
{
    __shared__ float red[(kTileWaves + 1) * kC];
    const int64_t rb = row_block<true>(), nblk = gridDim.x;
    Row27<double> g;
    g.init(rb, n, nrows, slice_ptr, val, 8u);
    const uint32_t colbytes = (uint32_t)(nrows * 8);
    const int ntile = (nc + kC - 1) / kC;
    for (int tile = 0; tile < ntile; ++tile) {
        float sq[kC];
        f8 r8;
        for_cut(g.cut, [&](auto cut) {
            constexpr bool CUT = decltype(cut)::value;
#pragma unroll
            for (int t = 0; t < kC; ++t) {
                const int c = tile * kC + t;
                r8.v[t] = sq[t] = 0.f;
                __builtin_amdgcn_sched_barrier(0);
                if (c < nc) {  // uniform
                    const auto rs = buffer_rsrc(Xv + (int64_t)c * ldx, colbytes);
                    double v[9], e[9], acc = 0.0;
#pragma unroll
                    for (int l = 0; l < 9; ++l) {
                        v[l] = buffer_load<double>(rs, g.line[l]);
                        e[l] = buffer_load<double>(rs, g.line[l] + g.step);
                    }
#pragma unroll
                    for (int l = 0; l < 9; ++l) acc = g.terms<CUT>(l, v[l], e[l], acc);
                    if (g.live) {
                        const float r = (float)(Bv[g.row + (int64_t)c * ldb] - acc);
                        r8.v[t] = r;
                        sq[t] = r * r;
                    }
                    asm volatile("" : "+v"(r8.v[t]));
                }
            }
        });
        if (g.live) store8(R + ((int64_t)tile * nrows + g.row) * kC, r8);
        block_sum8(sq, red);
        if (threadIdx.x < kC)
            partial[(int64_t)(tile * kC + threadIdx.x) * nblk + rb] =
                red[kTileWaves * kC + threadIdx.x];
        __syncthreads();
    }
}

// flag[0] = 1 when some row's entries are not those of the 27-point grid
// pattern (padding entries hold value 0 and the row's own index)
__global__ __launch_bounds__(kWG) void k_grid27_check(int n, int64_t nrows,
                                                      const int64_t *__restrict__ slice_ptr,
                                                      const int *__restrict__ col,
                                                      const double *__restrict__ val,
                                                      int *__restrict__ flag)
{
    const int64_t row = (int64_t)blockIdx.x * kWG + threadIdx.x;
    if (row >= nrows) return;
    const int64_t s = row >> 6, base = slice_ptr[s];
    const int w = (int)((slice_ptr[s + 1] - base) >> 6);
    const int64_t e0 = base + (row & 63);
    const int x = (int)(row % n), y = (int)(row / n % n), z = (int)(row / n / n);
    int j = 0;
    bool ok = true;
    for (int k = 0; k < 27; ++k) {
        const int dz = k / 9 - 1, dy = k / 3 % 3 - 1, dx = k % 3 - 1;
        if (x + dx < 0 || x + dx >= n || y + dy < 0 || y + dy >= n || z + dz < 0 || z + dz >= n)
            continue;
        const int64_t want = row + dx + (int64_t)n * (dy + (int64_t)n * dz);
        ok = ok && j < w && col[e0 + (int64_t)64 * j] == want;
        ++j;
    }
    for (; j < w; ++j)
        ok = ok && col[e0 + (int64_t)64 * j] == row && val[e0 + (int64_t)64 * j] == 0.0;
    if (!ok) *flag = 1;  // every writer stores 1
}

}  // namespace

void detect_grid27(SellMat &A, hipStream_t s)
{
    A.grid27_n = 0;
    if (A.max_width != 27) return;
    int n = 4;
    while (n < kGrid27MaxN && (int64_t)n * n * n < A.nrows) ++n;
    const int64_t m = 3 * (int64_t)n - 2;
    if ((int64_t)n * n * n != A.nrows || m * m * m != A.nnz_true) return;
    int *d = nullptr, h = 0;
    dev_alloc(&d, sizeof(int));
    HIPCHECK(hipMemsetAsync(d, 0, sizeof(int), s));
    k_grid27_check<<<(unsigned)((A.nrows + kWG - 1) / kWG), kWG, 0, s>>>(n, A.nrows, A.slice_ptr,
                                                                         A.col, A.val, d);
    HIPCHECK(hipMemcpyAsync(&h, d, sizeof(int), hipMemcpyDeviceToHost, s));
    HIPCHECK(hipStreamSynchronize(s));
    dev_free(d);
    if (h == 0) A.grid27_n = n;
}

bool spmm_grid27(const SellMat &A, const double *X, int64_t ldx, double *Y, int64_t ldy,
                 int ncols, hipStream_t s)
{
    if (A.grid27_n == 0 || ncols <= 0) return false;
    const int n = A.grid27_n;
    // From side 33 on the workgroups are more than the CUs; up to 38 the
    // general kernel's rows still take few columns faster (one column at 33^3:
    // 5.6 against 6.5-7.1 us, 4 at 36^3 9.2 against 8.9-9.6; at 32^3 5.6
    // against 5.0, at 40^3 6.9 against 6.1-7.2).
    if (n > 32 && n < 39 && ncols <= 3) return false;
    const int chunks = n <= 128 ? 1 : (n + 123) / 124;
    const int xlen = 2 * ((n + 2 * chunks - 1) / (2 * chunks));
    const int nby = (n + kPairWaves * kPairBy - 1) / (kPairWaves * kPairBy);
    const int nbz = (n + kPairBz - 1) / kPairBz;
    const unsigned g = (unsigned)(chunks * kPairBy * kPairBz * nby * nbz);
    if (n % 2 != 0)
        k_grid27_spmm<true><<<g, 64 * kPairWaves, 0, s>>>(
            n, A.nrows, chunks, xlen, nby, A.slice_ptr, A.val, X, ldx, Y, ldy, ncols);
    else
        k_grid27_spmm<false><<<g, 64 * kPairWaves, 0, s>>>(
            n, A.nrows, chunks, xlen, nby, A.slice_ptr, A.val, X, ldx, Y, ldy, ncols);
    return true;
}

bool grid27_pw(const SellMat &A, const int *tiles, const int *ntact_p, const float *P, float *W,
               float *partial, hipStream_t s)
{
    if (A.grid27_n == 0) return false;
    const unsigned g = (unsigned)((A.nrows + kWG - 1) / kWG);
    k_grid27_pw<<<g, kWG, 0, s>>>(A.grid27_n, A.nrows, A.slice_ptr, A.val32, tiles, ntact_p, P, W,
                                  partial);
    return true;
}

bool grid27_resid(const SellMat &A, int nc, const double *B, int64_t ldb, const double *X,
                  int64_t ldx, float *R, float *partial, hipStream_t s)
{
    if (A.grid27_n == 0) return false;
    const unsigned g = (unsigned)((A.nrows + kWG - 1) / kWG);
    k_grid27_resid<<<g, kWG, 0, s>>>(A.grid27_n, A.nrows, A.slice_ptr, A.val, nc, B, ldb, X, ldx,
                                     R, partial);
    return true;
}

}  // namespace gcge
