// Wavefront sums, and device helpers of the FP32 BlockPCG's 8-column tiles: element (row, col)
// of an interleaved block lies at ((col / 8) * n + row) * 8 + col % 8, so a
// row of a tile is one 32-byte access.  Workgroups have 256 threads.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "sell_rows.h"

namespace gcge {
namespace {

constexpr int kTileWaves = 4;
constexpr int kC = 8;      // columns per interleaved tile

struct alignas(32) f8 {
    float v[kC];
};

// A level of wave_sums and those below it: the lanes O apart keep H values
// each of the 2 H that both hold.  (A level is an instance of its own: the
// compiler does not unroll a loop over the levels of 64 values, and an array
// that is indexed at run time lies in scratch memory, in the caller's loop
// too.)
template <int H, int O, int M, typename T>
__device__ __forceinline__ void halve_sums(T (&v)[M], int &which)
{
    if constexpr (H > 0) {
        const bool up = (threadIdx.x & O) != 0;
#pragma unroll
        for (int i = 0; i < H; ++i) {
            const T keep = up ? v[i + H] : v[i], give = up ? v[i] : v[i + H];
            v[i] = keep + __shfl_xor(give, O, 64);
        }
        which += up ? H : 0;
        halve_sums<H / 2, O / 2>(v, which);
    }
}

// Sums of M values per lane over the wavefront, each over the pairs
// of lanes 32 apart, then 16, ...: the first log2(M) levels keep
// half of the values on each side, so 8 values take 10 exchanges instead of
// 48 (a BlockPCG call on 62,500 2D rows with 20 columns: 1.33 -> 1.25 ms).
// Returns the sum of value `which` (set to this lane's); lanes that
// agree in their upper log2(M) bits hold the same one.
template <int M, typename T>
__device__ __forceinline__ T wave_sums(T (&v)[M], int &which)
{
    which = 0;
    halve_sums<M / 2, 32>(v, which);
    T s = v[0];
#pragma unroll
    for (int o = 32 / M; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    return s;
}

// Sum over the workgroup of kC per-thread values; result in red[4*kC + t].
__device__ __forceinline__ void block_sum8(const float (&v)[kC], float *red)
{
    float w[kC];
#pragma unroll
    for (int t = 0; t < kC; ++t) w[t] = v[t];
    int which;
    const float s = wave_sums<kC>(w, which);
    if ((threadIdx.x & (64 / kC - 1)) == 0) red[(threadIdx.x >> 6) * kC + which] = s;
    __syncthreads();
    if (threadIdx.x < kC) {
        float t = 0.f;
#pragma unroll
        for (int k = 0; k < kTileWaves; ++k) t += red[k * kC + threadIdx.x];
        red[kTileWaves * kC + threadIdx.x] = t;
    }
    __syncthreads();
}

__device__ __forceinline__ f8 load8(const float *p)
{
    return *reinterpret_cast<const f8 *>(p);
}

__device__ __forceinline__ void store8(float *p, const f8 &x)
{
    *reinterpret_cast<f8 *>(p) = x;
}

typedef float f4v __attribute__((ext_vector_type(4)));

// load8 through a buffer resource at a byte offset (two 16-byte loads).
// The loaded vectors are bit-cast whole: a bit cast of one element of the
// integer vector reads the vector's first element for every index.
__device__ __forceinline__ f8 buffer_load8(__amdgpu_buffer_rsrc_t r, uint32_t off)
{
    const f4v a = __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
    const f4v b = __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(r, off, 16, 0));
    f8 x;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        x.v[i] = a[i];
        x.v[4 + i] = b[i];
    }
    return x;
}

}  // namespace
}  // namespace gcge
