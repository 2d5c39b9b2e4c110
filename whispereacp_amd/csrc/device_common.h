// Device helpers shared by the gfx950 kernels: weight widening, wave64
// reductions and the exact GELU. CDNA4 only: waves are 64 lanes wide.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace wsp
{
constexpr int kWave = 64;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float4u __attribute__((ext_vector_type(4), aligned(4))); // the same at any float

enum WeightType : int
{
    kF32 = 0,
    kF16 = 1,
    kBF16 = 2
};

// Global-memory views of pointers the compiler cannot place itself (pointers
// read from LDS or from memory). Accesses through them are global_load /
// global_store, which count only in vmcnt; the same access through a generic
// pointer is a flat access, which also counts in lgkmcnt, so every later LDS
// wait would also wait for it.
template <class T>
using global_ptr = __attribute__((address_space(1))) T*;

template <class T>
__device__ __forceinline__ const __attribute__((address_space(1))) T* global(const T* p)
{
    return (const __attribute__((address_space(1))) T*) p;
}

template <class T>
__device__ __forceinline__ __attribute__((address_space(1))) T* global_mut(T* p)
{
    return (__attribute__((address_space(1))) T*) p;
}

// Sums within a 16-lane DPP row in a fixed order: swap neighbours, swap
// pairs, mirror within 8 and mirror within 16 leave the row total in every
// lane, each step one v_add_f32_dpp. Every pair is added in an
// order-independent way (a + b == b + a), so every lane of the row holds the
// same bits. Every lane of the row must be active.
// (bound_ctrl set: every pattern used reads a lane of the same row, so no lane
// reads out of range, and the move folds into the consuming add as one
// v_add_f32_dpp.)
template <int CTRL>
__device__ __forceinline__ float dpp(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}

constexpr int kSwapNeighbours = 0xB1; // quad_perm [1,0,3,2]
constexpr int kSwapPairs = 0x4E;      // quad_perm [2,3,0,1]
constexpr int kMirrorHalfRow = 0x141; // row_half_mirror
constexpr int kMirrorRow = 0x140;     // row_mirror

__device__ __forceinline__ float sum16(float v)
{
    v += dpp<kSwapNeighbours>(v);
    v += dpp<kSwapPairs>(v);
    v += dpp<kMirrorHalfRow>(v);
    v += dpp<kMirrorRow>(v);
    return v;
}

// 16 bytes from global memory.
__device__ __forceinline__ uint4 load_global16(const void* p)
{
    const u32x4 v = *global(static_cast<const u32x4*>(p));
    return make_uint4(v[0], v[1], v[2], v[3]);
}

__device__ __forceinline__ float bf16_to_float(uint16_t bits)
{
    return __uint_as_float((uint32_t) bits << 16);
}

// Eight consecutive weights widened to float from one 16-byte load (F16,
// BF16) or two (F32). `index` is an element index, a multiple of 8.
template <int WT>
__device__ __forceinline__ void load8(const void* base, size_t index, float (&w)[8])
{
    if constexpr (WT == kF32)
    {
        const float4v* p = reinterpret_cast<const float4v*>(static_cast<const float*>(base) + index);
        const float4v a = p[0], b = p[1];
        w[0] = a[0]; w[1] = a[1]; w[2] = a[2]; w[3] = a[3];
        w[4] = b[0]; w[5] = b[1]; w[6] = b[2]; w[7] = b[3];
    }
    else if constexpr (WT == kF16)
    {
        const half8 h = *reinterpret_cast<const half8*>(static_cast<const _Float16*>(base) + index);
#pragma unroll
        for (int i = 0; i < 8; ++i)
            w[i] = (float) h[i];
    }
    else
    {
        const uint4 u = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(base) + index);
        const uint32_t v[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            w[2 * i] = __uint_as_float(v[i] << 16);
            w[2 * i + 1] = __uint_as_float(v[i] & 0xFFFF0000u);
        }
    }
}

template <int WT>
__device__ __forceinline__ float load1(const void* base, size_t index)
{
    if constexpr (WT == kF32)
        return static_cast<const float*>(base)[index];
    else if constexpr (WT == kF16)
        return (float) static_cast<const _Float16*>(base)[index];
    else
        return bf16_to_float(static_cast<const uint16_t*>(base)[index]);
}

__device__ __forceinline__ float wave_sum(float v)
{
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1)
        v += __shfl_xor(v, offset, kWave);
    return v;
}

__device__ __forceinline__ float wave_max(float v)
{
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1)
        v = fmaxf(v, __shfl_xor(v, offset, kWave));
    return v;
}

// Block-wide sum for blockDim.x a multiple of 64 (at most 1024). `scratch`
// holds one float per wave. Every thread returns the total.
__device__ __forceinline__ float block_sum(float v, float* scratch)
{
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int waves = blockDim.x / kWave;
    v = wave_sum(v);
    __syncthreads();
    if (lane == 0)
        scratch[wave] = v;
    __syncthreads();
    float total = 0.f;
    for (int i = 0; i < waves; ++i)
        total += scratch[i];
    return total;
}

__device__ __forceinline__ float block_max(float v, float* scratch)
{
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int waves = blockDim.x / kWave;
    v = wave_max(v);
    __syncthreads();
    if (lane == 0)
        scratch[wave] = v;
    __syncthreads();
    float best = scratch[0];
    for (int i = 1; i < waves; ++i)
        best = fmaxf(best, scratch[i]);
    return best;
}

// The sum over a wave, in every lane (all 64 active), by cross-lane operations
// of the vector units alone: no LDS round trips.
__device__ __forceinline__ float lanes_sum(float v)
{
    v = sum16(v);
    const uint32_t row = __builtin_bit_cast(uint32_t, v);
    const auto rows = __builtin_amdgcn_permlane16_swap(row, row, false, false);
    v = __builtin_bit_cast(float, (uint32_t) rows[0]) + __builtin_bit_cast(float, (uint32_t) rows[1]);
    const uint32_t half = __builtin_bit_cast(uint32_t, v);
    const auto halves = __builtin_amdgcn_permlane32_swap(half, half, false, false);
    return __builtin_bit_cast(float, (uint32_t) halves[0]) + __builtin_bit_cast(float, (uint32_t) halves[1]);
}

// One wave's LayerNorm of a row of `width` floats (a multiple of 4, at most
// 256·RUNS; rows at 16 bytes, the terms at any float): the mean, the centred squares' mean, then
// (x - mean)·rstd·gamma + beta (Kernels/LayerNorm.h:44-89). Lane l holds runs
// l, l + 64, ... of four in v. The row, gamma and beta are all in flight at
// once, and nothing waits for another wave: a launch is bound by its memory
// round trips and barriers, of which a block for each row had three and four
// (96 x 768: 4.6 us a launch so, 3.5 now; 1500 x 1280 written as parts, a wave
// for each row with the terms read behind the sums 7.5, 6.4 now).
template <int RUNS>
__device__ __forceinline__ void normalise_row(const float* __restrict__ src, const float* __restrict__ gamma,
                                              const float* __restrict__ beta, int width, float eps,
                                              float4v (&v)[RUNS])
{
    const int lane = threadIdx.x % kWave, runs = width / 4;
    float4v scales[RUNS], shifts[RUNS];
#pragma unroll
    for (int i = 0; i < RUNS; ++i)
    {
        const int r = min(lane + kWave * i, runs - 1);
        v[i] = reinterpret_cast<const float4v*>(src)[r];
        scales[i] = *reinterpret_cast<const float4u*>(gamma + 4 * r);
        shifts[i] = *reinterpret_cast<const float4u*>(beta + 4 * r);
    }
    float total = 0.f;
#pragma unroll
    for (int i = 0; i < RUNS; ++i)
        if (lane + kWave * i < runs)
            total += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
    const float mean = lanes_sum(total) / (float) width;
    float squares = 0.f;
#pragma unroll
    for (int i = 0; i < RUNS; ++i)
    {
        v[i] -= mean;
        if (lane + kWave * i < runs)
            squares += (v[i][0] * v[i][0] + v[i][1] * v[i][1]) + (v[i][2] * v[i][2] + v[i][3] * v[i][3]);
    }
    const float rstd = rsqrtf(lanes_sum(squares) / (float) width + eps);
#pragma unroll
    for (int i = 0; i < RUNS; ++i)
        v[i] = v[i] * rstd * scales[i] + shifts[i];
}

// x as 16-bit parts for products with 16-bit weights of type WT; part p in the
// low 16 bits of bits[p]. kBF16: three bf16 parts whose sum is x. kF16: fp16 hi
// + lo, for |x| < 65504, whose sum is within 2^-22 of x's magnitude or 2^-25
// (half the last place of fp16's least numbers), whichever is larger; past that
// hi is infinite and lo NaN.
template <int WT>
__device__ __forceinline__ void cut_parts(float x, uint32_t (&bits)[3])
{
    if constexpr (WT == kF16)
    {
        const _Float16 hi = (_Float16) x;
        const _Float16 lo = (_Float16) (x - (float) hi);
        bits[0] = __builtin_bit_cast(uint16_t, hi);
        bits[1] = __builtin_bit_cast(uint16_t, lo);
        bits[2] = 0;
    }
    else
    {
        float rest = x;
#pragma unroll
        for (int p = 0; p < 3; ++p)
        {
            const __bf16 b = (__bf16) rest;
            bits[p] = __builtin_bit_cast(uint16_t, b);
            rest -= (float) b;
        }
    }
}

// How many parts those are (an fp32 weight's rows are read as they are).
template <int WT>
constexpr int parts_of()
{
    return WT == kF32 ? 1 : WT == kF16 ? 2 : 3;
}

// c + a·b over 32 k of 16-bit values of type WT, a 16 x 16 tile.
template <int WT>
__device__ __forceinline__ float4v mfma16(u32x4 a, u32x4 b, float4v c)
{
    if constexpr (WT == kF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0,
                                                       0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                        0, 0, 0);
}

// The 16-byte slot of chunk c of LDS row r, rows of eight chunks (128 bytes): one
// chunk of eight consecutive rows lies in eight different bank groups.
__device__ __forceinline__ int chunk_slot(int r, int c)
{
    return 8 * r + (c ^ (r & 7));
}

// The LDS byte address of a shared-memory pointer.
__device__ __forceinline__ uint32_t lds_address(const void* p)
{
    return (uint32_t) (uintptr_t) (__attribute__((address_space(3))) char*) (p);
}

// One direct-to-LDS load: this lane's 16 bytes at base + offset land at LDS
// address lds + 16·lane (lds uniform over the wave).
__device__ __forceinline__ void load_lds16(const void* base, uint32_t offset, uint32_t lds)
{
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(offset), "s"(base)
                 : "memory");
}

template <int N>
__device__ __forceinline__ void wait_loads()
{
    static_assert(N >= 0 && N < 64, "vmcnt holds 0..63");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Where the encoder attention's transposed values keep key `row`: inside each
// 32 keys the eight that a lane group g of the score product's output holds
// (4g .. 4g + 3 and 16 + 4g .. 16 + 4g + 3) lie together, so they are one
// 16-byte operand read.
__host__ __device__ constexpr int attention_place(int row)
{
    return (row & ~31) | ((row >> 2 & 3) << 3) | ((row >> 4 & 1) << 2) | (row & 3);
}

// x * 0.5 * (1 + erf(x / sqrt(2))), the exact form (Kernels/Gelu.h:16-21),
// with the device library's erff.
__device__ __forceinline__ float exact_gelu(float x)
{
    return 0.5f * x * (1.f + erff(x * 0.70710678118654752f));
}
} // namespace wsp
