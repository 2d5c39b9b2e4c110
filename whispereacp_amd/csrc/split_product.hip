// Products of many rows on gfx950 matrix cores: y = X·Wᵀ for fp32 X and a 16-bit
// W with X in pre-split parts, or an fp32 W in fp32 arithmetic
// (Encoder/Encoder.cpp:82-174: the q/k/v, attention-output, fc1 and fc2
// products of every layer and the convolutions; the cross keys and values of
// every layer, and long prompts, through linear_product.hip).
//
// For 16-bit W, X is stored once in 16-bit parts (cut_parts: three bf16 parts for
// bf16 weights, together exact; fp16 hi + lo for fp16 weights, within 2^-22 of
// |x| < 65504 or 2^-25), part-major: part p of row r at parts + p·part_stride +
// r·inner. Every matrix-core product of a part with W is exact, and the fp32
// sums match an fp32 product with widened weights to fp32 rounding (fp16: to the
// parts'). The parts are written by split_rows (from fp32 rows) or by a
// product's own epilogue (fc1 writes its GELU output as parts for fc2), so
// the products' inner loops carry no conversion work.
//
// A block computes a TM x TN tile in 64-wide k-steps: every staged row segment
// is then one whole 128-byte line (with 32-wide steps each request fetched half
// a line, and the requests bound the products: 14-16 bytes a clock and CU).
// Both operands go straight from memory into LDS with direct-to-LDS loads (each
// lane's 16 bytes land at the wave's slot + 16·lane), into one of S stage
// buffers, so a step's loads are issued S - 1 steps before its products and
// hold no registers meanwhile. A 16-byte chunk c (8 k values) of tile row r
// sits at slot 8r + (c ^ (r & 7)): a 16-byte operand read serves eight lanes
// (128 bytes, the 32 banks) at a time, and the matrix-core operand reads (rows
// li of a 16-row tile, one chunk for each g, for lanes (li, g)) then give each
// eight lanes eight different bank groups. The loads are issued from inline
// assembly with explicit waits: the compiler's own wait insertion would drain
// every load in flight before each LDS read.
//
// W is the matrix cores' row operand and X their column operand, so a lane ends
// up with four consecutive outputs of one row and stores them together (16
// bytes of fp32, 8 of each 16-bit part).
//
// Tiles measured at 1500 rows, two parts (us a launch, the same products in
// 128 x 128 tiles of 32-wide steps on two stages or 128 x 64 on four before):
//   1280 -> 5120  128 x 256: 38 (46)     5120 -> 1280  64 x 128: 45 (65)
//   1280 -> 3840  128 x 256: 33 (38)     1280 -> 1280  64 x 128: 15 (19)
//    384 -> 1152  64 x 128: 6.5 (7.9)    1536 -> 384   32 x 128: 9.8 (20)
// and at 300 rows 5120 -> 1280 in 32 x 64 tiles 18.5 (57).
#include "device_common.h"
#include "once_per_device.h"
#include "ops.h"

#include <algorithm>

namespace wsp::ops
{
namespace
{
typedef uint16_t u16;

constexpr int kRowBytes = 128;              // of a tile row per step: 64 16-bit values or 32 fp32
constexpr int kChunks = kRowBytes / 16;
constexpr int kLoadRows = 1024 / kRowBytes; // tile rows one wave load (1 KB) covers
constexpr int kSplitThreads = 256;

template <int WT>
constexpr int value_bytes()
{
    return WT == kF32 ? 4 : 2;
}

// One 16-byte chunk of each operand: 32 k of 16-bit values, or 16 k of fp32 in
// four products (a lane's element e of chunk c stands for k = 4c + e in both).
// One sum in the order of k: even and odd elements summed apart would be a
// shorter chain, but where X is a signal and W its spectrum's basis each half
// is an aliased spectrum and the two cancel (the log-mel's error against 64
// bits grew from 1.2e-7 to 2.8e-7).
template <int WT>
__device__ __forceinline__ float4v multiply(u32x4 a, u32x4 b, float4v c)
{
    if constexpr (WT == kF32)
    {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[e]), __uint_as_float(b[e]), c, 0, 0, 0);
        return c;
    }
    else
        return mfma16<WT>(a, b, c);
}

// Eight consecutive values of a row as parts: part p's eight 16-bit values in
// out[p] (the first value in the low half of the first word).
template <int WT>
__device__ __forceinline__ void split8(const float (&v)[8], u32x4 (&out)[3])
{
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        uint32_t b0[3], b1[3];
        cut_parts<WT>(v[2 * j], b0);
        cut_parts<WT>(v[2 * j + 1], b1);
#pragma unroll
        for (int p = 0; p < 3; ++p)
            out[p][j] = b0[p] | (b1[p] << 16);
    }
}

// fp32 rows [rows][width] -> parts; one thread converts eight values.
template <int WT>
__global__ void __launch_bounds__(kSplitThreads) split_rows_kernel(const float* __restrict__ x, size_t count,
                                                                   u16* __restrict__ parts, size_t part_stride)
{
    constexpr int P = parts_of<WT>();
    const size_t i = ((size_t) blockIdx.x * kSplitThreads + threadIdx.x) * 8;
    if (i >= count)
        return;
    const float4v a = *reinterpret_cast<const float4v*>(x + i);
    const float4v b = *reinterpret_cast<const float4v*>(x + i + 4);
    const float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    u32x4 out[3];
    split8<WT>(v, out);
#pragma unroll
    for (int p = 0; p < P; ++p)
        *reinterpret_cast<u32x4*>(parts + p * part_stride + i) = out[p];
}

// normalise_row written as the parts of split_product's input, each part's four
// values of a run as one 8-byte store.
constexpr int kNormWidth = 2048; // the widest

template <int WT, int RUNS>
__global__ void __launch_bounds__(kWave) layernorm_parts_kernel(const float* __restrict__ x,
                                                                const float* __restrict__ gamma,
                                                                const float* __restrict__ beta, int width, float eps,
                                                                u16* __restrict__ parts, size_t part_stride)
{
    constexpr int P = parts_of<WT>();
    const size_t row = (size_t) blockIdx.x * width;
    float4v v[RUNS];
    normalise_row<RUNS>(x + row, gamma, beta, width, eps, v);
#pragma unroll
    for (int i = 0; i < RUNS; ++i)
    {
        const int at = 4 * ((int) threadIdx.x + kWave * i);
        if (at >= width)
            continue;
        uint32_t bits[4][3];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            cut_parts<WT>(v[i][e], bits[e]);
#pragma unroll
        for (int p = 0; p < P; ++p)
            *reinterpret_cast<uint2*>(parts + p * part_stride + row + at)
                = uint2 {bits[0][p] | (bits[1][p] << 16), bits[2][p] | (bits[3][p] << 16)};
    }
}

// WM x WN waves, each TM / WM rows by TN / WN columns; S stage buffers.
template <int WT, int TM_, int TN_, int WM_, int WN_, int S_>
struct Tile
{
    static constexpr int P = parts_of<WT>();
    static constexpr int TM = TM_, TN = TN_, WM = WM_, WN = WN_, S = S_;
    static constexpr int kWaves = WM * WN;
    static constexpr int kABytes = TM * kRowBytes; // one part's rows
    static constexpr int kStageBytes = P * kABytes + TN * kRowBytes;
    static constexpr int kLoads = (P * TM + TN) / kLoadRows;
    static_assert(kLoads % kWaves == 0, "whole loads per wave");
    static constexpr int kPerWave = kLoads / kWaves;
    static constexpr int MT = TM / 16 / WM, NT = TN / 16 / WN;
    static_assert(S * kStageBytes <= 160 * 1024, "the stages fit the LDS");
};

template <class T, int WT>
__global__ void __launch_bounds__(T::kWaves * kWave) split_product_kernel(SplitProduct a)
{
    constexpr int P = T::P, MT = T::MT, NT = T::NT, B = value_bytes<WT>();
    constexpr int kStep = kRowBytes / B; // k per step
    extern __shared__ __attribute__((aligned(16))) unsigned char stage_mem[];

    const int tid = threadIdx.x, lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave); // uniform, so the load bases are scalar
    const int li = lane % 16, g = lane / 16;
    const int wm = wave / T::WN, wn = wave % T::WN;
    const int n_block = blockIdx.x * T::TN, m_block = blockIdx.y * T::TM;
    const int steps = (a.inner + kStep - 1) / kStep;
    // The block's columns lie in one of the matrices.
    const int width = a.columns, seg = a.count > 1 ? n_block / width : 0, seg_first = seg * width;
    const ProductMatrix& matrix = a.matrix[seg];
    const void* w = matrix.w;

    // This wave's loads: load q = wave + waves·t of a stage covers 8 tile rows
    // (the parts' rows first, then W's); lane i moves row 8 q' + i / 8, chunk
    // (i % 8) ^ (row & 7), so it lands in that chunk's slot. Rows past the end
    // (and fp32 W's columns) re-read the last one.
    const void* src[T::kPerWave];
    uint32_t offset[T::kPerWave];
    uint32_t dst[T::kPerWave]; // byte offset in the stage
#pragma unroll
    for (int t = 0; t < T::kPerWave; ++t)
    {
        const int q = wave + T::kWaves * t;
        if (q < P * T::TM / kLoadRows)
        {
            const int p = q / (T::TM / kLoadRows), rq = q % (T::TM / kLoadRows);
            const int r = kLoadRows * rq + lane / kChunks;
            const int row = min(m_block + r, a.rows - 1);
            src[t] = a.parts;
            offset[t] = (uint32_t) (((size_t) p * a.part_stride + (size_t) row * a.inner) * B);
            dst[t] = p * T::kABytes + 1024 * rq;
        }
        else
        {
            const int wq = q - P * T::TM / kLoadRows;
            const int col = min(n_block - seg_first + kLoadRows * wq + lane / kChunks, width - 1);
            src[t] = w;
            offset[t] = (uint32_t) ((size_t) col * a.inner * B);
            dst[t] = P * T::kABytes + 1024 * wq;
        }
    }
    // (A load's first tile row is a multiple of 8, so every load of a lane
    // moves the same chunk.)
    const uint32_t chunk_bytes = 16 * ((lane % kChunks) ^ (lane / kChunks));
    const uint32_t stage0 = lds_address(stage_mem);
    // Issues step `step`'s loads into stage buffer `buf` (a step past the end
    // reloads the last one into a buffer no one reads again).
    auto issue = [&](int step, int buf) {
        uint32_t k_bytes = (uint32_t) min(step, steps - 1) * kRowBytes + chunk_bytes;
        if constexpr (WT == kF32) // a last step past the row's end: its last chunk instead (zeroed before use)
            k_bytes = min(k_bytes, (uint32_t) a.inner * B - 16);
#pragma unroll
        for (int t = 0; t < T::kPerWave; ++t)
            load_lds16(src[t], offset[t] + k_bytes,
                       __builtin_amdgcn_readfirstlane(stage0 + buf * T::kStageBytes + dst[t]));
    };

    float4v acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
            acc[i][j] = float4v {0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int s = 0; s < T::S - 1; ++s)
        issue(s, s);
    int buf = 0;
    for (int s = 0; s < steps; ++s)
    {
        // This wave's loads of step s are done once at most the later S - 2
        // steps' loads are in flight; the barrier then makes every wave's
        // loads visible and ends every read of the buffer refilled next.
        wait_loads<(T::S - 2) * T::kPerWave>();
        __syncthreads();
        issue(s + T::S - 1, buf == 0 ? T::S - 1 : buf - 1);
        unsigned char* const st = stage_mem + buf * T::kStageBytes;
        if constexpr (WT == kF32)
            if (s == steps - 1 && a.inner % kStep != 0) // the chunks past the rows' end
            {
                const int first = a.inner % kStep / 4; // (inner is a multiple of 4)
                for (int i = tid; i < (T::TM + T::TN) * kChunks; i += T::kWaves * kWave)
                    if (i % kChunks >= first)
                        reinterpret_cast<u32x4*>(st)[chunk_slot(i / kChunks, i % kChunks)] = u32x4 {0, 0, 0, 0};
                __syncthreads();
            }
#pragma unroll
        for (int kk = 0; kk < kChunks / 4; ++kk)
        {
            const int c = 4 * kk + g;
            u32x4 af[MT][P], bf[NT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int p = 0; p < P; ++p)
                    af[mt][p] = reinterpret_cast<const u32x4*>(st + p * T::kABytes)[chunk_slot(16 * (MT * wm + mt) + li, c)];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                bf[nt] = reinterpret_cast<const u32x4*>(st + P * T::kABytes)[chunk_slot(16 * (NT * wn + nt) + li, c)];
#pragma unroll
            for (int p = 0; p < P; ++p)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
                        acc[mt][nt] = multiply<WT>(bf[nt], af[mt][p], acc[mt][nt]);
        }
        buf = buf == T::S - 1 ? 0 : buf + 1;
    }
    wait_loads<0>();

    // acc[mt][nt][r] of lane (g, li) is row li, column 4g + r of that 16 x 16 tile.
    float* y = matrix.y;
    const float* bias = matrix.bias;
    const float scale = matrix.scale;
    // Four columns a lane go out as one store; fp32 products may end inside them.
    const bool quads = width % 4 == 0 && a.ldy % 4 == 0 && a.group_stride % 4 == 0
                       && reinterpret_cast<uintptr_t>(y) % 16 == 0
                       && reinterpret_cast<uintptr_t>(a.residual) % 16 == 0;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
    {
        const int c = n_block - seg_first + 16 * (NT * wn + nt) + 4 * g;
        if (WT == kF32 && c >= width)
            continue;
        float b[4] = {0.f, 0.f, 0.f, 0.f};
        if (bias != nullptr)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                b[r] = bias[WT == kF32 ? min(c + r, width - 1) : c + r];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
        {
            const int row = m_block + 16 * (MT * wm + mt) + li;
            if (row >= a.rows)
                continue;
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
                v[r] = acc[mt][nt][r] * scale + b[r];
                if (a.flags & kProductGelu)
                    v[r] = exact_gelu(v[r]);
            }
            if (WT != kF32 && a.out_parts != nullptr)
            {
                uint32_t bits[4][3];
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    cut_parts<WT>(v[r], bits[r]);
                u16* o = static_cast<u16*>(a.out_parts) + (size_t) row * width + c;
#pragma unroll
                for (int p = 0; p < P; ++p)
                    *reinterpret_cast<uint2*>(o + p * a.out_part_stride)
                        = uint2 {bits[0][p] | (bits[1][p] << 16), bits[2][p] | (bits[3][p] << 16)};
            }
            else if ((seg == 1 && a.y1_halves != nullptr) || (seg == 2 && a.y2_halves_t != nullptr))
            {
                uint32_t hi[4], lo[4];
#pragma unroll
                for (int r = 0; r < 4; ++r)
                {
                    const _Float16 h = (_Float16) v[r];
                    hi[r] = __builtin_bit_cast(u16, h);
                    lo[r] = __builtin_bit_cast(u16, (_Float16) (v[r] - (float) h));
                }
                const size_t part = (size_t) a.halves_pitch * width;
                if (seg == 1)
                {
                    u16* o = static_cast<u16*>(a.y1_halves) + (size_t) row * width + c;
                    *reinterpret_cast<uint2*>(o) = uint2 {hi[0] | (hi[1] << 16), hi[2] | (hi[3] << 16)};
                    *reinterpret_cast<uint2*>(o + part) = uint2 {lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16)};
                }
                else
                {
                    u16* o = static_cast<u16*>(a.y2_halves_t) + (size_t) c * a.halves_pitch + attention_place(row);
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                    {
                        o[(size_t) r * a.halves_pitch] = (u16) hi[r];
                        o[(size_t) r * a.halves_pitch + part] = (u16) lo[r];
                    }
                }
            }
            else if (WT == kF32 && (a.flags & kProductTaps))
            {
                const int p = row / 2;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (c + r < width)
                    {
                        float* o = y + ((size_t) p * width + c + r) * 3;
                        if (row % 2 != 0)
                        {
                            o[2] = v[r];
                            if (p + 1 < a.taps)
                                o[3 * (size_t) width] = v[r];
                            continue;
                        }
                        o[1] = v[r];
                        if (row == 0)
                            o[0] = 0.f;
                        if (row == a.rows - 1)
                            o[2] = 0.f;
                    }
            }
            else if (const size_t at = (size_t) (row / a.rows_per_group) * a.group_stride
                                       + (size_t) (row % a.rows_per_group) * a.ldy + c;
                     quads)
            {
                float4v* o = reinterpret_cast<float4v*>(y + at);
                float4v sum = {v[0], v[1], v[2], v[3]};
                if (a.flags & kProductResidual)
                    sum = (a.residual != nullptr ? *reinterpret_cast<const float4v*>(a.residual + at) : *o) + sum;
                *o = sum;
            }
            else
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (c + r < width)
                    {
                        float* o = y + at + r;
                        const float from = a.residual != nullptr ? a.residual[at + r] : *o;
                        *o = a.flags & kProductResidual ? from + v[r] : v[r];
                    }
        }
    }
}

template <class T, int WT>
hipError_t allow()
{
    return hipFuncSetAttribute(reinterpret_cast<const void*>(&split_product_kernel<T, WT>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, T::S * T::kStageBytes);
}

template <class T, int WT>
hipError_t launch(hipStream_t stream, const SplitProduct& a)
{
    hipLaunchKernelGGL((split_product_kernel<T, WT>), dim3((a.count * a.columns + T::TN - 1) / T::TN, (a.rows + T::TM - 1) / T::TM),
                       dim3(T::kWaves * kWave), T::S * T::kStageBytes, stream, a);
    return hipGetLastError();
}

template <int WT>
struct Tiles
{
    using Widest = Tile<WT, 128, 256, 2, 4, 2>;
    using Shared = Tile<WT, 64, 128, 2, 4, 2>; // (two blocks of a CU)
    using Alone = Tile<WT, 64, 128, 2, 4, 4>;
    using Short = Tile<WT, 32, 128, 2, WT == kF16 ? 4 : 2, 4>; // (bf16: 28 loads a stage)
    using Least = Tile<WT, 32, 64, 2, 2, 4>;
};

template <>
struct Tiles<kF32>
{
    using Whole = Tile<kF32, 64, 64, 2, 2, 2>;
    using Half = Tile<kF32, 32, 64, 2, 2, 2>;
    using Quarter = Tile<kF32, 32, 32, 2, 2, 4>;
};

template <int WT, class... T>
hipError_t allow_each()
{
    hipError_t e = hipSuccess;
    (void) ((e == hipSuccess && (e = allow<T, WT>()) != hipSuccess) || ...);
    return e;
}

template <int WT>
hipError_t allow_tiles()
{
    using T = Tiles<WT>;
    if constexpr (WT == kF32)
        return allow_each<WT, typename T::Whole, typename T::Half, typename T::Quarter>();
    else
        return allow_each<WT, typename T::Widest, typename T::Shared, typename T::Alone, typename T::Short,
                          typename T::Least>();
}

// The largest tile that still occupies half the CUs (the bytes a product moves
// into LDS fall with the tile's extents, but a launch of fewer blocks leaves
// CUs idle for all of it): 128 x 256, 64 x 128, 32 x 128, else 32 x 64. At 1500
// rows 1536 -> 384 ran 9.8 us as 141 blocks of 32 x 128, 13.6 as 72 of 64 x 128
// and 14.5 as 282 of 32 x 64; 768 -> 2304 17.3 as 432 of 64 x 128, 19.9 in 64 x
// 64 and 23 as 108 of 128 x 256. 128 x 256 tiles of several rounds over the
// CUs, or of up to 512 of K, also have to keep four fifths of their rounds busy,
// unless the columns are few and the rows' parts the larger operand: 3000 x 1280
// -> 3072 in two rounds of 288 (56%) 78.1 us, 65.3 as 1128 blocks of 64 x 128;
// 3000 x 256 -> 2048 as 192 (75%) 21.6 and 18.3; but 4500 x 512 -> 1536 as 216
// (84%) 29.1 and 29.9, 6000 x 512 -> 1024 as 188 29.3 and 31.6. With at most one 64 x 128 block a CU, four
// stages hide the loads (5120 -> 1280: 45 us against 60 with two); with more,
// two let the blocks share a CU (768 -> 2304: 17.3 against 19.6 with four).
template <int WT>
hipError_t launch_tiles(hipStream_t stream, const SplitProduct& a)
{
    const long long units = compute_units();
    const int out = a.count * a.columns;
    auto blocks = [&](int tm, int tn) { return (long long) ((a.rows + tm - 1) / tm) * (out / tn); };
    const long long widest = blocks(128, 256), rounds = (widest + units - 1) / units;
    if (a.columns % 256 == 0 && 2 * widest >= units
        && (out <= 1024 || (rounds == 1 && a.inner > 512) || 5 * widest >= 4 * rounds * units))
        return launch<typename Tiles<WT>::Widest, WT>(stream, a);
    if (blocks(64, 128) > units)
        return launch<typename Tiles<WT>::Shared, WT>(stream, a);
    if (2 * blocks(64, 128) >= units)
        return launch<typename Tiles<WT>::Alone, WT>(stream, a);
    if (2 * blocks(32, 128) >= units)
        return launch<typename Tiles<WT>::Short, WT>(stream, a);
    return launch<typename Tiles<WT>::Least, WT>(stream, a);
}
} // namespace

bool split_product_fits(int wdtype, int inner, int columns)
{
    return (wdtype == kF16 || wdtype == kBF16) && inner % 64 == 0 && columns % 128 == 0;
}

hipError_t split_rows(hipStream_t stream, const float* x, size_t count, int wdtype, void* parts, size_t part_stride)
{
    if (count % 8 != 0 || (wdtype != kF16 && wdtype != kBF16))
        return hipErrorInvalidValue;
    const dim3 grid((unsigned) ((count / 8 + kSplitThreads - 1) / kSplitThreads));
    if (wdtype == kF16)
        hipLaunchKernelGGL(split_rows_kernel<kF16>, grid, dim3(kSplitThreads), 0, stream, x, count,
                           static_cast<u16*>(parts), part_stride);
    else
        hipLaunchKernelGGL(split_rows_kernel<kBF16>, grid, dim3(kSplitThreads), 0, stream, x, count,
                           static_cast<u16*>(parts), part_stride);
    return hipGetLastError();
}

bool layernorm_parts_fits(int width)
{
    return width > 0 && width % 4 == 0 && width <= kNormWidth;
}

hipError_t layernorm_parts(hipStream_t stream, const float* x, const float* gamma, const float* beta, void* parts,
                           size_t part_stride, int rows, int width, float eps, int wdtype)
{
    if (!layernorm_parts_fits(width) || (wdtype != kF16 && wdtype != kBF16))
        return hipErrorInvalidValue;
    auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(rows), dim3(kWave), 0, stream, x, gamma, beta, width, eps,
                           static_cast<u16*>(parts), part_stride);
    };
    if (wdtype == kF16)
        width <= 512    ? run(layernorm_parts_kernel<kF16, 2>)
        : width <= 1280 ? run(layernorm_parts_kernel<kF16, 5>)
                        : run(layernorm_parts_kernel<kF16, 8>);
    else
        width <= 512    ? run(layernorm_parts_kernel<kBF16, 2>)
        : width <= 1280 ? run(layernorm_parts_kernel<kBF16, 5>)
                        : run(layernorm_parts_kernel<kBF16, 8>);
    return hipGetLastError();
}

// fp32 X and W through the same kernel, one "part" of four-byte values:
// v_mfma_f32_16x16x4_f32 in 32-wide steps.
bool fp32_split_fits(const SplitProduct& a)
{
    auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    bool fits = a.wdtype == kF32 && a.inner % 4 == 0 && aligned(a.parts) && (a.count == 1 || a.columns % 64 == 0)
                && (unsigned long long) std::max(a.rows, a.columns) * a.inner < 1ull << 30; // 32-bit byte offsets
    for (int i = 0; i < a.count; ++i)
        fits = fits && aligned(a.matrix[i].w);
    return fits;
}

// 64 x 64 tiles, 32 x 64 or 32 x 32, whichever finishes first by its rounds
// over the CUs: a smaller tile costs 1.07 or 1.2 of its share of a 64 x 64
// one's time (more loads a product), so it wins where the larger leaves a
// round part-filled. Measured at 1500 rows (us in that order): 512 -> 512
// 13.2, 13.1, 11.7; 512 -> 1536 30.4, 28.7, 30.6; 512 -> 2048 31.9, 33.3,
// 38.6; 2048 -> 512 41.4, 41.3, 35.4; 3840 -> 1280 129, 134, 153 (247 as 64 x
// 64 tiles of vector multiply-adds).
hipError_t fp32_split(hipStream_t stream, const SplitProduct& product)
{
    if (!fp32_split_fits(product))
        return hipErrorInvalidValue;
    SplitProduct a = product;
    if (a.rows_per_group <= 0)
        a.rows_per_group = a.rows;
    const long long units = compute_units();
    auto rounds = [&](int tm, int tn) {
        return ((long long) ((a.rows + tm - 1) / tm) * ((a.count * a.columns + tn - 1) / tn) + units - 1) / units;
    };
    const double whole = 1.0 * rounds(64, 64), half = 0.535 * rounds(32, 64), quarter = 0.3 * rounds(32, 32);
    if (whole <= half && whole <= quarter)
        return launch<Tiles<kF32>::Whole, kF32>(stream, a);
    if (half <= quarter)
        return launch<Tiles<kF32>::Half, kF32>(stream, a);
    return launch<Tiles<kF32>::Quarter, kF32>(stream, a);
}

hipError_t split_product(hipStream_t stream, const SplitProduct& product)
{
    if (!split_product_fits(product.wdtype, product.inner, product.columns) || product.count < 1
        || product.count > kMaxMatrices)
        return hipErrorInvalidValue;
    SplitProduct a = product;
    if (a.rows_per_group <= 0)
        a.rows_per_group = a.rows;
    return a.wdtype == kF16 ? launch_tiles<kF16>(stream, a) : launch_tiles<kBF16>(stream, a);
}

hipError_t prepare_split_products()
{
    static OncePerDevice prepared;
    int device = 0;
    const hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess)
        return e;
    return prepared(device, [] {
        hipError_t status = allow_tiles<kF16>();
        if (status == hipSuccess)
            status = allow_tiles<kBF16>();
        return status == hipSuccess ? allow_tiles<kF32>() : status;
    });
}
} // namespace wsp::ops
