// y = X·Wᵀ (bias, GELU, residual) for fp32 X in fp32 arithmetic on the matrix
// cores, any weight storage and any extents, and the products of few rows
// (Kernels/Linear.h:129-276, Kernels/SimdTiledMatMul.h:470-486).
//
// fp32_tile_kernel: many rows. v_mfma_f32_16x16x4_f32 multiplies and
// accumulates in fp32 (the same inputs, products and range as fused
// multiply-adds, twice their rate: 157 TFLOP/s against 79 without packed fp32
// instructions). 32 x 64 tiles in 32-wide k-steps, operands widened on their
// way through registers into two LDS buffers, so a step needs one barrier and
// its loads are in flight over the previous step's products. LDS chunk c (four
// k) of row r sits at slot 8r + (c ^ (r & 7)): the operand reads of eight rows
// hit eight bank groups. It takes what split_product's direct-to-LDS loads
// cannot: 16-bit weights to be widened (the 51865-column logits of 96 rows:
// 90 us, 153 as 64 x 64 tiles of vector multiply-adds), rows that are not
// whole 16-byte runs.
//
// row_product_kernel: few rows, where tiles over whole rows of K would leave
// most CUs idle behind a long serial chain (96 x 768 x 768 was 18 blocks of 24
// dependent steps, 28 us). A block takes a small tile and its eight waves
// split K; operands go straight from memory into the matrix-core operand
// registers (a lane's eight consecutive k; any assignment of k to lanes serves
// as long as both operands share it), and the eight partial tiles are added in
// wave order through LDS, so the result does not depend on timing. SPLIT takes
// 16-bit weights in their own type with X cut into 16-bit parts (as
// split_product's), otherwise everything is fp32.
//
// In these two W is the matrix cores' row operand, X their column operand: a
// lane ends up with four consecutive outputs of one row.
//
// cut_product_kernel: many rows of 16-bit weights that split_product does not
// take (K in odd multiples of 32, W not at 16 bytes, or parts that the scratch
// does not hold) and of short K, where storing the parts costs more than it gives. X is cut into its 16-bit parts on its way through registers into LDS, 32 k a step.
#include "device_common.h"
#include "ops.h"

#include <algorithm>

namespace wsp::ops
{
namespace
{
typedef uint16_t u16;
typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(2))); // u32x4 at any 16-bit value

// Up to three matrices a launch here.
constexpr int kMatrices = 3;
struct RowProduct
{
    const float* x;
    int rows, inner, columns, out; // out: every matrix's columns together
    ProductMatrix matrix[kMatrices];
    int ldy, rows_per_group;
    size_t group_stride;
    int flags;
};

// Output column n's matrix, and its column there.
struct Column
{
    const void* w;
    const float* bias;
    float* y;
    int c;
};

__device__ __forceinline__ Column column_of(const RowProduct& a, int n)
{
    if (n < a.columns)
        return {a.matrix[0].w, a.matrix[0].bias, a.matrix[0].y, n};
    if (n < 2 * a.columns)
        return {a.matrix[1].w, a.matrix[1].bias, a.matrix[1].y, n - a.columns};
    return {a.matrix[2].w, a.matrix[2].bias, a.matrix[2].y, n - 2 * a.columns};
}

__device__ __forceinline__ void store_output(const RowProduct& a, int row, int n, float v)
{
    const Column col = column_of(a, n);
    if (col.bias != nullptr)
        v += col.bias[col.c];
    if (a.flags & 1)
        v = exact_gelu(v);
    float* dst = col.y + (size_t) (row / a.rows_per_group) * a.group_stride + (size_t) (row % a.rows_per_group) * a.ldy
                 + col.c;
    if (a.flags & 2)
        v += *dst;
    *dst = v;
}

// COUNT consecutive values of a row from element `index` on, as loaded: kept
// raw until values() so that nothing waits for the load before its use. Past
// the row's end (`left` elements from `index` on) they read as zero. VEC:
// 16-byte loads (8 for four 16-bit values, which may lie at any of them), the
// row's end a multiple of COUNT; a run past it loads the matrix's first values
// instead.
template <int WT, int COUNT, bool VEC>
struct Run
{
    static constexpr int kWords = WT == kF32 || !VEC ? COUNT : COUNT / 2;
    uint32_t raw[kWords];

    __device__ __forceinline__ void load(const void* base, size_t index, int left)
    {
        if constexpr (VEC)
        {
            const size_t at = left > 0 ? index : 0;
            constexpr int kPiece = kWords >= 4 ? 4 : 2;
            typedef uint32_t piece __attribute__((ext_vector_type(kPiece), aligned(WT == kF32 ? 4 * kPiece : 2)));
            const piece* p = reinterpret_cast<const piece*>(static_cast<const char*>(base) + at * (WT == kF32 ? 4 : 2));
#pragma unroll
            for (int i = 0; i < kWords / kPiece; ++i)
            {
                const piece v = p[i];
#pragma unroll
                for (int j = 0; j < kPiece; ++j)
                    raw[kPiece * i + j] = v[j];
            }
        }
        else
#pragma unroll
            for (int i = 0; i < COUNT; ++i)
                raw[i] = __float_as_uint(i < left ? load1<WT>(base, index + i) : 0.f);
    }

    __device__ __forceinline__ void values(float (&v)[COUNT], int left) const
    {
#pragma unroll
        for (int i = 0; i < COUNT; ++i)
        {
            if constexpr (WT == kF32 || !VEC)
                v[i] = __uint_as_float(raw[i]);
            else
            {
                const u16 h = (u16) (raw[i / 2] >> (16 * (i % 2)));
                v[i] = WT == kF16 ? (float) __builtin_bit_cast(_Float16, h) : bf16_to_float(h);
            }
            if (VEC)
                v[i] = left > 0 ? v[i] : 0.f;
        }
    }
};

// ---------------------------------------------------------------------------
// Many rows
// ---------------------------------------------------------------------------
constexpr int kTileThreads = 256;
constexpr int kTileRows = 32, kTileColumns = 64;
constexpr int kTileStep = 32;

template <int WT, bool VEC>
__global__ void __launch_bounds__(kTileThreads, 2) fp32_tile_kernel(RowProduct a)
{
    constexpr int TM = kTileRows, TN = kTileColumns, KS = kTileStep, CH = KS / 4;
    constexpr int MT = TM / 32, NT = TN / 32; // 16 x 16 tiles a wave, waves 2 x 2
    constexpr int RP = kTileThreads / CH;     // rows staged at a time
    constexpr int XC = TM / RP, WC = TN / RP; // chunks a thread stages per step
    __shared__ float4v xs[2][TM * CH], ws[2][TN * CH];

    const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave, li = lane % 16, g = lane / 16;
    const int wm = wave / 2, wn = wave % 2;
    const int m_block = blockIdx.y * TM, n_block = blockIdx.x * TN;
    const int sc = tid % CH, sr = tid / CH; // this thread's chunk of rows sr, sr + RP, ...

    // Rows and columns past the end re-read the last one; their outputs are
    // not stored.
    size_t x_at[XC], w_at[WC];
    const void* w_base[WC];
#pragma unroll
    for (int j = 0; j < XC; ++j)
        x_at[j] = (size_t) min(m_block + sr + RP * j, a.rows - 1) * a.inner;
#pragma unroll
    for (int j = 0; j < WC; ++j)
    {
        const Column col = column_of(a, min(n_block + sr + RP * j, a.out - 1));
        w_base[j] = col.w;
        w_at[j] = (size_t) col.c * a.inner;
    }
    Run<kF32, 4, VEC> xr[XC];
    Run<WT, 4, VEC> wr[WC];
    auto fetch = [&](int k0) {
        const int k = k0 + 4 * sc;
#pragma unroll
        for (int j = 0; j < XC; ++j)
            xr[j].load(a.x, x_at[j] + k, a.inner - k);
#pragma unroll
        for (int j = 0; j < WC; ++j)
            wr[j].load(w_base[j], w_at[j] + k, a.inner - k);
    };
    auto stage = [&](int buf, int k0) {
        const int left = a.inner - k0 - 4 * sc;
        float v[4];
#pragma unroll
        for (int j = 0; j < XC; ++j)
        {
            xr[j].values(v, left);
            xs[buf][chunk_slot(sr + RP * j, sc)] = float4v {v[0], v[1], v[2], v[3]};
        }
#pragma unroll
        for (int j = 0; j < WC; ++j)
        {
            wr[j].values(v, left);
            ws[buf][chunk_slot(sr + RP * j, sc)] = float4v {v[0], v[1], v[2], v[3]};
        }
    };

    float4v acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
            acc[i][j] = float4v {0.f, 0.f, 0.f, 0.f};

    fetch(0);
    stage(0, 0);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < a.inner; k0 += KS)
    {
        const bool more = k0 + KS < a.inner;
        if (more)
            fetch(k0 + KS);
        float4v xf[2][MT], wf[2][NT];
        auto operands = [&](int kk, int set) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                xf[set][mt] = xs[buf][chunk_slot(16 * (MT * wm + mt) + li, 4 * kk + g)];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                wf[set][nt] = ws[buf][chunk_slot(16 * (NT * wn + nt) + li, 4 * kk + g)];
        };
        operands(0, 0);
#pragma unroll
        for (int kk = 0; kk < KS / 16; ++kk)
        {
            if (kk + 1 < KS / 16)
                operands(kk + 1, (kk + 1) % 2);
            __builtin_amdgcn_sched_barrier(0); // the next operands' reads stay ahead of these products
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
                        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[kk % 2][nt][e], xf[kk % 2][mt][e],
                                                                            acc[mt][nt], 0, 0, 0);
        }
        if (more)
            stage(buf ^ 1, k0 + KS); // last read before the previous step's barrier
        __syncthreads();
        buf ^= 1;
    }

#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
    {
        const int row = m_block + 16 * (MT * wm + mt) + li;
        if (row >= a.rows)
            continue;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
                const int n = n_block + 16 * (NT * wn + nt) + 4 * g + r;
                if (n < a.out)
                    store_output(a, row, n, acc[mt][nt][r]);
            }
    }
}

// ---------------------------------------------------------------------------
// Few rows
// ---------------------------------------------------------------------------
constexpr int kRowWaves = 8;
constexpr int kRowChunk = 32; // k a wave takes at a time

// One chunk's operands of a lane: eight k of MT rows and NT columns.
template <int WT, int MT, int NT>
struct RowChunk
{
    Run<kF32, 8, true> x[MT];
    Run<WT, 8, true> w[NT];
};

template <int WT, int MT, int NT, bool SPLIT>
__global__ void __launch_bounds__(kRowWaves * kWave) row_product_kernel(RowProduct a)
{
    static_assert(!SPLIT || WT != kF32, "parts go with 16-bit weights");
    constexpr int P = parts_of<WT>();
    // Interleaved sums per tile: shorter chains of dependent products (a single
    // one issues every 46 clocks instead of 32) and of roundings. With parts,
    // the first part and the smaller ones are summed apart.
    constexpr int SETS = SPLIT ? 2 : MT * NT >= 4 ? 1 : 4 / (MT * NT);
    __shared__ float4v sums[kRowWaves][MT * NT][kWave];

    const int tid = threadIdx.x, lane = tid % kWave, li = lane % 16, g = lane / 16;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int m_block = blockIdx.y * 16 * MT, n_block = blockIdx.x * 16 * NT;

    size_t x_at[MT], w_at[NT];
    const void* w_base[NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
        x_at[mt] = (size_t) min(m_block + 16 * mt + li, a.rows - 1) * a.inner;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
    {
        const Column col = column_of(a, min(n_block + 16 * nt + li, a.out - 1));
        w_base[nt] = col.w;
        w_at[nt] = (size_t) col.c * a.inner;
    }
    float4v acc[SETS][MT][NT];
#pragma unroll
    for (int i = 0; i < SETS; ++i)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                acc[i][mt][nt] = float4v {0.f, 0.f, 0.f, 0.f};

    using Chunk = RowChunk<WT, MT, NT>;
    auto load = [&](Chunk& ch, int chunk) {
        const int k = kRowChunk * chunk + 8 * g, left = a.inner - k;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
            ch.x[mt].load(a.x, x_at[mt] + k, left);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            ch.w[nt].load(w_base[nt], w_at[nt] + k, left);
    };
    auto multiply = [&](const Chunk& ch, int chunk) {
        const int left = a.inner - kRowChunk * chunk - 8 * g;
        float x[MT][8];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
            ch.x[mt].values(x[mt], left);
        if constexpr (SPLIT) // (whole chunks: left is never short)
        {
            u32x4 xb[MT][3], wb[NT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                {
                    uint32_t b0[3], b1[3];
                    cut_parts<WT>(x[mt][2 * j], b0);
                    cut_parts<WT>(x[mt][2 * j + 1], b1);
#pragma unroll
                    for (int p = 0; p < 3; ++p)
                        xb[mt][p][j] = b0[p] | (b1[p] << 16);
                }
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                wb[nt] = u32x4 {ch.w[nt].raw[0], ch.w[nt].raw[1], ch.w[nt].raw[2], ch.w[nt].raw[3]};
#pragma unroll
            for (int p = 0; p < P; ++p)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
                        {
                        float4v& sum = acc[p == 0 ? 0 : 1][mt][nt];
                        sum = mfma16<WT>(wb[nt], xb[mt][p], sum);
                    }
        }
        else
        {
            float w[NT][8];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                ch.w[nt].values(w[nt], left);
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
                    {
                        float4v& sum = acc[e % SETS][mt][nt];
                        sum = __builtin_amdgcn_mfma_f32_16x16x4f32(w[nt][e], x[mt][e], sum, 0, 0, 0);
                    }
        }
    };
    // Chunks wave, wave + 8, ..., the next one's loads ahead of this one's products.
    const int chunks = (a.inner + kRowChunk - 1) / kRowChunk;
    Chunk c0, c1;
    if (wave < chunks)
        load(c0, wave);
    for (int chunk = wave; chunk < chunks; chunk += 2 * kRowWaves)
    {
        const bool second = chunk + kRowWaves < chunks;
        if (second)
            load(c1, chunk + kRowWaves);
        multiply(c0, chunk);
        if (!second)
            break;
        if (chunk + 2 * kRowWaves < chunks)
            load(c0, chunk + 2 * kRowWaves);
        multiply(c1, chunk + kRowWaves);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
        {
            float4v total = acc[SETS - 1][mt][nt];
#pragma unroll
            for (int i = SETS - 2; i >= 0; --i)
                total += acc[i][mt][nt];
            sums[wave][mt * NT + nt][lane] = total;
        }
    __syncthreads();
    // Consecutive threads take consecutive columns of a row.
    constexpr int kOutputs = MT * NT * 256;
#pragma unroll
    for (int i = 0; i < (kOutputs + kRowWaves * kWave - 1) / (kRowWaves * kWave); ++i)
    {
        const int at = tid + i * kRowWaves * kWave;
        if (at >= kOutputs)
            break;
        const int n = at % (16 * NT), m = at / (16 * NT);
        const int tile = m / 16 * NT + n / 16, from = m % 16 + 16 * (n % 16 / 4);
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < kRowWaves; ++w)
            v += reinterpret_cast<const float*>(&sums[w][tile][from])[n % 4];
        if (m_block + m < a.rows && n_block + n < a.out)
            store_output(a, m_block + m, n_block + n, v);
    }
}

// ---------------------------------------------------------------------------
// Many rows, parts cut on the way
// ---------------------------------------------------------------------------
constexpr int kCutThreads = 256;
constexpr int kCutColumns = 128;
constexpr int kCutStep = 32;
constexpr int kCutRow = kCutStep + 16; // 16-bit values an LDS row: at 96 bytes its reads conflict half as often as at 80

// TM rows by 128 columns of one matrix a block, its four waves 2 x 2; the next
// step's loads are in flight over this one's products.
template <int WT, int TM>
__global__ void __launch_bounds__(kCutThreads) cut_product_kernel(RowProduct a)
{
    constexpr int P = parts_of<WT>(), NT = 4;
    constexpr int MT = TM / 32;                       // 16-row tiles a wave
    constexpr int kValues = TM * kCutStep / kCutThreads; // of X a thread moves a step: 16, 8 or 4
    constexpr int kRowThreads = kCutStep / kValues;
    __shared__ __attribute__((aligned(16))) u16 xs[P][TM][kCutRow];
    __shared__ __attribute__((aligned(16))) u16 ws[kCutColumns][kCutRow];

    const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave, li = lane % 16, g = lane / 16;
    const int wm = wave / 2, wn = wave % 2;
    const int m_block = blockIdx.y * TM, n_block = blockIdx.x * kCutColumns;
    const Column first = column_of(a, n_block);

    // Rows past the end re-read the last one; their outputs are not stored.
    const int xr = tid / kRowThreads, xk = tid % kRowThreads * kValues;
    constexpr int kRuns = kValues / 4;
    const int wr = tid / 2, wk = tid % 2 * 16;
    const float* const x = a.x + (size_t) min(m_block + xr, a.rows - 1) * a.inner + xk;
    const u16* const w = static_cast<const u16*>(first.w) + (size_t) (first.c + wr) * a.inner + wk;
    float4v xv[kRuns];
    u32x4 wv[2];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < kRuns; ++i)
            xv[i] = *reinterpret_cast<const float4v*>(x + k0 + 4 * i);
#pragma unroll
        for (int i = 0; i < 2; ++i)
            wv[i] = *reinterpret_cast<const u32x4u*>(w + k0 + 8 * i);
    };

    float4v acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            acc[mt][nt] = float4v {0.f, 0.f, 0.f, 0.f};

    fetch(0);
    for (int k0 = 0; k0 < a.inner; k0 += kCutStep)
    {
        __syncthreads(); // the previous step has been read
        uint2 cut[kRuns][P];
#pragma unroll
        for (int i = 0; i < kRuns; ++i)
        {
            uint32_t bits[4][3];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                cut_parts<WT>(xv[i][e], bits[e]);
#pragma unroll
            for (int p = 0; p < P; ++p)
                cut[i][p] = uint2 {bits[0][p] | (bits[1][p] << 16), bits[2][p] | (bits[3][p] << 16)};
        }
#pragma unroll
        for (int p = 0; p < P; ++p)
            if constexpr (kRuns == 1)
                *reinterpret_cast<uint2*>(&xs[p][xr][xk]) = cut[0][p];
            else
#pragma unroll
                for (int i = 0; i < kRuns; i += 2)
                    *reinterpret_cast<u32x4*>(&xs[p][xr][xk + 4 * i])
                        = u32x4 {cut[i][p].x, cut[i][p].y, cut[i + 1][p].x, cut[i + 1][p].y};
#pragma unroll
        for (int i = 0; i < 2; ++i)
            *reinterpret_cast<u32x4*>(&ws[wr][wk + 8 * i]) = wv[i];
        __syncthreads();
        if (k0 + kCutStep < a.inner)
            fetch(k0 + kCutStep);
        u32x4 xf[MT][P], wf[NT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int p = 0; p < P; ++p)
                xf[mt][p] = *reinterpret_cast<const u32x4*>(&xs[p][16 * (MT * wm + mt) + li][8 * g]);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            wf[nt] = *reinterpret_cast<const u32x4*>(&ws[16 * (NT * wn + nt) + li][8 * g]);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int p = 0; p < P; ++p)
                    acc[mt][nt] = mfma16<WT>(xf[mt][p], wf[nt], acc[mt][nt]);
    }

    // acc[mt][nt][r] of lane (g, li) is row 4g + r, column li of that tile.
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            const int row = m_block + 16 * (MT * wm + mt) + 4 * g + r;
            if (row >= a.rows)
                continue;
            float* const y = first.y + (size_t) (row / a.rows_per_group) * a.group_stride
                             + (size_t) (row % a.rows_per_group) * a.ldy;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
            {
                const int c = first.c + 16 * (NT * wn + nt) + li;
                float v = acc[mt][nt][r];
                if (first.bias != nullptr)
                    v += first.bias[c];
                if (a.flags & 1)
                    v = exact_gelu(v);
                y[c] = a.flags & 2 ? y[c] + v : v;
            }
        }
}

bool aligned(const void* p, size_t bytes)
{
    return reinterpret_cast<uintptr_t>(p) % bytes == 0;
}

// Whether X and every matrix take whole vector loads of `run` values.
bool whole_vectors(const Products& a, int run)
{
    bool fits = a.inner % run == 0 && aligned(a.x, 16);
    for (int i = 0; i < a.count; ++i)
        fits = fits && aligned(a.matrices[i].w, a.wdtype == kF32 ? 16 : 2 * run);
    return fits;
}

template <int WT, bool VEC>
hipError_t launch_tile(hipStream_t stream, const RowProduct& a)
{
    hipLaunchKernelGGL((fp32_tile_kernel<WT, VEC>), dim3((a.out + kTileColumns - 1) / kTileColumns,
                                                         (a.rows + kTileRows - 1) / kTileRows),
                       dim3(kTileThreads), 0, stream, a);
    return hipGetLastError();
}

template <int WT, int MT, int NT, bool SPLIT>
hipError_t launch_row(hipStream_t stream, const RowProduct& a)
{
    hipLaunchKernelGGL((row_product_kernel<WT, MT, NT, SPLIT>),
                       dim3((a.out + 16 * NT - 1) / (16 * NT), (a.rows + 16 * MT - 1) / (16 * MT)),
                       dim3(kRowWaves * kWave), 0, stream, a);
    return hipGetLastError();
}

template <int WT, int TM>
hipError_t launch_cut(hipStream_t stream, const RowProduct& a)
{
    hipLaunchKernelGGL((cut_product_kernel<WT, TM>), dim3(a.out / kCutColumns, (a.rows + TM - 1) / TM),
                       dim3(kCutThreads), 0, stream, a);
    return hipGetLastError();
}

RowProduct row_product(const Products& p, int first, int count)
{
    RowProduct a {};
    a.x = p.x;
    a.rows = p.rows;
    a.inner = p.inner;
    a.columns = p.columns;
    a.out = count * p.columns;
    for (int i = 0; i < count; ++i)
        a.matrix[i] = p.matrices[first + i];
    a.ldy = p.ldy;
    a.rows_per_group = p.rows_per_group;
    a.group_stride = p.group_stride;
    a.flags = p.flags;
    return a;
}

SplitProduct split_product_of(const Products& p, const void* parts, size_t part_stride, int first, int count)
{
    SplitProduct a {};
    a.parts = parts;
    a.part_stride = part_stride;
    a.rows = p.rows;
    a.inner = p.inner;
    a.count = count;
    a.columns = p.columns;
    for (int i = 0; i < count; ++i)
        a.matrix[i] = p.matrices[first + i];
    a.ldy = p.ldy;
    a.rows_per_group = p.rows_per_group;
    a.group_stride = p.group_stride;
    a.flags = p.flags;
    a.wdtype = p.wdtype;
    return a;
}

// Rows of X whose parts the scratch holds at a time: all of them, else half of
// them in whole 32-row tiles; 0 where it holds less or fewer than kLeastSlab
// rows, or where the output's rows lie in groups. (In shorter slabs each launch
// leaves CUs idle: 1500 x 16384 -> 1280 in six of 256 rows 365 us, 306 in
// cut_product_kernel, 3000 x 5120 -> 384 in four 110 against 102; 1000 x 8192 ->
// 512 in two 72 against 144.)
constexpr int kLeastSlab = 512;
int slab_rows(const Products& p, const Scratch& scratch)
{
    const size_t row_bytes = (size_t) p.inner * 2 * (p.wdtype == kF16 ? 2 : 3);
    const size_t held = std::min(scratch.bytes / row_bytes, ((size_t) (1u << 29) - 1) / p.inner); // (32-bit byte offsets)
    if ((size_t) p.rows <= held)
        return p.rows;
    const int whole = (int) (held / 32 * 32);
    const int half = ((p.rows + 1) / 2 + 31) / 32 * 32;
    return whole < kLeastSlab || half > whole || p.rows > p.rows_per_group ? 0 : half;
}

// Parts without storing them, two or three matrices at a time. Up to 2^17 outputs
// row_product_kernel in 16 x 32 tiles; more, in 32 x 64 tiles while those do not
// give each CU one, or two where K is long (a tile's eight waves share it):
// 300 x 1056 -> 1152 10.5 us against 18.5 in cut_product_kernel's tiles, 700 x
// 3104 -> 768 40 against 59, but 300 x 96 -> 5120 14 against 7.2 and 1500 x
// 2080 -> 5120 215 against 92. Those tiles are of 128 rows, halved while they
// give fewer than four blocks a CU, and again below one.
template <int WT>
hipError_t unstored_parts_product(hipStream_t stream, const Products& p)
{
    const long long units = compute_units(), out = (long long) p.columns * p.count;
    auto blocks = [&](int tm, int tn) { return (p.rows + tm - 1) / tm * (out / tn); };
    const bool few = p.rows * out <= 1 << 17, some = blocks(32, 64) <= (p.inner < 1024 ? units : 2 * units);
    hipError_t e = hipSuccess;
    for (int i = 0; i < p.count && e == hipSuccess; i += kMatrices)
    {
        const RowProduct a = row_product(p, i, std::min(kMatrices, p.count - i));
        e = few                               ? launch_row<WT, 1, 2, true>(stream, a)
            : some                            ? launch_row<WT, 2, 4, true>(stream, a)
            : blocks(64, 128) < units         ? launch_cut<WT, 32>(stream, a)
            : blocks(128, 128) < 4 * units    ? launch_cut<WT, 64>(stream, a)
                                              : launch_cut<WT, 128>(stream, a);
    }
    return e;
}

// 16-bit weights with X in 16-bit parts. From 2^17 outputs on (every matrix
// together) X is stored as parts, every matrix going through split_product in
// launches of up to 64; fewer, and what split_product or the scratch does not
// take, without (96 x 768 -> 768 runs 5.3 us there, 96 x 3072 -> 768 13; 200 x
// 5120 -> 1280 39, against 20 with the parts' launch). So do, where one launch
// takes every matrix, two shapes that do not make up for the launch that stores
// the parts: short K over many rows whose tiles in split_product are one round
// at most (300 x 64 -> 768 7.0 us, 5.5 without; 1500 x 384 -> 768 in three parts 14.3, 11.3 without; 3000 x 384 ->
// 384 in two 12.7 and 10.7; but 448 x 384 -> 1152 7.5 and 9.7, 1500 x 512 ->
// 1152 in two 14.8 and 15.6), and few columns under very many rows (12000 x 768 ->
// 768 in three parts 79.7 and 67.8, in two 62.3 and 56.8 but 6000 x 1280 -> 768
// 50.6 and 53.7: in two up to 512 of K).
template <int WT>
hipError_t parts_product(hipStream_t stream, const Products& p, const Scratch& scratch)
{
    const long long units = compute_units(), out = (long long) p.columns * p.count, outputs = p.rows * out;
    auto blocks = [&](int tm, int tn) { return (p.rows + tm - 1) / tm * (out / tn); };
    const int slab = slab_rows(p, scratch);
    const bool short_inner = p.count <= kMatrices && blocks(64, 128) <= units
                             && (p.inner <= 64 || (p.inner <= (WT == kF16 ? 384 : 512) && p.rows >= 700
                                                   && 2 * blocks(WT == kF16 ? 64 : 32, 128) >= units));
    const bool few_columns = p.count <= kMatrices && p.rows >= 4500
                             && (WT == kF16 ? out <= 768 && p.inner <= 512 : out <= 1024);
    if (outputs <= 1 << 17 || short_inner || few_columns || slab == 0 || !whole_vectors(p, 8)
        || !split_product_fits(p.wdtype, p.inner, p.columns) || (size_t) p.columns * p.inner >= 1u << 30) // (32-bit byte offsets)
        return unstored_parts_product<WT>(stream, p);
    hipError_t e = hipSuccess;
    for (int first = 0; first < p.rows && e == hipSuccess; first += slab)
    {
        const int rows = std::min(slab, p.rows - first);
        const size_t values = (size_t) rows * p.inner;
        e = split_rows(stream, p.x + (size_t) first * p.inner, values, p.wdtype, scratch.data, values);
        for (int i = 0; i < p.count && e == hipSuccess; i += kMaxMatrices)
        {
            SplitProduct a = split_product_of(p, scratch.data, values, i, std::min(kMaxMatrices, p.count - i));
            a.rows = rows;
            for (int m = 0; m < a.count; ++m)
                a.matrix[m].y += (size_t) first * p.ldy;
            e = split_product(stream, a);
        }
    }
    return e;
}

// fp32 arithmetic. Up to 16 rows, and while 32 x 32 tiles would not give each
// CU one, row_product_kernel: 96 x 3072 -> 768 ran 19 us against 36 in such
// tiles, 200 x 1280 -> 1280 (280 tiles) 20 against 17.6. fp32 weights
// otherwise take split_product's direct-to-LDS form (1500 x 2048 -> 512 35 us
// against 48 staged through registers), the rest fp32_tile_kernel.
template <int WT>
hipError_t fp32_product(hipStream_t stream, const Products& p)
{
    const long long units = compute_units();
    const int out = p.count * p.columns;
    auto blocks = [&](int tm, int tn) { return (long long) ((p.rows + tm - 1) / tm) * ((out + tn - 1) / tn); };
    const bool few = (p.rows <= kSplitRowLimit || blocks(32, 32) < units) && whole_vectors(p, 8);
    hipError_t e = hipSuccess;
    if (!few && WT == kF32 && p.count <= kMaxMatrices)
    {
        const SplitProduct a = split_product_of(p, p.x, 0, 0, p.count);
        if (fp32_split_fits(a))
            return fp32_split(stream, a);
    }
    for (int i = 0; i < p.count && e == hipSuccess; i += kMatrices)
    {
        const RowProduct a = row_product(p, i, std::min(kMatrices, p.count - i));
        if (few && p.rows > 16)
            e = launch_row<WT, 2, 1, false>(stream, a);
        else if (few) // (16 x 1280 -> 5120: 9.8 us with 32 columns a block, 11.3 with 16; 8 x 768 -> 3072: 6.1 and 4.4)
            e = blocks(16, 16) > units ? launch_row<WT, 1, 2, false>(stream, a)
                                       : launch_row<WT, 1, 1, false>(stream, a);
        else
            e = whole_vectors(p, 4) ? launch_tile<WT, true>(stream, a) : launch_tile<WT, false>(stream, a);
    }
    return e;
}
} // namespace

bool parts_fit(int wdtype, int inner, int columns, const void* x)
{
    return (wdtype == kF16 || wdtype == kBF16) && inner % 32 == 0 && columns % 128 == 0 && aligned(x, 16);
}

bool row_product_fits(const Products& product)
{
    return product.rows <= kSplitRowLimit && whole_vectors(product, 8);
}

namespace
{
// Rows of one call at most: their tiles (of 16 at least) are a launch's y extent,
// which ends at 65535.
constexpr int kMostRows = 1 << 19;

// Longer products of one group of rows, in equal calls.
hipError_t products_in_calls(hipStream_t stream, const Products& p, const Scratch& scratch)
{
    const int calls = (p.rows + kMostRows - 1) / kMostRows, most = (p.rows + calls - 1) / calls;
    hipError_t e = hipSuccess;
    for (int first = 0; first < p.rows && e == hipSuccess; first += most)
        for (int i = 0; i < p.count && e == hipSuccess; i += kMaxMatrices)
        {
            ProductMatrix matrices[kMaxMatrices];
            Products part = p;
            part.x += (size_t) first * p.inner;
            part.rows = part.rows_per_group = std::min(most, p.rows - first);
            part.matrices = matrices;
            part.count = std::min(kMaxMatrices, p.count - i);
            for (int m = 0; m < part.count; ++m)
            {
                matrices[m] = p.matrices[i + m];
                matrices[m].y += (size_t) first * p.ldy;
            }
            e = products(stream, part, scratch);
        }
    return e;
}
} // namespace

hipError_t products(hipStream_t stream, const Products& given, const Scratch& scratch)
{
    Products p = given;
    if (p.rows_per_group <= 0)
        p.rows_per_group = p.rows;
    if (p.rows > kMostRows && p.rows_per_group >= p.rows)
        return products_in_calls(stream, p, scratch);
    const bool parts = p.rows > kSplitRowLimit && parts_fit(p.wdtype, p.inner, p.columns, p.x);
    switch (p.wdtype)
    {
        case kF32: return fp32_product<kF32>(stream, p);
        case kF16: return parts ? parts_product<kF16>(stream, p, scratch) : fp32_product<kF16>(stream, p);
        default: return parts ? parts_product<kBF16>(stream, p, scratch) : fp32_product<kBF16>(stream, p);
    }
}
} // namespace wsp::ops
