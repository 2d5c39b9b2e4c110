// The Whisper encoder (Encoder/Encoder.cpp:82-111) on gfx950: the step before
// the decode path, producing the [positions, width] rows the decoder's cross
// keys and values are projected from.
//
//   x = gelu(conv1(mel))   stride 1, kernel 3, padding 1
//   x = gelu(conv2(x))     stride 2: the frames halve into positions
//   h = x + embed_positions
//   per layer: h += out_proj(attention(LN(h)));  h += fc2(gelu(fc1(LN(h))))
//   rows = LN(h)
//
// Both convolutions are products over rows that hold, for every output frame,
// the three taps of every input channel (index channel * 3 + tap, the order of
// a [out, in, 3] weight row), with zero past the frames the run was given
// (Encoder/Encoder.h:46-56). A column kernel gathers the first's from the mel;
// the first's product writes the second's itself, and the second's adds the
// positional table. The projections are split_product's or the library's
// products, the attention flash_attention_kernel for heads of 64 channels and
// the library's otherwise.
#include "../../include/wsp_hip.h"
#include "device_common.h"
#include "ops.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdio>
#include <new>
#include <vector>

namespace wsp::encoder
{
namespace
{
constexpr int kColumnThreads = 256;
constexpr int kFlashWaves = 4;     // queries per attention block: 16 per wave
constexpr int kFlashWideWaves = 8; // the same with twice the queries per K/V tile, when the blocks still fill the chip
constexpr int kMaxFlashSplits = 4; // key splits of the attention when its 64-query blocks leave CUs idle

// Kernels/Conv1d.h:121-124 with kernel 3 and padding 1.
int conv_length(int length, int stride)
{
    return (length + 2 - 3) / stride + 1;
}

// Row t of the first convolution's columns: mel[s][t + tap - 1] at
// s * 3 + tap. The mel is band-major with `stride` frames a band, of which
// the run reads the first `frames`.
//
// The first `clearing` blocks set the attention's values to zero from the run's
// `positions` to the end of their key tile: it reads them with weight zero,
// which hides what an earlier, longer run left there only while it is finite. A
// thread takes four keys of a channel, which attention_place keeps together.
// (A launch of their own would cost an encode a few microseconds; stale keys
// need no clearing, their scores are masked.)
constexpr int kClearedQuads = 16; // of a 64-key tile

__global__ void __launch_bounds__(kColumnThreads) mel_columns_kernel(const float* __restrict__ mel, int bins,
                                                                     int stride, int frames,
                                                                     float* __restrict__ columns, int clearing,
                                                                     int positions, int width, int pitch,
                                                                     uint16_t* __restrict__ vt_halves)
{
    const int t = (int) blockIdx.x - clearing;
    if (t < 0)
    {
        const int i = blockIdx.x * kColumnThreads + threadIdx.x, row = i / kClearedQuads; // [part][channel]
        const int key = (positions - 1) / (4 * kClearedQuads) * (4 * kClearedQuads) + 4 * (i % kClearedQuads);
        if (row >= 2 * width || key + 4 <= positions)
            return;
        uint16_t* const at = vt_halves + (size_t) row * pitch + attention_place(key);
        if (key >= positions)
            *reinterpret_cast<uint2*>(at) = uint2 {0, 0};
        else
            for (int e = positions - key; e < 4; ++e)
                at[e] = 0;
        return;
    }
    const int inner = bins * 3;
    for (int i = threadIdx.x; i < inner; i += kColumnThreads)
    {
        const int s = i / 3, at = t + i % 3 - 1;
        columns[(size_t) t * inner + i] = at >= 0 && at < frames ? mel[(size_t) s * stride + at] : 0.f;
    }
}

// ---------------------------------------------------------------------------
// Self attention of the encoder (Tests/Encoder/Common.h:547-594: every query
// sees every key, softmax(scale q.k) v per head) for head width 64, on the
// matrix cores, one pass over the keys with an online softmax.
//
// A block takes 16 queries per wave of one head; key tiles of 64 rows of K
// and V go through LDS once for all its waves (a large-v3 window took 12.19
// ms with 64-key tiles, 12.33 with 32, 12.30 with 128: half the barriers and
// softmax passes of 32, fewer registers than 128).
// Every fp32 operand is cut into fp16 parts, hi = fp16(x) and
// lo = fp16(x - hi), and a product takes
// the three terms hi·hi + hi·lo + lo·hi (v_mfma_f32_16x16x32_f16, fp32
// accumulation): what is dropped, lo·lo, is about 2^-22 of the product, so
// the sums stay at fp32 rather than fp16 accuracy.
//
// Layout: the wave computes S^T = K·Q^T, so lane (g, l) holds the scores of
// keys 4g..4g+3 and 16+4g..16+4g+3 of each 32-key block of the tile for
// query l — exactly the B operand of O^T = V^T·P^T once the key order
// inside each 32-key block is taken as (4g..4g+3, 16+4g..16+4g+3) for both
// operands, so P
// never leaves its registers. V is staged transposed for that A operand.
// Weights are exp2 of the scores in base-2 units (one fused multiply-add and
// one v_exp_f32 each); a new tile rescales the running row by
// exp2(m_old - m_new) (exact online softmax) where a maximum grew, and only the
// last tile masks keys. The vector instructions between the products are what
// a large-v3 layer's launch waits for: with the library exp2f's range
// handling, a mask per tile and a rescale per tile they were about 300 a tile
// against 48 products, 64 us a launch; now about 140, 55 us.
// ---------------------------------------------------------------------------
constexpr int kFlashKeys = 64;
constexpr int kFlashWidth = 64;
constexpr int kFlashStages = 2; // 32 KB each
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ _Float16 half_hi(float x)
{
    return (_Float16) x;
}

__device__ __forceinline__ _Float16 half_lo(float x)
{
    return (_Float16) (x - (float) (_Float16) x);
}

__device__ __forceinline__ f32x4 mfma3(const f16x8& ah, const f16x8& al, const f16x8& bh, const f16x8& bl, f32x4 c)
{
    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bh, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bl, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(al, bh, c, 0, 0, 0);
}

// K and V arrive cut into fp16 hi and lo (k_halves [2][pitch][width], vt_halves
// transposed [2][width][pitch] with each 32 keys in attention_place order, pitch
// a multiple of the key tile): the q/k/v product writes them, or halves_kernel.
// Tiles go straight from there into LDS (direct-to-LDS loads, two stages, one
// barrier a tile; chunk c of row r at slot 8r + (c ^ (r & 7)), so an operand
// read's eight rows hit eight bank groups).
//
// Key splits: blockIdx.z takes keys [z·span, min((z + 1)·span, count)); with
// one split the block writes the normalised rows to out (OUT = kF32) or as
// the 16-bit parts of the output product's input (OUT = kF16, kBF16:
// part p at out_parts + p·out_part_stride), with several it writes (max, sum,
// row) partials [split][head][query][66] for flash_combine_kernel.
template <int WAVES, int OUT>
__global__ void __launch_bounds__(WAVES * 64) flash_attention_kernel(const float* __restrict__ q, int count,
                                                                    int width, float scale2, float* __restrict__ out,
                                                                    int span, float* __restrict__ partials,
                                                                    const uint16_t* __restrict__ k_halves,
                                                                    const uint16_t* __restrict__ vt_halves, int pitch,
                                                                    uint16_t* __restrict__ out_parts,
                                                                    size_t out_part_stride)
{
    constexpr int KB = kFlashKeys / 32;            // 32-key blocks of a tile (P·V k-steps)
    constexpr int kPartBytes = kFlashKeys * 128;   // one part of a tile of K, or of V^T
    constexpr int kStageBytes = 4 * kPartBytes;    // K hi, K lo, V hi, V lo
    constexpr int kPerWave = kStageBytes / 1024 / WAVES;
    static_assert(kFlashKeys == 64 && kFlashWidth == 64, "rows of 64 halves, in both K and V^T");
    __shared__ __attribute__((aligned(16))) unsigned char stages[kFlashStages][kStageBytes];

    const int head = blockIdx.y;
    const int lane = threadIdx.x % 64, li = lane % 16, g = lane / 16;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int column = head * kFlashWidth;
    const int query = blockIdx.x * 16 * WAVES + 16 * wave + li;
    const bool query_in = query < count;
    const int k_begin = (int) blockIdx.z * span, k_end = min(count, k_begin + span);
    const int tiles = max(0, k_end - k_begin + kFlashKeys - 1) / kFlashKeys;

    // This wave's loads: load i moves eight rows (128 bytes each) of one part.
    const void* src[kPerWave];
    uint32_t offset[kPerWave], advance[kPerWave], dst[kPerWave];
#pragma unroll
    for (int t = 0; t < kPerWave; ++t)
    {
        const int i = wave + WAVES * t, part = i / 8 % 2, row = 8 * (i % 8) + lane / 8, chunk = (lane % 8) ^ (row & 7);
        const bool is_key = i < 16;
        src[t] = is_key ? k_halves : vt_halves;
        offset[t] = 2 * (uint32_t) (part * (size_t) pitch * width
                                    + (is_key ? (size_t) (k_begin + row) * width + column
                                              : (size_t) (column + row) * pitch + k_begin)
                                    + 8 * chunk);
        advance[t] = is_key ? 2 * kFlashKeys * width : 2 * kFlashKeys;
        dst[t] = 1024 * i;
    }
    const uint32_t stage0 = lds_address(stages);
    // (a tile past the last reloads it, into a stage no one reads again)
    auto issue = [&](int tile, int stage) {
#pragma unroll
        for (int t = 0; t < kPerWave; ++t)
            load_lds16(src[t], offset[t] + (uint32_t) min(tile, tiles - 1) * advance[t],
                       __builtin_amdgcn_readfirstlane(stage0 + stage * kStageBytes + dst[t]));
    };

    // This lane's B fragments of Q^T: query `query`, dims 32 s + 8 g .. + 7.
    f16x8 qh[2], ql[2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
    {
        const float* from = q + (size_t) min(query, count - 1) * width + column + 32 * s + 8 * g;
        const f32x4 a = *reinterpret_cast<const f32x4*>(from);
        const f32x4 b = *reinterpret_cast<const f32x4*>(from + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e)
        {
            qh[s][e] = half_hi(a[e]);
            ql[s][e] = half_lo(a[e]);
            qh[s][4 + e] = half_hi(b[e]);
            ql[s][4 + e] = half_lo(b[e]);
        }
    }

    float m = -INFINITY, l = 0.f;
    f32x4 o[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
        o[t] = f32x4 {0.f, 0.f, 0.f, 0.f};

    if (tiles > 0)
#pragma unroll
        for (int t = 0; t < kFlashStages - 1; ++t)
            issue(t, t);
    int stage = 0;
    for (int tile = 0; tile < tiles; ++tile)
    {
        // This wave's loads of the tile are done once only the later stages'
        // are in flight; the barrier makes every wave's visible and ends every
        // read of the stage refilled next.
        wait_loads<(kFlashStages - 2) * kPerWave>();
        __syncthreads();
        issue(tile + kFlashStages - 1, stage == 0 ? kFlashStages - 1 : stage - 1);
        const int first = k_begin + tile * kFlashKeys;
        const f16x8* const ks = reinterpret_cast<const f16x8*>(stages[stage]);
        const f16x8* const vs = ks + 2 * kPartBytes / 16;

        // S^T for keys 16 mt + 4 g + r of the tile, query li.
        f32x4 st_[2 * KB];
#pragma unroll
        for (int mt = 0; mt < 2 * KB; ++mt)
        {
            st_[mt] = f32x4 {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 2; ++s)
            {
                const int from = chunk_slot(16 * mt + li, 4 * s + g);
                st_[mt] = mfma3(ks[from], ks[kPartBytes / 16 + from], qh[s], ql[s], st_[mt]);
            }
        }
        if (first + kFlashKeys > k_end) // the last tile: its keys past the end
#pragma unroll
            for (int mt = 0; mt < 2 * KB; ++mt)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    st_[mt][r] = first + 16 * mt + 4 * g + r < k_end ? st_[mt][r] : -INFINITY;
        float tile_max = -INFINITY;
#pragma unroll
        for (int mt = 0; mt < 2 * KB; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                tile_max = fmaxf(tile_max, st_[mt][r]);
        tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 16));
        tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 32));
        // The running row is rescaled only where some query's maximum grew
        // (its factor is exactly 1 elsewhere).
        const float m_new = fmaxf(m, tile_max);
        if (__any(m_new != m))
        {
            const float alpha = __builtin_amdgcn_exp2f((m - m_new) * scale2);
            l *= alpha;
#pragma unroll
            for (int t = 0; t < 4; ++t)
                o[t] *= alpha;
            m = m_new;
        }
        const float top = m * scale2;
        float p[8 * KB], own = 0.f;
#pragma unroll
        for (int j = 0; j < 8 * KB; ++j)
        {
            p[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(st_[j / 4][j % 4], scale2, -top));
            own += p[j];
        }
        l += own;
        // Key block b (keys 32 b .. 32 b + 31 of the tile) takes p[8 b .. 8 b + 7].
        f16x8 ph[KB], pl[KB];
#pragma unroll
        for (int b = 0; b < KB; ++b)
#pragma unroll
            for (int j = 0; j < 8; ++j)
            {
                ph[b][j] = half_hi(p[8 * b + j]);
                pl[b][j] = half_lo(p[8 * b + j]);
            }
#pragma unroll
        for (int t = 0; t < 4; ++t)
        {
#pragma unroll
            for (int b = 0; b < KB; ++b)
            {
                const int from = chunk_slot(16 * t + li, 4 * b + g);
                o[t] = mfma3(vs[from], vs[kPartBytes / 16 + from], ph[b], pl[b], o[t]);
            }
        }
        stage = stage == kFlashStages - 1 ? 0 : stage + 1;
    }
    wait_loads<0>();
    // The row sum over the four lanes of query li, then O = O^T / l.
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (partials != nullptr)
    {
        if (query_in)
        {
            const int heads = gridDim.y;
            float* part = partials + (((size_t) blockIdx.z * heads + head) * count + query) * (kFlashWidth + 2);
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    part[2 + 16 * t + 4 * g + r] = o[t][r];
            if (g == 0)
            {
                part[0] = m * scale2;
                part[1] = l;
            }
        }
        return;
    }
    if (query_in)
    {
        const float inv = 1.f / l;
        // A lane holds four consecutive channels of its query: one store each.
#pragma unroll
        for (int t = 0; t < 4; ++t)
        {
            const size_t at = (size_t) query * width + column + 16 * t + 4 * g;
            if constexpr (OUT == kF32)
                *reinterpret_cast<f32x4*>(out + at) = o[t] * inv;
            else
            {
                uint32_t bits[4][3];
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    cut_parts<OUT>(o[t][r] * inv, bits[r]);
#pragma unroll
                for (int p = 0; p < (OUT == kF16 ? 2 : 3); ++p)
                    *reinterpret_cast<uint2*>(out_parts + p * out_part_stride + at)
                        = uint2 {bits[0][p] | (bits[1][p] << 16), bits[2][p] | (bits[3][p] << 16)};
            }
        }
    }
}

// fp32 k and v rows as the attention's halves, where their product does not
// write them itself.
__global__ void __launch_bounds__(kColumnThreads) halves_kernel(const float* __restrict__ k,
                                                                const float* __restrict__ v, int width, int pitch,
                                                                uint16_t* __restrict__ k_halves,
                                                                uint16_t* __restrict__ vt_halves)
{
    const int row = blockIdx.x;
    const size_t part = (size_t) pitch * width;
    for (int c = threadIdx.x; c < width; c += kColumnThreads)
    {
        const float kv = k[(size_t) row * width + c], vv = v[(size_t) row * width + c];
        const size_t at = (size_t) row * width + c, vat = (size_t) c * pitch + attention_place(row);
        k_halves[at] = __builtin_bit_cast(uint16_t, half_hi(kv));
        k_halves[part + at] = __builtin_bit_cast(uint16_t, half_lo(kv));
        vt_halves[vat] = __builtin_bit_cast(uint16_t, half_hi(vv));
        vt_halves[part + vat] = __builtin_bit_cast(uint16_t, half_lo(vv));
    }
}

// The key splits of every (query, head) combined in split order, in base-2
// units: out = Σ 2^(m_s - m)·row_s / Σ 2^(m_s - m)·l_s. One 64-lane wave per
// (query, head), a lane per channel, four waves a block; the rows go out in
// fp32 or as the output product's parts, like the attention's.
template <int OUT>
__global__ void __launch_bounds__(4 * kFlashWidth) flash_combine_kernel(const float* __restrict__ partials, int count,
                                                                        int heads, int splits, int width,
                                                                        float* __restrict__ out,
                                                                        uint16_t* __restrict__ out_parts,
                                                                        size_t out_part_stride)
{
    const int query = blockIdx.x * 4 + threadIdx.x / kFlashWidth, head = blockIdx.y, c = threadIdx.x % kFlashWidth;
    if (query >= count)
        return;
    const size_t stride = (size_t) heads * count * (kFlashWidth + 2);
    const float* base = partials + ((size_t) head * count + query) * (kFlashWidth + 2);
    float largest = -INFINITY;
    for (int s = 0; s < splits; ++s)
        largest = fmaxf(largest, base[s * stride]);
    float numerator = 0.f, denominator = 0.f;
    for (int s = 0; s < splits; ++s)
    {
        const float* part = base + s * stride;
        if (part[1] == 0.f) // a split with no key
            continue;
        const float f = exp2f(part[0] - largest);
        numerator += f * part[2 + c];
        denominator += f * part[1];
    }
    const size_t at = (size_t) query * width + head * kFlashWidth + c;
    const float v = numerator / denominator;
    if constexpr (OUT == kF32)
        out[at] = v;
    else
    {
        uint32_t bits[3];
        cut_parts<OUT>(v, bits);
#pragma unroll
        for (int p = 0; p < (OUT == kF16 ? 2 : 3); ++p)
            out_parts[p * out_part_stride + at] = (uint16_t) bits[p];
    }
}

// Row p of the second convolution's columns over frame-major rows x
// [frames, channels]: x[2p + tap - 1][s] at s * 3 + tap.
__global__ void __launch_bounds__(kColumnThreads) frame_columns_kernel(const float* __restrict__ x, int channels,
                                                                       int frames, float* __restrict__ columns)
{
    const int p = blockIdx.x;
    const int inner = channels * 3;
    for (int i = threadIdx.x; i < inner; i += kColumnThreads)
    {
        const int s = i / 3, at = 2 * p + i % 3 - 1;
        columns[(size_t) p * inner + i] = at >= 0 && at < frames ? x[(size_t) at * channels + s] : 0.f;
    }
}
} // namespace
} // namespace wsp::encoder

struct wsp_encoder
{
    wsp_encoder_shape shape {};
    int device = 0;
    hipStream_t stream = nullptr;
    float* columns = nullptr; // both convolutions' gathered rows
    float* conv = nullptr;    // [conv frames, width] frame-major, or the second convolution's gathered rows
    float* hidden = nullptr;  // [positions, width]
    float* normed = nullptr;
    float* q = nullptr;
    float* k = nullptr;
    float* v = nullptr;
    float* att = nullptr;
    float* ff = nullptr;      // [positions, feed_forward_width]
    // 16-bit weights: a product's input as 16-bit parts (split_product):
    // up to three [positions, width] parts, and fc2's [positions, feed_forward_width].
    void* parts = nullptr;
    void* ff_parts = nullptr;
    // The attention's keys and values as fp16 hi and lo halves, written by the
    // q/k/v product: [2][pitch][width] and transposed [2][width][pitch], pitch
    // the positions rounded up to the key tile. Past a run's positions the keys
    // are whatever earlier runs left; the values of its last tile are zero
    // (mel_columns_kernel).
    uint16_t* k_halves = nullptr;
    uint16_t* vt_halves = nullptr;
    int pitch = 0;
    float* workspace = nullptr;
    float* flash_partials = nullptr; // [kMaxFlashSplits][heads][positions][66], split-key attention
    std::vector<void*> owned;
    char error[512] = {0};
};

namespace
{
int encoder_fail(wsp_encoder* e, int code, const char* message)
{
    std::snprintf(e->error, sizeof e->error, "%s", message);
    return code;
}

int encoder_hip(wsp_encoder* e, hipError_t status, const char* what)
{
    if (status == hipSuccess)
        return WSP_OK;
    std::snprintf(e->error, sizeof e->error, "%s: %s", what, hipGetErrorString(status));
    return WSP_ERR_HIP;
}

// The products run over pre-split inputs (split_product) for 16-bit weights
// when every product's extents and the LayerNorm's width fit them.
bool pre_split_shape(int wdtype, int d, int f)
{
    namespace ops = wsp::ops;
    return d % 8 == 0 && ops::layernorm_parts_fits(d) && ops::split_product_fits(wdtype, d, d)
           && ops::split_product_fits(wdtype, d, f) && ops::split_product_fits(wdtype, f, d);
}

hipError_t encoder_allocate(wsp_encoder* e, float** out, size_t floats)
{
    void* p = nullptr;
    const hipError_t status = hipMalloc(&p, std::max<size_t>(floats, 1) * sizeof(float));
    if (status == hipSuccess)
    {
        e->owned.push_back(p);
        *out = static_cast<float*>(p);
    }
    return status;
}
} // namespace

extern "C" {

int wsp_encoder_create(const wsp_encoder_shape* shape, int device, void* stream, wsp_encoder** out)
{
    using wsp::encoder::conv_length;
    if (shape == nullptr || out == nullptr)
        return WSP_ERR_ARGUMENT;
    *out = nullptr;
    const wsp_encoder_shape& s = *shape;
    if (s.mel_bins <= 0 || s.width <= 0 || s.heads <= 0 || s.layers < 0 || s.feed_forward_width <= 0
        || s.input_frames <= 0)
        return WSP_ERR_ARGUMENT;
    if (s.width % s.heads != 0 || (s.width / s.heads) % 4 != 0 || s.width / s.heads > wsp::ops::kMaxHeadWidth)
        return WSP_ERR_SHAPE;

    wsp_encoder* e = new (std::nothrow) wsp_encoder;
    if (e == nullptr)
        return WSP_ERR_HIP;
    e->shape = s;
    e->device = device;
    e->stream = static_cast<hipStream_t>(stream);
    const size_t frames = (size_t) conv_length(s.input_frames, 1);
    const size_t positions = (size_t) conv_length((int) frames, 2);
    const size_t d = (size_t) s.width;
    hipError_t status = hipSetDevice(device);
    if (status == hipSuccess)
        status = wsp::ops::prepare_split_products();
    if (status == hipSuccess)
        status = encoder_allocate(e, &e->columns, std::max(frames * s.mel_bins * 3, positions * d * 3));
    if (status == hipSuccess)
        status = encoder_allocate(e, &e->conv, std::max(frames, 3 * positions) * d);
    float** rows[] = {&e->hidden, &e->normed, &e->q, &e->k, &e->v, &e->att};
    for (float** r : rows)
        if (status == hipSuccess)
            status = encoder_allocate(e, r, positions * d);
    if (status == hipSuccess)
        status = encoder_allocate(e, &e->ff, positions * s.feed_forward_width);
    // Three 16-bit parts take 1.5 floats a value.
    if (status == hipSuccess)
        status = encoder_allocate(e, reinterpret_cast<float**>(&e->parts), (positions * d * 3 + 1) / 2);
    if (status == hipSuccess)
        status = encoder_allocate(e, reinterpret_cast<float**>(&e->ff_parts),
                                  (positions * s.feed_forward_width * 3 + 1) / 2);
    e->pitch = (int) ((positions + wsp::encoder::kFlashKeys - 1) / wsp::encoder::kFlashKeys
                      * wsp::encoder::kFlashKeys);
    const size_t halves = (size_t) 2 * e->pitch * d; // two parts of 16 bits
    if (status == hipSuccess)
        status = encoder_allocate(e, reinterpret_cast<float**>(&e->k_halves), halves / 2);
    if (status == hipSuccess)
        status = encoder_allocate(e, reinterpret_cast<float**>(&e->vt_halves), halves / 2);
    if (status == hipSuccess)
        status = hipMemsetAsync(e->k_halves, 0, halves * sizeof(uint16_t), e->stream);
    if (status == hipSuccess)
        status = hipMemsetAsync(e->vt_halves, 0, halves * sizeof(uint16_t), e->stream);
    if (status == hipSuccess && s.heads > 0 && s.width == s.heads * wsp::encoder::kFlashWidth)
        status = encoder_allocate(e, &e->flash_partials,
                                  (size_t) wsp::encoder::kMaxFlashSplits * s.heads * positions
                                      * (wsp::encoder::kFlashWidth + 2));
    if (status == hipSuccess)
        status = encoder_allocate(e, &e->workspace,
                                  wsp::ops::attention_workspace_floats(s.heads, (int) positions, (int) positions,
                                                                       s.width / s.heads));
    // The attention workspace's counters start at zero.
    if (status == hipSuccess)
        status = hipMemsetAsync(e->workspace, 0, wsp::ops::kAttentionCounters * sizeof(unsigned), e->stream);
    if (status == hipSuccess)
        status = hipStreamSynchronize(e->stream);
    if (status != hipSuccess)
    {
        for (void* p : e->owned)
            (void) hipFree(p);
        delete e;
        return WSP_ERR_HIP;
    }
    *out = e;
    return WSP_OK;
}

void wsp_encoder_destroy(wsp_encoder* e)
{
    if (e == nullptr)
        return;
    (void) hipSetDevice(e->device);
    (void) hipStreamSynchronize(e->stream);
    for (void* p : e->owned)
        (void) hipFree(p);
    delete e;
}

const char* wsp_encoder_last_error(const wsp_encoder* e)
{
    return e == nullptr ? "null encoder" : e->error;
}

int wsp_encoder_encode(wsp_encoder* e, const wsp_encoder_tensors* T, const float* mel, float* output,
                       int position_count)
{
    using namespace wsp::encoder;
    namespace ops = wsp::ops;
    if (e == nullptr)
        return WSP_ERR_ARGUMENT;
    e->error[0] = 0;
    if (T == nullptr || mel == nullptr || output == nullptr || (e->shape.layers > 0 && T->layers == nullptr))
        return encoder_fail(e, WSP_ERR_ARGUMENT, "wsp_encoder_encode: null tensors, mel or output");
    const wsp_encoder_shape& s = e->shape;
    const int window_positions = conv_length(conv_length(s.input_frames, 1), 2);
    if (position_count < 0 || position_count > window_positions)
        return encoder_fail(e, WSP_ERR_SHAPE, "wsp_encoder_encode: more positions than the window holds");
    if (T->wdtype != WSP_F32 && T->wdtype != WSP_F16 && T->wdtype != WSP_BF16)
        return encoder_fail(e, WSP_ERR_LOGIC, "wsp_encoder_encode: unknown projection storage");
    const int frames = position_count == 0 ? s.input_frames : std::min(2 * position_count, s.input_frames);
    const int conv_frames = conv_length(frames, 1);
    const int positions = conv_length(conv_frames, 2);
    const int d = s.width, f = s.feed_forward_width, heads = s.heads;
    const float scale = 1.f / std::sqrt((float) (d / heads));
    const float eps = 1e-5f;
    hipStream_t st = e->stream;
    (void) hipSetDevice(e->device);
    hipError_t status;

    // Stored projection scales (powers of two in [2^-126, 2^126], so their
    // reciprocals are normal floats; 0 reads as 1) and whether any
    // projection carries one: those take the pre-split products at every
    // position count, the only products that divide a scale out.
    bool scaled = false;
    for (int l = 0; l < s.layers; ++l)
    {
        const wsp_encoder_layer_tensors& L = T->layers[l];
        for (const float c : {L.q_scale, L.k_scale, L.v_scale, L.out_scale, L.fc1_scale, L.fc2_scale})
        {
            int exponent = 0;
            if (c != 0.f && !(std::isfinite(c) && c > 0.f && std::frexp(c, &exponent) == 0.5f && exponent >= -125
                               && exponent <= 127))
                return encoder_fail(e, WSP_ERR_ARGUMENT,
                                    "wsp_encoder_encode: a projection scale is not a power of two in [2^-126, 2^126]");
            scaled = scaled || (c != 0.f && c != 1.f);
        }
    }
    if (scaled && !pre_split_shape(T->wdtype, d, f))
        return encoder_fail(e, WSP_ERR_SHAPE,
                            "wsp_encoder_encode: scaled projections need 16-bit storage and the pre-split products' "
                            "shapes");
    const bool flash = d / heads == kFlashWidth;
    static_assert(kFlashKeys == 4 * kClearedQuads, "the key tile's values are cleared");
    const int clearing = flash ? (2 * d * kClearedQuads + kColumnThreads - 1) / kColumnThreads : 0;
    hipLaunchKernelGGL(mel_columns_kernel, dim3(clearing + conv_frames), dim3(kColumnThreads), 0, st, mel, s.mel_bins,
                       s.input_frames, frames, e->columns, clearing, positions, d, e->pitch, e->vt_halves);
    if ((status = hipGetLastError()) != hipSuccess)
        return encoder_hip(e, status, "conv1 columns");
    // Both convolutions as direct-to-LDS fp32 products where they fit and give
    // each CU a tile: the first writes the second's columns itself, and the
    // second adds to the positional table's rows.
    auto convolution = [&](const float* x, int rows, int inner, const float* w, const float* bias, float* y, int flags) {
        ops::SplitProduct p {};
        p.parts = x;
        p.rows = rows;
        p.inner = inner;
        p.count = 1;
        p.columns = d;
        p.matrix[0] = {w, bias, y, 1.f};
        p.ldy = d;
        p.flags = flags;
        p.wdtype = WSP_F32;
        return p;
    };
    auto tiles = [&](int rows) { return (rows + 31) / 32 * ((d + 31) / 32); };
    ops::SplitProduct conv1 = convolution(e->columns, conv_frames, 3 * s.mel_bins, T->conv1_w, T->conv1_b, e->conv,
                                          ops::kProductGelu | ops::kProductTaps);
    conv1.taps = positions;
    ops::SplitProduct conv2 = convolution(e->conv, positions, 3 * d, T->conv2_w, T->conv2_b, e->hidden,
                                          ops::kProductGelu | ops::kProductResidual);
    conv2.residual = T->positions;
    if (tiles(positions) >= ops::compute_units() && ops::fp32_split_fits(conv1) && ops::fp32_split_fits(conv2))
    {
        if ((status = ops::fp32_split(st, conv1)) != hipSuccess)
            return encoder_hip(e, status, "conv1");
        if ((status = ops::fp32_split(st, conv2)) != hipSuccess)
            return encoder_hip(e, status, "conv2");
    }
    else
    {
        if ((status = ops::linear(st, e->columns, conv_frames, 3 * s.mel_bins, T->conv1_w, WSP_F32, T->conv1_b,
                                  e->conv, d, 1)) != hipSuccess)
            return encoder_hip(e, status, "conv1");
        hipLaunchKernelGGL(frame_columns_kernel, dim3(positions), dim3(kColumnThreads), 0, st, e->conv, d, conv_frames,
                           e->columns);
        if ((status = hipGetLastError()) != hipSuccess)
            return encoder_hip(e, status, "conv2 columns");
        // h = gelu(conv2) + embed_positions: the rows start as the positional
        // table's first rows and the product adds to them (bias, GELU, residual).
        if ((status = hipMemcpyAsync(e->hidden, T->positions, (size_t) positions * d * sizeof(float),
                                     hipMemcpyDeviceToDevice, st)) != hipSuccess)
            return encoder_hip(e, status, "positional rows");
        if ((status = ops::linear(st, e->columns, positions, 3 * d, T->conv2_w, WSP_F32, T->conv2_b, e->hidden, d, 3))
            != hipSuccess)
            return encoder_hip(e, status, "conv2");
    }

    const int wt = T->wdtype;
    auto unscale = [](float c) { return c == 0.f ? 1.f : 1.f / c; };
    // 16-bit weights take the products over pre-split inputs: each product's
    // input is stored once as its 16-bit parts (fc1 writes fc2's itself):
    // three exact bf16 parts, or fp16 hi + lo for fp16 and scaled weights.
    const size_t part_stride = (size_t) positions * d, ff_part_stride = (size_t) positions * f;
    const bool split = (positions > 16 || scaled) && part_stride % 8 == 0 && pre_split_shape(wt, d, f);
    auto split_product = [&](const void* parts, size_t stride, int inner, const void* w, const float* bias, float* y,
                             int out, int flags, void* out_parts, float stored_scale) {
        ops::SplitProduct p {};
        p.parts = parts;
        p.part_stride = stride;
        p.rows = positions;
        p.inner = inner;
        p.count = 1;
        p.columns = out;
        p.matrix[0] = {w, bias, y, unscale(stored_scale)};
        p.ldy = out;
        p.flags = flags;
        p.out_parts = out_parts;
        p.out_part_stride = ff_part_stride;
        p.wdtype = wt;
        return ops::split_product(st, p);
    };
    // q, k and v of an fp32 layer side by side, k and v as the attention's halves.
    auto fp32_projections = [&](const wsp_encoder_layer_tensors& L, bool as_halves) {
        ops::SplitProduct p {};
        p.parts = e->normed;
        p.rows = positions;
        p.inner = d;
        p.count = 3;
        p.columns = d;
        p.matrix[0] = {L.q_w, L.q_b, e->q, 1.f};
        p.matrix[1] = {L.k_w, nullptr, e->k, 1.f};
        p.matrix[2] = {L.v_w, L.v_b, e->v, 1.f};
        p.ldy = d;
        p.wdtype = WSP_F32;
        if (as_halves)
        {
            p.y1_halves = e->k_halves;
            p.y2_halves_t = e->vt_halves;
            p.halves_pitch = e->pitch;
        }
        return p;
    };
    // (Products that do not run over stored parts may store them there themselves.)
    const size_t window_rows = (size_t) window_positions;
    const ops::Scratch scratch {e->ff_parts, ops::parts_bytes(window_rows * f)};
    for (int l = 0; l < s.layers; ++l)
    {
        const wsp_encoder_layer_tensors& L = T->layers[l];
        bool halves = false; // the projections left k and v as the attention's halves
        status = split ? ops::layernorm_parts(st, e->hidden, L.attention_norm_w, L.attention_norm_b, e->parts,
                                              part_stride, positions, d, eps, wt)
                       : ops::layernorm(st, e->hidden, L.attention_norm_w, L.attention_norm_b, e->normed, positions,
                                        d, eps);
        if (status != hipSuccess)
            return encoder_hip(e, status, "self-attention norm");
        if (split)
        {
            // q, k and v side by side in one launch.
            ops::SplitProduct p {};
            p.parts = e->parts;
            p.part_stride = part_stride;
            p.rows = positions;
            p.inner = d;
            p.count = 3;
            p.columns = d;
            p.matrix[0] = {L.q_w, L.q_b, e->q, unscale(L.q_scale)};
            p.matrix[1] = {L.k_w, nullptr, e->k, unscale(L.k_scale)};
            p.matrix[2] = {L.v_w, L.v_b, e->v, unscale(L.v_scale)};
            p.ldy = d;
            p.wdtype = wt;
            if (flash)
            {
                // The attention takes k and v as fp16 halves.
                p.y1_halves = e->k_halves;
                p.y2_halves_t = e->vt_halves;
                p.halves_pitch = e->pitch;
                halves = true;
            }
            status = ops::split_product(st, p);
        }
        else if (const ops::SplitProduct three = fp32_projections(L, flash);
                 wt == WSP_F32 && positions > 16 && ops::fp32_split_fits(three))
        {
            halves = flash;
            status = ops::fp32_split(st, three);
        }
        else
        {
            // q, k and v side by side in one launch: three times the blocks of one.
            const ops::ProductMatrix matrices[] = {{L.q_w, L.q_b, e->q, 1.f},
                                                   {L.k_w, nullptr, e->k, 1.f},
                                                   {L.v_w, L.v_b, e->v, 1.f}};
            ops::Products p {};
            p.x = e->normed;
            p.rows = positions;
            p.inner = d;
            p.matrices = matrices;
            p.count = 3;
            p.columns = d;
            p.ldy = d;
            p.wdtype = wt;
            status = ops::products(st, p, scratch);
        }
        if (status != hipSuccess)
            return encoder_hip(e, status, "self-attention projections");
        if (flash)
        {
            if (!halves)
            {
                hipLaunchKernelGGL(halves_kernel, dim3(positions), dim3(kColumnThreads), 0, st, e->k, e->v, d,
                                   e->pitch, e->k_halves, e->vt_halves);
                if ((status = hipGetLastError()) != hipSuccess)
                    return encoder_hip(e, status, "self-attention keys and values");
            }
            // 128 queries a block share each K/V tile when that still leaves
            // at most an eighth of the CUs idle (large-v3: 240 blocks,
            // 14.2 -> 13.4 ms a window); else 64 (tiny.en's 72 blocks of 128
            // queries measured slower than 144 of 64).
            const int wide_blocks = (positions + 16 * kFlashWideWaves - 1) / (16 * kFlashWideWaves) * heads;
            const float scale2 = scale * 1.44269504088896340736f;
            // Fewer 64-query blocks than CUs (tiny.en: 144): the keys are
            // split over up to four blocks per query tile, at least 64 keys
            // each, and the splits combined after.
            const int narrow_blocks = (positions + 16 * kFlashWaves - 1) / (16 * kFlashWaves) * heads;
            int splits = 1;
            if (narrow_blocks < ops::compute_units() && e->flash_partials != nullptr)
                splits = std::max(1, std::min({kMaxFlashSplits, (ops::compute_units() + narrow_blocks - 1) / narrow_blocks,
                                               positions / 64}));
            const int span = ((positions + splits - 1) / splits + kFlashKeys - 1) / kFlashKeys * kFlashKeys;
            float* partials = splits > 1 ? e->flash_partials : nullptr;
            const bool wide = 8 * wide_blocks >= 7 * ops::compute_units();
            const dim3 grid = wide ? dim3((positions + 16 * kFlashWideWaves - 1) / (16 * kFlashWideWaves), heads)
                                   : dim3((positions + 16 * kFlashWaves - 1) / (16 * kFlashWaves), heads, splits);
            const int key_span = wide ? positions : span;
            // With the pre-split products the rows (or their combination) go
            // out as the output product's input parts.
            uint16_t* const out_parts = static_cast<uint16_t*>(e->parts);
            auto launch = [&](auto kernel, int waves) {
                hipLaunchKernelGGL(kernel, grid, dim3(64 * waves), 0, st, e->q, positions, d, scale2, e->att, key_span,
                                   wide ? nullptr : partials, e->k_halves, e->vt_halves, e->pitch, out_parts,
                                   part_stride);
            };
            auto combine = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3((positions + 3) / 4, heads), dim3(4 * kFlashWidth), 0, st,
                                   e->flash_partials, positions, heads, splits, d, e->att, out_parts, part_stride);
            };
            auto attend = [&](auto wide_kernel, auto narrow_kernel, auto combine_kernel) {
                if (wide)
                    launch(wide_kernel, kFlashWideWaves);
                else
                    launch(narrow_kernel, kFlashWaves);
                if (!wide && splits > 1)
                    combine(combine_kernel);
            };
            if (!split)
                attend(flash_attention_kernel<kFlashWideWaves, wsp::kF32>, flash_attention_kernel<kFlashWaves, wsp::kF32>,
                       flash_combine_kernel<wsp::kF32>);
            else if (wt == WSP_F16)
                attend(flash_attention_kernel<kFlashWideWaves, wsp::kF16>, flash_attention_kernel<kFlashWaves, wsp::kF16>,
                       flash_combine_kernel<wsp::kF16>);
            else
                attend(flash_attention_kernel<kFlashWideWaves, wsp::kBF16>,
                       flash_attention_kernel<kFlashWaves, wsp::kBF16>, flash_combine_kernel<wsp::kBF16>);
            status = hipGetLastError();
        }
        else
            status = ops::attention(st, e->q, positions, e->k, e->v, positions, d, heads, 0, scale, e->att,
                                    e->workspace);
        if (status != hipSuccess)
            return encoder_hip(e, status, "self attention");
        if (split)
        {
            if (flash || (status = ops::split_rows(st, e->att, part_stride, wt, e->parts, part_stride))
                                 == hipSuccess)
                status = split_product(e->parts, part_stride, d, L.out_w, L.out_b, e->hidden, d,
                                       ops::kProductResidual, nullptr, L.out_scale);
        }
        else
            status = ops::linear(st, e->att, positions, d, L.out_w, wt, L.out_b, e->hidden, d, 2, scratch);
        if (status != hipSuccess)
            return encoder_hip(e, status, "attention output");
        status = split ? ops::layernorm_parts(st, e->hidden, L.final_norm_w, L.final_norm_b, e->parts, part_stride,
                                              positions, d, eps, wt)
                       : ops::layernorm(st, e->hidden, L.final_norm_w, L.final_norm_b, e->normed, positions, d, eps);
        if (status != hipSuccess)
            return encoder_hip(e, status, "feed-forward norm");
        if (split)
        {
            if ((status = split_product(e->parts, part_stride, d, L.fc1_w, L.fc1_b, nullptr, f, ops::kProductGelu,
                                        e->ff_parts, L.fc1_scale))
                == hipSuccess)
                status = split_product(e->ff_parts, ff_part_stride, f, L.fc2_w, L.fc2_b, e->hidden, d,
                                       ops::kProductResidual, nullptr, L.fc2_scale);
        }
        else if ((status = ops::linear(st, e->normed, positions, d, L.fc1_w, wt, L.fc1_b, e->ff, f, 1, scratch)) == hipSuccess)
            status = ops::linear(st, e->ff, positions, f, L.fc2_w, wt, L.fc2_b, e->hidden, d, 2, scratch);
        if (status != hipSuccess)
            return encoder_hip(e, status, "feed-forward");
    }
    if ((status = ops::layernorm(st, e->hidden, T->final_norm_w, T->final_norm_b, output, positions, d, eps))
        != hipSuccess)
        return encoder_hip(e, status, "final norm");
    return WSP_OK;
}

int wsp_encoder_scaled_halves(const wsp_encoder_shape* shape, const void* bf16, size_t count, void* halves,
                              float* scale)
{
    if (shape == nullptr || scale == nullptr || (count > 0 && (bf16 == nullptr || halves == nullptr)))
        return WSP_ERR_ARGUMENT;
    if (!pre_split_shape(WSP_F16, shape->width, shape->feed_forward_width))
        return WSP_ERR_SHAPE;
    const uint16_t* in = static_cast<const uint16_t*>(bf16);
    uint16_t* out = static_cast<uint16_t*>(halves);
    auto widen = [](uint16_t bits) { return __builtin_bit_cast(float, (uint32_t) bits << 16); };
    // The shift puts the largest magnitude's binade at 2^15 (fp16's top one:
    // an 8-bit significand there is at most 65280 < 65504).
    int top = INT_MIN;
    for (size_t i = 0; i < count; ++i)
    {
        const float v = widen(in[i]);
        if (!std::isfinite(v))
            return WSP_ERR_LOGIC;
        if (v != 0.f)
            top = std::max(top, std::ilogb(v));
    }
    // (At most 126, so the scale stays a finite float and its reciprocal a normal one.)
    const int shift = top == INT_MIN ? 0 : std::min(15 - top, 126);
    for (size_t i = 0; i < count; ++i)
    {
        const float v = widen(in[i]);
        const _Float16 h = (_Float16) std::ldexp(v, shift);
        if (__builtin_bit_cast(uint32_t, std::ldexp((float) h, -shift)) != __builtin_bit_cast(uint32_t, v))
            return WSP_ERR_LOGIC;
        out[i] = __builtin_bit_cast(uint16_t, h);
    }
    *scale = std::ldexp(1.f, shift);
    return WSP_OK;
}

} // extern "C"
