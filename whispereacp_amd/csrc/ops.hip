// Per-op gfx950 kernels behind the C ABI: the split GEMV (Kernels/Linear.h;
// linear_product.hip has the products of more rows), LayerNorm (Kernels/LayerNorm.h), Embed
// (Kernels/Embed.h), split-key attention with its combine
// (Kernels/SingleQueryAttention.h, Kernels/Attention.h) and the two-stage
// argmax (Kernels/Argmax.h). Written for wave64 CDNA4; every reduction runs in
// a fixed order, so results are deterministic run to run.
#include "device_common.h"
#include "ops.h"

#include <algorithm>
#include <cmath>

namespace wsp::ops
{
namespace
{
constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kWave;

// ---------------------------------------------------------------------------
// Split GEMV: each wave owns OPW output columns for up to RMAX rows. Lane l
// walks the inner dimension in runs of 8 (one 16-byte weight load for F16 and
// BF16, two for F32) at k = 8l, 8l + 512, ...; the 64 lane partials are then
// summed by a fixed xor-butterfly. The epilogue is the reference's store
// (Kernels/Linear.h:213-227): bias, then GELU, then the residual.
// ---------------------------------------------------------------------------
template <int WT, int RMAX, int OPW>
__global__ void __launch_bounds__(kBlock) gemv_kernel(const float* __restrict__ x, int rows,
                                                      int inner, const void* __restrict__ w,
                                                      const float* __restrict__ bias,
                                                      float* __restrict__ y, int out, int flags,
                                                      int vectorised)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
    const int o0 = wave * OPW;

    if (o0 >= out)
        return;

    float acc[RMAX][OPW];
#pragma unroll
    for (int r = 0; r < RMAX; ++r)
#pragma unroll
        for (int j = 0; j < OPW; ++j)
            acc[r][j] = 0.f;

    if (vectorised)
    {
        for (int k = lane * 8; k < inner; k += kWave * 8)
        {
            float wv[OPW][8];
#pragma unroll
            for (int j = 0; j < OPW; ++j)
            {
                const int o = min(o0 + j, out - 1);
                load8<WT>(w, (size_t) o * inner + k, wv[j]);
            }
#pragma unroll
            for (int r = 0; r < RMAX; ++r)
            {
                if (r >= rows)
                    break;
                const float4v* xp = reinterpret_cast<const float4v*>(x + (size_t) r * inner + k);
                const float4v a = xp[0], b = xp[1];
                const float xv[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
#pragma unroll
                for (int j = 0; j < OPW; ++j)
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        acc[r][j] += xv[i] * wv[j][i];
            }
        }
    }
    else
    {
        for (int k = lane; k < inner; k += kWave)
        {
            float wv[OPW];
#pragma unroll
            for (int j = 0; j < OPW; ++j)
                wv[j] = load1<WT>(w, (size_t) min(o0 + j, out - 1) * inner + k);
#pragma unroll
            for (int r = 0; r < RMAX; ++r)
            {
                if (r >= rows)
                    break;
                const float xv = x[(size_t) r * inner + k];
#pragma unroll
                for (int j = 0; j < OPW; ++j)
                    acc[r][j] += xv * wv[j];
            }
        }
    }

#pragma unroll
    for (int r = 0; r < RMAX; ++r)
#pragma unroll
        for (int j = 0; j < OPW; ++j)
            acc[r][j] = wave_sum(acc[r][j]);

#pragma unroll
    for (int r = 0; r < RMAX; ++r)
#pragma unroll
        for (int j = 0; j < OPW; ++j)
        {
            const int o = o0 + j;
            if (r < rows && o < out && lane == ((r * OPW + j) & (kWave - 1)))
            {
                float v = acc[r][j] + (bias != nullptr ? bias[o] : 0.f);
                if (flags & 1)
                    v = exact_gelu(v);
                float* dst = y + (size_t) r * out + o;
                if (flags & 2)
                    v += *dst;
                *dst = v;
            }
        }
}

// ---------------------------------------------------------------------------
// LayerNorm: one block per row; mean, then the centred variance, then
// (x - mean) * rsqrt(var + eps) * gamma + beta (Kernels/LayerNorm.h:44-89).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(kBlock) layernorm_kernel(const float* __restrict__ x,
                                                           const float* __restrict__ gamma,
                                                           const float* __restrict__ beta,
                                                           float* __restrict__ y, int width,
                                                           float eps)
{
    __shared__ float scratch[kWavesPerBlock];
    const float* row = x + (size_t) blockIdx.x * width;
    float* dst = y + (size_t) blockIdx.x * width;

    float total = 0.f;
    for (int c = threadIdx.x; c < width; c += kBlock)
        total += row[c];
    const float mean = block_sum(total, scratch) / (float) width;

    float squares = 0.f;
    for (int c = threadIdx.x; c < width; c += kBlock)
    {
        const float centred = row[c] - mean;
        squares += centred * centred;
    }
    const float scale = rsqrtf(block_sum(squares, scratch) / (float) width + eps);

    for (int c = threadIdx.x; c < width; c += kBlock)
        dst[c] = (row[c] - mean) * scale * gamma[c] + beta[c];
}

// A wave for each row of up to 256·RUNS floats in whole 16-byte runs
// (normalise_row); other rows take layernorm_kernel.
template <int RUNS>
__global__ void __launch_bounds__(kWave) layernorm_row_kernel(const float* __restrict__ x,
                                                              const float* __restrict__ gamma,
                                                              const float* __restrict__ beta, float* __restrict__ y,
                                                              int width, float eps)
{
    const size_t row = (size_t) blockIdx.x * width;
    float4v v[RUNS];
    normalise_row<RUNS>(x + row, gamma, beta, width, eps, v);
#pragma unroll
    for (int i = 0; i < RUNS; ++i)
    {
        const int at = 4 * ((int) threadIdx.x + kWave * i);
        if (at < width)
            *reinterpret_cast<float4v*>(y + row + at) = v[i];
    }
}

// ---------------------------------------------------------------------------
// Embed: out[t, c] = tokens table row + position table row (Kernels/Embed.h).
// ---------------------------------------------------------------------------
// A token id outside the vocabulary (it arrives from device memory, so the host
// cannot check it) poisons its row with NaN rather than reading past the table.
__global__ void embed_kernel(const uint32_t* __restrict__ tokens,
                             const float* __restrict__ token_table,
                             const float* __restrict__ position_table, int first_position,
                             float* __restrict__ y, int width, int vocabulary)
{
    const int t = blockIdx.y;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= width)
        return;
    const uint32_t token = tokens[t];
    y[(size_t) t * width + c] = token < (uint32_t) vocabulary
                                    ? token_table[(size_t) token * width + c]
                                          + position_table[(size_t) (first_position + t) * width + c]
                                    : __builtin_nanf("");
}

// ---------------------------------------------------------------------------
// Split-key attention. Block (head h, query i, chunk c) scores its chunk of
// the keys query i can see (the last q_count of k_count positions when
// causal, Kernels/Attention.h:34-47), takes the chunk maximum, exponentiates
// and sums, and walks the value rows. One chunk writes the normalised row;
// several write (max, sum, unnormalised row) for the combine, which rescales
// each chunk by exp(max_c - max) exactly as Kernels/SingleQueryAttention.h
// :27-37 describes.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(kBlock) attention_chunk_kernel(
    const float* __restrict__ q, int q_count, const float* __restrict__ keys,
    const float* __restrict__ values, int k_count, int width, int head_width, int causal,
    float scale, int chunks, int chunk_length, float* __restrict__ out,
    float* __restrict__ partials)
{
    __shared__ float scores[kAttentionChunkKeys];
    __shared__ float scratch[kWavesPerBlock];
    __shared__ float rows_sum[4][kMaxHeadWidth];

    const int chunk = blockIdx.x % chunks;
    const int query = (blockIdx.x / chunks) % q_count;
    const int head = blockIdx.x / (chunks * q_count);
    const int column = head * head_width;

    const int visible = causal ? k_count - q_count + query + 1 : k_count;
    const int first = chunk * chunk_length;
    const int last = min(first + chunk_length, visible);
    const int count = max(0, last - first);

    // Scores: 16 lanes per key, each lane a run of four channels.
    const int sub = threadIdx.x % 16, group = threadIdx.x / 16;
    const float* qrow = q + (size_t) query * width + column;
    float4v qv = {0.f, 0.f, 0.f, 0.f};
    if (4 * sub < head_width)
        qv = *reinterpret_cast<const float4u*>(qrow + 4 * sub);

    float local_max = -INFINITY;
    for (int j = group; j < count; j += 16)
    {
        float part = 0.f;
        if (4 * sub < head_width)
        {
            const float4v kv =
                *reinterpret_cast<const float4u*>(keys + (size_t) (first + j) * width + column + 4 * sub);
            part = qv[0] * kv[0] + qv[1] * kv[1] + qv[2] * kv[2] + qv[3] * kv[3];
        }
#pragma unroll
        for (int offset = 8; offset > 0; offset >>= 1)
            part += __shfl_xor(part, offset, 16);
        const float s = scale * part;
        if (sub == 0)
            scores[j] = s;
        local_max = fmaxf(local_max, s);
    }
    const float chunk_max = block_max(local_max, scratch);

    float local_sum = 0.f;
    for (int j = threadIdx.x; j < count; j += kBlock)
    {
        const float p = expf(scores[j] - chunk_max);
        scores[j] = p;
        local_sum += p;
    }
    const float chunk_sum = block_sum(local_sum, scratch);

    // Values: channel c = t % 64, keys j = t / 64 (mod 4).
    const int c = threadIdx.x % kMaxHeadWidth, kg = threadIdx.x / kMaxHeadWidth;
    float acc = 0.f;
    if (c < head_width)
        for (int j = kg; j < count; j += 4)
            acc += scores[j] * values[(size_t) (first + j) * width + column + c];
    rows_sum[kg][c] = acc;
    __syncthreads();

    if (threadIdx.x < head_width)
    {
        const float row = (rows_sum[0][c] + rows_sum[1][c]) + (rows_sum[2][c] + rows_sum[3][c]);
        if (chunks == 1)
            out[(size_t) query * width + column + c] = row / chunk_sum;
        else
        {
            float* part = partials + ((size_t) (head * q_count + query) * chunks + chunk) * (head_width + 2);
            part[2 + c] = row;
            if (c == 0)
            {
                part[0] = count > 0 ? chunk_max : -INFINITY;
                part[1] = chunk_sum;
            }
        }
    }
}

// A wave for each fourth chunk, AHEAD chunks' loads in flight: walking them one
// after the other cost 18 us for 32 chunks of eight heads. (As many as there are
// four or eight: the loads of eight cost two chunks of 12 heads 0.4 us of 7.5.)
template <int AHEAD>
__global__ void __launch_bounds__(kBlock) attention_combine_kernel(const float* __restrict__ partials, int q_count,
                                                                   int width, int head_width, int chunks,
                                                                   float* __restrict__ out)
{
    __shared__ float sums[kWavesPerBlock][2][kMaxHeadWidth];
    const int query = blockIdx.x % q_count;
    const int head = blockIdx.x / q_count;
    const int c = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int pitch = head_width + 2;
    const float* base = partials + (size_t) (head * q_count + query) * chunks * pitch;

    float largest = -INFINITY;
    for (int k = c; k < chunks; k += kWave)
        largest = fmaxf(largest, base[(size_t) k * pitch]);
    largest = wave_max(largest);

    float numerator = 0.f, denominator = 0.f;
    for (int k0 = wave; k0 < chunks; k0 += AHEAD * kWavesPerBlock)
    {
        float top[AHEAD], sum[AHEAD], row[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
        {
            const float* part = base + (size_t) min(k0 + i * kWavesPerBlock, chunks - 1) * pitch;
            top[i] = part[0];
            sum[i] = part[1];
            row[i] = part[2 + min(c, head_width - 1)];
        }
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
            if (k0 + i * kWavesPerBlock < chunks && sum[i] != 0.f) // (a chunk with no visible key sums to zero)
            {
                const float factor = expf(top[i] - largest);
                numerator += factor * row[i];
                denominator += factor * sum[i];
            }
    }
    sums[wave][0][c] = numerator;
    sums[wave][1][c] = denominator;
    __syncthreads();
    if (threadIdx.x < head_width)
    {
        float n = 0.f, d = 0.f;
#pragma unroll
        for (int w = 0; w < kWavesPerBlock; ++w)
        {
            n += sums[w][0][c];
            d += sums[w][1][c];
        }
        out[(size_t) query * width + head * head_width + c] = n / d;
    }
}

// ---------------------------------------------------------------------------
// Attention of two and more queries with heads of 64 channels, in fp32 on the
// matrix cores (v_mfma_f32_16x16x4_f32), with the causal rule of
// Kernels/Attention.h:34-47. Block (head, 16·QT queries, key split): its eight
// waves take 32 keys at a time each, straight from memory into operand
// registers (no barrier in the loop), every key serving all the block's
// queries, and keep an online (max, sum, row) per query; the waves are merged
// in order through LDS at the end.
//
// S^T = K·Q^T leaves lane (li, g) with keys 4g + r of query li, which is the
// operand of O^T = V^T·P^T as it stands: product r takes key 4g + r from lane
// group g, and V's float4 of channels 4li .. 4li + 3 feeds the four products
// of channels 4·row + t. 96 queries over 1500 keys of 12 heads: 160 us as one
// block per (query, head, chunk) of vector code, 17 here. Bound by the
// K and V reads of each query tile from the L2s and, at these sizes, by the
// chain load, score, softmax, merge. The rows may start at any float (the loads
// are 16 bytes wide all the same).
// ---------------------------------------------------------------------------
constexpr int kQueryWaves = 8;
constexpr int kQueryKeys = 32; // keys a wave takes at a time

template <int QT>
__global__ void __launch_bounds__(kQueryWaves * kWave) query_attention_kernel(
    const float* __restrict__ q, int q_count, const float* __restrict__ keys, const float* __restrict__ values,
    int k_count, int width, int causal, float scale, int splits, int span, int first_tile, float* __restrict__ out,
    float* __restrict__ partials)
{
    __shared__ float tops[kQueryWaves][QT][16], totals[kQueryWaves][QT][16];
    __shared__ float4v rows[kQueryWaves][16][16]; // [wave][query][channel run of four]

    const int split = blockIdx.x % splits, head = blockIdx.x / splits;
    const int first_query = (first_tile + (int) blockIdx.y) * 16 * QT;
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave, li = lane % 16, g = lane / 16;
    const int column = head * 64;
    const int past = k_count - q_count; // causal: query i sees keys 0 .. past + i
    const int last_seen = causal ? past + min(first_query + 16 * QT, q_count) - 1 : k_count - 1;
    const int end = min(min(split * span + span, k_count), last_seen + 1);

    float4v qf[QT][4], o[QT][4];
    float m[QT], l[QT];
#pragma unroll
    for (int t = 0; t < QT; ++t)
    {
        const float* row = q + (size_t) min(first_query + 16 * t + li, q_count - 1) * width + column + 4 * g;
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            qf[t][j] = *reinterpret_cast<const float4u*>(row + 16 * j);
            o[t][j] = float4v {0.f, 0.f, 0.f, 0.f};
        }
        m[t] = -INFINITY;
        l[t] = 0.f;
    }
    for (int k0 = split * span + kQueryKeys * wave; k0 < end; k0 += kQueryKeys * kQueryWaves)
    {
        float4v kf[2][4], vf[2][4];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                const int key = min(k0 + 16 * b + li, end - 1);
                kf[b][j] = *reinterpret_cast<const float4u*>(keys + (size_t) key * width + column + 16 * j + 4 * g);
            }
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
                const int key = min(k0 + 16 * b + 4 * g + r, end - 1);
                vf[b][r] = *reinterpret_cast<const float4u*>(values + (size_t) key * width + column + 4 * li);
            }
        bool hidden_odd = false;
#pragma unroll
        for (int t = 0; t < QT; ++t)
        {
            // Four partial sums a score, added in pairs: chains of four roundings
            // instead of sixteen, and products that need not wait for each other.
            float4v part[2][4], s[2];
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int b = 0; b < 2; ++b)
                        part[b][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            kf[b][j][e], qf[t][j][e], e == 0 ? float4v {0.f, 0.f, 0.f, 0.f} : part[b][j], 0, 0, 0);
#pragma unroll
            for (int b = 0; b < 2; ++b)
                s[b] = (part[b][0] + part[b][1]) + (part[b][2] + part[b][3]);
            const int seen = causal ? min(end, past + first_query + 16 * t + li + 1) : end; // keys before this one
            float top = -INFINITY;
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                {
                    s[b][r] = k0 + 16 * b + 4 * g + r < seen ? scale * s[b][r] : -INFINITY;
                    top = fmaxf(top, s[b][r]);
                }
            top = fmaxf(top, __shfl_xor(top, 16));
            top = fmaxf(top, __shfl_xor(top, 32));
            const float m_new = fmaxf(m[t], top);
            const float alpha = m_new == -INFINITY ? 1.f : expf(m[t] - m_new);
            float own = 0.f;
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                {
                    s[b][r] = k0 + 16 * b + 4 * g + r < seen ? expf(s[b][r] - m_new) : 0.f;
                    own += s[b][r];
                }
            l[t] = l[t] * alpha + own;
            m[t] = m_new;
#pragma unroll
            for (int c = 0; c < 4; ++c)
                o[t][c] *= alpha;
            // Keys that some of these queries do not see, and the last key again in
            // place of those past the end (the last lane group's last key is that
            // one), get weight zero in the products, which hides a value only while
            // it is finite. (Without the causal rule a look at every value cost a
            // launch 0.5 us.)
            if (t == 0 && causal && k0 + kQueryKeys > past + first_query + 1)
            {
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int c = 0; c < 4; ++c)
                            hidden_odd = hidden_odd || !isfinite(vf[b][r][c]);
                hidden_odd = __any(hidden_odd);
            }
            else if (t == 0 && k0 + kQueryKeys > end)
            {
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    hidden_odd = hidden_odd || !isfinite(vf[1][3][c]);
                hidden_odd = __any(hidden_odd);
            }
            if (hidden_odd) // each query's own keys alone
            {
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        for (int from = 0; from < 4; ++from)
                        {
                            const float weight = __shfl(s[b][r], li + 16 * from);
                            const int key = k0 + 16 * b + 4 * from + r;
                            if (key >= seen)
                                continue;
                            const float* row = values + (size_t) key * width + column;
#pragma unroll
                            for (int c = 0; c < 4; ++c)
#pragma unroll
                                for (int i = 0; i < 4; ++i)
                                    o[t][c][i] += weight * row[4 * (4 * g + i) + c];
                        }
                continue;
            }
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        o[t][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[b][r][c], s[b][r], o[t][c], 0, 0, 0);
        }
    }
#pragma unroll
    for (int t = 0; t < QT; ++t)
    {
        l[t] += __shfl_xor(l[t], 16);
        l[t] += __shfl_xor(l[t], 32);
        if (g == 0)
        {
            tops[wave][t][li] = m[t];
            totals[wave][t][li] = l[t];
        }
    }
#pragma unroll
    for (int t = 0; t < QT; ++t)
    {
        // o[t][c][r] is channel 4 (4g + r) + c of query li.
#pragma unroll
        for (int r = 0; r < 4; ++r)
            rows[wave][li][4 * g + r] = float4v {o[t][0][r], o[t][1][r], o[t][2][r], o[t][3][r]};
        __syncthreads();
        for (int i = threadIdx.x; i < 16 * 64; i += kQueryWaves * kWave)
        {
            const int at = i / 64, c = i % 64, query = first_query + 16 * t + at;
            float largest = -INFINITY;
#pragma unroll
            for (int w = 0; w < kQueryWaves; ++w)
                largest = fmaxf(largest, tops[w][t][at]);
            float numerator = 0.f, denominator = 0.f;
#pragma unroll
            for (int w = 0; w < kQueryWaves; ++w)
                if (totals[w][t][at] != 0.f) // (a wave with no visible key)
                {
                    const float factor = expf(tops[w][t][at] - largest);
                    numerator += factor * reinterpret_cast<const float*>(&rows[w][at][c / 4])[c % 4];
                    denominator += factor * totals[w][t][at];
                }
            if (query >= q_count)
                continue;
            if (splits == 1)
                out[(size_t) query * width + column + c] = numerator / denominator;
            else
            {
                float* part = partials + ((size_t) (head * q_count + query) * splits + split) * (64 + 2);
                part[2 + c] = numerator;
                if (c == 0)
                {
                    part[0] = largest;
                    part[1] = denominator;
                }
            }
        }
        __syncthreads(); // (the rows are written again for the next queries)
    }
}

// ---------------------------------------------------------------------------
// Multi-query attention of a prompt step (2..16 queries): the scores, the
// softmax and the weighted value sum of Kernels/Attention.h:75-209, with its
// causal rule (query i of q stands at absolute position k - q + i and sees the
// keys up to it, Kernels/Attention.h:34-47), in one launch. Block (head,
// split) takes every query of its head over keys [split·span, +span) in tiles
// of 64 keys staged in LDS, and keeps per query an online (max, sum, row) with
// exact exp(m_old - m_new) rescaling: masked keys get weight exactly 0. Wave w
// owns queries 4w .. 4w + 3 in every phase (lane = key for the scores, lane =
// channel for the values), so a query's statistics never leave its wave. With
// several splits each block writes its (max, sum, row) per query, and the last
// block of the head to finish (a per-head counter it resets to zero) combines
// them in split order, so the result does not depend on which block is last.
// ---------------------------------------------------------------------------
constexpr int kPromptTile = 64;
constexpr int kPromptKeyStride = kMaxHeadWidth + 4; // padded rows: lanes reading key rows spread over the banks
constexpr int kPromptPartial = kMaxHeadWidth + 2;
static_assert(kMaxPromptQueries == 4 * kWavesPerBlock, "four queries per wave");

__global__ void __launch_bounds__(kBlock) prompt_attention_kernel(
    const float* __restrict__ q, int q_count, const float* __restrict__ keys, const float* __restrict__ values,
    int k_count, int width, int head_width, int causal, float scale, int splits, int span, float* __restrict__ out,
    float* __restrict__ partials, unsigned int* __restrict__ counters)
{
    __shared__ __attribute__((aligned(16))) float qs[kMaxPromptQueries][kMaxHeadWidth];
    __shared__ __attribute__((aligned(16))) float ks[kPromptTile][kPromptKeyStride];
    __shared__ float vs[kPromptTile][kMaxHeadWidth];
    __shared__ float ps[kMaxPromptQueries][kPromptTile];
    __shared__ int last_block;

    const int split = blockIdx.x % splits, head = blockIdx.x / splits;
    const int column = head * head_width;
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int first = split * span, end = min(first + span, k_count);

    for (int i = threadIdx.x; i < kMaxPromptQueries * kMaxHeadWidth; i += kBlock)
    {
        const int r = i / kMaxHeadWidth, c = i % kMaxHeadWidth;
        qs[r][c] = r < q_count && c < head_width ? q[(size_t) r * width + column + c] : 0.f;
    }

    float m[4], l[4], acc[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
        m[k] = -INFINITY;
        l[k] = 0.f;
        acc[k] = 0.f;
    }
    for (int t0 = first; t0 < end; t0 += kPromptTile)
    {
        const int n = min(kPromptTile, end - t0);
        __syncthreads(); // the previous tile's readers are done (and the queries are in)
        for (int i = threadIdx.x; i < kPromptTile * kMaxHeadWidth / 4; i += kBlock)
        {
            const int j = i / (kMaxHeadWidth / 4), c4 = 4 * (i % (kMaxHeadWidth / 4));
            float4v kv = {0.f, 0.f, 0.f, 0.f}, vv = {0.f, 0.f, 0.f, 0.f};
            if (j < n && c4 < head_width)
            {
                const size_t at = (size_t) (t0 + j) * width + column + c4;
                kv = *reinterpret_cast<const float4v*>(keys + at);
                vv = *reinterpret_cast<const float4v*>(values + at);
            }
            *reinterpret_cast<float4v*>(&ks[j][c4]) = kv;
            *reinterpret_cast<float4v*>(&vs[j][c4]) = vv;
        }
        __syncthreads();

        // Scores of key t0 + lane against this wave's four queries.
        float s[4] = {0.f, 0.f, 0.f, 0.f};
        for (int c = 0; c < head_width; c += 4)
        {
            const float4v kv = *reinterpret_cast<const float4v*>(&ks[lane][c]);
#pragma unroll
            for (int k = 0; k < 4; ++k)
            {
                const float4v qv = *reinterpret_cast<const float4v*>(&qs[4 * wave + k][c]);
                s[k] += (qv[0] * kv[0] + qv[1] * kv[1]) + (qv[2] * kv[2] + qv[3] * kv[3]);
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            const int query = 4 * wave + k;
            const int key = t0 + lane;
            const bool seen = query < q_count && lane < n && (!causal || key <= k_count - q_count + query);
            const float score = seen ? scale * s[k] : -INFINITY;
            const float m_new = fmaxf(m[k], wave_max(score));
            const float alpha = m_new == -INFINITY ? 1.f : expf(m[k] - m_new);
            const float p = seen ? expf(score - m_new) : 0.f;
            l[k] = l[k] * alpha + wave_sum(p);
            acc[k] *= alpha;
            m[k] = m_new;
            ps[query][lane] = p;
        }
        __syncthreads();

        // Values: lane = channel.
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            float sum = 0.f;
            for (int j = 0; j < n; ++j)
                sum += ps[4 * wave + k][j] * vs[j][lane];
            acc[k] += sum;
        }
    }

    if (splits == 1)
    {
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            const int query = 4 * wave + k;
            if (query < q_count && lane < head_width)
                out[(size_t) query * width + column + lane] = acc[k] / l[k];
        }
        return;
    }

    float* const head_parts = partials + (size_t) head * splits * kMaxPromptQueries * kPromptPartial;
#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
        const int query = 4 * wave + k;
        float* part = head_parts + ((size_t) split * kMaxPromptQueries + query) * kPromptPartial;
        if (query < q_count)
        {
            if (lane < head_width)
                part[2 + lane] = acc[k];
            if (lane == 0)
            {
                part[0] = m[k];
                part[1] = l[k];
            }
        }
    }
    __threadfence(); // the partial is visible device-wide before the count says so
    __syncthreads();
    if (threadIdx.x == 0)
        last_block = atomicAdd(&counters[head], 1u) == (unsigned) (splits - 1);
    __syncthreads();
    if (!last_block)
        return;
    __threadfence(); // every other block's partial is visible from here on

#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
        const int query = 4 * wave + k;
        if (query >= q_count)
            continue;
        float largest = -INFINITY;
        for (int sp = 0; sp < splits; ++sp)
        {
            const float* part = head_parts + ((size_t) sp * kMaxPromptQueries + query) * kPromptPartial;
            if (part[1] != 0.f)
                largest = fmaxf(largest, part[0]);
        }
        float numerator = 0.f, denominator = 0.f;
        for (int sp = 0; sp < splits; ++sp)
        {
            const float* part = head_parts + ((size_t) sp * kMaxPromptQueries + query) * kPromptPartial;
            if (part[1] == 0.f)
                continue;
            const float factor = expf(part[0] - largest);
            numerator += factor * (lane < head_width ? part[2 + lane] : 0.f);
            denominator += factor * part[1];
        }
        if (lane < head_width)
            out[(size_t) query * width + column + lane] = numerator / denominator;
    }
    if (threadIdx.x == 0)
        counters[head] = 0u; // zero again for the next launch
}

// ---------------------------------------------------------------------------
// Argmax (Kernels/Argmax.h:46-262): candidates are (value, index) pairs; a
// larger value wins and equal values keep the lower index, so the fold ends on
// the index a left-to-right scan stops at. Suppressed entries never compete;
// a row with none allowed yields 0.
// ---------------------------------------------------------------------------
constexpr uint32_t kUnchosen = 0xFFFFFFFFu;
constexpr int kArgmaxPerThread = 8;

__device__ __forceinline__ bool better(float v, uint32_t i, float bv, uint32_t bi)
{
    if (i == kUnchosen)
        return false;
    if (bi == kUnchosen)
        return true;
    return v > bv || (v == bv && i < bi);
}

__device__ __forceinline__ void block_argmax(float& v, uint32_t& i)
{
    __shared__ float sv[kWavesPerBlock];
    __shared__ uint32_t si[kWavesPerBlock];
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1)
    {
        const float ov = __shfl_xor(v, offset, kWave);
        const uint32_t oi = __shfl_xor(i, offset, kWave);
        if (better(ov, oi, v, i))
        {
            v = ov;
            i = oi;
        }
    }
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    if (lane == 0)
    {
        sv[wave] = v;
        si[wave] = i;
    }
    __syncthreads();
    v = sv[0];
    i = si[0];
    for (int k = 1; k < (int) (blockDim.x / kWave); ++k)
        if (better(sv[k], si[k], v, i))
        {
            v = sv[k];
            i = si[k];
        }
}

__global__ void __launch_bounds__(kBlock) argmax_partial_kernel(const float* __restrict__ logits,
                                                                size_t row_stride, int row_length,
                                                                const float* __restrict__ mask,
                                                                int groups,
                                                                float* __restrict__ pv,
                                                                uint32_t* __restrict__ pi)
{
    const int row = blockIdx.x / groups, part = blockIdx.x % groups;
    const float* values = logits + (size_t) row * row_stride;
    float bv = 0.f;
    uint32_t bi = kUnchosen;
    for (int j = part * kBlock + threadIdx.x; j < row_length; j += groups * kBlock)
    {
        if (mask != nullptr && mask[j] != 0.f)
            continue;
        const float v = values[j];
        if (bi == kUnchosen || v > bv)
        {
            bv = v;
            bi = (uint32_t) j;
        }
    }
    block_argmax(bv, bi);
    if (threadIdx.x == 0)
    {
        pv[blockIdx.x] = bv;
        pi[blockIdx.x] = bi;
    }
}

__global__ void __launch_bounds__(kWave) argmax_final_kernel(const float* __restrict__ pv,
                                                             const uint32_t* __restrict__ pi,
                                                             int groups, uint32_t* __restrict__ out)
{
    const int row = blockIdx.x;
    float bv = 0.f;
    uint32_t bi = kUnchosen;
    for (int k = threadIdx.x; k < groups; k += kWave)
        if (better(pv[row * groups + k], pi[row * groups + k], bv, bi))
        {
            bv = pv[row * groups + k];
            bi = pi[row * groups + k];
        }
    block_argmax(bv, bi);
    if (threadIdx.x == 0)
        out[row] = bi == kUnchosen ? 0u : bi;
}

template <int WT>
hipError_t launch_gemv(hipStream_t stream, const float* x, int rows, int inner, const void* w,
                       const float* bias, float* y, int out, int flags)
{
    const bool vectorised = inner % 8 == 0 && (reinterpret_cast<uintptr_t>(x) % 16) == 0
                            && (reinterpret_cast<uintptr_t>(w) % 16) == 0;
    // Enough waves to cover the chip at one output per wave; several outputs
    // per wave only once there are plenty of waves.
    const int opw = out >= 8192 ? 4 : 1;
    for (int r0 = 0; r0 < rows; r0 += 4)
    {
        const int rr = std::min(4, rows - r0);
        const float* xr = x + (size_t) r0 * inner;
        float* yr = y + (size_t) r0 * out;
        const int waves = (out + opw - 1) / opw;
        const dim3 grid((waves + kWavesPerBlock - 1) / kWavesPerBlock);
        if (rr == 1 && opw == 1)
            hipLaunchKernelGGL((gemv_kernel<WT, 1, 1>), grid, dim3(kBlock), 0, stream, xr, rr, inner, w, bias, yr, out, flags, (int) vectorised);
        else if (rr == 1)
            hipLaunchKernelGGL((gemv_kernel<WT, 1, 4>), grid, dim3(kBlock), 0, stream, xr, rr, inner, w, bias, yr, out, flags, (int) vectorised);
        else if (opw == 1)
            hipLaunchKernelGGL((gemv_kernel<WT, 4, 1>), grid, dim3(kBlock), 0, stream, xr, rr, inner, w, bias, yr, out, flags, (int) vectorised);
        else
            hipLaunchKernelGGL((gemv_kernel<WT, 4, 4>), grid, dim3(kBlock), 0, stream, xr, rr, inner, w, bias, yr, out, flags, (int) vectorised);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}

} // namespace

// (Asked once: a node's GPUs are alike, the number only steers the choice of
// tiles, and to ask for the current device at each launch costs 0.3 us.)
int compute_units()
{
    static const int units = [] {
        int device = 0, count = 0;
        if (hipGetDevice(&device) == hipSuccess
            && hipDeviceGetAttribute(&count, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && count > 0)
            return count;
        return 256;
    }();
    return units;
}

hipError_t linear(hipStream_t stream, const float* x, int rows, int inner, const void* weight,
                  int wdtype, const float* bias, float* y, int out, int flags, const Scratch& scratch)
{
    const ProductMatrix matrix {weight, bias, y, 1.f};
    Products p {};
    p.x = x;
    p.rows = rows;
    p.inner = inner;
    p.matrices = &matrix;
    p.count = 1;
    p.columns = out;
    p.ldy = out;
    p.flags = flags;
    p.wdtype = wdtype;
    // Up to four rows the GEMV (a wave per output, one read of W); from five
    // on it would read W again for every four rows (16 x 768 -> 3072: four
    // launches of 4 us against one of 5).
    if (rows > kSplitRowLimit || (rows > 4 && row_product_fits(p)))
        return products(stream, p, scratch);
    switch (wdtype)
    {
        case kF32: return launch_gemv<kF32>(stream, x, rows, inner, weight, bias, y, out, flags);
        case kF16: return launch_gemv<kF16>(stream, x, rows, inner, weight, bias, y, out, flags);
        default: return launch_gemv<kBF16>(stream, x, rows, inner, weight, bias, y, out, flags);
    }
}

hipError_t layernorm(hipStream_t stream, const float* x, const float* gamma, const float* beta,
                     float* y, int rows, int width, float eps)
{
    auto whole = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    if (width % 4 != 0 || width > 2048 || !whole(x) || !whole(y))
    {
        hipLaunchKernelGGL(layernorm_kernel, dim3(rows), dim3(kBlock), 0, stream, x, gamma, beta, y, width, eps);
        return hipGetLastError();
    }
    auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(rows), dim3(kWave), 0, stream, x, gamma, beta, y, width, eps);
    };
    width <= 512    ? run(layernorm_row_kernel<2>)
    : width <= 1280 ? run(layernorm_row_kernel<5>)
                    : run(layernorm_row_kernel<8>);
    return hipGetLastError();
}

hipError_t embed(hipStream_t stream, const uint32_t* tokens, int count, const float* token_table,
                 const float* position_table, int first_position, float* y, int width,
                 int vocabulary)
{
    const dim3 grid((width + kBlock - 1) / kBlock, count);
    hipLaunchKernelGGL(embed_kernel, grid, dim3(kBlock), 0, stream, tokens, token_table, position_table, first_position, y, width, vocabulary);
    return hipGetLastError();
}

int attention_chunks(int heads, int q_count, int k_count)
{
    // Enough blocks to cover the chip (about 256), at least 32 keys a chunk,
    // and no chunk longer than the shared score array.
    const int units = heads * q_count;
    int chunks = std::max(1, std::min((k_count + 31) / 32, (256 + units - 1) / units));
    while ((k_count + chunks - 1) / chunks > kAttentionChunkKeys)
        ++chunks;
    return chunks;
}

// Keys per split of a prompt step's attention: a whole number of 64-key tiles,
// as few as give about one round of blocks over the chip (256).
int prompt_attention_span(int heads, int k_count)
{
    const int tiles = std::max(1, (k_count + kPromptTile - 1) / kPromptTile);
    const int wanted = std::max(1, std::min(tiles, (256 + heads - 1) / heads));
    return (tiles + wanted - 1) / wanted * kPromptTile;
}

int prompt_attention_splits(int heads, int k_count)
{
    const int span = prompt_attention_span(heads, k_count);
    return std::max(1, (k_count + span - 1) / span);
}

bool takes_prompt_attention(int q_count, int heads)
{
    return q_count >= 2 && q_count <= kMaxPromptQueries && heads <= kAttentionCounters;
}

hipError_t combine(hipStream_t stream, const float* partials, int q_count, int width, int heads, int chunks, float* out)
{
    auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(heads * q_count), dim3(kBlock), 0, stream, partials, q_count, width,
                           width / heads, chunks, out);
    };
    chunks <= kWavesPerBlock       ? run(attention_combine_kernel<1>)
    : chunks <= 2 * kWavesPerBlock ? run(attention_combine_kernel<2>)
                                   : run(attention_combine_kernel<8>);
    return hipGetLastError();
}

size_t attention_workspace_floats(int heads, int q_count, int k_count, int head_width)
{
    if (takes_prompt_attention(q_count, heads))
    {
        const int splits = prompt_attention_splits(heads, k_count);
        return kAttentionCounters
               + (splits > 1 ? (size_t) heads * splits * kMaxPromptQueries * kPromptPartial : 0);
    }
    const int chunks = attention_chunks(heads, q_count, k_count);
    return kAttentionCounters + (chunks > 1 ? (size_t) heads * q_count * chunks * (head_width + 2) : 0);
}

// Two queries on, heads of 64 channels: query_attention_kernel over 16 queries
// a block, or 32 (each key and value read for twice as many) where blocks of 16
// over 256 keys each would not fit one round. As many key splits as leave each wave 32
// keys, while the blocks fit one round of the CUs; what they leave stays within
// kQueryAttentionFloats (at most 256·32 partial rows).
hipError_t query_attention(hipStream_t stream, const float* q, int q_count, const float* keys, const float* values,
                           int k_count, int width, int heads, int causal, float scale, float* out, float* partials)
{
    const int reach = kQueryKeys * kQueryWaves, reaches = (k_count + reach - 1) / reach;
    const int tile = (long long) heads * ((q_count + 15) / 16) * reaches > kQueryBlocks ? 32 : 16;
    const int tiles = (q_count + tile - 1) / tile;
    const int splits = std::max(1, std::min(reaches, kQueryBlocks / (heads * tiles)));
    const int span = ((k_count + splits - 1) / splits + kQueryKeys - 1) / kQueryKeys * kQueryKeys;
    const dim3 block(kQueryWaves * kWave);
    constexpr int kMostTiles = 65535; // a launch's y extent
    hipError_t e = hipSuccess;
    for (int first = 0; first < tiles && e == hipSuccess; first += kMostTiles)
    {
        const dim3 grid(heads * splits, std::min(tiles - first, kMostTiles));
        if (tile == 32)
            hipLaunchKernelGGL(query_attention_kernel<2>, grid, block, 0, stream, q, q_count, keys, values, k_count,
                               width, causal, scale, splits, span, first, out, partials);
        else
            hipLaunchKernelGGL(query_attention_kernel<1>, grid, block, 0, stream, q, q_count, keys, values, k_count,
                               width, causal, scale, splits, span, first, out, partials);
        e = hipGetLastError();
    }
    if (e != hipSuccess || splits == 1)
        return e;
    return combine(stream, partials, q_count, width, heads, splits, out);
}

hipError_t attention(hipStream_t stream, const float* q, int q_count, const float* keys,
                     const float* values, int k_count, int width, int heads, int causal,
                     float scale, float* out, float* workspace)
{
    const int head_width = width / heads;
    unsigned int* const counters = reinterpret_cast<unsigned int*>(workspace);
    float* const partials = workspace + kAttentionCounters;
    // More queries than a prompt step's over few keys: one launch of a block for
    // each (query, head), while those fit one round (eight a CU) and their scores
    // are few. 17 queries of 12 heads over 20 keys: 4.4 us, 5.0 in
    // query_attention_kernel; 40 of 20 heads over 20 keys 4.7 and 4.9, over 33
    // 5.5 and 5.3; 100 of 12 heads over 20 5.1 and 5.0.
    const long long units = (long long) heads * q_count;
    const bool few_keys = q_count > kMaxPromptQueries && k_count <= 40 && units <= 2048 && units * k_count <= 20000
                          && attention_chunks(heads, q_count, k_count) == 1;
    if (q_count > 1 && head_width == 64 && !few_keys)
        return query_attention(stream, q, q_count, keys, values, k_count, width, heads, causal, scale, out, partials);
    if (takes_prompt_attention(q_count, heads))
    {
        const int splits = prompt_attention_splits(heads, k_count);
        hipLaunchKernelGGL(prompt_attention_kernel, dim3(heads * splits), dim3(kBlock), 0, stream, q, q_count, keys,
                           values, k_count, width, head_width, causal, scale, splits,
                           prompt_attention_span(heads, k_count), out, partials, counters);
        return hipGetLastError();
    }
    workspace = partials;
    const int chunks = attention_chunks(heads, q_count, k_count);
    const int chunk_length = (k_count + chunks - 1) / chunks;
    hipLaunchKernelGGL(attention_chunk_kernel, dim3(heads * q_count * chunks), dim3(kBlock), 0, stream,
                       q, q_count, keys, values, k_count, width, head_width, causal, scale, chunks,
                       chunk_length, out, workspace);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || chunks == 1)
        return e;
    return combine(stream, workspace, q_count, width, heads, chunks, out);
}

int argmax_groups(int row_length)
{
    const int per_group = kBlock * kArgmaxPerThread;
    return std::max(1, (row_length + per_group - 1) / per_group);
}

hipError_t argmax(hipStream_t stream, const float* logits, int rows, int row_length,
                  const float* mask, uint32_t* out, float* partial_values,
                  uint32_t* partial_indices)
{
    return argmax_rows(stream, logits, rows, (size_t) row_length, row_length, mask, out, partial_values,
                       partial_indices);
}

hipError_t argmax_rows(hipStream_t stream, const float* logits, int rows, size_t row_stride,
                       int row_length, const float* mask, uint32_t* out, float* partial_values,
                       uint32_t* partial_indices)
{
    const int groups = argmax_groups(row_length);
    hipLaunchKernelGGL(argmax_partial_kernel, dim3(rows * groups), dim3(kBlock), 0, stream, logits,
                       row_stride, row_length, mask, groups, partial_values, partial_indices);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL(argmax_final_kernel, dim3(rows), dim3(kWave), 0, stream, partial_values,
                       partial_indices, groups, out);
    return hipGetLastError();
}
} // namespace wsp::ops
