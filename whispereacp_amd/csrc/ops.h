// Host-side launchers of the per-op gfx950 kernels. Each returns the launch's
// hipError_t; argument checking is the C ABI's job (capi.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace wsp::ops
{
// Up to this many rows the products stay in fp32 arithmetic, and those that
// the matrix cores cannot load in whole vectors take the split GEMV (the
// reference's splitRowLimit, Net/KernelNet.h:144-149).
constexpr int kSplitRowLimit = 16;
constexpr int kMaxHeadWidth = 64;
constexpr int kAttentionChunkKeys = 1024; // longest key chunk one workgroup scores

// CUs of a GPU.
int compute_units();

// One of the matrices side by side in a product: W [columns][inner], its bias
// (or null), its output, and the factor its sums are multiplied by before the
// bias (the reciprocal of the power of two its stored weights carry, exact; 1
// for weights stored as they are).
struct ProductMatrix
{
    const void* w = nullptr;
    const float* bias = nullptr;
    float* y = nullptr;
    float scale = 1.f;
};
constexpr int kMaxMatrices = 64;

// The products over X as split_product's kernel reads it: 16-bit parts for
// 16-bit W (cut_parts: three bf16 parts, or fp16 hi + lo), part p at
// parts + p·part_stride + r·inner, or fp32 X for fp32 W. `count` matrices of
// `columns` columns share the launch. Row r of a column lands at
// y[(r / rows_per_group)·group_stride + (r % rows_per_group)·ldy + c]
// (rows_per_group 0: one group; += with kProductResidual, after GELU with
// kProductGelu), or, with out_parts set, as the parts of the value (one matrix
// only, rows of `columns` values, part p at out_parts + p·out_part_stride).
constexpr int kProductGelu = 1;
constexpr int kProductResidual = 2;
// fp32 products, one matrix: row f is frame f of a convolution and goes out as
// the columns of the next, stride two: of output row p's three taps (channel·3 +
// tap, rows of 3·columns) tap t is frame 2p + t - 1, zero outside the frames.
constexpr int kProductTaps = 4;
struct SplitProduct
{
    const void* parts;
    size_t part_stride;
    int rows, inner;
    int count, columns;
    ProductMatrix matrix[kMaxMatrices];
    int ldy;
    int rows_per_group;
    size_t group_stride;
    int flags;
    const float* residual; // kProductResidual: what is added to, laid out as y (null: y)
    int taps;              // kProductTaps: the next convolution's rows
    void* out_parts;
    size_t out_part_stride;
    int wdtype;
    // Matrix 1 (y1_halves) and matrix 2 (y2_halves_t), when set, go out as fp16
    // hi = fp16(v) and lo = fp16(v - hi) instead of fp32: hi of row r, column c
    // at y1_halves[r·columns + c], lo halves_pitch·columns further; y2_halves_t
    // transposed, hi at [c·halves_pitch + attention_place(r)]. (The encoder's
    // keys and values for its attention; fp32 products need columns in quads.)
    void* y1_halves;
    void* y2_halves_t;
    int halves_pitch;
};

// What split_product and fp32_split ask of the current device before their first
// launch there (their stages pass the LDS a launch gets unasked).
hipError_t prepare_split_products();

// 16-bit weights, inner a multiple of 64, columns of 128.
bool split_product_fits(int wdtype, int inner, int columns);
hipError_t split_product(hipStream_t stream, const SplitProduct& product);
// fp32 weights: rows in whole 16-byte runs, several matrices in multiples of
// 64 columns.
bool fp32_split_fits(const SplitProduct& product);
hipError_t fp32_split(hipStream_t stream, const SplitProduct& product);
// count fp32 values (a multiple of 8) as parts for 16-bit weights of wdtype.
hipError_t split_rows(hipStream_t stream, const float* x, size_t count, int wdtype, void* parts,
                      size_t part_stride);

// Memory for a product's input as 16-bit parts; products that would want more
// read fp32 rows instead.
struct Scratch
{
    void* data = nullptr;
    size_t bytes = 0;
};
// Bytes for the parts of `values` fp32 values (three 16-bit parts at most).
constexpr size_t parts_bytes(size_t values)
{
    return 6 * values;
}

// y = X·Wᵀ for any rows, extents and weight storage (linear_product.hip), any
// number of matrices of `columns` columns over the same rows. More than
// kSplitRowLimit rows of 16-bit weights in whole parts (parts_fit) are computed
// in 16-bit parts, everything else in fp32.
bool parts_fit(int wdtype, int inner, int columns, const void* x);
struct Products
{
    const float* x;
    int rows, inner;
    const ProductMatrix* matrices;
    int count, columns;
    int ldy;
    int rows_per_group;  // as SplitProduct's
    size_t group_stride;
    int flags;
    int wdtype;
};
hipError_t products(hipStream_t stream, const Products& given, const Scratch& scratch);
// Whether a product of at most kSplitRowLimit rows goes there in one launch.
bool row_product_fits(const Products& product);

hipError_t linear(hipStream_t stream, const float* x, int rows, int inner, const void* weight,
                  int wdtype, const float* bias, float* y, int out, int flags, const Scratch& scratch = {});

hipError_t layernorm(hipStream_t stream, const float* x, const float* gamma, const float* beta,
                     float* y, int rows, int width, float eps);

// LayerNorm rows (as layernorm) written as the parts of split_product's input;
// widths that are multiples of 4 up to 2048 (layernorm_parts_fits).
bool layernorm_parts_fits(int width);
hipError_t layernorm_parts(hipStream_t stream, const float* x, const float* gamma, const float* beta, void* parts,
                           size_t part_stride, int rows, int width, float eps, int wdtype);
// Token ids at or past `vocabulary` poison their row with NaN.
hipError_t embed(hipStream_t stream, const uint32_t* tokens, int count, const float* token_table,
                 const float* position_table, int first_position, float* y, int width,
                 int vocabulary);

// Queries a prompt step's attention takes in one launch (prompt_attention).
constexpr int kMaxPromptQueries = 16;
// The attention workspace starts with this many per-head counters (the
// prompt attention's last-block election); they are zero between launches,
// and whoever provides a workspace zeroes them once before its first use.
constexpr int kAttentionCounters = 256;

// Blocks a round of the multi-query attention of 64-channel heads takes, and
// the workspace it may use whatever the call: a workspace handed to attention()
// for such heads holds at least this many floats.
constexpr int kQueryBlocks = 256;
constexpr size_t kQueryAttentionFloats = kAttentionCounters + (size_t) kQueryBlocks * 32 * (64 + 2);

// How many key chunks the split-key attention uses for this shape, and the
// workspace (floats) it needs: the counters, then the partials —
// chunks * (head_width + 2) per (head, query) for one query or more than
// kMaxPromptQueries, splits * kMaxPromptQueries * (kMaxHeadWidth + 2) per head
// for a prompt step. The entry points refuse what their workspace does not hold
// of this, several queries of 64-channel heads too, which never take more than
// kQueryAttentionFloats.
int attention_chunks(int heads, int q_count, int k_count);
int prompt_attention_splits(int heads, int k_count);
size_t attention_workspace_floats(int heads, int q_count, int k_count, int head_width);

hipError_t attention(hipStream_t stream, const float* q, int q_count, const float* keys,
                     const float* values, int k_count, int width, int heads, int causal,
                     float scale, float* out, float* workspace);

int argmax_groups(int row_length);
hipError_t argmax(hipStream_t stream, const float* logits, int rows, int row_length,
                  const float* mask, uint32_t* out, float* partial_values,
                  uint32_t* partial_indices);

// The same over rows `row_stride` floats apart.
hipError_t argmax_rows(hipStream_t stream, const float* logits, int rows, size_t row_stride,
                       int row_length, const float* mask, uint32_t* out, float* partial_values,
                       uint32_t* partial_indices);
} // namespace wsp::ops
