// The once-per-sequence cross-attention key/value projection
// (Decoder/Decoder.cpp:121-146): K = X·Wkᵀ, V = X·Wvᵀ + bv over the encoder
// rows with fp32 accumulation, side by side in one product.
#include "capi_internal.h"
#include "ops.h"

namespace wsp
{
int cross_kv_projection(Context* ctx, const float* x, int rows, int width, const void* wk, const void* wv,
                        const float* bv, int wdtype, float* k_out, float* v_out)
{
    const ops::ProductMatrix matrices[] = {{wk, nullptr, k_out, 1.f}, {wv, bv, v_out, 1.f}};
    ops::Products p {};
    p.x = x;
    p.rows = rows;
    p.inner = width;
    p.matrices = matrices;
    p.count = 2;
    p.columns = width;
    p.ldy = width;
    p.wdtype = wdtype;
    return context_hip(ctx, ops::products(ctx->stream, p, {ctx->parts, ctx->parts_bytes}), "cross K/V projection");
}
} // namespace wsp
