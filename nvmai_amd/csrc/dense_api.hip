// Entry points of the dense models: matrix products against BF16 weights, embedding rows, the cap of the
// logits, argmax.
#include "ctx.hpp"
#include "dense_kernels.hpp"
#include "ends_kernels.hpp"
#include "rules.hpp"

using namespace nvmai;

namespace nvmai {

// Rows of floats -> [row][3][k] BF16, the smallest part first.  Bound by its bytes (4 read, 6 written per value).
__global__ __launch_bounds__(256) void dense_split_kernel(const float* x, uint32_t x_stride, uint32_t k, uint16_t* planes) {
    const uint32_t at = (blockIdx.x * 256u + threadIdx.x) * 8u, row = blockIdx.y;
    if (at >= k) return;
    const float4 v[2] = {*reinterpret_cast<const float4*>(x + (size_t)row * x_stride + at), *reinterpret_cast<const float4*>(x + (size_t)row * x_stride + at + 4u)};
    const float f[8] = {v[0].x, v[0].y, v[0].z, v[0].w, v[1].x, v[1].y, v[1].z, v[1].w};
    uint32_t out[3][4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        uint32_t a[3], b[3];
        split3(f[2 * e], a[0], a[1], a[2]);
        split3(f[2 * e + 1], b[0], b[1], b[2]);
#pragma unroll
        for (int q = 0; q < 3; ++q) out[q][e] = a[q] | (b[q] << 16);
    }
#pragma unroll
    for (int q = 0; q < 3; ++q)
        *reinterpret_cast<uint4*>(planes + ((size_t)row * 3u + (2 - q)) * k + at) = make_uint4(out[q][0], out[q][1], out[q][2], out[q][3]);
}

void dense_split(hipStream_t s, const float* x, uint32_t x_stride, uint32_t rows, uint32_t k, uint16_t* planes) {
    dense_split_kernel<<<dim3((k + 2047) / 2048, rows), 256, 0, s>>>(x, x_stride, k, planes);
}

int dense_linear_check(const nvmai_hip_ctx* ctx, const DenseLinearParams& p) {
    if (!ctx || !p.w || !p.x || (!p.y && !p.y_f32)) return NVMAI_ERR_INVALID_ARG;
    if (ctx->act != NVMAI_ACT_BF16 && ctx->act != NVMAI_ACT_FP32) return NVMAI_ERR_UNSUPPORTED;
    if (p.k == 0 || p.k % 64 || p.n == 0 || p.w_stride < p.k || p.x_stride < p.k) return NVMAI_ERR_INVALID_ARG;
    if (p.activation < NVMAI_LINEAR_NONE || p.activation > NVMAI_LINEAR_SILU_PAIRS) return NVMAI_ERR_UNSUPPORTED;
    const bool pairs = p.activation == NVMAI_LINEAR_SILU_PAIRS;
    if (p.y_stride < (pairs ? p.n / 2 : p.n)) return NVMAI_ERR_INVALID_ARG;
    if (pairs && (p.n % 2 || p.y_stride % 2 || p.bias || p.mul)) return NVMAI_ERR_INVALID_ARG;
    if (p.mul && (!p.mul_ids || p.mul_stride < p.n)) return NVMAI_ERR_INVALID_ARG;
    if (!aligned16(p.w) || !aligned16(p.x) || p.w_stride % 8 || p.x_stride % 8) return NVMAI_ERR_ALIGNMENT;
    if (!p.loose && ((p.y && !aligned16(p.y)) || (p.y_f32 && !aligned16(p.y_f32)))) return NVMAI_ERR_ALIGNMENT;
    // 32-bit byte offsets inside an operand
    if ((uint64_t)p.n * p.w_stride * 2 > 0xFFFFFFFFull || !dense_rows_fit(p.rows, p.x_stride)) return NVMAI_ERR_UNSUPPORTED;
    return NVMAI_OK;
}

int dense_linear(nvmai_hip_ctx* ctx, hipStream_t s, const DenseLinearParams& p) {
    const int rc = dense_linear_check(ctx, p);
    if (rc) return rc;
    if (p.rows == 0) return NVMAI_OK;
    if (p.activation == NVMAI_LINEAR_SILU_PAIRS) return dense_launch_pairs(ctx, s, p);
    if (p.mul || p.activation == NVMAI_LINEAR_GELU_TANH || (p.bias && p.activation != NVMAI_LINEAR_NONE)) return dense_launch_full(ctx, s, p);
    if (p.bias) return dense_launch_bias(ctx, s, p);
    return p.activation == NVMAI_LINEAR_GELU_ERF ? dense_launch_erf(ctx, s, p) : dense_launch<DE_PLAIN>(ctx, s, p);
}

uint64_t dense_linear_ns(const nvmai_hip_ctx* ctx, uint32_t rows, uint32_t n, uint32_t k) {
    return (uint64_t)dense_plan(n, rows < 65u ? 65u : rows, k, 1, (uint32_t)ctx->compute_units, 5, dense_may_cut(ctx)).ns;
}

}  // namespace nvmai

namespace {

// An entry point's own call: the planes of 32-bit rows lie in the workspace.  Where it cannot be made large enough (while the
// stream is being captured, or without memory) the product is made without them.
int dense_linear_call(nvmai_hip_ctx* ctx, nvmai_stream stream, DenseLinearParams p) {
    const int rc = dense_linear_check(ctx, p);
    if (rc) return rc;
    if (ctx->act == NVMAI_ACT_FP32 && p.rows > 4) {
        const size_t bytes = dense_plane_bytes(p.rows, p.k);
        if (ws_begin(ctx, stream, ws_round(bytes)) == NVMAI_OK) p.planes = ws_take<uint16_t>(ctx, bytes / 2);
    }
    return dense_linear(ctx, (hipStream_t)stream, p);
}

// Rows of floats, and whether those of two of them share a value.
struct FloatRows {
    const float* base;
    uint32_t stride, cols;
};

bool overlap(const FloatRows& a, const FloatRows& b, uint32_t rows) {
    for (uint32_t i = 0; i < rows; ++i)
        for (uint32_t j = 0; j < rows; ++j) {
            const uintptr_t p = reinterpret_cast<uintptr_t>(a.base + (size_t)i * a.stride), q = reinterpret_cast<uintptr_t>(b.base + (size_t)j * b.stride);
            if (p < q + (size_t)b.cols * 4u && q < p + (size_t)a.cols * 4u) return true;
        }
    return false;
}

}  // namespace

extern "C" int nvmai_hip_dense_linear(nvmai_hip_ctx* ctx, nvmai_stream stream, const uint16_t* w, uint32_t w_stride,
                                      const void* x, uint32_t x_stride, uint32_t rows, uint32_t n, uint32_t k, void* y,
                                      float* y_f32, uint32_t y_stride, int activation) {
    const DenseLinearParams p{w, x, y, y_f32, w_stride, x_stride, y_stride, rows, n, k, activation};
    return dense_linear_call(ctx, stream, p);
}

extern "C" int nvmai_hip_dense_linear_ex(nvmai_hip_ctx* ctx, nvmai_stream stream, const uint16_t* w, uint32_t w_stride, const void* x,
                                         uint32_t x_stride, uint32_t rows, uint32_t n, uint32_t k, void* y, float* y_f32,
                                         uint32_t y_stride, const nvmai_linear_epilogue* e) {
    if (!e) return NVMAI_ERR_INVALID_ARG;
    const DenseLinearParams p{w, x, y, y_f32, w_stride, x_stride, y_stride, rows, n, k, e->activation, e->bias, e->mul, e->mul_ids,
                              e->mul_stride, e->mul_rows};
    return dense_linear_call(ctx, stream, p);
}

extern "C" int nvmai_hip_dense_linear_planes(nvmai_hip_ctx* ctx, nvmai_stream stream, const uint16_t* w, uint32_t w_stride, const uint16_t* x, uint32_t rows,
                                             uint32_t n, uint32_t k, float* y, uint32_t y_stride, uint16_t* y_planes, uint32_t y_k,
                                             const nvmai_linear_epilogue* e) {
    if (!ctx || !e || (y == nullptr) == (y_planes == nullptr)) return NVMAI_ERR_INVALID_ARG;
    if (ctx->act != NVMAI_ACT_FP32 || rows < 5 || !planes_fit(rows, k)) return NVMAI_ERR_UNSUPPORTED;
    // planes are stored two or four values at a time
    if (y_planes && (n % 4 || y_k % 4 || !planes_fit(rows, y_k))) return NVMAI_ERR_UNSUPPORTED;
    if (y_planes && y_k < (e->activation == NVMAI_LINEAR_SILU_PAIRS ? n / 2 : n)) return NVMAI_ERR_INVALID_ARG;
    DenseLinearParams p{w, x, y, nullptr, w_stride, 3 * k, y_stride, rows, n, k, e->activation, e->bias, e->mul, e->mul_ids, e->mul_stride, e->mul_rows};
    p.x_planes = true;
    if (y_planes) { p.y = y_planes; p.y_stride = 3 * y_k; p.y_k = y_k; }
    return dense_linear(ctx, (hipStream_t)stream, p);
}

extern "C" int nvmai_hip_rms_residual_linear(nvmai_hip_ctx* ctx, nvmai_stream stream, const float* x, uint32_t x_stride, const float* delta,
                                             uint32_t delta_stride, const uint16_t* post_weight, float post_add, float eps, float* x_out,
                                             uint32_t x_out_stride, const uint16_t* w, uint32_t w_stride, uint32_t rows, uint32_t n, uint32_t k,
                                             float* y, uint32_t y_stride, const nvmai_linear_epilogue* e) {
    if (!ctx || !e || !delta || !post_weight || !x_out) return NVMAI_ERR_INVALID_ARG;
    if (ctx->act != NVMAI_ACT_FP32 || rows > DENSE_RMS_ROWS || k > DENSE_RMS_K) return NVMAI_ERR_UNSUPPORTED;
    DenseLinearParams p{w, x, y, nullptr, w_stride, x_stride, y_stride, rows, n, k, e->activation, e->bias, e->mul, e->mul_ids, e->mul_stride, e->mul_rows};
    p.rms_delta = delta; p.rms_w = post_weight; p.rms_out = x_out; p.rms_delta_stride = delta_stride; p.rms_out_stride = x_out_stride;
    p.rms_add = post_add; p.rms_eps = eps;
    if (delta_stride < k || x_out_stride < k) return NVMAI_ERR_INVALID_ARG;
    if (!aligned16(delta) || !aligned16(post_weight) || !aligned16(x_out) || delta_stride % 4 || x_out_stride % 4) return NVMAI_ERR_ALIGNMENT;
    // every block reads x and delta whole, while the first one stores x_out and others that have ended store y
    const FloatRows out{x_out, x_out_stride, k}, product{y, y_stride, e->activation == NVMAI_LINEAR_SILU_PAIRS ? n / 2 : n};
    for (const FloatRows& in : {FloatRows{x, x_stride, k}, FloatRows{delta, delta_stride, k}})
        if (overlap(in, out, rows) || overlap(in, product, rows)) return NVMAI_ERR_INVALID_ARG;
    if (overlap(out, product, rows)) return NVMAI_ERR_INVALID_ARG;
    return dense_linear(ctx, (hipStream_t)stream, p);
}

extern "C" int nvmai_hip_embed_rows(nvmai_hip_ctx* ctx, nvmai_stream stream, const uint16_t* table, uint32_t table_stride,
                                    const uint32_t* token_ids, uint32_t n_tokens, float* out, uint32_t out_stride, uint32_t d,
                                    uint32_t vocab) {
    return nvmai_hip_embed_positions(ctx, stream, table, table_stride, token_ids, n_tokens, 1.0f, nullptr, nullptr, out, out_stride, nullptr, 0, d, vocab);
}

extern "C" int nvmai_hip_embed_positions(nvmai_hip_ctx* ctx, nvmai_stream stream, const uint16_t* table, uint32_t table_stride,
                                         const uint32_t* token_ids, uint32_t n_tokens, float scale, const double* inv_freq,
                                         const nvmai_row_map* map, float* out, uint32_t out_stride, void* act, uint32_t act_stride,
                                         uint32_t d, uint32_t vocab) {
    if (!ctx || !table || !token_ids || !out || d == 0 || table_stride < d || out_stride < d || vocab == 0) return NVMAI_ERR_INVALID_ARG;
    if ((inv_freq && !map) || (act && act_stride < d)) return NVMAI_ERR_INVALID_ARG;
    if (act && ctx->act != NVMAI_ACT_BF16 && ctx->act != NVMAI_ACT_FP32) return NVMAI_ERR_UNSUPPORTED;
    if (n_tokens == 0) return NVMAI_OK;
    if (n_tokens > 65535) return NVMAI_ERR_UNSUPPORTED;
    EmbedParams p{table, token_ids, out, act, inv_freq, SeqRows{}, table_stride, out_stride, act_stride, d, vocab, scale};
    if (map) p.rows = SeqRows{map->slots, map->positions, map->slot, map->position};
    const dim3 grid((d + 511) / 512, n_tokens);
    if (ctx->act == NVMAI_ACT_FP32) embed_rows_kernel<ACT_FP32><<<grid, 256, 0, (hipStream_t)stream>>>(p);
    else embed_rows_kernel<ACT_BF16><<<grid, 256, 0, (hipStream_t)stream>>>(p);
    return launch_status();
}

extern "C" int nvmai_hip_softcap_rows(nvmai_hip_ctx* ctx, nvmai_stream stream, float* x, uint32_t x_stride, uint32_t rows, uint32_t n,
                                      float cap) {
    if (!ctx || !x || n == 0 || x_stride < n || !(cap > 0.0f)) return NVMAI_ERR_INVALID_ARG;
    if (rows == 0) return NVMAI_OK;
    if (rows > 65535) return NVMAI_ERR_UNSUPPORTED;
    softcap_rows_kernel<<<dim3((n + 255) / 256, rows), 256, 0, (hipStream_t)stream>>>(x, x_stride, n, cap);
    return launch_status();
}

extern "C" int nvmai_hip_argmax_rows(nvmai_hip_ctx* ctx, nvmai_stream stream, const float* x, uint32_t x_stride, uint32_t rows,
                                     uint32_t n, uint32_t* out_index) {
    if (!ctx || !x || !out_index || n == 0 || x_stride < n) return NVMAI_ERR_INVALID_ARG;
    if (rows == 0) return NVMAI_OK;
    if (rows > 65535) return NVMAI_ERR_UNSUPPORTED;
    const int rc = ws_begin(ctx, stream, ws_round((size_t)rows * ARGMAX_BLOCKS * 8));
    if (rc) return rc;
    uint64_t* part = ws_take<uint64_t>(ctx, (size_t)rows * ARGMAX_BLOCKS);
    uint32_t blocks = (n + 1023) / 1024;
    if (blocks > ARGMAX_BLOCKS) blocks = ARGMAX_BLOCKS;
    argmax_stage1_kernel<<<dim3(blocks, rows), 256, 0, (hipStream_t)stream>>>(x, x_stride, n, part);
    argmax_stage2_kernel<<<rows, 256, 0, (hipStream_t)stream>>>(part, blocks, out_index);
    return launch_status();
}
