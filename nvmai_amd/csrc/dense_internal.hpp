// The dense product, callable from other entry-point files.
#pragma once

#include "ctx.hpp"
#include "rules.hpp"

namespace nvmai {

struct DenseLinearParams {
    const uint16_t* w;      // [n, w_stride] BF16
    const void* x;          // [rows, x_stride] activations
    void* y;                // activations, or nullptr
    float* y_f32;           // floats, or nullptr
    uint32_t w_stride, x_stride, y_stride, rows, n, k;
    int activation;         // NVMAI_LINEAR_*
    const uint16_t* bias;   // [n] BF16, or nullptr
    const uint16_t* mul;    // BF16 table [mul_rows, mul_stride]: y[t, r] *= mul[mul_ids[t], r]; or nullptr
    const uint32_t* mul_ids;
    uint32_t mul_stride, mul_rows;
    uint16_t* planes;       // dense_plane_bytes of scratch for the rows of a 32-bit context, or nullptr
    // the rows that are multiplied are x + RMS(rms_delta) * (rms_add + rms_w), which go to rms_out as well (y and rms_out: neither x nor rms_delta); nullptr: x
    const float* rms_delta;
    const uint16_t* rms_w;
    float* rms_out;
    uint32_t rms_delta_stride, rms_out_stride;
    float rms_add, rms_eps;
    bool x_planes;          // x: planes (planes.hpp), x_stride 3 k, five rows or more
    uint32_t y_k;           // y: planes of y_k values, y_stride 3 y_k (x_planes too); 0: activations
    bool loose;             // plain outputs need not lie at 16-byte boundaries: one value at a time
};

// What the form with rms_delta takes beside a 32-bit context: a row is held in the registers of one wave.
constexpr uint32_t DENSE_RMS_ROWS = 2, DENSE_RMS_K = 2048;

void dense_split(hipStream_t s, const float* x, uint32_t x_stride, uint32_t rows, uint32_t k, uint16_t* planes);

int dense_linear_check(const nvmai_hip_ctx* ctx, const DenseLinearParams& p);
// What a call of more than 64 rows in a 16-bit context is expected to take, in ns.
uint64_t dense_linear_ns(const nvmai_hip_ctx* ctx, uint32_t rows, uint32_t n, uint32_t k);
// The launches behind it by what stands between sum and store (dense_*_api.hip, built side by side).
int dense_launch_erf(nvmai_hip_ctx* ctx, hipStream_t s, const DenseLinearParams& p);
int dense_launch_bias(nvmai_hip_ctx* ctx, hipStream_t s, const DenseLinearParams& p);
int dense_launch_pairs(nvmai_hip_ctx* ctx, hipStream_t s, const DenseLinearParams& p);
int dense_launch_full(nvmai_hip_ctx* ctx, hipStream_t s, const DenseLinearParams& p);
// Launches it.  In a 32-bit context p.planes is the caller's scratch: a call between ws_takes must not start the workspace anew.
int dense_linear(nvmai_hip_ctx* ctx, hipStream_t s, const DenseLinearParams& p);

}  // namespace nvmai
