// Kernels of the dense models (BF16 weights; 16-bit BF16 or 32-bit activations; a 32-bit residual stream):
// the matrix products.  gfx950, wave64.
#pragma once

#include "dense_internal.hpp"
#include "dense_plan.hpp"
#include "common.hpp"
#include "planes.hpp"

namespace nvmai {

typedef __bf16 dn_b8 __attribute__((ext_vector_type(8)));
typedef float dn_f4 __attribute__((ext_vector_type(4)));
typedef uint32_t dn_u4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ dn_f4 dn_mfma(const uint4& a, const uint4& b, dn_f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dn_b8, a), __builtin_bit_cast(dn_b8, b), c, 0, 0, 0);
}

// The same onto a sum that stays where it is, in the second half of the register file: with 64 sums and 32 operands the compiler moves sums about between
// products (three copies per product).  The compiler does not see a product here: operands must not come straight from vector instructions, and
// dn_mfma_done stands before the first use of a sum.
__device__ __forceinline__ void dn_mfma_in_place(const uint4& a, const uint4& b, dn_f4& c) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(__builtin_bit_cast(dn_u4, a)), "v"(__builtin_bit_cast(dn_u4, b)));
#endif
}

// The last product's sum is written.
__device__ __forceinline__ void dn_mfma_done() {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#endif
}

// z/2 (1 + erf(z / sqrt 2))
__device__ __forceinline__ float gelu_erf(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }

// z/2 (1 + tanh(sqrt(2/pi) (z + 0.044715 z^3)))
__device__ __forceinline__ float gelu_tanh(float z) { return 0.5f * z * (1.0f + tanhf(0.79788456080286536f * fmaf(0.044715f * z * z, z, z))); }

// Both without the library's branches, for the tiles, whose stores erff and tanhf lengthen by a third (2048 x 8192 x 2048 with
// GELU_ERF: 85 us, 75 with this, 62 without an activation).  z Phi(z), Phi(z) = 1/2 + z R(z^2) for |z| < 1, and past it
// s or 1 - s with s = Phi(-|z|), which does not cancel: e^(-z^2 / 2) times a polynomial in 1 / (1 + 0.34 |z|), or 1 / (1 + e^(2 |u|)).  The
// polynomials are minimax fits to erf, erfc e^(z^2 / 2) and tanh in double.  Largest error against 64 bits on the device, in 2^-24 of z / 2,
// beside that of erff's form (tanhf's is alike): z in -8 .. -4 0.00 and 0.50, -4 .. -2 0.26 and 0.76, -2 .. -1 1.4 and 1.6, -1 .. 0 1.5 and 1.7,
// 0 .. 1 3.0 and 3.3, 1 .. 8 3.2 and 4.1.
__device__ __forceinline__ float gelu_join(float z, float inner, float tail) { return z * (fabsf(z) < 1.0f ? fmaf(z, inner, 0.5f) : z < 0.0f ? tail : 1.0f - tail); }

__device__ __forceinline__ float gelu_erf_parts(float z) {
    const float q = z * z, t = __builtin_amdgcn_rcpf(fmaf(0.34f, fabsf(z), 1.0f));
    const float inner = fmaf(q, fmaf(q, fmaf(q, fmaf(q, fmaf(q, -7.530304e-06f, 1.13143644e-04f), -1.1859847e-03f), 9.973171e-03f), -6.649033e-02f), 0.3989423f);
    const float tail = fmaf(t, fmaf(t, fmaf(t, fmaf(t, fmaf(t, -0.12013893f, 0.37782046f), -0.1036036f), 0.22889116f), 0.11511663f), 1.8795595e-03f);
    return gelu_join(z, inner, tail * __builtin_amdgcn_exp2f(-0.72134752044448170f * q));
}

__device__ __forceinline__ float gelu_tanh_parts(float z) {
    const float q = z * z, u = 0.79788456080286536f * fmaf(0.044715f * q, z, z);
    const float inner = fmaf(q, fmaf(q, fmaf(q, fmaf(q, fmaf(q, -7.0424426e-06f, 1.1754699e-04f), -1.2428056e-03f), 1.0201477e-02f), -6.681947e-02f), 0.3989423f);
    return gelu_join(z, inner, __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(2.8853900817779268f * fabsf(u))));
}

// What stands between a sum and its store, fixed when a kernel is built: a tile's store is unrolled many times, and code
// that a call does not need costs instruction fetches in all of them.  PLAIN: the activation NONE; ERF: GELU_ERF; BIAS: a
// bias; PAIRS: SILU_PAIRS; FULL: bias, any activation, the token's own multiplier.
enum DenseEpilogue : int { DE_PLAIN, DE_ERF, DE_BIAS, DE_PAIRS, DE_FULL };

// PARTS: the forms for tiles, in 16-bit contexts.
template <bool PARTS>
__device__ __forceinline__ float dense_activate(int activation, float v) {
    if (activation == NVMAI_LINEAR_GELU_ERF) return PARTS ? gelu_erf_parts(v) : gelu_erf(v);
    if (activation == NVMAI_LINEAR_GELU_TANH) return PARTS ? gelu_tanh_parts(v) : gelu_tanh(v);
    return v;
}

template <int EPI, bool PARTS>
__device__ __forceinline__ float dense_finish(const DenseLinearParams& p, uint32_t t, uint32_t r, float v) {
    if (EPI == DE_ERF) return dense_activate<PARTS>(NVMAI_LINEAR_GELU_ERF, v);
    if (EPI == DE_BIAS) return v + bf16_to_f32(p.bias[r]);
    if (EPI != DE_FULL) return v;
    if (p.bias) v += bf16_to_f32(p.bias[r]);
    v = dense_activate<PARTS>(p.activation, v);
    if (p.mul) {                                     // an id past the table: zero
        const uint32_t id = p.mul_ids[t];
        v *= id < p.mul_rows ? bf16_to_f32(p.mul[(size_t)id * p.mul_stride + r]) : 0.0f;
    }
    return v;
}

// The biases of four neighbouring rows (r0 a multiple of 4; past the matrix: what is there is not used).
template <int EPI>
__device__ __forceinline__ dn_f4 dense_bias4(const DenseLinearParams& p, uint32_t r0) {
    dn_f4 b{0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (EPI == DE_BIAS || EPI == DE_FULL) {
        if (p.bias && r0 + 4u <= p.n)
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = bf16_to_f32(p.bias[r0 + j]);
    }
    return b;
}

// dense_finish of four neighbouring rows whose biases the caller holds.
template <int EPI, bool PARTS>
__device__ __forceinline__ dn_f4 dense_finish4(const DenseLinearParams& p, uint32_t t, uint32_t r0, dn_f4 v, dn_f4 bias) {
    if constexpr (EPI == DE_FULL) {
        dn_f4 m{1.0f, 1.0f, 1.0f, 1.0f};
        if (p.mul) {
            const uint32_t id = p.mul_ids[t];
            m = dn_f4{0.0f, 0.0f, 0.0f, 0.0f};
            if (id < p.mul_rows) {                   // an id past the table, which may have no row at all, reads nothing
                const uint16_t* at = p.mul + (size_t)id * p.mul_stride + r0;
                if ((reinterpret_cast<uintptr_t>(p.mul) & 7u) == 0 && (p.mul_stride & 3u) == 0) {
                    const uint2 q = *reinterpret_cast<const uint2*>(at);
                    m = dn_f4{__uint_as_float(q.x << 16), __uint_as_float(q.x & 0xFFFF0000u), __uint_as_float(q.y << 16), __uint_as_float(q.y & 0xFFFF0000u)};
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) m[j] = bf16_to_f32(at[j]);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = dense_activate<PARTS>(p.activation, v[j] + bias[j]) * m[j];
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = EPI == DE_ERF ? dense_activate<PARTS>(NVMAI_LINEAR_GELU_ERF, v[j]) : EPI == DE_BIAS ? v[j] + bias[j] : v[j];
    }
    return v;
}

template <int ACT>
__device__ __forceinline__ void dense_put(const DenseLinearParams& p, uint32_t t, uint32_t r, float v) {
    if (p.y) static_cast<act_t<ACT>*>(p.y)[(size_t)t * p.y_stride + r] = f32_to_act<ACT>(v);
    if (p.y_f32) p.y_f32[(size_t)t * p.y_stride + r] = v;
}

template <int EPI, int ACT, bool PARTS = false>
__device__ __forceinline__ void dense_store(const DenseLinearParams& p, uint32_t t, uint32_t r, float v) {
    dense_put<ACT>(p, t, r, dense_finish<EPI, PARTS>(p, t, r, v));
}

// Rows 2 j and 2 j + 1 of the matrix make output j: silu(gate) * up.
template <int ACT>
__device__ __forceinline__ float dense_pair(float gate, float up) { return (ACT == ACT_FP32 ? silu(gate) : silu_fast(gate)) * up; }

// Four neighbouring outputs of one token (r0 a multiple of 4).
template <int EPI, int ACT, bool PARTS = false>
__device__ __forceinline__ void dense_store4(const DenseLinearParams& p, uint32_t t, uint32_t r0, dn_f4 v, dn_f4 bias) {
    if (EPI == DE_PAIRS) {                           // n and the row stride are even
        const float a = dense_pair<ACT>(v[0], v[1]), b = dense_pair<ACT>(v[2], v[3]);
        if (r0 + 4u <= p.n) {
            if (p.y) {
                act_t<ACT>* y = static_cast<act_t<ACT>*>(p.y) + (size_t)t * p.y_stride + r0 / 2u;
                if constexpr (ACT == ACT_FP32) *reinterpret_cast<float2*>(y) = float2{a, b};
                else *reinterpret_cast<uint32_t*>(y) = f32_to_bf16(a) | ((uint32_t)f32_to_bf16(b) << 16);
            }
            if (p.y_f32) *reinterpret_cast<float2*>(p.y_f32 + (size_t)t * p.y_stride + r0 / 2u) = float2{a, b};
        } else if (r0 < p.n) {
            dense_put<ACT>(p, t, r0 / 2u, a);
        }
    } else if (r0 + 4u <= p.n && (p.y_stride & 3u) == 0 && !(EPI == DE_PLAIN && p.loose)) {
        v = dense_finish4<EPI, PARTS>(p, t, r0, v, bias);
        if (p.y) {
            act_t<ACT>* y = static_cast<act_t<ACT>*>(p.y) + (size_t)t * p.y_stride + r0;
            if constexpr (ACT == ACT_FP32) {
                *reinterpret_cast<dn_f4*>(y) = v;
            } else {
                uint2 q;
                q.x = f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16);
                q.y = f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16);
                *reinterpret_cast<uint2*>(y) = q;
            }
        }
        if (p.y_f32) *reinterpret_cast<dn_f4*>(p.y_f32 + (size_t)t * p.y_stride + r0) = v;
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (r0 + j < p.n) dense_store<EPI, ACT, PARTS>(p, t, r0 + j, v[j]);
    }
}

// The same as planes (n a multiple of 4).
template <int EPI>
__device__ __forceinline__ void dense_store_planes(const DenseLinearParams& p, uint32_t t, uint32_t r0, dn_f4 v, dn_f4 bias) {
    uint16_t* const row = static_cast<uint16_t*>(p.y) + (size_t)t * p.y_stride;
    if constexpr (EPI == DE_PAIRS) {
        const float out[2] = {dense_pair<ACT_FP32>(v[0], v[1]), dense_pair<ACT_FP32>(v[2], v[3])};
        planes_put<2>(row, p.y_k, r0 / 2u, out);
    } else {
        v = dense_finish4<EPI, false>(p, t, r0, v, bias);
        const float out[4] = {v[0], v[1], v[2], v[3]};
        planes_put<4>(row, p.y_k, r0, out);
    }
}

// ---- 1 .. 4 input rows: a wave owns RW weight rows, its lanes split k in 16-byte pieces -------------
// Bound by the matrix's bytes.  The inputs are read from L1 / L2 beside the weights (no LDS, no barrier): every
// load of a k step is independent of the others, so a wave has RW + NT (32-bit inputs: RW + 2 NT) 16-byte loads per lane
// in flight.
// U steps of 512 k whose loads are all issued before the first product.
template <int EPI, int ACT, int NT, int RW, int U>
__global__ __launch_bounds__(256) void dense_gemv_kernel(DenseLinearParams p) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t r0 = (blockIdx.x * 4u + wave) * RW;
    if (r0 >= p.n) return;
    const uint16_t* wp[RW];
#pragma unroll
    for (int r = 0; r < RW; ++r) wp[r] = p.w + (size_t)min(r0 + r, p.n - 1u) * p.w_stride;
    const act_t<ACT>* x = static_cast<const act_t<ACT>*>(p.x);
    float acc[NT][RW];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < RW; ++r) acc[t][r] = 0.0f;
    constexpr int XP = ACT == ACT_FP32 ? 2 : 1;
    for (uint32_t k0 = 0; k0 < p.k; k0 += 512u * U) {
        uint4 wv[U][RW], xv[U][NT][XP];
#pragma unroll
        for (int s = 0; s < U; ++s) {
            const uint32_t at = min(k0 + 512u * s + lane * 8u, p.k - 8u);        // past the end: the last piece, whose sums are dropped
#pragma unroll
            for (int r = 0; r < RW; ++r) wv[s][r] = *reinterpret_cast<const uint4*>(wp[r] + at);
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int u = 0; u < XP; ++u) xv[s][t][u] = reinterpret_cast<const uint4*>(x + (size_t)t * p.x_stride + at)[u];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < U; ++s) {
            const bool live = k0 + 512u * s + lane * 8u < p.k;
            float wf[RW][8];
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                const uint4 q = wv[s][r];
                act2_to_f32<ACT_BF16>(q.x, wf[r][0], wf[r][1]);
                act2_to_f32<ACT_BF16>(q.y, wf[r][2], wf[r][3]);
                act2_to_f32<ACT_BF16>(q.z, wf[r][4], wf[r][5]);
                act2_to_f32<ACT_BF16>(q.w, wf[r][6], wf[r][7]);
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                float xf[8];
                if constexpr (ACT == ACT_FP32) {
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        xf[4 * u] = __uint_as_float(xv[s][t][u].x); xf[4 * u + 1] = __uint_as_float(xv[s][t][u].y);
                        xf[4 * u + 2] = __uint_as_float(xv[s][t][u].z); xf[4 * u + 3] = __uint_as_float(xv[s][t][u].w);
                    }
                } else {
                    act2_to_f32<ACT_BF16>(xv[s][t][0].x, xf[0], xf[1]);
                    act2_to_f32<ACT_BF16>(xv[s][t][0].y, xf[2], xf[3]);
                    act2_to_f32<ACT_BF16>(xv[s][t][0].z, xf[4], xf[5]);
                    act2_to_f32<ACT_BF16>(xv[s][t][0].w, xf[6], xf[7]);
                }
#pragma unroll
                for (int r = 0; r < RW; ++r) {
                    float sum = acc[t][r];
#pragma unroll
                    for (int j = 0; j < 8; ++j) sum = fmaf(wf[r][j], xf[j], sum);
                    acc[t][r] = live ? sum : acc[t][r];
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        float v[RW];
#pragma unroll
        for (int r = 0; r < RW; ++r) v[r] = wave_sum_bcast(acc[t][r]);
#pragma unroll
        for (int r = 0; r < RW; r += EPI == DE_PAIRS ? 2 : 1) {
            if (lane != (uint32_t)(t * RW + r) || r0 + r >= p.n || (uint32_t)t >= p.rows) continue;
            if constexpr (EPI == DE_PAIRS) dense_put<ACT>(p, t, (r0 + r) / 2u, dense_pair<ACT>(v[r], v[r + 1]));
            else dense_store<EPI, ACT>(p, t, r0 + r, v[r]);
        }
    }
}

// ---- 1 or 2 input rows in 32 bits that are the end of a sublayer: x + RMS(delta) (add + w), then the product -------------------
// A block norms the rows once, four values of every 1024 per thread as norm_residual_kernel does (the same bits as the two launches), and hands them to its waves through LDS while their first weight rows are on
// their way; a wave keeps them in registers (k <= 512 S) and goes over `turns` times RW weight rows, the next ones requested before the
// current ones are multiplied.  The first block stores the sum.  (With each wave norming for itself and one weight row per wave the loads of x, delta and
// w, five times a weight row's, took the time: 16.1 us for 12,352 x 2048.)  Little longer than dense_gemv_kernel alone (cold weights: 10.6 us, 12.0 with the norm; 11,264
// rows in pairs 10.3 and 10.9; 256 rows 2.3 and 2.9): the norm's own launch, 3.0 us, is saved.
template <int EPI, int NT, int RW, int S>
__global__ __launch_bounds__(256) void dense_gemv_rms_kernel(DenseLinearParams p, uint32_t turns) {
    __shared__ __attribute__((aligned(16))) float rows[NT][512 * S];
    __shared__ float part[NT][4];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t first = (blockIdx.x * 4u + wave) * turns * RW;
    const float* x = static_cast<const float*>(p.x);
    // this thread's values: 4 (tid + 256 u) .. + 3
    constexpr int P = S / 2;
    dn_f4 xv[NT][P], dv[NT][P];
    uint2 nv[P];
#pragma unroll
    for (int u = 0; u < P; ++u) {
        const uint32_t at = min(4u * tid + 1024u * u, p.k - 4u);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            dv[t][u] = *reinterpret_cast<const dn_f4*>(p.rms_delta + (size_t)t * p.rms_delta_stride + at);
            xv[t][u] = *reinterpret_cast<const dn_f4*>(x + (size_t)t * p.x_stride + at);
        }
        nv[u] = *reinterpret_cast<const uint2*>(p.rms_w + at);
    }
    uint4 wv[S][RW];
    auto fetch = [&](uint32_t r0) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const uint32_t at = min(512u * s + lane * 8u, p.k - 8u);         // past the end: the last piece, which meets zeros
#pragma unroll
            for (int r = 0; r < RW; ++r) wv[s][r] = *reinterpret_cast<const uint4*>(p.w + (size_t)min(r0 + r, p.n - 1u) * p.w_stride + at);
        }
    };
    fetch(first);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        float q = 0.0f;
#pragma unroll
        for (int u = 0; u < P; ++u)
            if (4u * tid + 1024u * u < p.k)
#pragma unroll
                for (int e = 0; e < 4; ++e) q = fmaf(dv[t][u][e], dv[t][u][e], q);
        const float sum = wave_sum_bcast(q);
        if (lane == 0) part[t][wave] = sum;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < P; ++u) {
        const uint32_t at = 4u * tid + 1024u * u;
        const bool own = at < p.k;
        float nw[4];
        act2_to_f32<ACT_BF16>(nv[u].x, nw[0], nw[1]);
        act2_to_f32<ACT_BF16>(nv[u].y, nw[2], nw[3]);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const float inv = 1.0f / sqrtf(((part[t][0] + part[t][1]) + (part[t][2] + part[t][3])) / (float)p.k + p.rms_eps);
#pragma unroll
            for (int e = 0; e < 4; ++e) xv[t][u][e] += dv[t][u][e] * inv * (nw[e] + p.rms_add);
            if (own && blockIdx.x == 0) *reinterpret_cast<dn_f4*>(p.rms_out + (size_t)t * p.rms_out_stride + at) = xv[t][u];
            *reinterpret_cast<dn_f4*>(rows[t] + at) = own ? xv[t][u] : dn_f4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    __syncthreads();
    dn_f4 in[S][NT][2];
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int u = 0; u < 2; ++u) in[s][t][u] = reinterpret_cast<const dn_f4*>(rows[t] + 512u * s + lane * 8u)[u];
    for (uint32_t turn = 0; turn < turns; ++turn) {
        const uint32_t r0 = first + turn * RW;
        if (r0 >= p.n) return;
        uint4 cur[S][RW];
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int r = 0; r < RW; ++r) cur[s][r] = wv[s][r];
        if (turn + 1u < turns) fetch(r0 + RW);
        float acc[NT][RW];
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < RW; ++r) acc[t][r] = 0.0f;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const bool live = 512u * s + lane * 8u < p.k;
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                const uint4 q = live ? cur[s][r] : make_uint4(0u, 0u, 0u, 0u);
                float wf[8];
                act2_to_f32<ACT_BF16>(q.x, wf[0], wf[1]);
                act2_to_f32<ACT_BF16>(q.y, wf[2], wf[3]);
                act2_to_f32<ACT_BF16>(q.z, wf[4], wf[5]);
                act2_to_f32<ACT_BF16>(q.w, wf[6], wf[7]);
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int e = 0; e < 8; ++e) acc[t][r] = fmaf(wf[e], in[s][t][e >> 2][e & 3], acc[t][r]);
            }
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            float v[RW];
#pragma unroll
            for (int r = 0; r < RW; ++r) v[r] = wave_sum_bcast(acc[t][r]);
#pragma unroll
            for (int r = 0; r < RW; r += EPI == DE_PAIRS ? 2 : 1) {
                if (lane != (uint32_t)(t * RW + r) || r0 + r >= p.n) continue;
                if constexpr (EPI == DE_PAIRS) dense_put<ACT_FP32>(p, t, (r0 + r) / 2u, dense_pair<ACT_FP32>(v[r], v[r + 1]));
                else dense_store<EPI, ACT_FP32>(p, t, r0 + r, v[r]);
            }
        }
    }
}

// Every read of LDS done, all but the last N requests landed, for every wave of the block.
template <int N>
__device__ __forceinline__ void dense_stage_barrier() {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"i"(N) : "memory");
    __builtin_amdgcn_sched_barrier(0);
#endif
}

// All but this wave's last N requests have landed.
template <int N>
__device__ __forceinline__ void dense_landed() {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
    __builtin_amdgcn_sched_barrier(0);
#endif
}

// This wave's reads of LDS are done.
__device__ __forceinline__ void dense_read() {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#endif
}

// ---- 5 .. 64 input rows: 16 NR weight rows per block (HALF: eight), the waves split k, MFMA, sums through LDS ---------
// Steps of 64 k go round the NW waves, and every wave has a ring of S steps of its own in LDS: weights and inputs are requested in whole
// lines of 128 bytes and read back as operands (no barrier: a wave waits for its own requests alone).  Requested as operands, which is
// sixteen rows by lane, a load costs the address unit a cycle per lane, and that was what it took.  16 rows, cold weights, against sixteen
// and fewer waves that did: 2048 x 8192 18.6 -> 11.6 us, 8192 x 2048 11.5 -> 10.3, 2048 x 2048 6.1 -> 4.8, 1024 x 4096 10.3 -> 6.3, 49,664 x 2048 57 -> 48 (4.3 TB/s).  A line's pieces of 16 bytes lie in the order piece ^ skinny_swizzle(row): the sixteen lanes that a read serves at once cover 256
// bytes.  Stages are arrays of their own, so that a read does not wait for the requests behind it.
// An output is the sum of P = NW V partial sums: step s goes to the (s mod P)th, a wave's V of them in accumulators of its own, and they are added in
// order.  P is the launch's rule of n and k alone (skinny_sums), so that neither the waves nor the rows of a block change a bit; with
// one chain of products per wave the sums were up to 2.9 times as far from those in 64 bits (2048 x 8192, 17 rows 4.0e-7 and 1.5e-7), at 0 to 10 % less time.
constexpr int skinny_stages(int tt, int nr, int nw) {
    return nw * (nr + tt) * 2048 * 4 <= 128 * 1024 ? 4 : nw * (nr + tt) * 2048 * 3 <= 144 * 1024 ? 3 : 2;
}

// Partial sums of an output: chains of at most sixteen products up to 8192 k; many weight rows, four chains.
inline uint32_t skinny_sums(uint32_t n, uint32_t k) { return n >= 8192 || k <= 1024 ? 4 : k <= 2048 ? 8 : 16; }

// A lane's operand is the pieces 2 g and 2 g + 1 of row i; a read serves the rows 0 .. 3 and 12 .. 15 of one g with 4 .. 11 of the next at once, or sixteen rows
// of one: pairs of rows in the order 0 1 4 5 6 7 2 3 cover eight pieces either way.
__device__ __forceinline__ uint32_t skinny_swizzle(uint32_t row) { return (0x32765410u >> (row >> 1 << 2)) & 7u; }

// The threads that the compiler is told of: 512 leave a wave 256 registers, where the sums need no copies between the two halves of the register file
// (256 x 2048, 33 rows 7.2 us, 6.1 so; 2048 x 1536 6.5 and 5.6).  The largest sums are faster with them (6144 x 5632, 33 rows 29.1 and 31.3).
constexpr int skinny_threads(int tt, int nw, int v) { return tt * v >= 32 ? 64 * nw : 512; }

template <int EPI, int TT, int NR, int NW, int V, bool HALF = false>
__global__ __launch_bounds__(skinny_threads(TT, NW, V)) void dense_skinny_kernel(DenseLinearParams p) {
    static_assert(!HALF || NR == 1, "eight weight rows, the operand's other eight repeat them");
    constexpr int S = skinny_stages(TT, NR, NW), LW = HALF ? 1 : 2 * NR, L = LW + 2 * TT;      // 1 KB requests per step
    constexpr int U = S > V ? S : V;                         // steps of a turn round both the ring and the sums
    constexpr uint32_t STEP = L * 1024u, SUMS = NW * TT * NR * 1024u;
    static_assert(U % S == 0 && U % V == 0 && SUMS * ((V + S - 1) / S) <= NW * STEP, "the stages hold the sums");
    __shared__ __attribute__((aligned(1024))) uint8_t l0[NW * STEP], l1[NW * STEP], l2[S > 2 ? NW * STEP : 16], l3[S > 3 ? NW * STEP : 16];
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i = lane & 15u, g = lane >> 4;
    const uint32_t r0 = blockIdx.x * (HALF ? 8u : 16u * NR);
    const uint32_t steps = p.k / 64u, count = steps > wave ? (steps - wave + NW - 1u) / NW : 0u;
    [[maybe_unused]] const uint32_t w_bytes = (p.n - 1u) * p.w_stride * 2u + p.k * 2u, x_bytes = (p.rows - 1u) * p.x_stride * 2u + p.k * 2u;
    auto buf = [&](int j) -> uint8_t* { return (j == 0 ? l0 : j == 1 ? l1 : j == 2 ? l2 : l3) + wave * STEP; };
    // request q: rows 8 q .. 8 q + 7 of the weights' 16 NR, then of the inputs' 16 TT (rows past the last: the last one, whose sums are not stored)
    const uint32_t lr = lane >> 3;
    uint32_t off[L];
#pragma unroll
    for (int q = 0; q < L; ++q) {
        const uint32_t row = 8u * (q < LW ? q : q - LW) + lr, piece = ((lane & 7u) ^ skinny_swizzle(row & 15u)) * 16u;
        off[q] = (q < LW ? min(r0 + row, p.n - 1u) * p.w_stride : min(row, p.rows - 1u) * p.x_stride) * 2u + piece;
    }
    auto request = [&](uint32_t nth, int j) {
#if defined(__HIP_DEVICE_COMPILE__)     // the host pass rejects the 16-byte form of the load
        const bool live = nth < count;                       // a step past the last reads no bytes
        const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.w), 0, live ? (int)w_bytes : 0, 0x00020000);
        const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.x), 0, live ? (int)x_bytes : 0, 0x00020000);
        const uint32_t k = (wave + nth * NW) * 128u;
#pragma unroll
        for (int q = 0; q < L; ++q)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(q < LW ? wr : xr, (__attribute__((address_space(3))) void*)(buf(j) + q * 1024u), 16, off[q], k, 0, 0);
#endif
    };
    const uint32_t at0 = i * 128u + (((2u * g) ^ skinny_swizzle(i)) * 16u), at1 = at0 ^ 16u;
    [[maybe_unused]] const uint32_t half0 = (i & 7u) * 128u + (((2u * g) ^ skinny_swizzle(i & 7u)) * 16u), half1 = half0 ^ 16u;
    dn_f4 acc[V][NR][TT];
#pragma unroll
    for (int v = 0; v < V; ++v)
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
            for (int t = 0; t < TT; ++t) acc[v][r][t] = dn_f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < S; ++j) request(j, j);
    auto step = [&](uint32_t nth, int n) {                   // nth % U = n
        const int j = n % S, v = n % V;
        dense_landed<(S - 1) * L>();
        uint4 a[NR][2], b[TT][2];
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            a[r][0] = *reinterpret_cast<const uint4*>(buf(j) + 2048u * r + (HALF ? half0 : at0));
            a[r][1] = *reinterpret_cast<const uint4*>(buf(j) + 2048u * r + (HALF ? half1 : at1));
        }
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            b[t][0] = *reinterpret_cast<const uint4*>(buf(j) + 1024u * LW + 2048u * t + at0);
            b[t][1] = *reinterpret_cast<const uint4*>(buf(j) + 1024u * LW + 2048u * t + at1);
        }
        dense_read();                                        // the operands are in registers: the place is free
        request(nth + S, j);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int r = 0; r < NR; ++r)
#pragma unroll
                for (int t = 0; t < TT; ++t) acc[v][r][t] = dn_mfma(a[r][h], b[t][h], acc[v][r][t]);
    };
    uint32_t nth = 0;
    for (; nth + (uint32_t)U <= count; nth += U) {
#pragma unroll
        for (int n = 0; n < U; ++n) step(nth + n, n);
    }
#pragma unroll
    for (int n = 0; n < U - 1; ++n)
        if (nth + (uint32_t)n < count) step(nth + n, n);
    dense_stage_barrier<0>();                                // no request outlives its wave, and no other wave reads its places any more
    // The waves take the tiles of the sums in turn: part(v, w, at) is wave w's v-th sum of tile at, which is for another wave.
    auto part = [&](int v, int w, int at) {
        return reinterpret_cast<dn_f4*>((v % S == 0 ? l0 : v % S == 1 ? l1 : v % S == 2 ? l2 : l3) + v / S * SUMS + (w * NR * TT + at) * 1024u) + lane;
    };
#pragma unroll
    for (int v = 0; v < V; ++v)
#pragma unroll
        for (int at = 0; at < NR * TT; ++at)
            if (at % NW != (int)wave) *part(v, (int)wave, at) = acc[v][at / TT][at % TT];
    __syncthreads();
#pragma unroll
    for (int at = 0; at < NR * TT; ++at) {
        const int r = at / TT, t = at % TT;
        if (at % NW != (int)wave) continue;
        dn_f4 sum;
#pragma unroll
        for (int v = 0; v < V; ++v)
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const dn_f4 add = w == at % NW ? acc[v][r][t] : *part(v, w, at);
                sum = v + w == 0 ? add : sum + add;
            }
        // sum[j] = y[token 16 t + i, row r0 + 16 r + 4 g + j]
        if (16u * t + i < p.rows && (!HALF || g < 2u)) dense_store4<EPI, ACT_BF16>(p, 16u * t + i, r0 + 16u * r + 4u * g, sum, dense_bias4<EPI>(p, r0 + 16u * r + 4u * g));
    }
}

// ---- many input rows: tiles of BN weight rows x BM tokens, k in steps of 64 through a ring of S stages in LDS ----------
// Four waves, each a quarter of the tile (BN / 2 x BM / 2) in 16 x 16 x 32 products.  Bound by the rate at which a compute
// unit takes operands into LDS (about 60 bytes per ns; a tile of 256 x 256 is where the products take as long), below
// one tile per compute unit by the latency of a step, and where all units multiply by the clock that the card's power leaves.  A tile's rows are 128 bytes
// of LDS, whose eight 16-byte pieces lie in the order piece ^ tile_swizzle(row).  An operand is four pieces in a row, and a product adds them in their order:
// the bits of 32 x 32 x 16 products one after another, whatever the tile.
//   Which products, and in which order, is a matter of power.  From registers alone, random values, all units: 32 x 32 x 16 1,750 TFLOP/s,
// 16 x 16 x 32 with the first operand held for runs and the second going to and fro 2,070, in any order that changes the first each time 1,570 to 1,750.
// With 32 x 32 x 16 these kernels also left the clock of whatever ran next 13 % lower (a router product of 58 us took 66 beside them; 59 now).
// Cold weights, one call after another: 2048 x 2048 x 2048 23.7 -> 22.8 us, in the tiles of 256 x 256 below 4096 x 12,288 x 2048 179 -> 170 and 8192 x 8192 x 8192 769 -> 718.
//   A stage is multiplied in four phases, half of the weight rows by 32 k each.  The operands of the phases after the next one are read, and a quarter of a
// stage ahead is requested, between the products of a phase: a wave alone on its SIMD has products to issue at all times, and
// requests spread over the phases keep the wave from waiting at the memory pipe (in one burst behind the barrier: 96 us for
// 2048 x 2048 x 8192 in tiles of 256 x 128, spread 93, and 125 with a branch around the burst).  One barrier per stage,
// in its middle: by then every wave has read the stage to its end (its place is free for stage + S) and waits for
// its own part of the next one.  Requests are never conditional, so the counter's meaning is the same in every step; a
// stage past the last reads no bytes (a buffer of size 0).  Stages are separate arrays: the compiler then knows
// which requests a read of LDS has to wait for.
//   32-bit activations come as three BF16 planes (dense_split), [row][plane][k], the smallest first: the products of a step
// of 64 k are exact, and their sum goes to a running total of its own, which keeps the rounding of a long k small.
// Measured (tiles of 128 x 128 x 64 in two stages before): 2048 x 8192 x 2048 77 -> 64 us, 2048 x 2048 x 8192 140 -> 67, 1501 x
// 2048 x 2048 34 -> 17, 512 x 2048 x 2048 33 -> 9.5 (rows x n x k, cold weights).
// A read serves the rows 0 .. 3 and 12 .. 15 of one g with 4 .. 11 of the next at once, or sixteen rows of one: pairs of rows in their own order cover eight
// pieces either way where neighbouring g read neighbouring pieces.
__device__ __forceinline__ uint32_t tile_swizzle(uint32_t row) { return (row >> 1) & 7u; }

// One sum of the planes again by a whole wave, in fp32 multiply-adds of the values that the planes stand for.  An infinite weight makes
// NaN of a value's lower planes where they are zero, and planes of sums that overflow can cancel: a NaN comes from here or not
// at all.  It ends where the sum has become NaN, which it stays; poisoned: by an input that is NaN, so that all sums of its row are.
__device__ __forceinline__ float dense_sum_again(const DenseLinearParams& p, uint32_t t, uint32_t r, bool& poisoned) {
    const uint16_t *w = p.w + (size_t)r * p.w_stride, *x = static_cast<const uint16_t*>(p.x) + (size_t)t * p.x_stride;
    const uint32_t lane = threadIdx.x & 63u;
    float sum = 0.0f;
    bool none = false;
#pragma unroll 1
    for (uint32_t k0 = 0; k0 < p.k; k0 += 512u) {
        const uint32_t k = k0 + lane * 8u;
        if (k < p.k) {
            const uint4 a = *reinterpret_cast<const uint4*>(w + k), lo = *reinterpret_cast<const uint4*>(x + k),
                        mid = *reinterpret_cast<const uint4*>(x + p.k + k), hi = *reinterpret_cast<const uint4*>(x + 2u * p.k + k);
            const uint32_t av[4] = {a.x, a.y, a.z, a.w}, lv[4] = {lo.x, lo.y, lo.z, lo.w}, mv[4] = {mid.x, mid.y, mid.z, mid.w}, hv[4] = {hi.x, hi.y, hi.z, hi.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                auto part = [&](const uint32_t* v) { return bf16_to_f32((uint16_t)(v[e / 2] >> (16 * (e & 1)))); };
                const float value = (part(hv) + part(mv)) + part(lv);
                none |= value != value;
                sum = fmaf(part(av), value, sum);
            }
        }
        if (__any(sum != sum)) break;
    }
    poisoned = __any(none);
    return wave_sum_bcast(sum);
}

// Which tile a block takes, and which part of its k.
struct DenseTileAt {
    uint32_t m, n, tile, part;
};

__device__ __forceinline__ DenseTileAt dense_tile_at(uint32_t tiles_n, uint32_t tiles_m, uint32_t parts = 1) {
    // blocks are dealt to the eight XCDs in turn: give each XCD a run of neighbouring tiles (shared L2 lines); parts of k
    // outermost, so that an XCD reads as little of both operands as can be
    const uint32_t tiles = tiles_n * tiles_m, all = tiles * parts, xcd = blockIdx.x & 7u, nth = blockIdx.x >> 3;
    const uint32_t base = all / 8u, extra = all % 8u;
    uint32_t tile = xcd * base + min(xcd, extra) + nth, part = 0;
    if (parts > 1u) {                                        // a division that a launch without parts is spared
        part = tile / tiles;
        tile -= part * tiles;
    }
    // in bands of eight token tiles, weight tiles outermost within the band
    const uint32_t band = tile / (8u * tiles_n), in_band = tile % (8u * tiles_n);
    const uint32_t band_m = min(8u, tiles_m - band * 8u);
    return {band * 8u + in_band % band_m, in_band / band_m, tile, part};
}

// Tiles cut along k: `parts` blocks per tile, whose sums meet in `sums` (one tile of floats per block).  tickets: a zeroed word per tile.
struct DenseCut {
    uint32_t parts;
    float* sums;
    uint32_t* tickets;
};

constexpr int COHERENT = 16;                                 // sc1: a store goes through this XCD's L2, a load does not stop at it

// A block's sums of a tile go to memory, and the block that ends last takes all of them back and adds them in the order of k.  Nobody waits: a
// block that is not the last one has ended.  The stores are written through and have all arrived before the ticket is drawn (a release
// at device scope would write back everything that this XCD's L2 holds).  Returns whether this block holds the tile's sums.
template <int TN, int TM>
__device__ __forceinline__ bool dense_join(dn_f4 (&sum)[TN][TM], const DenseCut& cut, const DenseTileAt& at, uint32_t* shared) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr uint32_t WAVE = TN * TM * 1024u, TILE = 4u * WAVE;                    // bytes
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, own = wave * WAVE + lane * 16u;
    float* const sums = cut.sums + (size_t)at.tile * cut.parts * (TILE / 4u);
    const __amdgpu_buffer_rsrc_t all = __builtin_amdgcn_make_buffer_rsrc(sums, 0, (int)(cut.parts * TILE), 0x00020000);
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(dn_u4, sum[a][b]), all, own + (a * TM + b) * 1024u, at.part * TILE, COHERENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t before = __hip_atomic_fetch_add(cut.tickets + at.tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool last = before == cut.parts - 1u;
        if (last) __hip_atomic_store(cut.tickets + at.tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // ready for the next launch
        *shared = last;
    }
    __syncthreads();
    if (*shared == 0u) return false;
    __syncthreads();                                         // the word is read: its place is free
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) sum[a][b] = dn_f4{};
#pragma unroll 2
    for (uint32_t part = 0; part < cut.parts; ++part) {
        dn_f4 q[TN][TM];
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int b = 0; b < TM; ++b)
                q[a][b] = __builtin_bit_cast(dn_f4, __builtin_amdgcn_raw_buffer_load_b128(all, own + (a * TM + b) * 1024u, part * TILE, COHERENT));
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int b = 0; b < TM; ++b) sum[a][b] += q[a][b];
    }
#endif
    return true;
}

// Of 160 KB, one block per compute unit; 64 x 64 tiles of 16-bit inputs fit twice.  Planes come in threes: six stages where they fit
// (64 x 64, 700 x 1024 x 1024 in 32 bits: 17.4 us with three, 13.5 with six).
constexpr int dense_stages(int act, int bn, int bm) {
    return act == ACT_FP32 ? (bn + bm <= 192 ? 6 : 3) : bn + bm <= 192 ? 5 : bn + bm <= 256 ? 4 : 3;
}

constexpr int dense_blocks(int act, int bn, int bm) { return 2 * dense_stages(act, bn, bm) * (bn + bm) * 128 <= 160 * 1024 ? 2 : 1; }

template <int EPI, int ACT, int BN, int BM>
__global__ __launch_bounds__(256, dense_blocks(ACT, BN, BM)) void dense_tile_kernel(DenseLinearParams p, uint32_t tiles_n, uint32_t tiles_m, DenseCut cut) {
    constexpr bool SPLIT = ACT == ACT_FP32;
    constexpr int S = dense_stages(ACT, BN, BM);
    constexpr int LA = BN / 32, LB = BM / 32, L = LA + LB;   // 1 KB requests per wave and stage
    constexpr int TN = BN / 32, TM = BM / 32;                // 16 x 16 tiles per wave
    constexpr uint32_t STAGE = (BN + BM) * 128u;
    __shared__ __attribute__((aligned(1024))) uint8_t l0[STAGE], l1[STAGE], l2[STAGE], l3[S > 3 ? STAGE : 16], l4[S > 4 ? STAGE : 16], l5[S > 5 ? STAGE : 16];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const DenseTileAt at = dense_tile_at(tiles_n, tiles_m, cut.parts);
    const uint32_t m0 = at.m * BM, n0 = at.n * BN;

    // the part's first 64 k and how many: all of them, or an even share
    uint32_t first = 0, steps = p.k / 64u;
    if (cut.parts > 1u) {
        const uint32_t all = steps;
        first = all * at.part / cut.parts;
        steps = all * (at.part + 1u) / cut.parts - first;
    }
    if (SPLIT) steps *= 3u;
    [[maybe_unused]] const uint32_t w_bytes = (p.n - 1u) * p.w_stride * 2u + p.k * 2u;
    [[maybe_unused]] const uint32_t x_bytes = (p.rows - 1u) * p.x_stride * 2u + p.k * (SPLIT ? 6u : 2u);
    const uint32_t lr = lane >> 3;
    // request r of a wave: rows 8 r .. 8 r + 7 of its part (8 r + lane / 8 has two values of the swizzle)
    [[maybe_unused]] const uint32_t piece[2] = {((lane & 7u) ^ tile_swizzle(lr)) * 16u, ((lane & 7u) ^ tile_swizzle(lr + 8u)) * 16u};
    // rows past the last: the last one, whose sums are not stored
    [[maybe_unused]] const uint32_t a8 = p.w_stride * 16u, a0 = (n0 + wave * (LA * 8u) + lr) * p.w_stride * 2u, amax = (p.n - 1u) * p.w_stride * 2u;
    [[maybe_unused]] const uint32_t b8 = p.x_stride * 16u, b0 = (m0 + wave * (LB * 8u) + lr) * p.x_stride * 2u, bmax = (p.rows - 1u) * p.x_stride * 2u;
    auto buf = [&](int j) -> uint8_t* { return j == 0 ? l0 : j == 1 ? l1 : j == 2 ? l2 : j == 3 ? l3 : j == 4 ? l4 : l5; };
    // requests [from, to) of stage st into its place j = st % S (of a 32-bit input: plane j % 3, S is 3 or 6)
    auto request = [&](uint32_t st, int j, int from, int to) {
#if defined(__HIP_DEVICE_COMPILE__)     // the host pass rejects the 16-byte form of the load
        const bool live = st < steps;
        const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.w), 0, live ? (int)w_bytes : 0, 0x00020000);
        const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.x), 0, live ? (int)x_bytes : 0, 0x00020000);
        const uint32_t wk = (first + (SPLIT ? st / 3u : st)) * 128u, xk = SPLIT ? wk + j % 3 * p.k * 2u : wk;
        uint8_t* dst = buf(j);
#pragma unroll
        for (int r = 0; r < L; ++r) {
            if (r < from || r >= to) continue;
            if (r < LA) __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (__attribute__((address_space(3))) void*)(dst + (wave * LA + r) * 1024u), 16, min(a0 + r * a8, amax) + piece[r & 1], wk, 0, 0);
            else __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (__attribute__((address_space(3))) void*)(dst + BN * 128u + (wave * LB + r - LA) * 1024u), 16, min(b0 + (r - LA) * b8, bmax) + piece[(r - LA) & 1], xk, 0, 0);
        }
#endif
    };
    const uint32_t i = lane & 15u, g = lane >> 4;
    const uint32_t wn = (wave >> 1) * (BN / 2), wm = (wave & 1u) * (BM / 2);
    const uint32_t arow = (wn + i) * 128u, brow = BN * 128u + (wm + i) * 128u;
    uint4 fa[2][TN], fb[2][TM];
    // operands of the half h (32 k: the pieces 4 h + g) of the stage at place j: the tokens' and the first half of the weights' (part 0), the rest (part 1)
    auto fetch = [&](int j, int h, int part) {
        const uint32_t sw = ((4u * h + g) ^ tile_swizzle(i)) * 16u;
        if (part == 0) {
#pragma unroll
            for (int b = 0; b < TM; ++b) fb[h][b] = *reinterpret_cast<const uint4*>(buf(j) + brow + 2048u * b + sw);
        }
#pragma unroll
        for (int a = part * (TN / 2); a < (part + 1) * (TN / 2); ++a) fa[h][a] = *reinterpret_cast<const uint4*>(buf(j) + arow + 2048u * a + sw);
    };
    dn_f4 acc[TN][TM];
    [[maybe_unused]] dn_f4 total[SPLIT ? TN : 1][SPLIT ? TM : 1];
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) {
            acc[a][b] = dn_f4{};
            if constexpr (SPLIT) total[a][b] = dn_f4{};
        }
    // phase q: half q / 2 of the stage, the weights' half q % 2; a weight operand stays for a run, a token operand from one run to the next
    auto multiply = [&](auto phase, auto requests, bool fresh) {
        constexpr int Q = decltype(phase)::value, H = Q / 2, NP = TN * TM / 2, NF = TN / 2 + (Q % 2 == 0 ? TM : 0), NR = decltype(requests)::value;
#pragma unroll
        for (int e = 0; e < NP; ++e) {
            const int a = Q % 2 * (TN / 2) + e / TM, b = a & 1 ? TM - 1 - e % TM : e % TM;
            acc[a][b] = dn_mfma(fa[H][a], fb[H][b], fresh ? dn_f4{} : acc[a][b]);
        }
#pragma unroll
        for (int k = 0; k < NP; ++k) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);                                     // a product,
            __builtin_amdgcn_sched_group_barrier(0x100, (NF + NP - 1) / NP, 0);                  // operands to come,
            if constexpr (NR > 0) __builtin_amdgcn_sched_group_barrier(0x20, (NR + NP - 1) / NP, 0);  // and the requests
        }
        __builtin_amdgcn_sched_barrier(0);
    };
#define NVMAI_SHARE(q) (L * (q) / 4)
#define NVMAI_SHARES(q) std::integral_constant<int, NVMAI_SHARE(q + 1) - NVMAI_SHARE(q)>{}
    constexpr std::integral_constant<int, 0> q0{};
    constexpr std::integral_constant<int, 1> q1{};
    constexpr std::integral_constant<int, 2> q2{};
    constexpr std::integral_constant<int, 3> q3{};
    auto step = [&](uint32_t st, int j) {
        constexpr int B = S - 1;
        fetch(j, 1, 0);
        request(st + B, (j + B) % S, NVMAI_SHARE(2), NVMAI_SHARE(3));
        multiply(q0, NVMAI_SHARES(2), SPLIT && j % 3 == 0);
        fetch(j, 1, 1);
        request(st + B, (j + B) % S, NVMAI_SHARE(3), NVMAI_SHARE(4));
        multiply(q1, NVMAI_SHARES(3), SPLIT && j % 3 == 0);
        dense_stage_barrier<(S - 2) * L>();
        fetch((j + 1) % S, 0, 0);
        request(st + S, j, NVMAI_SHARE(0), NVMAI_SHARE(1));
        multiply(q2, NVMAI_SHARES(0), false);
        fetch((j + 1) % S, 0, 1);
        request(st + S, j, NVMAI_SHARE(1), NVMAI_SHARE(2));
        multiply(q3, NVMAI_SHARES(1), false);
        if constexpr (SPLIT) {
            if (j % 3 == 2) {
#pragma unroll
                for (int a = 0; a < TN; ++a)
#pragma unroll
                    for (int b = 0; b < TM; ++b) total[a][b] += acc[a][b];
            }
        }
    };
#pragma unroll
    for (int j = 0; j < S; ++j) request(j, j, 0, j == S - 1 ? NVMAI_SHARE(2) : L);
    dense_stage_barrier<(S - 2) * L + NVMAI_SHARE(2)>();
#undef NVMAI_SHARES
#undef NVMAI_SHARE
    fetch(0, 0, 0);
    fetch(0, 0, 1);
    uint32_t st = 0;
    for (; st + (uint32_t)S <= steps; st += S) {
#pragma unroll
        for (int j = 0; j < S; ++j) step(st + j, j);
    }
#pragma unroll
    for (int j = 0; j < S - 1; ++j)
        if (st + (uint32_t)j < steps) step(st + j, j);
    dense_stage_barrier<0>();                                // no request outlives its block; the stages' places are free
    if (cut.parts > 1u) {
        if constexpr (SPLIT) {
            if (!dense_join<TN, TM>(total, cut, at, reinterpret_cast<uint32_t*>(l2))) return;
        } else {
            if (!dense_join<TN, TM>(acc, cut, at, reinterpret_cast<uint32_t*>(l2))) return;
        }
    }
    // The sums change places through LDS, 32 tokens of the wave's part at a time, so that neighbouring lanes hold
    // neighbouring outputs of one token (stores of whole lines) and what stands between sum and store is a short loop: unrolled
    // over the sums of a tile it is longer than the instruction cache (GELU on 256 x 128: 122 us instead of 71 for 2048 x 8192 x 2048).
    constexpr uint32_t ROWS = BN / 2, PITCH = ROWS + 4, PER = ROWS / 4, AT_ONCE = 64 / PER;
    constexpr int UNROLL = EPI == DE_ERF ? 2 : 4;
    float* turn = reinterpret_cast<float*>((wave & 1u) ? l1 : l0) + (wave >> 1) * (32u * PITCH);
    static_assert(2u * 32u * PITCH * 4u <= STAGE, "two waves per stage");
    const uint32_t r = n0 + wn + lane % PER * 4u;
    const dn_f4 bias = dense_bias4<EPI>(p, r);
#pragma unroll
    for (int b = 0; b < TM / 2; ++b) {
        [[maybe_unused]] bool again = false;
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int t = 0; t < 2; ++t) {                    // element e of a lane: row 4 g + e, token i
                dn_f4 v = acc[a][2 * b + t];
                if constexpr (SPLIT) v = total[a][2 * b + t];
                *reinterpret_cast<dn_f4*>(turn + (16 * t + i) * PITCH + 16 * a + 4u * g) = v;
                if constexpr (SPLIT) {
                    bool none = false;
#pragma unroll
                    for (int e = 0; e < 4; ++e) none |= v[e] != v[e];
                    again |= none;
                }
            }
        if constexpr (SPLIT) {
            if (__any(again)) {
                uint32_t poisoned_token = 32;                // sums of one token follow each other
                for (uint32_t e0 = 0; e0 < 32u * ROWS; e0 += 64u) {
                    const uint32_t own = e0 + lane;
                    const float old = turn[own / ROWS * PITCH + own % ROWS];
                    for (uint64_t left = __ballot(old != old); left != 0; left &= left - 1) {
                        const uint32_t e = e0 + (uint32_t)__builtin_ctzll(left), token = e / ROWS, t = m0 + wm + 32 * b + token, row = n0 + wn + e % ROWS;
                        if (token == poisoned_token || t >= p.rows || row >= p.n) continue;
                        bool poisoned;
                        const float sum = dense_sum_again(p, t, row, poisoned);
                        if (poisoned) poisoned_token = token;
                        else if (lane == 0) turn[token * PITCH + e % ROWS] = sum;
                    }
                }
            }
        }
#pragma unroll UNROLL
        for (uint32_t k = 0; k < 32u / AT_ONCE; ++k) {
            const uint32_t token = lane / PER + k * AT_ONCE, t = m0 + wm + 32 * b + token;
            const dn_f4 v = *reinterpret_cast<const dn_f4*>(turn + token * PITCH + lane % PER * 4u);
            if (t >= p.rows || r >= p.n) continue;
            if constexpr (SPLIT) {
                if (p.y_k) {
                    dense_store_planes<EPI>(p, t, r, v, bias);
                    continue;
                }
            }
            dense_store4<EPI, ACT, !SPLIT>(p, t, r, v, bias);
        }
    }
}

// ---- the same in tiles of 256 x 256, 16-bit activations --------------------------------------------------------------------
// Two stages of 64 KB are all that fits, and a ring that frees a stage as a whole leaves the last requests for the next one a quarter of a
// stage to arrive.  Here a stage is two halves of both operands (rows 0 .. 63 of every 128, and the others), freed and asked for one by one:
// a wave's part is four products of half by half, in the order (0, 0), (1, 0), (1, 1), (0, 1), so that the halves 0 are read while the
// last two products of the stage before run and the halves 1 during the first two; a half is then out of LDS for registers (128 of them hold a
// stage) one to one and a half stages before its successor is needed.  Barriers stand behind the first eight of the 32 matrix instructions of
// a product: the reads before them arrive in the meantime.  Requests go out evenly over the stage.  Bound by the rate of requests into LDS and the
// power of the products.  Rows x n x k, cold weights, 32 x 32 x 16 products and these: 4096 x 12,288 x 2048 179 and 170 us (1,210 TFLOP/s).
// Not kept: a third place for the halves 0 (no change), requests of 64 bytes per row in stages of 32 k (half
// the rate).
template <int EPI>
__global__ __launch_bounds__(256, 1) void dense_wide_kernel(DenseLinearParams p, uint32_t tiles_n, uint32_t tiles_m) {
    constexpr uint32_t HALF = 128u * 128u;
    // weights and tokens: place (stage % 2), half
    __shared__ __attribute__((aligned(1024))) uint8_t w00[HALF], w01[HALF], w10[HALF], w11[HALF], x00[HALF], x01[HALF], x10[HALF], x11[HALF];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const DenseTileAt at = dense_tile_at(tiles_n, tiles_m);
    const uint32_t m0 = at.m * 256u, n0 = at.n * 256u;
    const uint32_t steps = p.k / 64u;
    [[maybe_unused]] const uint32_t w_bytes = (p.n - 1u) * p.w_stride * 2u + p.k * 2u, x_bytes = (p.rows - 1u) * p.x_stride * 2u + p.k * 2u;
    // request r of a wave: rows 32 wave + 8 r .. + 7 of a half (8 r + lane / 8 has two values of the swizzle)
    const uint32_t lr = lane >> 3;
    [[maybe_unused]] const uint32_t piece[2] = {((lane & 7u) ^ tile_swizzle(lr)) * 16u, ((lane & 7u) ^ tile_swizzle(lr + 8u)) * 16u};
    const uint32_t row = (wave & 1u) * 32u + (wave >> 1) * 128u + lr;
    [[maybe_unused]] const uint32_t w8 = p.w_stride * 16u, w0 = (n0 + row) * p.w_stride * 2u, wmax = (p.n - 1u) * p.w_stride * 2u;
    [[maybe_unused]] const uint32_t x8 = p.x_stride * 16u, x0 = (m0 + row) * p.x_stride * 2u, xmax = (p.rows - 1u) * p.x_stride * 2u;
    auto wbuf = [&](int j, int h) -> uint8_t* { return j == 0 ? (h == 0 ? w00 : w01) : (h == 0 ? w10 : w11); };
    auto xbuf = [&](int j, int h) -> uint8_t* { return j == 0 ? (h == 0 ? x00 : x01) : (h == 0 ? x10 : x11); };
    // request q of eight (four of weights, four of tokens) of half h of stage st into its place j = st % 2
    auto request = [&](uint32_t st, int j, int h, int q) {
#if defined(__HIP_DEVICE_COMPILE__)     // the host pass rejects the 16-byte form of the load
        const bool live = st < steps;
        const uint32_t k = st * 128u, r = (uint32_t)q & 3u;
        if (q < 4) {
            const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.w), 0, live ? (int)w_bytes : 0, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (__attribute__((address_space(3))) void*)(wbuf(j, h) + (wave * 4u + r) * 1024u), 16, min(w0 + (8u * h + r) * w8, wmax) + piece[r & 1u], k, 0, 0);
        } else {
            const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.x), 0, live ? (int)x_bytes : 0, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (__attribute__((address_space(3))) void*)(xbuf(j, h) + (wave * 4u + r) * 1024u), 16, min(x0 + (8u * h + r) * x8, xmax) + piece[r & 1u], k, 0, 0);
        }
#endif
    };
    const uint32_t i = lane & 15u, g = lane >> 4;
    const uint32_t wn = (wave >> 1) * 128u, wm = (wave & 1u) * 128u;
    const uint32_t arow = ((wave >> 1) * 64u + i) * 128u, brow = ((wave & 1u) * 64u + i) * 128u;
    uint4 A[2][2][4], B[2][2][4];                            // [half][32 k][tile of 16]
    // operand e of eight of a half
    auto read_w = [&](int j, int h, int e) { A[h][e >> 2][e & 3] = *reinterpret_cast<const uint4*>(wbuf(j, h) + arow + 2048u * (e & 3) + (((4u * (e >> 2) + g) ^ tile_swizzle(i)) * 16u)); };
    auto read_x = [&](int j, int h, int e) { B[h][e >> 2][e & 3] = *reinterpret_cast<const uint4*>(xbuf(j, h) + brow + 2048u * (e & 3) + (((4u * (e >> 2) + g) ^ tile_swizzle(i)) * 16u)); };
    dn_f4 acc[8][8];
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
        for (int b = 0; b < 8; ++b) acc[a][b] = dn_f4{};
    // matrix instruction e of 32 of the product of two halves: a weight operand stays for four, a token operand from one four to the next
    auto multiply = [&](int ha, int hb, int e) {
        const int k = e >> 4, a = (e >> 2) & 3, b = a & 1 ? 3 - (e & 3) : e & 3;
        dn_mfma_in_place(A[ha][k][a], B[hb][k][b], acc[4 * ha + a][4 * hb + b]);
    };
    // The half products (h, h) and (1 - h, h): the halves 1 - of the weights, then of the tokens, are read under the first two, those of the
    // next stage under the last two, where the weights' half 0 is still an operand and is replaced behind its last use.
    auto stage = [&](uint32_t st, int j) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int next = h == 0 ? j : 1 - j;
#pragma unroll
            for (int e = 0; e < 8; ++e) multiply(h, h, e);
            __builtin_amdgcn_sched_barrier(0);
            dense_stage_barrier<16>();                       // two halves of both operands stay on their way
#pragma unroll
            for (int e = 8; e < 32; ++e) {
                multiply(h, h, e);
                if ((e & 1) == 0 && e < 24) {
                    if (h == 0) read_w(next, 1, (e - 8) / 2);
                    else read_x(next, 0, (e - 8) / 2);
                }
                if (e % 6 == 1) request(st + 2u, j, h, e / 6 - 2);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int e = 0; e < 32; ++e) {
                multiply(1 - h, h, e);
                if (h == 0) {
                    if ((e & 1) == 0 && e < 16) read_x(next, 1, e / 2);
                } else if ((e & 3) == 3) {
                    read_w(next, 0, e >> 2);
                }
                if (e % 8 == 2) request(st + 2u, j, h, 4 + e / 8);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int q = 0; q < 8; ++q) request(j, j, h, q);
    dense_stage_barrier<24>();
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        read_w(0, 0, e);
        read_x(0, 0, e);
    }
    uint32_t st = 0;
    for (; st + 2u <= steps; st += 2u) {
        stage(st, 0);
        stage(st + 1u, 1);
    }
    if (st < steps) stage(st, 0);
    dn_mfma_done();
    dense_stage_barrier<0>();                                // no request outlives its block; the places are free
    // The sums change places as in dense_tile_kernel, in a row of 128 per token whose pieces of four are exchanged by the token.
    float* turn = reinterpret_cast<float*>(wave == 0u ? w00 : wave == 1u ? w01 : wave == 2u ? w10 : w11);
    constexpr int UNROLL = EPI == DE_ERF ? 2 : 4;
    const uint32_t r = n0 + wn + lane % 32u * 4u;
    const dn_f4 bias = dense_bias4<EPI>(p, r);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
#pragma unroll
        for (int a = 0; a < 8; ++a)
#pragma unroll
            for (int h = 0; h < 2; ++h)                      // element e of a lane: row 4 g + e, token i
                *reinterpret_cast<dn_f4*>(turn + (16u * h + i) * 128u + (((4u * a + g) ^ (16u * h + i)) * 4u)) = acc[a][2 * b + h];
#pragma unroll UNROLL
        for (uint32_t k = 0; k < 16u; ++k) {
            const uint32_t token = lane / 32u + k * 2u, t = m0 + wm + 32 * b + token;
            const dn_f4 v = *reinterpret_cast<const dn_f4*>(turn + token * 128u + ((lane % 32u) ^ token) * 4u);
            if (t < p.rows && r < p.n) dense_store4<EPI, ACT_BF16, true>(p, t, r, v, bias);
        }
    }
}

// ---- 32-bit activations, more than four rows, no place for their planes (a call that is captured before any other has
// sized the workspace): 64 x 64 tiles on the vector pipe, BF16 weights widened, fp32 FMA ---------------------------------
// Sums are two-level (a step of 16 k, then the running total), which keeps the rounding error of a long k small.
template <int EPI>
__global__ __launch_bounds__(256) void dense_f32_kernel(DenseLinearParams p) {
    __shared__ float ws[16][65], xs[16][65];
    const uint32_t tid = threadIdx.x, tx = tid & 15u, ty = tid >> 4;
    const uint32_t n0 = blockIdx.x * 64u, m0 = blockIdx.y * 64u;
    const float* x = static_cast<const float*>(p.x);
    float acc[4][4] = {};
    for (uint32_t k0 = 0; k0 < p.k; k0 += 16u) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t r = (tid >> 4) + 16u * j, k = tid & 15u;
            ws[k][r] = bf16_to_f32(p.w[(size_t)min(n0 + r, p.n - 1u) * p.w_stride + k0 + k]);
            xs[k][r] = x[(size_t)min(m0 + r, p.rows - 1u) * p.x_stride + k0 + k];
        }
        __syncthreads();
        float part[4][4] = {};
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            float a[4], b[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) { a[j] = xs[k][ty + 16 * j]; b[j] = ws[k][tx + 16 * j]; }
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int n = 0; n < 4; ++n) part[m][n] = fmaf(a[m], b[n], part[m][n]);
        }
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int n = 0; n < 4; ++n) acc[m][n] += part[m][n];
        __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            const uint32_t t = m0 + ty + 16u * m, r = n0 + tx + 16u * n;
            const float next = EPI == DE_PAIRS ? shfl_xor_f(acc[m][n], 1) : 0.0f;        // the neighbouring weight row's sum
            if (t >= p.rows || r >= p.n) continue;
            if (EPI != DE_PAIRS) dense_store<EPI, ACT_FP32>(p, t, r, acc[m][n]);
            else if ((r & 1u) == 0) dense_put<ACT_FP32>(p, t, r / 2u, dense_pair<ACT_FP32>(acc[m][n], next));
        }
}

// ---- launches ---------------------------------------------------------------------------------------------
template <int EPI, int ACT, int NT>
void launch_gemv(const DenseLinearParams& p, hipStream_t s) {
    constexpr int X = NT * (ACT == ACT_FP32 ? 2 : 1);        // loads of the inputs per step
    auto go = [&](auto rw, auto u) {
        constexpr int RW = decltype(rw)::value, U = decltype(u)::value;
        dense_gemv_kernel<EPI, ACT, NT, RW, U><<<(p.n + 4 * RW - 1) / (4 * RW), 256, 0, s>>>(p);
    };
    constexpr std::integral_constant<int, 1> one{};
    constexpr std::integral_constant<int, 2> two{};
    constexpr std::integral_constant<int, 4> four{};
    constexpr bool PAIRS = EPI == DE_PAIRS;
    // Rows per wave: one (short blocks, many of them) until the inputs' own loads weigh more than that.  Steps past the end of k are loads for nothing: where k ends
    // before they do, fewer steps and more rows (BF16 us, one row per wave and four steps, and so: 24,833 x 576 one input 11.2 and 7.2, two 14.8 and 8.4; 21,845 x 1024
    // 12.1 and 9.9, 15.3 and 10.2; 2048 x 1024 3.0 and 2.8; 4096 x 512 3.3 and 2.8, 4.1 and 3.2; 30,000 x 192 11.1 and 5.2; three inputs of 4096 x 512 in two steps 3.8 and 3.2).
    // The bits depend on neither.
    if (p.k <= 512) {
        if (p.n >= 8192) go(four, one);
        else if (PAIRS || (X <= 2 && p.n >= 2048)) go(two, one);
        else if constexpr (!PAIRS) go(one, one);
    } else if (p.n >= 65536) {
        go(four, two);
    } else if (X <= 2 && p.k <= 1024 && p.n >= 2048) {
        go(two, two);
    } else if (PAIRS || (X > 2 && p.n >= 8192)) {
        go(two, std::integral_constant<int, X == 1 ? 4 : 2>{});
    } else if constexpr (!PAIRS) {
        go(one, std::integral_constant<int, X <= 2 ? 4 : 2>{});
    }
}

template <int EPI, int NT, int S>
void launch_gemv_rms(const DenseLinearParams& p, uint32_t cus, hipStream_t s) {
    constexpr int RW = EPI == DE_PAIRS ? 2 : 1;
    // as few turns as leave no more than six blocks per compute unit (2, 4, 6, 8: 12.7, 12.7, 12.5, 12.2 us for 12,352 x 2048, 10.8, 11.0, 10.6, 10.5 for
    // 11,264 rows in pairs; with eight a small matrix's rows are dealt out one by one again)
    const uint32_t groups = (p.n + 4 * RW - 1) / (4 * RW), turns = (groups + 6 * cus - 1) / (6 * cus);
    dense_gemv_rms_kernel<EPI, NT, RW, S><<<(groups + turns - 1) / turns, 256, 0, s>>>(p, turns);
}

template <int EPI>
int gemv_rms(const DenseLinearParams& p, uint32_t cus, hipStream_t s) {
    if (p.rows == 1 && p.k <= 1024) launch_gemv_rms<EPI, 1, 2>(p, cus, s);
    else if (p.rows == 1) launch_gemv_rms<EPI, 1, 4>(p, cus, s);
    else if (p.k <= 1024) launch_gemv_rms<EPI, 2, 2>(p, cus, s);
    else launch_gemv_rms<EPI, 2, 4>(p, cus, s);
    return launch_status();
}

template <int EPI, int ACT>
int gemv(const DenseLinearParams& p, hipStream_t s) {
    if (p.rows == 1) launch_gemv<EPI, ACT, 1>(p, s);
    else if (p.rows == 2) launch_gemv<EPI, ACT, 2>(p, s);
    else if (p.rows == 3) launch_gemv<EPI, ACT, 3>(p, s);
    else launch_gemv<EPI, ACT, 4>(p, s);
    return launch_status();
}

inline bool dense_may_cut(const nvmai_hip_ctx* ctx) { return ctx->cut_sums != nullptr && (uint32_t)ctx->compute_units <= CUT_BLOCKS; }

template <int EPI, int ACT, int COUNT>
void launch_tile(nvmai_hip_ctx* ctx, hipStream_t s, const DenseLinearParams& p, const DensePlan& plan) {
    const int c = plan.tile;
    const uint32_t tn = (p.n + DENSE_TILES[c].bn - 1) / DENSE_TILES[c].bn, tm = (p.rows + DENSE_TILES[c].bm - 1) / DENSE_TILES[c].bm, blocks = tn * tm * plan.parts;
    const DenseCut cut{plan.parts, ctx->cut_sums, ctx->tickets + TICKET_CUTS};
    if (c == 0) dense_tile_kernel<EPI, ACT, 64, 64><<<blocks, 256, 0, s>>>(p, tn, tm, cut);
    else if (c == 1) dense_tile_kernel<EPI, ACT, 128, 64><<<blocks, 256, 0, s>>>(p, tn, tm, cut);
    else if (c == 2) dense_tile_kernel<EPI, ACT, 128, 128><<<blocks, 256, 0, s>>>(p, tn, tm, cut);
    if constexpr (COUNT > 3) {
        if (c == 3) dense_tile_kernel<EPI, ACT, 256, 128><<<blocks, 256, 0, s>>>(p, tn, tm, cut);
        else if (c == 4) dense_wide_kernel<EPI><<<blocks, 256, 0, s>>>(p, tn, tm);
    }
}

template <int EPI, int ACT>
void launch_tiles(nvmai_hip_ctx* ctx, hipStream_t s, const DenseLinearParams& p) {
    constexpr int COUNT = ACT == ACT_FP32 ? 3 : 5;           // 32-bit inputs keep a running total beside the sums: no registers for the larger tiles
    const uint32_t cus = (uint32_t)ctx->compute_units, planes = ACT == ACT_FP32 ? 3u : 1u;
    const DenseSplit plan = dense_plan(p.n, p.rows, p.k, planes, cus, COUNT, dense_may_cut(ctx));
    const uint32_t first = plan.first;
    DenseLinearParams q = p;
    q.n = first;
    launch_tile<EPI, ACT, COUNT>(ctx, s, q, plan.head);
    if (first == p.n) return;
    q.n = p.n - first;                                       // first is a multiple of 64: every operand stays aligned
    q.w = p.w + (size_t)first * p.w_stride;
    const uint32_t out = EPI == DE_PAIRS ? first / 2 : first;
    if (p.y) q.y = p.y_k ? static_cast<void*>(static_cast<uint16_t*>(p.y) + out) : static_cast<void*>(static_cast<act_t<ACT>*>(p.y) + out);
    if (p.y_f32) q.y_f32 = p.y_f32 + out;
    if (p.bias) q.bias = p.bias + first;
    if (p.mul) q.mul = p.mul + first;
    launch_tile<EPI, ACT, COUNT>(ctx, s, q, plan.tail);
}

// 32-bit inputs: their planes, in portions of rows, then the product.
template <int EPI>
int launch_split(nvmai_hip_ctx* ctx, hipStream_t s, const DenseLinearParams& p) {
    const uint32_t most = dense_plane_rows(p.k);
    for (uint32_t at = 0; at < p.rows; at += most) {
        DenseLinearParams q = p;
        q.rows = p.rows - at < most ? p.rows - at : most;
        dense_split(s, static_cast<const float*>(p.x) + (size_t)at * p.x_stride, p.x_stride, q.rows, p.k, p.planes);
        q.x = p.planes;
        q.x_stride = 3 * p.k;
        if (p.y) q.y = static_cast<float*>(p.y) + (size_t)at * p.y_stride;
        if (p.y_f32) q.y_f32 = p.y_f32 + (size_t)at * p.y_stride;
        if (p.mul_ids) q.mul_ids = p.mul_ids + at;
        launch_tiles<EPI, ACT_FP32>(ctx, s, q);
    }
    return launch_status();
}

template <int EPI>
int dense_launch(nvmai_hip_ctx* ctx, hipStream_t s, const DenseLinearParams& p) {
    if (p.rms_delta) return gemv_rms<EPI>(p, (uint32_t)ctx->compute_units, s);
    if (p.rows <= 4) return ctx->act == NVMAI_ACT_FP32 ? gemv<EPI, ACT_FP32>(p, s) : gemv<EPI, ACT_BF16>(p, s);
    if (ctx->act == NVMAI_ACT_FP32) {
        const dim3 grid((p.n + 63) / 64, (p.rows + 63) / 64);
        if (grid.y > 65535) return NVMAI_ERR_UNSUPPORTED;
        if (p.x_planes) return launch_tiles<EPI, ACT_FP32>(ctx, s, p), launch_status();
        if (p.planes) return launch_split<EPI>(ctx, s, p);
        dense_f32_kernel<EPI><<<grid, 256, 0, s>>>(p);
        return launch_status();
    }
    if (p.rows <= 64) {
        // Two waves leave room for several blocks per compute unit.  Several row tiles per block where the inputs, which every block reads, would
        // weigh more than its weights (32 rows: 8192 x 2048 11.5 -> 10.0 us; 64: 14.5 -> 12.3, 49,664 x 2048 83 -> 65 with four).  Past 16 rows, against sixteen
        // waves that load operands (17 and 64 rows): 2048 x 8192 19.5 -> 15.7 and 46.2 -> 24.2 us, 2048 x 5632 14.5 -> 11.6 and 33.9 -> 19.4, 2128 x 2048 8.4 -> 5.9 and
        // 14.2 -> 8.6, 1024 x 2816 8.3 -> 5.8 and 15.8 -> 8.9.
        const uint32_t sums = skinny_sums(p.n, p.k);
        auto launch = [&](auto tt, auto nr, auto nw) {
            constexpr int TT = decltype(tt)::value, NR = decltype(nr)::value, NW = decltype(nw)::value;
            const uint32_t blocks = (p.n + 16 * NR - 1) / (16 * NR);
            if constexpr (NR == 1) {                          // four waves: k past 2048
                if (sums == 16) return dense_skinny_kernel<EPI, TT, NR, NW, 16 / NW><<<blocks, 64 * NW, 0, s>>>(p);
                if constexpr (NW == 2)
                    if (sums == 8) return dense_skinny_kernel<EPI, TT, NR, NW, 8 / NW><<<blocks, 64 * NW, 0, s>>>(p);
            }
            dense_skinny_kernel<EPI, TT, NR, NW, 4 / NW><<<blocks, 64 * NW, 0, s>>>(p);
        };
        constexpr std::integral_constant<int, 1> one{};
        constexpr std::integral_constant<int, 2> two{};
        constexpr std::integral_constant<int, 4> four{};
        if (p.rows <= 16) {
            // Eight weight rows per block where sixteen leave half the units without one, past rows of 1024 (sixteen weight rows in two waves and eight, us for 5 rows:
            // 2048 x 8192 14.1 and 10.0, 2048 x 2112 5.6 and 4.6, 1024 x 4096 7.5 and 5.6, 2048 x 1536 3.7 and 3.5, 2048 x 1024 3.1 and 3.2, 2048 x 512 2.8 and 2.9).
            // Four waves where a row is long and the blocks are few, or the row so long that two take too many turns (two and four: 2064 x 4096 8.2 and 7.3,
            // 4096 x 2816 8.3 and 7.1, 8190 x 8192 31.7 and 30.0; but 6144 x 2112 8.0 and 8.8, 12,352 x 2816 16.8 and 17.4, 3072 x 1536 4.6 and 4.5, 2048 x 1024 3.1 and 3.3).
            if (p.k > 1024 && (p.n + 15) / 16 * 2 <= (uint32_t)ctx->compute_units) {
                if (sums == 16) dense_skinny_kernel<EPI, 1, 1, 4, 4, true><<<(p.n + 7) / 8, 256, 0, s>>>(p);
                else dense_skinny_kernel<EPI, 1, 1, 4, 2, true><<<(p.n + 7) / 8, 256, 0, s>>>(p);
            } else if (p.k <= 2048 || (p.n > 4096 && p.k < 4096)) launch(one, one, two);
            else launch(one, one, four);
        } else if (p.rows <= 32) {
            if (p.n < 8192) launch(two, one, two);
            else launch(two, two, two);
        } else if (p.n < 8192) launch(four, one, two);
        else if (p.n < 32768) launch(four, two, two);
        else launch(four, four, four);
        return launch_status();
    }
    launch_tiles<EPI, ACT_BF16>(ctx, s, p);
    return launch_status();
}

}  // namespace nvmai
