// Attention of a prompt's rows in 32 bits, shared by the latent and the windowed form.  gfx950, wave64.
#pragma once

#include "common.hpp"

namespace nvmai {

typedef float f32_f4 __attribute__((ext_vector_type(4)));

constexpr float FLASH32_NONE = -1e30f;      // maximum of no scores; a masked score is twice that

// One block: 16 queries of one head; its four waves take the tiles of 16 keys in turn and put their parts together at the end.
// S^T[key, query] = K Q^T and O^T[value, query] += V^T P^T on v_mfma_f32_16x16x4_f32: fp32 products and sums, nothing
// rounded on the way.  Lane (i = lane % 16, g = lane / 16) of a chunk of 16 dims holds dims 4 g .. 4 g + 3 of key (query) i, so
// a 16-byte load feeds four products; register j of S^T is key 4 g + j of query i and stands as the B operand of the second
// product beside values of key 4 g + j.  Keys come straight from L2 (no LDS: a tile is read by one wave), the next tile's
// under this tile's softmax and second product.  Bound by the latency of that chain at a few hundred rows, by the matrix
// pipe (157 TFLOP/s) at thousands.
//   KC: chunks of 16 dims; NV: 16-wide parts of the values.  query(c), key(tile, c): 16 bytes of dims 16 c + 4 g of query / key i
// (zeros where there are none).  VT: values(tile, n) is value 16 n + i of keys 4 g .. 4 g + 3; otherwise values(tile, j * NV / 4 + b)
// is values 64 b + 4 i .. + 3 of key 4 g + j.  score(tile, j, s): the score of key 4 g + j in powers of two.  whole(tile): every query of the
// block sees all of the tile (the same in all lanes); sees(tile, j, query): a query of the block sees key 4 g + j.  put(value, v): the block's
// result of query i at a value index.  shared: NV * 1024 + 128 floats.
//   A key that a query does not see has probability zero, and zero times an infinity or NaN among its values would be NaN.  A tile
// that is not seen whole is looked over for such values, and where there are any it is multiplied for one query at a time, with the
// values of the keys that this query does not see set to zero.
template <int KC, int NV, bool VT, class Query, class Key, class Values, class Score, class Whole, class Sees, class Put>
__device__ __forceinline__ void flash32_block(uint32_t tiles, float* shared, Query query, Key key, Values values, Score score, Whole whole, Sees sees, Put put) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, i = lane & 15u, g = lane >> 4;
    f32_f4 q[KC], k[KC], v[NV], acc[NV];
#pragma unroll
    for (int c = 0; c < KC; ++c) q[c] = query(c);
#pragma unroll
    for (int n = 0; n < NV; ++n) acc[n] = f32_f4{0.0f, 0.0f, 0.0f, 0.0f};
    float m = FLASH32_NONE, l = 0.0f;
    if (wave < tiles)
#pragma unroll
        for (int c = 0; c < KC; ++c) k[c] = key(wave, c);
    for (uint32_t t = wave; t < tiles; t += 4u) {
#pragma unroll
        for (int n = 0; n < NV; ++n) v[n] = values(t, n);
        f32_f4 s{0.0f, 0.0f, 0.0f, 0.0f}, s1 = s;
#pragma unroll
        for (int c = 0; c < KC; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (e & 1) s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[c][e], q[c][e], s1, 0, 0, 0);
                else s = __builtin_amdgcn_mfma_f32_16x16x4f32(k[c][e], q[c][e], s, 0, 0, 0);
            }
        const uint32_t next = min(t + 4u, tiles - 1u);
#pragma unroll
        for (int c = 0; c < KC; ++c) k[c] = key(next, c);
        s += s1;
#pragma unroll
        for (int j = 0; j < 4; ++j) s[j] = score(t, j, s[j]);
        const bool part = !whole(t);
        if (part) {
#pragma unroll
            for (int j = 0; j < 4; ++j) s[j] = sees(t, j, i) ? s[j] : 2.0f * FLASH32_NONE;
        }
        float tm = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
        tm = max_xor<16>(tm);
        tm = max_xor<32>(tm);
        if (__any(tm > m)) {
            const float mn = fmaxf(m, tm), alpha = __builtin_amdgcn_exp2f(m - mn);
            m = mn;
            l *= alpha;
#pragma unroll
            for (int n = 0; n < NV; ++n) acc[n] *= alpha;
        }
        // a query without a key so far has m = FLASH32_NONE, and exp2(2 FLASH32_NONE - FLASH32_NONE) = 0
#pragma unroll
        for (int j = 0; j < 4; ++j) s[j] = __builtin_amdgcn_exp2f(s[j] - m);
        l += (s[0] + s[1]) + (s[2] + s[3]);
        auto value = [&](int n, int j) { return VT ? v[n][j] : v[j * (NV / 4) + n / 4][n % 4]; };      // of key 4 g + j
        if (part) {
            uint32_t largest = 0;
#pragma unroll
            for (int n = 0; n < NV; ++n)
#pragma unroll
                for (int j = 0; j < 4; ++j) largest = max(largest, __float_as_uint(v[n][j]) & 0x7FFFFFFFu);
            if (__any(largest >= 0x7F800000u)) {
#pragma unroll 1
                for (uint32_t one = 0; one < 16u; ++one) {
                    bool seen[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) seen[j] = sees(t, j, one);
#pragma unroll
                    for (int n = 0; n < NV; ++n) {
                        f32_f4 sum{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                        for (int j = 0; j < 4; ++j) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(seen[j] ? value(n, j) : 0.0f, i == one ? s[j] : 0.0f, sum, 0, 0, 0);
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc[n][j] += i == one ? sum[j] : 0.0f;
                    }
                }
                continue;
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int n = 0; n < NV; ++n) acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(value(n, j), s[j], acc[n], 0, 0, 0);
    }
    l = add_xor<16>(l);
    l = add_xor<32>(l);
    float* ml = shared + NV * 1024;
    if (g == 0) {
        ml[wave * 32u + i] = m;
        ml[wave * 32u + 16u + i] = l;
    }
    __syncthreads();
    const float top = fmaxf(fmaxf(ml[i], ml[32u + i]), fmaxf(ml[64u + i], ml[96u + i]));
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) sum = fmaf(ml[w * 32 + 16 + i], __builtin_amdgcn_exp2f(ml[w * 32 + i] - top), sum);
    const float own = __builtin_amdgcn_exp2f(m - top);
#pragma unroll
    for (int n = 0; n < NV; ++n)
#pragma unroll
        for (int j = 0; j < 4; ++j) shared[wave * (NV * 256u) + (4 * n + j) * 64 + lane] = acc[n][j] * own;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NV / 4; ++u) {
        const uint32_t n = wave * (NV / 4) + u;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float* at = shared + (4u * n + j) * 64u + lane;
            const float o = (at[0] + at[NV * 256]) + (at[2 * NV * 256] + at[3 * NV * 256]);
            put(VT ? 16u * n + 4u * g + j : 64u * (n / 4u) + 16u * g + 4u * j + n % 4u, o / sum);
        }
    }
}

}  // namespace nvmai
