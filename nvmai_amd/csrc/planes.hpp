// Rows of floats as three BF16 planes, [row][3][k], the smallest part first: what the products of 32-bit contexts multiply.
//
// A row that only such products read is stored as planes by whatever makes it (a norm, another product, the latents' gather), which saves a launch in front of every product
// that would read 4 bytes a value and write 6: of 36 such launches (5 us each, 0.18 of 1.24 ms) of a prompt of 700 tokens (Pakirax 1k, 8 layers) 12 are left: 1243 -> 1138 us, 60 tokens
// 645 -> 602; Kemuzen 1k, 700 tokens 1994 -> 1844, 100 tokens 996 -> 910.
#pragma once

#include "common.hpp"

namespace nvmai {

// A float as three BF16 values that add up to it exactly (8 + 8 + 8 bits of mantissa, by truncation; below 2^-110 the
// last bits may be lost).  Infinities and NaN stay in the first one.
__device__ __forceinline__ void split3(float x, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
    const uint32_t u = __float_as_uint(x);
    const bool finite = (u & 0x7F800000u) != 0x7F800000u;
    const float r1 = x - __uint_as_float(u & 0xFFFF0000u);
    const float r2 = r1 - __uint_as_float(__float_as_uint(r1) & 0xFFFF0000u);
    hi = (u >> 16) | (!finite && (u & 0x007FFFFFu) ? 0x40u : 0u);
    mid = finite ? __float_as_uint(r1) >> 16 : 0u;
    lo = finite ? __float_as_uint(r2) >> 16 : 0u;
}

// N (1, 2 or 4) neighbouring values of a row of planes from `at` (a multiple of N) on.
template <int N>
__device__ __forceinline__ void planes_put(uint16_t* row, uint32_t k, uint32_t at, const float* v) {
    if constexpr (N == 1) {
        uint32_t hi, mid, lo;
        split3(v[0], hi, mid, lo);
        row[at] = (uint16_t)lo;
        row[k + at] = (uint16_t)mid;
        row[2u * (size_t)k + at] = (uint16_t)hi;
        return;
    }
    uint32_t out[3][(N + 1) / 2];
#pragma unroll
    for (int e = 0; e < N / 2; ++e) {
        uint32_t a[3], b[3];
        split3(v[2 * e], a[2], a[1], a[0]);
        split3(v[2 * e + 1], b[2], b[1], b[0]);
#pragma unroll
        for (int q = 0; q < 3; ++q) out[q][e] = a[q] | (b[q] << 16);
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        uint16_t* const to = row + (size_t)q * k + at;
        if constexpr (N == 4) *reinterpret_cast<uint2*>(to) = make_uint2(out[q][0], out[q][1]);
        else *reinterpret_cast<uint32_t*>(to) = out[q][0];
    }
}

}  // namespace nvmai
