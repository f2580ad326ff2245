// Choices between the forms of a call that sizes alone decide: plain C++, without a device.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace nvmai {

// Widths whose rows the row engine reads in 16, 32, 64 or 128 pieces of sixteen bytes, with its inputs as fp16 numbers (moe_kernels.hpp).  At
// others it takes floats.
inline bool rows_engine_fp16(uint32_t bits, uint32_t n) {
    const uint64_t width = (uint64_t)n * bits;
    return width == 16u * 128u || width == 32u * 128u || width == 64u * 128u || width == 128u * 128u;
}

// Whether three or four input rows of an affine matrix take the matrix-core product, as five do: where it is faster than the row engine and the engine
// takes the inputs as fp16 numbers too.  Engine and product, us, 4 bits, four rows: 12,352 x 2048 13.0 and 9.7, 2048 x 4096 10.1 and 9.3, 512 x 1024 6.7 and 5.4,
// 2048 x 512 5.6 and 5.4; three: 12,352 x 2048 11.3 and 9.8, 4096 x 2048 6.6 and 6.5, 1024 x 2048 5.5 and 5.7, 2048 x 4096 8.2 and 9.4; 8 bits, four: 12,352 x 2048 15.4
// and 12.0, 4096 x 2048 8.2 and 8.2, 512 x 1024 5.6 and 6.1; sums against 64 bits 8e-6 and 2e-6, 8 bits 5e-7 and 3e-7.  Three rows and 8 bits: the widths of one
// size are level below 8192 matrix rows (6 % for either), so the line lies where the gain is sure.  Up to 30,000 rows were measured (20.8 and 18.8); larger
// matrices stay.
inline bool few_rows_mfma(uint32_t bits, uint32_t n_tokens, uint32_t m, uint32_t n) {
    if (m >= 32768u || !rows_engine_fp16(bits, n)) return false;
    if (n_tokens == 4) return bits == 4 || (n == 2048 && m >= 8192);
    return n_tokens == 3 && n == 2048 && m >= 8192;
}

// Whether the matrix-core product of few rows requests its inputs ahead of the weights, without a look at which there are: all rows of a tile of 16 or 32, so that it
// pays where few are missing, and whole panels of 2048 or 1024 values.  4 bits, 2048 x 4096: 16 rows 9.6 -> 8.9 us, 9 rows 9.4 -> 9.0, 8 rows 9.4 both ways; 28 rows 18.2 -> 17.9, 24
// rows 18.0 -> 17.9 and at 512 x 2048 9.7 -> 9.9.  8 bits, 12,352 x 2048: 16 rows 12.0 -> 11.2, 14 rows 11.9 -> 11.7, 12 rows 11.8 both ways and at 2048 x 4096 12.0 -> 12.2; 32 rows
// 18.5 -> 18.0, 28 rows 18.2 -> 18.5.  Panels that are not whole, 16 rows of 1024 x 4096: 5.6 -> 5.8.
inline bool gemv_inputs_first(uint32_t bits, uint32_t n_tokens, uint32_t n) {
    if (n_tokens <= 16) return n % 2048 == 0 && n_tokens >= (bits == 4 ? 9u : 14u);
    return n % 1024 == 0 && n_tokens >= (bits == 4 ? 28u : 31u);
}

// Whether a dense product can address `rows` input rows of `stride` values with 32-bit byte offsets (values of up to four bytes).
inline bool dense_rows_fit(uint32_t rows, uint32_t stride) { return (uint64_t)rows * stride * 4 <= 0xFFFFFFFFull; }

// The same of both products of a shared expert: its tokens, and the f values that it holds of each between them.
inline bool expert_rows_fit(uint32_t tokens, uint32_t x_stride, uint32_t f) { return dense_rows_fit(tokens, x_stride) && dense_rows_fit(tokens, f); }

// How many tokens of a shared expert the products that dequantize per tile take in one call: x, the f values between them and the output have 32-bit
// byte offsets, in 16 bits.  0: the codes themselves are too many.
inline uint32_t expert_block_tokens(uint32_t x_stride, uint32_t d, uint32_t f, uint32_t bits) {
    if ((uint64_t)d * f * bits / 8 > 0xFFFFFFFFull) return 0;
    const uint32_t widest = x_stride > d ? (x_stride > f ? x_stride : f) : (d > f ? d : f);
    return 0xFFFFFFFFu / 2u / widest / 128u * 128u;
}

// 32-bit rows are multiplied as three BF16 planes, at most this many rows at a time: 128 MB of planes, or one row's (1.3 GB for
// the longest that a call accepts), so that byte offsets inside them stay within 32 bits.
inline uint32_t dense_plane_rows(uint32_t k) {
    const uint64_t rows = (128u << 20) / (6ull * k);
    return rows >= 32768u ? 32768u : rows >= 256u ? (uint32_t)(rows / 256u * 256u) : rows ? (uint32_t)rows : 1u;
}
inline size_t dense_plane_bytes(uint32_t rows, uint32_t k) {
    const uint32_t most = dense_plane_rows(k);
    return (size_t)(rows < most ? rows : most) * k * 6u;
}
// Whether a call takes rows that are planes already, in memory of its caller's.
inline bool planes_fit(uint32_t rows, uint32_t k) { return (uint64_t)rows * k * 6u <= (128u << 20); }
// Whether dense_plane_bytes is room for the planes of all rows at once, which products that share them need: the latents of an expanded 32-bit attention.
// Past it each product makes its own, in portions.
inline bool planes_at_once(uint32_t rows, uint32_t k) { return rows <= dense_plane_rows(k); }

// Rows of values of 16 bits by their addresses, 0: none.
struct Rows16 {
    uint64_t at;
    uint32_t stride;
};

// Whether `rows` rows of `d` values at a and at b have bytes in common.
inline bool rows_overlap(const Rows16& a, const Rows16& b, uint32_t rows, uint32_t d) {
    if (!a.at || !b.at) return false;
    const uint64_t na = ((uint64_t)(rows - 1) * a.stride + d) * 2, nb = ((uint64_t)(rows - 1) * b.stride + d) * 2;
    return a.at < b.at + nb && b.at < a.at + na;
}

// Whether what the prologue of a launch stores lies over the rows that all of its blocks read.
inline bool prologue_overlaps(const Rows16& x, const Rows16& delta, const Rows16& hidden_out, const Rows16& normed_out, uint32_t rows, uint32_t d) {
    return rows_overlap(hidden_out, x, rows, d) || rows_overlap(hidden_out, delta, rows, d) || rows_overlap(normed_out, x, rows, d) || rows_overlap(normed_out, delta, rows, d);
}

// The same of a launch that holds the whole MoE block: y, too, lies over nothing that other blocks read, nor over what another block stores, which nothing orders (a block
// that waits in vain stores the prologue's rows once more, after others have stored y).
inline bool block_overlaps(const Rows16& x, const Rows16& delta, const Rows16& hidden_out, const Rows16& normed_out, const Rows16& y, uint32_t rows, uint32_t d) {
    return prologue_overlaps(x, delta, hidden_out, normed_out, rows, d) || rows_overlap(y, x, rows, d) || rows_overlap(y, delta, rows, d) ||
           rows_overlap(y, hidden_out, rows, d) || rows_overlap(y, normed_out, rows, d);
}

}  // namespace nvmai
