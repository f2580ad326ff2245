// The MoE block of one token in one launch: router, selection, gate and up, down, weighted sum.
//
// As three launches (router_logits_kernel, expert_rows_routed, down_combine_kernel) the block is bound by their chain: 4.4 + 7.2 + 7.4 us at 4
// bits, 17 MB of weights among them, which HBM delivers in 3.4.  Here the steps are blocks of one launch that hand their values on (hand.hpp): the inputs of gate and up are
// staged while the router's rows are summed, and a block of the down projection asks for its experts' rows as soon as the router has chosen, beside gate and up.  One token, 2048 x 512, 256
// experts: 18.2 -> 14.3 to 15.2 us a block, from process to process, 24 -> 19 with the norm before it, at 4 and at 8 bits.  By the clock in its blocks: inputs staged at 1.9 us, logits at 3.0, seen at 5.3, experts chosen at
// 5.6 to 6.5, the first rows of gate and up at 7.4 and the last at 8.4, all seen at 10.0, taken at 11.6, summed at 13.2.  Two tokens take longer so than in three launches (23.3 and 21.7 us at 4 bits, 27.7 and
// 23.1 at 8): the blocks do not all fit the device at once, and each asks for all activations of its token.
#pragma once

#include "hand.hpp"
#include "moe_kernels.hpp"

namespace nvmai {

struct MoeOneParams {
    RouterParams router;
    SelectParams sel;            // logits unused
    RowsParams rows;             // gate and up; x as the router's (the residual stream with pre_weight set)
    DownCombineParams down;      // acts, idx, w unused
    RoutedStats stats;
    Hand hand;
    uint32_t router_blocks;      // per token
    uint32_t slots;
    uint32_t down_blocks;        // per token
    uint32_t blocks, lds;        // of the launch
};

// The launch takes one token (moe_one_fits).  Its blocks are numbered by token all the same: without the divisions, and without the statistics over several tokens, the compiler lays
// the kernel out otherwise, and at 8 bits a block whose weights come from HBM took 18.6 us instead of 18.2 (twelve layers in turn; 4 bits 14.7 and 15.2).
constexpr uint32_t MOE_ONE_TOKENS = 1;
constexpr uint32_t MOE_ONE_THREADS = 512;                // fewer blocks than of 256, and so fewer that ask for the same words
constexpr uint32_t MOE_ONE_ROWS = 16;                    // rows of gate and up per block, two per wave
constexpr uint32_t MOE_ONE_LOGITS = 8;                   // rows of the router per block: half-waves of one wave per SIMD
constexpr uint32_t MOE_ONE_SLOTS = 4 * DC_SLOTS_PER_WAVE;                   // top_k + shared at most

// Every word is written several times over, by neighbouring lanes of one store, and a block reads the copy that its number names: one line asked for by all
// of the blocks answers one after another (about 2.3 ns each), and what is to be written to it waits with them.
constexpr uint32_t MOE_ONE_COPIES = 8;                   // of logits and choices
constexpr uint32_t MOE_ONE_ACT_COPIES = 4;               // of activations

// Words: per token its logits (those of the experts that a lane takes lie 64 apart, so that a load is of neighbours) and its gate's, the chosen experts and
// their weights, the activations of every slot.
__host__ __device__ inline uint32_t moe_one_per_lane(uint32_t experts) { return experts <= 256 ? 4 : TOPK_MAX_PER_LANE; }
__host__ __device__ inline uint32_t moe_one_copy_words(uint32_t experts) { return 64 * moe_one_per_lane(experts) + 16 + 2 * 16; }
__host__ __device__ inline uint32_t moe_one_token_words(uint32_t experts, uint32_t slots, uint32_t f) {
    return MOE_ONE_COPIES * moe_one_copy_words(experts) + MOE_ONE_ACT_COPIES * slots * f;
}

// A slot's activations in LDS, in pieces of four that lanes of a row read without conflict: piece j of lane sl at j * (SEG + 1) + sl.
template <int BITS, int SEG>
struct DownActs {
    static constexpr uint32_t EPC = Chunk<BITS>::elems, PIECES = EPC / 4, FLOATS = PIECES * (SEG + 1) * 4;
    static __device__ uint32_t at(uint32_t f) { return ((f % EPC / 4) * (SEG + 1) + f / EPC) * 4 + f % 4; }
};

inline size_t moe_one_down_lds(uint32_t bits, uint32_t seg, uint32_t slots) { return (size_t)slots * (128 / bits / 4) * (seg + 1) * 16; }

struct MoeOneToken {
    uint64_t *first, *acts;      // copy 0
    uint32_t copy, gate, act;    // words of a copy; where in it the gate's is, and 16 behind it the chosen experts and 32 behind it their weights
    __device__ MoeOneToken(const MoeOneParams& p, uint32_t t) {
        first = p.hand.words + (size_t)t * moe_one_token_words(p.router.num_experts, p.slots, p.rows.rows);
        copy = moe_one_copy_words(p.router.num_experts);
        gate = copy - 48;
        acts = first + MOE_ONE_COPIES * copy;
        act = p.slots * p.rows.rows;
    }
    __device__ const uint64_t* mine() const { return first + blockIdx.x % MOE_ONE_COPIES * copy; }
    __device__ const uint64_t* my_acts() const { return acts + blockIdx.x % MOE_ONE_ACT_COPIES * act; }
};

// The selection of a token by one wave, from the router's words: as many of the chosen as `rounds`.
__device__ __forceinline__ bool moe_one_select(const MoeOneParams& p, uint32_t e, uint32_t t, int lane, uint32_t rounds, float& score, uint32_t& idx) {
    const uint32_t E = p.router.num_experts;
    const uint64_t* const words = MoeOneToken(p, t).mine();
    // past the last expert: the last one's word again
    auto at = [&](int j) {
        const uint32_t per = moe_one_per_lane(E), x = min((uint32_t)lane * per + j, E - 1u);
        return words + 64u * (x % per) + x / per;
    };
    if (E <= 256) {
        float val[4];
        if (!hand_take<4>(p.hand, e, at, val)) return false;
        select_topk_values<4>(p.sel, val, lane, score, idx, rounds);
    } else {
        float val[TOPK_MAX_PER_LANE];
        if (!hand_take<TOPK_MAX_PER_LANE>(p.hand, e, at, val)) return false;
        select_topk_values<TOPK_MAX_PER_LANE>(p.sel, val, lane, score, idx, rounds);
    }
    return true;
}

template <int ACT>
__device__ __forceinline__ void moe_one_router(const MoeOneParams& p, uint32_t e, uint32_t item, uint4* lds) {
    const RouterParams& r = p.router;
    const uint32_t t = item / p.router_blocks, b = item % p.router_blocks;
    const int hw = threadIdx.x >> 5, hl = threadIdx.x & 31;
    const uint32_t row = b * MOE_ONE_LOGITS + hw, total = r.num_experts + (r.gate.kind ? 1u : 0u);
    const bool live = hw < (int)MOE_ONE_LOGITS && row < total, is_gate = row >= r.num_experts;
    const RowsDesc& rd = is_gate ? r.gate : r.router;
    uint16_t* xl = reinterpret_cast<uint16_t*>(lds);
    RouterRowRegs<8> g;
    if (live) router_row_prefetch<8>(r, rd, is_gate ? 0u : row, hl, g);
    if (r.pre_weight) {
        const PreNormArgs a{(const uint16_t*)r.x, r.x_stride, r.pre_delta, r.pre_delta_stride, r.pre_weight, r.pre_hidden_out,
                            r.pre_hidden_stride, r.pre_normed_out, r.pre_normed_stride, r.pre_eps, r.d};
        stage_prenorm_rows<ACT>(a, t, 1, xl, xl + r.d, b == 0);
    } else {
        router_stage_x(r, t, 1, xl);
    }
    if (live) {
        float acc[1];
        router_row_any<ACT, 8, 2048>(r, rd.kind, g, xl, 1, hl, acc);
        const MoeOneToken token(p, t);
        const uint32_t per = moe_one_per_lane(r.num_experts);
        if (hl < (int)MOE_ONE_COPIES) hand_put(token.first + hl * token.copy + (is_gate ? token.gate : 64u * (row % per) + row / per), acc[0], e);
    }
}

// The choice of a token, handed to the blocks of the down projection and stored for the caller, with the statistics of the step; a block of its own, so that no block of
// gate and up is late for it.
__device__ __forceinline__ bool moe_one_choice(const MoeOneParams& p, uint32_t e, uint32_t t, uint32_t* ids) {
    const uint32_t K = p.sel.top_k, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const bool counts = p.stats.stats && t == 0;
    bool ok = true;
    float score;
    uint32_t idx = 0;
    if (wave == 0) {
        ok = moe_one_select(p, e, t, lane, K, score, idx);
        if (ok) {
            const uint16_t w = select_weight(p.sel, lane, score, idx);
            const MoeOneToken token(p, t);
            if (lane < K) {
#pragma unroll
                for (uint32_t c = 0; c < MOE_ONE_COPIES; ++c) {
                    hand_put(token.first + c * token.copy + token.gate + 16 + lane, __uint_as_float(idx), e);
                    hand_put(token.first + c * token.copy + token.gate + 32 + lane, f16_to_f32(w), e);
                }
                p.sel.out_idx[(size_t)t * K + lane] = idx;
                p.sel.out_w[(size_t)t * K + lane] = w;
            }
        }
    } else if (counts && wave < p.sel.tokens) {
        ok = moe_one_select(p, e, wave, lane, K, score, idx);
    }
    if (counts) {                // the distinct experts of the step: tokens * top_k <= 64 indices
        const uint32_t n = p.sel.tokens * K;
        if (wave < p.sel.tokens && lane < K) ids[wave * K + lane] = idx;
        if (!__syncthreads_and(ok)) return false;
        bool fresh = lane < n;
        for (uint32_t j = 0; j < lane && lane < n; ++j) fresh = fresh && ids[j] != ids[lane];
        const uint32_t distinct = (uint32_t)__popcll(__ballot(fresh));
        if (threadIdx.x == 0) {
            p.stats.stats[0] = p.sel.tokens * p.slots;
            p.stats.stats[1] = p.sel.tokens > 1 ? distinct : K;        // one token: as the launch that selects for itself says it, also where an expert is chosen again
        }
        return true;
    }
    return __syncthreads_and(ok);
}

// Two rows of gate and up per wave, for one input of up to 2048: the arithmetic of expert_rows_body, with the inputs staged before the expert is known.
// LDS: the packed inputs, their chunks' sums (all, odd pairs), the waves' maxima; behind them a normed row and its raw one.
template <int ACT, int BITS, int NCH>
__device__ __forceinline__ bool moe_one_rows(const MoeOneParams& p, uint32_t e, uint32_t item, uint4* lds, uint32_t* shared) {
    constexpr int EPC = Chunk<BITS>::elems, PAIRS = EPC / 2, H = PAIRS / 4, CHUNKS = 64 * NCH, ROWS = 2;
    constexpr uint32_t n = (uint32_t)CHUNKS * EPC;
    static_assert(n <= 2048, "eight inputs per thread of four waves");
    const RowsParams& r = p.rows;
    const uint32_t per_token = p.slots * r.blocks_per_entry;
    const uint32_t t = item / per_token, slot = item % per_token / r.blocks_per_entry, rb = item % r.blocks_per_entry;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const NibbleConsts nib = nibble_consts();
    uint4* const xw = lds;
    float* const sums = reinterpret_cast<float*>(lds + n / 8);
    float* const maxima = sums + 2 * CHUNKS;
    const uint32_t e0 = threadIdx.x * 8;
    const bool live = e0 < n;
    float v[8] = {};
    if (r.pre_weight) {
        uint16_t* const xl = reinterpret_cast<uint16_t*>(maxima + 4);
        const PreNormArgs a{(const uint16_t*)r.x, r.x_stride, r.pre_delta, r.pre_delta_stride, r.pre_weight, nullptr, 0, nullptr, 0, r.pre_eps, n};
        stage_prenorm_rows<ACT>(a, t, 1, xl, xl + n, false);
        if (live) load8<ACT, false>(xl, e0, v);
    } else if (live) {
        load8<ACT, false>(r.x, (size_t)t * r.x_stride + e0, v);
    }
    float most = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) most = fmaxf(most, fabsf(v[j]));
    most = wave_max_f32(most);
    if (lane == 0 && wave < 4) maxima[wave] = most;
    __syncthreads();
    float sc, isc;
    pow2_scale(fmaxf(fmaxf(maxima[0], maxima[1]), fmaxf(maxima[2], maxima[3])), sc, isc);
    if (live) {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] *= sc;
        const uint32_t chunk = e0 / EPC, piece = (e0 % EPC) / 8;
        xw[((chunk % NCH) * H + piece) * 64 + chunk / NCH] = pack_inputs<BITS>(v);
    }
    __syncthreads();
    if (threadIdx.x < CHUNKS) {
        const uint32_t c = threadIdx.x / 64, l = threadIdx.x % 64;
        float sum = 0.0f, odd = 0.0f;                 // odd: the pairs 1, 3, 5, ... of the chunk
#pragma unroll
        for (int h = 0; h < H; ++h) {
            const uint4 w = xw[(c * H + h) * 64 + l];
            const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const float both = f16_to_f32((uint16_t)(ws[d] & 0xFFFFu)) + f16_to_f32((uint16_t)(ws[d] >> 16));
                sum += both;
                if (d & 1) odd += both;
            }
        }
        sums[threadIdx.x * 2] = sum;
        sums[threadIdx.x * 2 + 1] = odd;
    }
    uint32_t expert = NVMAI_SLOT_FLAG | 8u;
    if (slot < p.sel.top_k && wave == 0) {
        float score;
        uint32_t idx;
        const bool ok = moe_one_select(p, e, t, lane, slot + 1, score, idx);      // the first experts are asked for while the last are chosen
        expert = ok ? (uint32_t)__builtin_amdgcn_readlane((int)idx, (int)slot) : 0xFFFFFFFFu;
        if (lane == 0) *shared = expert;
    }
    __syncthreads();
    if (slot < p.sel.top_k) expert = (uint32_t)__builtin_amdgcn_readfirstlane((int)*shared);
    if (expert == 0xFFFFFFFFu) return false;

    const uint8_t* const blob = blob_ptr(r.src, expert);
    const uint32_t row0 = (rb * (MOE_ONE_THREADS / 64) + wave) * ROWS, groups = n / NVMAI_GROUP, row_bytes = n * BITS / 8;
    uint4 q[2][ROWS][NCH];                            // gate, up
    uint16_t s[2][ROWS][NCH], b[2][ROWS][NCH];
    const int64_t w_at[2] = {r.wA, r.wB}, s_at[2] = {r.sA, r.sB}, b_at[2] = {r.bA, r.bB};
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
        const uint32_t row = min(row0 + i, r.rows - 1u);
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const uint32_t chunk = lane * NCH + c, g = chunk * EPC / NVMAI_GROUP;
            const bool fresh = c == 0 || NCH * EPC > NVMAI_GROUP;
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                q[m][i][c] = *reinterpret_cast<const uint4*>(blob + w_at[m] + (size_t)row * row_bytes + chunk * 16);
                s[m][i][c] = fresh ? reinterpret_cast<const uint16_t*>(blob + s_at[m])[(size_t)row * groups + g] : s[m][i][0];
                b[m][i][c] = fresh ? reinterpret_cast<const uint16_t*>(blob + b_at[m])[(size_t)row * groups + g] : b[m][i][0];
            }
        }
    }
    const MoeOneToken token(p, t);
    uint32_t xp[NCH][PAIRS];
    float xs[NCH], xo[NCH];
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
#pragma unroll
        for (int h = 0; h < H; ++h) {
            const uint4 w = xw[(c * H + h) * 64 + lane];
            xp[c][4 * h] = w.x; xp[c][4 * h + 1] = w.y; xp[c][4 * h + 2] = w.z; xp[c][4 * h + 3] = w.w;
        }
        xs[c] = sums[(c * 64 + lane) * 2];
        xo[c] = sums[(c * 64 + lane) * 2 + 1];
    }
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
        float out[2];
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            float acc = 0.0f;
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
                uint32_t qp[PAIRS];
                unpack_pairs<BITS>(q[m][i][c], qp, nib);
                float dot = 0.0f;
#pragma unroll
                for (int k = 0; k < PAIRS; ++k) dot = dot2_acc(qp[k], xp[c][k], dot);
                dot = fmaf(-1024.0f, xs[c], dot);
                if (BITS == 4) dot = fmaf(ODD_PAIR_OFFSET_GAP, xo[c], dot);
                acc = fmaf(bf16_to_f32(s[m][i][c]), dot, acc);
                acc = fmaf(bf16_to_f32(b[m][i][c]), xs[c], acc);
            }
            out[m] = readlane_f(seg_reduce_sum<64>(acc), 63) * isc;
        }
        const float y = silu_fast(out[0]) * out[1];
        if (row0 + i < r.rows && lane < (int)MOE_ONE_ACT_COPIES) hand_put(token.acts + (size_t)lane * token.act + (size_t)slot * r.rows + row0 + i, y, e);
    }
    return true;
}

// Bytes of LDS of a block of gate and up.
inline size_t moe_one_rows_lds(uint32_t n, uint32_t nch) { return (size_t)n * 2 + (size_t)nch * 64 * 8 + 16 + (size_t)2 * n * 2; }

// A unit is 64 / SEG output rows of one slot; the block's waves share those of its DC_ROWS rows.
template <int ACT, int BITS, int SEG>
__device__ __forceinline__ bool moe_one_down(const MoeOneParams& p, uint32_t e, uint32_t item, float* acts, float (*part)[DC_ROWS], uint32_t* shared) {
    constexpr int EPC = Chunk<BITS>::elems, RPL = 64 / SEG, PASSES = DC_ROWS / RPL, WAVES = MOE_ONE_THREADS / 64;
    constexpr int UNITS = ((int)MOE_ONE_SLOTS * PASSES + WAVES - 1) / WAVES;
    using A = DownActs<BITS, SEG>;
    const DownCombineParams& d = p.down;
    const uint32_t t = item / p.down_blocks, row0 = item % p.down_blocks * DC_ROWS, K = p.sel.top_k;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, seg_id = lane / SEG, sl = lane % SEG;
    const uint32_t groups = d.n / NVMAI_GROUP, row_bytes = d.n * BITS / 8, g = (uint32_t)sl * EPC / NVMAI_GROUP;
    const uint32_t units = p.slots * PASSES;
    const MoeOneToken token(p, t);
    float wk = 0.0f, gate = 0.0f;
    if (wave == 0) {
        // lane k: the expert of slot k and its weight; every lane the gate's logit
        float v[3];
        const uint32_t k = min((uint32_t)lane, K - 1u);
        const uint64_t* const choice = token.mine() + token.gate + 16;
        const bool ok = hand_take<3>(p.hand, e, [&](int j) { return j == 0 ? choice + k : j == 1 ? choice + 16 + k : d.gate_logit ? choice - 16 : choice; }, v);
        wk = (uint32_t)lane < K ? v[1] : 0.0f;
        gate = v[2];
        if ((uint32_t)lane < K) shared[lane] = ok ? __float_as_uint(v[0]) : 0xFFFFFFFFu;
    }
    __syncthreads();
    if (shared[0] == 0xFFFFFFFFu) return false;
    uint4 q[UNITS];
    uint16_t sc[UNITS], bi[UNITS];
#pragma unroll
    for (int j = 0; j < UNITS; ++j) {
        const uint32_t u = min((uint32_t)(wave + WAVES * j), units - 1u), slot = u / PASSES;
        const uint8_t* blob = blob_ptr(d.src, slot < K ? (uint32_t)__builtin_amdgcn_readfirstlane((int)shared[slot]) : (NVMAI_SLOT_FLAG | 8u));
        const uint32_t row = row0 + u % PASSES * RPL + seg_id, r = row < d.rows ? row : d.rows - 1;
        q[j] = *reinterpret_cast<const uint4*>(blob + d.wA + (size_t)r * row_bytes + sl * 16);
        sc[j] = reinterpret_cast<const uint16_t*>(blob + d.sA)[(size_t)r * groups + g];
        bi[j] = reinterpret_cast<const uint16_t*>(blob + d.bA)[(size_t)r * groups + g];
    }
    // The activations: while the last rows of the slots' blocks are not there, one wave looks at one word of each (all of them, from every
    // block, would be 40 KB per look), then every thread takes its words.
    constexpr uint32_t F = SEG * EPC;              // d.n
    const uint32_t count = p.slots * F;
    const uint64_t* const words = token.my_acts();
    bool ok = true;
    if (wave == 0) {
        float v[1];
        const uint32_t step = count / 64;
        ok = hand_take<1>(p.hand, e, [&](int) { return words + (lane + 1) * step - 1; }, v);
    }
    if (!__syncthreads_and(ok)) return false;
    constexpr int PER = 9;
    for (uint32_t f0 = threadIdx.x; f0 < count; f0 += MOE_ONE_THREADS * PER) {
        float v[PER];
        ok = ok && hand_take<PER>(p.hand, e, [&](int j) { return words + min(f0 + MOE_ONE_THREADS * j, count - 1u); }, v);
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const uint32_t f = f0 + MOE_ONE_THREADS * j;
            if (f < count) acts[f / F * A::FLOATS + A::at(f % F)] = v[j];
        }
    }
    if (!__syncthreads_and(ok)) return false;
#pragma unroll
    for (int j = 0; j < UNITS; ++j) {
        const uint32_t u = wave + WAVES * j, slot = u / PASSES;
        if (u >= units) break;                    // uniform per wave
        float a[EPC], xs = 0.0f;
#pragma unroll
        for (int i = 0; i < (int)A::PIECES; ++i) {
            const float4 v = *reinterpret_cast<const float4*>(acts + slot * A::FLOATS + (i * (SEG + 1) + sl) * 4);
            a[4 * i] = v.x; a[4 * i + 1] = v.y; a[4 * i + 2] = v.z; a[4 * i + 3] = v.w;
        }
#pragma unroll
        for (int i = 0; i < EPC; ++i) xs += a[i];
        const float acc = down_rows<BITS, SEG>(q[j], sc[j], bi[j], a, xs);
        if (seg_result_lane<SEG>(lane)) part[slot][u % PASSES * RPL + seg_id] = acc;
    }
    __syncthreads();
    if (wave == 0) down_store<ACT>(d, t, row0, lane, part, wk, gate, 0.0f);
    return true;
}

// Blocks: the router's of every token, the rows' of gate and up, the choices', the down projection's, so that a block's producers stand before it.
template <int ACT, int BITS, int NCH, int SEG>
__device__ __forceinline__ bool moe_one_item(const MoeOneParams& p, uint32_t e, uint32_t item, uint4* lds, float (*part)[DC_ROWS], uint32_t* shared) {
    const uint32_t T = p.sel.tokens, rows_from = T * p.router_blocks, choice_from = rows_from + T * p.slots * p.rows.blocks_per_entry, down_from = choice_from + T;
    if (item < rows_from) {
        moe_one_router<ACT>(p, e, item, lds);
        return true;
    }
    if (item < choice_from) return moe_one_rows<ACT, BITS, NCH>(p, e, item - rows_from, lds, shared);
    if (item < down_from) return moe_one_choice(p, e, item - choice_from, reinterpret_cast<uint32_t*>(lds));
    return moe_one_down<ACT, BITS, SEG>(p, e, item - down_from, reinterpret_cast<float*>(lds), part, shared);
}

// The same as a call, one item at a time: a loop around the steps themselves would be compiled with all that they read loaded ahead of it.
template <int ACT, int BITS, int NCH, int SEG>
__device__ __attribute__((noinline, cold)) void moe_one_item_again(const MoeOneParams* p, uint32_t e, uint32_t item, uint4* lds, float (*part)[DC_ROWS], uint32_t* shared) {
    (void)moe_one_item<ACT, BITS, NCH, SEG>(*p, e, item, lds, part, shared);
}

template <int ACT, int BITS, int NCH, int SEG>
__global__ __launch_bounds__(MOE_ONE_THREADS, 4) void moe_one_kernel(MoeOneParams p) {
    extern __shared__ uint4 one_lds[];
    __shared__ float part[MOE_ONE_SLOTS][DC_ROWS];
    __shared__ uint32_t shared[MOE_ONE_SLOTS];
    const uint32_t e = hand_open(p.hand);
    if (!moe_one_item<ACT, BITS, NCH, SEG>(p, e, blockIdx.x, one_lds, part, shared))
        // What the block waited for in vain, in order, and then its own: never the case while the blocks before it run.
        for (uint32_t item = 0; item <= blockIdx.x; ++item) {
            __syncthreads();
            moe_one_item_again<ACT, BITS, NCH, SEG>(kernel_args<MoeOneParams>(), e, item, one_lds, part, shared);
        }
    hand_close(p.hand, e);
}

}  // namespace nvmai
