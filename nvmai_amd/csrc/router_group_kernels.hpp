// Router, selection and work list of a small decode batch in one launch.
//
// As two launches (router_logits_kernel, select_group_kernel) the step is bound by two chains of trips to memory, the start of a launch and the trip past the L2 that
// fetches what the other wrote.  Here the logits are handed on inside the launch (hand.hpp): blocks of the router's rows, then blocks that choose for
// four tokens each, a wave per token, then one block that groups the chosen pairs by expert, so that a block's producers stand before it.  d 2048, 256 experts: 16 tokens
// 8.3 + 7.9 -> 13.9 us with the norm before them, 32 tokens 7.3 + 9.5 -> 14.1 without.  A layer of 512 wide experts at 4 bits: 8 tokens 45.3 -> 44.1 us, 16 61.0 -> 58.7, 24 75.1 -> 71.0,
// 32 85.9 -> 82.2; at 8 bits 32 128.0 -> 125.2, 63 181.2 -> 179.2.
#pragma once

#include "hand.hpp"
#include "moe_kernels.hpp"

namespace nvmai {

struct RouterGroupParams {
    RouterParams router;         // logits unused
    GroupParams group;           // ticket unused
    Hand hand;
    uint32_t router_blocks;      // per token
};

constexpr uint32_t RG_THREADS = 256;
constexpr uint32_t RG_ROWS = RG_THREADS / 32;                // rows of the router per block
constexpr uint32_t RG_TOKENS = RG_THREADS / 64;              // tokens per block that chooses

// Words: the logits of every token (those of the experts that a lane takes lie 64 apart, so that a load is of neighbours), then the chosen experts.
__host__ __device__ inline uint32_t rg_per_lane(uint32_t experts) { return experts <= 256 ? 4 : TOPK_MAX_PER_LANE; }
__host__ __device__ inline uint32_t rg_logit_words(uint32_t experts) { return 64 * rg_per_lane(experts); }
__host__ __device__ inline uint32_t rg_words(uint32_t tokens, uint32_t experts, uint32_t top_k) { return tokens * (rg_logit_words(experts) + top_k); }

template <int ACT, int CPL>
__device__ __forceinline__ void rg_router(const RouterGroupParams& p, uint32_t e, uint32_t item, uint32_t* lds) {
    const RouterParams& r = p.router;
    const uint32_t t = item / p.router_blocks, b = item % p.router_blocks;
    const int hw = threadIdx.x >> 5, hl = threadIdx.x & 31;
    const uint32_t row = b * RG_ROWS + hw;
    const bool live = row < r.num_experts + (r.gate.kind ? 1u : 0u), is_gate = row >= r.num_experts;
    const RowsDesc& rd = is_gate ? r.gate : r.router;
    uint16_t* const xl = reinterpret_cast<uint16_t*>(lds);
    RouterRowRegs<CPL> g;
    if (live) router_row_prefetch<CPL>(r, rd, is_gate ? 0u : row, hl, g);      // in flight while the inputs are staged
    if (r.pre_weight) {
        const PreNormArgs a{(const uint16_t*)r.x, r.x_stride, r.pre_delta, r.pre_delta_stride, r.pre_weight, r.pre_hidden_out,
                            r.pre_hidden_stride, r.pre_normed_out, r.pre_normed_stride, r.pre_eps, r.d};
        stage_prenorm_rows<ACT>(a, t, 1, xl, xl + r.d, b == 0);
    } else {
        router_stage_x(r, t, 1, xl);
    }
    if (!live) return;                               // uniform per half-wave
    float acc[1];
    router_row_any<ACT, CPL>(r, rd.kind, g, xl, 1, hl, acc);
    if (hl != 0) return;
    const uint32_t per = rg_per_lane(r.num_experts);
    if (is_gate) r.gate_logit[t] = acc[0];
    else hand_put(p.hand.words + (size_t)t * rg_logit_words(r.num_experts) + 64u * (row % per) + row / per, acc[0], e);
}

template <int PER>
__device__ __forceinline__ bool rg_choose(const RouterGroupParams& p, uint32_t e, uint32_t t, int lane) {
    const SelectParams& sel = p.group.sel;
    const uint64_t* const words = p.hand.words + (size_t)t * rg_logit_words(sel.num_experts);
    float val[PER];
    // past the last expert: the last one's word again
    if (!hand_take<PER>(p.hand, e, [&](int j) { const uint32_t x = min((uint32_t)(PER * lane + j), sel.num_experts - 1u); return words + 64u * (x % PER) + x / PER; }, val))
        return false;
    float score;
    uint32_t idx;
    select_topk_values<PER>(sel, val, lane, score, idx, sel.top_k);
    uint64_t* const chosen = p.hand.words + (size_t)sel.tokens * rg_logit_words(sel.num_experts) + (size_t)t * sel.top_k;
    if ((uint32_t)lane < sel.top_k) hand_put(chosen + lane, __uint_as_float(idx), e);
    select_store_routes(sel, t, lane, score, idx);
    return true;
}

__device__ __forceinline__ bool rg_list(const RouterGroupParams& p, uint32_t e, uint32_t* lds) {
    const SelectParams& sel = p.group.sel;
    const uint32_t pairs = sel.tokens * sel.top_k;
    uint32_t* const idx = lds + 4u * sel.num_experts + 8u + pairs;             // behind what build_work_list keeps
    const uint64_t* const chosen = p.hand.words + (size_t)sel.tokens * rg_logit_words(sel.num_experts);
    clear_work_list(p.group, lds);
    bool ok = true;
    for (uint32_t i0 = threadIdx.x & ~63u; i0 < pairs; i0 += RG_THREADS) {     // uniform per wave
        const uint32_t i = min(i0 + (threadIdx.x & 63u), pairs - 1u);
        float v[1];
        ok = ok && hand_take<1>(p.hand, e, [&](int) { return chosen + i; }, v);
        idx[i] = __float_as_uint(v[0]);
    }
    if (!__syncthreads_and(ok)) return false;
    build_work_list(p.group, lds, idx);
    return true;
}

template <int ACT, int CPL>
__device__ __forceinline__ bool rg_item(const RouterGroupParams& p, uint32_t e, uint32_t item, uint32_t* lds) {
    const SelectParams& sel = p.group.sel;
    const uint32_t choose_from = sel.tokens * p.router_blocks, list = choose_from + (sel.tokens + RG_TOKENS - 1u) / RG_TOKENS;
    if (item < choose_from) {
        rg_router<ACT, CPL>(p, e, item, lds);
        return true;
    }
    if (item == list) return rg_list(p, e, lds);
    const uint32_t t = (item - choose_from) * RG_TOKENS + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    bool ok = true;
    if (t < sel.tokens) ok = sel.num_experts <= 256 ? rg_choose<4>(p, e, t, lane) : rg_choose<TOPK_MAX_PER_LANE>(p, e, t, lane);
    return __syncthreads_and(ok);
}

template <int ACT, int CPL>
__device__ __attribute__((noinline, cold)) void rg_item_again(const RouterGroupParams* p, uint32_t e, uint32_t item, uint32_t* lds) {
    (void)rg_item<ACT, CPL>(*p, e, item, lds);
}

template <int ACT, int CPL>
__global__ __launch_bounds__(RG_THREADS, 4) void router_group_kernel(RouterGroupParams p) {
    extern __shared__ uint4 rg_lds[];
    uint32_t* const lds = reinterpret_cast<uint32_t*>(rg_lds);
    const uint32_t e = hand_open(p.hand);
    if (!rg_item<ACT, CPL>(p, e, blockIdx.x, lds))
        // What the block waited for in vain, in order, and then its own: never the case while the blocks before it run.
        for (uint32_t item = 0; item <= blockIdx.x; ++item) {
            __syncthreads();
            rg_item_again<ACT, CPL>(kernel_args<RouterGroupParams>(), e, item, lds);
        }
    hand_close(p.hand, e);
}

}  // namespace nvmai
