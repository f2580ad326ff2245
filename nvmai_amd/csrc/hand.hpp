// Values handed from block to block inside one launch: what lets a launch hold several steps that depend on one another.
//
// A launch that follows another starts 1.6 us after it at the least, and what the other wrote costs its first read a trip past the L2 (4.0 us per launch of a chain
// whose blocks read 8 KB and write a share of them, in a graph).  A value handed on inside a launch is there after 1.4 to 1.8 us, its sum and
// the waiting of 256 blocks included, and a consumer's weights are on their way meanwhile.  (The same with stores, a wait, a counter and then loads is three
// trips one after another: 4.0 to 6.2 us.)
//
// A word of 64 bits carries 32 bits of a value and the number of the launch that wrote it, so a consumer reads the value itself until its
// number is this launch's: relaxed 64-bit atomics of device scope, nothing to order, nothing to clear.
//   - The launch's number: a word of its own per block (hand_open), which the block moves on as it ends (hand_close); block 0 moves the words of blocks that
//     this launch does not have.  A captured launch so has another number at every replay.
//   - A number comes round after 2^32 launches: block 0 clears a stripe of the words that this launch does not use, so that none keeps a number that long.
//   - A consumer does not count on a producer's running beside it: one that has polled `polls` times in vain makes the producers' values itself, in the order of the
//     launch's blocks, and goes on.  Every wait ends so, whatever else holds the device; the same value written twice is the same word.  For that, a launch must not
//     overwrite what its producers read.
#pragma once

#include "common.hpp"

namespace nvmai {

constexpr uint32_t HAND_BLOCKS = 4096;                  // blocks of such a launch at most
constexpr uint32_t HAND_WORDS = 1u << 18;               // words of a context
constexpr size_t HAND_BYTES = HAND_BLOCKS * 4 + (size_t)HAND_WORDS * 8;
constexpr uint32_t HAND_POLLS = 1u << 14;               // about 15 ms

struct Hand {
    uint32_t* numbers;       // [HAND_BLOCKS] the last launch's
    uint64_t* words;         // [HAND_WORDS]
    uint32_t used;           // words of this launch, from the first on
    uint32_t polls;
};

__device__ __forceinline__ uint32_t hand_open(const Hand& h) {
    const uint32_t e = h.numbers[blockIdx.x] + 1u;
    return e ? e : 1u;                                   // 0 is a cleared word's
}

__device__ __forceinline__ void hand_close(const Hand& h, uint32_t e) {
    if (threadIdx.x == 0) h.numbers[blockIdx.x] = e;
    if (blockIdx.x == 0) {
        for (uint32_t i = gridDim.x + threadIdx.x; i < HAND_BLOCKS; i += blockDim.x) h.numbers[i] = e;
        const uint32_t i = e % (HAND_WORDS / 256u) * 256u + threadIdx.x;
        if (i >= h.used && threadIdx.x < 256u) h.words[i] = 0;
    }
}

__device__ __forceinline__ void hand_put(uint64_t* word, float v, uint32_t e) {
    __hip_atomic_store(word, ((uint64_t)e << 32) | __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A wave's words at[lane's index j], all of them this launch's; false where they did not come.
template <int N, typename At>
__device__ __forceinline__ bool hand_take(const Hand& h, uint32_t e, const At& at, float (&v)[N]) {
    for (uint32_t n = 0;; ++n) {
        uint64_t got[N];
        bool ok = true;
#pragma unroll
        for (int j = 0; j < N; ++j) got[j] = __hip_atomic_load(at(j), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int j = 0; j < N; ++j) {
            ok = ok && (uint32_t)(got[j] >> 32) == e;
            v[j] = __uint_as_float((uint32_t)got[j]);
        }
        if (__all(ok)) return true;
        if (n >= h.polls) return false;
        __builtin_amdgcn_s_sleep(1);
    }
}

// The running kernel's first argument where it lies, for a function that is called and not inlined.
template <typename P>
__device__ __forceinline__ const P* kernel_args() {
#if defined(__HIP_DEVICE_COMPILE__)
    return (const P*)__builtin_amdgcn_kernarg_segment_ptr();
#else
    return nullptr;
#endif
}

}  // namespace nvmai
