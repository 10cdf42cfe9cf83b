// Device helpers of the MoE router shared by the kernels that select routes
// (kernels/cuda/model/moe.py:413-494): the routing launch itself and the single-token expert
// projection that selects its token's routes in its own set-up.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "a8_device.h"

namespace orx {

// Total order on finite fp32 with -0 == +0 (moe.py:449-465): larger key = larger score.
__device__ __forceinline__ uint32_t ordered_key(float value) {
    const uint32_t bits = __float_as_uint(value);
    if (value == 0.f) return 0x80000000u;
    return (bits & 0x80000000u) ? ~bits : bits ^ 0x80000000u;
}
__device__ __forceinline__ float key_value(uint32_t ordered) {
    return __uint_as_float((ordered & 0x80000000u) ? ordered ^ 0x80000000u : ~ordered);
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) v += __shfl_xor(v, offset, 64);
    return v;
}

// Inclusive sum over the lanes in front, by lane moves: shifts by 1, 2, 4 and 8 within a row of 16, then the last lane of rows 0 and 2 to the row
// behind, then lane 31 to the upper half.  (A shuffle is an LDS round trip, six of them one after another.)
__device__ __forceinline__ int wave_prefix_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);
    return v;
}

// The logits of one row as one wave holds them: LOCAL = ceil(E/64) (rounded up to a power of two) per lane.
template <int LOCAL>
__device__ __forceinline__ void load_route_logits(float (&values)[LOCAL], const float* __restrict__ logits, int e, int lane) {
#pragma unroll
    for (int j = 0; j < LOCAL; ++j) values[j] = logits[min(j * 64 + lane, e - 1)];
}

// What depends on the selected scores alone: lane `rank` has the key of that rank and writes prob[rank].
template <int LOCAL>
__device__ __forceinline__ void route_probabilities(const float (&values)[LOCAL], float local_max, uint32_t my_key, float* prob, int e, int top_k, int renormalize, int lane) {
    float global_max = local_max;
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) global_max = fmaxf(global_max, __shfl_xor(global_max, offset, 64));
    float all_exp = 0.f;
    if (!renormalize) {
#pragma unroll
        for (int j = 0; j < LOCAL; ++j)
            if (j * 64 + lane < e) all_exp += expf(values[j] - global_max);
        all_exp = wave_sum(all_exp);
    }
    const float mine = lane < top_k ? expf(key_value(my_key) - global_max) : 0.f;
    const float selected_sum = wave_sum(mine);
    if (lane < top_k) prob[lane] = __fdiv_rn(mine, renormalize ? selected_sum : all_exp);
}

// The routes of one row, by one wave: the largest score first, the lowest id on ties.  A rank is one maximum of 32-bit keys and
// one ballot per held key for the lowest id that has it; what depends on the score alone waits for the end.  (64-bit keys of
// score and id, with the exponential inside the loop, took 0.3 us a rank.)  Lane `rank` writes ids[rank] and, where `prob` is
// not null, prob[rank].
template <int LOCAL>
__device__ __forceinline__ void select_routes(const float (&values)[LOCAL], int* ids, float* prob, int e, int top_k, int renormalize,
                                              int lane) {
    uint32_t keys[LOCAL];
    uint32_t open = 0;  // bit j: key j is there and not taken yet
    float local_max = -INFINITY;
#pragma unroll
    for (int j = 0; j < LOCAL; ++j) {
        const bool live = j * 64 + lane < e;
        keys[j] = live ? ordered_key(values[j]) : 0u;
        open |= live ? 1u << j : 0u;
        if (live) local_max = fmaxf(local_max, values[j]);
    }
    int my_id = e;
    uint32_t my_key = 0;  // of rank == lane
    for (int rank = 0; rank < top_k; ++rank) {
        uint32_t best = keys[0];
#pragma unroll
        for (int j = 1; j < LOCAL; ++j) best = max(best, keys[j]);
        best = wave_max_u32(best);
        int id = e;  // (never more ranks than ids)
#pragma unroll
        for (int j = LOCAL - 1; j >= 0; --j) {
            const unsigned long long having = __ballot(keys[j] == best && (open >> j & 1u));
            if (having != 0) id = j * 64 + __builtin_ctzll(having);
        }
#pragma unroll
        for (int j = 0; j < LOCAL; ++j)
            if (j * 64 + lane == id) keys[j] = 0u, open &= ~(1u << j);
        if (lane == rank) my_id = id, my_key = best;
    }
    if (lane < top_k) ids[lane] = my_id;
    if (prob != nullptr) route_probabilities<LOCAL>(values, local_max, my_key, prob, e, top_k, renormalize, lane);
}

// The same selection by all waves of a workgroup: a wave counts, for every expert, those of its own share (kShare experts from wave * kShare on) that come in front of it, so a
// rank is the sum over the waves and no rank waits for the one before it.  (One wave, rank after rank: the projection of one token was ready to name
// its expert after 2.7 us with eight of 128, now after 1.9.)
// counts[j]: for expert j * 64 + lane; at most kShare.  lds_keys: LOCAL * 64 words that all waves write the same to, and each reads behind its own writes (readlanes and comparisons of
// every pair for a tie: 17 instructions where these are 5).
template <int LOCAL, int WAVES>
__device__ __forceinline__ void count_in_front(const float (&values)[LOCAL], uint32_t (&counts)[LOCAL], uint32_t* lds_keys, int e, int wave, int lane) {
    constexpr int kShare = LOCAL * 64 / WAVES;
    static_assert(kShare % 4 == 0 && 64 % kShare == 0, "a share is whole reads and lies among the experts of one register");
    uint32_t keys[LOCAL];
#pragma unroll
    for (int j = 0; j < LOCAL; ++j) {
        keys[j] = j * 64 + lane < e ? ordered_key(values[j]) : 0u, counts[j] = 0;  // (behind the end: in front of nobody)
        lds_keys[j * 64 + lane] = keys[j];
    }
    asm volatile("" ::: "memory");
    uint4 share[kShare / 4];
#pragma unroll
    for (int i = 0; i < kShare / 4; ++i) share[i] = reinterpret_cast<const uint4*>(lds_keys + wave * kShare)[i];
    const int own = wave * kShare / 64, first = wave * kShare % 64;
#pragma unroll
    for (int i = 0; i < kShare; ++i) {
        const uint4& four = share[i / 4];
        const uint32_t key = i % 4 == 0 ? four.x : i % 4 == 1 ? four.y : i % 4 == 2 ? four.z : four.w;
        const uint64_t behind = ~1ull << (first + i);  // lanes whose expert in the share's register has a larger id
#pragma unroll
        for (int j = 0; j < LOCAL; ++j) {
            // in front: a larger key, or the same and a smaller id: keys[j] - key - (smaller id) borrows
            const uint64_t smaller = j == own ? behind : j > own ? ~0ull : 0ull;
            uint32_t difference;
            asm("v_subb_co_u32_e64 %0, vcc, %2, %3, %4\n\tv_addc_co_u32_e32 %1, vcc, 0, %1, vcc" : "=&v"(difference), "+v"(counts[j]) : "v"(keys[j]), "v"(key), "s"(smaller) : "vcc");
        }
    }
}

}  // namespace orx
