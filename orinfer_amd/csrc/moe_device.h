// Device helpers of the MoE router shared by the kernels that select routes
// (kernels/cuda/model/moe.py:413-494): the routing launch itself and the single-token expert
// projection that selects its token's routes in its own set-up.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <type_traits>

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

// Sums of lanes 32, 16, 8, 4, 2 and 1 apart, in this order, by lane moves: the swap of two copies' halves (rows) puts a lane's value beside that of its
// partner, and once all are alike 8 apart a turn by 4 within a row is the exchange.  (As shuffles, six LDS round trips one after another.)
__device__ __forceinline__ float wave_sum(float v) {
    auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(halves[0]) + __uint_as_float(halves[1]);
    auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(rows[0]) + __uint_as_float(rows[1]);
    auto from = [](float x, auto control) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(control)::value, 0xF, 0xF, true)); };
    v += from(v, std::integral_constant<int, 0x128>{});  // row_ror:8
    v += from(v, std::integral_constant<int, 0x124>{});  // row_ror:4
    v += from(v, std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
    v += from(v, std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
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
__device__ __forceinline__ void route_probabilities(const float (&values)[LOCAL], uint32_t my_key, float* prob, int e, int top_k, int renormalize, int lane) {
    const float global_max = key_value((uint32_t)__builtin_amdgcn_readfirstlane((int)my_key));  // of rank 0
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

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // (m0 is reserved: it holds nothing of the compiler's from one statement to the next)
// The routes of one row, by one wave: the largest score first, the lowest id on ties.  A rank is one maximum of 32-bit keys and
// one ballot per held key for the lowest id that has it; what depends on the score alone waits for the end.  (64-bit keys of
// score and id, with the exponential inside the loop, took 0.3 us a rank.)  Lane `rank` writes ids[rank] and, where `prob` is
// not null, prob[rank].
// With many rows this is bound by its instructions: which keys are taken is kept as scalar masks, and a rank's id and key are put into their lane as
// they are, 15 vector instructions a rank with two keys a lane instead of 45.
template <int LOCAL>
__device__ __forceinline__ void select_routes(const float (&values)[LOCAL], int* ids, float* prob, int e, int top_k, int renormalize,
                                              int lane) {
    uint32_t keys[LOCAL];
    uint64_t open[LOCAL];  // lanes whose key j is there and not taken yet
#pragma unroll
    for (int j = 0; j < LOCAL; ++j) {
        const bool live = j * 64 + lane < e;
        keys[j] = live ? ordered_key(values[j]) : 0u;
        open[j] = __ballot(live);
    }
    uint32_t my_id = (uint32_t)e, my_key = 0;  // of rank == lane
    const int ranks = __builtin_amdgcn_readfirstlane(top_k);
    for (int rank = 0; rank < ranks; ++rank) {
        uint32_t best = keys[0];
#pragma unroll
        for (int j = 1; j < LOCAL; ++j) best = max(best, keys[j]);
        best = wave_max_u32(best);
        int chosen = -1;  // (never more ranks than ids)
        uint64_t lowest = 0;
#pragma unroll
        for (int j = LOCAL - 1; j >= 0; --j) {
            const uint64_t having = __ballot(keys[j] == best) & open[j];
            if (having != 0) chosen = j, lowest = having;
        }
        lowest &= 0 - lowest;
        const uint32_t id = chosen < 0 ? (uint32_t)e : (uint32_t)(chosen * 64 + __builtin_ctzll(lowest));
#pragma unroll
        for (int j = 0; j < LOCAL; ++j) {
            const uint64_t taken = j == chosen ? lowest : 0;
            open[j] &= ~taken;
            asm("v_cndmask_b32_e64 %0, %0, 0, %1" : "+v"(keys[j]) : "s"(taken));
        }
        // (an instruction reads one scalar register: the lane's number goes by m0)
        asm("s_mov_b32 m0, %4\n\ts_nop 0\n\tv_writelane_b32 %0, %2, m0\n\tv_writelane_b32 %1, %3, m0"
            : "+v"(my_id), "+v"(my_key)
            : "s"(id), "s"(best), "s"(__builtin_amdgcn_readfirstlane(rank))
            : "m0");
    }
    if (lane < top_k) ids[lane] = (int)my_id;
    if (prob != nullptr) route_probabilities<LOCAL>(values, my_key, prob, e, top_k, renormalize, lane);
}
#pragma clang diagnostic pop

// The same selection by all waves of a workgroup: a wave counts, for every expert, those of its own share (kShare experts from wave * kShare on) that come in front of it, so a
// rank is the sum over the waves and no rank waits for the one before it.  (One wave, rank after rank: the projection of one token was ready to name
// its expert after 2.7 us with eight of 128, now after 1.9.)
// counts[j]: for expert j * 64 + lane; at most kShare.  lds_keys: LOCAL * 64 words that all waves write the same to, and each reads behind its own writes.  Two
// instructions a pair and a wait for every four pairs; the layer of one token takes what it took without the waits, 10.3 us with 8 of 128 experts, 2048 x 512.
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
    for (int i = 0; i < kShare; i += 4) {
        const uint4& key = share[i / 4];
        uint64_t behind[4];  // lanes whose expert in the share's register has a larger id
#pragma unroll
        for (int q = 0; q < 4; ++q) behind[q] = ~1ull << (first + i + q);
#pragma unroll
        for (int j = 0; j < LOCAL; ++j) {
            // In front: a larger key, or the same and a smaller id: keys[j] - key - (smaller id) borrows.  Four at a time, each with a borrow of its own: between a vector
            // instruction that writes a scalar register and one that reads it stand two others, which nobody sees to inside an asm statement.  (s_nop: the masks may come from one too.)
            uint64_t smaller[4], borrow[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) smaller[q] = j == own ? behind[q] : j > own ? ~0ull : 0ull;
            uint32_t difference;
            asm("s_nop 1\n\t"
                "v_subb_co_u32_e64 %0, %2, %6, %7, %11\n\t"
                "v_subb_co_u32_e64 %0, %3, %6, %8, %12\n\t"
                "v_subb_co_u32_e64 %0, %4, %6, %9, %13\n\t"
                "v_subb_co_u32_e64 %0, %5, %6, %10, %14\n\t"
                "v_addc_co_u32_e64 %1, %2, 0, %1, %2\n\t"
                "v_addc_co_u32_e64 %1, %3, 0, %1, %3\n\t"
                "v_addc_co_u32_e64 %1, %4, 0, %1, %4\n\t"
                "v_addc_co_u32_e64 %1, %5, 0, %1, %5"
                : "=&v"(difference), "+v"(counts[j]), "=&s"(borrow[0]), "=&s"(borrow[1]), "=&s"(borrow[2]), "=&s"(borrow[3])
                : "v"(keys[j]), "v"(key.x), "v"(key.y), "v"(key.z), "v"(key.w), "s"(smaller[0]), "s"(smaller[1]), "s"(smaller[2]), "s"(smaller[3]));
        }
    }
}

}  // namespace orx
