// Device helpers of the A8 activation quantiser, shared by the kernels that quantise activations
// (kernels/cuda/operators/op30_activation_quantization.py:14-18, 49-65).
#pragma once
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <cstdint>

namespace orx {

// Maximum of a 32-bit key over the wave with data-parallel-primitive moves only: a shuffle is an LDS round trip, and the few-row
// kernels wait for every one of them.  Quad swaps, half-row and row mirrors give every lane its row's maximum; two
// broadcasts carry it across rows into lane 63, which is then read back as a scalar.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp_max_step(uint32_t v) {
    // lanes outside ROW_MASK receive 0, which raises nothing: the move is part of the maximum then (their own value back was three instructions)
    return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xF, ROW_MASK == 0xF));
}
__device__ __forceinline__ uint32_t row_max_u32(uint32_t v) {  // over each row of 16 lanes, known to the row
    v = dpp_max_step<0xB1, 0xF>(v);      // quad_perm [1,0,3,2]
    v = dpp_max_step<0x4E, 0xF>(v);      // quad_perm [2,3,0,1]
    v = dpp_max_step<0x141, 0xF>(v);     // row_half_mirror
    return dpp_max_step<0x140, 0xF>(v);  // row_mirror
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    v = row_max_u32(v);
    v = dpp_max_step<0x142, 0xA>(v);  // row_bcast:15 into rows 1 and 3
    v = dpp_max_step<0x143, 0xC>(v);  // row_bcast:31 into rows 2 and 3
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
// of magnitudes (never NaN, never -0): their bits order as they do
__device__ __forceinline__ float wave_max_magnitude(float v) { return __uint_as_float(wave_max_u32(__float_as_uint(v))); }

// Sum over groups of LANES neighbouring lanes, known to all of them, without an LDS round trip: pairs, quads, mirrored half rows and rows of 16, then the
// swap of two copies' rows and halves, which puts a lane's sum beside its partner's.  All lanes of the wave take part.
template <int FIRST, int LANES>
__device__ __forceinline__ int group_sum(int v) {  // of lanes FIRST, 2 FIRST .. LANES / 2 apart
    if constexpr (FIRST <= 1 && LANES > 1) v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true);
    if constexpr (FIRST <= 2 && LANES > 2) v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true);
    if constexpr (FIRST <= 1 && LANES > 4) v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, true);
    if constexpr (FIRST <= 1 && LANES > 8) v += __builtin_amdgcn_update_dpp(0, v, 0x140, 0xF, 0xF, true);
    if constexpr (FIRST <= 16 && LANES > 16) {
        auto rows = __builtin_amdgcn_permlane16_swap((uint32_t)v, (uint32_t)v, false, false);
        v = (int)(rows[0] + rows[1]);
    }
    if constexpr (LANES > 32) {
        auto halves = __builtin_amdgcn_permlane32_swap((uint32_t)v, (uint32_t)v, false, false);
        v = (int)(halves[0] + halves[1]);
    }
    return v;
}

// fp16 scale of a group from its largest magnitude: max(amax / 127, 2^-24), or 1 for an all-zero group.
__device__ __forceinline__ __half a8_scale(float amax) {
    const float raw_scale = fmaxf(__fdiv_rn(amax, 127.0f), 5.9604644775390625e-08f);
    return amax > 0.f ? __float2half_rn(raw_scale) : __float2half_rn(1.0f);
}

// rint(value / scale), clamped: the product with the reciprocal decides, except within 2^-14 of a
// tie, where the correctly rounded quotient does.  The product is within 4 units in the last place
// of the quotient (|quotient| < 128.5, so 2^-15 at most), so the two round alike everywhere else;
// the reference's kernel takes the same shortcut (kernels/cuda/model/rotation_a8.py:153-164).
__device__ __forceinline__ int8_t quantise(float value, float scale, float inverse) {
    const float guess = value * inverse;
    float r = rintf(guess);
    if (fabsf(fabsf(guess - r) - 0.5f) < 6.103515625e-05f) r = rintf(__fdiv_rn(value, scale));
    return (int8_t)fmaxf(-127.f, fminf(127.f, r));
}

// Four codes packed into one word; one test (and, rarely, four exact quotients) for the four.
// The multiply-add rounds the exact product to an integer (1.5 * 2^23 more; the code is that word's low byte in two's complement),
// and its distance from the product is at most 0.5, so "within 2^-14 of a tie" is "farther than 0.5 - 2^-14 from the rounded value".
// The clamp is on the word: scales below 2^-14 are rounded so coarsely that quotients pass 127; a NaN gives -127.  The hint keeps
// the quotients behind their branch: executed for every value they cost a one-piece form a fifth of its time.
__device__ __forceinline__ uint32_t quantise4(const float (&value)[4], float scale, float inverse) {
    constexpr float kInteger = 12582912.0f;
    float r[4];
    float farthest = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        r[j] = __builtin_fmaf(value[j], inverse, kInteger);
        farthest = fmaxf(farthest, fabsf(__builtin_fmaf(value[j], inverse, kInteger - r[j])));
    }
    if (__builtin_expect(farthest > 0.49993896484375f, 0)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) r[j] = rintf(__fdiv_rn(value[j], scale)) + kInteger;
    }
    uint32_t word[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) word[j] = __float_as_uint(__builtin_amdgcn_fmed3f(r[j], kInteger - 127.f, kInteger + 127.f));
    // byte 0 of the first operand's partner (second argument), then byte 0 of the first argument
    const uint32_t low = __builtin_amdgcn_perm(word[1], word[0], 0x0C0C0400u);
    const uint32_t high = __builtin_amdgcn_perm(word[3], word[2], 0x0C0C0400u);
    return low | (high << 16);
}

typedef _Float16 half_pair __attribute__((ext_vector_type(2)));
// Largest magnitude of `count` pieces of eight fp16 values.  NaN does not count: as largest and smallest value by three-operand instructions that hand a
// NaN on, one instruction to a pair (without its sign through the maximum that drops NaN it is three), and that way only where a NaN came out.
template <int COUNT, typename WORDS>
__device__ __forceinline__ float largest_magnitude(const WORDS (&pieces)[COUNT]) {
    half_pair high = {(_Float16)0.f, (_Float16)0.f}, low = high;
#pragma unroll
    for (int p = 0; p < COUNT; ++p)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const half_pair pair = __builtin_bit_cast(half_pair, (uint32_t)pieces[p][j]);
            high = __builtin_elementwise_maximum(high, pair), low = __builtin_elementwise_minimum(low, pair);
        }
    half_pair largest = __builtin_elementwise_maximum(high, -low);
    if (__builtin_expect(largest[0] != largest[0] || largest[1] != largest[1], 0)) {
        largest = half_pair{(_Float16)0.f, (_Float16)0.f};
#pragma unroll
        for (int p = 0; p < COUNT; ++p)
#pragma unroll
            for (int j = 0; j < 4; ++j) largest = __builtin_elementwise_max(largest, __builtin_bit_cast(half_pair, (uint32_t)(pieces[p][j] & 0x7FFF7FFFu)));
    }
    return fmaxf((float)largest[0], (float)largest[1]);
}

// The codes of such a piece.
template <typename WORDS>
__device__ __forceinline__ uint2 quantise_eight(const WORDS& piece, float scale, float inverse) {
    float value[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const half_pair pair = __builtin_bit_cast(half_pair, (uint32_t)piece[j]);
        value[2 * j] = (float)pair[0], value[2 * j + 1] = (float)pair[1];
    }
    const float low[4] = {value[0], value[1], value[2], value[3]}, high[4] = {value[4], value[5], value[6], value[7]};
    return make_uint2(quantise4(low, scale, inverse), quantise4(high, scale, inverse));
}

// A stable sigmoid in fp32: e = exp(-|gate|), (gate >= 0 ? 1 : e) / (1 + e).
// exp(x) = 2^whole 2^part, whole = rint(x log2 e) (the sum with 1.5 * 2^23 has it in its low bits), part = x log2 e - whole by
// two fused multiply-adds over log2 e as a pair of fp32 numbers: |part| is at most a half, so its rounding is below that of
// the hardware exponential, and one fp32 log2 e alone would cost 1.3e-8 * |x|.  The power of two goes on last because the
// hardware exponential gives 0 instead of subnormal numbers: e is subnormal below -87.4 and 0 from -104 on (2^-150), where
// the argument stops, as the fp32 formula has it; a gate of minus infinity thus gives -inf * 0 = NaN, which a quantiser's
// maximum drops, and not an infinity that would be the row's scale.
// The quotient is the product with the hardware reciprocal and one residual correction: the product is within two units in the
// last place, so the residual is exact and the correction leaves half a unit and a 2^-22 part of one.
// With a correctly rounded exponential of part the largest relative error over all fp16 gates is 1.06e-7 from -1 up, 1.55e-7 in
// [-20, -1) and 6.4e-8 below, as that of a correctly rounded exp and quotient (1.04e-7, 1.55e-7, 5.7e-8); the hardware exponential's
// own unit in the last place comes on top.  Sixteen instructions, two of them transcendental, where the library exponential and
// quotient took about thirty (8192 rows of 17408 values were bound by them).
__device__ __forceinline__ float sigmoid_value(float gate) {
    const float x = fmaxf(-fabsf(gate), -104.f);
    const float shifted = __builtin_fmaf(x, 1.44269502162933349609375f, 12582912.0f);  // fp32(log2 e)
    const float whole = shifted - 12582912.0f;
    const float rest = __builtin_fmaf(x, 1.44269502162933349609375f, -whole);
    const float part = __builtin_fmaf(x, 1.925963033500011e-08f, rest);  // fp32(log2 e - fp32(log2 e))
    const float e = __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(part), __float_as_int(shifted) - 0x4B400000);
    const float denominator = 1.0f + e, numerator = gate >= 0.f ? 1.0f : e;
    const float reciprocal = __builtin_amdgcn_rcpf(denominator);
    const float quotient = numerator * reciprocal;
    return __builtin_fmaf(__builtin_fmaf(-denominator, quotient, numerator), reciprocal, quotient);
}

// fp16(silu(gate) * up) (kernels/cuda/operators/op04_swiglu.py:6-17).
__device__ __forceinline__ float swiglu_value(__half gate, __half up) {
    const float g = __half2float(gate), u = __half2float(up);
    float value = (g * sigmoid_value(g)) * u;
    // opaque: the fp32 product rounds, then the fp16 cast does (a fused multiply-convert rounds once, and which of the
    // two the compiler takes would differ between the kernels that share this)
    asm("" : "+v"(value));
    // the value a downstream quantiser sees is the materialised fp16
    return __half2float(__float2half_rn(value));
}

// ---- nibble planes ------------------------------------------------------------------------------
// The reference's INT4 expert kernels take A8 codes as two planes of u32 words: nibble i of a word holds the low
// (unsigned) or high (signed) nibble of code {0,2,1,3,4,6,5,7}[i] of its group of eight
// (kernels/cuda/model/e8p_core.py:63-78, rotation_a8.py:489-491).  x = codes 0..3, y = codes 4..7, one byte each.
__device__ __forceinline__ uint32_t low_word_first(uint32_t x) { return (x & 0x00000F0Fu) | ((x >> 12) & 0x0000F0F0u); }
__device__ __forceinline__ uint32_t low_word_second(uint32_t y) { return ((y << 16) & 0x0F0F0000u) | ((y << 4) & 0xF0F00000u); }
__device__ __forceinline__ uint32_t high_word_first(uint32_t x) { return ((x >> 4) & 0x00000F0Fu) | ((x >> 16) & 0x0000F0F0u); }
__device__ __forceinline__ uint32_t high_word_second(uint32_t y) { return ((y << 12) & 0x0F0F0000u) | (y & 0xF0F00000u); }
__device__ __forceinline__ uint32_t low_word(uint32_t x, uint32_t y) { return low_word_first(x) | low_word_second(y); }
__device__ __forceinline__ uint32_t high_word(uint32_t x, uint32_t y) { return high_word_first(x) | high_word_second(y); }

// Word j of plane row `row`: row-major (rows, K/8), or K64-major (K/64, rows, 8) (kernels/cuda/model/e8p_prefill.py:79-80)
__device__ __forceinline__ int64_t plane_index(int group_major, int plane_rows, int words, int64_t row, int j) {
    return group_major ? ((int64_t)(j >> 3) * plane_rows + row) * 8 + (j & 7) : row * words + j;
}

}  // namespace orx
