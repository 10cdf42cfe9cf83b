// Projections of two-stage (Q4) codes and of int8 weights for some dozens of rows to some thousand: token rows as packed panels, straight into
// the operand registers, the weights of a workgroup decoded (or brought) once into LDS.
//
// Reference counterparts: the Tensor Core schedules of kernels/cuda/model/integer_core.py behind
// kernels/cuda/model/e8p_q4.py:143-264 and int8_projection.py:15-62.  Arithmetic: exact int32 over the full K, (float(acc) * ws) * as.
//
//  * The quantiser leaves the int8 rows as panels besides (k_quant.hip): 1 KiB for 16 rows and 64 of K, in the order in which the
//    lanes of v_mfma_i32_16x16x64_i8 hold them: half s of a chunk of 128, lane (quarter q, row i): bytes [32 q + 16 s, +16) of row i,
//    the weights that the 16 bytes of codes of a lane (quarter q of a chunk) decode to.  A wave loads a fragment as 1 KiB in a row
//    (108-115 GB/s per CU, all CUs reading the same rows with 16 loads a wave in flight; out of row-major memory 16 rows x 64 bytes at a time 35 GB/s).  Through LDS,
//    as k_gemm_big.hip's 512-row runs take row-major rows, whole lines arrive as fast, but what is in flight has to have its place there: 128 of the
//    160 KiB, which leaves the decode tables without copies and every lookup in bank conflicts.
//  * A workgroup owns up to 512 token rows and a run of up to CB blocks of 16 channels over the whole K; wave w of eight owns TB or TB - 1 blocks
//    of 16 rows (w, w + 8, ...) and all channels of the run.  The tokens of D MFMA slices of 64 are on their way in registers (TB D = 16 KiB a wave).
//  * K goes by in phases of PH chunks of 128.  While the weights of one phase are multiplied, those of the next are decoded: a unit is 16
//    channels x 128 of K, 16 bytes of codes to a lane, four lookups a code in tables of eight copies (QuadLookup: no bank conflicts),
//    and what a lane decodes is what a lane of the fragment reads, so both sides of the LDS are linear.  One barrier a phase, behind its
//    second last slice.  Row sums (75 times them comes off, see QuadLookup) are the quantiser's.
//  * int8 weights go to the same places by direct-to-LDS loads, two to a unit, in the first slices of the phase before.
//
// What bounds it: the token stream and the LDS (fragments 8 KiB x CB a slice for the eight waves, lookups 4 KiB x CB), which add up more than they overlap:
// 64 of K take 0.08 us per 16 KiB of tokens and 0.045 us per channel block, the multiplies beside them 0.005 us per block of 16 x 16 and wave.  17408 x 5120 at 512
// rows, us: 49.5; without the token requests 40.7, without the lookups 44.9, with a quarter of the multiplies 44.3.  Four waves of twice the rows (half the fragment
// reads, sums in accumulation registers) 50-54, eight token slices instead of four, two slices to a step, a raised wave priority, lookups
// put together later: all within 2 %.  Against the best of all other kernels, with the A8 quantiser in front of either (here 0.2-0.7 us slower up to 512 rows, for the second
// copy of the codes), graphs whose weights come from memory, K-major: 17408 x 5120 at 200 / 512 rows 55.4 / 72.4 -> 34.4 / 53.8, 7168 x 5120 at 200 / 256 / 512 rows 26.1 / 41.9 /
// 56.4 -> 23.1 / 25.9 / 40.4, 9728 x 2560 at 200 / 512 29.2 / 39.7 -> 17.6 / 27.1; with one set of weights, in cache, 0.7 to 3 us less over panels and 1 to 7 without.
#include <hip/hip_fp16.h>

#include <algorithm>
#include <type_traits>

#include "e8p_device.h"
#include "lds_asm.h"
#include "orx_internal.h"

namespace orx {

uint32_t gemm_tall_units(int n);  // k_gemm_big.hip: workgroups of at most five blocks of 16 channels, whole rounds of the CUs
constexpr int kPanelMaxRows = 2048;

namespace {

using namespace lds_asm;

#define ORX_INLINE __attribute__((always_inline))

constexpr int kPanelWaves = 8, kPanelThreads = kPanelWaves * 64, kPanelRows = 512;

struct PanelParams {
    const uint8_t* panels;
    const int* sums;
    const uint8_t* w;
    const uint32_t* book;
    const __half* ws;
    const __half* as;
    void* out;
    int n, k, stride, m, out_f32;
    int tile_rows;                                   // rows of a row tile, a multiple of 16
    uint32_t row_stride, chunk_stride, half_stride;  // code bytes between channels, K chunks of 128, and halves of a chunk
};

enum PanelCodec { kPanelQ4 = 0, kPanelW8 = 1 };
template <int CODEC>
constexpr uint32_t kPanelWeights = CODEC == kPanelQ4 ? kQuadTableBytes<256> : 0;
template <int CB>
constexpr int kPhaseChunks = CB <= 2 ? 8 : 4;
template <int CB>
constexpr uint32_t kPhaseBytes = CB * kPhaseChunks<CB> * 2048;
template <int CODEC, int CB>
constexpr uint32_t kPanelScales = kPanelWeights<CODEC> + 2 * kPhaseBytes<CB>;  // 512 token scales, 512 sums, 16 CB channel scales
template <int CODEC, int CB>
constexpr uint32_t kPanelLds = kPanelScales<CODEC, CB> + kPanelRows * 8 + CB * 64;

template <int OFFSET>
__device__ __forceinline__ void write_16_at(uint32_t address, v4u value) {
    asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(address), "v"(value), "n"(OFFSET) : "memory");
}

// EVEN: every wave has TB blocks of rows (a branch less, and all multiplies to put the side work behind: 17408 x 5120 at 512 rows 51.2 -> 49.9; the other form leaves
// out what is not there: 7168 x 5120 at 130 / 200 rows 18.4 / 19.2 -> 16.2 / 18.3, 17408 x 5120 at 130 rows 31.1 -> 28.1)
template <int CODEC, int TB, int CB, bool EVEN>
__global__ __launch_bounds__(kPanelThreads) void panel_kernel(PanelParams p) {
    constexpr bool Q4 = CODEC == kPanelQ4;
    constexpr uint32_t kWeights = kPanelWeights<CODEC>, kScales = kPanelScales<CODEC, CB>;
    constexpr int PH = kPhaseChunks<CB>, S = 2 * PH;      // chunks and MFMA slices of a phase
    constexpr int D = 4;                                  // token slices on their way (eight are not faster)
    constexpr int UNITS = PH * CB, U = (UNITS + kPanelWaves - 1) / kPanelWaves;
    constexpr bool kUneven = UNITS % kPanelWaves != 0;    // the last unit of a phase is some waves' only
    static_assert((Q4 ? 2 * U + 1 < S : U + D < S) && S % D == 0 && S - 1 > D, "the decode of a phase ends in front of its barrier");
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int column = lane & 15, quarter = lane >> 4;
    const int blocks = (p.n + 15) / 16;
    const int first_block = (int)((int64_t)blockIdx.x * blocks / gridDim.x), end_block = (int)((int64_t)(blockIdx.x + 1) * blocks / gridDim.x);
    const int first_channel = first_block * 16, channels = min(end_block * 16, p.n) - first_channel;
    const int first_row = (int)blockIdx.y * p.tile_rows, rows = min(p.tile_rows, p.m - first_row);
    const int chunks = p.k / 128;

    // ---- requests: what the set-up needs, the codes of two phases, the first token slices ----
    uint32_t selector = 0, token_scale_bits, channel_scale_bits;
    int row_sum = 0;
    {
        const uint32_t entry_at = (uint32_t)(tid & 255) * 4, row_at = (uint32_t)min(tid, rows - 1), channel_at = (uint32_t)min(tid, channels - 1);
        if constexpr (Q4) asm volatile("global_load_dword %0, %1, %2" : "=v"(selector) : "v"(entry_at), "s"(uniform_pointer(p.book)) : "memory");
        asm volatile("global_load_ushort %0, %1, %2" : "=v"(token_scale_bits) : "v"(row_at * 2), "s"(uniform_pointer(p.as + first_row)) : "memory");
        if constexpr (Q4) asm volatile("global_load_dword %0, %1, %2" : "=v"(row_sum) : "v"(row_at * 4), "s"(uniform_pointer(p.sums + first_row)) : "memory");
        asm volatile("global_load_ushort %0, %1, %2" : "=v"(channel_scale_bits) : "v"(channel_at * 2), "s"(uniform_pointer(p.ws + first_channel)) : "memory");
    }
    const uint8_t* const w_base = uniform_pointer(p.w + (int64_t)first_channel * p.row_stride);
    // units of this wave: unit u is number wave + 8 u of the phase, chunk number / CB of it and channel block number % CB
    int unit_chunk[U];
    uint32_t unit_codes[U], unit_weights[U];
    Each<U>::run([&](auto tag) ORX_INLINE {
        constexpr int u = decltype(tag)::value;
        const int number = min(wave + kPanelWaves * u, UNITS - 1), block = number % CB;
        unit_chunk[u] = number / CB;
        unit_codes[u] = (uint32_t)min(16 * block + column, channels - 1) * p.row_stride;
        if constexpr (Q4)
            unit_codes[u] += (uint32_t)(quarter >> 1) * p.half_stride + (uint32_t)(quarter & 1) * 16;
        else
            unit_codes[u] += (uint32_t)quarter * 32;
        unit_weights[u] = kWeights + (uint32_t)(unit_chunk[u] * 2 * CB + block) * 1024 + (Q4 ? (uint32_t)lane * 16 : 0u);
    });
    const bool last_unit = !kUneven || wave + kPanelWaves * (U - 1) < UNITS;
    v4u codes[U];
    auto request_codes = [&](int phase, auto tag, v4u& to) ORX_INLINE {
        constexpr int u = decltype(tag)::value;
        load_16(to, unit_codes[u], w_base + (uint64_t)(uint32_t)min(phase * PH + unit_chunk[u], chunks - 1) * p.chunk_stride);
    };
    auto bring = [&](int phase, auto tag) ORX_INLINE {  // int8: a unit of a phase to its place
        constexpr int u = decltype(tag)::value;
        const uint8_t* const from = w_base + (uint64_t)(uint32_t)min(phase * PH + unit_chunk[u], chunks - 1) * p.chunk_stride;
        const uint32_t to = unit_weights[u] + (phase & 1 ? kPhaseBytes<CB> : 0u);
        if (u < U - 1 || last_unit) request_16<0>(unit_codes[u], from, to), request_16<0>(unit_codes[u] + 16, from, to + CB * 1024);
    };
    const int row_blocks = (rows + 15) / 16;
    const uint8_t* token_base[TB];
    Each<TB>::run([&](auto tag) ORX_INLINE {
        constexpr int i = decltype(tag)::value;
        token_base[i] = uniform_pointer(p.panels + (int64_t)(first_row / 16 + min(i * kPanelWaves + wave, row_blocks - 1)) * 16 * p.k);
    });
    const bool last_block = EVEN || (TB - 1) * kPanelWaves + wave < row_blocks;  // (all others every wave has: row_blocks > 8 (TB - 1), see panel_shape)
    v4i token[D][TB];
    const int last_slice = 2 * chunks - 1;
    auto token_offset = [&](int slice) ORX_INLINE { return (uint32_t)lane * 16 + (uint32_t)min(slice, last_slice) * 1024; };
    auto request_token = [&](v4i& to, uint32_t offset, const uint8_t* base) ORX_INLINE {
        asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(to) : "v"(offset), "s"(base) : "memory");
    };
    v4u first_codes[U];
    if constexpr (Q4) {
        Each<U>::run([&](auto tag) ORX_INLINE { request_codes(0, tag, first_codes[decltype(tag)::value]); });
        Each<U>::run([&](auto tag) ORX_INLINE { request_codes(1, tag, codes[decltype(tag)::value]); });
    } else {
        Each<U>::run([&](auto tag) ORX_INLINE { bring(0, tag); });
    }
    Each<D>::run([&](auto s_tag) ORX_INLINE {
        const uint32_t offset = token_offset(decltype(s_tag)::value);
        Each<TB>::run([&](auto i_tag) ORX_INLINE {
            constexpr int i = decltype(i_tag)::value;
            if (i < TB - 1 || last_block) request_token(token[decltype(s_tag)::value][i], offset, token_base[i]);
        });
    });

    // ---- tables: half an entry to a thread ----
    constexpr int kLater = (Q4 ? 2 * U : 0) + (TB - 1) * D;  // at least
    asm volatile("s_waitcnt vmcnt(%4)" : "+v"(selector), "+v"(token_scale_bits), "+v"(row_sum), "+v"(channel_scale_bits) : "n"(kLater > 63 ? 63 : kLater));
    if constexpr (Q4) {
        const uint32_t entry = (uint32_t)tid & 255, half = (uint32_t)tid >> 8, turn = entry & 7;
        const int shift = half ? 0 : 2;
        const uint2 basis = byte_basis_biased(selector, shift), mask = byte_mask_biased(entry, shift);
        const bool swap = (turn & 4) != 0;
        const v4u low = swap ? v4u{mask.x, mask.y, mask.x, mask.y} : v4u{basis.x, basis.y, basis.x, basis.y};
        const v4u high = swap ? v4u{basis.x, basis.y, basis.x, basis.y} : v4u{mask.x, mask.y, mask.x, mask.y};
        const uint32_t at = entry * 256 + half * 128;
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) lds_write_16(at + ((i ^ turn) * 16), i < 4 ? low : high);
    }
    {
        const uint32_t scales = kScales + (uint32_t)tid * 4;
        const float token_scale = __half2float(__ushort_as_half((unsigned short)token_scale_bits));
        asm volatile("ds_write_b32 %0, %1" ::"v"(scales), "v"(token_scale) : "memory");
        asm volatile("ds_write_b32 %0, %1" ::"v"(scales + kPanelRows * 4), "v"(row_sum) : "memory");
        if (tid < 16 * CB) {
            const float channel_scale = __half2float(__ushort_as_half((unsigned short)channel_scale_bits));
            asm volatile("ds_write_b32 %0, %1" ::"v"(scales + kPanelRows * 8), "v"(channel_scale) : "memory");
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    // ---- the decode: two codes a slice, looked up in one and put together in the next ----
    const QuadLookup<256> lookup(lane);
    v2u entry[2][4];
    auto read_code = [&](auto w_tag, uint32_t code) ORX_INLINE {
        constexpr int w = decltype(w_tag)::value;
        lookup.template read<0>(entry[w][0], code);
        lookup.template read<1>(entry[w][1], code);
        lookup.template read<2>(entry[w][2], code);
        lookup.template read<3>(entry[w][3], code);
    };
    auto combine = [&]() ORX_INLINE {
        v4u out;
#pragma unroll
        for (int w = 0; w < 2; ++w)
#pragma unroll
            for (int d = 0; d < 2; ++d) out[2 * w + d] = (entry[w][0][d] ^ entry[w][1][d]) + (entry[w][2][d] ^ entry[w][3][d]);
        return out;
    };
    auto keep_entries = [&]() ORX_INLINE {
#pragma unroll
        for (int w = 0; w < 2; ++w)
#pragma unroll
            for (int e = 0; e < 4; ++e) keep(entry[w][e]);
    };
    std::integral_constant<int, 0> zero;
    std::integral_constant<int, 1> one;
    // the first phase by itself
    if constexpr (!Q4) {
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((TB - 1) * D) : "memory");
    } else {
        constexpr int kAfter = U + (TB - 1) * D;
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kAfter > 63 ? 63 : kAfter) : "memory");
        Each<U>::run([&](auto tag) ORX_INLINE { keep(first_codes[decltype(tag)::value]); });
        Each<U>::run([&](auto tag) ORX_INLINE {
            constexpr int u = decltype(tag)::value;
            if (u < U - 1 || last_unit) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    read_code(zero, first_codes[u][2 * h]);
                    read_code(one, first_codes[u][2 * h + 1]);
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    keep_entries();
                    lds_write_16(unit_weights[u] + (uint32_t)h * (CB * 1024), combine());
                }
            }
        });
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }

    v4i acc[TB][CB];
#pragma unroll
    for (int i = 0; i < TB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            acc[i][j] = v4i{0, 0, 0, 0};
            keep(acc[i][j]);
        }
    v4i weight[2][CB];
    uint32_t phase_weights = kWeights + (uint32_t)lane * 16;  // of the phase that is multiplied
    Each<CB>::run([&](auto tag) ORX_INLINE { lds_read_16<decltype(tag)::value * 1024>(weight[0][decltype(tag)::value], phase_weights); });
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
        for (int e = 0; e < 4; ++e) entry[w][e] = v2u{0, 0};

    int phase = 0;
    uint32_t other = kPhaseBytes<CB>;  // from the buffer that is multiplied to the one that is written, modulo 2^32
    // One slice: its operands were requested before; the next slice's weights, the next lookups and token slice + D go out between its
    // multiplies.
    auto slice = [&](auto s_tag) ORX_INLINE {
        constexpr int s = decltype(s_tag)::value, set = s & 1, token_set = s % D;
        constexpr bool kLooksUp = Q4 && s < 2 * U, kPutsTogether = Q4 && s >= 1 && s <= 2 * U;
        constexpr int u = s / 2, before = (s - 1) / 2;
        // this slice's tokens, and with them the codes, which were requested S - 1 slices ago: at most the tokens of D - 1 slices are younger
        if (last_block)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(TB * (D - 1)) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((TB - 1) * (D - 1)) : "memory");
        Each<CB>::run([&](auto tag) ORX_INLINE { keep(weight[set][decltype(tag)::value]); });
        Each<TB>::run([&](auto tag) ORX_INLINE { keep(token[token_set][decltype(tag)::value]); });
        if constexpr (kLooksUp) keep(codes[u]);
        if constexpr (s == S - 1) asm volatile("s_barrier" ::: "memory");  // the next phase is written, and nobody reads this one any more
        if constexpr (kPutsTogether) {
            keep_entries();
            if (before < U - 1 || last_unit) write_16_at<((s - 1) & 1) * (CB * 1024)>(unit_weights[before] + (phase & 1 ? 0u : kPhaseBytes<CB>), combine());
        }
        const uint32_t offset = token_offset(phase * S + s + D);
        const uint32_t next = s == S - 1 ? phase_weights + other : phase_weights;
        // Side work behind the multiplies that every wave has, one piece each where there are that many: two codes of four lookups, then CB fragment
        // reads (what goes out last is waited for first, at the next slice's start).
        constexpr int kBefore = Q4 ? 2 : 0, kMultiplies = (EVEN ? TB : TB - 1) * CB, kSide = CB + kBefore, kSpan = kMultiplies < 2 * kSide ? kMultiplies : 2 * kSide;
        Each<kMultiplies>::run([&](auto m_tag) ORX_INLINE {
            constexpr int m = decltype(m_tag)::value, i = m / CB, j = (i & 1) ? CB - 1 - m % CB : m % CB;
            multiply_in_place<false>(acc[i][j], weight[set][j], token[token_set][i]);
            constexpr int from = m * kSide / kSpan, to = (m + 1) * kSide / kSpan;
            Each<kSide>::run([&](auto n_tag) ORX_INLINE {
                constexpr int n = decltype(n_tag)::value;
                if constexpr (n >= from && n < to) {
                    if constexpr (n >= kBefore) {
                        lds_read_16<((s + 1) % S) * (CB * 1024) + (n - kBefore) * 1024>(weight[set ^ 1][n - kBefore], next);
                    } else if constexpr (kLooksUp) {
                        if (u < U - 1 || last_unit) read_code(std::integral_constant<int, n>{}, codes[u][2 * (s & 1) + n]);
                    }
                }
            });
            if constexpr (m % CB == CB - 1) request_token(token[token_set][i], offset, token_base[i]);
        });
        // (Here and behind `done` stretches of code meet with multiplies and requests on their way, of which the compiler knows nothing: it must move no sum and no
        // token between registers there.  It has no reason to, and tests/test_codegen.py finds it in the built kernels if it does; a pause of 16 cycles a slice would
        // take its place.)
        if (!EVEN && last_block) {
            Each<CB>::run([&](auto j_tag) ORX_INLINE {
                constexpr int i = TB - 1, j = (i & 1) ? CB - 1 - decltype(j_tag)::value : decltype(j_tag)::value;
                multiply_in_place<false>(acc[i][j], weight[set][j], token[token_set][i]);
            });
            request_token(token[token_set][TB - 1], offset, token_base[TB - 1]);
        }
        // (in front of the tokens of slice S - 1 - D, so that the wait of slice S - 1 covers them)
        if constexpr (!Q4 && s < U) bring(phase + 1, std::integral_constant<int, (s < U ? s : 0)>{});
        if constexpr (kLooksUp && (s & 1) == 1) request_codes(phase + 2, std::integral_constant<int, u>{}, codes[u]);
    };
    for (;; ++phase) {
        const int here = 2 * (chunks - phase * PH);  // slices left
        bool done = false;
        Each<S>::run([&](auto tag) ORX_INLINE {
            constexpr int s = decltype(tag)::value;
            if constexpr (s > 0 && s % 2 == 0) done = done || s >= here;
            if (!done) slice(tag);
        });
        asm volatile("s_nop 15" ::: "memory");
        if (here <= S) break;
        phase_weights += other, other = 0u - other;
    }
    // what is still on its way lands before its registers are anybody else's
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    Each<D>::run([&](auto s_tag) ORX_INLINE { Each<TB>::run([&](auto tag) ORX_INLINE { keep(token[decltype(s_tag)::value][decltype(tag)::value]); }); });
    Each<CB>::run([&](auto tag) ORX_INLINE { keep(weight[0][decltype(tag)::value]), keep(weight[1][decltype(tag)::value]); });
    if constexpr (Q4) {
        Each<U>::run([&](auto tag) ORX_INLINE { keep(codes[decltype(tag)::value]); });
        keep_entries();
    }
    Each<TB>::run([&](auto i_tag) ORX_INLINE { Each<CB>::run([&](auto j_tag) ORX_INLINE { keep(acc[decltype(i_tag)::value][decltype(j_tag)::value]); }); });
    asm volatile("s_barrier" ::: "memory");  // tables and weights are nobody's any more

    // ---- epilogue: blocks of 16 rows through LDS (private to the wave), whole rows of the run out ----
    const float* const token_scales = reinterpret_cast<const float*>(lds + kScales);
    const int* const sums = reinterpret_cast<const int*>(token_scales + kPanelRows);
    constexpr int kDouble = Q4 ? 2 : 1;
    float4 channel_scale[CB];
    float token_scale[TB];
    int bias[TB];
#pragma unroll
    for (int j = 0; j < CB; ++j) channel_scale[j] = *reinterpret_cast<const float4*>(lds + kScales + kPanelRows * 8 + (16 * j + 4 * quarter) * 4);
#pragma unroll
    for (int i = 0; i < TB; ++i) {
        const int row = (i * kPanelWaves + wave) * 16 + column;
        token_scale[i] = token_scales[row], bias[i] = Q4 ? kQuadBias * sums[row] : 0;
    }
    if (p.out_f32) {
#pragma unroll
        for (int i = 0; i < TB; ++i) {
            const int row = (i * kPanelWaves + wave) * 16 + column;
            if (row >= rows) continue;
            float* const to = reinterpret_cast<float*>(p.out) + (int64_t)(first_row + row) * p.stride + first_channel;
#pragma unroll
            for (int j = 0; j < CB; ++j) {
                const float scale[4] = {channel_scale[j].x, channel_scale[j].y, channel_scale[j].z, channel_scale[j].w};
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int channel = 16 * j + 4 * quarter + r;
                    if (channel < channels) to[channel] = rescale(kDouble * acc[i][j][r] - bias[i], scale[r], token_scale[i]);
                }
            }
        }
        return;
    }
    constexpr int kPitch = CB * 32 + 16, kPieces = 2 * CB;
    uint8_t* const image = lds + wave * (2 * 16 * kPitch);
    static_assert(kPanelWaves * 2 * 16 * kPitch <= (int)(Q4 ? kWeights : kScales), "the images lie where the tables (the weights) were");
    __half* const out = reinterpret_cast<__half*>(p.out) + (int64_t)first_row * p.stride + first_channel;
    const bool aligned = p.stride % 8 == 0 && (reinterpret_cast<uintptr_t>(p.out) & 15) == 0;
    auto store_block = [&](int i) {
        const uint8_t* const from = image + (i & 1) * (16 * kPitch);
#pragma unroll
        for (int t = 0; t < (16 * kPieces + 63) / 64; ++t) {
            const int number = t * 64 + lane, local = number / kPieces, piece = number % kPieces;
            const int row = (i * kPanelWaves + wave) * 16 + local;
            if (local >= 16 || row >= rows || piece * 8 >= channels) continue;
            const uint4 value = *reinterpret_cast<const uint4*>(from + local * kPitch + piece * 16);
            __half* const to = out + (int64_t)row * p.stride + piece * 8;
            if (aligned && piece * 8 + 8 <= channels) {
                *reinterpret_cast<uint4*>(to) = value;
            } else {
                const uint32_t words[4] = {value.x, value.y, value.z, value.w};
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (piece * 8 + e < channels) to[e] = __ushort_as_half((unsigned short)(words[e >> 1] >> (16 * (e & 1))));
            }
        }
    };
#pragma unroll
    for (int i = 0; i < TB; ++i) {
        uint8_t* const to = image + (i & 1) * (16 * kPitch) + column * kPitch + quarter * 8;
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            const v4i a = acc[i][j];
            *reinterpret_cast<uint2*>(to + j * 32) =
                make_uint2(pack_halves(rescale(kDouble * a[0] - bias[i], channel_scale[j].x, token_scale[i]), rescale(kDouble * a[1] - bias[i], channel_scale[j].y, token_scale[i])),
                           pack_halves(rescale(kDouble * a[2] - bias[i], channel_scale[j].z, token_scale[i]), rescale(kDouble * a[3] - bias[i], channel_scale[j].w, token_scale[i])));
        }
        if (i > 0) store_block(i - 1);
    }
    store_block(TB - 1);
}

// ---- host side ----
struct PanelForm {
    const void* kernel;
    uint32_t shared;
};
// by codec, blocks of 16 rows to a wave (2 to 4), whether every wave has as many, and blocks of channels to a workgroup (1 to 5)
constexpr int kPanelForms = 60;
const PanelForm& panel_form(int index) {
#define ORX_PANEL(K, T, E, C) {reinterpret_cast<const void*>(&panel_kernel<K, T, C, E>), kPanelLds<K, C>}
#define ORX_PANELS(K, T, E) ORX_PANEL(K, T, E, 1), ORX_PANEL(K, T, E, 2), ORX_PANEL(K, T, E, 3), ORX_PANEL(K, T, E, 4), ORX_PANEL(K, T, E, 5)
#define ORX_CODEC(K) ORX_PANELS(K, 2, false), ORX_PANELS(K, 2, true), ORX_PANELS(K, 3, false), ORX_PANELS(K, 3, true), ORX_PANELS(K, 4, false), ORX_PANELS(K, 4, true)
    static const PanelForm forms[kPanelForms] = {ORX_CODEC(kPanelQ4), ORX_CODEC(kPanelW8)};
#undef ORX_CODEC
#undef ORX_PANELS
#undef ORX_PANEL
    return forms[index];
}

struct PanelShape {
    const PanelForm* form;
    int row_tiles, tile_rows, units;
};
PanelShape panel_shape(int codec, int rows, int n) {
    PanelShape s = {};
    s.row_tiles = (rows + kPanelRows - 1) / kPanelRows;
    s.tile_rows = ((rows + s.row_tiles - 1) / s.row_tiles + 15) / 16 * 16;
    s.units = (int)gemm_tall_units(n);
    const int blocks = (n + 15) / 16, tb = std::max(2, (s.tile_rows / 16 + kPanelWaves - 1) / kPanelWaves);
    const int last_rows = rows - (s.row_tiles - 1) * s.tile_rows;  // of the last tile
    const bool even = s.tile_rows == tb * kPanelWaves * 16 && last_rows > s.tile_rows - 16;
    s.form = &panel_form(((codec * 3 + tb - 2) * 2 + even) * 5 + (blocks + s.units - 1) / s.units - 1);
    return s;
}

}  // namespace

// (offsets of a code request are 32 bits: a run's channels times the bytes of a row)
bool panel_eligible(int rows, int n, int k) { return rows >= 1 && rows <= kPanelMaxRows && k % 128 == 0 && k >= 256 && (int64_t)n * k < (1ll << 31); }

void panel_geometry(int codec, int rows, int n, Geometry* g) {
    const PanelShape s = panel_shape(codec, rows, n);
    g->grid[0] = (uint32_t)s.units, g->grid[1] = (uint32_t)s.row_tiles, g->grid[2] = 1;
    g->block[0] = kPanelThreads;
    g->shared = s.form->shared;
}

int panel_launch(int codec, const uint8_t* panels, const int* sums, const void* w, const uint32_t* book, const __half* ws, const __half* as, void* out,
                 int rows, int n, int k, int stride, int packed_k, bool out_f32, hipStream_t stream) {
    static DeviceOnce opted_in;  // dynamic LDS above 64 KiB needs an opt-in per kernel and device
    const int ready = opted_in.run([] {
        for (int of = 0; of < kPanelForms; ++of) {
            const PanelForm& form = panel_form(of);
            const int code = hip_check(hipFuncSetAttribute(form.kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)form.shared),
                                       "hipFuncSetAttribute");
            if (code != ORX_OK) return code;
        }
        return (int)ORX_OK;
    });
    if (ready != ORX_OK) return ready;
    const PanelShape s = panel_shape(codec, rows, n);
    PanelParams p = {};
    p.panels = panels, p.sums = sums, p.w = static_cast<const uint8_t*>(w), p.book = book, p.ws = ws, p.as = as, p.out = out;
    p.n = n, p.k = k, p.stride = stride, p.m = rows, p.out_f32 = out_f32, p.tile_rows = s.tile_rows;
    if (codec == kPanelW8)
        p.row_stride = (uint32_t)k, p.chunk_stride = 128;
    else if (packed_k == 128)
        p.row_stride = 64, p.chunk_stride = (uint32_t)n * 64, p.half_stride = 32;
    else if (packed_k == 64)
        p.row_stride = 32, p.chunk_stride = (uint32_t)n * 64, p.half_stride = (uint32_t)n * 32;
    else
        p.row_stride = (uint32_t)k / 2, p.chunk_stride = 64, p.half_stride = 32;
    typedef void (*Panel)(PanelParams);
    const Panel kernel = reinterpret_cast<Panel>(const_cast<void*>(s.form->kernel));
    ORX_LAUNCH(kernel, dim3(s.units, s.row_tiles), dim3(kPanelThreads), s.form->shared, stream, p);
    return hip_check(hipGetLastError(), "launch projection (panels)");
}

}  // namespace orx
