// Projections of two-stage (Q4) codes and int8 weights for a few to a few hundred token rows: channel runs, K split over waves.
//
// Reference counterparts: the small-row Tensor Core schedules of kernels/cuda/model/integer_core.py behind
// kernels/cuda/model/e8p_q4.py:143-264 and int8_projection.py.  Arithmetic: exact int32 over the full K, (float(acc) * ws) * as.
//
//  * A workgroup owns a run of output channels (up to CB blocks of 16) and a tile of token rows (up to TB blocks of 16) over the
//    whole K, so every weight is decoded once per row tile and nothing is summed across workgroups.
//  * Its waves split K and never meet before their slices are added: each brings the operand rows of its own slice into a
//    ring of D chunks of 128 in LDS by direct loads (one cache line per row, eight rows per request), reads fragments of
//    v_mfma_i32_16x16x64_i8 back, and asks for the chunk after next when it has read one.  Read straight into operand
//    layout, 16 bytes per lane from 16 rows, the same bytes cost the CU one L1 access per lane: 16 bytes per cycle, which
//    bounded a first form of this kernel (int8, 5120 x 17408: 31 us at 24 rows, 8.5 us more per 16 rows).
//  * Codes go from memory into registers, 16 bytes per lane, block of channels and chunk, and through four tables in shared entries
//    (QuadLookup) into the weight operands: no bank conflicts, and the sum of two XORs is half of weight + 75 as it stands.  The rows' sums of
//    codes, which correct for the 75, come out of the token fragments.  The lookups of a block for the next step of 64 run
//    under the multiplies of that block, and are combined under those of the block after it.
//  * Multiplies of codes are asm statements that add in place: as builtins the compiler had copied sums between registers for a tenth
//    of the loop.
//  What bounds it: a wave issues an instruction every 4.5 cycles and an LDS read every 8, multiplies of 16 cycles run beside them, and with
//  one wave to a SIMD (five row blocks and more, whose rings and sums leave no room for two) the loop takes what its
//  instructions take: 7168 x 5120 codes of 200 rows, 322 -> 203 a step of 64 and 28 multiplies, 2050 -> 1400 cycles, the launch 28.9 -> 22.7 us.
//  With eight waves it is the LDS (17408 x 5120 of 48 rows 20.4 -> 18.0 us) and below 17 rows the stream (8 rows, by name, 17.3 -> 14.1 us in
//  cache and 14.6 out of memory, where `auto` keeps the loader-wave kernel at 14.5).
//  int8, 24 rows of 5120 x 17408: the stream, 4.6 TB/s.
//  * Quarter q of a wave multiplies bytes [32 q, +32) of a chunk, 16 in each of two steps: piece c = 2 q + s of row r sits at
//    position (q + 4 s) ^ swizzle(r).
#include <hip/hip_fp16.h>

#include <algorithm>
#include <type_traits>

#include "e8p_device.h"
#include "lds_asm.h"
#include "orx_internal.h"

namespace orx {
namespace {

using namespace lds_asm;

// a step is one stretch of code: a lambda left as a call would keep the fragments in scratch memory
#define ORX_INLINE __attribute__((always_inline))

enum RunsCodec { kRunsQ4 = 0, kRunsW8 = 2 };

struct RunsParams {
    const int8_t* a;
    const uint8_t* w;
    const uint32_t* book;
    const __half* ws;
    const __half* as;
    void* out;
    int n, k, stride, m, out_f32;
    int run, tile_rows;                              // channels of a workgroup, rows of a tile
    uint32_t row_stride, chunk_stride, half_stride;  // weight bytes between channels, K chunks of 128, and (codes) halves of a chunk
};

template <int CODEC, int TB, int CB>
constexpr uint32_t runs_stage() { return 2048u * (TB + (CODEC == kRunsW8 ? CB : 0)); }
// table entries of 256 bytes where the rings of all waves fit beside them, else of 128
template <int CODEC, int TB, int WAVES, int D>
constexpr int runs_entry() { return WAVES * D * TB * 2048 + 256 * 256 <= 160 * 1024 ? 256 : 128; }
template <int CODEC, int TB, int WAVES, int D>
constexpr uint32_t runs_tables() { return CODEC == kRunsQ4 ? 256u * runs_entry<CODEC, TB, WAVES, D>() : 0; }
// The slices are added in LDS: whole accumulators of all waves side by side, or of half of them where all do not fit.
template <int TB, int CB>
constexpr uint32_t runs_scales() { return (TB * 16 + CB * 16) * 4; }
template <int TB, int CB, int WAVES>
constexpr int runs_parts() { return WAVES * TB * (CB * 1024 + 64) + runs_scales<TB, CB>() <= 160 * 1024 ? WAVES : WAVES / 2; }
template <int CODEC, int TB, int CB, int WAVES, int D>
constexpr uint32_t runs_lds() {
    const uint32_t rings = runs_tables<CODEC, TB, WAVES, D>() + runs_stage<CODEC, TB, CB>() * WAVES * D;
    const uint32_t sums = runs_parts<TB, CB, WAVES>() * TB * CB * 1024 + WAVES * TB * 64 + runs_scales<TB, CB>();
    return rings > sums ? rings : sums;
}

// fragments FIRST .. FIRST + COUNT - 1 of 16 rows each
template <int COUNT, int FIRST>
__device__ __forceinline__ void read_fragments(v4i* to, uint32_t address) {
    lds_read_16<FIRST * 2048>(to[0], address);
    if constexpr (COUNT > 1) read_fragments<COUNT - 1, FIRST + 1>(to + 1, address);
}

template <int CODEC, int TB, int CB, int WAVES, int D>
__global__ __launch_bounds__(WAVES * 64) void runs_kernel(RunsParams p) {
    constexpr uint32_t kStage = runs_stage<CODEC, TB, CB>();
    constexpr int kEntry = runs_entry<CODEC, TB, WAVES, D>();
    constexpr int kRequests = 2 * TB + (CODEC == kRunsQ4 ? CB : 2 * CB);  // per chunk
    static_assert(D >= 2 && (D - 1) * kRequests < 64, "requests in flight are counted in six bits");
    static_assert(runs_lds<CODEC, TB, CB, WAVES, D>() <= 160 * 1024, "the rings of all waves fit LDS");
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int column = lane & 15, quarter = lane >> 4;
    const int first_channel = (int)blockIdx.x * p.run, channels = min(p.run, p.n - first_channel);
    const int first_row = (int)blockIdx.y * p.tile_rows, rows = min(p.tile_rows, p.m - first_row);
    if (channels <= 0 || rows <= 0) return;  // the whole workgroup
    const int chunks = p.k / 128;
    const int begin = chunks * wave / WAVES, count = chunks * (wave + 1) / WAVES - begin, last = max(begin + count - 1, begin);

    // token scales of the tile (threads 0-127) and scales of the run's channels: read here, used behind the K loop
    uint32_t scale_bits = 0, selector = 0;
    {
        const uint32_t at = 2 * (uint32_t)(tid < 128 ? min(tid, rows - 1) : min(tid - 128, channels - 1));
        const __half* const from = tid < 128 ? p.as + first_row : p.ws + first_channel;
        asm volatile("global_load_ushort %0, %1, off" : "=v"(scale_bits) : "v"(reinterpret_cast<uint64_t>(from) + at) : "memory");
    }
    if constexpr (CODEC == kRunsQ4)
        asm volatile("global_load_dword %0, %1, %2" : "=v"(selector) : "v"((uint32_t)(tid & 255) * 4), "s"(uniform_pointer(p.book)) : "memory");

    uint8_t* const ring = lds + runs_tables<CODEC, TB, WAVES, D>() + (uint32_t)wave * (D * kStage);
    const int8_t* const a_base = uniform_pointer(p.a + (int64_t)first_row * p.k);
    const uint8_t* const w_base = uniform_pointer(p.w + (int64_t)first_channel * p.row_stride);
    v4i acc[TB][CB];
#pragma unroll
    for (int i = 0; i < TB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) acc[i][j] = v4i{0, 0, 0, 0};
    const uint32_t frag = lds_address_of(ring) + (uint32_t)column * 128 + (uint32_t)((quarter ^ swizzle(column)) * 16);
    std::integral_constant<int, 0> zero;
    std::integral_constant<int, 1> one;
    int row_sum[TB] = {};  // codes: the sums of the wave's slice of every row

    if constexpr (CODEC == kRunsQ4) {
        // ---- requests: eight rows of 128 bytes each; behind the last row they repeat it, so that every chunk counts the same.  Four
        // requests share an LDS base: the offset of the others is the instruction's, taken off the lane offset (and 4096 off
        // the base, so that none is negative) ----
        uint32_t row_offset[2 * TB], code_offset[CB];
#pragma unroll
        for (int i = 0; i < 2 * TB; ++i) {
            const int row = min(8 * i + (lane >> 3), rows - 1), position = (lane & 7) ^ swizzle(8 * i + (lane >> 3));
            row_offset[i] = (uint32_t)row * (uint32_t)p.k + (uint32_t)(((position & 3) << 1) | (position >> 2)) * 16 + 4096u - (uint32_t)(i & 3) * 1024u;
        }
#pragma unroll
        for (int j = 0; j < CB; ++j)
            code_offset[j] = (uint32_t)min(16 * j + column, channels - 1) * p.row_stride + (uint32_t)(quarter >> 1) * p.half_stride + (uint32_t)(quarter & 1) * 16;
        v4u codes[D][CB];
        const uint32_t ring_address = lds_address_of(ring);
        auto request_one = [&](const uint8_t* rows_from, const uint8_t* weights, auto index_tag, auto slot_tag) ORX_INLINE {
            constexpr int INDEX = decltype(index_tag)::value, SLOT = decltype(slot_tag)::value, ROW = INDEX - CB;
            if constexpr (INDEX < CB)
                load_16(codes[SLOT][INDEX], code_offset[INDEX], weights);
            else if constexpr ((ROW & 3) == 0)
                request_16<0>(row_offset[ROW], rows_from, ring_address + SLOT * kStage + ROW * 1024);
            else
                request_16_behind<(ROW & 3) * 1024>(row_offset[ROW], rows_from);
        };
        auto rows_of_chunk = [&](int index) ORX_INLINE { return reinterpret_cast<const uint8_t*>(a_base) + (int64_t)min(begin + index, last) * 128 - 4096; };
        auto codes_of_chunk = [&](int index) ORX_INLINE { return w_base + (uint64_t)min(begin + index, last) * p.chunk_stride; };
        auto request = [&](int index, auto slot_tag) ORX_INLINE {  // chunk begin + index of this wave's slice
            const uint8_t *const rows_from = rows_of_chunk(index), *const weights = codes_of_chunk(index);
            Each<kRequests>::run([&](auto index_tag) ORX_INLINE { request_one(rows_from, weights, index_tag, slot_tag); });
        };
        // waits until at most YOUNGER requests are still on their way
        auto wait_requests = [&](auto younger_tag) ORX_INLINE {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(younger_tag)::value) : "memory");
#pragma unroll
            for (int d = 0; d < D; ++d)
#pragma unroll
                for (int j = 0; j < CB; ++j) keep(codes[d][j]);
        };
        // One chunk in front of the tables, whose selector words are on their way, the others behind: a wave that issues requests waits
        // for its turn in the CU's memory pipe.  (Of eight waves four make the tables; their words would come back behind the
        // requests of the others, so these four wait for them first.)
        uint2 coarse_mask = byte_mask_biased((uint32_t)tid & 255, 2), fine_mask = byte_mask_biased((uint32_t)tid & 255, 0);
        keep(coarse_mask.x), keep(coarse_mask.y), keep(fine_mask.x), keep(fine_mask.y);  // in front of the wait
        const bool makes_tables = wave < 4;
        if (WAVES == 4 || !makes_tables) request(0, zero);
        if (makes_tables) {
            asm volatile("s_waitcnt vmcnt(%2)" : "+v"(selector), "+v"(scale_bits) : "n"(WAVES == 4 ? kRequests : 0));
            const uint2 basis = byte_basis_biased(selector, 0);
            write_quad_entry<kEntry>(tid, make_uint2(basis.x << 2, basis.y << 2), coarse_mask, basis, fine_mask);
            if (WAVES != 4) request(0, zero);
        }
        request(1, one);
        if constexpr (D > 2) request(2, std::integral_constant<int, 2>{});
        if constexpr (D > 3) request(3, std::integral_constant<int, 3>{});
        // (the waves that make no tables have not waited for their selector word, whose register is free from here on)
        asm volatile("s_waitcnt vmcnt(%2) lgkmcnt(0)\n\ts_barrier" : "+v"(selector), "+v"(scale_bits) : "n"(std::min(D * kRequests, 63)) : "memory");

        const QuadLookup<kEntry> tables(lane);
        // Sums in accumulation registers where a wave has its SIMD to itself.  The rows' sums of codes then by a multiply with ones, of four registers
        // and one instruction; else by four dot products into one register.
        constexpr bool kOwnSimd = WAVES == 4;
        v4i token[2][TB], weight[CB], sums_of_rows[kOwnSimd ? TB : 1];
        v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
        keep(ones);  // a value of its own: made again in front of a multiply it would be written too late
        auto add_row_sum = [&](auto i_tag, const v4i& fragment) ORX_INLINE {
            constexpr int I = decltype(i_tag)::value;
            if constexpr (kOwnSimd) {
                multiply_in_place<true>(sums_of_rows[I], ones, fragment);
            } else {
#pragma unroll
                for (int w = 0; w < 4; ++w) row_sum[I] = __builtin_amdgcn_sdot4(fragment[w], 0x01010101, row_sum[I], false);
            }
        };
        v2u looked[2][2][4];  // of a block and of the one before it: two codes, four rounds
        auto lookup = [&](auto set_tag, auto part_tag, uint32_t code) ORX_INLINE {  // part: code * 2 + half of its rounds
            constexpr int SET = decltype(set_tag)::value, CODE = decltype(part_tag)::value >> 1, HALF = decltype(part_tag)::value & 1;
            tables.template read<2 * HALF>(looked[SET][CODE][2 * HALF], code);
            tables.template read<2 * HALF + 1>(looked[SET][CODE][2 * HALF + 1], code);
        };
        auto combine = [&](auto set_tag, v4i& w, int word) ORX_INLINE {
            constexpr int SET = decltype(set_tag)::value;
            const int c = word >> 1, e = word & 1;
            w[word] = (int)((looked[SET][c][0][e] ^ looked[SET][c][1][e]) + (looked[SET][c][2][e] ^ looked[SET][c][3][e]));
        };
        // LDS reads return in order: at most YOUNGER are still on their way
        auto wait_lookups = [&](auto set_tag, auto younger_tag) ORX_INLINE {
            constexpr int SET = decltype(set_tag)::value;
            asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(decltype(younger_tag)::value) : "memory");
#pragma unroll
            for (int c = 0; c < 2; ++c) keep(looked[SET][c][0]), keep(looked[SET][c][1]), keep(looked[SET][c][2]), keep(looked[SET][c][3]);
        };
        auto wait_tokens = [&](auto set_tag, auto younger_tag) ORX_INLINE {
            asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(decltype(younger_tag)::value) : "memory");
#pragma unroll
            for (int i = 0; i < TB; ++i) keep(token[decltype(set_tag)::value][i]);
        };
        auto read_token = [&](auto set_tag, auto i_tag, auto slot_tag, uint32_t address) ORX_INLINE {
            constexpr int I = decltype(i_tag)::value;
            lds_read_16<decltype(slot_tag)::value * (int)kStage + I * 2048>(token[decltype(set_tag)::value][I], address);
        };
        // The multiplies of a step of 64 (HALF: which of the chunk), a block of channels at a time.  Between a block's multiplies: the lookups of its
        // next weights go out, the lookups of the block before it (a whole block old) are combined, and all blocks but the last ask for
        // their share of the next fragments.  A wave has its SIMD to itself, or shares it with one other, and issues an
        // instruction in four cycles: what is between two multiplies of 16 cycles is what they cost, so it is dealt out evenly.  In the second step of a
        // chunk the requests of the chunk D ahead go out as well, into the slot whose last fragments have been waited for.
        const uint32_t frag_half = frag ^ 64u;
        auto step = [&](auto half_tag, auto next_slot_tag, const v4u(&next_codes)[CB], auto slot_tag, const uint8_t* rows_from, const uint8_t* weights) ORX_INLINE {
            constexpr int HALF = decltype(half_tag)::value, NEXT = 1 - HALF;  // next step: its half of a chunk
            constexpr int kSpots = CB * TB;
            const uint32_t next_fragments = NEXT ? frag_half : frag;
            wait_tokens(half_tag, std::integral_constant<int, CB == 1 ? 0 : 8>{});
            Each<CB>::run([&](auto j_tag) ORX_INLINE {
                constexpr int j = decltype(j_tag)::value, before = (j + CB - 1) % CB;
                constexpr int kSet = CB == 1 ? 0 : (HALF * CB + j) & 1, kHeld = CB == 1 ? 0 : 1 - kSet;
                constexpr int kTokensHere = CB == 1 ? TB : j < CB - 1 ? (TB - j + CB - 2) / (CB > 1 ? CB - 1 : 1) : 0;  // i with i % (CB - 1) == j
                std::integral_constant<int, kSet> set;
                std::integral_constant<int, kHeld> held;
                Each<TB>::run([&](auto i_tag) ORX_INLINE {
                    constexpr int i = decltype(i_tag)::value;
                    multiply_in_place<kOwnSimd>(acc[i][j], weight[j], token[HALF][i]);
                    if constexpr (j == CB - 1) add_row_sum(i_tag, token[HALF][i]);
                    __builtin_amdgcn_sched_barrier(0);
                    // token reads of this block in front of its lookups
                    if constexpr (i == 0)
                        Each<TB>::run([&](auto n_tag) ORX_INLINE {
                            constexpr int n = decltype(n_tag)::value;
                            if constexpr (CB == 1 || (j < CB - 1 && n % (CB > 1 ? CB - 1 : 1) == j)) read_token(std::integral_constant<int, NEXT>{}, n_tag, next_slot_tag, next_fragments);
                        });
                    constexpr int kSpread = TB > 4 ? 4 : TB;  // multiplies over which the four pairs of lookups are spread
                    Each<4>::run([&](auto part_tag) ORX_INLINE {
                        constexpr int PART = decltype(part_tag)::value;
                        if constexpr (PART * kSpread / 4 == i) lookup(set, part_tag, next_codes[j][2 * NEXT + (PART >> 1)]);
                    });
                    if constexpr (HALF == 1)
                        Each<kRequests>::run([&](auto index_tag) ORX_INLINE {
                            constexpr int INDEX = decltype(index_tag)::value;
                            if constexpr (INDEX * kSpots / kRequests == j * TB + i) request_one(rows_from, weights, index_tag, slot_tag);
                        });
                    if constexpr (CB > 1) {
                        constexpr int kFirst = TB > 4 ? 4 : TB - 1, kOver = TB - kFirst;
                        if constexpr (i == kFirst) wait_lookups(held, std::integral_constant<int, std::min(8 + kTokensHere, 15)>{});
                        Each<4>::run([&](auto word_tag) ORX_INLINE {
                            constexpr int WORD = decltype(word_tag)::value;
                            if constexpr (i >= kFirst && WORD * kOver / 4 == i - kFirst) combine(held, weight[before], WORD);
                        });
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
                if constexpr (CB == 1) {
                    wait_lookups(set, zero);
#pragma unroll
                    for (int word = 0; word < 4; ++word) combine(set, weight[0], word);
                }
                if constexpr (CB <= 2) asm volatile("s_nop 1");  // the weights just combined are the next ones to be multiplied
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        if constexpr (kOwnSimd) {
#pragma unroll
            for (int i = 0; i < TB; ++i) sums_of_rows[i] = v4i{0, 0, 0, 0};
        }
        if (count > 0) {
            wait_requests(std::integral_constant<int, (D - 1) * kRequests>{});
            Each<TB>::run([&](auto i_tag) ORX_INLINE { read_token(zero, i_tag, zero, frag); });
            Each<CB>::run([&](auto j_tag) ORX_INLINE {  // (the last block's lookups are combined under the first multiplies)
                constexpr int j = decltype(j_tag)::value;
                std::integral_constant<int, CB == 1 ? 0 : (CB + j) & 1> set;
                Each<4>::run([&](auto part_tag) ORX_INLINE { lookup(set, part_tag, codes[0][j][decltype(part_tag)::value >> 1]); });
                if constexpr (j < CB - 1 || CB == 1) {
                    wait_lookups(set, zero);
#pragma unroll
                    for (int word = 0; word < 4; ++word) combine(set, weight[j], word);
                }
            });
#pragma unroll
            for (int i = 0; i < TB; ++i) {  // zeroed above the pause
                if constexpr (kOwnSimd) keep_sum<true>(sums_of_rows[i]);
#pragma unroll
                for (int j = 0; j < CB; ++j) keep_sum<kOwnSimd>(acc[i][j]);
            }
            asm volatile("s_nop 7");
            auto chunk_step = [&](int t, auto slot_tag, bool tail) ORX_INLINE {
                constexpr int SLOT = decltype(slot_tag)::value, NEXT = (SLOT + 1) % D;
                std::integral_constant<int, NEXT> next;
                asm volatile("s_nop 3");
                step(zero, slot_tag, codes[SLOT], slot_tag, nullptr, nullptr);
                wait_requests(std::integral_constant<int, (D - 2) * kRequests>{});  // chunk t + 1 is here
                step(one, next, codes[NEXT], slot_tag, rows_of_chunk(t + D), codes_of_chunk(t + D));
                // Where stretches of this code meet, the compiler may move sums to other registers, and knows nothing of multiplies on their way:
                // they have ended here, and what it writes is old enough for the next one (s_nop above).
                if (SLOT == D - 1 || tail) asm volatile("s_nop 15");
            };
            int t = 0;
            for (; t + D <= count; t += D) {
                chunk_step(t, zero, false);
                chunk_step(t + 1, one, false);
                if constexpr (D > 2) chunk_step(t + 2, std::integral_constant<int, 2>{}, false);
                if constexpr (D > 3) chunk_step(t + 3, std::integral_constant<int, 3>{}, false);
            }
            if (t < count) chunk_step(t, zero, true);
            if constexpr (D > 2)
                if (t + 1 < count) chunk_step(t + 1, one, true);
            if constexpr (D > 3)
                if (t + 2 < count) chunk_step(t + 2, std::integral_constant<int, 2>{}, true);
        }
        // the requests behind the slice (repeats of its last chunk) and the reads ahead have landed before their registers and slots are
        // reused, and the last multiplies have written their sums
        wait_requests(zero);
        wait_tokens(zero, zero), wait_tokens(one, zero), wait_lookups(zero, zero), wait_lookups(one, zero);
        asm volatile("s_nop 15");
#pragma unroll
        for (int i = 0; i < TB; ++i) {
            if constexpr (kOwnSimd) {
                keep_sum<true>(sums_of_rows[i]);
                row_sum[i] = sums_of_rows[i][0];
            } else {
                row_sum[i] += __shfl_xor(row_sum[i], 16, 64);
                row_sum[i] += __shfl_xor(row_sum[i], 32, 64);
            }
#pragma unroll
            for (int j = 0; j < CB; ++j) keep_sum<kOwnSimd>(acc[i][j]);
        }
    } else {
        // ---- requests: eight rows of 128 bytes each.  Requests behind the one that holds the last row repeat that one, so that every
        // chunk counts the same.  int8: where the last request of a tile or a run would be such a repeat it is left out of every
        // chunk (what its rows hold in LDS reaches no stored sum): 5120 x 17408 of 24 rows, 20 channels to a CU, has six requests
        // a chunk instead of eight, 24.7 -> 24.1 us with the quantiser, of one row 18.7 -> 17.9 without it.  (Codes: the branch
        // costs the step between the chunks more than a request: 17408 x 5120 of 48 rows 21.7 -> 25.3.) ----
        struct Rows {
            uint32_t even, odd, last;  // lane offsets in an even and an odd request, and in the last one
            int last_request;
        };
        auto rows_of = [&](int count_here) {
            const int row = lane >> 3, position = (lane & 7) ^ (lane >> 4);
            auto piece = [](int at) { return (uint32_t)(((at & 3) << 1) | (at >> 2)) * 16; };
            Rows r;
            r.last_request = (count_here - 1) >> 3;
            r.even = (uint32_t)row * (uint32_t)p.k + piece(position), r.odd = (uint32_t)row * (uint32_t)p.k + piece(position ^ 4);
            r.last = (uint32_t)min(row, count_here - 1 - 8 * r.last_request) * (uint32_t)p.k + piece(r.last_request & 1 ? position ^ 4 : position);
            return r;
        };
        const Rows token_rows = rows_of(rows), weight_rows = rows_of(channels);
        const int left_out = (token_rows.last_request < 2 * TB - 1) + (weight_rows.last_request < 2 * CB - 1);
        auto request_rows = [&](const void* base, const Rows& r, auto blocks_tag, uint8_t* to) ORX_INLINE {
            constexpr int BLOCKS = decltype(blocks_tag)::value;
    #pragma unroll
            for (int i = 0; i < 2 * BLOCKS; ++i) {
                if (i == 2 * BLOCKS - 1 && r.last_request < i) break;  // uniform
                const bool tail = i >= r.last_request;  // uniform
                uint32_t offset = tail ? r.last : i & 1 ? r.odd : r.even;
                asm volatile("" : "+v"(offset));  // 32 bits beside a uniform base
                const uint64_t first = (uint64_t)(uint32_t)(8 * min(i, r.last_request)) * (uint32_t)p.k;
                direct_load_16(static_cast<const uint8_t*>(base) + first + (uint64_t)offset, to + i * 1024);
            }
        };
        auto request = [&](int index, auto slot_tag) ORX_INLINE {  // chunk begin + index of this wave's slice
            constexpr int SLOT = decltype(slot_tag)::value;
            const int chunk = min(begin + index, last);
            request_rows(w_base + (uint64_t)chunk * p.chunk_stride, weight_rows, std::integral_constant<int, CB>{}, ring + SLOT * kStage + TB * 2048);
            request_rows(a_base + (uint64_t)chunk * 128, token_rows, std::integral_constant<int, TB>{}, ring + SLOT * kStage);
        };
        // waits until at most `CHUNKS` of the youngest chunks requested are still on their way
        auto wait_requests = [&](auto chunks_tag) ORX_INLINE {
            constexpr int CHUNKS = decltype(chunks_tag)::value;
            if (CHUNKS == 0 || left_out == 0)
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(CHUNKS * kRequests) : "memory");
            else if (left_out == 1)
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(CHUNKS * (kRequests - 1)) : "memory");
            else
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(CHUNKS * (kRequests - 2)) : "memory");
        };
        request(0, zero);
        request(1, one);
        if constexpr (D > 2) request(2, std::integral_constant<int, 2>{});
        if constexpr (D > 3) request(3, std::integral_constant<int, 3>{});
        v4i token[2][TB], weight[2][CB];
        auto chunk_step = [&](int t, auto slot_tag) {
            constexpr int SLOT = decltype(slot_tag)::value;
            wait_requests(std::integral_constant<int, D - 1>{});
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const uint32_t address = (frag + SLOT * kStage) ^ (64u * s);
                read_fragments<TB, 0>(token[s], address);
                read_fragments<CB, TB>(weight[s], address);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int s = 0; s < 2; ++s) {
#pragma unroll
                for (int i = 0; i < TB; ++i) asm volatile("" : "+v"(token[s][i]));
#pragma unroll
                for (int j = 0; j < CB; ++j) asm volatile("" : "+v"(weight[s][j]));
            }
            request(t + D, slot_tag);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int i = 0; i < TB; ++i)
#pragma unroll
                    for (int j = 0; j < CB; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(weight[s][j], token[s][i], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        int t = 0;
        for (; t + D <= count; t += D) {
            chunk_step(t, std::integral_constant<int, 0>{});
            chunk_step(t + 1, std::integral_constant<int, 1>{});
            if constexpr (D > 2) chunk_step(t + 2, std::integral_constant<int, 2>{});
            if constexpr (D > 3) chunk_step(t + 3, std::integral_constant<int, 3>{});
        }
        if (t < count) chunk_step(t, std::integral_constant<int, 0>{});
        if constexpr (D > 2)
            if (t + 1 < count) chunk_step(t + 1, std::integral_constant<int, 1>{});
        if constexpr (D > 3)
            if (t + 2 < count) chunk_step(t + 2, std::integral_constant<int, 2>{});
        // the requests behind the slice (repeats of its last chunk) have landed before their slots are reused
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" : "+v"(scale_bits)::"memory");
    }
    asm volatile("s_barrier" ::: "memory");

    // ---- the slices are added where the rings and tables were.  Accumulator register r of a lane: channel 4 quarter + r of the block,
    // token `column`.  A wave leaves its blocks whole, 16 bytes to a lane, and adds whole blocks of all waves ----
    constexpr int kBlocks = TB * CB, kParts = runs_parts<TB, CB, WAVES>();
    v4i* const sums = reinterpret_cast<v4i*>(lds);
    int* const row_sums = reinterpret_cast<int*>(lds + kParts * kBlocks * 1024);  // of every wave
    float* const token_scales = reinterpret_cast<float*>(row_sums + WAVES * TB * 16);
    float* const channel_scales = token_scales + TB * 16;
    asm volatile("" : "+v"(scale_bits));  // converted here, not where it was read
    const float scale = __half2float(__ushort_as_half((unsigned short)scale_bits));
    if (tid < TB * 16) token_scales[tid] = scale;
    if (tid >= 128 && tid < 128 + CB * 16) channel_scales[tid - 128] = scale;
    int own = threadIdx.x & 63;
    asm volatile("" : "+v"(own));
    // column c of quarter q of a block lies at 16 q + (c ^ 4 q): no two of the 16 lanes that write or read together meet in a bank
    v4i* const mine = sums + (wave % kParts) * kBlocks * 64 + ((own & 48) | ((own & 15) ^ (own >> 4 << 2)));
    if constexpr (CODEC == kRunsQ4) {
        if (own < 16) {
#pragma unroll
            for (int i = 0; i < TB; ++i) row_sums[(wave * TB + i) * 16 + own] = row_sum[i];
        }
    }
    auto leave = [&]() ORX_INLINE {
#pragma unroll
        for (int i = 0; i < TB; ++i)
#pragma unroll
            for (int j = 0; j < CB; ++j) mine[(i * CB + j) * 64] = acc[i][j];
    };
    if constexpr (kParts < WAVES) {
        if (wave >= kParts) leave();
        __syncthreads();
        if (wave < kParts) {
#pragma unroll
            for (int i = 0; i < TB; ++i)
#pragma unroll
                for (int j = 0; j < CB; ++j) acc[i][j] += mine[(i * CB + j) * 64];
            leave();
        }
    } else {
        leave();
    }
    __syncthreads();
    // Four lanes take a row of 32 channels of two blocks beside each other, eight channels to a lane (few blocks: of 16 channels, four to a
    // lane, so that every wave has one): 16 bytes to a lane and 64 in a row where 8 bytes of 16 rows took 115 cycles
    // an instruction (200 rows of 7168 x 5120: 3200 of the 41000 cycles of a workgroup).
    constexpr int kQuads = TB * ((CB + 1) / 2) >= WAVES ? 2 : 1, kPerRow = kQuads == 2 ? (CB + 1) / 2 : CB;
    constexpr int kUnits = TB * kPerRow, kTurns = (kUnits + WAVES - 1) / WAVES, kBatch = kTurns > 1 ? 2 : 1;
    const int row_of_block = own >> 2, share = own & 3;
    auto cell_of = [&](int block, int quarter_here) ORX_INLINE { return sums + block * 64 + quarter_here * 16 + (row_of_block ^ (quarter_here * 4)); };
#pragma unroll 1
    for (int turn = 0; turn < kTurns; turn += kBatch) {
        v4i sum[kBatch][kQuads];
        int correction[kBatch];
        float token_scale[kBatch];
        float4 ws[kBatch][kQuads];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const int unit = min(wave + (turn + u) * WAVES, kUnits - 1), i = unit / kPerRow;
            const int j = kQuads == 2 ? min(unit % kPerRow * 2 + (share >> 1), CB - 1) : unit % kPerRow, quarter_here = kQuads == 2 ? 2 * (share & 1) : share;
            const int local = i * 16 + row_of_block;
#pragma unroll
            for (int h = 0; h < kQuads; ++h) {
                const v4i* const cell = cell_of(i * CB + j, quarter_here + h);
                sum[u][h] = *cell;
#pragma unroll
                for (int w = 1; w < kParts; ++w) sum[u][h] += cell[w * kBlocks * 64];
                ws[u][h] = *reinterpret_cast<const float4*>(channel_scales + j * 16 + 4 * (quarter_here + h));
            }
            correction[u] = 0;
            if constexpr (CODEC == kRunsQ4) {
#pragma unroll
                for (int w = 0; w < WAVES; ++w) correction[u] += row_sums[w * TB * 16 + local];
                correction[u] *= kQuadBias;
            }
            token_scale[u] = token_scales[local];
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            constexpr int kEach = 4 * kQuads;  // channels of a lane
            const int unit = wave + (turn + u) * WAVES, local = unit / kPerRow * 16 + row_of_block, channel = unit % kPerRow * (4 * kEach) + share * kEach;
            if (unit >= kUnits || local >= rows || channel >= channels) continue;
            constexpr int kTimes = CODEC == kRunsQ4 ? 2 : 1;
            float value[kEach];
#pragma unroll
            for (int h = 0; h < kQuads; ++h) {
                const float scale_of[4] = {ws[u][h].x, ws[u][h].y, ws[u][h].z, ws[u][h].w};
#pragma unroll
                for (int r = 0; r < 4; ++r) value[4 * h + r] = rescale(kTimes * sum[u][h][r] - correction[u], scale_of[r], token_scale[u]);
            }
            const int64_t at = (int64_t)(first_row + local) * p.stride + first_channel + channel;
            const bool whole = channel + kEach <= channels;
            if (p.out_f32) {
                float* const dst = static_cast<float*>(p.out) + at;
                if (whole) {
                    __builtin_memcpy(dst, value, sizeof value);
                } else {
#pragma unroll
                    for (int r = 0; r < kEach; ++r)
                        if (channel + r < channels) dst[r] = value[r];
                }
            } else {
                __half* const dst = static_cast<__half*>(p.out) + at;
                __half h[kEach];
                uint32_t words[2 * kQuads];
#pragma unroll
                for (int r = 0; r < kEach; ++r) h[r] = __float2half_rn(value[r]);
#pragma unroll
                for (int r = 0; r < 2 * kQuads; ++r) words[r] = (uint32_t)__half_as_ushort(h[2 * r]) | (uint32_t)__half_as_ushort(h[2 * r + 1]) << 16;
                if (whole) {  // (one store at any address: a run of 38 channels, 9728 of them, leaves its rows at multiples of 4)
                    __builtin_memcpy(dst, words, sizeof words);
                } else {
#pragma unroll
                    for (int r = 0; r < kEach; r += 2) {
                        if (channel + r + 2 <= channels)
                            __builtin_memcpy(dst + r, &words[r / 2], 4);
                        else if (channel + r < channels)
                            dst[r] = h[r];
                    }
                }
            }
        }
    }
}

// ---- host side ----
struct RunsForm {
    int codec, tb, cb, waves;
    const void* kernel;
};
// every form asks for the same LDS: one workgroup per CU either way, and the record of a launch then holds for all the row
// counts that share a grid and a block
constexpr uint32_t kRunsLds = 160 * 1024;
const RunsForm* runs_forms(int* count) {
#define ORX_RUNS(C, T, B, W, D) {C, T, B, W, reinterpret_cast<const void*>(&runs_kernel<C, T, B, W, D>)}
    static const RunsForm forms[] = {
        ORX_RUNS(kRunsQ4, 1, 1, 8, 4), ORX_RUNS(kRunsQ4, 1, 2, 8, 4), ORX_RUNS(kRunsQ4, 1, 3, 8, 4), ORX_RUNS(kRunsQ4, 1, 5, 8, 3),
        ORX_RUNS(kRunsQ4, 2, 1, 8, 3), ORX_RUNS(kRunsQ4, 2, 2, 8, 3), ORX_RUNS(kRunsQ4, 2, 3, 8, 3), ORX_RUNS(kRunsQ4, 2, 5, 8, 3),
        ORX_RUNS(kRunsQ4, 3, 1, 8, 2), ORX_RUNS(kRunsQ4, 3, 2, 8, 2), ORX_RUNS(kRunsQ4, 3, 3, 8, 2), ORX_RUNS(kRunsQ4, 3, 5, 8, 2),
        ORX_RUNS(kRunsQ4, 4, 1, 8, 2), ORX_RUNS(kRunsQ4, 4, 2, 8, 2), ORX_RUNS(kRunsQ4, 4, 3, 8, 2), ORX_RUNS(kRunsQ4, 4, 5, 8, 2),
        ORX_RUNS(kRunsQ4, 5, 1, 4, 3), ORX_RUNS(kRunsQ4, 5, 2, 4, 3), ORX_RUNS(kRunsQ4, 5, 3, 4, 3), ORX_RUNS(kRunsQ4, 5, 4, 4, 3),
        ORX_RUNS(kRunsQ4, 6, 1, 4, 2), ORX_RUNS(kRunsQ4, 6, 2, 4, 2), ORX_RUNS(kRunsQ4, 6, 3, 4, 2), ORX_RUNS(kRunsQ4, 6, 4, 4, 2),
        ORX_RUNS(kRunsQ4, 7, 1, 4, 2), ORX_RUNS(kRunsQ4, 7, 2, 4, 2), ORX_RUNS(kRunsQ4, 7, 3, 4, 2), ORX_RUNS(kRunsQ4, 7, 4, 4, 2),
        ORX_RUNS(kRunsQ4, 8, 1, 4, 2), ORX_RUNS(kRunsQ4, 8, 2, 4, 2), ORX_RUNS(kRunsQ4, 8, 3, 4, 2), ORX_RUNS(kRunsQ4, 8, 4, 4, 2),
        ORX_RUNS(kRunsW8, 1, 1, 8, 4), ORX_RUNS(kRunsW8, 1, 2, 8, 3), ORX_RUNS(kRunsW8, 1, 3, 8, 2), ORX_RUNS(kRunsW8, 1, 5, 4, 3),
        ORX_RUNS(kRunsW8, 2, 1, 8, 3), ORX_RUNS(kRunsW8, 2, 2, 8, 2), ORX_RUNS(kRunsW8, 2, 3, 8, 2), ORX_RUNS(kRunsW8, 2, 5, 4, 2),
        ORX_RUNS(kRunsW8, 3, 1, 8, 2), ORX_RUNS(kRunsW8, 3, 2, 8, 2), ORX_RUNS(kRunsW8, 3, 3, 4, 3), ORX_RUNS(kRunsW8, 3, 5, 4, 2),
        ORX_RUNS(kRunsW8, 4, 1, 8, 2), ORX_RUNS(kRunsW8, 4, 2, 4, 3), ORX_RUNS(kRunsW8, 4, 3, 4, 2), ORX_RUNS(kRunsW8, 4, 5, 4, 2),
        ORX_RUNS(kRunsW8, 5, 2, 4, 2), ORX_RUNS(kRunsW8, 5, 3, 4, 2), ORX_RUNS(kRunsW8, 5, 5, 4, 2),
        ORX_RUNS(kRunsW8, 6, 2, 4, 2), ORX_RUNS(kRunsW8, 6, 3, 4, 2),
        ORX_RUNS(kRunsW8, 7, 2, 4, 2), ORX_RUNS(kRunsW8, 7, 3, 4, 2),
        ORX_RUNS(kRunsW8, 8, 2, 4, 2),
    };
#undef ORX_RUNS
    *count = (int)(sizeof forms / sizeof forms[0]);
    return forms;
}

// the forms of a codec and a tile height, widest last: they follow one another in the list (every call of a handle asks several
// times, so the list is not searched each time)
struct RunsFormRange {
    const RunsForm* first;
    int count;
};
RunsFormRange runs_forms_of(int codec, int tb) {
    struct Index {
        RunsFormRange of[2][9] = {};
        Index() {
            int count = 0;
            const RunsForm* forms = runs_forms(&count);
            for (int i = 0; i < count; ++i) {
                RunsFormRange& range = of[forms[i].codec == kRunsW8][forms[i].tb];
                if (range.count++ == 0) range.first = &forms[i];
            }
        }
    };
    static const Index index;
    return index.of[codec == kRunsW8][tb];
}

constexpr int kRunsMaxRows = 512;

// How a launch is cut: rows into tiles of up to 128, channels into runs so that the workgroups fill whole rounds of the CUs.
struct RunsShape {
    const RunsForm* form;
    int row_tiles, tile_rows, runs, run;
    int grid_runs;  // a row of the grid: the runs, and workgroups without one that end at once
};
RunsShape runs_shape(int codec, int rows, int n) {
    RunsShape s = {};
    s.row_tiles = (rows + 127) / 128;
    s.tile_rows = (rows + s.row_tiles - 1) / s.row_tiles;
    const int blocks = (s.tile_rows + 15) / 16;
    const RunsFormRange forms = runs_forms_of(codec, blocks);
    const int most = forms.first[forms.count - 1].cb;
    const int cus = device_compute_units();
    const int column_blocks = (n + 15) / 16;
    // fewest rounds of the CUs whose runs fit the widest form, then the runs as even as whole rounds make them
    const int least_runs = (column_blocks + most - 1) / most;
    const int rounds = (least_runs * s.row_tiles + cus - 1) / cus;
    s.runs = std::max(least_runs, rounds * cus / s.row_tiles);
    s.run = (n + s.runs - 1) / s.runs;
    // Stores that start on 16 bytes, where that leaves no CU without work that others wait for: a wide run takes no block of 16 more (240 rows of 7000 x
    // 2560: 55 channels 16.0 us, 56 15.5), a narrow one leaves a sixth of the CUs idle (int8, 40 rows of 5120 x 17408: 20 channels 25.8, 24 26.7).
    if (rows > 32 && s.run >= 40) s.run = (s.run + 7) / 8 * 8;
    s.runs = (n + s.run - 1) / s.run;
    // Several row tiles: rows of the grid are a multiple of the 8 XCDs, so that the workgroups of a run, a row apart, read its weights through one L2, unless an XCD
    // would get a round more that way.  int8 9728 x 2560 at 129 / 160 rows (122 runs) 15.0 / 15.5 -> 13.7 / 14.2 us, 7000 x 2560 at 300 22.5 -> 20.5; codes, half the bytes,
    // 7000 x 2560 at 200 / 300 rows 15.1 / 23.1 -> 14.6 / 22.3; with a round more 19000 x 2048 at 300 rows 44.4 -> 51.7.
    const int even_runs = (s.runs + 7) / 8 * 8, rounds_here = (s.runs * s.row_tiles + cus - 1) / cus;
    s.grid_runs = s.row_tiles > 1 && even_runs * s.row_tiles <= rounds_here * cus ? even_runs : s.runs;
    for (int i = forms.count - 1; i >= 0; --i)
        if (16 * forms.first[i].cb >= s.run) s.form = &forms.first[i];
    return s;
}

}  // namespace

bool runs_eligible(int codec, int rows, int n, int k) {
    return rows >= 1 && rows <= kRunsMaxRows && k % 128 == 0 && (int64_t)n * k < (1ll << 31) && (int64_t)rows * k < (1ll << 31) &&
           runs_shape(codec, rows, n).form != nullptr;
}

// rounds of the CUs that the launch takes, the rows of its tiles and the channels of its runs
int runs_rounds(int codec, int rows, int n, int* tile_rows, int* run) {
    const RunsShape s = runs_shape(codec, rows, n);
    const int cus = device_compute_units();
    *tile_rows = s.tile_rows, *run = s.run;
    return (s.runs * s.row_tiles + cus - 1) / cus;
}

void runs_geometry(int codec, int rows, int n, Geometry* g) {
    const RunsShape s = runs_shape(codec, rows, n);
    g->grid[0] = (uint32_t)s.grid_runs, g->grid[1] = (uint32_t)s.row_tiles, g->grid[2] = 1;
    g->block[0] = (uint32_t)s.form->waves * 64;
    g->shared = kRunsLds;
}

int runs_launch(int codec, const int8_t* a, const void* w, const uint32_t* book, const __half* ws, const __half* as, void* out,
                int rows, int n, int k, int stride, int packed_k, bool out_f32, hipStream_t stream) {
    static DeviceOnce opted_in;  // dynamic LDS above 64 KiB needs an opt-in per kernel and device
    const int ready = opted_in.run([] {
        int count = 0;
        const RunsForm* forms = runs_forms(&count);
        for (int i = 0; i < count; ++i) {
            const int code = hip_check(hipFuncSetAttribute(forms[i].kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kRunsLds),
                                       "hipFuncSetAttribute");
            if (code != ORX_OK) return code;
        }
        return (int)ORX_OK;
    });
    if (ready != ORX_OK) return ready;
    const RunsShape s = runs_shape(codec, rows, n);
    RunsParams p = {};
    p.a = a, p.w = static_cast<const uint8_t*>(w), p.book = book, p.ws = ws, p.as = as, p.out = out;
    p.n = n, p.k = k, p.stride = stride, p.m = rows, p.out_f32 = out_f32, p.run = s.run, p.tile_rows = s.tile_rows;
    if (codec == kRunsW8)
        p.row_stride = (uint32_t)k, p.chunk_stride = 128, p.half_stride = 64;
    else if (packed_k == 128)
        p.row_stride = 64, p.chunk_stride = (uint32_t)n * 64, p.half_stride = 32;
    else if (packed_k == 64)
        p.row_stride = 32, p.chunk_stride = (uint32_t)n * 64, p.half_stride = (uint32_t)n * 32;
    else
        p.row_stride = (uint32_t)k / 2, p.chunk_stride = 64, p.half_stride = 32;
    typedef void (*Runs)(RunsParams);
    const Runs kernel = reinterpret_cast<Runs>(const_cast<void*>(s.form->kernel));
    ORX_LAUNCH(kernel, dim3(s.grid_runs, s.row_tiles), dim3(s.form->waves * 64), kRunsLds, stream, p);
    return hip_check(hipGetLastError(), "launch projection (channel runs)");
}

}  // namespace orx
