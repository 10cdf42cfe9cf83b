// Routed single-stage (Q2) expert projections of long prompts: 128-row tiles, codes decoded into MFMA operands.
//
// Reference counterpart: the routed decode kernels/cuda/model/e8p_decode.py:36-245 over the tile list of
// kernels/cuda/model/routing.py.  Arithmetic: exact int32 over the full K, (float(acc) * ws) * as, rounded to fp16 once.
//
// With hundreds of rows per expert the projection is a matrix product: 4096 tokens x top-8 of 128 experts are 137 GOP in
// gate_up and 69 GOP in down, which the 32-row tiles of the weight-streaming kernels ran at 460 TOP/s, decoding every code
// once per 32 rows.
//  * A unit is (tile of up to 128 slots, 256 output channels or, see below, 128), a workgroup four waves, two workgroups to a CU, so that the
//    set-up and the epilogue of one run beside the K loop of the other.
//  * A wave owns 64 channels and all rows of the tile, 8 x 4 blocks of v_mfma_i32_16x16x64_i8 (128 accumulator
//    registers).  Its codes go from memory into registers (8 bytes per lane, block of 16 channels and 128 of K) and through
//    the byte tables straight into the weight operands: no decoded weight passes through LDS, and a code is
//    decoded once per 128 rows.  Per 64 of K a wave then asks LDS for 8 fragments of 1 KiB and 16 lookups of 512 bytes while
//    it multiplies 32 times.  Tiles of at most 64 or 32 rows take 4 or 2 row blocks.
//  * Token rows come through LDS by direct loads in whole cache lines (K chunks of 128, two slots of 16 KiB); with GATHER
//    the rows are those of the slots' tokens, so no launch copies a token's row top_k times.
//  * The two tables share 32 KiB without conflicts (PairedLookup); two tables of eight copies, read one after the other, had half
//    as many conflict cycles again, and sixteen copies of each leave room for one workgroup per CU.
// Measured at 4096 tokens x top-8 of 128 experts (H = 2048, I = 512; popularity of the experts like 1 / rank^1.1):
// gate_up 296 -> 100 us, down 215 -> 67 us.  What bounds it now: the loop, where two waves of a SIMD keep its matrix pipe busy
// in 0.85 of the cycles, is 9800 of the 21000 cycles of a unit of down and 38000 of 57000 of gate_up; set-up (tile, tables, first
// chunks) takes 5200, the epilogue 4600 and, with the SwiGLU's sixteen instructions a sigmoid, 11000.
// With tile units the tiles come largest first and in one read: a unit of gate_up takes 30 us, and in the order of the experts the
// last ones started when most of the chip was done (gate_up 97-107 -> 96 us over three routings, down 71-77 -> 70; the layer at 2000
// tokens 140.7 -> 133.1 us over eight, at 4096, where two whole rounds are full, 229.6 -> 228.7).
// One persistent workgroup of eight waves per CU that requests the next unit's chunks early measured 118 and 75 us.
// A workgroup that takes 2, 4 or 8 spans of a tile in a row, the next one's chunks requested in the last steps, and 512
// persistent workgroups of this form with even shares both measured level or slower (whole layer 227 / 241 / 247 and 243 against
// 226 us): what the set-up saves, the uneven ends lose.
//  * Units of 128 channels where those of 256 leave CUs without one (grouped_bulk_narrow): a wave has two blocks of 16 channels instead of four.
//  * SWIGLU: a wave owns 32 gate and the 32 matching up channels, so gate and up of one (slot, channel) meet in one
//    lane; the epilogue writes fp16(silu(gate) * up) and, where asked, gate | up and the slots' largest magnitudes.
#include <hip/hip_fp16.h>

#include <algorithm>
#include <type_traits>

#include "a8_device.h"
#include "e8p_device.h"
#include "lds_asm.h"
#include "orx_internal.h"

namespace orx {
namespace {

using namespace lds_asm;

constexpr int kThreads = 256;
constexpr int kTileRows = 128;
// Output channels of a unit of waves with CB blocks of 16 channels (SWIGLU: half of them gate, half up).
constexpr int span_of(int cb) { return 64 * cb; }
constexpr int kSpan = span_of(4);
constexpr uint32_t kTokens = kPairedTableBytes;
constexpr uint32_t kTokenBytes = 2 * kTileRows * 128;  // two chunks of 128 rows, four of 64
constexpr uint32_t kTokenScale = kTokens + kTokenBytes;
constexpr uint32_t kChannelScale = kTokenScale + kTileRows * 4;
constexpr uint32_t kLds = kChannelScale + kSpan * 4;

struct BulkParams {
    const int8_t* a;        // (slots, K), or (tokens, K) when gathered
    const __half* as;
    const int* slot_token;  // GATHER: token of every slot
    const uint8_t* w;       // (E, K/128, N, 16) u16
    const uint32_t* book;
    const __half* ws;       // (E, N)
    __half* out;            // (slots, N); may be null with SWIGLU
    __half* act;            // SWIGLU: (slots, N/2)
    int* row_max;           // SWIGLU: raised to the fp32 bits of the slot's largest |act|; may be null
    const int* counts;
    const int* offsets;
    const int* tile_expert;
    const int* tile_row;
    const int* tile_count;
    const int4* tile_units;  // or null
    int n, k, tile_capacity, spans;
};

// until at most COUNT requests of this wave are on their way
template <int COUNT>
__device__ __forceinline__ void wait_requests() {
    static_assert(COUNT < 64, "the counter has six bits");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(COUNT) : "memory");
}

template <bool GATHER, bool SWIGLU, int CB>
__global__ __launch_bounds__(kThreads, 2) void grouped_bulk_kernel(BulkParams p) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // ---- unit: workgroups 8 apart (one XCD) take the spans of one tile, whose rows that XCD's L2 then holds ----
    const int b = (int)blockIdx.x, region = 8 * p.spans;
    const int tile = (b / region) * 8 + b % 8, span = (b / 8) % p.spans;
    if (tile >= p.tile_capacity) return;
    uint32_t selector;
    asm volatile("global_load_dword %0, %1, %2" : "=v"(selector) : "v"((uint32_t)tid * 4), "s"(uniform_pointer(p.book)) : "memory");
    // the list's length and its entry in one trip; behind the end an entry is whatever the buffer holds
    const int listed = p.tile_count[0];
    int expert, rows, row0;
    if (p.tile_units != nullptr) {
        const int4 unit = p.tile_units[tile];
        if (tile >= listed) return;
        expert = unit.x, row0 = unit.y, rows = min(kTileRows, unit.z);
    } else {
        const int listed_expert = p.tile_expert[tile], first = p.tile_row[tile];
        if (tile >= listed) return;
        expert = listed_expert, rows = min(kTileRows, p.counts[expert] - first), row0 = p.offsets[expert] + first;
    }
    expert = __builtin_amdgcn_readfirstlane(expert), rows = __builtin_amdgcn_readfirstlane(rows), row0 = __builtin_amdgcn_readfirstlane(row0);
    if (rows <= 0) return;
    const int inner = p.n / 2;
    const int chunks = p.k / 128;

    // ---- this wave's channels: plain n0 .. n0 + 63; SWIGLU gate n0 .. n0 + 31 and up inner + n0 .. ----
    const int group = span * 4 + wave;
    constexpr int kOwn = 16 * CB, kHalf = SWIGLU ? kOwn / 2 : kOwn;  // channels of a wave, and beside each other
    const int limit = SWIGLU ? inner / kHalf : p.n / kOwn;
    const bool live_wave = group < limit;  // the others help with the token rows
    const int n0 = (live_wave ? group : 0) * kHalf;
    const uint8_t* const codes_base = uniform_pointer(p.w + (int64_t)expert * p.n * (p.k / 4));
    const uint32_t chunk_stride = (uint32_t)p.n * 32;
    const uint32_t code_offset = (uint32_t)(n0 + (lane & 15)) * 32 + (uint32_t)(lane >> 4) * 8;
    const uint32_t code_offset_up = code_offset + (SWIGLU ? (uint32_t)inner * 32 : CB * 256u);
    const int8_t* const a_base = uniform_pointer(p.a);

    auto run = [&](auto blocks_tag) {
        constexpr int NB = decltype(blocks_tag)::value;  // 16-row blocks
        constexpr int LOADS = NB / 2;                    // 16 NB rows are 2 NB requests of 8 rows, over four waves
        constexpr int PHASES = NB >= 4 ? 4 : 1;          // a step of 64 in phases of RB row blocks,
        constexpr int RB = NB / PHASES;                  // each looking up LB of the next step's CB weight blocks, while there are any
        constexpr int LB = CB > PHASES ? CB / PHASES : 1;
        constexpr int DEPTH = NB == 8 ? 2 : 4;           // chunks in LDS and in code registers
        static_assert(DEPTH * NB * 16 * 128 <= kTokenBytes, "the chunks fit");
        constexpr uint32_t SLOT = NB * 16 * 128;
        constexpr int kChunkRequests = CB + LOADS;
        // ---- token rows: request b of this wave brings rows 8 (LOADS wave + b) .. +7 of a chunk, 128 bytes each.  The
        // quarter q of a wave multiplies K bytes [32 q, +32) of a chunk in two steps of 16, so piece c = 2 q + s of row r sits
        // at position (q + 4 s) ^ swizzle(r): a fragment read touches four neighbouring positions of 16 rows ----
        uint32_t slot_of[LOADS + 1];  // of this lane's row of each request, and of row `tid` for its scale; GATHER: then of their tokens
#pragma unroll
        for (int i = 0; i < LOADS; ++i) slot_of[i] = (uint32_t)(row0 + min((wave * LOADS + i) * 8 + (lane >> 3), rows - 1));
        slot_of[LOADS] = (uint32_t)(row0 + min(tid, rows - 1));
        if constexpr (GATHER) {
            const int* const tokens_of = uniform_pointer(p.slot_token);
            Each<LOADS + 1>::run([&](auto i) { load_4(slot_of[i], slot_of[i] * 4, tokens_of); });
        }
        // DEPTH register sets of codes, chunk c in set c % DEPTH: CB blocks of 16 channels, 8 bytes to a lane
        v2u codes[DEPTH][CB];
        Each<DEPTH>::run([&](auto set) { Each<CB>::run([&](auto j) { anything(codes[set][j]); }); });  // (anything, but in a register)
        // Chunks that do not exist are requested by no lane where waits behind them count requests, else not at all.
        std::true_type counted;
        std::bool_constant<(DEPTH > 2)> counted_in_loop;
        auto issue_codes = [&](int chunk, auto set_tag, auto counted_tag) {
            auto& set = codes[decltype(set_tag)::value];
            const uint8_t* const base = codes_base + (uint64_t)chunk * chunk_stride;
            if constexpr (CB == 4) load_8_of_four<decltype(counted_tag)::value>(set, code_offset, code_offset_up, base, chunk, chunks);
            else load_8_of_two<decltype(counted_tag)::value>(set, code_offset, code_offset_up, base, chunk, chunks);
        };
        std::integral_constant<int, 0> zero;
        std::integral_constant<int, 1> one;
        issue_codes(0, zero, counted);  // two chunks' are on their way while the rows' tokens are looked up
        issue_codes(1, one, counted);
        if constexpr (GATHER) {
            wait_requests<2 * CB>();
            Each<LOADS + 1>::run([&](auto i) { keep(slot_of[i]); });
        }
        uint32_t row_offset[LOADS];
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int position = (lane & 7) ^ swizzle((wave * LOADS + i) * 8 + (lane >> 3));
            const int piece = ((position & 3) << 1) | (position >> 2);
            row_offset[i] = slot_of[i] * (uint32_t)p.k + (uint32_t)piece * 16 + 4096u - (uint32_t)i * 1024u;
        }
        const uint32_t token_slots = lds_address_of(lds) + kTokens + (uint32_t)wave * (LOADS * 1024);
        auto issue_tokens = [&](int chunk, int slot, auto counted_tag) {  // (the instruction's offset counts in memory too and is taken off the lane's)
            const int8_t* const base = a_base + (int64_t)chunk * 128 - 4096;
            request_rows_16<LOADS, decltype(counted_tag)::value>(row_offset, base, token_slots + (uint32_t)slot * SLOT, chunk, chunks);
        };
        // scales of the tile's rows and of this wave's channels (in the order of its blocks), waited for by hand like all that follows
        uint32_t token_scale_bits, channel_scale_bits;
        {
            const uint64_t of_row = reinterpret_cast<uint64_t>(p.as + slot_of[LOADS]);
            const int own = lane & (kOwn - 1), channel = own >= kHalf ? inner + n0 + own - kHalf : n0 + own;
            const uint64_t of_channel = reinterpret_cast<uint64_t>(p.ws + (int64_t)expert * p.n + channel);
            asm volatile("global_load_ushort %0, %1, off" : "=v"(token_scale_bits) : "v"(of_row) : "memory");
            asm volatile("global_load_ushort %0, %1, off" : "=v"(channel_scale_bits) : "v"(of_channel) : "memory");
        }
        issue_tokens(0, 0, counted);
        issue_tokens(1, 1, counted);
        Each<DEPTH - 2>::run([&](auto i) {
            constexpr int CHUNK = decltype(i)::value + 2;
            issue_codes(CHUNK, std::integral_constant<int, CHUNK>{}, counted), issue_tokens(CHUNK, CHUNK, counted);
        });

        // ---- tables, scales (beside the first loads) ----
        wait_requests<2 * LOADS + (DEPTH - 2) * kChunkRequests>();
        asm volatile("" : "+v"(selector), "+v"(token_scale_bits), "+v"(channel_scale_bits));
        write_paired_entry(lds, tid, false, byte_basis_signed(selector));
        write_paired_entry(lds, tid, true, byte_mask_signed((uint32_t)tid));
        if (tid < kTileRows) reinterpret_cast<float*>(lds + kTokenScale)[tid] = __half2float(__ushort_as_half((unsigned short)token_scale_bits));
        reinterpret_cast<float*>(lds + kChannelScale)[tid] = __half2float(__ushort_as_half((unsigned short)channel_scale_bits));

        v4i acc[NB][CB];
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int j = 0; j < CB; ++j) acc[i][j] = v4i{0, 0, 0, 0};

        // ---- LDS reads ----
        const uint32_t lds_base = lds_address_of(lds);
        const PairedLookup tables(lds_base, lane);
        const uint32_t frag = lds_base + kTokens + (uint32_t)(lane & 15) * 128 + (uint32_t)(((lane >> 4) ^ swizzle(lane & 15)) * 16);
        const uint32_t frag_half = frag ^ 64u;  // of a chunk's second step
        v4i token[2][RB];  // fragments of even and odd phases
        auto read_tokens = [&](auto phase_tag, auto set_tag, auto slot_tag, uint32_t address) {
            constexpr int SET = decltype(set_tag)::value, OFFSET = decltype(slot_tag)::value * (int)SLOT + decltype(phase_tag)::value * RB * 2048;
            lds_read_16<OFFSET>(token[SET][0], address);
            if constexpr (RB > 1) lds_read_16<OFFSET + 2048>(token[SET][1], address);
        };
        v2u looked[LB][2][2];
        auto lookup = [&](int at, uint32_t word) {  // both entries of two codes
            tables.read<0>(looked[at][0], word);
            tables.read<1>(looked[at][1], word);
        };
        auto combine = [&](int at) {
            const v2u first = looked[at][0][0] ^ looked[at][0][1], second = looked[at][1][0] ^ looked[at][1][1];
            return v4i{(int)first[0], (int)first[1], (int)second[0], (int)second[1]};
        };
        auto wait_reads = [&]() {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int l = 0; l < LB; ++l)
                asm volatile("" : "+v"(looked[l][0][0]), "+v"(looked[l][0][1]), "+v"(looked[l][1][0]), "+v"(looked[l][1][1]));
#pragma unroll
            for (int i = 0; i < RB; ++i) asm volatile("" : "+v"(token[0][i]), "+v"(token[1][i]));
        };
        v4i weight[2][CB];  // of a chunk's two steps
        // Phase PHASE of step STEP: its multiplies (one operand changing between consecutive ones), and behind the first of them
        // the fragments of the phase after it and LB blocks of the next step's codes; all of these have come when it ends.
        auto phase = [&](auto step_tag, auto phase_tag, auto next_slot, uint32_t next_fragments, const v2u(&next_codes)[CB], auto requests) {
            constexpr int STEP = decltype(step_tag)::value, PHASE = decltype(phase_tag)::value;
            constexpr int NEXT = (PHASE + 1) % PHASES, TOKENS = (STEP * PHASES + PHASE) & 1;
            constexpr bool LOOKS = PHASE * LB < CB;
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int j = 0; j < CB; ++j) {
                    const int jj = (i & 1) ? CB - 1 - j : j;
                    v4i& sum = acc[PHASE * RB + i][jj];
                    sum = __builtin_amdgcn_mfma_i32_16x16x64_i8(weight[STEP][jj], token[TOKENS][i], sum, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if (i == 0 && j == 0) read_tokens(std::integral_constant<int, NEXT>{}, std::integral_constant<int, 1 - TOKENS>{}, next_slot, next_fragments);
                    if (LOOKS && i == 0 && j >= 1 && j - 1 < LB) lookup(j - 1, next_codes[PHASE * LB + j - 1][1 - STEP]);
                    if (LB == CB && i == 1 && j == 0) lookup(CB - 1, next_codes[CB - 1][1 - STEP]);
                    if (i == 0 && j == CB - 1) requests();
                    __builtin_amdgcn_sched_barrier(0);
                }
            wait_reads();
#pragma unroll
            for (int l = 0; l < (LOOKS ? LB : 0); ++l) weight[1 - STEP][PHASE * LB + l] = combine(l);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto nothing = [] {};
        std::integral_constant<int, 2> two;
        std::integral_constant<int, 3> three;

        // ---- prologue: chunk 0 in LDS, the weights of its first step decoded, its first fragments read ----
        wait_requests<LOADS + (DEPTH - 2) * kChunkRequests>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        Each<CB>::run([&](auto j) { keep(codes[0][j]); });
        read_tokens(zero, zero, zero, frag);
#pragma unroll
        for (int j = 0; j < CB; j += 2) {  // two blocks of channels at a time
            v2u pair[2][2][2];
#pragma unroll
            for (int l = 0; l < 2; ++l) tables.read<0>(pair[l][0], codes[0][j + l][0]), tables.read<1>(pair[l][1], codes[0][j + l][0]);
            wait_reads();
#pragma unroll
            for (int l = 0; l < 2; ++l) {
                keep(pair[l][0][0]), keep(pair[l][0][1]), keep(pair[l][1][0]), keep(pair[l][1][1]);
                const v2u first = pair[l][0][0] ^ pair[l][0][1], second = pair[l][1][0] ^ pair[l][1][1];
                weight[0][j + l] = v4i{(int)first[0], (int)first[1], (int)second[0], (int)second[1]};
            }
        }

        // One chunk: two steps of 64.  In front of its last phase the workgroup meets once: chunk t + 1 has landed,
        // everybody has read chunk t, and the requests of chunk t + DEPTH go out into its slot and its code registers.
        auto chunk_step = [&](int t, auto set_tag) {
            constexpr int SET = decltype(set_tag)::value, NEXT_SET = (SET + 1) % DEPTH;
            std::integral_constant<int, NEXT_SET> other;
            auto meet = [&]() {
                wait_requests<(DEPTH - 2) * kChunkRequests>();
                asm volatile("s_barrier" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            };
            auto request = [&]() {
                issue_codes(t + DEPTH, set_tag, counted_in_loop), issue_tokens(t + DEPTH, SET, counted_in_loop);
            };
            if constexpr (PHASES == 4) {
                phase(zero, zero, set_tag, frag, codes[SET], nothing);
                phase(zero, one, set_tag, frag, codes[SET], nothing);
                phase(zero, two, set_tag, frag, codes[SET], nothing);
                phase(zero, three, set_tag, frag_half, codes[SET], nothing);
            } else {
                phase(zero, zero, set_tag, frag_half, codes[SET], nothing);
            }
            wait_requests<(DEPTH - 2) * kChunkRequests + LOADS>();  // the codes of chunk t + 1 are older than its token rows
            Each<CB>::run([&](auto j) { keep(codes[NEXT_SET][j]); });
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (PHASES == 4) {
                phase(one, zero, set_tag, frag_half, codes[NEXT_SET], nothing);
                phase(one, one, set_tag, frag_half, codes[NEXT_SET], nothing);
                phase(one, two, set_tag, frag_half, codes[NEXT_SET], nothing);
                meet();
                phase(one, three, other, frag, codes[NEXT_SET], request);
            } else {
                meet();
                phase(one, zero, other, frag, codes[NEXT_SET], request);
            }
        };
        for (int t = 0; t < chunks; t += DEPTH)
            Each<DEPTH>::run([&](auto set) {
                if (t + decltype(set)::value < chunks) chunk_step(t + decltype(set)::value, set);
            });

        // ---- epilogue: a lane holds four consecutive channels of one slot in every block.  Stored from there, every instruction touches 16
        // rows in an order that leaves each lane an access of its own, more than a hundred cycles apiece (128 slots of 64
        // channels to a wave: 11300 cycles beside 9800 of the whole K loop at K = 512).  So a block of 16 rows goes through LDS, where
        // the token rows were and private to the wave, and leaves with neighbouring lanes beside each other in a row ----
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");  // nobody's token rows are on their way any more
        if (!live_wave) return;
        int own = threadIdx.x & 63;
        asm volatile("" : "+v"(own));  // nothing of the addresses below is carried through the K loop
        const int quarter = own >> 4, column = own & 15;
        // the scales once, into registers: read where they are used, behind each write of a row, every value waited for an LDS read of its own
        // (13000 of the 29000 cycles of a unit of down)
        float token_scale[NB];
        float4 channel_scale[CB];
#pragma unroll
        for (int i = 0; i < NB; ++i) token_scale[i] = reinterpret_cast<const float*>(lds + kTokenScale)[i * 16 + column];
#pragma unroll
        for (int j = 0; j < CB; ++j)
            channel_scale[j] = *reinterpret_cast<const float4*>(lds + kChannelScale + (wave * 64 + j * 16 + 4 * quarter) * 4);
        constexpr int kWidth = 2 * kHalf, kPitch = kWidth + 16, kLanes = kWidth / 16, kRowsAtOnce = std::min(16, 64 / kLanes);  // bytes of a row; lanes to a row
        uint8_t* const image = lds + kTokens + wave * 8192;  // two blocks of 16 rows
        static_assert(2 * 16 * kPitch <= 8192, "the images of four waves fit where two chunks were");
        __half* const rows_out = (SWIGLU ? p.act : p.out) + (int64_t)row0 * (SWIGLU ? inner : p.n) + n0;
        const int row_stride = SWIGLU ? inner : p.n;
        const bool aligned = ((reinterpret_cast<uintptr_t>(rows_out) | (uintptr_t)row_stride * 2) & 15) == 0;  // (a buffer may be aligned to its elements only)
        auto store_block = [&](int i) {
            const uint8_t* const from = image + (i & 1) * (16 * kPitch);
#pragma unroll
            for (int h = 0; h < 16 / kRowsAtOnce; ++h) {
                const int row = h * kRowsAtOnce + own / kLanes, local = i * 16 + row;
                const uint4 piece = *reinterpret_cast<const uint4*>(from + row * kPitch + own % kLanes * 16);
                if (local >= rows || (kLanes * kRowsAtOnce < 64 && own >= kLanes * kRowsAtOnce)) continue;
                __half* const to = rows_out + (int64_t)local * row_stride + own % kLanes * 8;
                if (aligned) {
                    *reinterpret_cast<uint4*>(to) = piece;
                } else {
                    const uint32_t words[4] = {piece.x, piece.y, piece.z, piece.w};
#pragma unroll
                    for (int e = 0; e < 8; ++e) to[e] = __ushort_as_half((unsigned short)(words[e >> 1] >> (16 * (e & 1))));
                }
            }
        };
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int local = i * 16 + column;
            const bool live = local < rows;
            const int64_t slot = row0 + local;
            uint8_t* const to = image + (i & 1) * (16 * kPitch) + column * kPitch + quarter * 8;
            auto values = [&](int j) {  // of four channels, rounded to fp16 once
                return make_uint2(pack_halves(rescale(acc[i][j][0], channel_scale[j].x, token_scale[i]), rescale(acc[i][j][1], channel_scale[j].y, token_scale[i])),
                                  pack_halves(rescale(acc[i][j][2], channel_scale[j].z, token_scale[i]), rescale(acc[i][j][3], channel_scale[j].w, token_scale[i])));
            };
            if constexpr (!SWIGLU) {
#pragma unroll
                for (int j = 0; j < CB; ++j) *reinterpret_cast<uint2*>(to + j * 32) = values(j);
            } else {
                const bool maxima = p.row_max != nullptr;
                float amax = 0.f;
#pragma unroll
                for (int e = 0; e < CB / 2; ++e) {
                    const uint2 gate = values(e), up = values(e + CB / 2);
                    const uint32_t gates[2] = {gate.x, gate.y}, ups[2] = {up.x, up.y};
                    float v[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        auto half_of = [&](const uint32_t(&words)[2]) { return __ushort_as_half((unsigned short)(words[r >> 1] >> (16 * (r & 1)))); };
                        v[r] = swiglu_value(half_of(gates), half_of(ups));
                        if (maxima) amax = fmaxf(amax, fabsf(v[r]));
                    }
                    *reinterpret_cast<uint2*>(to + e * 32) = make_uint2(pack_halves(v[0], v[1]), pack_halves(v[2], v[3]));
                    if (live && p.out != nullptr) {
                        __half* dst = p.out + slot * p.n + n0 + 16 * e + 4 * quarter;
                        *reinterpret_cast<uint2*>(dst) = gate;
                        *reinterpret_cast<uint2*>(dst + inner) = up;
                    }
                }
                if (maxima) {
                    amax = fmaxf(amax, __shfl_xor(amax, 16, 64));
                    amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
                    if (live && quarter == 0) atomicMax(p.row_max + slot, __float_as_int(amax));
                }
            }
            if (i > 0) store_block(i - 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        store_block(NB - 1);
    };
    if (rows > 64)
        run(std::integral_constant<int, 8>{});
    else if (rows > 32)
        run(std::integral_constant<int, 4>{});
    else
        run(std::integral_constant<int, 2>{});
}

}  // namespace

// What the kernel takes: K-major codes, tiles of 128 rows, whole 64-channel groups per wave, row offsets of 32 bits.
bool grouped_bulk_eligible(int n, int k, int block_m, int packed_k, int64_t rows) {
    return block_m == kTileRows && packed_k == 128 && k % 128 == 0 && n % 64 == 0 && rows * k < (1ll << 31) &&
           (int64_t)n * 32 < (1ll << 31);
}

void grouped_bulk_geometry(int n, int tiles, bool swiglu, Geometry* g) {
    const uint32_t spans = ceil_div((uint32_t)n, (uint32_t)kSpan);
    g->grid[0] = ceil_div((uint32_t)tiles, 8u) * 8u * spans;
    g->grid[1] = g->grid[2] = 1;
    g->block[0] = kThreads;
    g->shared = kLds;
}

// Units of 128 channels: where units of 256 (by what the routed rows of `experts` come to, half a tile each beyond whole ones) leave CUs without one, as a unit of few blocks takes
// as long per step of K whatever the others do.  One to a CU is bound by the chain of a step (reads of LDS, multiplies): 128 x 3200 channels and K 22 us, 256 channels 32; deeper requests
// (three chunks of 128 rows, 80 KiB of LDS) and phases of eight and sixteen multiplies measured within 3 % of it.  gate | up, us, 256 / 128 channels: 2185 tokens of 16 experts
// x top-2, 3200 x 384 31.6 / 22.6; 800 tokens 32.0 / 22.0; 3493 of 128 x 2, 2560 x 256 29.0 / 24.1; with both projections the layer 600 of 32 x 4, 1280 x 512 46.7 / 38.8, 500 of 16 x 8, 4096 x 256 77.5 / 65.1.  The reported geometry is that of the units of 256, as a record of
// a launch names it.
// Tiles go to the eight XCDs in turn, so what counts is the XCD with the most of them: the line is at one unit of 256 to a CU of it (820 projections, time of 256 over 128 channels: up to there
// 0.91-1.56, median 1.32, three of 591 below 0.98; up to a fourth more 0.81-1.20, median 0.99, then 0.80-1.17, 0.93; by the tiles that came, which a launch does not know, 574 of 574 are 1.00
// or more.  Units summed over the chip had 1890 tokens of 8 x 1, 3200 x 1536, in 216 of 36 to an XCD: 37 -> 43 us).
bool grouped_bulk_narrow(int64_t rows, int experts, int n) {
    const int64_t tiles = (rows / kTileRows + experts / 2 + 7) / 8 * 8;
    return tiles * ceil_div((uint32_t)n, (uint32_t)kSpan) <= device_compute_units();
}

int grouped_bulk_launch(const GroupedBuffers& b, int n, int k, int tiles, bool gather, bool swiglu, bool narrow, hipStream_t stream) {
    static DeviceOnce opted_in;  // dynamic LDS above 64 KiB needs an opt-in per kernel and device
    const int ready = opted_in.run([] {
        // (named in this order they also stand so in the code: behind the others the units of 256 took 1 % longer, 1357 tokens, 16 x 8, 1024 x 768 77.9 / 78.5)
#define ORX_BULK(GATHER, SWIGLU, CB) reinterpret_cast<const void*>(&grouped_bulk_kernel<GATHER, SWIGLU, CB>)
        for (const void* kernel : {ORX_BULK(false, false, 4), ORX_BULK(true, false, 4), ORX_BULK(false, true, 4), ORX_BULK(true, true, 4),
                                   ORX_BULK(false, false, 2), ORX_BULK(true, false, 2), ORX_BULK(false, true, 2), ORX_BULK(true, true, 2)}) {
            const int code = hip_check(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds),
                                       "hipFuncSetAttribute");
            if (code != ORX_OK) return code;
        }
#undef ORX_BULK
        return (int)ORX_OK;
    });
    if (ready != ORX_OK) return ready;
    Geometry g;
    grouped_bulk_geometry(n, tiles, swiglu, &g);
    BulkParams p = {};
    p.a = reinterpret_cast<const int8_t*>(b.a), p.as = reinterpret_cast<const __half*>(b.as), p.slot_token = b.slot_token;
    p.w = reinterpret_cast<const uint8_t*>(b.w), p.book = b.book, p.ws = reinterpret_cast<const __half*>(b.ws);
    p.out = reinterpret_cast<__half*>(b.out), p.act = reinterpret_cast<__half*>(b.act);
    p.row_max = swiglu ? const_cast<int*>(b.row_max) : nullptr;
    p.counts = b.counts, p.offsets = b.offsets, p.tile_expert = b.tile_expert, p.tile_row = b.tile_row;
    p.tile_count = b.tile_count, p.tile_units = static_cast<const int4*>(b.tile_units);
    p.n = n, p.k = k, p.tile_capacity = tiles;
    p.spans = (int)ceil_div((uint32_t)n, (uint32_t)span_of(narrow ? 2 : 4));
    const dim3 grid(ceil_div((uint32_t)tiles, 8u) * 8u * (uint32_t)p.spans), block(kThreads);
#define ORX_BULK(GATHER, SWIGLU)                                                                           \
    {                                                                                                      \
        if (narrow) ORX_LAUNCH((grouped_bulk_kernel<GATHER, SWIGLU, 2>), grid, block, g.shared, stream, p); \
        else ORX_LAUNCH((grouped_bulk_kernel<GATHER, SWIGLU, 4>), grid, block, g.shared, stream, p);        \
    }
    if (gather && swiglu) ORX_BULK(true, true)
    else if (gather) ORX_BULK(true, false)
    else if (swiglu) ORX_BULK(false, true)
    else ORX_BULK(false, false)
#undef ORX_BULK
    return hip_check(hipGetLastError(), "launch routed projection (bulk)");
}

}  // namespace orx
