// The first routed single-stage (Q2) expert projection of a decode batch or a short prompt, from the ids of all routes: it works out its tiles by itself, gathers the
// token rows and ends in SwiGLU.
//
// Reference counterpart: the warp-owned routed decode kernels/cuda/model/e8p_decode.py:36-245 behind the tile metadata of kernels/cuda/model/moe.py:713-770.
// Arithmetic: exact int32 over the full K, (float(acc) * ws) * as, rounded to fp16; SwiGLU of those.
//
// The metadata as a launch of its own is one workgroup at work on a chain of reads, ranks and prefixes while the rest of the chip waits, 5.3 us and a launch's gap
// of the layer's 47.5 at 256 tokens x top-8 of 128 experts (2048 x 512), where this kernel takes 2 us more than the one that is handed its tiles: the layer 47.5 -> 42.9 us.
// Here every workgroup reads all ids while its tables are built.  It counts the experts' rows by LDS additions, which need no order; every wave scans the counts
// by itself, finds the tile of its unit among them, and only that tile's routes are ranked: a comparison and a ballot per 64 ids.  Who holds a tile's first span
// writes the tile's part of the metadata for the launches behind, which find what route_metadata leaves.
//
// One resident workgroup of eight waves per CU; a unit is (tile of up to 32 rows, 256 gate and the 256 matching up channels), a wave's share 32 of each over the full K: no
// split of K, no barrier inside a unit.  What bounds the loop is the LDS pipe (a lookup of 8 bytes per lane takes it 4 clocks, a fragment of 1 KiB 8) and behind it the codes'
// stream.  At the size above: ids 1.0 us, tables 1.6,
// rows requested 3.4 and there at 5.0, then a loop of 11.2 us for 16 K blocks of 512 channels (without the codes' traffic 10.9 where it was 12.6, without lookups 8.7) and 1.4 of epilogue.
// Sixteen waves of 32 channels, which read every fragment twice as often: 13.2.  Tables, rows and ring registers leave one workgroup to a CU.
//  * A step is 64 of K: 16 lookups (one v_perm_b32 an address, the paired tables of k_grouped.hip), one fragment per 16 rows, 4 multiplies for each of those.  The
//    reads of a step go out in front of the multiplies of the one before it and are waited for behind them.
//  * Tiles of up to 16 rows read and multiply half as many fragments.
//  * Codes come through a ring of two pairs of K blocks of 128 in registers, refilled right after use, also across the end of a unit into the next one's first pairs.  Where there
//    is none, all lanes read one and the same word: a load under a branch has the compiler wait for all of them.
//  * A tile's rows come by direct loads, 1 KiB to a request, into rows padded by 16 bytes, so that the 16-byte fragment reads do not collide.
//  * Units are dealt in contiguous runs, so a run mostly stays inside one tile, and each XCD gets a stretch of neighbouring workgroups: tiles of one expert meet in one L2.
// The arithmetic of every value is that of the separate launches, so the bits are the same.
#include <hip/hip_fp16.h>

#include <algorithm>

#include "a8_device.h"
#include "e8p_device.h"
#include "lds_asm.h"
#include "moe_device.h"
#include "orx_internal.h"

namespace orx {
namespace {

using lds_asm::v2u;
using lds_asm::v4i;
using lds_asm::v4u;

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;
constexpr int kSpan = kWaves * 32;              // gate channels of a unit, and up channels
constexpr int kRows = 32;                       // of a tile
constexpr int kDepth = 2;                       // pairs of K blocks whose codes are in registers
constexpr int kRowPad = 16;
constexpr int kMaxExperts = 512;
constexpr uint32_t kLdsLimit = 160 * 1024;
// LDS: 256 entries x (16 copies of basis, 16 of mask) x 8 bytes; scales of the tile's rows; the waves' matches; the routes of the tile's rows; the experts' counts, which
// are read again for every tile above 128 experts; the staged rows behind them
constexpr uint32_t kRowScale = 65536, kMatches = kRowScale + kRows * 4, kTileRoutes = kMatches + kWaves * 16, kCounts = kTileRoutes + kRows * 2,
                   kStaged = kCounts + kMaxExperts * 4;
static_assert(kMatches % 16 == 0 && kStaged % 16 == 0, "whole requests, and pairs of words for the matches");

struct RoutedParams {
    const int8_t* a;       // (tokens, K)
    const __half* as;      // (tokens)
    __half* act;           // (slots, N/2)
    int* row_max;          // raised to the fp32 bits of the slot's largest |act|
    __half* out;           // (slots, N) gate | up; may be null
    const uint8_t* w;
    const uint32_t* book;
    const __half* ws;
    int n, k, k_major, routes;
    float inverse_groups, inverse_spans;
    int64_t expert_weight_stride;  // bytes
    RoutedOutputs to;
};

struct Tile {
    int number, expert, row0, rows;  // row0: first slot
    int in_expert;                   // the first row among those of the expert
};

// a barrier that publishes LDS and lets loads from memory stay on their way
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// floor(x / d) from 1 / d, exact for what there are of units: (x + 0.5) / d is at least 0.5 / d away from a whole number
__device__ __forceinline__ int quotient(int x, float inverse) { return __builtin_amdgcn_readfirstlane((int)(((float)x + 0.5f) * inverse)); }

// HELD: ids to a thread, at most; RUN: experts to a lane
template <int HELD, int RUN>
__global__ __launch_bounds__(kThreads) void routed_gate_up_kernel(RoutedParams p) {
    static_assert(HELD == 4 || HELD == 8, "matches of four steps to a word pair");
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, column = lane & 15, quarter = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int chunks = p.k / 128, pairs = (chunks + 1) / 2, inner = p.n / 2, spans = (inner + kSpan - 1) / kSpan;
    const int groups = (int)gridDim.x, b = (int)blockIdx.x;
    const int group = groups % 8 == 0 ? b % 8 * (groups / 8) + b / 8 : b;
    const int row_stride = pairs * 256 + kRowPad;
    uint8_t* const staged_rows = lds + kStaged;
    float* const row_scale = reinterpret_cast<float*>(lds + kRowScale);
    uint16_t* const tile_routes = reinterpret_cast<uint16_t*>(lds + kTileRoutes);
    int* const expert_rows = reinterpret_cast<int*>(lds + kCounts);

    // ---- set-up: the selector table and all ids in one trip; tables and counts ----
    const uint32_t selector = wave < 4 ? p.book[tid] : 0u;
    int id[HELD];  // of route tid + kThreads s
#pragma unroll
    for (int s = 0; s < HELD; ++s) {
        const int at = tid + s * kThreads;
        id[s] = at < p.routes ? p.to.ids[at] : -1;
    }
#pragma unroll
    for (int e = 0; e < 64 * RUN; e += kThreads)
        if (64 * RUN >= kThreads || tid < 64 * RUN) expert_rows[e + tid] = 0;
    if ((chunks & 1) && tid < 8 * kRows) *reinterpret_cast<uint4*>(staged_rows + (tid >> 3) * row_stride + p.k + (tid & 7) * 16) = make_uint4(0, 0, 0, 0);
    lds_barrier();  // (nobody waits for the ids here)
#pragma unroll
    for (int s = 0; s < HELD; ++s)
        if ((uint32_t)id[s] < (uint32_t)p.to.experts) atomicAdd(expert_rows + id[s], 1);
    lds_asm::write_paired_entry<8>(lds, tid & 255, wave >= 4, wave < 4 ? byte_basis_signed(selector) : byte_mask_signed((uint32_t)tid & 255u));
    lds_barrier();
    // a lane has a run of experts; rows in the low half of a word, tiles in the high half
    int packed[RUN], scan = 0;
    auto read_run = [&]() {
#pragma unroll
        for (int j = 0; j < RUN; ++j) packed[j] = expert_rows[lane * RUN + j];
#pragma unroll
        for (int j = 0; j < RUN; ++j) packed[j] |= (packed[j] + kRows - 1) / kRows << 16;
    };
    read_run();
#pragma unroll
    for (int j = 0; j < RUN; ++j) scan += packed[j];
    const int run_sum = scan;
    scan = wave_prefix_sum(scan);
    const int run_first = scan - run_sum, tile_count = __builtin_amdgcn_readlane(scan, 63) >> 16;
    auto tile_at = [&](int number) {
        int before = run_first, expert = 0, row0 = 0, rows = 0, in_expert = 0;
        if constexpr (RUN > 2) {  // (read again: eight registers more are spilled)
            asm volatile("" ::: "memory");
            read_run();
        }
#pragma unroll
        for (int j = 0; j < RUN; ++j) {
            const int nth = number - (before >> 16);
            if (nth >= 0 && nth < packed[j] >> 16) expert = lane * RUN + j, in_expert = kRows * nth, row0 = (before & 0xFFFF) + in_expert, rows = (packed[j] & 0xFFFF) - in_expert;
            before += packed[j];
        }
        const int owner = __builtin_ctzll(__ballot(rows > 0) | 1ull << 63);
        return Tile{number, __builtin_amdgcn_readlane(expert, owner), __builtin_amdgcn_readlane(row0, owner), min(kRows, __builtin_amdgcn_readlane(rows, owner)),
                    __builtin_amdgcn_readlane(in_expert, owner)};
    };

    // ---- units: the same number to every workgroup, one more to the first ones ----
    const int units = tile_count * spans, full = quotient(units, p.inverse_groups), leftover = units - full * groups;
    const int first_unit = group * full + min(group, leftover), my_units = full + (group < leftover ? 1 : 0);
    if (group == groups - 1 && wave == 0) {  // (the workgroup with the fewest units)
        int before = run_first;
#pragma unroll
        for (int j = 0; j < RUN; ++j) {
            const int e = lane * RUN + j;
            if (e < p.to.experts) p.to.counts[e] = packed[j] & 0xFFFF, p.to.row_offsets[e] = before & 0xFFFF, p.to.tile_offsets[e] = before >> 16;
            before += packed[j];
        }
        if (lane == 0) p.to.tile_count[0] = tile_count;
    }

    // ---- the routes of a tile's rows, which are those of its expert in token order: 64 to a step of a wave, the waves of a step one after another ----
    const uint32_t token_magic = __builtin_amdgcn_readfirstlane(((1u << 20) + p.to.top_k - 1) / p.to.top_k);  // (4096 routes x 64 < 2^20)
    auto token_of_route = [&](uint32_t at) { return (int)(__umul24(at, token_magic) >> 20); };
    auto find_routes = [&](const Tile& t) {
        uint64_t same[HELD];
        uint2 matches[HELD / 4];  // of four steps, 16 bits each
#pragma unroll
        for (int s = 0; s < HELD; ++s) same[s] = __ballot(id[s] == t.expert);
#pragma unroll
        for (int h = 0; h < HELD / 4; ++h)
            matches[h] = make_uint2((uint32_t)__popcll(same[4 * h]) | (uint32_t)__popcll(same[4 * h + 1]) << 16,
                                    (uint32_t)__popcll(same[4 * h + 2]) | (uint32_t)__popcll(same[4 * h + 3]) << 16);
#pragma unroll
        for (int h = 0; h < HELD / 4; ++h)
            if (lane == 0) reinterpret_cast<uint2*>(lds + kMatches)[h * kWaves + wave] = matches[h];
        lds_barrier();
        int before = -t.in_expert;  // in front of the step
#pragma unroll
        for (int h = 0; h < HELD / 4; ++h) {
            const uint2 of_wave = reinterpret_cast<const uint2*>(lds + kMatches)[h * kWaves + (lane & (kWaves - 1))];
            // inclusive sums over the eight waves (every eight lanes of a row of 16 hold the same: what the shifts bring from in front of lane 8 is not read)
            auto sum_of = [](uint32_t v) {
                v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);
                v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
                v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
                return v;
            };
            const uint32_t sums[2] = {sum_of(of_wave.x), sum_of(of_wave.y)};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int s = 4 * h + q, shift = 16 * (q & 1);
                const int through = (int)(__builtin_amdgcn_readlane(sums[q >> 1], wave) >> shift & 0xFFFF), all = (int)(__builtin_amdgcn_readlane(sums[q >> 1], kWaves - 1) >> shift & 0xFFFF);
                const int row = before + through - (int)__popcll(same[s]) + (int)__popcll(same[s] & ((1ull << lane) - 1ull));
                if ((same[s] >> lane & 1) && row >= 0 && row < t.rows) tile_routes[row] = (uint16_t)(tid + s * kThreads);
                before += all;
            }
        }
        lds_barrier();
    };
    auto publish = [&](const Tile& t) {  // a tile's part of the metadata, by one wave behind the tile's requests
        if (lane < t.rows) {
            const uint32_t at = tile_routes[lane];
            p.to.relative[at] = t.in_expert + lane, p.to.slot_map[at] = t.row0 + lane, p.to.slot_token[t.row0 + lane] = token_of_route(at);
        }
        if (lane == 0) {
            p.to.tile_expert[t.number] = t.expert, p.to.tile_row[t.number] = t.in_expert;
            p.to.tile_units[t.number] = make_int4(t.expert, t.row0, t.rows, 0);
        }
    };

    // ---- staging: no registers and no address but the row's; requests past a row's end are left out ----
    const uint32_t staged_at = lds_asm::lds_address_of(staged_rows);
    float held_scale = 0.f;
    auto stage = [&](const Tile& t) {
        const int own_token = token_of_route(tile_routes[min(lane & (kRows - 1), t.rows - 1)]);
        held_scale = __half2float(p.as[own_token]);
        const int segments = (p.k + 1023) >> 10;
        for (int row = wave, segment = 0; row < t.rows;) {
            const int token = __builtin_amdgcn_readlane(own_token, row);
            if (segment * 1024 + lane * 16 < p.k)
                lds_asm::request_16<0>((uint32_t)lane * 16, p.a + (int64_t)token * p.k + segment * 1024, staged_at + (uint32_t)(row * row_stride + segment * 1024));
            if (++segment == segments) segment = 0, row += kWaves;
        }
    };

    // ---- a wave's share of a unit: blocks j of 16 channels, gate n0 + 16 j and up inner + n0 + 16 (j - 2) ----
    auto live_block = [&](int n0, int j) { return n0 + 16 * (j & 1) < inner; };
    auto channel_of = [&](int n0, int j) {  // first channel of a block (the wave's first, or the very first, in the place of those behind the end)
        return (live_block(n0, j) ? n0 + 16 * (j & 1) : live_block(n0, 0) ? n0 : 0) + (j >= 2 ? inner : 0);
    };
    // codes: 16 bytes to a lane, of channel `column` of a block; the quarter q multiplies K [64 q, +64) of a pair of K blocks in four steps of 16.  (8 bytes of one block, twice the loads: the loop
    // 12.3 us for 11.0.)  Behind an odd block the rows are zero and the last two quarters read its codes again.
    const uint32_t channel_pitch = p.k_major ? 32u : (uint32_t)chunks * 32u;
    const uint32_t chunk_pitch = p.k_major ? (uint32_t)p.n * 32u : 32u;
    const uint32_t lane_codes = (uint32_t)column * channel_pitch + (uint32_t)(quarter & 1) * 16, lane_second = (uint32_t)(quarter >> 1) * chunk_pitch;
    v4u codes[kDepth][4];
    struct Stream {
        const uint8_t* block[4];
    };
    auto stream_of = [&](int expert, int n0) {
        Stream s;
        const uint8_t* const base = p.w + (int64_t)expert * p.expert_weight_stride;
#pragma unroll
        for (int j = 0; j < 4; ++j) s.block[j] = base + (uint64_t)((uint32_t)channel_of(n0, j) * channel_pitch);
        return s;
    };
    auto fetch = [&](v4u(&set)[4], const Stream& s, int pair, bool wanted) {
        const uint64_t at = wanted ? (uint64_t)((uint32_t)(2 * pair) * chunk_pitch) : 0;
        const uint32_t own = wanted ? lane_codes + (2 * pair + 1 < chunks ? lane_second : 0u) : 0u;
#pragma unroll
        for (int j = 0; j < 4; ++j) set[j] = *reinterpret_cast<const v4u*>(s.block[j] + at + own);
    };

    // ---- decode ----
    const lds_asm::WidePairedLookup paired(lane);
    auto lookup = [&](uint32_t word, uint32_t which) { return *reinterpret_cast<const v2u*>(lds + paired.address(word, which)); };

    if (my_units == 0) return;
    int span;  // of the unit at hand
    Tile cur;
    {
        const int number = quotient(first_unit, p.inverse_spans);
        span = first_unit - number * spans, cur = tile_at(number);
    }
    Stream ahead = stream_of(cur.expert, span * kSpan + wave * 32);  // of the codes requested next: this unit's, from its last blocks on the next one's
    bool fresh = true;  // the rows of the tile at hand are not there yet
    for (int u = 0; u < my_units; ++u) {
        const bool more_units = u + 1 < my_units, same_tile = span + 1 < spans;
        const int n0 = span * kSpan + wave * 32, next_span = same_tile ? span + 1 : 0, next_n0 = next_span * kSpan + wave * 32;
        // Half of the ring in front of the first tile's rows, half behind them: all at once puts off the rows by as much.
        if (u == 0) fetch(codes[0], ahead, 0, true);
        if (fresh) {
            if (u > 0) lds_barrier();  // every wave has finished with the rows staged before
            find_routes(cur);
            stage(cur);
        }
        if (u == 0) fetch(codes[1], ahead, 1, 1 < pairs);
        if (fresh) {
            if (u > 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(4)" ::: "memory");  // the codes behind the rows
            if (tid < kRows) row_scale[tid] = held_scale;
            lds_barrier();
            if (span == 0 && wave == kWaves - 1) publish(cur);
        }
        const Tile nxt = more_units && !same_tile ? tile_at(cur.number + 1) : cur;
        const bool live_wave = live_block(n0, 0), have_next = more_units && live_block(next_n0, 0);
        v2u scale_bits[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) scale_bits[j] = *reinterpret_cast<const v2u*>(p.ws + (int64_t)cur.expert * p.n + channel_of(n0, j) + 4 * quarter);

        auto work = [&](auto blocks_tag) {
            constexpr int NB = decltype(blocks_tag)::value;  // 16-row blocks
            const uint8_t* fragment[NB];
#pragma unroll
            for (int i = 0; i < NB; ++i) fragment[i] = staged_rows + min(i * 16 + column, cur.rows - 1) * row_stride + quarter * 64;
            v4i acc[NB][4], weight[4], token[NB];
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = v4i{0, 0, 0, 0};
            v2u looked[4][4];
            v4i coming[NB];
            auto request = [&](const v4u(&set)[4], auto word_tag, int pair) {  // the reads of one step
                constexpr int word = decltype(word_tag)::value;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t code = set[j][word];
                    looked[j][0] = lookup(code, paired.first_low), looked[j][1] = lookup(code, paired.second_low);
                    looked[j][2] = lookup(code, paired.first_high), looked[j][3] = lookup(code, paired.second_high);
                }
#pragma unroll
                for (int i = 0; i < NB; ++i) coming[i] = *reinterpret_cast<const v4i*>(fragment[i] + pair * 256 + word * 16);
            };
            auto take = [&]() {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const v2u low = looked[j][0] ^ looked[j][1], high = looked[j][2] ^ looked[j][3];
                    weight[j] = v4i{(int)low[0], (int)low[1], (int)high[0], (int)high[1]};
                }
#pragma unroll
                for (int i = 0; i < NB; ++i) token[i] = coming[i];
            };
            auto multiply = [&]() {
#pragma unroll
                for (int i = 0; i < NB; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(weight[j], token[i], acc[i][j], 0, 0, 0);
            };
            std::integral_constant<int, 0> zero;
            std::integral_constant<int, 1> one;
            std::integral_constant<int, 2> two;
            std::integral_constant<int, 3> three;
            request(codes[0], zero, 0);
            take();
            // a step's reads go out in front of the multiplies of the step before it
            auto step = [&](const v4u(&set)[4], auto word_tag, int pair, auto behind) {
                __builtin_amdgcn_sched_barrier(0);
                request(set, word_tag, pair);
                __builtin_amdgcn_sched_barrier(0);
                multiply();
                behind();
                __builtin_amdgcn_sched_barrier(0);
                take();
            };
            auto nothing = [] {};
            auto pair_step = [&](int t, auto set_tag) {
                constexpr int SET = decltype(set_tag)::value, NEXT = (SET + 1) % kDepth;
                step(codes[SET], one, t, nothing);
                step(codes[SET], two, t, nothing);
                step(codes[SET], three, t, [&] {
                    if (t == max(pairs - kDepth, 0)) ahead = stream_of(nxt.expert, next_n0);
                    const bool own = t + kDepth < pairs;
                    fetch(codes[SET], ahead, own ? t + kDepth : SET, own || (have_next && SET < pairs));
                });
                step(codes[NEXT], zero, min(t + 1, pairs - 1), nothing);  // (behind the last pair: read and not used)
                return t + 1 < pairs;
            };
            for (int t = 0;;) {
                if (!pair_step(t++, zero)) break;
                if (!pair_step(t++, one)) break;
            }

            // ---- epilogue: a lane holds channels 4 quarter .. + 3 of every block for the rows `column` of every row block ----
            int own_lane = lane;
            asm volatile("" : "+v"(own_lane));  // (or its addresses are carried through the K loop)
            const int column = own_lane & 15, quarter = own_lane >> 4;
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int local = i * 16 + column;
                const bool live = local < cur.rows;
                const int64_t row = cur.row0 + local;
                const float token_scale = row_scale[min(local, cur.rows - 1)];
                auto value = [&](int j, int r) {
                    const uint32_t bits = scale_bits[j][r >> 1];
                    return __float2half_rn(rescale(acc[i][j][r], __half2float(__ushort_as_half((unsigned short)(bits >> (16 * (r & 1))))), token_scale));
                };
                auto pack4 = [](const __half(&h)[4]) {
                    return make_uint2((uint32_t)__half_as_ushort(h[0]) | (uint32_t)__half_as_ushort(h[1]) << 16,
                                      (uint32_t)__half_as_ushort(h[2]) | (uint32_t)__half_as_ushort(h[3]) << 16);
                };
                float amax = 0.f;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if (!live_block(n0, j)) continue;
                    __half gate[4], up[4], act[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        gate[r] = value(j, r), up[r] = value(j + 2, r);
                        const float v = swiglu_value(gate[r], up[r]);  // already rounded to fp16
                        act[r] = __float2half_rn(v);
                        amax = fmaxf(amax, fabsf(v));
                    }
                    if (live) {
                        const int64_t at = n0 + 16 * j + 4 * quarter;
                        *reinterpret_cast<uint2*>(p.act + row * inner + at) = pack4(act);
                        if (p.out != nullptr) {
                            *reinterpret_cast<uint2*>(p.out + row * p.n + at) = pack4(gate);
                            *reinterpret_cast<uint2*>(p.out + row * p.n + inner + at) = pack4(up);
                        }
                    }
                }
                // the four quarters hold different channels of the same row (non-negative fp32 bits order like integers)
                amax = fmaxf(amax, __shfl_xor(amax, 16, 64));
                amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
                if (live && quarter == 0) atomicMax(p.row_max + row, __float_as_int(amax));
            }
        };
        if (live_wave) {
            if (cur.rows > 16) work(std::integral_constant<int, 2>{});
            else work(std::integral_constant<int, 1>{});
        } else if (more_units) {  // nothing to do in this unit, but perhaps in the next
            ahead = stream_of(nxt.expert, next_n0);
#pragma unroll
            for (int d = 0; d < kDepth; ++d) fetch(codes[d], ahead, d, have_next && d < pairs);
        }
        fresh = !same_tile;
        if (more_units) span = next_span, cur = nxt;
    }
}

uint32_t routed_gate_up_lds(int k) { return kStaged + (uint32_t)kRows * ((uint32_t)(k + 255) / 256 * 256 + kRowPad); }

}  // namespace

// Shapes it takes: whole blocks of 16 gate channels, rows that fit beside the tables, up to 4096 routes in ids of 16 bits' reach.
bool routed_gate_up_eligible(int n, int k, int block_m, int experts, int routes) {
    return block_m == kRows && n % 32 == 0 && k % 128 == 0 && k >= 256 && experts <= kMaxExperts && routes <= 8 * kThreads && routed_gate_up_lds(k) <= kLdsLimit;
}

void routed_gate_up_geometry(int k, Geometry* g) {
    g->grid[0] = (uint32_t)device_compute_units();
    g->grid[1] = g->grid[2] = 1;
    g->block[0] = kThreads;
    g->shared = routed_gate_up_lds(k);
}

int routed_gate_up_launch(const GroupedBuffers& b, int n, int k, int packed_k, int routes, hipStream_t stream) {
    static DeviceOnce opted_in;  // dynamic LDS above 64 KiB needs an opt-in per kernel and device
    const int ready = opted_in.run([] {
        for (const void* kernel : {reinterpret_cast<const void*>(&routed_gate_up_kernel<4, 2>), reinterpret_cast<const void*>(&routed_gate_up_kernel<8, 2>),
                                   reinterpret_cast<const void*>(&routed_gate_up_kernel<4, 8>), reinterpret_cast<const void*>(&routed_gate_up_kernel<8, 8>)}) {
            const int code = hip_check(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsLimit), "hipFuncSetAttribute");
            if (code != ORX_OK) return code;
        }
        return (int)ORX_OK;
    });
    if (ready != ORX_OK) return ready;
    RoutedParams p = {};
    p.a = reinterpret_cast<const int8_t*>(b.a), p.as = reinterpret_cast<const __half*>(b.as);
    p.act = reinterpret_cast<__half*>(b.act), p.row_max = const_cast<int*>(b.row_max), p.out = reinterpret_cast<__half*>(b.out);
    p.w = reinterpret_cast<const uint8_t*>(b.w), p.book = b.book, p.ws = reinterpret_cast<const __half*>(b.ws);
    p.n = n, p.k = k, p.k_major = packed_k != 0, p.routes = routes;
    p.expert_weight_stride = (int64_t)n * (k / 8) * 2;
    p.to = b.routed;
    Geometry g;
    routed_gate_up_geometry(k, &g);
    p.inverse_groups = 1.f / (float)g.grid[0], p.inverse_spans = 1.f / (float)ceil_div((uint32_t)n / 2, (uint32_t)kSpan);
    const dim3 grid(g.grid[0]), block(kThreads);
    if (b.routed.experts <= 128) {
        if (routes <= 4 * kThreads) ORX_LAUNCH((routed_gate_up_kernel<4, 2>), grid, block, g.shared, stream, p);
        else ORX_LAUNCH((routed_gate_up_kernel<8, 2>), grid, block, g.shared, stream, p);
    } else {
        if (routes <= 4 * kThreads) ORX_LAUNCH((routed_gate_up_kernel<4, 8>), grid, block, g.shared, stream, p);
        else ORX_LAUNCH((routed_gate_up_kernel<8, 8>), grid, block, g.shared, stream, p);
    }
    return hip_check(hipGetLastError(), "launch routed projection (gate and up from routes)");
}

}  // namespace orx
