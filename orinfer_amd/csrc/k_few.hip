// The two routed single-stage (Q2) projections of an expert layer where the routed tiles are too few for workgroups that own 512 channels
// (k_grouped.hip): decode batches and short prompts, any K whose sums int32 holds.
//
// Reference counterpart: the warp-owned routed decode kernels/cuda/model/e8p_decode.py:36-245 behind the tile metadata of
// kernels/cuda/model/routing.py.  Arithmetic: exact int32 over the full K, (float(acc) * ws) * as, rounded to fp16 once; fp16(silu(gate) * up).
//
//  * A workgroup of eight waves owns a tile (one expert, up to 32 of its rows) and 32 channels per group of SPLITS waves, which split K between them; the
//    sums meet in LDS.  K blocks of 128: 16 bytes of codes to a lane (a wave's are 1 KiB in a row), two lookups a code, v_mfma_i32_32x32x32_i8.
//  * gate | up: token rows go through a wave's own LDS, a K block at a time: whole cache lines in, eight lanes to a row (fetched as fragments, a lane its own row, an
//    instruction is 64 accesses of the L1 instead of 16, and those were what the streaming kernel waited for).  Nobody else reads them: no barrier in the loop.
//  * gate | up (ACT false): int8 token rows by way of the slot's token, no dispatch copy; a group's 32 channels are 16 of gate and the 16 of up, and
//    the epilogue leaves fp16(silu(gate) * up) and raises the slot's largest magnitude.
//  * down (ACT true): those values, quantised by the A8 rule on their way into LDS, the whole tile once for all groups of the workgroup.
//  * What a tile is comes in one load (TileUnits), so memory is asked three times in a row, not five: tile, token of the slot, row.
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "a8_device.h"
#include "e8p_device.h"
#include "orx_internal.h"

namespace orx {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8, kThreads = kWaves * 64, kRows = 32;
constexpr int kPitch = 128 + 16;                // bytes of a row of a wave's own block: fragment reads spread over the banks
constexpr int kRegion = kRows * kPitch;         // a wave's own LDS: rows of a K block, then its sums
constexpr int kSumPitch = kRows + 1;            // ints of a channel's sums
constexpr int kRowPad = 16;                     // down: bytes behind a staged row of K
constexpr uint32_t kLdsLimit = 160 * 1024;
static_assert(32 * kSumPitch * 4 <= kRegion, "the sums lie where the rows were");

struct FewParams {
    const void* rows;       // gate | up: int8 (tokens, K); down: fp16 (slots, K)
    const __half* scales;   // gate | up: of the token rows
    const int* slot_token;  // gate | up
    int* row_max;           // fp32 bits of a slot's largest magnitude: raised by gate | up, read by down
    const uint8_t* w;
    const uint32_t* book;
    const __half* ws;
    __half* out;            // gate | up: (slots, N / 2); down: (slots, N)
    const int4* units;      // expert, first slot, rows
    const int* tile_count;
    int n, k, tile_rows;    // the most of a tile
    int64_t expert_stride;  // bytes of codes of an expert
};

template <bool ACT, int SPLITS>
__global__ __launch_bounds__(kThreads) void few_rows_kernel(FewParams p) {
    constexpr int GROUPS = kWaves / SPLITS;
    extern __shared__ __align__(16) uint8_t lds[];  // a region to a wave, tables; down: the tile's rows
    uint8_t(*const regions)[kRegion] = reinterpret_cast<uint8_t(*)[kRegion]>(lds);
    Q2ByteTables& tables = *reinterpret_cast<Q2ByteTables*>(lds + kWaves * kRegion);
    uint8_t* const tile_rows = lds + kWaves * kRegion + sizeof(Q2ByteTables);
    const int tile_pitch = p.k + kRowPad;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int split = wave % SPLITS, group = wave / SPLITS;
    const int half = lane >> 5, frag = lane & 31;
    uint8_t* const region = regions[wave];

    // ---- set-up ----
    const uint32_t selector = p.book[tid & 255];
    const int4 unit = p.units[blockIdx.y];  // (nothing there behind the last tile)
    if ((int)blockIdx.y >= p.tile_count[0]) return;
    const int expert = unit.x, row0 = unit.y, rows = min(p.tile_rows, unit.z);  // (a list of taller tiles: the rows that LDS holds)
    if (rows <= 0) return;
    const int inner = p.n / 2;

    // weight row of this lane (clamped: channels beyond the last are computed and not stored)
    const int first = (blockIdx.x * GROUPS + group) * (ACT ? 32 : 16);
    const int w_row = ACT ? min(first + frag, p.n - 1) : min(first + (frag & 15), inner - 1) + (frag < 16 ? 0 : inner);
    const uint8_t* const codes_at = p.w + (int64_t)expert * p.expert_stride + (int64_t)w_row * 32 + half * 16;
    const int64_t kb_step = (int64_t)p.n * 32;
    const int k_blocks = p.k / 128;
    const int kb_first = k_blocks * split / SPLITS, kb_last = k_blocks * (split + 1) / SPLITS;
    auto fetch_codes = [&](int kb) { return *reinterpret_cast<const v4u*>(codes_at + min(kb, k_blocks - 1) * kb_step); };

    // What the epilogue multiplies by: a thread has one channel (a pair, gate and up) of one group and GROUPS (2 GROUPS) of the tile's rows.
    constexpr int kChannels = ACT ? 32 : 16;                                   // of a group in the epilogue
    constexpr int kTurns = GROUPS * kChannels * kRows / kThreads, kTurnRows = kRows / kTurns;
    const int channel = tid % kChannels, out_group = tid / kChannels % GROUPS, out_row = tid / (kChannels * GROUPS);
    const int out_channel = (blockIdx.x * GROUPS + out_group) * kChannels + channel;
    const bool out_live = out_channel < (ACT ? p.n : inner);
    const __half* const ws = p.ws + (int64_t)expert * p.n;
    const int safe_channel = out_live ? out_channel : 0;
    const __half own_scale = ws[safe_channel], up_scale = ACT ? own_scale : ws[inner + safe_channel];
    __half token_scale[kTurns];
    int row_word[kTurns];  // largest magnitude, token
#pragma unroll
    for (int t = 0; t < kTurns; ++t) row_word[t] = (ACT ? p.row_max : p.slot_token)[row0 + min(out_row + t * kTurnRows, rows - 1)];

    // tables: half of the threads each
    auto build = [&]() {
        if (tid < 256)
            tables.basis[tid] = byte_basis_signed(selector);
        else
            tables.mask[tid - 256] = byte_mask_signed((uint32_t)(tid - 256));
    };
    v16i acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0;
    auto multiply = [&](const v4u& codes, const uint8_t* fragment) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const uint2 low = decode_q2(tables, codes[s] & 0xFFFFu), high = decode_q2(tables, codes[s] >> 16);
            const v4i weights = {(int)low.x, (int)low.y, (int)high.x, (int)high.y};
            const v4i tokens = *reinterpret_cast<const v4i*>(fragment + 16 * s);
            acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(weights, tokens, acc, 0, 0, 0);
        }
    };
    if constexpr (ACT) {
        // the tile's rows, quantised once for all groups
        v4u codes[2] = {fetch_codes(kb_first), fetch_codes(kb_first + 1)};
        const int pieces_per_row = p.k / 8, pieces = rows * pieces_per_row;
        const v4u* const values = reinterpret_cast<const v4u*>(reinterpret_cast<const __half*>(p.rows) + (int64_t)row0 * p.k);
        build();
        constexpr int kTogether = 2;
        for (int at = tid; at < pieces; at += kTogether * kThreads) {
            v4u held[kTogether];
            int row[kTogether], bits[kTogether];
#pragma unroll
            for (int i = 0; i < kTogether; ++i) {
                const int piece = min(at + i * kThreads, pieces - 1);
                row[i] = piece / pieces_per_row;
                held[i] = values[piece];
                bits[i] = p.row_max[row0 + row[i]];
            }
#pragma unroll
            for (int i = 0; i < kTogether; ++i) {
                const int piece = min(at + i * kThreads, pieces - 1), col = piece - row[i] * pieces_per_row;
                const float scale = __half2float(a8_scale(__int_as_float(bits[i]))), inverse = __frcp_rn(scale);
                const __half* h = reinterpret_cast<const __half*>(&held[i]);
                const float low[4] = {__half2float(h[0]), __half2float(h[1]), __half2float(h[2]), __half2float(h[3])};
                const float high[4] = {__half2float(h[4]), __half2float(h[5]), __half2float(h[6]), __half2float(h[7])};
                *reinterpret_cast<uint2*>(tile_rows + row[i] * tile_pitch + col * 8) = make_uint2(quantise4(low, scale, inverse), quantise4(high, scale, inverse));
            }
        }
        __syncthreads();
        const uint8_t* const fragment = tile_rows + min(frag, rows - 1) * tile_pitch + half * 64;
        for (int kb = kb_first; kb < kb_last; kb += 2) {
            multiply(codes[0], fragment + kb * 128);
            codes[0] = fetch_codes(kb + 2);
            if (kb + 1 < kb_last) {
                multiply(codes[1], fragment + kb * 128 + 128);
                codes[1] = fetch_codes(kb + 3);
            }
        }
    } else {
        // rows that this lane brings, piece i of a K block: row 8 i + lane / 8, bytes 16 (lane % 8)
        auto run = [&](auto pieces_tag) {
            constexpr int PIECES = decltype(pieces_tag)::value;  // 8 rows each
            const uint8_t* row_at[PIECES];
            const int staged_row = lane / 8, staged_piece = lane % 8;
            int token[PIECES];
#pragma unroll
            for (int i = 0; i < PIECES; ++i) token[i] = p.slot_token[row0 + min(i * 8 + staged_row, rows - 1)];
            v4u codes[2] = {fetch_codes(kb_first), fetch_codes(kb_first + 1)}, piece[2][PIECES];
#pragma unroll
            for (int i = 0; i < PIECES; ++i) row_at[i] = reinterpret_cast<const uint8_t*>(p.rows) + (int64_t)token[i] * p.k + staged_piece * 16;
            auto fetch_rows = [&](v4u(&to)[PIECES], int kb) {
#pragma unroll
                for (int i = 0; i < PIECES; ++i) to[i] = *reinterpret_cast<const v4u*>(row_at[i] + min(kb, k_blocks - 1) * 128);
            };
            fetch_rows(piece[0], kb_first);
            fetch_rows(piece[1], kb_first + 1);
#pragma unroll
            for (int t = 0; t < kTurns; ++t) token_scale[t] = p.scales[row_word[t]];
            build();
            __syncthreads();
            const uint8_t* const fragment = region + min(frag, PIECES * 8 - 1) * kPitch + half * 64;
            auto block = [&](const v4u& of, const v4u(&from)[PIECES]) {
#pragma unroll
                for (int i = 0; i < PIECES; ++i) *reinterpret_cast<v4u*>(region + (i * 8 + staged_row) * kPitch + staged_piece * 16) = from[i];
                __builtin_amdgcn_wave_barrier();  // (LDS serves a wave in order)
                multiply(of, fragment);
                __builtin_amdgcn_wave_barrier();
            };
            for (int kb = kb_first; kb < kb_last; kb += 2) {
                block(codes[0], piece[0]);
                codes[0] = fetch_codes(kb + 2);
                fetch_rows(piece[0], kb + 2);
                if (kb + 1 < kb_last) {
                    block(codes[1], piece[1]);
                    codes[1] = fetch_codes(kb + 3);
                    fetch_rows(piece[1], kb + 3);
                }
            }
        };
        if (rows <= 8)
            run(std::integral_constant<int, 1>{});
        else if (rows <= 16)
            run(std::integral_constant<int, 2>{});
        else
            run(std::integral_constant<int, 4>{});
    }

    // ---- epilogue.  Accumulator register r of a lane: channel 8 (r / 4) + 4 half + r % 4 of the group, row `frag` ----
    int* const sums = reinterpret_cast<int*>(region);
#pragma unroll
    for (int r = 0; r < 16; ++r) sums[(8 * (r >> 2) + 4 * half + (r & 3)) * kSumPitch + frag] = acc[r];
    __syncthreads();
    auto total = [&](int of_channel, int row) {
        int sum = 0;
#pragma unroll
        for (int s = 0; s < SPLITS; ++s) sum += reinterpret_cast<const int*>(regions[out_group * SPLITS + s])[of_channel * kSumPitch + row];
        return sum;
    };
#pragma unroll
    for (int t = 0; t < kTurns; ++t) {
        const int row = out_row + t * kTurnRows;
        const int64_t slot = row0 + row;
        const bool live = out_live && row < rows;
        if constexpr (ACT) {
            const float token = __half2float(a8_scale(__int_as_float(row_word[t])));
            if (live) p.out[slot * p.n + out_channel] = __float2half_rn(rescale(total(channel, row), __half2float(own_scale), token));
        } else {
            const float token = __half2float(token_scale[t]);
            const __half gate = __float2half_rn(rescale(total(channel, row), __half2float(own_scale), token));
            const __half up = __float2half_rn(rescale(total(channel + 16, row), __half2float(up_scale), token));
            const float value = swiglu_value(gate, up);
            if (live) p.out[slot * inner + out_channel] = __float2half_rn(value);
            // of the workgroup's channels of this row, 16 GROUPS neighbouring lanes; NaN is no magnitude
            uint32_t largest = row_max_u32(__float_as_uint(live ? fmaxf(0.f, fabsf(value)) : 0.f));
            if constexpr (GROUPS > 1) largest = max(largest, (uint32_t)__shfl_xor((int)largest, 16, 64));
            if constexpr (GROUPS > 2) largest = max(largest, (uint32_t)__shfl_xor((int)largest, 32, 64));
            if (row < rows && tid % (16 * GROUPS) == 0) atomicMax(p.row_max + slot, (int)largest);
        }
    }
}

// ---- host side ----
// slots used: K, N, E, tiles, capacity, flags (bit 0: fp16 rows)
// Waves that share a group.  gate | up: a wave's K blocks one after another (0.75 us each) against set-up, tables and sums of the workgroups that have to be run (about
// 0.005 us each over the chip, tiles by uniform popularity): 2, 4 and 8 of them are the fastest of the three within 3 % on 16 of 18 shapes by this rule (layer,
// us, 2 / 4 / 8: 29 tokens, 128 experts x top-4, 3840 x 256 37.2 / 32.0 / 31.0; 5, 64 x 8, 2432 x 768 30.8 / 30.7 / 33.9; 85, 32 x 8, 1920 x 1280 62.9 / 66.0 / 71.5).
// down: a workgroup quantises the whole tile, so few of them: two waves to a group, 128 channels, and one, 256, where rows are long and CUs have several
// (85, 32 x 8, 1920 x 1280 66.0 -> 62.9, otherwise 1 to 8 % slower; four waves 2 % faster to 13 % slower).
int splits_for(const orx_function& f) {
    const bool act = f.flags & 1;
    const double hit = f.E * (1.0 - std::exp(-(double)f.capacity / f.E)), tiles = std::max(hit, f.capacity / 32.0);
    const int blocks = f.K / 128;
    if (act) return blocks >= 8 && tiles * ((f.N + 127) / 128) >= 2 * device_compute_units() ? 1 : 2;
    int best = 0;
    double least = 0;
    for (const int splits : {2, 4, 8}) {
        const int of_workgroup = kWaves / splits * 16;
        const double time = 0.75 * blocks / splits + 0.005 * tiles * ((f.N / 2 + of_workgroup - 1) / of_workgroup);
        if (best == 0 || time < least) best = splits, least = time;
    }
    return best;
}

// rows of a tile, for which down has LDS
int most_rows(const orx_function& f) { return std::min(kRows, f.capacity); }

int few_geometry(const orx_function& f, int, Geometry* g) {
    const bool act = f.flags & 1;
    const int channels = (kWaves / splits_for(f)) * (act ? 32 : 16);
    g->grid[0] = ceil_div((uint32_t)(act ? f.N : f.N / 2), (uint32_t)channels);
    g->grid[1] = (uint32_t)f.tiles;
    g->block[0] = kThreads;
    g->shared = kWaves * kRegion + (uint32_t)sizeof(Q2ByteTables) + (act ? (uint32_t)most_rows(f) * (f.K + kRowPad) : 0u);
    return ORX_OK;
}

// gate | up: A, AS, Act, Book, P, RowMax, SlotToken, TileCount, TileUnits, WS; down: A, Book, C, P, RowMax, TileCount, TileUnits, WS
int few_launch(const orx_function& f, int, const Geometry& g, hipStream_t stream, void** args) {
    static DeviceOnce opted_in;  // dynamic LDS above 64 KiB needs an opt-in per kernel and device
    const int ready = opted_in.run([] {
        for (const void* kernel : {reinterpret_cast<const void*>(&few_rows_kernel<true, 1>), reinterpret_cast<const void*>(&few_rows_kernel<true, 2>)}) {
            const int code = hip_check(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsLimit), "hipFuncSetAttribute");
            if (code != ORX_OK) return code;
        }
        return (int)ORX_OK;
    });
    if (ready != ORX_OK) return ready;
    const bool act = f.flags & 1;
    FewParams p = {};
    int next = 0;
    p.rows = pointer_arg<const void>(args, next++);
    if (!act) p.scales = pointer_arg<const __half>(args, next++), p.out = pointer_arg<__half>(args, next++);
    p.book = pointer_arg<const uint32_t>(args, next++);
    if (act) p.out = pointer_arg<__half>(args, next++);
    p.w = pointer_arg<const uint8_t>(args, next++);
    p.row_max = pointer_arg<int>(args, next++);
    if (!act) p.slot_token = pointer_arg<const int>(args, next++);
    p.tile_count = pointer_arg<const int>(args, next++);
    p.units = pointer_arg<const int4>(args, next++);
    p.ws = pointer_arg<const __half>(args, next++);
    p.n = f.N, p.k = f.K, p.tile_rows = most_rows(f), p.expert_stride = (int64_t)f.N * (f.K / 8) * 2;
    const dim3 grid(g.grid[0], g.grid[1]), block(kThreads);
#define ORX_FEW(ACT, S) ORX_LAUNCH((few_rows_kernel<ACT, S>), grid, block, g.shared, stream, p)
    const int splits = splits_for(f);
    if (act) {
        if (splits == 2) ORX_FEW(true, 2);
        else ORX_FEW(true, 1);
    } else {
        if (splits == 8) ORX_FEW(false, 8);
        else if (splits == 4) ORX_FEW(false, 4);
        else ORX_FEW(false, 2);
    }
#undef ORX_FEW
    return hip_check(hipGetLastError(), "launch routed projection (few rows)");
}

}  // namespace

// e8p_decode_grouped with few_rows=true: rows (slots), E, tiles, N, K; gather=true with epilogue=swiglu, or input_dtype=float16
int make_few_rows(const Variant& v, orx_function* f) {
    bool bad = false;
    f->capacity = f->M = (int)v.integer("rows", 0, &bad);
    f->E = (int)v.integer("E", 0, &bad);
    f->tiles = (int)v.integer("tiles", 0, &bad);
    f->N = (int)v.integer("N", 0, &bad);
    f->K = (int)v.integer("K", 0, &bad);
    f->block_m = (int)v.integer("block_m", 32, &bad);
    f->packed_k = (int)v.integer("packed_k", 128, &bad);
    const bool act = v.string("input_dtype", "int8", &bad) == "float16", gather = v.boolean("gather", false, &bad);
    const std::string epilogue = v.string("epilogue", "none", &bad), algorithm = v.string("algorithm", "auto", &bad);
    if (bad) return ORX_ERR_BAD_VARIANT;
    if (f->M <= 0 || f->E <= 0 || f->tiles <= 0 || f->tiles > 65535 || f->N <= 0 || f->N % 32 || f->K <= 0 || f->K % 128 ||
        (int64_t)f->K * 128 * 128 > 2147483647LL || f->block_m != 32 || f->packed_k != 128 || algorithm != "auto" ||
        (act ? gather || epilogue != "none" : !gather || epilogue != "swiglu")) {
        set_error("%s: few_rows=true serves lists of up to 65535 32-row tiles, packed_k=128, N a multiple of 32, K of 128 with K * 2^14 < 2^31, algorithm auto: gather=true "
                  "with epilogue=swiglu, or input_dtype=float16", f->symbol.c_str());
        return ORX_ERR_BAD_VARIANT;
    }
    f->flags = act ? 1 : 0;
    Geometry g;
    few_geometry(*f, f->capacity, &g);
    if (g.shared > kLdsLimit) {
        set_error("%s: few_rows=true stages the fp16 rows of a tile: K=%d is too long for LDS", f->symbol.c_str(), f->K);
        return ORX_ERR_BAD_VARIANT;
    }
    if (act)
        f->args = {{"A", ArgPointer, 16}, {"Book", ArgPointer, 4}, {"C", ArgPointer, 2}, {"P", ArgPointer, 16}, {"RowMax", ArgPointer, 4},
                   {"TileCount", ArgPointer, 4}, {"TileUnits", ArgPointer, 16}, {"WS", ArgPointer, 2}};
    else
        f->args = {{"A", ArgPointer, 16}, {"AS", ArgPointer, 2}, {"Act", ArgPointer, 2}, {"Book", ArgPointer, 4}, {"P", ArgPointer, 16},
                   {"RowMax", ArgPointer, 4}, {"SlotToken", ArgPointer, 4}, {"TileCount", ArgPointer, 4}, {"TileUnits", ArgPointer, 16}, {"WS", ArgPointer, 2}};
    f->geometry = few_geometry;
    f->launch = few_launch;
    f->device_function = nullptr;
    return ORX_OK;
}

}  // namespace orx
