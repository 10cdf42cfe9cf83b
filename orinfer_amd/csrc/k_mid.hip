// int8 x int8 projections of some hundred to some thousand rows whose 256 x 256 tiles (k_gemm_big.hip) leave CUs idle: 128 x 128 tiles, whole or with the K
// steps of all tiles dealt evenly to the workgroups.
//
// Reference counterpart: the Tensor Core schedules of kernels/cuda/model/integer_core.py:162-272 at block_m 128.  Arithmetic: exact int32 over the full K,
// (float(acc) * ws) * as.
//
//  * Four waves of 64 rows x 64 channels, v_mfma_i32_16x16x64_i8, weights as the row operand: a lane holds four channels of one token.  Operands go from memory
//    to LDS directly, K steps of 128 in whole lines, in stages of 32 KiB: four where CUs have one workgroup each, two where they have two, of which one multiplies
//    while the other waits.
//  * A step is two slices of 64.  The fragments of a slice arrive while the other one is multiplied; one barrier a step, behind the last fragment reads of its
//    stage, and right behind it the wave's eight requests for the stage go out between the multiplies.
//  * A workgroup takes a tile, or one of a few parts of its K where tiles are few: then it leaves its int32 sums, and mid_finish_kernel adds a tile's parts
//    (integers: exact in any order).
#include <hip/hip_fp16.h>

#include <algorithm>

#include "e8p_device.h"
#include "lds_asm.h"
#include "orx_internal.h"

namespace orx {
namespace {

using namespace lds_asm;

constexpr int kTile = 128, kStep = 128, kThreads = 256;
constexpr uint32_t kOperand = kTile * kStep, kStage = 2 * kOperand;  // 16 KiB of token rows, 16 KiB of weights
constexpr int kSlotInts = kTile * kTile;

struct MidParams {
    const int8_t* a;
    const int8_t* w;
    const __half* ws;
    const __half* as;
    void* out;
    int* partials;
    int n, k, stride, m, out_f32;
    int tiles_m, tiles_n, parts;
};

// down M in groups of 8 for each N: neighbouring tiles share operands
__device__ __forceinline__ void tile_at(int number, int tiles_m, int tiles_n, int* tm, int* tn) {
    constexpr int kGroup = 8;
    const int first = number / (kGroup * tiles_n) * kGroup, rows = min(kGroup, tiles_m - first), within = number % (kGroup * tiles_n);
    *tm = first + within % rows, *tn = within / rows;
}

template <int N>
__device__ __forceinline__ void wait_for(v4i (&f)[4], v4i (&g)[4]) {
    asm volatile("s_waitcnt lgkmcnt(%8)"
                 : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(g[0]), "+v"(g[1]), "+v"(g[2]), "+v"(g[3])
                 : "n"(N)
                 : "memory");
}

template <int STAGES>
__global__ __launch_bounds__(kThreads, STAGES == 2 ? 2 : 1) void gemm_mid_kernel(MidParams p) {
    extern __shared__ __align__(16) uint8_t lds[];  // the stages
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_m = wave >> 1, wave_n = wave & 1;
    const uint32_t lds_base = lds_address_of(lds);
    // consecutive workgroups go to the eight XCDs in turn: each gets one stretch of the list, whose neighbours share operands (a part of K of all tiles
    // before the next part); the first workgroups % 8 stretches are one longer.  (Without stretches where the count was no multiple of eight, 560 shapes took 1.19 (codes) and 1.05 times (int8)
    // as long in the median: linears of codes, 833 x 6912 x 4864 60.7 -> 50.8 us, 803 x 7029 x 16256 211 -> 140.)  Up to eight columns of tiles, whose weights every L2 holds, lose up to 5 % by it
    // and seldom gain, so such a list without a multiple of eight goes as it is: rows of tiles are then dealt to the XCDs.
    const int workgroups = gridDim.x, tiles = p.tiles_m * p.tiles_n, xcd = (int)blockIdx.x & 7;
    const bool stretches = p.tiles_n > 8 || (workgroups & 7) == 0;
    const int number = stretches ? xcd * (workgroups >> 3) + min(xcd, workgroups & 7) + ((int)blockIdx.x >> 3) : (int)blockIdx.x;
    const int part = number / tiles, tile = number % tiles, k_tiles = p.k / kStep;
    const int kt_begin = k_tiles * part / p.parts, steps = k_tiles * (part + 1) / p.parts - kt_begin;

    // fragment: K bytes [16 (lane / 16), +16) of a slice, row lane % 16 of a block; the second slice is bit 6 of the address
    const int frag_row = lane & 15, quarter = lane >> 4;
    const uint32_t a_frag = lds_base + (uint32_t)(wave_m * 64 + frag_row) * kStep + (uint32_t)((quarter ^ swizzle(frag_row)) * 16);
    const uint32_t w_frag = lds_base + kOperand + (uint32_t)(wave_n * 64 + frag_row) * kStep + (uint32_t)((quarter ^ swizzle(frag_row)) * 16);
    // requests: rows 32 wave + 8 b + lane / 8 of either operand, b < 4, the piece of 16 bytes that belongs at lane % 8
    const int load_row = wave * 32 + (lane >> 3);
    const uint32_t load_piece = (uint32_t)(((lane & 7) ^ swizzle(load_row)) * 16);  // of even b; odd b: bit 6 the other way round

    v4i ft[2][4], fw[2][4];
    int tm, tn;
    tile_at(tile, p.tiles_m, p.tiles_n, &tm, &tn);
    const int row0 = tm * kTile, col0 = tn * kTile, rows = min(kTile, p.m - row0), cols = min(kTile, p.n - col0);
    const int8_t* const a_base = uniform_pointer(p.a + (int64_t)row0 * p.k + (int64_t)kt_begin * kStep);
    const int8_t* const w_base = uniform_pointer(p.w + (int64_t)col0 * p.k + (int64_t)kt_begin * kStep);
    // (an offset of a request counts on both sides: 1 KiB further in LDS, and here taken off again)
    uint32_t a_offset[4], w_offset[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const uint32_t piece = (load_piece ^ (uint32_t)((b & 1) * 64)) + (uint32_t)(3 - b) * 1024;
        a_offset[b] = (uint32_t)min(load_row + 8 * b, rows - 1) * (uint32_t)p.k + piece;
        w_offset[b] = (uint32_t)min(load_row + 8 * b, cols - 1) * (uint32_t)p.k + piece;
    }
    // the wave's four requests of a step for either operand, by no lane behind the last step: they are waited for by number
    auto request = [&](auto weights_tag, int step, uint32_t stage) {
        constexpr bool weights = decltype(weights_tag)::value != 0;
        request_rows_16<4, true>(weights ? w_offset : a_offset, (weights ? w_base : a_base) + (int64_t)step * kStep - 3072,
                                 lds_base + stage + (weights ? kOperand : 0u) + (uint32_t)wave * 4096, step, steps);
    };
    auto read_slice = [&](auto slice_tag, uint32_t stage) {
        constexpr int slice = decltype(slice_tag)::value;
        const uint32_t a = (a_frag ^ (uint32_t)(slice * 64)) + stage, w = (w_frag ^ (uint32_t)(slice * 64)) + stage;
        Each<4>::run([&](auto tag) { lds_read_16<decltype(tag)::value * 16 * kStep>(ft[slice][decltype(tag)::value], a); });
        Each<4>::run([&](auto tag) { lds_read_16<decltype(tag)::value * 16 * kStep>(fw[slice][decltype(tag)::value], w); });
    };
    std::integral_constant<int, 0> zero;
    std::integral_constant<int, 1> one;

    v4i acc[4][4];
    // a slice, token by token back and forth over the channels; `between` behind every second multiply
    auto multiply = [&](auto slice_tag, auto... between) {
        constexpr int slice = decltype(slice_tag)::value;
        Each<16>::run([&](auto m_tag) {
            constexpr int m = decltype(m_tag)::value, i = m / 4, j = (i & 1) ? 3 - m % 4 : m % 4;
            multiply_in_place<false>(acc[i][j], fw[slice][j], ft[slice][i]);
            if constexpr ((m & 1) == 1) {
                __builtin_amdgcn_sched_barrier(0);
                (between(std::integral_constant<int, m / 2>{}), ...);
                __builtin_amdgcn_sched_barrier(0);
            }
        });
    };
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            acc[i][j] = v4i{0, 0, 0, 0};
            keep(acc[i][j]);
        }
    Each<STAGES>::run([&](auto stage_tag) {
        constexpr int stage = decltype(stage_tag)::value;
        request(zero, stage, stage * kStage), request(one, stage, stage * kStage);
    });
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(8 * (STAGES - 1)) : "memory");
    read_slice(zero, 0);
    // One body for all steps (copies of it for the last ones would move fragments between registers while they are on their way): requests behind the last step
    // bring nothing, and what is read for the step behind it nobody uses.
    uint32_t current = 0;
    for (int step = 0; step < steps; ++step) {
        read_slice(one, current);
        wait_for<8>(ft[0], fw[0]);
        __builtin_amdgcn_sched_barrier(0);
        multiply(zero);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 * (STAGES - 2)) : "memory");
        wait_for<0>(ft[1], fw[1]);
        asm volatile("s_barrier" ::: "memory");  // the next step is in LDS, and nobody reads this one any more
        const uint32_t next = STAGES == 2 ? current ^ kStage : (current + kStage) % (STAGES * kStage);
        read_slice(zero, next);
        __builtin_amdgcn_sched_barrier(0);
        multiply(one, [&](auto tag) {
            constexpr int m = decltype(tag)::value;
            if constexpr (m == 0) request(zero, step + STAGES, current);
            if constexpr (m == 4) request(one, step + STAGES, current);
        });
        __builtin_amdgcn_sched_barrier(0);
        current = next;
    }
    wait_for<0>(ft[0], fw[0]);
    asm volatile("s_nop 15" ::: "memory");  // the last sums are written
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) keep(acc[i][j]);

    if (p.parts > 1) {
        // block (i, j) of thread tid, four sums, at ((4 i + j) 256 + tid) 4: 1 KiB to a store
        v4i* const slot = reinterpret_cast<v4i*>(p.partials + (int64_t)number * kSlotInts) + tid;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) slot[(4 * i + j) * kThreads] = acc[i][j];
    } else {
        float channel_scale[4][4], token_scale[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            token_scale[j] = __half2float(p.as[row0 + min(wave_m * 64 + j * 16 + frag_row, rows - 1)]);
#pragma unroll
            for (int r = 0; r < 4; ++r) channel_scale[j][r] = __half2float(p.ws[col0 + min(wave_n * 64 + j * 16 + 4 * quarter + r, cols - 1)]);
        }
        if (p.out_f32) {
            // (a lane's four channels in one store: 249 x 19456 x 512 24.0 -> 12.4 us, value by value)
            const bool aligned = p.stride % 4 == 0 && (reinterpret_cast<uintptr_t>(p.out) & 15) == 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = wave_m * 64 + i * 16 + frag_row;
                if (row >= rows) continue;
                float* const to = reinterpret_cast<float*>(p.out) + (int64_t)(row0 + row) * p.stride + col0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int col = wave_n * 64 + j * 16 + 4 * quarter;
                    const float value[4] = {rescale(acc[i][j][0], channel_scale[j][0], token_scale[i]), rescale(acc[i][j][1], channel_scale[j][1], token_scale[i]),
                                            rescale(acc[i][j][2], channel_scale[j][2], token_scale[i]), rescale(acc[i][j][3], channel_scale[j][3], token_scale[i])};
                    if (aligned && col + 4 <= cols) {
                        *reinterpret_cast<float4*>(to + col) = make_float4(value[0], value[1], value[2], value[3]);
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (col + r < cols) to[col + r] = value[r];
                    }
                }
            }
        } else {
            // 16 rows x 64 channels at a time through the wave's own LDS (nobody reads the stages any more), whole rows of 128 bytes out
            uint8_t* const image = lds + wave * 4096;
            __half* const out = reinterpret_cast<__half*>(p.out) + (int64_t)(row0 + wave_m * 64) * p.stride + col0;
            const bool aligned = p.stride % 8 == 0 && (reinterpret_cast<uintptr_t>(p.out) & 15) == 0;
            const int local_col = wave_n * 64 + (lane & 7) * 8;
            auto store_block = [&](int i) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int local = h * 8 + (lane >> 3), row = i * 16 + local;
                    const uint4 piece = *reinterpret_cast<const uint4*>(image + (i & 1) * 2048 + local * 128 + ((lane & 7) ^ (local & 7)) * 16);
                    if (wave_m * 64 + row >= rows || local_col >= cols) continue;
                    __half* const to = out + (int64_t)row * p.stride + local_col;
                    if (aligned && local_col + 8 <= cols) {
                        *reinterpret_cast<uint4*>(to) = piece;
                    } else {
                        const uint32_t parts[4] = {piece.x, piece.y, piece.z, piece.w};
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            if (local_col + e < cols) to[e] = __ushort_as_half((unsigned short)(parts[e >> 1] >> (16 * (e & 1))));
                    }
                }
            };
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    *reinterpret_cast<uint2*>(image + (i & 1) * 2048 + frag_row * 128 + (((2 * j + (quarter >> 1)) ^ (frag_row & 7)) * 16) + (quarter & 1) * 8) =
                        make_uint2(pack_halves(rescale(acc[i][j][0], channel_scale[j][0], token_scale[i]), rescale(acc[i][j][1], channel_scale[j][1], token_scale[i])),
                                   pack_halves(rescale(acc[i][j][2], channel_scale[j][2], token_scale[i]), rescale(acc[i][j][3], channel_scale[j][3], token_scale[i])));
                if (i > 0) store_block(i - 1);
            }
            store_block(3);
        }
    }
}

// Four workgroups per tile, one per row block of every wave: the sums of the tile's parts, rescaled.
__global__ __launch_bounds__(kThreads) void mid_finish_kernel(MidParams p) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int tile = blockIdx.x >> 2, i = blockIdx.x & 3, tiles = p.tiles_m * p.tiles_n;
    v4i acc[4] = {};
#pragma unroll 2
    for (int part = 0; part < p.parts; ++part) {
        const v4i* const slot = reinterpret_cast<const v4i*>(p.partials + ((int64_t)part * tiles + tile) * kSlotInts) + tid;
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] += slot[(4 * i + j) * kThreads];
    }
    int tm, tn;
    tile_at(tile, p.tiles_m, p.tiles_n, &tm, &tn);
    const int row0 = tm * kTile, col0 = tn * kTile, rows = min(kTile, p.m - row0), cols = min(kTile, p.n - col0);
    const int row = (wave >> 1) * 64 + i * 16 + (lane & 15);
    if (row >= rows) return;
    const float token_scale = __half2float(p.as[row0 + row]);
    const bool aligned = p.stride % 4 == 0 && (reinterpret_cast<uintptr_t>(p.out) & (p.out_f32 ? 15 : 7)) == 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int col = (wave & 1) * 64 + j * 16 + 4 * (lane >> 4);
        if (col >= cols) continue;
        float value[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) value[r] = rescale(acc[j][r], __half2float(p.ws[col0 + min(col + r, cols - 1)]), token_scale);
        const int64_t at = (int64_t)(row0 + row) * p.stride + col0 + col;
        if (p.out_f32 && aligned && col + 4 <= cols) {
            *reinterpret_cast<float4*>(reinterpret_cast<float*>(p.out) + at) = make_float4(value[0], value[1], value[2], value[3]);
        } else if (aligned && col + 4 <= cols) {
            *reinterpret_cast<uint2*>(reinterpret_cast<__half*>(p.out) + at) = make_uint2(pack_halves(value[0], value[1]), pack_halves(value[2], value[3]));
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (col + r >= cols) continue;
                if (p.out_f32)
                    reinterpret_cast<float*>(p.out)[at + r] = value[r];
                else
                    reinterpret_cast<__half*>(p.out)[at + r] = __float2half_rn(value[r]);
            }
        }
    }
}

}  // namespace

// Tiles in `parts` of K: one, or `partials` holds 64 KiB for each of them.  Up to one workgroup to a CU has four stages, more have two.
// (offsets of a request are 32 bits: 128 rows of K)
int gemm_mid_launch(const int8_t* a, const void* w, const __half* ws, const __half* as, void* out, int rows, int n, int k, int stride, bool out_f32, int parts,
                    int* partials, hipStream_t stream) {
    static DeviceOnce opted_in;  // dynamic LDS above 64 KiB needs an opt-in per kernel and device
    const int ready = opted_in.run([] {
        return hip_check(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_mid_kernel<4>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)(4 * kStage)),
                         "hipFuncSetAttribute");
    });
    if (ready != ORX_OK) return ready;
    MidParams p = {};
    p.a = a, p.w = static_cast<const int8_t*>(w), p.ws = ws, p.as = as, p.out = out, p.partials = partials;
    p.n = n, p.k = k, p.stride = stride, p.m = rows, p.out_f32 = out_f32, p.parts = parts;
    p.tiles_m = (rows + kTile - 1) / kTile, p.tiles_n = (n + kTile - 1) / kTile;
    const int tiles = p.tiles_m * p.tiles_n, workgroups = tiles * parts;
    if (workgroups <= device_compute_units())
        ORX_LAUNCH(gemm_mid_kernel<4>, dim3(workgroups), dim3(kThreads), 4 * kStage, stream, p);
    else
        ORX_LAUNCH(gemm_mid_kernel<2>, dim3(workgroups), dim3(kThreads), 2 * kStage, stream, p);
    const int code = hip_check(hipGetLastError(), "launch projection (128 x 128 tiles)");
    if (code != ORX_OK || parts == 1) return code;
    ORX_LAUNCH(mid_finish_kernel, dim3(4 * tiles), dim3(kThreads), 0, stream, p);
    return hip_check(hipGetLastError(), "launch projection (sum of a tile's parts)");
}

}  // namespace orx
