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
//  * Codes go from memory into registers, 16 bytes per lane, block of channels and chunk, and through the paired tables into
//    the weight operands; the lookups of a block for the next step of 64 run under the multiplies of that block, and are
//    combined under those of the block after it.
//  What bounds it (7168 x 5120 codes of 200 rows, 28.5 us): latency, with one wave to a SIMD and the LDS at about half its rate;
//  without the token requests, the lookups or the stores it takes 3.6, 4.6 or 2.3 us less.  int8, 24 rows of 5120 x 17408: the stream, 4.6 TB/s.
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

template <int CODEC>
constexpr uint32_t runs_tables() { return CODEC == kRunsQ4 ? kPairedTableBytes : 0; }
template <int CODEC, int TB, int CB>
constexpr uint32_t runs_stage() { return 2048u * (TB + (CODEC == kRunsW8 ? CB : 0)); }
template <int CODEC, int TB, int CB, int WAVES, int D>
constexpr uint32_t runs_lds() {
    const uint32_t rings = runs_stage<CODEC, TB, CB>() * WAVES * D, sums = (CB * 16 * (TB * 16 + 4) + 128 + CB * 16) * 4;  // sums and scales follow the rings
    return runs_tables<CODEC>() + (rings > sums ? rings : sums);
}

// fragments FIRST .. FIRST + COUNT - 1 of 16 rows each
template <int COUNT, int FIRST>
__device__ __forceinline__ void read_fragments(v4i* to, uint32_t address) {
    lds_read_16<FIRST * 2048>(to[0], address);
    if constexpr (COUNT > 1) read_fragments<COUNT - 1, FIRST + 1>(to + 1, address);
}

template <int CODEC, int TB, int CB, int WAVES, int D>
__global__ __launch_bounds__(WAVES * 64) void runs_kernel(RunsParams p) {
    constexpr int kThreads = WAVES * 64;
    constexpr int kPitch = TB * 16 + 4;  // 4 (mod 16): the 64 lanes of an accumulator register hit 64 banks
    constexpr uint32_t kStage = runs_stage<CODEC, TB, CB>();
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
    uint32_t scale_bits = reinterpret_cast<const unsigned short*>(tid < 128 ? p.as + first_row : p.ws + first_channel)
        [tid < 128 ? min(tid, rows - 1) : min(tid - 128, channels - 1)];
    uint32_t selector = 0;
    if constexpr (CODEC == kRunsQ4)
        if (tid < 256) selector = p.book[tid];

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
    const int left_out = CODEC == kRunsW8 ? (token_rows.last_request < 2 * TB - 1) + (weight_rows.last_request < 2 * CB - 1) : 0;
    uint8_t* const ring = lds + runs_tables<CODEC>() + (uint32_t)wave * (D * kStage);
    const int8_t* const a_base = uniform_pointer(p.a + (int64_t)first_row * p.k);
    const uint8_t* const w_base = uniform_pointer(p.w + (int64_t)first_channel * p.row_stride);
    auto request_rows = [&](const void* base, const Rows& r, auto blocks_tag, uint8_t* to) ORX_INLINE {
        constexpr int BLOCKS = decltype(blocks_tag)::value;
#pragma unroll
        for (int i = 0; i < 2 * BLOCKS; ++i) {
            if (CODEC == kRunsW8 && i == 2 * BLOCKS - 1 && r.last_request < i) break;  // uniform
            const bool tail = i >= r.last_request;  // uniform
            uint32_t offset = tail ? r.last : i & 1 ? r.odd : r.even;
            asm volatile("" : "+v"(offset));  // 32 bits beside a uniform base
            const uint64_t first = (uint64_t)(uint32_t)(8 * min(i, r.last_request)) * (uint32_t)p.k;
            direct_load_16(static_cast<const uint8_t*>(base) + first + (uint64_t)offset, to + i * 1024);
        }
    };
    uint32_t code_offset[CB];
#pragma unroll
    for (int j = 0; j < CB; ++j)
        code_offset[j] = (uint32_t)min(16 * j + column, channels - 1) * p.row_stride + (uint32_t)(quarter >> 1) * p.half_stride + (uint32_t)(quarter & 1) * 16;
    v4u codes[CODEC == kRunsQ4 ? D : 1][CB];
    auto request = [&](int index, auto slot_tag) ORX_INLINE {  // chunk begin + index of this wave's slice
        constexpr int SLOT = decltype(slot_tag)::value;
        const int chunk = min(begin + index, last);
        const uint8_t* const weights = w_base + (uint64_t)chunk * p.chunk_stride;
        if constexpr (CODEC == kRunsQ4) {
#pragma unroll
            for (int j = 0; j < CB; ++j)
                load_16(codes[SLOT][j], code_offset[j], weights);
        } else {
            request_rows(weights, weight_rows, std::integral_constant<int, CB>{}, ring + SLOT * kStage + TB * 2048);
        }
        request_rows(a_base + (uint64_t)chunk * 128, token_rows, std::integral_constant<int, TB>{}, ring + SLOT * kStage);
    };
    auto name_codes = [&]() ORX_INLINE {
        if constexpr (CODEC == kRunsQ4) {
#pragma unroll
            for (int d = 0; d < D; ++d)
#pragma unroll
                for (int j = 0; j < CB; ++j) asm volatile("" : "+v"(codes[d][j]));
        }
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
        name_codes();
    };
    request(0, std::integral_constant<int, 0>{});
    request(1, std::integral_constant<int, 1>{});
    if constexpr (D > 2) request(2, std::integral_constant<int, 2>{});
    if constexpr (D > 3) request(3, std::integral_constant<int, 3>{});

    if constexpr (CODEC == kRunsQ4) {
        if (tid < 256) {
            write_paired_entry(lds, tid, false, byte_basis_biased(selector, 0));
            write_paired_entry(lds, tid, true, byte_mask_biased((uint32_t)tid, 0));
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }

    v4i acc[TB][CB];
#pragma unroll
    for (int i = 0; i < TB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) acc[i][j] = v4i{0, 0, 0, 0};
    const uint32_t lds_base = lds_address_of(lds);
    const uint32_t frag = lds_address_of(ring) + (uint32_t)column * 128 + (uint32_t)((quarter ^ swizzle(column)) * 16);
    auto read_fragment = [&](v4i& to, auto block_tag, uint32_t address) ORX_INLINE { lds_read_16<decltype(block_tag)::value * 2048>(to, address); };

    if constexpr (CODEC == kRunsQ4) {
        const PairedLookup tables(lds_base, lane);
        // Two sets each: the fragments of a step and of the next, the lookups of a block and of the block before it.
        constexpr int SETS = CB > 1 ? 2 : 1;
        v4i token[SETS][TB], weight[CB];
        v2u looked[SETS][2][2][2];  // of two codes: stages, basis and mask entries
        auto lookup = [&](auto set_tag, const v4u& words, auto step_tag) ORX_INLINE {
            constexpr int SET = decltype(set_tag)::value % SETS, STEP = decltype(step_tag)::value;
            tables.read<0>(looked[SET][0][0], words[2 * STEP]);
            tables.read<1>(looked[SET][0][1], words[2 * STEP]);
            tables.read<0>(looked[SET][1][0], words[2 * STEP + 1]);
            tables.read<1>(looked[SET][1][1], words[2 * STEP + 1]);
        };
        auto combine = [&](auto set_tag, v4i& w, int word) ORX_INLINE {  // w + 128 = 8 (v0 + 8) + 2 (v1 + 8) + 53 in every byte
            constexpr int SET = decltype(set_tag)::value % SETS;
            const int c = word >> 1, e = word & 1;
            const uint32_t coarse = looked[SET][c][0][0][e] ^ looked[SET][c][0][1][e], fine = looked[SET][c][1][0][e] ^ looked[SET][c][1][1][e];
            w[word] = (int)(((((coarse << 2) + fine) << 1) + 0x35353535u) ^ 0x80808080u);
        };
        auto wait_reads = [&]() ORX_INLINE {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int set = 0; set < SETS; ++set) {
#pragma unroll
                for (int c = 0; c < 2; ++c)
                    asm volatile("" : "+v"(looked[set][c][0][0]), "+v"(looked[set][c][0][1]), "+v"(looked[set][c][1][0]), "+v"(looked[set][c][1][1]));
#pragma unroll
                for (int i = 0; i < TB; ++i) asm volatile("" : "+v"(token[set][i]));
            }
        };
        auto read_token = [&](auto set_tag, auto i_tag, uint32_t address) ORX_INLINE {
            read_fragment(token[decltype(set_tag)::value % SETS][decltype(i_tag)::value], i_tag, address);
        };
        auto for_tokens = [&](auto body) ORX_INLINE {
            body(std::integral_constant<int, 0>{});
            if constexpr (TB > 1) body(std::integral_constant<int, 1>{});
            if constexpr (TB > 2) body(std::integral_constant<int, 2>{});
            if constexpr (TB > 3) body(std::integral_constant<int, 3>{});
            if constexpr (TB > 4) body(std::integral_constant<int, 4>{});
            if constexpr (TB > 5) body(std::integral_constant<int, 5>{});
            if constexpr (TB > 6) body(std::integral_constant<int, 6>{});
            if constexpr (TB > 7) body(std::integral_constant<int, 7>{});
        };
        auto for_blocks = [&](auto body) ORX_INLINE {
            body(std::integral_constant<int, 0>{});
            if constexpr (CB > 1) body(std::integral_constant<int, 1>{});
            if constexpr (CB > 2) body(std::integral_constant<int, 2>{});
            if constexpr (CB > 3) body(std::integral_constant<int, 3>{});
            if constexpr (CB > 4) body(std::integral_constant<int, 4>{});
        };
        // The multiplies of a step of 64 (HALF: which of the chunk), a block of channels at a time.  Under a block's multiplies:
        // the lookups of its next weights go out, the lookups of the block before it (a whole block old, so that nothing
        // waits for them) are combined, and all blocks but the last ask for their share of the next fragments (so those
        // have returned when the step ends).  With one wave to a SIMD nothing else would fill these waits.
        auto step = [&](auto half_tag, uint32_t next_fragments, const v4u(&next_codes)[CB], auto next_step_tag) ORX_INLINE {
            constexpr int HALF = decltype(half_tag)::value;
            for_blocks([&](auto j_tag) ORX_INLINE {
                constexpr int j = decltype(j_tag)::value, before = (j + CB - 1) % CB;
                std::integral_constant<int, HALF * CB + j> lookups;            // set parity of this block's lookups
                std::integral_constant<int, HALF * CB + j + 2 * CB - 1> held;  // and of the block's before it
                std::integral_constant<int, HALF + 1> next;
                if constexpr (CB > 1) wait_reads();
                for_tokens([&](auto i_tag) ORX_INLINE {
                    constexpr int i = decltype(i_tag)::value;
                    acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(weight[j], token[HALF % SETS][i], acc[i][j], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (i == 0) lookup(lookups, next_codes[j], next_step_tag);
                    if constexpr (CB == 1 || (j < CB - 1 && i % (CB - 1) == j)) read_token(next, i_tag, next_fragments);
                    if constexpr (CB > 1) {
#pragma unroll
                        for (int word = 0; word < 4; ++word)
                            if (word * TB / 4 == i) combine(held, weight[before], word);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
                if constexpr (CB == 1) {
                    wait_reads();
#pragma unroll
                    for (int word = 0; word < 4; ++word) combine(lookups, weight[0], word);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        std::integral_constant<int, 0> zero;
        std::integral_constant<int, 1> one;
        if (count > 0) {
            wait_requests(std::integral_constant<int, D - 1>{});
            for_tokens([&](auto i_tag) ORX_INLINE { read_token(zero, i_tag, frag); });
            for_blocks([&](auto j_tag) ORX_INLINE {  // (the last block's lookups are combined under the first multiplies)
                constexpr int j = decltype(j_tag)::value;
                std::integral_constant<int, CB + j> set;
                lookup(set, codes[0][j], zero);
                if constexpr (j < CB - 1 || CB == 1) {
                    wait_reads();
#pragma unroll
                    for (int word = 0; word < 4; ++word) combine(set, weight[j], word);
                }
            });
            auto chunk_step = [&](int t, auto slot_tag) ORX_INLINE {
                constexpr int SLOT = decltype(slot_tag)::value, NEXT = (SLOT + 1) % D;
                step(zero, (frag + SLOT * kStage) ^ 64u, codes[SLOT], one);
                wait_requests(std::integral_constant<int, D - 2>{});  // chunk t + 1 is here, and nobody reads chunk t any more
                request(t + D, slot_tag);
                __builtin_amdgcn_sched_barrier(0);
                step(one, frag + NEXT * kStage, codes[NEXT], zero);
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
            wait_reads();
        }
    } else {
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
    }
    // the requests behind the slice (repeats of its last chunk) have landed before their registers and slots are reused
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    name_codes();
    asm volatile("s_barrier" ::: "memory");

    // ---- the slices are added where the rings were: wave 0 stores, the others add ----
    // accumulator register r of a lane: channel 4 quarter + r of the block, token `column`
    int* const sums = reinterpret_cast<int*>(lds + runs_tables<CODEC>());
    float* const token_scales = reinterpret_cast<float*>(sums + CB * 16 * kPitch);
    float* const channel_scales = token_scales + 128;
    asm volatile("" : "+v"(scale_bits));  // converted here, not where it was read
    if (tid < 128 + CB * 16) token_scales[tid] = __half2float(__ushort_as_half((unsigned short)scale_bits));
    int own = threadIdx.x & 63;
    asm volatile("" : "+v"(own));
    int* const mine = sums + 4 * (own >> 4) * kPitch + (own & 15);
    if (wave == 0) {
#pragma unroll
        for (int i = 0; i < TB; ++i)
#pragma unroll
            for (int j = 0; j < CB; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) mine[(16 * j + r) * kPitch + 16 * i] = acc[i][j][r];
    }
    __syncthreads();
    if (wave != 0) {
#pragma unroll
        for (int i = 0; i < TB; ++i)
#pragma unroll
            for (int j = 0; j < CB; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) atomicAdd(mine + (16 * j + r) * kPitch + 16 * i, acc[i][j][r]);
    }
    __syncthreads();
    // four channels of a row per thread and store
    const int element = p.out_f32 ? 4 : 2;
    for (int e = tid; e < rows * CB * 4; e += kThreads) {
        const int local = e / (CB * 4), channel = e % (CB * 4) * 4;
        if (channel >= channels) continue;
        const float token_scale = token_scales[local];
        const float4 ws = *reinterpret_cast<const float4*>(channel_scales + channel);
        const int* cell = sums + channel * kPitch + local;
        const float value[4] = {rescale(cell[0], ws.x, token_scale), rescale(cell[kPitch], ws.y, token_scale),
                                rescale(cell[2 * kPitch], ws.z, token_scale), rescale(cell[3 * kPitch], ws.w, token_scale)};
        char* const dst = static_cast<char*>(p.out) + ((int64_t)(first_row + local) * p.stride + first_channel + channel) * element;
        const bool whole = channel + 3 < channels && (reinterpret_cast<uintptr_t>(dst) & (uintptr_t)(4 * element - 1)) == 0;
        if (p.out_f32) {
            if (whole) {
                *reinterpret_cast<float4*>(dst) = make_float4(value[0], value[1], value[2], value[3]);
            } else {
                for (int i = 0; i < 4; ++i)
                    if (channel + i < channels) reinterpret_cast<float*>(dst)[i] = value[i];
            }
        } else {
            __half h[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) h[i] = __float2half_rn(value[i]);
            if (whole) {
                *reinterpret_cast<uint2*>(dst) = make_uint2((uint32_t)__half_as_ushort(h[0]) | (uint32_t)__half_as_ushort(h[1]) << 16,
                                                            (uint32_t)__half_as_ushort(h[2]) | (uint32_t)__half_as_ushort(h[3]) << 16);
            } else {
                for (int i = 0; i < 4; ++i)
                    if (channel + i < channels) reinterpret_cast<__half*>(dst)[i] = h[i];
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
    s.runs = (n + s.run - 1) / s.run;
    for (int i = forms.count - 1; i >= 0; --i)
        if (16 * forms.first[i].cb >= s.run) s.form = &forms.first[i];
    return s;
}

}  // namespace

bool runs_eligible(int codec, int rows, int n, int k) {
    return rows >= 1 && rows <= kRunsMaxRows && k % 128 == 0 && (int64_t)n * k < (1ll << 31) && (int64_t)rows * k < (1ll << 31) &&
           runs_shape(codec, rows, n).form != nullptr;
}

// rounds of the CUs that the launch takes, and the rows of its tiles
int runs_rounds(int codec, int rows, int n, int* tile_rows) {
    const RunsShape s = runs_shape(codec, rows, n);
    const int cus = device_compute_units();
    *tile_rows = s.tile_rows;
    return (s.runs * s.row_tiles + cus - 1) / cus;
}

void runs_geometry(int codec, int rows, int n, Geometry* g) {
    const RunsShape s = runs_shape(codec, rows, n);
    g->grid[0] = (uint32_t)s.runs, g->grid[1] = (uint32_t)s.row_tiles, g->grid[2] = 1;
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
    ORX_LAUNCH(kernel, dim3(s.runs, s.row_tiles), dim3(s.form->waves * 64), kRunsLds, stream, p);
    return hip_check(hipGetLastError(), "launch projection (channel runs)");
}

}  // namespace orx
