// LDS and memory accesses from asm statements, waited for by hand, for the kernels whose token rows arrive by direct-to-LDS
// loads: the compiler waits for every such load in flight in front of an LDS read it can see.  A register named here as a
// result holds nothing until the wait that covers it: name it in that wait, and keep it named until then.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace orx {
namespace lds_asm {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

// body(0) .. body(COUNT - 1), each with its number as a constant
template <int COUNT>
struct Each {
    template <typename Body>
    static __device__ __forceinline__ void run(Body body) {
        if constexpr (COUNT > 0) {
            Each<COUNT - 1>::run(body);
            body(std::integral_constant<int, COUNT - 1>{});
        }
    }
};

// Rows of 128 bytes in LDS: the piece at position p of a row is kept at p ^ swizzle(row), so that the 16 rows of a
// fragment read spread over the banks.
__device__ __forceinline__ int swizzle(int row) { return (row >> 1) & 7; }
__device__ __forceinline__ uint32_t lds_address_of(const void* pointer) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)pointer;
}
__device__ __forceinline__ void direct_load_16(const void* global, void* lds_wave_base) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)global,
                                     (__attribute__((address_space(3))) void*)lds_wave_base, 16, 0, 0);
}
// The same from an asm statement: a uniform base and 32 bits per lane, and no wait in front of the LDS accesses that the compiler
// can see.  OFFSET counts on both sides.  The statements that set m0 name it: else the compiler holds what its last direct_load_16 left there for unchanged.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // (m0 is reserved: it holds nothing of the compiler's from one statement to the next)
template <int OFFSET>
__device__ __forceinline__ void request_16(uint32_t lane_offset, const void* uniform_base, uint32_t lds_wave_base) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 offset:%3" ::"v"(lane_offset), "s"(uniform_base), "s"(lds_wave_base), "n"(OFFSET)
                 : "memory", "m0");
}
// COUNT (1, 2 or 4) requests of 1 KiB, one behind the other in LDS, if index < count.  Else none, by a branch inside the statement; COUNTED: requests by no
// lane, which bring nothing and count all the same, where requests that follow are waited for by number.
#define ORX_BELOW_OR_SKIPPED(INDEX, COUNT, BODY) "s_cmp_lt_i32 " INDEX ", " COUNT "\n\ts_cbranch_scc0 .Lskipped%=\n\t" BODY ".Lskipped%=:"
#define ORX_BELOW_OR_EMPTY(INDEX, COUNT, ALL, BODY) \
    "s_mov_b64 " ALL ", exec\n\ts_cmp_lt_i32 " INDEX ", " COUNT "\n\ts_cselect_b64 exec, exec, 0\n\t" BODY "s_mov_b64 exec, " ALL
template <int COUNT, bool COUNTED>
__device__ __forceinline__ void request_rows_16(const uint32_t (&lane_offset)[COUNT], const void* uniform_base, uint32_t lds_wave_base, int index, int count) {
    static_assert(COUNT == 1 || COUNT == 2 || COUNT == 4, "one, two or four requests to a statement");
    uint64_t all;
#define ORX_REQUEST_4 \
    "s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %5, %1\n\tglobal_load_lds_dwordx4 %6, %1 offset:1024\n\t" \
    "global_load_lds_dwordx4 %7, %1 offset:2048\n\tglobal_load_lds_dwordx4 %8, %1 offset:3072\n\t"
#define ORX_REQUEST_2 "s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %5, %1\n\tglobal_load_lds_dwordx4 %6, %1 offset:1024\n\t"
#define ORX_REQUEST_1 "s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %5, %1\n\t"
#define ORX_REQUEST(TEXT, ...)                                                                                              \
    do {                                                                                                                    \
        if constexpr (COUNTED)                                                                                              \
            asm volatile(ORX_BELOW_OR_EMPTY("%3", "%4", "%0", TEXT)                                                         \
                         : "=&s"(all)                                                                                       \
                         : "s"(uniform_base), "s"(lds_wave_base), "s"(index), "s"(count), __VA_ARGS__                       \
                         : "memory", "m0", "scc");                                                                          \
        else                                                                                                                \
            asm volatile(ORX_BELOW_OR_SKIPPED("%3", "%4", TEXT)                                                             \
                         : "=&s"(all)                                                                                       \
                         : "s"(uniform_base), "s"(lds_wave_base), "s"(index), "s"(count), __VA_ARGS__                       \
                         : "memory", "m0", "scc");                                                                          \
    } while (0)
    if constexpr (COUNT == 1)
        ORX_REQUEST(ORX_REQUEST_1, "v"(lane_offset[0]));
    else if constexpr (COUNT == 2)
        ORX_REQUEST(ORX_REQUEST_2, "v"(lane_offset[0]), "v"(lane_offset[1]));
    else
        ORX_REQUEST(ORX_REQUEST_4, "v"(lane_offset[0]), "v"(lane_offset[1]), "v"(lane_offset[2]), "v"(lane_offset[3]));
#undef ORX_REQUEST
#undef ORX_REQUEST_1
#undef ORX_REQUEST_2
#undef ORX_REQUEST_4
}
#pragma clang diagnostic pop
// A request OFFSET behind the last request_16, by the m0 that this one left: for a kernel whose only writes of m0 are request_16's, so for none with a
// direct_load_16 or another builtin that needs m0 (the check of the built kernels in tests/test_codegen.py counts them).
template <int OFFSET>
__device__ __forceinline__ void request_16_behind(uint32_t lane_offset, const void* uniform_base) {
    asm volatile("global_load_lds_dwordx4 %0, %1 offset:%2" ::"v"(lane_offset), "s"(uniform_base), "n"(OFFSET) : "memory");
}
__device__ __forceinline__ void lds_write_16(uint32_t address, v4u value) {
    asm volatile("ds_write_b128 %0, %1" ::"v"(address), "v"(value) : "memory");
}
template <int OFFSET>
__device__ __forceinline__ void lds_read_16(v4i& value, uint32_t address) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(value) : "v"(address), "n"(OFFSET));
}
template <int OFFSET>
__device__ __forceinline__ void lds_read_8(v2u& value, uint32_t address) {
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(value) : "v"(address), "n"(OFFSET));
}
template <int OFFSET>
__device__ __forceinline__ void load_8(v2u& value, uint32_t lane_offset, const void* uniform_base) {
    asm volatile("global_load_dwordx2 %0, %1, %2 offset:%3"
                 : "=v"(value)
                 : "v"(lane_offset), "s"(uniform_base), "n"(OFFSET)
                 : "memory");
}
// Four times 8 bytes, at both lane offsets and 512 behind them, where index < count as above; else the registers keep what they have.
template <bool COUNTED>
__device__ __forceinline__ void load_8_of_four(v2u (&value)[4], uint32_t lane_offset, uint32_t other_offset, const void* uniform_base, int index, int count) {
    uint64_t all;
#define ORX_LOADS                                                                                                      \
    "global_load_dwordx2 %0, %5, %7\n\tglobal_load_dwordx2 %1, %5, %7 offset:512\n\tglobal_load_dwordx2 %2, %6, %7\n\t" \
    "global_load_dwordx2 %3, %6, %7 offset:512\n\t"
    if constexpr (COUNTED)
        asm volatile(ORX_BELOW_OR_EMPTY("%8", "%9", "%4", ORX_LOADS)
                     : "+v"(value[0]), "+v"(value[1]), "+v"(value[2]), "+v"(value[3]), "=&s"(all)
                     : "v"(lane_offset), "v"(other_offset), "s"(uniform_base), "s"(index), "s"(count)
                     : "memory", "scc");
    else
        asm volatile(ORX_BELOW_OR_SKIPPED("%8", "%9", ORX_LOADS)
                     : "+v"(value[0]), "+v"(value[1]), "+v"(value[2]), "+v"(value[3]), "=&s"(all)
                     : "v"(lane_offset), "v"(other_offset), "s"(uniform_base), "s"(index), "s"(count)
                     : "memory", "scc");
#undef ORX_LOADS
}
// The same of two, at both lane offsets.
template <bool COUNTED>
__device__ __forceinline__ void load_8_of_two(v2u (&value)[2], uint32_t lane_offset, uint32_t other_offset, const void* uniform_base, int index, int count) {
    uint64_t all;
#define ORX_LOADS "global_load_dwordx2 %0, %3, %5\n\tglobal_load_dwordx2 %1, %4, %5\n\t"
    if constexpr (COUNTED)
        asm volatile(ORX_BELOW_OR_EMPTY("%6", "%7", "%2", ORX_LOADS)
                     : "+v"(value[0]), "+v"(value[1]), "=&s"(all)
                     : "v"(lane_offset), "v"(other_offset), "s"(uniform_base), "s"(index), "s"(count)
                     : "memory", "scc");
    else
        asm volatile(ORX_BELOW_OR_SKIPPED("%6", "%7", ORX_LOADS)
                     : "+v"(value[0]), "+v"(value[1]), "=&s"(all)
                     : "v"(lane_offset), "v"(other_offset), "s"(uniform_base), "s"(index), "s"(count)
                     : "memory", "scc");
#undef ORX_LOADS
}
#undef ORX_BELOW_OR_EMPTY
#undef ORX_BELOW_OR_SKIPPED
__device__ __forceinline__ void load_4(uint32_t& value, uint32_t lane_offset, const void* uniform_base) {
    asm volatile("global_load_dword %0, %1, %2" : "=v"(value) : "v"(lane_offset), "s"(uniform_base) : "memory");
}
__device__ __forceinline__ void load_16(v4u& value, uint32_t lane_offset, const void* uniform_base) {
    asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(value) : "v"(lane_offset), "s"(uniform_base) : "memory");
}
template <typename T>
__device__ __forceinline__ void keep(T& value) { asm volatile("" : "+v"(value)); }
// a register of its own, whatever it holds
template <typename T>
__device__ __forceinline__ void anything(T& value) { asm volatile("" : "=v"(value)); }
// In and out in one register: left to itself the compiler moves sums about between unrolled steps, a tenth of a loop's
// instructions.  What it would have inserted is on the caller: two instructions between the last write of an operand and the multiply,
// and a pause (s_nop 15) in front of the first reading of a sum.
// ACC: the sum in accumulation registers (the kernel then has half of its registers of either kind).
template <bool ACC>
__device__ __forceinline__ void multiply_in_place(v4i& sum, const v4i& weight, const v4i& token) {
    if constexpr (ACC)
        asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+a"(sum) : "v"(weight), "v"(token));
    else
        asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+v"(sum) : "v"(weight), "v"(token));
}
template <bool ACC>
__device__ __forceinline__ void keep_sum(v4i& sum) {
    if constexpr (ACC)
        asm volatile("" : "+a"(sum));
    else
        asm volatile("" : "+v"(sum));
}
template <typename T>
__device__ __forceinline__ T* uniform_pointer(T* pointer) {
    const uint64_t bits = reinterpret_cast<uint64_t>(pointer);
    const uint32_t low = __builtin_amdgcn_readfirstlane((uint32_t)bits), high = __builtin_amdgcn_readfirstlane((uint32_t)(bits >> 32));
    return reinterpret_cast<T*>((uint64_t)high << 32 | low);
}

// Lookups in two tables that lie side by side, entry i of both in bytes 128 i: eight copies of the first table's entry, then
// eight of the second's.  Of 16 neighbouring lanes eight read one table and eight the other, each its own copy, so no two
// meet in a bank; the next lookup goes the other way round.  (Their results are XORed, so the order does not matter.)
struct PairedLookup {
    uint32_t first_table, second_table, first_bit, second_bit;  // bit: of the code byte that indexes the table
    __device__ __forceinline__ PairedLookup(uint32_t base, int lane) {
        const uint32_t other = (uint32_t)(lane >> 3) & 1;
        first_table = base + (uint32_t)(lane & 7) * 8 + other * 64, second_table = first_table ^ 64u;
        first_bit = 8 - 8 * other, second_bit = 8 - first_bit;
    }
    // both entries of the code in the low (HALF 0) or the high half of a word: bits 8-15 index the first table, 0-7 the second
    template <int HALF>
    __device__ __forceinline__ void read(v2u (&entry)[2], uint32_t word) const {
        lds_read_8<0>(entry[0], (__builtin_amdgcn_ubfe(word, first_bit + 16 * HALF, 8) << 7) + first_table);
        lds_read_8<0>(entry[1], (__builtin_amdgcn_ubfe(word, second_bit + 16 * HALF, 8) << 7) + second_table);
    }
};
constexpr uint32_t kPairedTableBytes = 256 * 128;
// The same in entries of 256 bytes, 16 copies of either table: of 32 neighbouring lanes 16 read one table and 16 the other.
// Byte 0 of an address is the lane's column, byte 1 a byte of the code: one v_perm_b32 of (code, columns) and a selector.
struct WidePairedLookup {
    uint32_t columns, first_low, second_low, first_high, second_high;
    __device__ __forceinline__ explicit WidePairedLookup(int lane) {
        const uint32_t copy = (uint32_t)(lane & 15) * 8, other = (uint32_t)(lane >> 4) & 1;
        columns = (copy | other * 128) | (copy | (other ^ 1) * 128) << 8;
        first_low = 0x0C0C0500u - (other << 8), second_low = 0x0C0C0401u + (other << 8);
        first_high = first_low + 0x200u, second_high = second_low + 0x200u;
    }
    __device__ __forceinline__ uint32_t address(uint32_t code, uint32_t selector) const {
        return __builtin_amdgcn_perm(code, columns, selector);
    }
};
// Two-stage codes: four tables (basis and mask of the coarse code, basis and mask of the fine one) share entries of BYTES, 256 or 128, in
// copies of 8 bytes.  Of BYTES / 8 neighbouring lanes a quarter reads each table, each lane its own copy, so no two meet in a bank;
// round r of a code reads table group ^ r: rounds 0 and 1 one stage's pair, rounds 2 and 3 the other's.
// The entries are byte_basis_biased and byte_mask_biased, the coarse ones shifted by 2, so that
// (e0 ^ e1) + (e2 ^ e3) = 4 (v0 + 8) + (v1 + 8) = (w + 75) / 2, between 10 and 65 in every byte: two instructions per four weights, and a
// signed byte as it is.  sum(a w) is then 2 sum(a W) - 75 sum(a).
constexpr int kQuadBias = 75;
template <int BYTES>
constexpr uint32_t kQuadTableBytes = 256 * BYTES;
template <int BYTES>
struct QuadLookup {
    static_assert(BYTES == 256 || BYTES == 128, "eight or four copies");
    uint32_t columns[BYTES == 256 ? 1 : 4], select[4];
    __device__ __forceinline__ explicit QuadLookup(int lane) {
        constexpr uint32_t kCopies = BYTES / 32;
        const uint32_t group = (uint32_t)lane / kCopies & 3, copy = (uint32_t)lane % kCopies * 8;
        if constexpr (BYTES == 256) columns[0] = 0;
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) {
            const uint32_t table = group ^ r, column = table * (BYTES / 4) + copy, byte = table ^ 1;  // of the code, the index of the table
            if constexpr (BYTES == 256)  // byte 0 of an address is the column, byte 1 the index: one v_perm_b32
                columns[0] |= column << (8 * r), select[r] = 0x0C0C0000u | (4 + byte) << 8 | r;
            else
                columns[r] = column, select[r] = 8 * byte;
        }
    }
    template <int ROUND>
    __device__ __forceinline__ void read(v2u& entry, uint32_t code) const {  // the tables lie at LDS address 0
        if constexpr (BYTES == 256)
            lds_read_8<0>(entry, __builtin_amdgcn_perm(code, columns[0], select[ROUND]));
        else
            lds_read_8<0>(entry, (__builtin_amdgcn_ubfe(code, select[ROUND], 8) << 7) + columns[ROUND]);
    }
};
// Every lane of a wave writes its own entry, whole entries apart: the order of the 16-byte slots turns with the entry, so that
// the lanes of a write spread over the banks.
template <int BYTES>
__device__ __forceinline__ void write_quad_entry(int entry, uint2 coarse_basis, uint2 coarse_mask, uint2 fine_basis, uint2 fine_mask) {
    constexpr uint32_t kSlots = BYTES / 16, kEach = kSlots / 4;  // kEach slots of a table in a row
    uint2 value[4] = {coarse_basis, coarse_mask, fine_basis, fine_mask};
    const uint32_t turn = BYTES == 256 ? (uint32_t)entry & 15 : (uint32_t)entry >> 1 & 7;
    auto swap_if = [](bool swap, uint2& a, uint2& b) {
        const uint2 x = swap ? b : a, y = swap ? a : b;
        a = x, b = y;
    };
    swap_if(turn & kEach, value[0], value[1]), swap_if(turn & kEach, value[2], value[3]);
    swap_if(turn & (2 * kEach), value[0], value[2]), swap_if(turn & (2 * kEach), value[1], value[3]);
#pragma unroll
    for (uint32_t i = 0; i < kSlots; ++i) {
        const uint2 v = value[i / kEach];
        lds_write_16((uint32_t)entry * BYTES + (i ^ turn) * 16, v4u{v.x, v.y, v.x, v.y});
    }
}

// One half of a paired entry: SLOTS 16-byte slots of two copies each.  Every lane of a wave writes its own entry, so the slot
// order turns with the entry: in the same order for all, the lanes, whole entries apart, would write to the same banks (the
// 16-wave kernels spent 2 us of every launch on 64 KB of tables that way, 0.3 us now).
template <int SLOTS = 4>
__device__ __forceinline__ void write_paired_entry(uint8_t* tables, int entry, bool second, uint2 value) {
    static_assert(SLOTS == 4 || SLOTS == 8, "an entry is 128 or 256 bytes");
    const uint32_t turn = SLOTS == 8 ? (uint32_t)entry & 7 : (uint32_t)entry >> 1 & 3;
    const uint32_t first = (uint32_t)entry * (32 * SLOTS) + (second ? 16 * SLOTS : 0) + 16 * turn;
#pragma unroll
    for (uint32_t i = 0; i < SLOTS; ++i) *reinterpret_cast<uint4*>(tables + (first ^ 16 * i)) = make_uint4(value.x, value.y, value.x, value.y);
}

}  // namespace lds_asm
}  // namespace orx
