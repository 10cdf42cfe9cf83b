// LDS and memory accesses from asm statements, waited for by hand, for the kernels whose token rows arrive by direct-to-LDS
// loads: the compiler waits for every such load in flight in front of an LDS read it can see.  A register named here as a
// result holds nothing until the wait that covers it: name it in that wait, and keep it named until then.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace orx {
namespace lds_asm {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

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
__device__ __forceinline__ void load_16(v4u& value, uint32_t lane_offset, const void* uniform_base) {
    asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(value) : "v"(lane_offset), "s"(uniform_base) : "memory");
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
