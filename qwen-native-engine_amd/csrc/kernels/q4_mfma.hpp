// q4 weights as operands of the f16 matrix instructions.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace qne {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float float16_t __attribute__((ext_vector_type(16)));

// (v & mask) | 0x64006400 in one instruction: the constants have to sit in registers (`magic` in a
// vector one), which the compiler gives up for a literal each and two instructions.
__device__ __forceinline__ uint32_t and_or(uint32_t v, uint32_t mask, uint32_t magic) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(mask), "v"(magic));
    return r;
}

// The integer r in 0..15 nearest a scale / zero word's zero point, as what nibbles8 subtracts: 1024 + r and
// -64 - r, twice each. A sum of 1024 or more rounds to a whole number in f16, so z + 1024 is the rounding.
struct ZeroInt {
    half2_t high, low;
};
__device__ __forceinline__ ZeroInt zero_int(uint32_t szw) {
    const half2_t k1024 = {(_Float16)1024.0f, (_Float16)1024.0f}, k1039 = {(_Float16)1039.0f, (_Float16)1039.0f};
    const half2_t k960 = {(_Float16)960.0f, (_Float16)960.0f};
    const _Float16 z = __builtin_bit_cast(half2_t, szw).y;
    const half2_t high = __builtin_elementwise_min(__builtin_elementwise_max(half2_t{z, z} + k1024, k1024), k1039);
    return ZeroInt{high, k960 - high};
}

// The 8 nibbles of a q4 word (nibble i at bits 4i: column 8j + i of word j), minus r, as exact
// f16 values, in the order [q0, q4, q1, q5, q2, q6, q3, q7]: 0x6400 | q is the f16 1024 + q, and
// 0x6400 | (q << 4) is 1024 + 16 q, so four and-or, one shift, two packed subtracts and two packed
// fmas (x / 16 - 64 - r) give all eight. The x operand of a q4 GEMM is staged in the same column order.
__device__ __forceinline__ half8_t nibbles8(uint32_t v, const ZeroInt& r) {
    typedef uint32_t u32;
    const u32 v2 = v >> 8, magic = 0x64006400u;
    const u32 t0 = and_or(v, 0x000F000Fu, magic), t1 = and_or(v, 0x00F000F0u, magic);
    const u32 t2 = and_or(v2, 0x000F000Fu, magic), t3 = and_or(v2, 0x00F000F0u, magic);
    const half2_t k16 = {(_Float16)0.0625f, (_Float16)0.0625f};
    const half2_t h0 = __builtin_bit_cast(half2_t, t0) - r.high;
    const half2_t h1 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, t1), k16, r.low);
    const half2_t h2 = __builtin_bit_cast(half2_t, t2) - r.high;
    const half2_t h3 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, t3), k16, r.low);
    return half8_t{h0.x, h0.y, h1.x, h1.y, h2.x, h2.y, h3.x, h3.y};
}
__device__ __forceinline__ half8_t nibbles8(uint32_t v) {
    const half2_t high = {(_Float16)1024.0f, (_Float16)1024.0f}, low = {(_Float16)-64.0f, (_Float16)-64.0f};
    return nibbles8(v, ZeroInt{high, low});
}

}  // namespace qne
