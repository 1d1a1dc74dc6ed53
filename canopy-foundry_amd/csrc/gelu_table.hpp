// bf16(gelu(x)) of bf16 values by table.  The result is a function of x's 16 bits; with erff it costs about 40 vector instructions, a look-up
// five and an LDS read.  The table holds every x with 2^-18 <= |x| < 16, 5632 entries in 11 KiB, which a workgroup of 1024 builds with
// five or six evaluations per lane (all 65536 bit patterns took 64 and 128 KiB); what lies outside (zeros, tiny, huge, non-finite
// values) is evaluated directly.  The same bits either way: the table is built with gelu_fwd.
#pragma once
#include "common.hpp"

namespace cf {

constexpr uint32_t kGeluLo = 0x3680u, kGeluSpan = 22u * 128u;       // bits of 2^-18; magnitudes in the table
constexpr int kGeluEntries = 2 * kGeluSpan;                         // entry 2 * magnitude + sign

// lane `lane` of `lanes`
__device__ __forceinline__ void gelu_table_build(uint16_t* table, uint32_t lane, uint32_t lanes) {
    for (uint32_t i = lane; i < kGeluEntries; i += lanes)
        table[i] = f32_to_bf16(gelu_fwd(bf16_to_f32(static_cast<uint16_t>((i >> 1) + kGeluLo + ((i & 1u) << 15)))));
}
// Both halves of a pair.  worst keeps the largest index met, per half: kGeluEntries or more means that some value lay outside and
// that what was returned for it is of no use.
__device__ __forceinline__ uint32_t gelu_look2(const uint16_t* table, uint32_t pair, u16x2& worst) {
    const u16x2 b = __builtin_bit_cast(u16x2, pair);
    const u16x2 lo = {static_cast<unsigned short>(2 * kGeluLo), static_cast<unsigned short>(2 * kGeluLo)};
    const u16x2 last = {static_cast<unsigned short>(kGeluEntries - 1), static_cast<unsigned short>(kGeluEntries - 1)};
    const u16x2 one = {1, 1}, fifteen = {15, 15};
    const u16x2 at = ((b << one) | (b >> fifteen)) - lo;            // sign to the lowest bit; below the table: wraps far beyond it
    worst = __builtin_elementwise_max(worst, at);
    const uint32_t i = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(at, last));
    return static_cast<uint32_t>(table[i & 0xffffu]) | (static_cast<uint32_t>(table[i >> 16]) << 16);
}
__device__ __forceinline__ bool gelu_outside(const u16x2& worst) { return max(worst.x, worst.y) >= kGeluEntries; }
// Four pairs, evaluated directly where one lies outside
__device__ __forceinline__ uint4 gelu_look8(const uint16_t* table, const uint4& v) {
    u16x2 worst = {0, 0};
    const uint4 g = make_uint4(gelu_look2(table, v.x, worst), gelu_look2(table, v.y, worst), gelu_look2(table, v.z, worst), gelu_look2(table, v.w, worst));
    if (!gelu_outside(worst)) return g;
    return make_uint4(gelu2(v.x), gelu2(v.y), gelu2(v.z), gelu2(v.w));
}

}  // namespace cf
