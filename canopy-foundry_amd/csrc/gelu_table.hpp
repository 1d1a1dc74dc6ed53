// bf16(gelu(x)) of bf16 values by table.  The result is a function of x's 16 bits; with erff it costs about 40 vector instructions, a look-up
// five and an LDS read.  The table holds every x with 2^-18 <= |x| < 16, 5632 entries in 11 KiB, which a workgroup of 1024 builds with
// five or six evaluations per lane (all 65536 bit patterns took 64 and 128 KiB); what lies outside (zeros, tiny, huge
// values) has a closed form, infinities and NaN are evaluated directly.  The same bits every way: the table is built with gelu_fwd.
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
// A pair of which a half may lie outside the table, `found` being what the table gave: below it erff(x / sqrt 2) is too small to reach the
// bf16 result, x / 2; from 16 on erff is 1 or -1, and the result x or -0.  Infinities and NaN: `special`.
__device__ __forceinline__ uint32_t gelu_edge2(uint32_t pair, uint32_t found, bool& special) {
    const uint32_t half = pack_bf16x2_hw(0.5f * bf16_lo(pair), 0.5f * bf16_hi(pair));
    auto one = [&](uint32_t x, uint32_t f, uint32_t h) {
        const uint32_t m = x & 0x7fffu;
        special |= m >= 0x7f80u;
        return m < kGeluLo ? h : m < kGeluLo + kGeluSpan ? f : (x & 0x8000u) ? 0x8000u : x;
    };
    return one(pair & 0xffffu, found & 0xffffu, half & 0xffffu) | (one(pair >> 16, found >> 16, half >> 16) << 16);
}
// Four pairs.  A wavefront with one value outside takes the second half; evaluating its values with gelu_fwd there made data with a zero here
// and there the slowest: 98304 x 1408 with per-row scales, half of the values zero, 221 us, now 125 (normal values 84, one in a thousand
// 40.0 109 and 94).
__device__ __forceinline__ uint4 gelu_look8(const uint16_t* table, const uint4& v) {
    u16x2 worst = {0, 0};
    const uint4 g = make_uint4(gelu_look2(table, v.x, worst), gelu_look2(table, v.y, worst), gelu_look2(table, v.z, worst), gelu_look2(table, v.w, worst));
    if (!gelu_outside(worst)) return g;
    bool special = false;
    const uint4 o = make_uint4(gelu_edge2(v.x, g.x, special), gelu_edge2(v.y, g.y, special), gelu_edge2(v.z, g.z, special), gelu_edge2(v.w, g.w, special));
    if (!special) return o;
    return make_uint4(gelu2(v.x), gelu2(v.y), gelu2(v.z), gelu2(v.w));
}

}  // namespace cf
