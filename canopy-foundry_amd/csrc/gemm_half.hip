// The persistent FP8 GEMM at half the tile, one workgroup per CU:  C[M,N] = epilogue( (A[M,K] * sa) . (B[N,K] * sb)^T ).
//
// Tile 256 activation rows x 128 weight rows, or 128 x 256 (the SiLU gate: 128 x 128 outputs), four wavefronts 2 x 2.  It is for
// problems whose 256 x 256 tiles fill the last round badly: 2048 rows and 4096 columns are 128 of those, half the CUs.  Smaller
// tiles than this one (128 x 128, in gemm_duo.hip and gemm_direct.hip) need twice the bytes of the 256 x 256 tile per FLOP,
// and a CU takes in about 37 of its nominal 64 bytes a cycle; this one needs one and a half times as many.
//   - A K-tile of 128 bytes is 48 KiB; three LDS stages, filled by buffer_load ... lds three K-tiles ahead.
//   - The scheme of gemm_bf16_duo.hip: a K-tile's operands are in registers before its barrier, so that its stage is free for the
//     copies right behind it; the narrow operand's four 16-row blocks have two register sets, the wide one's eight are refilled
//     one by one behind the four v_mfma_f32_16x16x128_f8f6f4 that use them.
//   - Rows of the operands beyond their last and bytes beyond K are read as zeros: K only has to be a multiple of 16.
//   - C leaves through 2 KiB of LDS per wavefront in whole 128-byte lines.
#include "gemm_common.hpp"

#include <mutex>

namespace cf {
namespace {

constexpr int kThreads = 256;
constexpr int kWide = 256, kNarrow = 128;                      // rows of the two operands' tiles
constexpr int kWideTile = kWide * BK;                          // 32 KiB
constexpr int kStageBytes = kWideTile + kNarrow * BK;          // 48 KiB
constexpr int kRingBytes = 3 * kStageBytes;
constexpr int kStageOut = 2048;                                // per wavefront: what the epilogue turns round at a time
constexpr int kLdsBytes = kRingBytes + 4 * kStageOut;          // 152 KiB
constexpr int kNonTemporal = 2;                                // cache policy of a buffer access
constexpr int kWaitVm0 = 0x0f70, kWaitVm12 = 0x0f7c;           // s_waitcnt vmcnt(n), the other counters left alone
constexpr uint32_t kOutside = 0x80000000u;                     // an offset beyond every operand's descriptor

typedef int s32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float acc_read(float a) {
    float v;
    asm("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(a));
    return v;
}
// One 16 x 16 x 128 MFMA on an accumulator that stays where it is; X5: the activations are E5M2
template <bool X5, bool FIRST>
__device__ __forceinline__ void mfma(v4f& acc, const v8i& w, const v8i& x) {
    v4f c;
    if constexpr (FIRST) {
        if constexpr (X5) asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, 0 blgp:1" : "=a"(c) : "v"(w), "v"(x));
        else asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, 0" : "=a"(c) : "v"(w), "v"(x));
    } else {
        c = acc;
        if constexpr (X5) asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0 blgp:1" : "+a"(c) : "v"(w), "v"(x));
        else asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0" : "+a"(c) : "v"(w), "v"(x));
    }
    acc = c;
}
// 16-byte chunk swizzle of a 128-byte row: the rows 0-7 of one k-group and 8-15 of the next, which one read serves together,
// land in the sixteen 16-byte slots of 256 bytes
__device__ __forceinline__ int swz_row(int row) { return (row ^ ((row >> 3) & 1)) & 7; }

// A5: A is E5M2.  WIDE_M: the tile is 256 activation rows x 128 weight rows, otherwise 128 x 256.
template <bool A5, int EPI, int SCALE, bool WIDE_M>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
void k_gemm_nt_half(const GemmArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    constexpr bool GATE = EPI == EPI_SILU_GATE;
    static_assert(!(GATE && WIDE_M), "a wavefront's 128 weight rows are gate and up of 64 columns");
    constexpr int TM = WIDE_M ? kWide : kNarrow, TW = WIDE_M ? kNarrow : kWide;        // activation rows, weight rows
    constexpr int OUT_BN = GATE ? TW / 2 : TW;
    constexpr int MB = TM / 32, NB = TW / 32;       // 16-row blocks per wavefront
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int ww = WIDE_M ? wm : wn, wsm = WIDE_M ? wn : wm;

    // position b = (XCD x = b % 8, that XCD's i-th workgroup); XCD x walks a contiguous range of the tile order
    const int x = blockIdx.x % kXcds, xi_step = gridDim.x / kXcds;
    const int total = p.tiles_m * p.tiles_n, per = (total + kXcds - 1) / kXcds;
    const int nk = max((p.K + 2 * BK - 1) / (2 * BK) * 2, 4);       // K-tiles: an even number; those beyond K add zeros
    struct Tile {
        int m0, n0;
        bool valid;
    };
    auto decode = [&](int xi) {
        Tile t{0, 0, xi < per && x * per + xi < total};
        if (t.valid) {
            int tm, tn;
            tile_coords(x * per + xi, p.tiles_m, p.tiles_n, tm, tn);
            t.m0 = __builtin_amdgcn_readfirstlane(tm * TM);
            t.n0 = __builtin_amdgcn_readfirstlane(tn * OUT_BN);
        }
        return t;
    };

    // ---- global -> LDS: 8 rows x 128 bytes per instruction ----
    // A descriptor per operand; a row at or beyond the operand's last gets the offset of the descriptor's end, bytes beyond K kOutside.
    auto descriptor = [](const uint8_t* base, uint32_t bytes) {
        const uint64_t a = reinterpret_cast<uint64_t>(base);
        return s32x4{__builtin_amdgcn_readfirstlane(static_cast<int>(a)), __builtin_amdgcn_readfirstlane(static_cast<int>((a >> 32) & 0xffffu)),
                     __builtin_amdgcn_readfirstlane(static_cast<int>(bytes)), 0x00020000};
    };
    const s32x4 xrs = descriptor(p.A, static_cast<uint32_t>(p.M) * static_cast<uint32_t>(p.lda));
    const s32x4 wrs = descriptor(p.B, static_cast<uint32_t>(p.N) * static_cast<uint32_t>(p.ldb));
    [[maybe_unused]] const s32x4 urs = descriptor(GATE ? p.B2 : p.B, static_cast<uint32_t>(p.N) * static_cast<uint32_t>(p.ldb));
    constexpr int XI = WIDE_M ? 8 : 4, WI = 12 - XI;                // copy instructions per wavefront and K-tile
    uint32_t xoff[XI], woff[WI];
    int xi_fetch = blockIdx.x / kXcds;
    Tile F = decode(xi_fetch);
    if (!F.valid) return;
    int fk = 0;
    // the 16 bytes of its row that land in this lane's slot (rows 8 j + lane / 8: the swizzle alternates with j)
    auto chunk16 = [&](int j) { return static_cast<uint32_t>((lane & 7) ^ swz_row((j & 1) * 8 + (lane >> 3))) * 16u; };
    auto aim = [&]() {
#pragma unroll
        for (int j = 0; j < XI; ++j) {
            const int row = wave * (8 * XI) + 8 * j + (lane >> 3);
            xoff[j] = F.valid ? static_cast<uint32_t>(min(F.m0 + row, p.M)) * static_cast<uint32_t>(p.lda) + chunk16(j) : kOutside;
        }
#pragma unroll
        for (int j = 0; j < WI; ++j) {
            int n = F.n0 + wave * (8 * WI) + 8 * j + (lane >> 3);
            // SiLU gate: wavefront column c's 128 weight rows are gate, up of its first 32 columns, gate, up of its last 32
            if constexpr (GATE) n = F.n0 + (wave >> 1) * 64 + (wave & 1) * 32 + (j & 3) * 8 + (lane >> 3);
            woff[j] = F.valid ? static_cast<uint32_t>(min(n, p.N)) * static_cast<uint32_t>(p.ldb) + chunk16(j) : kOutside;
        }
    };
    aim();
    // before the copies of a K-tile: the next tile, if the fetch has been through this one; lanes whose bytes lie beyond K sent outside
    auto enter = [&]() {
        if (fk == nk) {
            xi_fetch += xi_step;
            F = decode(xi_fetch);
            fk = 0;
            aim();
        }
        if ((fk + 1) * BK > p.K) {
            const int left = p.K - fk * BK;
#pragma unroll
            for (int j = 0; j < XI; ++j) xoff[j] |= static_cast<int>(chunk16(j)) < left ? 0u : kOutside;
#pragma unroll
            for (int j = 0; j < WI; ++j) woff[j] |= static_cast<int>(chunk16(j)) < left ? 0u : kOutside;
        }
    };
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem));
    const uint32_t lds_x = lds0 + (WIDE_M ? 0 : kWideTile) + wave * (1024 * XI), lds_w = lds0 + (WIDE_M ? kWideTile : 0) + wave * (1024 * WI);
    auto dma = [&](int stage, auto ic) {
        constexpr int I = decltype(ic)::value;
        constexpr bool X = I < XI;
        constexpr int J = X ? I : I - XI;
        const uint32_t dst = (X ? lds_x : lds_w) + stage, off = X ? xoff[X ? J : 0] : woff[X ? 0 : J];
        const s32x4 rs = X ? xrs : (GATE && J >= 4) ? urs : wrs;
        const int k0 = min(fk * BK, p.K);           // (a K-tile beyond K: every lane is outside already)
        asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds"
                     :: "s"(dst), "n"(J * 1024), "v"(off), "s"(rs), "s"(k0) : "memory", "scc");
    };

    // ---- LDS -> MFMA operands: lane l holds the 32 bytes of k-group l / 16 of row l % 16 ----
    const int r16 = lane & 15, kg = lane >> 4;
    const int rd0 = r16 * BK + (((2 * kg) ^ swz_row(r16)) << 4);            // the second 16 bytes: rd0 ^ 16
    const int rd_w = ww * (128 * BK) + rd0, rd_s = kWideTile + wsm * (64 * BK) + rd0;
    v8i wset[8], sset[2][4];
    v4f acc[NB][MB];
    auto read_block = [&](int at, auto ic) {
        constexpr int I = decltype(ic)::value;
        const uint4 lo = *reinterpret_cast<const uint4*>(smem + at + I * 16 * BK), hi = *reinterpret_cast<const uint4*>(smem + (at ^ 16) + I * 16 * BK);
        return v8i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
    };
    auto read_w = [&](int at, auto ic) { wset[decltype(ic)::value] = read_block(at, ic); };
    auto read_s = [&](int at, auto pc, auto jc) { sset[decltype(pc)::value][decltype(jc)::value] = read_block(at, jc); };

    int s0 = 0, s1 = kStageBytes, s2 = 2 * kStageBytes;
    // One K-tile: 32 MFMAs, wide block by wide block, with one or two other items behind most of them
    auto ktile = [&](auto pc, auto first_c, auto wait_c) {
        constexpr int P = decltype(pc)::value;
        constexpr bool FIRST = decltype(first_c)::value, WAIT = decltype(wait_c)::value;
        const int nxt_w = rd_w + s1, nxt_s = rd_s + s1;
        read_w(rd_w + s0, std::integral_constant<int, 7>{});
        static_for<0, 32>([&](auto mc) {
            constexpr int m = decltype(mc)::value, g = m / 4, t = (g & 1) ? 3 - m % 4 : m % 4;
            if constexpr (WIDE_M) mfma<A5, FIRST>(acc[t][g], sset[P][t], wset[g]);
            else mfma<A5, FIRST>(acc[g][t], wset[g], sset[P][t]);
            if constexpr (m == 7) {
                if constexpr (WAIT) __builtin_amdgcn_s_waitcnt(kWaitVm12);
                __syncthreads();
                __builtin_amdgcn_sched_barrier(0);
                enter();
            }
            // wide block g is read behind its last MFMA, block 0 and 1 and the narrow ones from the barrier on
            using Z = std::integral_constant<int, 1 - P>;
            if constexpr (m == 8) read_w(nxt_w, std::integral_constant<int, 0>{});
            if constexpr (m == 9) read_s(nxt_s, Z{}, std::integral_constant<int, 0>{});
            if constexpr (m == 10) read_w(nxt_w, std::integral_constant<int, 1>{});
            if constexpr (m == 11) read_s(nxt_s, Z{}, std::integral_constant<int, 1>{});
            if constexpr (m == 13) read_w(nxt_w, std::integral_constant<int, 2>{});
            if constexpr (m == 15) read_s(nxt_s, Z{}, std::integral_constant<int, 2>{});
            if constexpr (m == 17) read_w(nxt_w, std::integral_constant<int, 3>{});
            if constexpr (m == 19) read_s(nxt_s, Z{}, std::integral_constant<int, 3>{});
            if constexpr (m == 21) read_w(nxt_w, std::integral_constant<int, 4>{});
            if constexpr (m == 25) read_w(nxt_w, std::integral_constant<int, 5>{});
            if constexpr (m == 29) read_w(nxt_w, std::integral_constant<int, 6>{});
            if constexpr (m >= 8 && m % 2 == 0) dma(s0, std::integral_constant<int, (m - 8) / 2>{});
            __builtin_amdgcn_sched_barrier(0);
        });
        ++fk;
        const int b = s0;
        s0 = s1; s1 = s2; s2 = b;
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;

    float s_one = 0.0f;
    [[maybe_unused]] float s_up = 0.0f;
    if constexpr (SCALE == SCALE_TENSOR) {
        s_one = p.sa[0] * p.sb[0];
        if constexpr (GATE) s_up = p.sa[0] * p.sb2[0];
    }

    Tile cur = F;
    static_for<0, 3>([&](auto sc) {
        enter();
        static_for<0, 12>([&](auto ic) { dma(decltype(sc)::value * kStageBytes, ic); });
        ++fk;
    });
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
    __syncthreads();
    static_for<0, 4>([&](auto jc) { read_s(rd_s, I0{}, jc); });
    static_for<0, 7>([&](auto ic) { read_w(rd_w, ic); });

    while (true) {
        // the first pair's copies were waited for in the prologue or in the epilogue before
        ktile(I0{}, std::true_type{}, std::false_type{});
        ktile(I1{}, std::false_type{}, std::false_type{});
        for (int kt = 2; kt < nk; kt += 2) {
            ktile(I0{}, std::false_type{}, std::true_type{});
            ktile(I1{}, std::false_type{}, std::true_type{});
        }
        // the MFMAs are opaque to the compiler's hazard handling
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");

        // ---- epilogue: accumulator register q of block (j, i) is activation row m0 + wm*16*MB + 16 i + lane % 16, weight row
        //      wn*16*NB + 16 j + 4 (lane / 16) + q ----
        int lane_e = lane;
        asm volatile("" : "+v"(lane_e));            // the epilogue's lane offsets are formed here, not kept through the K loop
        const int r_e = lane_e & 15, kg_e = lane_e >> 4, row_l = lane_e >> 3, col_l = 8 * (lane_e & 7);
        const int row_w = cur.m0 + wm * 16 * MB, col_w = cur.n0 + wn * (OUT_BN / 2);
        const uint32_t row_bytes = static_cast<uint32_t>(p.ldc) * 2u;
        uint8_t* const stg = smem + kRingBytes + wave * kStageOut;
        // rows 16 i .. of the wavefront's block of C: rows beyond M lie beyond the descriptor
        auto c_rsrc = [&](int i) {
            const int row = row_w + 16 * i, rows = max(min(p.M - row, 16), 0);
            const uint64_t at = reinterpret_cast<uint64_t>(p.C) + (static_cast<size_t>(rows > 0 ? row : 0) * p.ldc + col_w) * 2;
            const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<int>(at)), hi = __builtin_amdgcn_readfirstlane(static_cast<int>(at >> 32));
            return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>((static_cast<uint64_t>(hi) << 32) | lo), 0,
                                                     __builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(rows) * row_bytes)), 0x00020000);
        };
        auto quad = [](const v4f& a) { return make_float4(acc_read(a[0]), acc_read(a[1]), acc_read(a[2]), acc_read(a[3])); };
        if constexpr (!GATE) {
            // a pass: eight rows x 64 columns, staged in fp32; a lane reads back eight columns of a row and scales them
            constexpr int HN = NB / 4, PASSES = 16, ROWS = PASSES / HN;
            const uint32_t lane_off = row_l * row_bytes + col_l * 2;
            float cs[HN][8], sa[ROWS];
            uint4 bias[HN];
#pragma unroll
            for (int jp = 0; jp < HN; ++jp) {
                const int col = min(col_w + 64 * jp + col_l, p.N - 8);
                if constexpr (SCALE == SCALE_ROWCOL) {
                    const float4 lo = *reinterpret_cast<const float4*>(p.sb + col), hi = *reinterpret_cast<const float4*>(p.sb + col + 4);
                    cs[jp][0] = lo.x; cs[jp][1] = lo.y; cs[jp][2] = lo.z; cs[jp][3] = lo.w;
                    cs[jp][4] = hi.x; cs[jp][5] = hi.y; cs[jp][6] = hi.z; cs[jp][7] = hi.w;
                } else {
#pragma unroll
                    for (int q = 0; q < 8; ++q) cs[jp][q] = s_one;
                }
                if constexpr (EPI == EPI_BIAS) bias[jp] = *reinterpret_cast<const uint4*>(p.bias + col);
            }
#pragma unroll
            for (int r = 0; r < ROWS; ++r) sa[r] = SCALE == SCALE_ROWCOL ? p.sa[min(row_w + 8 * r + row_l, p.M - 1)] : 1.0f;
            __builtin_amdgcn_sched_barrier(0);
            // everything in flight, the copies of the next tile's first K-tiles among it, is waited for before the first store (one
            // counter for loads and stores): the tile that follows does not wait for its first pair
            __builtin_amdgcn_s_waitcnt(kWaitVm0);
            __builtin_amdgcn_sched_barrier(0);
            auto piece = [](int row, int chunk) { return row * 256 + ((chunk ^ row) << 4); };
#pragma unroll
            for (int u = 0; u < PASSES; ++u) {
                const int jp = u % HN, h = u / HN % 2, i = u / HN / 2;
                float4 v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = quad(acc[4 * jp + j][i]);
                if ((r_e >> 3) == h) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) *reinterpret_cast<float4*>(stg + piece(r_e & 7, 4 * j + kg_e)) = v[j];
                }
                const float4 lo = *reinterpret_cast<const float4*>(stg + piece(row_l, 2 * (lane_e & 7)));
                const float4 hi = *reinterpret_cast<const float4*>(stg + piece(row_l, 2 * (lane_e & 7) + 1));
                const float d[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
                float r[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) r[q] = d[q] * (sa[u / HN] * cs[jp][q]);
                u32x4 o;
                o.x = pack_bf16x2_hw(r[0], r[1]); o.y = pack_bf16x2_hw(r[2], r[3]);
                o.z = pack_bf16x2_hw(r[4], r[5]); o.w = pack_bf16x2_hw(r[6], r[7]);
                if constexpr (EPI == EPI_BIAS) {            // added to the bf16 result, as the separate kernel does
                    const uint4 bv = bias[jp];
                    o.x = pack_bf16x2_hw(bf16_lo(o.x) + bf16_lo(bv.x), bf16_hi(o.x) + bf16_hi(bv.x));
                    o.y = pack_bf16x2_hw(bf16_lo(o.y) + bf16_lo(bv.y), bf16_hi(o.y) + bf16_hi(bv.y));
                    o.z = pack_bf16x2_hw(bf16_lo(o.z) + bf16_lo(bv.z), bf16_hi(o.z) + bf16_hi(bv.z));
                    o.w = pack_bf16x2_hw(bf16_lo(o.w) + bf16_lo(bv.w), bf16_hi(o.w) + bf16_hi(bv.w));
                }
                const uint32_t at = col_w + 64 * jp + col_l < p.N ? lane_off + 128u * jp + 8 * h * row_bytes : kOutside;
                __builtin_amdgcn_raw_buffer_store_b128(o, c_rsrc(i), static_cast<int>(at), 0, kNonTemporal);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            // gate and up of the same columns meet in the accumulator layout (blocks 4 b + s: gate, 4 b + 2 + s: up of columns
            // 32 b + 16 s ..); what is staged is bf16, sixteen rows x 64 columns
            float sa[MB];
#pragma unroll
            for (int i = 0; i < MB; ++i) sa[i] = SCALE == SCALE_ROWCOL ? p.sa[min(row_w + 16 * i + r_e, p.M - 1)] : 1.0f;
            float4 cg[4], cu[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if constexpr (SCALE == SCALE_ROWCOL) {
                    const int col = min(col_w + 16 * c + 4 * kg_e, p.N - 4);
                    cg[c] = *reinterpret_cast<const float4*>(p.sb + col);
                    cu[c] = *reinterpret_cast<const float4*>(p.sb2 + col);
                } else {
                    cg[c] = make_float4(s_one, s_one, s_one, s_one);
                    cu[c] = make_float4(s_up, s_up, s_up, s_up);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(kWaitVm0);           // as above
            __builtin_amdgcn_sched_barrier(0);
            const uint32_t lane_off = col_w + col_l < p.N ? row_l * row_bytes + col_l * 2 : kOutside;
            auto piece = [](int row, int chunk) { return row * 128 + ((chunk ^ (row & 7)) << 4); };
#pragma unroll
            for (int i = 0; i < MB; ++i) {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int gb = 4 * (c >> 1) + (c & 1);
                    const float4 ga = quad(acc[gb][i]), ua = quad(acc[gb + 2][i]);
                    // the reference rounds gate and up to bf16 before the SiLU product
                    const uint32_t x0 = pack_bf16x2_hw(ga.x * (sa[i] * cg[c].x), ua.x * (sa[i] * cu[c].x));
                    const uint32_t x1 = pack_bf16x2_hw(ga.y * (sa[i] * cg[c].y), ua.y * (sa[i] * cu[c].y));
                    const uint32_t x2 = pack_bf16x2_hw(ga.z * (sa[i] * cg[c].z), ua.z * (sa[i] * cu[c].z));
                    const uint32_t x3 = pack_bf16x2_hw(ga.w * (sa[i] * cg[c].w), ua.w * (sa[i] * cu[c].w));
                    *reinterpret_cast<uint2*>(stg + piece(r_e, 2 * c + (kg_e >> 1)) + (kg_e & 1) * 8) =
                        make_uint2(pack_bf16x2_hw(fast_silu(bf16_lo(x0)) * bf16_hi(x0), fast_silu(bf16_lo(x1)) * bf16_hi(x1)),
                                   pack_bf16x2_hw(fast_silu(bf16_lo(x2)) * bf16_hi(x2), fast_silu(bf16_lo(x3)) * bf16_hi(x3)));
                }
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const u32x4 v = *reinterpret_cast<const u32x4*>(stg + piece(row_l + 8 * t, lane_e & 7));
                    __builtin_amdgcn_raw_buffer_store_b128(v, c_rsrc(i), static_cast<int>(lane_off + 8 * t * row_bytes), 0, kNonTemporal);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // the fetch, three K-tiles ahead in tiles of at least four, is in the tile that follows
        cur = F;
        if (!cur.valid) break;
    }
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
}

template <bool A5, int EPI, int SCALE, bool WIDE_M>
int launch(GemmArgs p, hipStream_t st) {
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [] {
        err = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm_nt_half<A5, EPI, SCALE, WIDE_M>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
    });
    if (err != hipSuccess) return static_cast<int>(err);
    constexpr int TM = WIDE_M ? kWide : kNarrow, OUT_BN = (WIDE_M ? kNarrow : kWide) / (EPI == EPI_SILU_GATE ? 2 : 1);
    p.tiles_m = (p.M + TM - 1) / TM;
    p.tiles_n = (p.N + OUT_BN - 1) / OUT_BN;
    const int want = 8 * ((p.tiles_m * p.tiles_n + 7) / 8), most = num_cus() / 8 * 8;
    k_gemm_nt_half<A5, EPI, SCALE, WIDE_M><<<want < most ? want : most, kThreads, kLdsBytes, st>>>(p);
    return launch_status();
}
// whether the tile lies along the rows: fewer tiles that way
bool along_rows(const GemmArgs& p) {
    return static_cast<long long>((p.M + 255) / 256) * ((p.N + 127) / 128) <= static_cast<long long>((p.M + 127) / 128) * ((p.N + 255) / 256);
}
template <bool A5, int EPI, int SCALE>
int launch_along(const GemmArgs& p, hipStream_t st) {
    return along_rows(p) ? launch<A5, EPI, SCALE, true>(p, st) : launch<A5, EPI, SCALE, false>(p, st);
}
template <bool A5, int SCALE>
int launch_plain(const GemmArgs& p, int epi, hipStream_t st) {
    return epi == EPI_BIAS ? launch_along<A5, EPI_BIAS, SCALE>(p, st) : launch_along<A5, EPI_NONE, SCALE>(p, st);
}

}  // namespace

bool half_ok(const GemmArgs& p, int fmt, int epi, int scale_mode) {
    // offsets travel in 32 bits with the top one marking "outside"
    if (p.tile_map || epi > EPI_SILU_GATE || fmt > 1 || scale_mode > SCALE_ROWCOL || p.K % 16 != 0 || p.K <= BK || p.ldc >= (1 << 21) ||
        static_cast<size_t>(p.M + kWide) * p.lda >= (1ull << 31) || static_cast<size_t>(p.N + kWide) * p.ldb >= (1ull << 31))
        return false;
    if (p.N % 8 != 0 || p.ldc % 8 != 0 || !aligned16(p.C) || (scale_mode == SCALE_ROWCOL && !aligned16(p.sb))) return false;
    if (epi == EPI_SILU_GATE) return fmt == 0 && (scale_mode == SCALE_TENSOR || aligned16(p.sb2));
    return epi != EPI_BIAS || aligned16(p.bias);
}

// Microseconds, measured at 300 sizes (130 to 8192 rows, 1024 to 50304 columns, K 1024 to 50304): 0.74 a K-tile where the round fills
// the chip and the L2s, 0.57 where up to 144 CUs have a tile; per tile the store, which a long K hides part of; 6 (gate 4) for the launch
// and the first fill.  Against the fastest of the other kernels there: 2048 x 4096 over K 14336 102.6 -> 90.8 us, over 50304 361 -> 317;
// 700 x 2 x 14336 over 4096 88.7 -> 79.3; 4000 x 2048 over 32000 302 -> 189.
// shared: with rows of K that share lines (K no multiple of 128).  A K-tile's copies then take 0.8 to 0.9 whatever the number of CUs, 0.95 in
// problems of several rounds.
float half_estimate_us(const GemmArgs& p, int epi, bool shared) {
    const int out_bn = 128;
    const long long tiles = epi == EPI_SILU_GATE ? static_cast<long long>((p.M + 127) / 128) * ((p.N + out_bn - 1) / out_bn)
                            : along_rows(p)      ? static_cast<long long>((p.M + 255) / 256) * ((p.N + 127) / 128)
                                                 : static_cast<long long>((p.M + 127) / 128) * ((p.N + 255) / 256);
    const int cus = num_cus();
    const long long full = tiles / cus, rest = tiles % cus;
    const float nk = static_cast<float>(p.K <= 2 * BK ? 4 : (p.K + 2 * BK - 1) / (2 * BK) * 2);
    const float busy = static_cast<float>(rest) / static_cast<float>(cus), tile = 2.5f + 20.0f / nk;
    const float crowd = busy > 0.5625f ? busy - 0.5625f : 0.0f;
    const float whole = shared ? 0.95f : 0.74f, slow = !shared ? 0.57f + 0.4f * crowd : full ? 0.95f : 0.80f + 0.2f * crowd;
    return (epi == EPI_SILU_GATE ? 4.0f : 6.0f) + static_cast<float>(full) * (nk * whole + tile) + (rest ? nk * slow + tile : 0.0f);
}

int gemm_nt_half(const GemmArgs& p, int fmt, int epi, int scale_mode, hipStream_t st) {
    if (epi == EPI_SILU_GATE)
        return scale_mode == SCALE_TENSOR ? launch<false, EPI_SILU_GATE, SCALE_TENSOR, false>(p, st) : launch<false, EPI_SILU_GATE, SCALE_ROWCOL, false>(p, st);
    if (fmt == 1) return scale_mode == SCALE_TENSOR ? launch_plain<true, SCALE_TENSOR>(p, epi, st) : launch_plain<true, SCALE_ROWCOL>(p, epi, st);
    return scale_mode == SCALE_TENSOR ? launch_plain<false, SCALE_TENSOR>(p, epi, st) : launch_plain<false, SCALE_ROWCOL>(p, epi, st);
}

}  // namespace cf
