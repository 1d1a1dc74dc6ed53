// bf16 weight gradients, C[M,N] += A[K,M]^T . B[K,N], dense and grouped per expert (gemm_bf16_tn_f32 of
// src/trainer.cu:3069-3160, called per expert at :7727-7740): the contraction runs over tokens, an expert's n rows, which both
// operands have as their SLOW dimension.  A tile is copied to LDS as it lies in memory, [k][columns], and read with
// ds_read_b64_tr_b16 (gemm_bf16.hip says how).
//
// What bounds it: C.  A weight gradient reads and writes M x N x 4 (2) bytes for a short K, so with one workgroup per CU all of
// them multiplied and then all of them waited for HBM (50304 x 4096 fp32 over 2048 rows: 600 us of products, 330 of C, 970 in
// all).  Here a CU holds TWO workgroups, one of which multiplies while the other adds its tile to C.
//   - Tile 256 x 128 (or 128 x 256) by steps of 32 k, four wavefronts 2 x 2, each 128 x 64 = 8 x 4 blocks of
//     v_mfma_f32_16x16x32_bf16: 128 accumulator registers, so that two wavefronts share a SIMD.  At 128 x 128 the copies
//     into LDS would take twice the bytes per FLOP and a CU takes in about 37 of its nominal 64 bytes a cycle; a third of the tile's
//     time would be theirs.
//   - LDS: a ring of three 24 KiB stages, filled by buffer_load ... lds three steps ahead (no staging registers).  The step's
//     operands are in registers before its barrier, so that the stage they came from is free for the copies right after it:
//     the narrow operand's four blocks have two register sets, the wide one's eight are refilled one by one behind the four
//     MFMAs that use them.
//   - 16-byte pieces of a row are xor-swizzled in the copy's source addresses (unit_swz), which no padding could do: a copy
//     instruction writes 1 KiB of LDS in a row.
//   - C passes through 2 KiB of LDS per wavefront, so that an instruction covers eight whole 128-byte lines.  Read and written from the
//     accumulator layout (neighbouring lanes sixteen rows apart) it took the memory pipe 64 accesses and held up the other
//     workgroup's copies: 890 us instead of 815 for the size above.
// Measured, before (one workgroup of 256 x 256 per CU) and after, C from memory: 50304 x 4096 fp32 over 2048 rows 970 -> 810 us; 64
// experts of 2048 x 1408 bf16 over 384 rows each 270 -> 205 us (0.9 GB: 174 us at the rate of a copy), over 1536 rows 620 -> 540;
// 1408 x 2048 over 8192 rows 172 -> 97; 1024 x 1024 over 8192 rows 183 -> 95 (twice the tiles).  Same bits: every output is summed over the
// same sequence of MFMAs.
#include "common.hpp"
#include "internal.hpp"

#include <algorithm>
#include <mutex>
#include <type_traits>

namespace cf {
namespace {

constexpr int kThr = 256;
constexpr int KS = 32;                          // k rows per step: one MFMA deep
constexpr int kWide = 256, kNarrow = 128;       // columns of the two operands' tiles
constexpr int kWidePitch = kWide * 2, kNarrowPitch = kNarrow * 2;
constexpr int kWideTile = KS * kWidePitch, kNarrowTile = KS * kNarrowPitch;
constexpr int kStageBytes = kWideTile + kNarrowTile;       // 24 KiB
constexpr int kStages = 3;
constexpr int kRingBytes = kStages * kStageBytes;
constexpr int kStageOut = 2048;                            // per wavefront: what the epilogue turns round at a time
constexpr int kLdsBytes = kRingBytes + 4 * kStageOut;      // 80 KiB: two workgroups per CU
constexpr long long kStreamBytes = 96ll << 20;             // a larger C is streamed (see launch)
constexpr long long kNearOperands = 300000000, kFarOperands = 600000000, kReadAgain = 1600000000;      // bytes (see large_operands)
constexpr int kTurn = 8;                                   // steps, an even number
constexpr int kNonTemporal = 2;                            // cache policy of a buffer access
constexpr int kWaitVm0 = 0x0f70, kWaitVm6 = 0x0f76;        // s_waitcnt vmcnt(n), the other counters left alone

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v4bf __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef int s32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4bf* lds_v4bf_ptr;

struct TnArgs {
    const uint16_t* A; int lda;     // [K rows][M]
    const uint16_t* B; int ldb;     // [K rows][N]
    void* C; int ldc;               // [M][N]
    int M, N, K;
    int tiles_m, tiles_n;
    int num_experts;
    const int* counts; const int* offsets;
    long long c_expert_stride;
};

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

__device__ __forceinline__ float acc_read(float a) {
    float v;
    asm("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(a));
    return v;
}

// Which 32-byte unit of a row (modulo 8) unit 0 of k row `row` is parked in: the rows one transposing read serves together
// (four consecutive ones of two neighbouring groups of eight) land in the eight different 32-byte units of 256 bytes.
__device__ __forceinline__ int unit_swz(int row) { return ((row & 3) << 1) | ((row >> 3) & 1); }

// STREAM: C is read and written past the caches.  TURNS: a CU's two workgroups go first by turns of kTurn steps, not of a tile.
template <bool WIDE_M, bool F32, bool GROUPED, bool STREAM, bool TURNS>
__global__ __launch_bounds__(kThr) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_gemm_bf16_tn_duo(const TnArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    constexpr int TM = WIDE_M ? kWide : kNarrow, TN = WIDE_M ? kNarrow : kWide;
    constexpr int MB = TM / 32, NB = TN / 32;           // 16-wide blocks per wavefront
    constexpr int CE = F32 ? 4 : 2;                      // bytes per element of C
    constexpr int AUX = STREAM ? kNonTemporal : 0;
    constexpr uint32_t kOutside = 0x80000000u;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int ww = WIDE_M ? wm : wn, wsm = WIDE_M ? wn : wm;

    const int x = blockIdx.x % 8, xi_step = gridDim.x / 8;
    const int tiles_mn = p.tiles_m * p.tiles_n, per = (tiles_mn + 7) / 8;

    struct Tile {
        int m0, n0, k_begin, k_end, nk;
        size_t c_base;
        bool valid;
    };
    // tile `i` of an order that walks the tiles in patches of `rows` row tiles, column after column
    auto place = [&](Tile& t, int i, int rows) {
        const int group = i / (rows * p.tiles_n), first = group * rows;
        const int gm = min(rows, p.tiles_m - first), in_group = i - group * rows * p.tiles_n;
        t.m0 = __builtin_amdgcn_readfirstlane((first + in_group % gm) * TM);
        t.n0 = __builtin_amdgcn_readfirstlane((in_group / gm) * TN);
    };
    auto decode = [&](int xi) {
        Tile t{};
        if constexpr (GROUPED) {
            const int round = xi / tiles_mn, e = x + 8 * round, ti = xi - round * tiles_mn;
            t.valid = e < p.num_experts;
            if (t.valid) {
                // An expert's tiles in patches too, of 1024 columns of A where it has 2048 or more: 64 tiles are worked on at a time, and of an
                // expert with many rows of tiles (14336 x 1024: 56) that would be all of A.  16 experts of 14336 x 1024 over 4473 rows
                // each 3298 us without, 1812 so (2048 columns: 2051); of 8192 x 1024 over 3305 1214 and 806; 8 of 8192 x 8192 over 2310
                // 3591 and 2522; of 2048 x 8192 over 11371 2966 and 2571.  1920 x 8064 over 3750 827 without, 850 in such patches.
                place(t, ti, p.M < 2048 ? p.tiles_m : 1024 / TM);
                // an expert's row range is cut at the rows the compact buffers hold
                t.k_begin = min(max(__builtin_amdgcn_readfirstlane(p.offsets[e]), 0), p.K);
                t.k_end = min(t.k_begin + min(max(__builtin_amdgcn_readfirstlane(p.counts[e]), 0), p.K), p.K);
                t.c_base = static_cast<size_t>(e) * p.c_expert_stride;
            }
        } else {
            const int lin = x * per + xi;
            t.valid = xi < per && lin < tiles_mn;
            if (t.valid) {
                place(t, lin, 8);
                t.k_end = p.K;
            }
        }
        t.nk = max(((t.k_end - t.k_begin + 2 * KS - 1) / (2 * KS)) * 2, 4);
        return t;
    };

    // ---- global -> LDS ----
    const uint16_t* const Wp = WIDE_M ? p.A : p.B;
    const uint16_t* const Sp = WIDE_M ? p.B : p.A;
    const uint32_t ldw = 2u * static_cast<uint32_t>(WIDE_M ? p.lda : p.ldb), lds_ = 2u * static_cast<uint32_t>(WIDE_M ? p.ldb : p.lda);
    const int ext_w = WIDE_M ? p.M : p.N, ext_s = WIDE_M ? p.N : p.M;
    uint32_t voff_w[4], voff_s[2];
    uint64_t base_w = 0, base_s = 0;
    int left_rows = 0;                              // k rows of the fetch tile from the fetch position on
    int xi_fetch = blockIdx.x / 8;
    Tile F = decode(xi_fetch);
    if (!F.valid) return;
    int fk = 0;
    // (A k row beyond the operand's last starts at its end: 32 bits hold that offset for every stride, which row * stride they
    // would not, fewer than 32 rows of more than 128 Mi elements being within the launcher's limits.)
    auto aim = [&]() {
        const int w0 = WIDE_M ? F.m0 : F.n0, s0 = WIDE_M ? F.n0 : F.m0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = 8 * wave + 2 * j + (lane >> 5), chunk = (lane & 31) ^ (unit_swz(row) << 1);
            voff_w[j] = w0 + chunk * 8 < ext_w ? static_cast<uint32_t>(min(row, p.K)) * ldw + chunk * 16u : kOutside;
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int row = 8 * wave + 4 * j + (lane >> 4), chunk = (lane & 15) ^ (unit_swz(row) << 1);
            voff_s[j] = s0 + chunk * 8 < ext_s ? static_cast<uint32_t>(min(row, p.K)) * lds_ + chunk * 16u : kOutside;
        }
        base_w = reinterpret_cast<uint64_t>(Wp) + static_cast<uint64_t>(F.k_begin) * ldw + 2ull * w0;
        base_s = reinterpret_cast<uint64_t>(Sp) + static_cast<uint64_t>(F.k_begin) * lds_ + 2ull * s0;
        left_rows = F.k_end - F.k_begin;
    };
    aim();
    s32x4 rs_w = s32x4{0, 0, 0, 0}, rs_s = rs_w;
    auto descriptors = [&]() {
        const uint32_t rows = static_cast<uint32_t>(max(left_rows, 0));
        rs_w = s32x4{__builtin_amdgcn_readfirstlane(static_cast<int>(base_w)), __builtin_amdgcn_readfirstlane(static_cast<int>((base_w >> 32) & 0xffffu)),
                     __builtin_amdgcn_readfirstlane(static_cast<int>(rows * ldw)), 0x00020000};
        rs_s = s32x4{__builtin_amdgcn_readfirstlane(static_cast<int>(base_s)), __builtin_amdgcn_readfirstlane(static_cast<int>((base_s >> 32) & 0xffffu)),
                     __builtin_amdgcn_readfirstlane(static_cast<int>(rows * lds_)), 0x00020000};
    };
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem));
    const uint32_t lds_w = lds0 + wave * (kWideTile / 4), lds_s = lds0 + kWideTile + wave * (kNarrowTile / 4);
    // copy I (0..5) of the fetch position's step: four of the wide operand, two of the narrow one
    auto dma = [&](int stage, auto ic) {
        constexpr int I = decltype(ic)::value;
        constexpr bool WIDE = I < 4;
        const uint32_t dst = (WIDE ? lds_w : lds_s) + stage, off = WIDE ? voff_w[WIDE ? I : 0] : voff_s[WIDE ? 0 : I - 4];
        const s32x4 rs = WIDE ? rs_w : rs_s;
        asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, 0 offen lds"
                     :: "s"(dst), "n"((WIDE ? I : I - 4) * 1024), "v"(off), "s"(rs) : "memory", "scc");
    };
    auto advance = [&]() {
        base_w += static_cast<uint64_t>(KS) * ldw;
        base_s += static_cast<uint64_t>(KS) * lds_;
        left_rows -= KS;
        ++fk;
    };
    // before the copies of a step: the next tile, if the fetch has been through this one
    auto enter = [&]() {
        if (fk == F.nk) {
            xi_fetch += xi_step;
            F = decode(xi_fetch);
            fk = 0;
            aim();
        }
        descriptors();
    };

    // ---- LDS -> MFMA operands ----
    const int r16 = lane & 15, kg = lane >> 4;
    const int row_l = 8 * kg + (r16 >> 2), unit_l = unit_swz(row_l);
    const int rd_w = row_l * kWidePitch + ww * 256 + unit_l * 32 + 8 * (r16 & 3);
    const int rd_s = kWideTile + row_l * kNarrowPitch + (((wsm * 4) ^ unit_l) << 5) + 8 * (r16 & 3);
    v8bf wset[8], sset[2][4];
    v4f acc[NB][MB];
    auto read_tr = [&](int off, auto pitch_c) {
        constexpr int PITCH = decltype(pitch_c)::value;
        const v4bf lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_v4bf_ptr)(smem + off));
        const v4bf hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_v4bf_ptr)(smem + off + 4 * PITCH));
        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    auto read_w = [&](int at, auto ic) {
        constexpr int I = decltype(ic)::value;
        wset[I] = read_tr(at ^ (I << 5), std::integral_constant<int, kWidePitch>{});
    };
    auto read_s = [&](int at, auto pc, auto jc) {
        constexpr int J = decltype(jc)::value;
        sset[decltype(pc)::value][J] = read_tr(at ^ (J << 5), std::integral_constant<int, kNarrowPitch>{});
    };

    int s0 = 0, s1 = kStageBytes, s2 = 2 * kStageBytes;
    // One step of 32 k: 32 MFMAs, wide block by wide block.
    auto step = [&](auto pc, auto first_c, auto wait_c) {
        constexpr int P = decltype(pc)::value;
        constexpr bool FIRST = decltype(first_c)::value, WAIT = decltype(wait_c)::value;
        const int cur_w = rd_w + s0, nxt_w = rd_w + s1, nxt_s = rd_s + s1;
        read_w(cur_w, std::integral_constant<int, 7>{});
        static_for<0, 32>([&](auto mc) {
            constexpr int m = decltype(mc)::value, g = m / 4, t = (g & 1) ? 3 - m % 4 : m % 4;
            constexpr int jn = WIDE_M ? t : g, im = WIDE_M ? g : t;
            const v8bf nreg = WIDE_M ? sset[P][t] : wset[g], mreg = WIDE_M ? wset[g] : sset[P][t];
            v4f c;
            if constexpr (FIRST) {
                asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(c) : "v"(nreg), "v"(mreg));
            } else {
                c = acc[jn][im];
                asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(nreg), "v"(mreg));
            }
            acc[jn][im] = c;
            if constexpr (m == 7) {
                if constexpr (WAIT) __builtin_amdgcn_s_waitcnt(kWaitVm6);
                __syncthreads();
                __builtin_amdgcn_sched_barrier(0);
                enter();
            }
            using Z = std::integral_constant<int, 1 - P>;
            if constexpr (m == 8) read_w(nxt_w, std::integral_constant<int, 0>{});
            if constexpr (m == 9) read_s(nxt_s, Z{}, std::integral_constant<int, 0>{});
            if constexpr (m == 10) dma(s0, std::integral_constant<int, 0>{});
            if constexpr (m == 11) read_w(nxt_w, std::integral_constant<int, 1>{});
            if constexpr (m == 12) read_s(nxt_s, Z{}, std::integral_constant<int, 1>{});
            if constexpr (m == 13) dma(s0, std::integral_constant<int, 1>{});
            if constexpr (m == 14) read_w(nxt_w, std::integral_constant<int, 2>{});
            if constexpr (m == 15) read_s(nxt_s, Z{}, std::integral_constant<int, 2>{});
            if constexpr (m == 16) dma(s0, std::integral_constant<int, 2>{});
            if constexpr (m == 17) read_w(nxt_w, std::integral_constant<int, 3>{});
            if constexpr (m == 18) read_s(nxt_s, Z{}, std::integral_constant<int, 3>{});
            if constexpr (m == 19) dma(s0, std::integral_constant<int, 3>{});
            if constexpr (m == 21) read_w(nxt_w, std::integral_constant<int, 4>{});
            if constexpr (m == 22) dma(s0, std::integral_constant<int, 4>{});
            if constexpr (m == 25) read_w(nxt_w, std::integral_constant<int, 5>{});
            if constexpr (m == 26) dma(s0, std::integral_constant<int, 5>{});
            if constexpr (m == 29) read_w(nxt_w, std::integral_constant<int, 6>{});
            __builtin_amdgcn_sched_barrier(0);
        });
        advance();
        const int b = s0;
        s0 = s1; s1 = s2; s2 = b;
    };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;

    // Left alone the matrix cores serve the older of a CU's two workgroups first, which then runs ahead by a quarter of the launch
    // (and out of step with what its XCD's L2 holds).  So the other one (its LDS starts above the first one's) goes first in
    // every second of its tiles.  With one tile per workgroup and many steps that would leave the other one alone for the second
    // half, when one wavefront per SIMD cannot fill the matrix cores: there they take turns inside the tile (TURNS; 1360 x 8944 fp32 over 17430 rows
    // 509 -> 447 us, 2360 x 4984 bf16 over 11926 304 -> 287, 14384 x 840 over 3545 99 -> 91).
    unsigned lds_alloc;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_LDS_ALLOC, 0, 12)" : "=s"(lds_alloc));
    bool first_now = lds_alloc != 0;
    auto go_first = [&]() {
        if (first_now) __builtin_amdgcn_s_setprio(3);
        else __builtin_amdgcn_s_setprio(0);
        first_now = lds_alloc != 0 && !first_now;
    };

    Tile cur = F;
    // the wavefront's block of C, rows from 16 im on: rows beyond the tile's end lie beyond the descriptor
    const uint32_t row_bytes = static_cast<uint32_t>(p.ldc) * CE;
    auto c_rsrc = [&](int im) {
        const int row_w = cur.m0 + wm * 16 * MB + 16 * im, rows = max(min(p.M - row_w, 16 * (MB - im)), 0);
        const uint64_t at = reinterpret_cast<uint64_t>(p.C) + (cur.c_base + static_cast<size_t>(rows > 0 ? row_w : 0) * p.ldc + cur.n0 + wn * 16 * NB) * CE;
        const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<int>(at)), hi = __builtin_amdgcn_readfirstlane(static_cast<int>(at >> 32));
        return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>((static_cast<uint64_t>(hi) << 32) | lo), 0,
                                                 __builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(rows) * row_bytes)), 0x00020000);
    };
    static_for<0, 3>([&](auto sc) {
        enter();
        static_for<0, 6>([&](auto ic) { dma(decltype(sc)::value * kStageBytes, ic); });
        advance();
    });
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
    __syncthreads();
    static_for<0, 4>([&](auto jc) { read_s(rd_s, B0{}, jc); });
    static_for<0, 7>([&](auto ic) { read_w(rd_w, ic); });

    while (true) {
        go_first();
        // the first pair's copies were waited for in the prologue or in the epilogue before
        step(B0{}, std::true_type{}, std::false_type{});
        step(B1{}, std::false_type{}, std::false_type{});
        for (int ks = 2; ks < cur.nk;) {
            const int stop = TURNS ? min(cur.nk, ks + kTurn) : cur.nk;
            for (; ks < stop; ks += 2) {
                step(B0{}, std::false_type{}, std::true_type{});
                step(B1{}, std::false_type{}, std::true_type{});
            }
            if constexpr (TURNS) go_first();
        }
        // the MFMAs are opaque to the compiler's hazard handling
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
        if (cur.k_end <= cur.k_begin) {
            // an empty k range adds nothing (and must not turn a -0 of C into +0)
            __builtin_amdgcn_s_waitcnt(kWaitVm0);
        } else {
            // accumulator register q of block (j, i): row m0 + wm*16*MB + 16 i + lane % 16, column n0 + wn*16*NB + 16 j + 4 (lane / 16) + q
            // From there a store instruction's neighbouring lanes would lie in sixteen rows, 16 bytes each, and so would the reads
            // of C: the memory pipe takes such an instruction lane by lane and the partner's copies wait behind it.  So sixteen rows
            // x 32 columns (bf16: eight x 64) at a time go through the wavefront's 2 KiB of LDS, 16-byte pieces xor-swizzled, and
            // C is read and written eight rows x 128 bytes per instruction.
            int lane_e = lane;
            asm volatile("" : "+v"(lane_e));        // the epilogue's lane offsets are formed here, not kept through the K loop
            const int r16e = lane_e & 15, kge = lane_e >> 4;
            const int col_w = cur.n0 + wn * 16 * NB;
            uint8_t* const stg = smem + kRingBytes + wave * kStageOut;
            constexpr int PN = F32 ? 32 : 64, HN = 16 * NB / PN;    // columns of a pass; passes side by side
            constexpr int PASSES = 16, kAhead = F32 ? 3 : 4;        // and the passes whose part of C is on its way
            const int row_l = lane_e >> 3, col_l = (F32 ? 4 : 8) * (lane_e & 7);
            const uint32_t lane_off = row_l * row_bytes + col_l * CE;
            // fp32: pass u = row block u / HN, all sixteen rows; bf16: row block u / (2 HN), rows 8 h .. with h = u / HN % 2
            auto row_block = [](int u) { return F32 ? u / HN : u / (2 * HN); };
            constexpr int LPP = F32 ? 2 : 1;                        // reads of C, and stores, per pass
            u32x4 old[kAhead][LPP];
            auto at = [&](int u, int t) {
                const uint32_t rows_down = F32 ? 8 * t : 8 * (u / HN % 2);
                return col_w + PN * (u % HN) + col_l < p.N ? lane_off + PN * CE * (u % HN) + rows_down * row_bytes : kOutside;
            };
            auto load = [&](int u) {
#pragma unroll
                for (int t = 0; t < LPP; ++t)
                    old[u % kAhead][t] = __builtin_amdgcn_raw_buffer_load_b128(c_rsrc(row_block(u)), static_cast<int>(at(u, t)), 0, AUX);
            };
#pragma unroll
            for (int u = 0; u < kAhead; ++u) load(u);
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt vmcnt(%0)" :: "n"(LPP * kAhead) : "memory");        // the copies of the next tile's first steps
            __builtin_amdgcn_sched_barrier(0);
            auto quad = [](const v4f& a) { return make_float4(acc_read(a[0]), acc_read(a[1]), acc_read(a[2]), acc_read(a[3])); };
#pragma unroll
            for (int u = 0; u < PASSES; ++u) {
                const int im = row_block(u);
                u32x4 o[LPP];
                if constexpr (F32) {
                    const int jn = 2 * (u % HN);
                    auto piece = [](int row, int chunk) { return row * 128 + ((chunk ^ (row & 7)) << 4); };
#pragma unroll
                    for (int j = 0; j < 2; ++j) *reinterpret_cast<float4*>(stg + piece(r16e, kge + 4 * j)) = quad(acc[jn + j][im]);
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        const float4 v = *reinterpret_cast<const float4*>(stg + piece(row_l + 8 * t, lane_e & 7));
                        const u32x4 c = old[u % kAhead][t];
                        o[t].x = __float_as_uint(__uint_as_float(c.x) + v.x);
                        o[t].y = __float_as_uint(__uint_as_float(c.y) + v.y);
                        o[t].z = __float_as_uint(__uint_as_float(c.z) + v.z);
                        o[t].w = __float_as_uint(__uint_as_float(c.w) + v.w);
                    }
                } else {
                    const int jn = 4 * (u % HN), h = u / HN % 2;
                    auto piece = [](int row, int chunk) { return row * 256 + ((chunk ^ row) << 4); };
                    float4 v[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[j] = quad(acc[jn + j][im]);
                    if ((r16e >> 3) == h) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) *reinterpret_cast<float4*>(stg + piece(r16e & 7, kge + 4 * j)) = v[j];
                    }
                    const float4 lo = *reinterpret_cast<const float4*>(stg + piece(row_l, 2 * (lane_e & 7)));
                    const float4 hi = *reinterpret_cast<const float4*>(stg + piece(row_l, 2 * (lane_e & 7) + 1));
                    const u32x4 c = old[u % kAhead][0];
                    // fp32 sum of the old value and the product, one rounding (cublasGemmEx with a bf16 C, beta = 1)
                    o[0].x = pack_bf16x2_hw(lo.x + bf16_lo(c.x), lo.y + bf16_hi(c.x));
                    o[0].y = pack_bf16x2_hw(lo.z + bf16_lo(c.y), lo.w + bf16_hi(c.y));
                    o[0].z = pack_bf16x2_hw(hi.x + bf16_lo(c.z), hi.y + bf16_hi(c.z));
                    o[0].w = pack_bf16x2_hw(hi.z + bf16_lo(c.w), hi.w + bf16_hi(c.w));
                }
                if (u + kAhead < PASSES) load(u + kAhead);
#pragma unroll
                for (int t = 0; t < LPP; ++t)
                    __builtin_amdgcn_raw_buffer_store_b128(o[t], c_rsrc(im), static_cast<int>(at(u, t)), 0, AUX);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // the fetch, three steps ahead in tiles of at least four steps, is in the tile that follows
        cur = F;
        if (!cur.valid) break;
    }
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
}

// two workgroups per CU, a multiple of 8 of them (launch position % 8 is the XCD)
int resident_workgroups() {
    static const int n = [] {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v < 8) return 512;
        return 2 * (v - v % 8);
    }();
    return n;
}
long long tiles_of(int M, int N, int tm, int tn) { return static_cast<long long>((M + tm - 1) / tm) * ((N + tn - 1) / tn); }

template <bool WIDE_M, bool F32, bool GROUPED, bool STREAM, bool TURNS>
int launch(TnArgs p, hipStream_t st) {
    static std::once_flag once;
    static hipError_t attr = hipSuccess;      // kept: a failed set-up is reported by every call, not only the first
    auto kern = k_gemm_bf16_tn_duo<WIDE_M, F32, GROUPED, STREAM, TURNS>;
    std::call_once(once, [&] {
        attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
    });
    if (attr != hipSuccess) return static_cast<int>(attr);
    const int most = resident_workgroups();         // and no more than there are tiles
    constexpr int TM = WIDE_M ? kWide : kNarrow, TN = WIDE_M ? kNarrow : kWide;
    p.tiles_m = (p.M + TM - 1) / TM;
    p.tiles_n = (p.N + TN - 1) / TN;
    const long long mn = static_cast<long long>(p.tiles_m) * p.tiles_n;
    const long long want = GROUPED ? 8 * mn * ((p.num_experts + 7) / 8) : 8 * ((mn + 7) / 8);
    if (want >= (1LL << 31)) return CF_ERR_UNSUPPORTED;
    kern<<<dim3(static_cast<unsigned>(want < most ? want : most)), kThr, kLdsBytes, st>>>(p);
    return launch_status();
}
template <bool WIDE_M, bool F32, bool GROUPED>
int launch(const TnArgs& p, hipStream_t st) {
    // A C that the 256 MiB memory-side cache still holds from the call that added to it before is best left there, one that comes from
    // memory is best streamed: 64 MiB fp32 (4096^2 over 256 rows) over and over 28 us, streamed 36, from memory 44 and 42; 96 MiB 39
    // and 45, 59 and 50; 144 MiB 60 and 69, 85 and 73; 192 MiB 73 and 102, 110 and 105; 256 MiB 124 and 125, 133 and 132.  The larger, the less
    // of it is likely to be left, so the line lies inside that range.
    // Streamed rows have to begin at lines: a line shared by two rows' accesses would be read and written twice (32000 x 2968 bf16 over
    // 848 rows 225 us streamed, 171 not; 30000 x 2056 fp32 over 256 213 and 107; rows at half lines 14336 x 4080 fp32 313 and 317).
    const long long bytes = static_cast<long long>(p.M) * p.ldc * (F32 ? 4 : 2) * (GROUPED ? p.num_experts : 1);
    const bool lines = (static_cast<long long>(p.ldc) * (F32 ? 4 : 2)) % 128 == 0 && (reinterpret_cast<uintptr_t>(p.C) & 127u) == 0;
    if (bytes > kStreamBytes && lines) return launch<WIDE_M, F32, GROUPED, true, false>(p, st);
    if constexpr (!GROUPED) {
        const long long tiles = WIDE_M ? tiles_of(p.M, p.N, kWide, kNarrow) : tiles_of(p.M, p.N, kNarrow, kWide);
        if (tiles <= resident_workgroups() && 2 * tiles > resident_workgroups()) return launch<WIDE_M, F32, GROUPED, false, true>(p, st);
    }
    return launch<WIDE_M, F32, GROUPED, false, false>(p, st);
}
template <bool F32, bool GROUPED>
int launch(const TnArgs& p, hipStream_t st) {
    // the tile lies along C whichever way it covers it with fewer (2048 x 1408: 88 tiles against 96); where both ways are alike and C is one wide tile
    // across, it takes whole rows, since two tiles would read and write the lines they share twice (64 experts of 6040 x 136 fp32
    // over 572 rows 143 us in two, 102 in one; 386560 x 136 over 9 136 and 93)
    const long long wide_m = tiles_of(p.M, p.N, kWide, kNarrow), wide_n = tiles_of(p.M, p.N, kNarrow, kWide);
    return wide_m < wide_n || (wide_m == wide_n && p.N > kWide) ? launch<true, F32, GROUPED>(p, st) : launch<false, F32, GROUPED>(p, st);
}

// Which dense problems go to one workgroup of 256 x 256 per CU instead (gemm_bf16.hip, the same sums).  The 64 workgroups of an XCD drift apart in k,
// beyond the 700 rows that its L2 holds of what they read; what they then read again comes from the 256 MiB memory-side cache, and from
// memory where the operands are larger (8192 x 8192 over 32768 rows: 29 GB through the L2s instead of 8).  Their 32 larger tiles take a third less
// per product and stay together.  Measured at 315 sizes, this kernel and that one: in several rounds of tiles the operands are read once a round
// and the line is where that comes to 1.6 GB: 8192 x 8192 bf16 over 32768 4411 and 3589 us, over 16384 1966 and 1828, over 8192 814 and 914; 128256 x
// 4096 fp32 over 2048 2830 and 2319, 50304 x 4096 over 2048 770 and 1000; 23168 x 49344 over 3234 9740 and 7600; 6072 x 18064 bf16 over 25114 7140 and
// 4820.  Narrow ones (one side up to 2048) gain little until their operands are twice that large: 80192 x 1536 over 1917 403 and 501, 25600 x 2728
// over 20295 3630 and 2622.  In a single round the partner's tile costs as much as the other half of a 256 x 256: 1136 x 9976 over 28204 810 and
// 594, 11008 x 768 over 21389 392 and 442.  Where it decides wrongly: 2624 x 54016 over 4371 1020 and 1275, 50304 x 4096 over 8192 2600 and 3010,
// and, kept here, 2760 x 5144 over 25895 868 and 585, 1848 x 13256 over 11575 662 and 518.
bool large_operands(int M, int N, int K) {
    if (K < 64) return false;
    const long long most = resident_workgroups(), bytes = 2ll * K * (static_cast<long long>(M) + N);
    const long long tiles = std::min(tiles_of(M, N, kWide, kNarrow), tiles_of(M, N, kNarrow, kWide)), rounds = (tiles + most - 1) / most;
    if (rounds == 1) return bytes > kFarOperands && 2 * tiles > most && 2 * tiles_of(M, N, kWide, kWide) <= most;
    return bytes * rounds > kReadAgain && (bytes > kFarOperands || (bytes > kNearOperands && std::min(M, N) > 2048));
}

// C[M,N] += A[K,M]^T . B[K,N]; grouped: per expert, K running over its rows of the compact buffers, C[E,M,N]
template <bool F32>
int gemm_tn(int M, int N, int K, int E, const int* counts, const int* offsets, const uint16_t* A, int lda, const uint16_t* B,
            int ldb, void* C, int ldc, bool grouped, cf_stream_t stream) {
    if (M < 0 || N < 0 || K < 0 || E < 0) return CF_ERR_INVALID_ARG;
    if (M == 0 || N == 0 || K == 0 || (grouped && E == 0)) return CF_OK;
    if (!A || !B || !C || (grouped && (!counts || !offsets))) return CF_ERR_INVALID_ARG;
    if (lda < M || ldb < N || ldc < N) return CF_ERR_INVALID_ARG;
    if (N % 8 != 0 || M % 8 != 0 || !bf16_operands_ok(A, lda, B, ldb, C, ldc, F32 ? 4 : 2)) return CF_ERR_UNSUPPORTED;
    if (static_cast<size_t>(K) * lda >= (1ull << 30) || static_cast<size_t>(K) * ldb >= (1ull << 30)) return CF_ERR_UNSUPPORTED;
    if (!grouped && large_operands(M, N, K)) return gemm_bf16_tn_large(M, N, K, A, lda, B, ldb, C, ldc, F32, as_stream(stream));
    TnArgs p{};
    p.A = A; p.lda = lda; p.B = B; p.ldb = ldb; p.C = C; p.ldc = ldc;
    p.M = M; p.N = N; p.K = K;
    if (!grouped) return launch<F32, false>(p, as_stream(stream));
    p.counts = counts; p.offsets = offsets;
    p.num_experts = E;
    p.c_expert_stride = static_cast<long long>(M) * ldc;
    return launch<F32, true>(p, as_stream(stream));
}

}  // namespace
}  // namespace cf

using namespace cf;

extern "C" {

int cf_gemm_bf16_tn_accum_f32(int M, int N, int K, const uint16_t* A, int lda, const uint16_t* B, int ldb, float* C, int ldc,
                              cf_stream_t stream) {
    return gemm_tn<true>(M, N, K, 0, nullptr, nullptr, A, lda, B, ldb, C, ldc, false, stream);
}
int cf_gemm_bf16_tn_accum_bf16(int M, int N, int K, const uint16_t* A, int lda, const uint16_t* B, int ldb, uint16_t* C,
                               int ldc, cf_stream_t stream) {
    return gemm_tn<false>(M, N, K, 0, nullptr, nullptr, A, lda, B, ldb, C, ldc, false, stream);
}
int cf_moe_grouped_gemm_bf16_tn_accum_f32(int M, int N, int total_rows, int num_experts, const int* d_counts,
                                          const int* d_offsets, const uint16_t* A, int lda, const uint16_t* B, int ldb,
                                          float* C, cf_stream_t stream) {
    return gemm_tn<true>(M, N, total_rows, num_experts, d_counts, d_offsets, A, lda, B, ldb, C, N, true, stream);
}
int cf_moe_grouped_gemm_bf16_tn_accum_bf16(int M, int N, int total_rows, int num_experts, const int* d_counts,
                                           const int* d_offsets, const uint16_t* A, int lda, const uint16_t* B, int ldb,
                                           uint16_t* C, cf_stream_t stream) {
    return gemm_tn<false>(M, N, total_rows, num_experts, d_counts, d_offsets, A, lda, B, ldb, C, N, true, stream);
}

}  // extern "C"
