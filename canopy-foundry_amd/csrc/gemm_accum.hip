// FP8 weight gradients over a ragged K (no multiple of 128), C[M,N] fp32 += s A[M,K] . B[N,K]^T with A in E4M3 and B in E5M2, on 256 x 256 tiles:
// eight wavefronts per workgroup, each 64 x 128, one workgroup per CU.
//
// What bounds it: C (14336 x 4096: 470 MB read and written, 90 us) and the bytes that the copies fetch.  Rows of K bytes that begin off the lines cost
// the 128 x 128 tiles of gemm_duo.hip a third of their rate, and those fetch twice the bytes per FLOP of these tiles to begin with.  The
// persistent kernel of gemm.hip has the same tile and hides more, but copies whole K-tiles of aligned rows only; where K is a multiple of 128
// it stays ahead (14336 x 4096, K 4096: 215 us, 235 here).  Here a CU multiplies and then adds with the matrix cores idle, and it is the CUs that
// overlap: they start at different times and so take turns at memory.
// 14336 x 4096, two workgroups per CU and this kernel: K 1488 152 -> 144 us, 2000 180 -> 164, 3008 221 -> 201, 4016 310 -> 256, 8176 563 -> 435;
// 28672 x 8192: K 2000 724 -> 572, 8176 2276 -> 1643; 8192 x 8192: K 4016 355 -> 291.  The backward of a 14336 x 4096 projection: 2000 tokens 372 -> 355 us,
// 4016 639 -> 589, 6800 987 -> 881, 8176 1153 -> 1028.
//
// The K loop is that of gemm_block.hip (v_mfma_f32_16x16x128_f8f6f4, two stages of 64 KiB, one barrier per K-tile before its last group of
// MFMAs), accumulating in place.  16-byte pieces of a row beyond K are sent beyond the copy's descriptor, which reads zeros.
#include "gemm_common.hpp"

#include <mutex>

namespace cf {
namespace {

constexpr int kAccThreads = 512;
constexpr int kAccStage = (BM + BN) * BK;               // 64 KiB: A rows, then B rows
constexpr int kAccOut = 2 * kAccStage;                  // 2 KiB per wavefront in which the products are turned round
constexpr int kAccLds = kAccOut + 8 * 2048;             // 147,456 bytes
constexpr int kAccWaitVm0 = 0x0f70;
constexpr uint32_t kAccOutside = 0x80000000u;           // beyond every descriptor (operands below 2 GiB)

typedef int s32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int acc_swz(int row) { return (row ^ ((row >> 3) & 1)) & 7; }

// Passes of 16 rows x 32 columns of C that a wavefront has on their way: 128 KiB per CU.
constexpr int kAhead = 8;
constexpr int kManyTiles = 6;      // tiles per workgroup

__global__ __launch_bounds__(kAccThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_gemm_nt_accum_wide(const GemmArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);      // 0..7
    const int wm = wave & 3, wn = wave >> 2;              // 64 rows x 128 columns
    const int ktiles = (p.K + BK - 1) / BK;               // >= 3, checked by the launcher
    const int total_tiles = p.tiles_m * p.tiles_n;
    int my_tiles, lin0, lstep;
    if (gridDim.x % kXcds == 0) {
        const int per = (total_tiles + kXcds - 1) / kXcds;
        const int x = blockIdx.x % kXcds, i = blockIdx.x / kXcds;
        lstep = gridDim.x / kXcds;
        const int cnt = max(0, min(per, total_tiles - x * per));
        my_tiles = (cnt - i + lstep - 1) / lstep;
        lin0 = x * per + i;
    } else {
        lstep = gridDim.x;
        my_tiles = (total_tiles - static_cast<int>(blockIdx.x) + lstep - 1) / lstep;
        lin0 = blockIdx.x;
    }
    if (my_tiles <= 0) return;
    // Turns at memory: the workgroups start in eight groups within about the time that C takes (24 us; `late` counts in us, a K-tile takes 1.42), which
    // costs the last group that much once, so over many tiles each, or a few of few K-tiles.  Over few otherwise, those with a tile fewer start late by
    // 1 us a K-tile and still end before the others.  In step, the second and the first: 14336 x 4096 (four tiles or three) K 2000 179, 164, 159 us, within
    // a step 376, 367, 354; K 4016 there 645, 595, 600.  28672 x 8192 (14 tiles), K 2000: 634, 571 in eight groups.  8192 x 8192 (four whole rounds), K 2000:
    // 197, 171.  The line at 20 K-tiles, within a step, second and first: 14336 x 4096 K 2000 382 and 367, 2512 452 and 441, 2768 470 and 463, 3024 489 and 485,
    // 3536 567 and 572; 12288 x 4096 K 2512 362 and 355, 3536 461 and 462; 11008 x 5120 (3.4 rounds) K 2000 388 and 392, 2512 and 3024 the same.
    int late = 0;
    if (total_tiles >= kManyTiles * static_cast<int>(gridDim.x)) late = min(ktiles, 24) * static_cast<int>(blockIdx.x / 8 % 8) / 8;
    else if (ktiles <= 20 && total_tiles >= 3 * static_cast<int>(gridDim.x)) late = ktiles * 3 * static_cast<int>(blockIdx.x / 8 % 8) / 16;
    else if (my_tiles * static_cast<int>(gridDim.x) < total_tiles) late = ktiles;
    for (int i = 0; i < late; ++i) __builtin_amdgcn_s_sleep(32);
    auto tile_at = [&](int seq, int& m0, int& n0) {
        int tm, tn;
        tile_coords(lin0 + seq * lstep, p.tiles_m, p.tiles_n, tm, tn);
        m0 = tm * BM;
        n0 = tn * BN;
    };
    const float scale = p.sa[0] * p.sb[0];

    // ---- global -> LDS: wavefront w copies rows [32 w, 32 w + 32) of both operands, eight lanes to a row of 128 bytes ----
    const int lrow = lane >> 3, lslot = lane & 7;
    uint32_t xoff[4], woff[4];
    auto aim = [&](int seq) {
        int m0, n0;
        tile_at(seq, m0, n0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = wave * 32 + j * 8 + lrow;
            const uint32_t chunk = (lslot ^ acc_swz(row)) * 16;
            xoff[j] = static_cast<uint32_t>(min(m0 + row, p.M - 1)) * static_cast<uint32_t>(p.lda) + chunk;
            woff[j] = static_cast<uint32_t>(min(n0 + row, p.N - 1)) * static_cast<uint32_t>(p.ldb) + chunk;
        }
    };
    const uint32_t x_bytes = static_cast<uint32_t>(p.M) * static_cast<uint32_t>(p.lda), w_bytes = static_cast<uint32_t>(p.N) * static_cast<uint32_t>(p.ldb);
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem));
    const uint32_t chunk_at[2] = {static_cast<uint32_t>((lslot ^ acc_swz(lrow)) * 16), static_cast<uint32_t>((lslot ^ acc_swz(lrow + 8)) * 16)};
    // The copies are issued through inline assembly: the compiler cannot tell that an LDS-DMA write and a later LDS read touch
    // different stages.  Their completion is tracked by hand before the barriers.
    auto dma16 = [&](uint32_t dst, uint32_t voff, const uint8_t* base, uint32_t bytes) {
        const uint64_t at = reinterpret_cast<uint64_t>(base);
        const s32x4 rs = {__builtin_amdgcn_readfirstlane(static_cast<int>(at)), __builtin_amdgcn_readfirstlane(static_cast<int>((at >> 32) & 0xffffu)),
                          __builtin_amdgcn_readfirstlane(static_cast<int>(bytes)), 0x00020000};
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" :: "s"(dst), "v"(voff), "s"(rs) : "memory");
    };
    // copy J (0..7) of the K-tile at position kt of its tile into the stage at `stage` (0 or kAccStage)
    auto copy_one = [&](int stage, int kt, auto jc) {
        constexpr int J = decltype(jc)::value;
        const uint32_t k0 = static_cast<uint32_t>(kt) * BK;
        const bool inside = chunk_at[J & 1] + k0 < static_cast<uint32_t>(p.K);
        if constexpr (J < 4) dma16(lds0 + stage + (wave * 32 + J * 8) * BK, inside ? xoff[J] : kAccOutside, p.A + k0, x_bytes - k0);
        else                 dma16(lds0 + stage + BM * BK + (wave * 32 + (J - 4) * 8) * BK, inside ? woff[J - 4] : kAccOutside, p.B + k0, w_bytes - k0);
    };

    // ---- LDS -> MFMA operands ----
    const int r16 = lane & 15, kg = lane >> 4;
    int xat[2], wat[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int rd = r16 * BK + (((kg * 2 + c) ^ acc_swz(r16)) << 4);
        xat[c] = wm * 64 * BK + rd;
        wat[c] = BM * BK + wn * 128 * BK + rd;
    }
    v4f acc[8][4];                // [B block][A block]
    v8i W[2][2], X[4];
    auto put = [](v8i& dst, int half, const uint4 v) {
        dst[4 * half + 0] = (int)v.x; dst[4 * half + 1] = (int)v.y; dst[4 * half + 2] = (int)v.z; dst[4 * half + 3] = (int)v.w;
    };
    auto read_w = [&](int stage, auto gc, auto rc) {
        constexpr int G = decltype(gc)::value, R = decltype(rc)::value;
        put(W[G & 1][R >> 1], R & 1, *reinterpret_cast<const uint4*>(smem + stage + wat[R & 1] + (G * 2 + (R >> 1)) * 16 * BK));
    };
    auto read_x = [&](int stage, auto rc) {
        constexpr int R = decltype(rc)::value;
        put(X[R >> 1], R & 1, *reinterpret_cast<const uint4*>(smem + stage + xat[R & 1] + (R >> 1) * 16 * BK));
    };
    // MFMA n (0..31): groups 0 to 2 take a B block at a time, the last one an A block (as in gemm_block.hip)
    auto mfma = [&](auto nc, auto first_c) {
        constexpr int n = decltype(nc)::value;
        constexpr int i = n < 24 ? 2 * (n >> 3) + ((n >> 2) & 1) : 6 + (n & 1), j = n < 24 ? n & 3 : (n - 24) >> 1;
        v4f c = acc[i][j];
        if constexpr (decltype(first_c)::value != 0) c = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(W[(i >> 1) & 1][i & 1], X[j], c, 1, 0, 0, 0, 0, 0);
    };

    int s0 = 0;
    // FIRST: the accumulators start at zero.  LAST: the next tile's operands are read after C, whose registers they would take.
    auto ktile = [&](auto first_c, auto last_c, int dkt) {
        constexpr bool LAST = decltype(last_c)::value != 0;
        const int s1 = s0 ^ kAccStage;
        static_for<0, 24>([&](auto nc) {
            constexpr int n = decltype(nc)::value;
            mfma(nc, first_c);
            if constexpr ((n & 7) < 4) read_w(s0, std::integral_constant<int, (n >> 3) + 1>{}, std::integral_constant<int, n & 3>{});
            __builtin_amdgcn_sched_barrier(0);
        });
        mfma(std::integral_constant<int, 24>{}, first_c);
        __builtin_amdgcn_sched_barrier(0);
        // The next K-tile's copies have landed; those of a tile's second one before the first pass of C came in, which set out after them (the
        // first tile's: above), so that the last stores of C are not waited for.
        if constexpr (decltype(first_c)::value == 0) __builtin_amdgcn_s_waitcnt(kAccWaitVm0);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        static_for<25, 32>([&](auto nc) {
            constexpr int n = decltype(nc)::value, m = n - 25;
            mfma(nc, first_c);
            if constexpr (!LAST && m < 2) {
                read_w(s1, std::integral_constant<int, 0>{}, std::integral_constant<int, (m < 2 ? 2 * m : 0)>{});
                read_w(s1, std::integral_constant<int, 0>{}, std::integral_constant<int, (m < 2 ? 2 * m + 1 : 0)>{});
            }
            if constexpr (!LAST && m >= 1) read_x(s1, std::integral_constant<int, (m >= 1 ? m - 1 : 0)>{});
            copy_one(s0, dkt, std::integral_constant<int, m>{});
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (!LAST) {
            read_x(s1, std::integral_constant<int, 6>{});
            read_x(s1, std::integral_constant<int, 7>{});
        }
        copy_one(s0, dkt, std::integral_constant<int, 7>{});
        __builtin_amdgcn_sched_barrier(0);
        s0 = s1;
    };

    aim(0);
    static_for<0, 8>([&](auto jc) { copy_one(0, 0, jc); });
    static_for<0, 8>([&](auto jc) { copy_one(kAccStage, 1, jc); });
    __builtin_amdgcn_s_waitcnt(kAccWaitVm0);
    __syncthreads();

    // copy position: two K-tiles ahead of the compute position; past the last tile the stream re-reads that tile and what it copies
    // is never used
    int dkt = 2, dseq = 0;
    auto advance_copy = [&]() {
        if (++dkt == ktiles) {
            dkt = 0;
            if (++dseq < my_tiles) aim(dseq);
        }
    };

    uint8_t* const stg = smem + kAccOut + wave * 2048;
    for (int seq = 0; seq < my_tiles; ++seq) {
        // The wavefront's 64 x 128 products go to C in sixteen passes of 16 rows x 32 columns: a lane holds four consecutive columns of one row
        // per block, so a pass is turned round in LDS (128-byte rows, 16-byte pieces xor-swizzled by row) and C is read and written eight
        // rows x 128 bytes per instruction.
        int m0, n0;
        tile_at(seq, m0, n0);
        int lane_d = lane;
        asm volatile("" : "+v"(lane_d));
        const int row = lane_d & 15, cq = lane_d >> 4, rr = lane_d >> 3, rc = lane_d & 7;
        float* const cb = p.Cf + static_cast<size_t>(m0 + wm * 64) * p.ldc + n0 + wn * 128;
        const int rows_left = p.M - m0 - wm * 64, cols_left = p.N - n0 - wn * 128 - rc * 4;
        u32x4 old[kAhead][2];
        const uint32_t row_bytes = static_cast<uint32_t>(p.ldc) * 4u;
        // the wavefront's block through a descriptor: rows at or beyond M lie beyond it, columns at or beyond N are sent there
        const uint64_t cat = reinterpret_cast<uint64_t>(cb);
        const uint32_t clo = __builtin_amdgcn_readfirstlane(static_cast<int>(cat)), chi = __builtin_amdgcn_readfirstlane(static_cast<int>(cat >> 32));
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            reinterpret_cast<void*>((static_cast<uint64_t>(chi) << 32) | clo), 0,
            __builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(max(min(rows_left, 64), 0)) * row_bytes)), 0x00020000);
        const uint32_t lane_at = static_cast<uint32_t>(rr) * row_bytes + rc * 16u;
        auto at = [&](int u, int t) {          // pass u: row block u / 4, columns 32 (u % 4)
            return (u & 3) * 32 < cols_left ? lane_at + ((u >> 2) * 16 + t * 8) * row_bytes + (u & 3) * 128u : kAccOutside;
        };
        auto load = [&](int u) {
#pragma unroll
            for (int t = 0; t < 2; ++t) old[u % kAhead][t] = __builtin_amdgcn_raw_buffer_load_b128(rs, static_cast<int>(at(u, t)), 0, 2);
        };
        static_for<0, 4>([&](auto rc) { read_w(s0, std::integral_constant<int, 0>{}, rc); });
        static_for<0, 8>([&](auto rc) { read_x(s0, rc); });
        ktile(std::integral_constant<int, 1>{}, std::integral_constant<int, 0>{}, dkt);
        advance_copy();
        for (int kt = 1; kt < ktiles - 1; ++kt) {
            ktile(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, dkt);
            advance_copy();
        }
        ktile(std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{}, dkt);
        advance_copy();
#pragma unroll
        for (int u = 0; u < kAhead; ++u) load(u);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int j = u >> 2, i = 2 * (u & 3);
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const v4f v = acc[i + b][j];
                *reinterpret_cast<float4*>(stg + row * 128 + (((b * 4 + cq) ^ (row & 7)) << 4)) =
                    make_float4(v[0] * scale, v[1] * scale, v[2] * scale, v[3] * scale);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            u32x4 o[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int r = rr + 8 * t;
                const float4 v = *reinterpret_cast<const float4*>(stg + r * 128 + ((rc ^ (r & 7)) << 4));
                const u32x4 c = old[u % kAhead][t];
                o[t].x = __float_as_uint(__uint_as_float(c.x) + v.x);
                o[t].y = __float_as_uint(__uint_as_float(c.y) + v.y);
                o[t].z = __float_as_uint(__uint_as_float(c.z) + v.z);
                o[t].w = __float_as_uint(__uint_as_float(c.w) + v.w);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            if (u + kAhead < 16) load(u + kAhead);
#pragma unroll
            for (int t = 0; t < 2; ++t) __builtin_amdgcn_raw_buffer_store_b128(o[t], rs, static_cast<int>(at(u, t)), 0, 2);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // the copies started past the end of the stream must have landed before the LDS is given back
    __builtin_amdgcn_s_waitcnt(kAccWaitVm0);
}

}  // namespace

// Operands and rows of C as the accumulating kernels of gemm_duo.hip take them, with three K-tiles at least.
bool accum_wide_ok(const GemmArgs& p, int fmt, int epi, int scale_mode) {
    return epi == EPI_ACCUM_F32 && scale_mode == SCALE_TENSOR && fmt == 2 && !p.tile_map && p.K % 16 == 0 && p.K > 2 * BK && p.K % BK != 0 &&
           p.lda % 16 == 0 && p.ldb % 16 == 0 && aligned16(p.A) && aligned16(p.B) && p.N % 4 == 0 && p.ldc % 4 == 0 && aligned16(p.Cf) &&
           p.ldc < (1 << 23) && static_cast<size_t>(p.M) * p.lda < (1ull << 31) && static_cast<size_t>(p.N) * p.ldb < (1ull << 31);
}

// Microseconds: per round of tiles 1.42 a K-tile and, for C, 21; 26 where a few rounds, the last of them more than four fifths full, leave hardly a workgroup to
// start later, 34 where there is one round and all go to C at once, 39 where the rows of C do not begin at lines.  Beside the two workgroups per CU (them,
// this), a line on each side: 14336 x 4096, K 1040 123 and 120 alone, K 1488 152 and 144; 14336 x 4100, K 1488 209 and 222, K 2000 241 and 237; 10620 x 3072, K
// 800 64.4 and 70.7 (504 tiles); 5632 x 2048 (one round, part filled), K 4016 70.7 and 66.4 alone but no difference within a step, K 8176 121 and 110; 5120 x 4096
// (a quarter of the second round filled), K 8176 198 and 210.  Of 453 random sizes that come here 14 are slower by more than 3 %, the worst 1.06 times (K 800 to 1350).
float accum_wide_estimate_us(const GemmArgs& p) {
    const int most = num_cus();
    const long long tiles = static_cast<long long>((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN), rounds = (tiles + most - 1) / most;
    const float c = c_lines_shared(p, 4) ? 39.0f : rounds == 1 ? 34.0f : 5 * (rounds * most - tiles) < most && rounds < kManyTiles ? 26.0f : 21.0f;
    return static_cast<float>(rounds) * (static_cast<float>((p.K + BK - 1) / BK) * 1.42f + c);
}

int gemm_nt_accum_wide(GemmArgs p, hipStream_t st) {
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [] {
        err = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm_nt_accum_wide), hipFuncAttributeMaxDynamicSharedMemorySize, kAccLds);
    });
    if (err != hipSuccess) return static_cast<int>(err);
    p.tiles_m = (p.M + BM - 1) / BM;
    p.tiles_n = (p.N + BN - 1) / BN;
    k_gemm_nt_accum_wide<<<persistent_grid(p.tiles_m * p.tiles_n, num_cus()), kAccThreads, kAccLds, st>>>(p);
    return launch_status();
}

}  // namespace cf
