// Block-scaled FP8 GEMM on 256 x 256 tiles and on 128 x 128 tiles (1 x 128 activation scales, 128 x 128 weight-block scales), persistent, one
// workgroup of eight wavefronts per CU.  The large ones first.
//
// What bounds it: the socket's power, and with it the bytes an operation moves.  A 128-wide K-tile is one scale group, so its partial
// products start from zero and are folded into running sums on the vector ALU, which cannot write accumulation registers while the
// matrix cores run.  With v_mfma_f32_32x32x64 a wavefront held 64 registers of partial products and its tile was 64 x 64; with
// v_mfma_f32_16x16x128 one MFMA is a whole scale group of a 16 x 16 block, its four registers are folded three MFMAs later, and
// the tile is 64 x 128 (sums 128 registers, activations 32, weights 2 x 16, partial products 16 of the 256 that two wavefronts per SIMD have).
// A workgroup's 256 x 256 tile takes two thirds of the L2-to-LDS bytes per FLOP of the 128 x 256 tile of k_gemm_nt_block_ring, three
// quarters of its LDS reads and half of its barriers.  4096 x 7168 x 7168, quantized normal operands: 210 -> 186 us (2.26 PFLOP/s) on one pair of
// operands over and over, 243 -> 199 on eight pairs in turn, so from memory (202 in a profile of the quantize and it); 1.75 rounds of tiles, so 87.5 % at best.
//
// LDS: two stages of 64 KiB.  A K-tile is 32 MFMAs per wavefront in four groups of eight (two weight blocks x four activation blocks).
// The weights of the next group are read under the current one; before the last group every wavefront has the rest of the K-tile in
// registers, so the barrier stands there: behind it the next K-tile is visible and read under the last group, and the copies of the
// K-tile after that go into the stage just left.
#include "gemm_common.hpp"

#include <mutex>

namespace cf {
namespace {

constexpr int kWideThreads = 512;
constexpr int kWideStage = (BM + BN) * BK;              // 64 KiB: activations, then weights
constexpr int kWideSa = 2 * kWideStage;                 // activation scales: 2 stages x 256 floats
constexpr int kWideSb = kWideSa + 2 * BM * 4;           // weight-block scales: 2 tile parities x 2 column blocks x 256 floats
constexpr int kWideMaxKb = 256;
constexpr int kWideOut = kWideSb + 2 * 2 * kWideMaxKb * 4;      // 2 KiB per wavefront in which the output is turned round
constexpr int kWideLds = kWideOut + 8 * 2048;           // 153,600 bytes
constexpr int kWideWaitVm0 = 0x0f70;                    // s_waitcnt vmcnt(0) only

// 16-byte pieces of a row are xor-swizzled: the 16-lane groups of a ds_read_b128 meet 16 different slots (the pattern repeats every 16 rows)
__device__ __forceinline__ int swz_rows16(int row) { return (row ^ ((row >> 3) & 1)) & 7; }

__global__ __launch_bounds__(kWideThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_gemm_nt_block_wide(const GemmArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);      // 0..7
    const int wm = wave & 3, wn = wave >> 2;              // 64 rows x 128 columns: the four wavefronts of a wn share a column block
    const int ktiles = p.K / BK;          // >= 3, checked by the launcher; also the number of scale groups along K
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
    auto tile_at = [&](int seq, int& m0, int& n0) {
        int tm, tn;
        tile_coords(lin0 + seq * lstep, p.tiles_m, p.tiles_n, tm, tn);
        m0 = tm * BM;
        n0 = tn * BN;
    };

    // ---- global -> LDS: wavefront w copies rows [32 w, 32 w + 32) of both operands and the scales of those activation rows ----
    const int lrow = lane >> 3, lslot = lane & 7;
    uint32_t xoff[4], woff[4], saoff = 0;              // per-lane byte offsets
    const uint8_t* sbsrc = nullptr;                    // the tile's rows of weight-block scales
    auto aim = [&](int seq) {
        int m0, n0;
        tile_at(seq, m0, n0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = wave * 32 + j * 8 + lrow;
            const uint32_t chunk = (lslot ^ swz_rows16(row)) * 16;
            xoff[j] = static_cast<uint32_t>(min(m0 + row, p.M - 1)) * static_cast<uint32_t>(p.lda) + chunk;
            woff[j] = static_cast<uint32_t>(n0 + row) * static_cast<uint32_t>(p.ldb) + chunk;        // N % 256 == 0
        }
        saoff = static_cast<uint32_t>(min(m0 + wave * 32 + (lane & 31), p.M - 1)) * static_cast<uint32_t>(ktiles) * 4u;
        sbsrc = reinterpret_cast<const uint8_t*>(p.sb + static_cast<size_t>((n0 >> 7) + (wave & 1)) * ktiles);
    };
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem));
    auto dma16 = [&](uint32_t dst, uint32_t voff, const uint8_t* base) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(dst), "v"(voff), "s"(base) : "memory");
    };
    // 4-byte copies by the low 32 lanes only: lane l lands at dst + 4 l.  Every call site is in wavefront-uniform control flow with
    // all 64 lanes active, so "all ones" is what the execution mask was.
    auto dma4_lo32 = [&](uint32_t dst, uint32_t voff, const uint8_t* base) {
        asm volatile("s_mov_b32 m0, %0\n\ts_mov_b32 exec_hi, 0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2\n\ts_mov_b32 exec_hi, -1\n\ts_nop 0"
                     :: "s"(dst), "v"(voff), "s"(base) : "memory");
    };
    auto dma4 = [&](uint32_t dst, uint32_t voff, const uint8_t* base) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" :: "s"(dst), "v"(voff), "s"(base) : "memory");
    };
    // copy J (0..8) of the K-tile at position kt of its tile into the stage at `stage` (0 or kWideStage)
    auto copy_one = [&](int stage, int kt, auto jc) {
        constexpr int J = decltype(jc)::value;
        if constexpr (J < 4)      dma16(lds0 + stage + (wave * 32 + J * 8) * BK, xoff[J], p.A + kt * BK);
        else if constexpr (J < 8) dma16(lds0 + stage + BM * BK + (wave * 32 + (J - 4) * 8) * BK, woff[J - 4], p.B + kt * BK);
        else dma4_lo32(lds0 + kWideSa + (stage ? BM * 4 : 0) + wave * 128, saoff, reinterpret_cast<const uint8_t*>(p.sa + kt));
    };
    // the weight-block scales of the tile the stream has just turned to, by wavefronts 0 and 1 (one per column block), into the half of
    // the scale table selected by the tile's parity
    auto copy_sb = [&](int parity) {
        if (wave < 2) {
            for (int c = 0; c * 64 < ktiles; ++c) {
                const uint32_t v = static_cast<uint32_t>(min(c * 64 + lane, ktiles - 1)) * 4u;
                dma4(lds0 + kWideSb + (parity * 2 + wave) * (kWideMaxKb * 4) + c * 256, v, sbsrc);
            }
        }
    };

    // ---- LDS -> MFMA operands: block b is rows 16 b ... + 15; lane l reads row l % 16, the 32 bytes of k-group l / 16 ----
    const int r16 = lane & 15, kg = lane >> 4;
    int xat[2], wat[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int rd = r16 * BK + (((kg * 2 + c) ^ swz_rows16(r16)) << 4);
        xat[c] = wm * 64 * BK + rd;
        wat[c] = BM * BK + wn * 128 * BK + rd;
    }
    v4f sum[8][4];                // [weight block][activation block]: running sums, already scaled
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) sum[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    v8i W[2][2], X[4];            // weight blocks of two groups, the K-tile's activation blocks
    v4f part[4];                  // partial products on their way into the sums
    float f[4], fn[4];            // factors of this K-tile's activation blocks, and the next one's
    auto put = [](v8i& dst, int half, const uint4 v) {
        dst[4 * half + 0] = (int)v.x; dst[4 * half + 1] = (int)v.y; dst[4 * half + 2] = (int)v.z; dst[4 * half + 3] = (int)v.w;
    };
    // read R (0..3) of weight group G (blocks 2 G, 2 G + 1); read R (0..7) of the activations
    auto read_w = [&](int stage, auto gc, auto rc) {
        constexpr int G = decltype(gc)::value, R = decltype(rc)::value;
        put(W[G & 1][R >> 1], R & 1, *reinterpret_cast<const uint4*>(smem + stage + wat[R & 1] + (G * 2 + (R >> 1)) * 16 * BK));
    };
    auto read_x = [&](int stage, auto rc) {
        constexpr int R = decltype(rc)::value;
        put(X[R >> 1], R & 1, *reinterpret_cast<const uint4*>(smem + stage + xat[R & 1] + (R >> 1) * 16 * BK));
    };
    // MFMA n (0..31) of a K-tile: groups 0 to 2 take a weight block at a time, the last one an activation block, so that the next
    // K-tile's activations can be read as this one's fall free
    auto mfma = [&](auto nc) {
        constexpr int n = decltype(nc)::value;
        constexpr int i = n < 24 ? 2 * (n >> 3) + ((n >> 2) & 1) : 6 + (n & 1), j = n < 24 ? n & 3 : (n - 24) >> 1;
        part[n & 3] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(W[(i >> 1) & 1][i & 1], X[j], v4f{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0, 0, 0, 0);
    };
    auto fold = [&](auto nc) {
        constexpr int n = decltype(nc)::value;
        constexpr int i = n < 24 ? 2 * (n >> 3) + ((n >> 2) & 1) : 6 + (n & 1), j = n < 24 ? n & 3 : (n - 24) >> 1;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float v = __builtin_fmaf(part[n & 3][r], f[j], sum[i][j][r]);
            asm volatile("" : "+v"(v));         // here, not gathered at the end of the loop body with 128 partial products alive
            sum[i][j][r] = v;
        }
    };
    auto read_factors = [&](int stage, int parity, int kt) {
        const float sbv = *reinterpret_cast<const float*>(smem + kWideSb + (parity * 2 + wn) * (kWideMaxKb * 4) + kt * 4);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            fn[j] = *reinterpret_cast<const float*>(smem + kWideSa + (stage ? BM * 4 : 0) + (wm * 64 + j * 16 + r16) * 4) * sbv;
    };

    int s0 = 0;                   // stage of the current K-tile; the other one holds, or receives, the next
    // One K-tile.  FIRST: a tile's first (nothing is left to fold).  (nkt, npar): position and tile parity of the K-tile after it,
    // dkt: position of the one after that, whose copies start behind the barrier.
    auto ktile = [&](auto first_c, int nkt, int npar, int dkt) {
        constexpr bool FIRST = decltype(first_c)::value != 0;
        const int s1 = s0 ^ kWideStage;
        static_for<0, 24>([&](auto nc) {
            constexpr int n = decltype(nc)::value;
            mfma(nc);
            if constexpr (n >= 3) {
                fold(std::integral_constant<int, (n >= 3 ? n - 3 : 0)>{});
            } else if constexpr (!FIRST) {
                fold(std::integral_constant<int, 29 + n>{});
            }
            if constexpr (n == 2) {
#pragma unroll
                for (int j = 0; j < 4; ++j) f[j] = fn[j];
            }
            if constexpr ((n & 7) < 4) read_w(s0, std::integral_constant<int, (n >> 3) + 1>{}, std::integral_constant<int, n & 3>{});
            __builtin_amdgcn_sched_barrier(0);
        });
        mfma(std::integral_constant<int, 24>{});
        fold(std::integral_constant<int, 21>{});
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(kWideWaitVm0);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        static_for<25, 32>([&](auto nc) {
            constexpr int n = decltype(nc)::value, m = n - 25;
            mfma(nc);
            fold(std::integral_constant<int, n - 3>{});
            if constexpr (m < 2) {
                read_w(s1, std::integral_constant<int, 0>{}, std::integral_constant<int, (m < 2 ? 2 * m : 0)>{});
                read_w(s1, std::integral_constant<int, 0>{}, std::integral_constant<int, (m < 2 ? 2 * m + 1 : 0)>{});
            }
            // activation block j falls free with MFMA 25 + 2 j
            if constexpr (m >= 1) read_x(s1, std::integral_constant<int, (m >= 1 ? m - 1 : 0)>{});
            copy_one(s0, dkt, std::integral_constant<int, m>{});
            if constexpr (m == 2) read_factors(s1, npar, nkt);
            __builtin_amdgcn_sched_barrier(0);
        });
        read_x(s1, std::integral_constant<int, 6>{});
        read_x(s1, std::integral_constant<int, 7>{});
        copy_one(s0, dkt, std::integral_constant<int, 7>{});
        copy_one(s0, dkt, std::integral_constant<int, 8>{});
        __builtin_amdgcn_sched_barrier(0);
        s0 = s1;
    };

    // prologue: K-tiles 0 and 1 in LDS, K-tile 0's first operands and factors in registers
    aim(0);
    copy_sb(0);
    static_for<0, 9>([&](auto jc) { copy_one(0, 0, jc); });
    static_for<0, 9>([&](auto jc) { copy_one(kWideStage, 1, jc); });
    __builtin_amdgcn_s_waitcnt(kWideWaitVm0);
    __syncthreads();
    static_for<0, 4>([&](auto rc) { read_w(0, std::integral_constant<int, 0>{}, rc); });
    static_for<0, 8>([&](auto rc) { read_x(0, rc); });
    read_factors(0, 0, 0);

    // copy position: two K-tiles ahead of the compute position; past the last tile the stream re-reads that tile and what it copies
    // is never used
    int dkt = 2, dseq = 0;
    auto advance_copy = [&]() {
        if (++dkt == ktiles) {
            dkt = 0;
            if (++dseq < my_tiles) aim(dseq);
            copy_sb(dseq & 1);
        }
    };

    uint8_t* stg = smem + kWideOut + wave * 2048;
    for (int seq = 0; seq < my_tiles; ++seq) {
        const int parity = seq & 1;
        ktile(std::integral_constant<int, 1>{}, 1, parity, dkt);
        advance_copy();
        for (int kt = 1; kt < ktiles; ++kt) {
            const bool last = kt + 1 == ktiles;
            ktile(std::integral_constant<int, 0>{}, last ? 0 : kt + 1, last ? parity ^ 1 : parity, dkt);
            advance_copy();
        }
        static_for<29, 32>([&](auto nc) { fold(nc); });
        // The sums leave as bf16.  A lane holds four consecutive columns of one row per block; 16 rows x 64 columns at a time are
        // turned round in LDS (128-byte rows, 16-byte pieces xor-swizzled by row) and stored as whole lines, eight rows per instruction.
        int m0, n0;
        tile_at(seq, m0, n0);
        int lane_d = lane;
        asm volatile("" : "+v"(lane_d));        // the drain's per-lane constants are worked out here, not kept through the K loop
        const int row = lane_d & 15, cq = lane_d >> 4, rr = lane_d >> 3, rc = lane_d & 7;
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        uint16_t* cp = p.C + static_cast<size_t>(m0 + wm * 64) * p.ldc + n0 + wn * 128;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    v4f& v = sum[h * 4 + b][j];
                    *reinterpret_cast<uint2*>(stg + row * 128 + (((b * 2 + (cq >> 1)) ^ ((row >> 1) & 7)) << 4) + (cq & 1) * 8) =
                        make_uint2(pack_bf16x2_hw(v[0], v[1]), pack_bf16x2_hw(v[2], v[3]));
                    v = v4f{0.0f, 0.0f, 0.0f, 0.0f};
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const int r = rr + 8 * t;
                    const uint4 v = *reinterpret_cast<const uint4*>(stg + r * 128 + ((rc ^ ((r >> 1) & 7)) << 4));
                    if (m0 + wm * 64 + j * 16 + r < p.M) {
                        const u32x4 vv = {v.x, v.y, v.z, v.w};
                        __builtin_nontemporal_store(vv, reinterpret_cast<u32x4*>(cp + static_cast<size_t>(j * 16 + r) * p.ldc + h * 64 + rc * 8));
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_sched_barrier(0);
            }
    }
    // the copies started past the end of the stream must have landed before the LDS is given back
    __builtin_amdgcn_s_waitcnt(kWideWaitVm0);
}

// The same on 128 x 128 tiles, for problems that give the 128 x 256 tiles of k_gemm_nt_block_ring to half of the CUs or fewer: eight wavefronts of 32 x 64,
// a ring of four 32 KiB stages, one barrier per K-tile.
// What bounds it: the copies.  A K-tile is 512 cycles of MFMAs per SIMD and 32 KiB, of which a CU takes in about 37 bytes a cycle (0.4 us); LDS reads
// (96 KiB) take 768 cycles.  So the stages are many rather than large, and operands are single: block by block the next K-tile's are read as this one's
// fall free, with the other wavefront of the SIMD under way.
constexpr int kSlimEdge = 128;
constexpr int kSlimStage = 2 * kSlimEdge * BK;          // 32 KiB: activations, then weights
constexpr int kSlimStages = 4;
constexpr int kSlimSa = kSlimStages * kSlimStage;       // activation scales: a row of 128 floats per stage
constexpr int kSlimSb = kSlimSa + kSlimStages * kSlimEdge * 4;      // weight-block scales: 2 tile parities x 256 floats
constexpr int kSlimOut = kSlimSb + 2 * kWideMaxKb * 4;  // 2 KiB per wavefront in which the output is turned round
constexpr int kSlimLds = kSlimOut + 8 * 2048;           // 151,552 bytes
// five copy instructions per wavefront and K-tile (2 activations, 2 weights, 1 scales)
constexpr int kSlimWaitVm10 = 0x0f7a, kSlimWaitVm15 = 0x0f7f;

__global__ __launch_bounds__(kWideThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_gemm_nt_block_slim(const GemmArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);      // 0..7
    const int wm = wave & 3, wn = wave >> 2;              // 32 rows x 64 columns
    const int ktiles = p.K / BK;          // >= 4, checked by the launcher
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
    auto tile_at = [&](int seq, int& m0, int& n0) {
        int tm, tn;
        tile_coords(lin0 + seq * lstep, p.tiles_m, p.tiles_n, tm, tn);
        m0 = tm * kSlimEdge;
        n0 = tn * kSlimEdge;
    };

    // ---- global -> LDS: wavefront w copies rows [16 w, 16 w + 16) of both operands and the scales of those activation rows ----
    const int lrow = lane >> 3, lslot = lane & 7;
    uint32_t xoff[2], woff[2], saoff = 0;
    const uint8_t* sbsrc = nullptr;
    auto aim = [&](int seq) {
        int m0, n0;
        tile_at(seq, m0, n0);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int row = wave * 16 + j * 8 + lrow;
            const uint32_t chunk = (lslot ^ swz_rows16(row)) * 16;
            xoff[j] = static_cast<uint32_t>(min(m0 + row, p.M - 1)) * static_cast<uint32_t>(p.lda) + chunk;
            woff[j] = static_cast<uint32_t>(n0 + row) * static_cast<uint32_t>(p.ldb) + chunk;        // N % 128 == 0
        }
        saoff = static_cast<uint32_t>(min(m0 + wave * 16 + (lane & 15), p.M - 1)) * static_cast<uint32_t>(ktiles) * 4u;
        sbsrc = reinterpret_cast<const uint8_t*>(p.sb + static_cast<size_t>(n0 >> 7) * ktiles);
    };
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem));
    auto dma16 = [&](uint32_t dst, uint32_t voff, const uint8_t* base) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(dst), "v"(voff), "s"(base) : "memory");
    };
    // by the low 16 lanes only; as in the kernel above
    auto dma4_lo16 = [&](uint32_t dst, uint32_t voff, const uint8_t* base) {
        asm volatile("s_mov_b32 m0, %0\n\ts_mov_b32 exec_lo, 0xffff\n\ts_mov_b32 exec_hi, 0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2\n\t"
                     "s_mov_b32 exec_lo, -1\n\ts_mov_b32 exec_hi, -1\n\ts_nop 0"
                     :: "s"(dst), "v"(voff), "s"(base) : "memory");
    };
    auto dma4 = [&](uint32_t dst, uint32_t voff, const uint8_t* base) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" :: "s"(dst), "v"(voff), "s"(base) : "memory");
    };
    // a stage's scale row begins at kSlimSa + stage / 64
    auto copy_one = [&](int stage, int kt, auto jc) {
        constexpr int J = decltype(jc)::value;
        if constexpr (J < 2)      dma16(lds0 + stage + (wave * 16 + J * 8) * BK, xoff[J], p.A + kt * BK);
        else if constexpr (J < 4) dma16(lds0 + stage + kSlimEdge * BK + (wave * 16 + (J - 2) * 8) * BK, woff[J - 2], p.B + kt * BK);
        else dma4_lo16(lds0 + kSlimSa + (stage >> 6) + wave * 64, saoff, reinterpret_cast<const uint8_t*>(p.sa + kt));
    };
    auto copy_sb = [&](int parity) {
        if (wave == 0) {
            for (int c = 0; c * 64 < ktiles; ++c) {
                const uint32_t v = static_cast<uint32_t>(min(c * 64 + lane, ktiles - 1)) * 4u;
                dma4(lds0 + kSlimSb + parity * (kWideMaxKb * 4) + c * 256, v, sbsrc);
            }
        }
    };

    const int r16 = lane & 15, kg = lane >> 4;
    int xat[2], wat[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int rd = r16 * BK + (((kg * 2 + c) ^ swz_rows16(r16)) << 4);
        xat[c] = wm * 32 * BK + rd;
        wat[c] = kSlimEdge * BK + wn * 64 * BK + rd;
    }
    v4f sum[4][2];                // [weight block][activation block]
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) sum[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    v8i W[4], X[2];
    v4f part[4];
    float f[2] = {0.0f, 0.0f}, fn[2];
    auto put = [](v8i& dst, int half, const uint4 v) {
        dst[4 * half + 0] = (int)v.x; dst[4 * half + 1] = (int)v.y; dst[4 * half + 2] = (int)v.z; dst[4 * half + 3] = (int)v.w;
    };
    auto read_w = [&](int stage, auto ic) {
        constexpr int I = decltype(ic)::value;
#pragma unroll
        for (int c = 0; c < 2; ++c) put(W[I], c, *reinterpret_cast<const uint4*>(smem + stage + wat[c] + I * 16 * BK));
    };
    auto read_x = [&](int stage) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int c = 0; c < 2; ++c) put(X[j], c, *reinterpret_cast<const uint4*>(smem + stage + xat[c] + j * 16 * BK));
    };
    auto fold = [&](auto nc) {
        constexpr int n = decltype(nc)::value, i = n >> 1, j = n & 1;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float v = __builtin_fmaf(part[n & 3][r], f[j], sum[i][j][r]);
            asm volatile("" : "+v"(v));         // here, not gathered at the end of the loop body
            sum[i][j][r] = v;
        }
    };
    auto read_factors = [&](int stage, int parity, int kt) {
        const float sbv = *reinterpret_cast<const float*>(smem + kSlimSb + parity * (kWideMaxKb * 4) + kt * 4);
#pragma unroll
        for (int j = 0; j < 2; ++j)
            fn[j] = *reinterpret_cast<const float*>(smem + kSlimSa + (stage >> 6) + (wm * 32 + j * 16 + r16) * 4) * sbv;
    };

    int s0 = 0;                   // stage of the current K-tile, whose operands are in registers
    // (nkt, npar): position and tile parity of the next K-tile; dkt: position of the one four on, whose copies go into this one's stage
    auto ktile = [&](auto first_c, int nkt, int npar, int dkt) {
        constexpr bool FIRST = decltype(first_c)::value != 0;
        const int s1 = (s0 + kSlimStage) & (kSlimStages * kSlimStage - 1);
        // the next K-tile has landed, and every wavefront has this one in registers
        __builtin_amdgcn_s_waitcnt(kSlimWaitVm10);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        static_for<0, 8>([&](auto nc) {
            constexpr int n = decltype(nc)::value, i = n >> 1, j = n & 1;
            part[n & 3] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(W[i], X[j], v4f{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0, 0, 0, 0);
            if constexpr (n >= 3) {
                fold(std::integral_constant<int, (n >= 3 ? n - 3 : 0)>{});
            } else if constexpr (!FIRST) {
                fold(std::integral_constant<int, 5 + n>{});
            }
            if constexpr (n == 2) {
                f[0] = fn[0];
                f[1] = fn[1];
            }
            if constexpr (n < 5) copy_one(s0, dkt, nc);
            if constexpr (n == 3) read_factors(s1, npar, nkt);
            if constexpr (j == 1) read_w(s1, std::integral_constant<int, i>{});
            __builtin_amdgcn_sched_barrier(0);
        });
        read_x(s1);
        __builtin_amdgcn_sched_barrier(0);
        s0 = s1;
    };

    // copy position: four K-tiles ahead of the compute position (ktiles >= 4, so at most one tile ahead); past the last tile the stream
    // re-reads that tile and what it copies is never used
    int dkt = 0, dseq = 0;
    auto advance_copy = [&]() {
        if (++dkt == ktiles) {
            dkt = 0;
            if (++dseq < my_tiles) aim(dseq);
            copy_sb(dseq & 1);
        }
    };
    aim(0);
    copy_sb(0);
    static_for<0, 4>([&](auto kc) {
        static_for<0, 5>([&](auto jc) { copy_one(decltype(kc)::value * kSlimStage, dkt, jc); });
        advance_copy();
    });
    __builtin_amdgcn_s_waitcnt(kSlimWaitVm15);
    __syncthreads();
    static_for<0, 4>([&](auto ic) { read_w(0, ic); });
    read_x(0);
    read_factors(0, 0, 0);

    uint8_t* stg = smem + kSlimOut + wave * 2048;
    for (int seq = 0; seq < my_tiles; ++seq) {
        const int parity = seq & 1;
        ktile(std::integral_constant<int, 1>{}, 1, parity, dkt);
        advance_copy();
        for (int kt = 1; kt < ktiles; ++kt) {
            const bool last = kt + 1 == ktiles;
            ktile(std::integral_constant<int, 0>{}, last ? 0 : kt + 1, last ? parity ^ 1 : parity, dkt);
            advance_copy();
        }
        static_for<5, 8>([&](auto nc) { fold(nc); });
        // out as in the kernel above
        int m0, n0;
        tile_at(seq, m0, n0);
        int lane_d = lane;
        asm volatile("" : "+v"(lane_d));
        const int row = lane_d & 15, cq = lane_d >> 4, rr = lane_d >> 3, rc = lane_d & 7;
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        uint16_t* cp = p.C + static_cast<size_t>(m0 + wm * 32) * p.ldc + n0 + wn * 64;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                v4f& v = sum[b][j];
                *reinterpret_cast<uint2*>(stg + row * 128 + (((b * 2 + (cq >> 1)) ^ ((row >> 1) & 7)) << 4) + (cq & 1) * 8) =
                    make_uint2(pack_bf16x2_hw(v[0], v[1]), pack_bf16x2_hw(v[2], v[3]));
                v = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int r = rr + 8 * t;
                const uint4 v = *reinterpret_cast<const uint4*>(stg + r * 128 + ((rc ^ ((r >> 1) & 7)) << 4));
                if (m0 + wm * 32 + j * 16 + r < p.M) {
                    const u32x4 vv = {v.x, v.y, v.z, v.w};
                    __builtin_nontemporal_store(vv, reinterpret_cast<u32x4*>(cp + static_cast<size_t>(j * 16 + r) * p.ldc + rc * 8));
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __builtin_amdgcn_s_waitcnt(kWideWaitVm0);
}

}  // namespace

bool block_wide_ok(const GemmArgs& p) {
    const int kb = p.K / BK;
    return p.K % BK == 0 && kb >= 3 && kb <= kWideMaxKb && p.N % BN == 0 && static_cast<size_t>(p.M) * p.lda < (1ull << 32) &&
           static_cast<size_t>(p.N) * p.ldb < (1ull << 32) && static_cast<size_t>(p.M) * kb * 4 < (1ull << 32) && p.ldc % 8 == 0 &&
           aligned16(p.C);
}

// Microseconds: 1.12 a K-tile and 10 a tile beside the 0.65 and 6 of k_gemm_nt_block_ring's 128 x 256 tiles.  Whole rounds: 186 against 210 (4096 x 7168
// x 7168), 61 against 68 (4096^3), 93 against 104 (2048 x 7168 x 7168).  Where the large tiles leave a round nearly empty or half of the CUs
// without one the small ones stay: 169 against 154 (2560 x 7168 x 7168, 1.1 rounds and 2.2), 78 against 60 (4096 x 2048 x 7168, half a round and one).
// With few K-tiles the fixed part decides.  At 6 these went to the large ones: 3000 x 7168 x 2048 54.5 against 48.2, 2892 x 11008 x 640 34.9 and 27.7,
// 3644 x 5888 x 1536 44.1 and 38.4; 3500 x 7168 x 2048 still does, 54.2 against 63.0.  Of 1400 sizes (K 384 to 9000) 44 of 900 were slower than before these
// kernels by more than 3 %, the worst 1.19 times; now 3 of 500 are, all with K 512 to 768.
float block_wide_estimate_us(const GemmArgs& p) {
    const long long tiles = static_cast<long long>((p.M + BM - 1) / BM) * (p.N / BN);
    const int cus = num_cus();
    return static_cast<float>((tiles + cus - 1) / cus) * (static_cast<float>(p.K / BK) * 1.12f + 10.0f);
}

int gemm_nt_block_wide(GemmArgs p, hipStream_t st) {
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [] {
        err = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm_nt_block_wide), hipFuncAttributeMaxDynamicSharedMemorySize, kWideLds);
    });
    if (err != hipSuccess) return static_cast<int>(err);
    p.tiles_m = (p.M + BM - 1) / BM;
    p.tiles_n = p.N / BN;
    k_gemm_nt_block_wide<<<persistent_grid(p.tiles_m * p.tiles_n, num_cus()), kWideThreads, kWideLds, st>>>(p);
    return launch_status();
}

bool block_slim_ok(const GemmArgs& p) {
    const int kb = p.K / BK;
    return p.K % BK == 0 && kb >= kSlimStages && kb <= kWideMaxKb && p.N % kSlimEdge == 0 && static_cast<size_t>(p.M) * p.lda < (1ull << 32) &&
           static_cast<size_t>(p.N) * p.ldb < (1ull << 32) && static_cast<size_t>(p.M) * kb * 4 < (1ull << 32) && p.ldc % 8 == 0 &&
           aligned16(p.C);
}

// Microseconds: 0.50 a K-tile and 6 a tile.  Quantize and product, before and with these tiles: 2048 x 7168 over K 2048, 350 rows 20.6 and 15.8, 512 21.4 and
// 16.5; 4096 x 4096, 512 rows 27.8 (K split over wavefronts) and 25.1, 700 35.9 (128 x 256 tiles) and 27.0, 1000 38.1 and 29.7; 2048 columns over K 7168, 1400 rows
// 65.1 and 48.2, 2048 68.2 and 51.4; 7168 x 7168, 512 rows 59.7 and 43.3.  In a second round the larger tiles have it: 7168 x 7168, 700 rows 61.1 and
// 70.7.  Columns that the larger ones do not take (N % 256 = 128, the register-staged kernel before): 600 x 8576 over 2048 38.4 and 24.6, 4096 x 4224 over
// 4096 185 and 108.  The K-splitting ones stay where K is long: 2048 columns over K 7168, 700 rows 42.5 and 43.2, 1000 44.2 and 45.4.
float block_slim_estimate_us(const GemmArgs& p) {
    const long long tiles = static_cast<long long>((p.M + kSlimEdge - 1) / kSlimEdge) * (p.N / kSlimEdge);
    const int cus = num_cus();
    return static_cast<float>((tiles + cus - 1) / cus) * (static_cast<float>(p.K / BK) * 0.50f + 6.0f);
}

int gemm_nt_block_slim(GemmArgs p, hipStream_t st) {
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [] {
        err = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm_nt_block_slim), hipFuncAttributeMaxDynamicSharedMemorySize, kSlimLds);
    });
    if (err != hipSuccess) return static_cast<int>(err);
    p.tiles_m = (p.M + kSlimEdge - 1) / kSlimEdge;
    p.tiles_n = p.N / kSlimEdge;
    k_gemm_nt_block_slim<<<persistent_grid(p.tiles_m * p.tiles_n, num_cus()), kWideThreads, kSlimLds, st>>>(p);
    return launch_status();
}

}  // namespace cf
