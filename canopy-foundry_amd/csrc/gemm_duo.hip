// The persistent FP8 GEMM at half the tile edge, two workgroups per CU:
//     C[M,N] = epilogue( (A[M,K] * sa) . (B[N,K] * sb)^T ),   or   C += that  (fp32 or bf16 C).
//
// Workgroup tile 128 x 128 x 128, four wavefronts 2 x 2, each 64 x 64 = 2 x 2 tiles of v_mfma_f32_32x32x64_f8f6f4 (64
// accumulator registers), a ring of five 16 KiB slots: 80 KiB, so a CU holds TWO workgroups and every SIMD two wavefronts.  The
// price is twice the LDS and L2 bytes per FLOP of the 256 x 256 tile: a K-tile takes 0.44 us where the CU's two workgroups share
// the matrix cores (0.24 at the 256 x 256 kernel's rate), what the L2s deliver being the limit.  Two kinds of problem gain:
//   - too few 256 x 256 tiles to fill the chip (4096 columns, 1000 rows, K 4096: 38 -> 19 us; 2048 rows, K 14336: 123 -> 98);
//   - the accumulating forms over a short K: while one workgroup of a CU adds its tile to what C holds, the other multiplies.
//     With one workgroup per CU all of them multiply and all of them wait for memory in turn.  14336 x 4096 fp32 (470 MB read
//     and written, 85 us): K 1024 126 -> 108 us, K 2048 164 -> 147, K 2000 262 (register-staged kernel) -> 188 (164 in gemm_accum.hip, which has
//     the longer K that are no multiple of 128), K 4096 240 -> 250.
// Operand rows and bytes of K beyond the operands are read as zeros (buffer copies with the operand's size in their
// descriptor), so K only has to be a multiple of 16.
#include "gemm_common.hpp"

#include <mutex>

namespace cf {
namespace {

constexpr int DM = 128;
constexpr int kSlots = 5;
constexpr int kDuoSlot = DM * BK;                  // 16 KiB
constexpr int kDuoLds = kSlots * kDuoSlot;         // 80 KiB
constexpr int kThreads = 256;
// s_waitcnt immediates: vmcnt in bits [3:0] and [15:14], the other counters left at no-wait
constexpr int kWaitVm0 = 0x0f70, kWaitVm4 = 0x0f74, kWaitVm8 = 0x0f78;

// FMT bit 0: A is E5M2, bit 1: B is E5M2.  KTAIL: K is not a multiple of 128.
template <int FMT, int EPI, int SCALE, bool KTAIL>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_gemm_nt_duo(const GemmArgs p, const int stagger) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    constexpr bool GATE = EPI == EPI_SILU_GATE;
    constexpr bool ACCUM = EPI == EPI_ACCUM_F32 || EPI == EPI_ACCUM_BF16;
    constexpr int OUT_BN = GATE ? DM / 2 : DM;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
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
    const int ktiles = (p.K + BK - 1) / BK;      // >= 2, checked by the launcher

    if (stagger) {
        // the second workgroup of a CU (its LDS starts above the first one's) waits about half a tile's MFMA time
        unsigned alloc;
        asm volatile("s_getreg_b32 %0, hwreg(HW_REG_LDS_ALLOC, 0, 12)" : "=s"(alloc));
        if (alloc != 0) {
            for (int i = 0; i < (ktiles + 15) / 16; ++i) __builtin_amdgcn_s_sleep(127);
        }
    }

    auto tile_at = [&](int seq, int& m0, int& n0) {
        int tm, tn;
        tile_coords(lin0 + seq * lstep, p.tiles_m, p.tiles_n, tm, tn);
        m0 = tm * DM;
        n0 = tn * OUT_BN;
    };

    // ---- global -> LDS: wave w copies rows [32w, 32w+32) of an operand tile, 8 rows per instruction ----
    // A descriptor per operand; a row at or beyond the operand's last gets the offset of the descriptor's end.
    typedef int s32x4 __attribute__((ext_vector_type(4)));
    auto descriptor = [](const uint8_t* base, uint32_t bytes) {
        const uint64_t a = reinterpret_cast<uint64_t>(base);
        return s32x4{__builtin_amdgcn_readfirstlane(static_cast<int>(a)),
                     __builtin_amdgcn_readfirstlane(static_cast<int>((a >> 32) & 0xffffu)),
                     __builtin_amdgcn_readfirstlane(static_cast<int>(bytes)), 0x00020000};
    };
    const s32x4 xrs = descriptor(p.A, static_cast<uint32_t>(p.M) * static_cast<uint32_t>(p.lda));
    // SiLU-gate: the W tile's rows are [gate 32 | up 32] for the columns of wavefront column 0, then the same for
    // column 1, so wave w copies from one matrix only: gate for even w, up for odd w
    const s32x4 wrs = descriptor((GATE && (wave & 1)) ? p.B2 : p.B, static_cast<uint32_t>(p.N) * static_cast<uint32_t>(p.ldb));
    const int lrow = lane >> 3, lslot = lane & 7;
    uint32_t xoff[4], woff[4];
    auto aim = [&](int seq) {
        int m0, n0;
        tile_at(seq, m0, n0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = wave * 32 + j * 8 + lrow;
            const uint32_t gchunk = (lslot ^ swz(row)) * 16;
            xoff[j] = static_cast<uint32_t>(min(m0 + row, p.M)) * static_cast<uint32_t>(p.lda) + gchunk;
            const int n = GATE ? n0 + (row >> 6) * 32 + (row & 31) : n0 + row;
            woff[j] = static_cast<uint32_t>(min(n, p.N)) * static_cast<uint32_t>(p.ldb) + gchunk;
        }
    };
    // the last K-tile of a tile whose K ends inside it: lanes whose 16 bytes lie beyond K are sent past the descriptors' ends
    auto clip = [&]() {
        const uint32_t left = static_cast<uint32_t>(p.K - (ktiles - 1) * BK);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t gchunk = (lslot ^ swz(wave * 32 + j * 8 + lrow)) * 16;
            const uint32_t out = gchunk < left ? 0u : 0x80000000u;
            xoff[j] |= out;
            woff[j] |= out;
        }
    };
    uint32_t lds_wave = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem)) + wave * (32 * BK);
    auto dma = [&](int slot, uint32_t voff, const s32x4& rs, int k0, auto jc) {
        constexpr int J = decltype(jc)::value;
        const uint32_t dst = lds_wave + slot;
        asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds"
                     :: "s"(dst), "n"(J * 8 * BK), "v"(voff), "s"(rs), "s"(k0) : "memory", "scc");
    };
    auto dma_x = [&](int slot, int k0, auto jc) { dma(slot, xoff[decltype(jc)::value], xrs, k0, jc); };
    auto dma_w = [&](int slot, int k0, auto jc) { dma(slot, woff[decltype(jc)::value], wrs, k0, jc); };

    // ---- LDS -> MFMA operands ----
    const int frow = lane & 31, khalf = lane >> 5, fs = swz(frow);
    int rd[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 2; ++j) rd[h][j] = frow * BK + (((h * 4 + khalf * 2 + j) ^ fs) << 4);
    const uint8_t* xrd = smem + wm * 64 * BK;
    const uint8_t* wrd = smem + wn * 64 * BK;

    v16f acc[2][2];       // [weight tile][activation tile]
    v8i wq[2][2], xq[2][2];
    auto put = [](v8i& dst, int half, const uint4 v) {
        dst[4 * half + 0] = (int)v.x; dst[4 * half + 1] = (int)v.y; dst[4 * half + 2] = (int)v.z; dst[4 * half + 3] = (int)v.w;
    };
    // read I (0..7) of k-half H: w0 x0 x1 w1, two reads each
    auto read_one = [&](int sx, int sw, auto hc, auto ic) {
        constexpr int H = decltype(hc)::value, I = decltype(ic)::value;
        constexpr int t = I >> 1, half = I & 1;
        const int r = rd[H][half];
        if constexpr (t == 0)      put(wq[H][0], half, *reinterpret_cast<const uint4*>(wrd + sw + r));
        else if constexpr (t <= 2) put(xq[H][t - 1], half, *reinterpret_cast<const uint4*>(xrd + sx + (t - 1) * 32 * BK + r));
        else                       put(wq[H][1], half, *reinterpret_cast<const uint4*>(wrd + sw + 32 * BK + r));
    };
    auto mfma_one = [&](auto hc, auto ic, auto first_c) {
        constexpr int H = decltype(hc)::value, I = decltype(ic)::value;
        constexpr int a = I >> 1, b = I & 1;
        v16f c = acc[a][b];
        if constexpr (decltype(first_c)::value != 0) {
#pragma unroll
            for (int r = 0; r < 16; ++r) c[r] = 0.0f;
        }
        acc[a][b] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wq[H][a], xq[H][b], c, (FMT >> 1) & 1, FMT & 1, 0, 0, 0, 0);
    };
    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;

    int a0 = 0, a1 = kDuoSlot, a2 = 2 * kDuoSlot, a3 = 3 * kDuoSlot, a4 = 4 * kDuoSlot;

    // What the drain needs in registers, fetched under the tile's last MFMAs.  bf16 outputs: row descales of this lane's two
    // output rows and the channel descales of its columns (plain: cs[a][g] = four columns of quad g of weight tile a; SiLU-gate:
    // cs[0][g] gate, cs[1][g] up).  Accumulating forms: this lane's part of C, four columns of four rows per 32 x 32 block.
    float sa[2] = {1.0f, 1.0f};
    float4 cs[2][4];
    float s1 = 0.0f, s2 = 0.0f;
    if constexpr (SCALE == SCALE_TENSOR) {
        s1 = p.sa[0] * p.sb[0];
        if constexpr (GATE) s2 = p.sa[0] * p.sb2[0];
    }
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    constexpr bool OUT_BF16 = EPI != EPI_ACCUM_F32;
    constexpr uint32_t ES = OUT_BF16 ? 2u : 4u;                 // bytes per element of C
    using Raw = std::conditional_t<OUT_BF16, u32x2, f32x4>;
    Raw old[ACCUM ? 4 : 1][4];
    const int rr = lane >> 3, rc = lane & 7;
    auto c_at = [&](int m, int n) -> uint8_t* {
        const size_t at = static_cast<size_t>(m) * p.ldc + n;
        return OUT_BF16 ? reinterpret_cast<uint8_t*>(p.C + at) : reinterpret_cast<uint8_t*>(p.Cf + at);
    };
    auto load_scales = [&](int m0, int n0) {
        if constexpr (ACCUM) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int b = k >> 1, a = k & 1, col = n0 + wn * 64 + a * 32 + rc * 4;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int row = m0 + wm * 64 + b * 32 + i * 8 + rr;
                    // clamped, not skipped: a load under a condition would be waited for on the spot
                    old[k][i] = __builtin_nontemporal_load(reinterpret_cast<const Raw*>(c_at(min(row, p.M - 1), min(col, p.N - 4))));
                }
            }
        }
        if constexpr (SCALE == SCALE_ROWCOL) {
#pragma unroll
            for (int b = 0; b < 2; ++b) sa[b] = p.sa[min(m0 + wm * 64 + b * 32 + (lane & 31), p.M - 1)];
            if constexpr (GATE) {
                const int col = n0 + wn * 32 + khalf * 4;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    cs[0][g] = *reinterpret_cast<const float4*>(p.sb + col + g * 8);
                    cs[1][g] = *reinterpret_cast<const float4*>(p.sb2 + col + g * 8);
                }
            } else {
                const int col = n0 + wn * 64 + khalf * 4;
#pragma unroll
                for (int a = 0; a < 2; ++a)
#pragma unroll
                    for (int g = 0; g < 4; ++g) cs[a][g] = *reinterpret_cast<const float4*>(p.sb + min(col + a * 32 + g * 8, p.N - 4));
            }
        }
    };

    auto ktile = [&](auto first_c, auto end_c, int dk0, int m0, int n0, bool wait) {
        constexpr bool END = decltype(end_c)::value != 0;
        // step (g,0): 4 MFMAs, the operand reads of (g,1), the copies of X(g+2)
        static_for<0, 4>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            mfma_one(C0{}, ic, first_c);
            read_one(a0, a1, C1{}, std::integral_constant<int, 2 * i>{});
            read_one(a0, a1, C1{}, std::integral_constant<int, 2 * i + 1>{});
            dma_x(a4, dk0, ic);
            __builtin_amdgcn_sched_barrier(0);
        });
        // step (g,1)
        mfma_one(C1{}, C0{}, C0{});
        __builtin_amdgcn_sched_barrier(0);
        if (wait) __builtin_amdgcn_s_waitcnt(kWaitVm4);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        static_for<1, 4>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            mfma_one(C1{}, ic, C0{});
            if constexpr (!END) {
                static_for<0, 3>([&](auto jc) {
                    constexpr int j = (i - 1) * 3 + decltype(jc)::value;
                    if constexpr (j < 8) read_one(a2, a3, C0{}, std::integral_constant<int, j < 8 ? j : 0>{});
                });
            }
            if constexpr (i == 1) { dma_w(a0, dk0, C0{}); dma_w(a0, dk0, C1{}); }
            if constexpr (i == 2) dma_w(a0, dk0, std::integral_constant<int, 2>{});
            if constexpr (i == 3) dma_w(a0, dk0, std::integral_constant<int, 3>{});
            if constexpr (END && i == 1) load_scales(m0, n0);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto rotate = [&]() {
        const int b0 = a0, b1 = a1;
        a0 = a2; a1 = a3; a2 = a4; a3 = b0; a4 = b1;
    };

    // copy position: two K-tiles ahead of the compute position; past the last tile the stream re-reads that tile
    int dkt = 2 % ktiles, dseq = 2 / ktiles;
    aim(0);
    static_for<0, 4>([&](auto jc) { dma_x(a0, 0, jc); });
    static_for<0, 4>([&](auto jc) { dma_w(a1, 0, jc); });
    if (KTAIL && ktiles == 2) clip();
    static_for<0, 4>([&](auto jc) { dma_x(a2, BK, jc); });
    static_for<0, 4>([&](auto jc) { dma_w(a3, BK, jc); });
    if (dseq == 1) aim(my_tiles > 1 ? 1 : 0);
    if (KTAIL && dkt == ktiles - 1) clip();
    __builtin_amdgcn_s_waitcnt(kWaitVm8);
    __syncthreads();
    static_for<0, 8>([&](auto ic) { read_one(a0, a1, C0{}, ic); });

    auto advance_copy = [&]() {
        if (++dkt == ktiles) {
            dkt = 0;
            if (++dseq < my_tiles) aim(dseq);
            else if (KTAIL) aim(my_tiles - 1);       // the re-read starts from unclipped offsets again
        }
        if (KTAIL && dkt == ktiles - 1) clip();
    };

    for (int seq = 0; seq < my_tiles; ++seq) {
        int m0, n0;
        tile_at(seq, m0, n0);
        ktile(C1{}, C0{}, dkt * BK, m0, n0, seq == 0);
        rotate(); advance_copy();
        for (int kt = 1; kt + 1 < ktiles; ++kt) {
            ktile(C0{}, C0{}, dkt * BK, m0, n0, true);
            rotate(); advance_copy();
        }
        ktile(C0{}, C1{}, dkt * BK, m0, n0, true);
        rotate(); advance_copy();

        // ---- drain: a4 is free until this workgroup's own copies of the stream's next K-tile but one ----
        const int row = lane & 31;
        const int wswz = (row >> 1) & 7;
        if constexpr (ACCUM) {
            // per 32 x 32 block: scaled, parked as 32 rows x 128 bytes of fp32 in this wavefront's own 4 KiB, read back four
            // columns of a row per lane, added to what C holds and stored: whole 128-byte (bf16: 64-byte) pieces
            uint8_t* stage = smem + a4 + wave * (32 * BK);
            uint8_t* wr = stage + row * 128;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int b = k >> 1, a = k & 1;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    float4 v;
                    v.x = acc[a][b][g * 4 + 0] * s1; v.y = acc[a][b][g * 4 + 1] * s1;
                    v.z = acc[a][b][g * 4 + 2] * s1; v.w = acc[a][b][g * 4 + 3] * s1;
                    *reinterpret_cast<float4*>(wr + (((g * 2 + khalf) ^ (row & 7)) << 4)) = v;
                }
                __builtin_amdgcn_sched_barrier(0);
                if (k == 0) __builtin_amdgcn_s_waitcnt(kWaitVm0);
                const int col = n0 + wn * 64 + a * 32 + rc * 4;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int r = i * 8 + rr, m = m0 + wm * 64 + b * 32 + r;
                    const float4 v = *reinterpret_cast<const float4*>(stage + r * 128 + ((rc ^ (r & 7)) << 4));
                    const Raw c = old[k][i];
                    if (m < p.M && col < p.N) {
                        if constexpr (OUT_BF16) {
                            const u32x2 o = {pack_bf16x2_hw(v.x + bf16_lo(c[0]), v.y + bf16_hi(c[0])),
                                             pack_bf16x2_hw(v.z + bf16_lo(c[1]), v.w + bf16_hi(c[1]))};
                            __builtin_nontemporal_store(o, reinterpret_cast<u32x2*>(c_at(m, col)));
                        } else {
                            const f32x4 o = {c[0] + v.x, c[1] + v.y, c[2] + v.z, c[3] + v.w};
                            __builtin_nontemporal_store(o, reinterpret_cast<f32x4*>(c_at(m, col)));
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        } else if constexpr (GATE) {
            // the two wavefronts of a row half share 64 rows x 128 bytes: each writes the 64 bytes per row of its 32
            // output columns, then (barrier) each streams out 32 whole rows
            uint8_t* stage = smem + a4 + wm * (64 * 128);
            uint8_t* wr = stage + row * 128 + khalf * 8;
#pragma unroll
            for (int b = 0; b < 2; ++b) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    float4 c = make_float4(s1, s1, s1, s1), u = make_float4(s2, s2, s2, s2);
                    if constexpr (SCALE == SCALE_ROWCOL) { c = cs[0][g]; u = cs[1][g]; }
                    const float c4[4] = {c.x, c.y, c.z, c.w}, u4[4] = {u.x, u.y, u.z, u.w};
                    float v[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        // the reference rounds gate and up to bf16 before the SiLU product
                        const uint32_t gu = pack_bf16x2_hw(acc[0][b][g * 4 + q] * (sa[b] * c4[q]), acc[1][b][g * 4 + q] * (sa[b] * u4[q]));
                        v[q] = fast_silu(bf16_lo(gu)) * bf16_hi(gu);
                    }
                    *reinterpret_cast<uint2*>(wr + b * 32 * 128 + (((wn * 4 + g) ^ wswz) << 4)) =
                        make_uint2(pack_bf16x2_hw(v[0], v[1]), pack_bf16x2_hw(v[2], v[3]));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            // every copy in flight is waited for before the first store (stores and copies share one counter); the tile
            // that follows skips the wait of its first K-tile
            __builtin_amdgcn_s_waitcnt(kWaitVm0);
            __syncthreads();
            const uint8_t* rdp0 = stage + (wn * 32 + rr) * 128 + ((rc ^ (rr >> 1)) << 4);
            const uint8_t* rdp1 = stage + (wn * 32 + rr) * 128 + ((rc ^ (rr >> 1) ^ 4) << 4);
            uint8_t* cu = reinterpret_cast<uint8_t*>(p.C + static_cast<size_t>(m0 + wm * 64 + wn * 32) * p.ldc + n0);
            const uint32_t coff = (static_cast<uint32_t>(rr) * static_cast<uint32_t>(p.ldc) + rc * 8u) * 2u;
            const size_t cstep = static_cast<size_t>(p.ldc) * 16;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint4 v = *reinterpret_cast<const uint4*>(((i & 1) ? rdp1 : rdp0) + i * 8 * 128);
                if (m0 + wm * 64 + wn * 32 + rr + i * 8 < p.M) {
                    const u32x4 vv = {v.x, v.y, v.z, v.w};
                    __builtin_nontemporal_store(vv, reinterpret_cast<u32x4*>(cu + i * cstep + coff));
                }
            }
        } else {
            // per 32 output rows: 32 rows x 128 bytes in this wavefront's own 4 KiB, then out as whole lines
            uint8_t* stage = smem + a4 + wave * (32 * BK);
            uint8_t* wr = stage + row * 128 + khalf * 8;
            const uint8_t* rdp0 = stage + rr * 128 + ((rc ^ (rr >> 1)) << 4);
            const uint8_t* rdp1 = stage + rr * 128 + ((rc ^ (rr >> 1) ^ 4) << 4);
            uint8_t* cu = reinterpret_cast<uint8_t*>(p.C + static_cast<size_t>(m0 + wm * 64) * p.ldc + n0 + wn * 64);
            const uint32_t coff = (static_cast<uint32_t>(rr) * static_cast<uint32_t>(p.ldc) + rc * 8u) * 2u;
            const size_t cstep = static_cast<size_t>(p.ldc) * 16;
            const int ncol = n0 + wn * 64 + rc * 8;             // N is a multiple of 8: a lane's columns are in or out together
            uint4 bv = make_uint4(0, 0, 0, 0);
            if constexpr (EPI == EPI_BIAS) bv = *reinterpret_cast<const uint4*>(p.bias + min(ncol, p.N - 8));
            const float bf[8] = {bf16_lo(bv.x), bf16_hi(bv.x), bf16_lo(bv.y), bf16_hi(bv.y),
                                 bf16_lo(bv.z), bf16_hi(bv.z), bf16_lo(bv.w), bf16_hi(bv.w)};
#pragma unroll
            for (int b = 0; b < 2; ++b) {
#pragma unroll
                for (int a = 0; a < 2; ++a)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        float4 c = make_float4(s1, s1, s1, s1);
                        if constexpr (SCALE == SCALE_ROWCOL) c = cs[a][g];
                        const float c4[4] = {c.x, c.y, c.z, c.w};
                        float v[4];
#pragma unroll
                        for (int q = 0; q < 4; ++q) v[q] = acc[a][b][g * 4 + q] * (sa[b] * c4[q]);
                        *reinterpret_cast<uint2*>(wr + (((a * 4 + g) ^ wswz) << 4)) =
                            make_uint2(pack_bf16x2_hw(v[0], v[1]), pack_bf16x2_hw(v[2], v[3]));
                    }
                __builtin_amdgcn_sched_barrier(0);
                if (b == 0) __builtin_amdgcn_s_waitcnt(kWaitVm0);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    uint4 v = *reinterpret_cast<const uint4*>(((i & 1) ? rdp1 : rdp0) + i * 8 * 128);
                    if constexpr (EPI == EPI_BIAS) {            // added to the bf16 result, as the separate kernel does
                        v.x = pack_bf16x2_hw(bf16_lo(v.x) + bf[0], bf16_hi(v.x) + bf[1]);
                        v.y = pack_bf16x2_hw(bf16_lo(v.y) + bf[2], bf16_hi(v.y) + bf[3]);
                        v.z = pack_bf16x2_hw(bf16_lo(v.z) + bf[4], bf16_hi(v.z) + bf[5]);
                        v.w = pack_bf16x2_hw(bf16_lo(v.w) + bf[6], bf16_hi(v.w) + bf[7]);
                    }
                    if (m0 + wm * 64 + b * 32 + rr + i * 8 < p.M && ncol < p.N) {
                        const u32x4 vv = {v.x, v.y, v.z, v.w};
                        __builtin_nontemporal_store(vv, reinterpret_cast<u32x4*>(cu + (b * 4 + i) * cstep + coff));
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        static_for<0, 8>([&](auto ic) { read_one(a0, a1, C0{}, ic); });
    }
    __builtin_amdgcn_s_waitcnt(kWaitVm0);
}

template <int FMT, int EPI, int SCALE, bool KTAIL>
int launch(GemmArgs p, hipStream_t st) {
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [] {
        err = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm_nt_duo<FMT, EPI, SCALE, KTAIL>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, kDuoLds);
    });
    if (err != hipSuccess) return static_cast<int>(err);
    constexpr int out_bn = EPI == EPI_SILU_GATE ? DM / 2 : DM;
    p.tiles_m = (p.M + DM - 1) / DM;
    p.tiles_n = (p.N + out_bn - 1) / out_bn;
    const int grid = persistent_grid(p.tiles_m * p.tiles_n, 2 * num_cus());
    k_gemm_nt_duo<FMT, EPI, SCALE, KTAIL><<<grid, kThreads, kDuoLds, st>>>(p, p.duo == 1);
    return launch_status();
}
template <int FMT, int EPI, int SCALE>
int launch_k(const GemmArgs& p, hipStream_t st) {
    return p.K % BK == 0 ? launch<FMT, EPI, SCALE, false>(p, st) : launch<FMT, EPI, SCALE, true>(p, st);
}
template <int FMT, int SCALE>
int launch_plain(const GemmArgs& p, int epi, hipStream_t st) {
    return epi == EPI_BIAS ? launch_k<FMT, EPI_BIAS, SCALE>(p, st) : launch_k<FMT, EPI_NONE, SCALE>(p, st);
}

}  // namespace

bool duo_ok(const GemmArgs& p, int fmt, int epi, int scale_mode) {
    // offsets travel in 32 bits with the top one marking "outside"
    if (p.tile_map || p.K % 16 != 0 || p.K <= BK || static_cast<size_t>(p.M + DM) * p.lda >= (1ull << 31) ||
        static_cast<size_t>(p.N + DM) * p.ldb >= (1ull << 31))
        return false;
    if (epi == EPI_ACCUM_F32 || epi == EPI_ACCUM_BF16)
        return fmt == 2 && scale_mode == SCALE_TENSOR && p.N % 4 == 0 && p.ldc % 4 == 0 &&
               (epi == EPI_ACCUM_F32 ? aligned16(p.Cf) : (reinterpret_cast<uintptr_t>(p.C) & 7u) == 0);
    if (fmt > 1 || scale_mode > SCALE_ROWCOL || p.ldc % 8 != 0 || !aligned16(p.C) || (scale_mode == SCALE_ROWCOL && !aligned16(p.sb))) return false;
    if (epi == EPI_SILU_GATE)
        return fmt == 0 && p.N % (DM / 2) == 0 && (scale_mode == SCALE_TENSOR || aligned16(p.sb2));
    return p.N % 8 == 0 && (epi != EPI_BIAS || aligned16(p.bias));
}

// Microseconds: 0.48 a K-tile where a CU holds one workgroup (0.62 with the SiLU gate), 0.875 for both where it holds two, less where
// only some CUs hold two and there is one round (measured, 4096 columns, K 4096 to 14336: 288 workgroups 0.70 to 0.74, 384 0.77 to 0.80, 448 0.82); a third more where K is no multiple of 128 and a row's 128-byte pieces therefore
// lie across lines.  Per round of tiles 2.5 for the fill and the bf16 store (hidden in a last round that follows others), 3 for
// those and the SiLU gate's arithmetic (1.2 there).  512 x 2 x 14336 over K 1024, a round and three quarters: 26.0 us, 20.8 in
// the ring kernel; 1500 x 2 x 4096: 16.5, 19.1.
// Accumulating forms, per round: 8 for what is left of adding to an fp32 C under the other workgroup's MFMAs, 5.5 to a bf16 C,
// whose 64-byte pieces are half lines; more where the rows of C do not begin at lines.  So a short K and a bf16 C stay with
// the ring kernel (+= bf16 4096 x 4096: K 256 21.8 us there, 29.2 here; 4096 x 14336: K 512 74.2, 85.6), as do rows off the
// lines (fp32 4096 x 14336, ldc + 4, K 512: 191, 222); few tiles come here (fp32 1024 x 4096, K 1024: 24.1, 13.5).  One
// shape is still misjudged: fp32 4096 x 8192, K up to 512, whose two whole rounds take the ring 70 us, this kernel 75.
float duo_estimate_us(const GemmArgs& p, int epi) {
    const int out_bn = epi == EPI_SILU_GATE ? DM / 2 : DM, most = num_cus();
    const long long wgs = static_cast<long long>((p.M + DM - 1) / DM) * ((p.N + out_bn - 1) / out_bn);
    const long long full = wgs / (2 * most), rest = wgs % (2 * most);
    const float kt = static_cast<float>((p.K + BK - 1) / BK) * (p.K % BK ? 1.33f : 1.0f);
    const bool gate = epi == EPI_SILU_GATE, accum = epi == EPI_ACCUM_F32 || epi == EPI_ACCUM_BF16;
    const float tile = epi == EPI_ACCUM_F32 ? (c_lines_shared(p, 4) ? 14.0f : 8.0f) : epi == EPI_ACCUM_BF16 ? (c_lines_shared(p, 2) ? 6.2f : 5.5f)
                     : gate ? 3.0f : 2.5f;
    const float two = accum || full > 0 || p.M <= DM ? 0.875f : 0.70f + 0.175f * static_cast<float>(rest - most) / static_cast<float>(most);
    const float last = full == 0 || accum ? tile : gate ? 1.2f : 0.0f;
    return static_cast<float>(full) * (kt * 0.875f + tile) + (rest == 0 ? 0.0f : kt * (rest > most ? two : gate ? 0.62f : 0.48f) + last);
}

int gemm_nt_duo(GemmArgs p, int fmt, int epi, int scale_mode, hipStream_t st) {
    if (epi == EPI_ACCUM_F32) return launch_k<2, EPI_ACCUM_F32, SCALE_TENSOR>(p, st);
    if (epi == EPI_ACCUM_BF16) return launch_k<2, EPI_ACCUM_BF16, SCALE_TENSOR>(p, st);
    if (epi == EPI_SILU_GATE)
        return scale_mode == SCALE_TENSOR ? launch_k<0, EPI_SILU_GATE, SCALE_TENSOR>(p, st) : launch_k<0, EPI_SILU_GATE, SCALE_ROWCOL>(p, st);
    if (fmt == 1) return scale_mode == SCALE_TENSOR ? launch_plain<1, SCALE_TENSOR>(p, epi, st) : launch_plain<1, SCALE_ROWCOL>(p, epi, st);
    return scale_mode == SCALE_TENSOR ? launch_plain<0, SCALE_TENSOR>(p, epi, st) : launch_plain<0, SCALE_ROWCOL>(p, epi, st);
}

}  // namespace cf
