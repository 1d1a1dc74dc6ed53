// FP8 GEMM on small tiles, K split over a workgroup's wavefronts:
//     C[M,N] = epilogue( (A[M,K] * sa) . (B[N,K] * sb)^T )  for few rows, few tiles or few rows per expert.
//
// The persistent kernels of gemm.hip stage 256 x 256 tiles through LDS, one workgroup per tile: a decode batch of 16 rows
// against a [4096, 14336] weight is 16 tiles, so 240 of the 256 CUs idle and each of the others streams 3.7 MB of weights
// alone (108 us).  Here a workgroup owns a small output tile and its four wavefronts split K: wavefront w takes K-tiles w,
// w + 4, w + 8, ... of 128 bytes and copies their operand rows to LDS for itself alone, so that nothing synchronises inside
// the K loop; the fp32 partial sums are added through LDS at the end, in wavefront order.
//
// What bounds it.  Few rows: HBM (16 rows: 10.9 us, the 58.7 MB weight at 5.4 TB/s; 64 rows 13.4 us).  More rows: what the
// eight L2s deliver, about 24 TB/s here, 93 KB per microsecond and CU, whatever the tile: 256 rows 24 us, 512 rows 36 us,
// 1000 rows 53 us (256 x 256 tiles: 108-110 us throughout).  So the rule is the largest tile that still gives every CU one.
// Reading the operands from memory straight into registers was built first: a lane's MFMA row is lane % 16, so 16 consecutive
// lanes read 16 different lines, and the same L2s delivered 8.6 TB/s (16 rows 15.0 us, 256 rows 52 us).  Copies to LDS take
// whole 128-byte lines, eight lanes each.
#include "gemm_common.hpp"

#include <mutex>

namespace cf {
namespace {

// vmcnt(n), the other counters left alone
constexpr int wait_vm(int n) { return 0x0f70 | (n & 15) | ((n >> 4) << 14); }
constexpr int kWaitLgkm0 = 0xc07f;

template <int FMT, bool GATE, bool BLOCK, bool GROUPED, int MB, int NB, int WK, int S>
// BLOCK: two wavefronts per SIMD at most 256 registers each, so that the products land where the vector ALU can fold them
__global__ __launch_bounds__(64 * WK) __attribute__((amdgpu_waves_per_eu(BLOCK ? 2 : 1)))
void k_gemm_nt_direct(const GemmArgs p, const int rowcol, const int bias, const int c_vec) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    constexpr int NT = GATE ? 2 * NB : NB;          // weight blocks: NB gate blocks, then NB up blocks
    constexpr int TM = 16 * MB, TN = 16 * NB;
    constexpr int kBlk = 16 * BK;                   // a 16-row block of a K-tile
    constexpr int kStage = (MB + NT) * kBlk;
    constexpr int kCopies = 2 * (MB + NT);          // copy instructions per K-tile
    // block rows whose partial sums fit LDS together
    constexpr int MR = WK * MB * NT * 1024 > 128 * 1024 ? MB / 2 : MB;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, g = lane >> 4;

    const int total = p.tiles_m * p.tiles_n;
    const int pos = blockIdx.x;
    const int t = total % kXcds == 0 ? (pos % kXcds) * (total / kXcds) + pos / kXcds : pos;
    const int tm = t % p.tiles_m, tn = t / p.tiles_m;
    const int n0 = tn * TN;
    int m_first = tm * TM, m_end = min(m_first + TM, p.M), m_step = TM, expert = 0;
    if constexpr (GROUPED) {
        // A table entry is up to 256 rows of an expert, walked TM at a time.  Where the rows lie on few experts there are fewer entries
        // than workgroups to a column of tiles: those beyond the last entry take every second, third, ... pass of the entries
        // before.  (64 experts of 2 x 1408 x 2048, 1280 rows all on one: 53 us with its entries walked by a workgroup each.)
        const int* e = p.tile_map + 1 + kMapWords * min(tm, p.map_entries - 1);            // the usual one, read beside the number of entries
        int number = e[0], first = e[1], last = e[2], first_tile = e[3];
        const int entries = __builtin_amdgcn_readfirstlane(min(p.tile_map[0], p.map_entries));
        if (entries <= 0) return;
        int entry = tm, part = 0, parts = tm + entries < p.tiles_m ? 2 : 1;
        if (tm >= entries || 2 * entries < p.tiles_m) {
            part = tm / entries;
            entry = tm - part * entries;
            parts = (p.tiles_m - 1 - entry) / entries + 1;
            e = p.tile_map + 1 + kMapWords * entry;
            number = e[0]; first = e[1]; last = e[2]; first_tile = e[3];
        }
        expert = __builtin_amdgcn_readfirstlane(number);
        m_first = __builtin_amdgcn_readfirstlane(first) + (entry - __builtin_amdgcn_readfirstlane(first_tile)) * BM;
        m_end = min(m_first + BM, __builtin_amdgcn_readfirstlane(last));
        m_first += part * TM;
        m_step = parts * TM;
    }
    const uint8_t* B = p.B + static_cast<size_t>(expert) * p.b_expert_stride;
    const uint8_t* B2 = GATE ? p.B2 + static_cast<size_t>(expert) * p.b_expert_stride : B;

    // ---- memory -> LDS: one instruction copies 8 whole 128-byte row pieces, so that every line is asked for once ----
    const int crow = lane >> 3;
    uint32_t cchunk[2];                             // this lane's 16-byte chunk of rows 0-7 and 8-15 of a block
    cchunk[0] = ((lane & 7) ^ crow) * 16u;
    cchunk[1] = ((lane & 7) ^ crow ^ 1) * 16u;
    uint32_t woff[NB][2];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int h = 0; h < 2; ++h)
            woff[b][h] = static_cast<uint32_t>(min(n0 + b * 16 + h * 8 + crow, p.N - 1)) * static_cast<uint32_t>(p.ldb) + cchunk[h];
    uint8_t* const mine = smem + wave * (S * kStage);
    const uint32_t lds_mine = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem)) + wave * (S * kStage);
    // ---- LDS -> operands: row r16, chunks 2 g and 2 g + 1 ----
    const int fs = (r16 ^ (r16 >> 3)) & 7;
    const int rd0 = r16 * BK + (((2 * g) ^ fs) << 4), rd1 = r16 * BK + (((2 * g + 1) ^ fs) << 4);

    const int kfull = p.K / BK;
    const int nk = kfull > wave ? (kfull - wave + WK - 1) / WK : 0;
    const int kgroups = (p.K + BK - 1) / BK;        // scale groups along K (BLOCK)
    const int kpad = kgroups | 1;
    float* const lds_sa = reinterpret_cast<float*>(smem + WK * S * kStage);
    float* const lds_sb = lds_sa + TM * kpad;

    for (int m0 = m_first; m0 < m_end; m0 += m_step) {
        uint32_t xoff[MB][2];
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                int row = min(m0 + b * 16 + h * 8 + crow, m_end - 1);
                if (GROUPED && p.a_row_index) row = p.a_row_index[row];
                xoff[b][h] = static_cast<uint32_t>(row) * static_cast<uint32_t>(p.lda) + cchunk[h];
            }
        if constexpr (BLOCK) {
            // the tile's scales: [TM][groups] of the activations, [groups] of the weights
            for (int i = threadIdx.x; i < TM * kgroups; i += 64 * WK) {
                const int r = i / kgroups, k = i - r * kgroups;
                lds_sa[r * kpad + k] = p.sa[static_cast<size_t>(min(m0 + r, m_end - 1)) * kgroups + k];
            }
            for (int i = threadIdx.x; i < kgroups; i += 64 * WK) lds_sb[i] = p.sb[static_cast<size_t>(n0 / 128) * kgroups + i];
            __syncthreads();
        }

        // the epilogue's factors, on their way while K is walked: one row and one column per lane
        float f_row = 0.0f, f_col = 0.0f, f_col2 = 0.0f;
        const int tid = threadIdx.x;
        if constexpr (!BLOCK) {
            const float* sb = p.sb + static_cast<size_t>(expert) * p.sb_expert_stride;
            const float* sb2 = GATE ? p.sb2 + static_cast<size_t>(expert) * p.sb_expert_stride : sb;
            int row = min(m0 + (tid < TM ? tid : 0), m_end - 1), col = min(n0 + (tid < TN ? tid : 0), p.N - 1);
            if (GROUPED && p.a_row_index) row = p.a_row_index[row];
            f_row = p.sa[rowcol ? row : 0];
            f_col = sb[rowcol ? col : 0];
            if constexpr (GATE) f_col2 = sb2[rowcol ? col : 0];
        }

        v4f acc[MB][NT];
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

        auto copy = [&](uint32_t dst, uint32_t voff, const uint8_t* base) {
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(dst), "v"(voff), "s"(base) : "memory");
        };
        auto fetch = [&](int stage, int kt) {
            const size_t k0 = static_cast<size_t>(kt) * BK;
            const uint32_t dst = lds_mine + stage * kStage;
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    copy(dst + b * kBlk + h * (kBlk / 2), woff[b][h], B + k0);
                    if constexpr (GATE) copy(dst + (NB + b) * kBlk + h * (kBlk / 2), woff[b][h], B2 + k0);
                }
#pragma unroll
            for (int b = 0; b < MB; ++b)
#pragma unroll
                for (int h = 0; h < 2; ++h) copy(dst + (NT + b) * kBlk + h * (kBlk / 2), xoff[b][h], p.A + k0);
        };
        v8i x[MB], w[NT];
        auto read = [&](int stage) {
            const uint8_t* s = mine + stage * kStage;
            auto one = [&](v8i& d, const uint8_t* blk) {
                const uint4 lo = *reinterpret_cast<const uint4*>(blk + rd0), hi = *reinterpret_cast<const uint4*>(blk + rd1);
                d = v8i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
            };
#pragma unroll
            for (int j = 0; j < NT; ++j) one(w[j], s + j * kBlk);
#pragma unroll
            for (int i = 0; i < MB; ++i) one(x[i], s + (NT + i) * kBlk);
        };
        auto multiply = [&](int kt) {
            float fx[MB], fw = 0.0f;
            if constexpr (BLOCK) {
                fw = lds_sb[kt];
#pragma unroll
                for (int i = 0; i < MB; ++i) fx[i] = lds_sa[(i * 16 + r16) * kpad + kt] * fw;
            }
            if constexpr (BLOCK) {
                // a column's products are folded while the next column's are on the matrix cores
                v4f part[2][MB];
#pragma unroll
                for (int j = 0; j <= NT; ++j) {
                    if (j < NT) {
#pragma unroll
                        for (int i = 0; i < MB; ++i) {
                            const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
                            part[j & 1][i] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w[j < NT ? j : 0], x[i], zero, (FMT >> 1) & 1, FMT & 1, 0, 0, 0, 0);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    if (j > 0) {
#pragma unroll
                        for (int i = 0; i < MB; ++i)
#pragma unroll
                            for (int q = 0; q < 4; ++q)
                                acc[i][j > 0 ? j - 1 : 0][q] = __builtin_fmaf(part[(j + 1) & 1][i][q], fx[i], acc[i][j > 0 ? j - 1 : 0][q]);
                    }
                }
            } else {
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int i = 0; i < MB; ++i)
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w[j], x[i], acc[i][j], (FMT >> 1) & 1, FMT & 1, 0, 0, 0, 0);
            }
        };

        // (loads issued before the copies are older than them: a wait that leaves n copies in flight covers them)
#pragma unroll
        for (int s = 0; s < S; ++s)
            if (s < nk) fetch(s, wave + s * WK);
        int i = 0, stage = 0;
        for (; i + S < nk; ++i) {
            __builtin_amdgcn_s_waitcnt(wait_vm((S - 1) * kCopies));
            __builtin_amdgcn_sched_barrier(0);
            read(stage);
            __builtin_amdgcn_s_waitcnt(kWaitLgkm0);    // the stage is free for the copies of the K-tile S ahead
            __builtin_amdgcn_sched_barrier(0);
            fetch(stage, wave + (i + S) * WK);
            multiply(wave + i * WK);
            stage = stage + 1 == S ? 0 : stage + 1;
        }
        for (; i < nk; ++i) {
            // the last K-tiles: nothing is issued behind them
            if (nk - i >= S) __builtin_amdgcn_s_waitcnt(wait_vm((S - 1) * kCopies));
            else             __builtin_amdgcn_s_waitcnt(wait_vm(0));
            __builtin_amdgcn_sched_barrier(0);
            read(stage);
            multiply(wave + i * WK);
            stage = stage + 1 == S ? 0 : stage + 1;
        }
        // the last, partial K-tile (K % 16 == 0): bytes beyond K count as zeros
        if (kfull * BK < p.K && wave == kfull % WK) {
            const uint32_t left = p.K - kfull * BK;
            const size_t k0 = static_cast<size_t>(kfull) * BK;
            auto part = [&](int blk, int h, uint32_t voff, const uint8_t* base) {
                uint4 v = make_uint4(0, 0, 0, 0);
                if (cchunk[h] < left) v = *reinterpret_cast<const uint4*>(base + k0 + voff);
                *reinterpret_cast<uint4*>(mine + blk * kBlk + h * (kBlk / 2) + lane * 16) = v;
            };
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    part(b, h, woff[b][h], B);
                    if constexpr (GATE) part(NB + b, h, woff[b][h], B2);
                }
#pragma unroll
                for (int b = 0; b < MB; ++b) part(NT + b, h, xoff[b][h], p.A);
            }
            read(0);
            multiply(kfull);
        }
        __syncthreads();          // every wavefront is done with its stages: their LDS takes the partial sums

        // ---- the wavefronts' partial sums, added in wavefront order; MR block rows at a time ----
        float4* red = reinterpret_cast<float4*>(smem);
        float* const lds_f = reinterpret_cast<float*>(smem + WK * MR * NT * 1024);      // [TM] rows, [TN] columns, [TN] up columns
        if constexpr (!BLOCK) {
            if (tid < TM) lds_f[tid] = f_row;
            if (tid < TN) lds_f[TM + tid] = f_col;
            if (GATE && tid < TN) lds_f[TM + TN + tid] = f_col2;
        }
        static_for<0, MB / MR>([&](auto pass) {
        constexpr int base = decltype(pass)::value * MR;
        if constexpr (base > 0) __syncthreads();
#pragma unroll
        for (int b = 0; b < MR; ++b)
#pragma unroll
            for (int j = 0; j < NT; ++j)
                red[(wave * (MR * NT) + b * NT + j) * 64 + lane] =
                    make_float4(acc[base + b][j][0], acc[base + b][j][1], acc[base + b][j][2], acc[base + b][j][3]);
        __syncthreads();
        auto summed = [&](int blk, float (&v)[4]) {
            v[0] = v[1] = v[2] = v[3] = 0.0f;
#pragma unroll
            for (int k = 0; k < WK; ++k) {
                const float4 s = red[(k * (MR * NT) + blk) * 64 + lane];
                v[0] += s.x; v[1] += s.y; v[2] += s.z; v[3] += s.w;
            }
        };
        // ---- epilogue: one 16 x 16 block of outputs per wavefront and step; a lane holds four columns of one row ----
#pragma unroll
        for (int u = 0; u < (MR * NB + WK - 1) / WK; ++u) {
            const int unit = wave + u * WK;
            if (MR * NB % WK != 0 && unit >= MR * NB) break;
            const int mb = unit / NB, nb = unit % NB;
            const int ml = (base + mb) * 16 + r16, nl = nb * 16 + g * 4;
            const int m = m0 + ml, n = n0 + nl;
            float v[4], up[4];
            summed(mb * NT + nb, v);
            if constexpr (GATE) summed(mb * NT + NB + nb, up);
            if constexpr (!BLOCK) {
                const float sa = lds_f[ml];
                const float4 c = *reinterpret_cast<const float4*>(lds_f + TM + nl);
                const float c4[4] = {c.x, c.y, c.z, c.w};
                float4 d = c;
                if constexpr (GATE) d = *reinterpret_cast<const float4*>(lds_f + TM + TN + nl);
                const float d4[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    v[q] *= sa * c4[q];
                    if constexpr (GATE) {
                        // the reference rounds gate and up to bf16 before the SiLU product
                        const uint32_t gu = pack_bf16x2_hw(v[q], up[q] * (sa * d4[q]));
                        v[q] = fast_silu(bf16_lo(gu)) * bf16_hi(gu);
                    }
                }
            }
            if (m >= m_end || n >= p.N) continue;
            const bool whole = n + 3 < p.N;
            if (bias)
#pragma unroll
                for (int q = 0; q < 4; ++q) v[q] = round_bf16_hw(v[q]) + bf16_to_f32(p.bias[min(n + q, p.N - 1)]);
            uint16_t* c = p.C + static_cast<size_t>(m) * p.ldc + n;
            const uint32_t o01 = pack_bf16x2_hw(v[0], v[1]), o23 = pack_bf16x2_hw(v[2], v[3]);
            if (whole && c_vec) {
                *reinterpret_cast<uint2*>(c) = make_uint2(o01, o23);
            } else {
                c[0] = static_cast<uint16_t>(o01);
                if (n + 1 < p.N) c[1] = static_cast<uint16_t>(o01 >> 16);
                if (n + 2 < p.N) c[2] = static_cast<uint16_t>(o23);
                if (n + 3 < p.N) c[3] = static_cast<uint16_t>(o23 >> 16);
            }
        }
        });
        if (GROUPED) __syncthreads();          // the sums' LDS takes the next pass's stages
    }
}

constexpr int kLds = 160 * 1024;

// bytes of LDS the scales of a block-scaled tile take beside the operands: [16 mb] rows and one row of weights
constexpr size_t block_scale_bytes(int mb, int K) {
    const size_t kg = (static_cast<size_t>(K) + BK - 1) / BK;
    return (16 * mb * (kg | 1) + kg) * 4;
}

template <int FMT, bool GATE, bool BLOCK, bool GROUPED, int MB, int NB, int WK, int S>
int launch(GemmArgs p, int epi, int scale_mode, hipStream_t st) {
    constexpr int NT = GATE ? 2 * NB : NB;
    constexpr int stages = WK * S * (MB + NT) * 2048;
    constexpr int one = WK * MB * NT * 1024, sums = (one > 128 * 1024 ? one / 2 : one) + (16 * MB + 32 * NB) * 4;
    constexpr int base = stages > sums ? stages : sums;
    static_assert(base <= kLds);
    const size_t lds = base + (BLOCK ? block_scale_bytes(MB, p.K) : 0);
    if (lds > kLds) return CF_ERR_UNSUPPORTED;          // direct_takes() is stricter
    static std::once_flag once;
    static hipError_t err = hipSuccess;
    std::call_once(once, [] {
        err = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm_nt_direct<FMT, GATE, BLOCK, GROUPED, MB, NB, WK, S>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    });
    if (err != hipSuccess) return static_cast<int>(err);
    if (!GROUPED) p.tiles_m = (p.M + 16 * MB - 1) / (16 * MB);
    p.tiles_n = (p.N + 16 * NB - 1) / (16 * NB);
    k_gemm_nt_direct<FMT, GATE, BLOCK, GROUPED, MB, NB, WK, S><<<p.tiles_m * p.tiles_n, 64 * WK, lds, st>>>(
        p, scale_mode == SCALE_ROWCOL, epi == EPI_BIAS, p.ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(p.C) & 7u) == 0);
    return launch_status();
}

// The tile shapes, smallest first: 16 mb rows x 16 nt weight rows (nt counts gate and up blocks), whether two workgroups fit a
// CU's LDS, and what a workgroup costs beside its operand bytes (pipeline fill, reduction, epilogue; microseconds).
struct Shape { int mb, nt; bool shared; float fixed; };
constexpr Shape kPlain[6] = {{1, 1, true, 1.5f}, {2, 2, true, 2.0f}, {4, 2, false, 2.5f}, {4, 4, false, 4.0f}, {8, 4, false, 6.0f}, {8, 8, false, 12.0f}};
// Grouped only: the first two with 64 weight rows per workgroup.  With experts enough to fill the chip many times over, the cost
// per workgroup counts for more than their number: 64 experts of 2048 x 1408 and 6 rows each,
// the routed layer around them 157 -> 145 us; 18 rows each 157 -> 148; 16 tokens, 1.5 rows each 129 -> 114.
constexpr Shape kWide[2] = {{1, 4, true, 2.0f}, {2, 4, true, 2.5f}};
constexpr int kWideShape = 6;           // shape numbers 6 and 7
constexpr double kBlockRate[4] = {70e3, 75e3, 62e3, 72e3};     // bytes per microsecond and CU with block scales
constexpr Shape kGate[4] = {{1, 2, true, 1.5f}, {2, 4, true, 2.5f}, {4, 8, false, 6.0f}, {8, 8, false, 12.0f}};

template <int FMT, bool BLOCK, bool GROUPED>
int launch_plain(const GemmArgs& p, int epi, int scale_mode, int shape, hipStream_t st) {
    switch (shape) {
        case 0: return launch<FMT, false, BLOCK, GROUPED, 1, 1, 4, 3>(p, epi, scale_mode, st);
        case 1: return launch<FMT, false, BLOCK, GROUPED, 2, 2, 4, 2>(p, epi, scale_mode, st);
        case 2:
            if constexpr (GROUPED) return CF_ERR_UNSUPPORTED;          // of two shapes of as many rows the wider is taken
            else return launch<FMT, false, BLOCK, GROUPED, 4, 2, 4, 2>(p, epi, scale_mode, st);
        case 3: return launch<FMT, false, BLOCK, GROUPED, 4, 4, 4, 2>(p, epi, scale_mode, st);
        default:
            if constexpr (GROUPED) {
                return shape == kWideShape ? launch<FMT, false, BLOCK, GROUPED, 1, 4, 4, 2>(p, epi, scale_mode, st)
                                           : launch<FMT, false, BLOCK, GROUPED, 2, 4, 4, 1>(p, epi, scale_mode, st);
            } else if constexpr (BLOCK) return CF_ERR_UNSUPPORTED;
            else return shape == 4 ? launch<FMT, false, BLOCK, GROUPED, 8, 4, 4, 1>(p, epi, scale_mode, st) : launch<FMT, false, BLOCK, GROUPED, 8, 8, 4, 1>(p, epi, scale_mode, st);
    }
}
template <bool GROUPED>
int launch_gate(const GemmArgs& p, int scale_mode, int shape, hipStream_t st) {
    switch (shape) {
        case 0: return launch<0, true, false, GROUPED, 1, 1, 4, 3>(p, EPI_SILU_GATE, scale_mode, st);
        case 1: return launch<0, true, false, GROUPED, 2, 2, 4, 1>(p, EPI_SILU_GATE, scale_mode, st);
        case 2: return launch<0, true, false, GROUPED, 4, 4, 4, 1>(p, EPI_SILU_GATE, scale_mode, st);
        default:
            if constexpr (GROUPED) return CF_ERR_UNSUPPORTED;
            else return launch<0, true, false, GROUPED, 8, 4, 4, 1>(p, EPI_SILU_GATE, scale_mode, st);
    }
}

}  // namespace

bool direct_ok(const GemmArgs& p, int fmt, int epi, int scale_mode) {
    return epi <= EPI_SILU_GATE && !(fmt & 2) && !(epi == EPI_SILU_GATE && fmt) && !(scale_mode == SCALE_BLOCK && (fmt || epi != EPI_NONE)) &&
           p.K >= BK && static_cast<size_t>(p.M) * p.lda < (1ull << 32) && static_cast<size_t>(p.N) * p.ldb < (1ull << 32);
}
// Whether the shape exists for the epilogue and scales and its LDS suffices (block scales: the stages of the four shapes take 48,
// 64, 96 and 128 KiB, their sums less, the scales the rest)
bool direct_takes(const GemmArgs& p, int epi, int scale_mode, int shape) {
    if (shape < 0 || shape >= (epi == EPI_SILU_GATE ? 4 : scale_mode == SCALE_BLOCK ? 4 : 6)) return false;
    if (scale_mode != SCALE_BLOCK) return true;
    constexpr size_t stages[4] = {48 * 1024, 64 * 1024, 96 * 1024, 128 * 1024};
    return stages[shape] + block_scale_bytes(kPlain[shape].mb, p.K) <= kLds;
}

// Picks the tile shape and says what it would take, in microseconds: every workgroup moves K bytes of each of its rows and weight
// rows, and a CU takes them in at 93 KB per microsecond whatever the shape (measured, K 1024 to 14336); a CU whose LDS holds one
// workgroup works in whole rounds.  With block scales the folds lower the rate (fitted to 1400 sizes):
// 3000 x 512 over K 4096 takes 33.9, 42.4 and 28.7 us in the last three shapes and 29.9 in the persistent kernel, 1000 x 512:
// 11.7, 12.1, 13.7 and 28.6; 100 x 1000 over K 4096 8.3, 6.7, 8.9 and 11.5 in the four shapes.
// A shape with more rows than the next one smaller would do is not looked at: its extra rows are copies.
float direct_estimate_us(const GemmArgs& p, int epi, int scale_mode, int* shape) {
    const bool gate = epi == EPI_SILU_GATE, block = scale_mode == SCALE_BLOCK;
    const int M = p.M, N = p.N, K = p.K;
    const Shape* s = gate ? kGate : kPlain;
    const int count = gate ? 4 : block ? 4 : 6;
    float best = 1e30f;
    for (int i = 0; i < count; ++i) {
        if (i > 0 && s[i].mb > s[i - 1].mb && M <= 16 * s[i - 1].mb) break;
        if (!direct_takes(p, epi, scale_mode, i)) break;
        const int tn = 16 * s[i].nt / (gate ? 2 : 1);
        const double wgs = static_cast<double>((M + 16 * s[i].mb - 1) / (16 * s[i].mb)) * ((N + tn - 1) / tn);
        double rounds = wgs / num_cus();
        if (!s[i].shared) rounds = static_cast<double>(static_cast<long long>(rounds + 0.999));
        if (rounds < 1.0) rounds = 1.0;
        const double rate = block ? kBlockRate[i] : 93e3;
        const float t = static_cast<float>(rounds * (s[i].fixed + static_cast<double>(K) * 16.0 * (s[i].mb + s[i].nt) / rate));
        if (t < best) { best = t; *shape = i; }
    }
    return best;
}

float grouped_direct_estimate_us(int total_rows, int N, int K, int num_experts, bool gate, int* shape) {
    const Shape* s = gate ? kGate : kPlain;
    const int count = gate ? 3 : 4;
    const float rows = static_cast<float>(total_rows) / static_cast<float>(num_experts);
    int i = 0;
    while (i + 1 < count && (16 * s[i].mb < 1.5f * rows + 2.0f || s[i + 1].mb == s[i].mb)) ++i;
    *shape = i;
    auto estimate = [&](const Shape& sh) {
        const int tn = 16 * sh.nt / (gate ? 2 : 1);
        const float rounds = static_cast<float>(num_experts) * static_cast<float>((N + tn - 1) / tn) / static_cast<float>(num_cus());
        return (rounds < 1.0f ? 1.0f : rounds) * (sh.fixed + static_cast<float>(K) * 16.0f * static_cast<float>(sh.mb + sh.nt) / 93e3f);
    };
    float best = estimate(s[i]);
    if (!gate && i < 2 && estimate(kWide[i]) < best) {
        best = estimate(kWide[i]);
        *shape = kWideShape + i;
    }
    return best;
}

// The same in passes of 64 rows that run side by side; to be compared with 0.89 us a K-tile and 6.1 a round (gate 0.88 and 8.3) of the ring kernel.
// Passes: 0.6 an expert more than the rows fill (even counts leave less open, Zipf's more).  An XCD's workgroups are a run of whole columns of
// weights in which those that have rows come first, so a part of a column counts as one.  Beyond a round half a round more, for what is left uneven.
// Fitted, to 15 %, to 1200 sizes of 1 to 64 experts with counts even, random, after Zipf, half on one and all on one; 15 % on top for those that are not even.
// Without the XCDs and those 15 %, 56 of the 1200 were slower than the ring kernel by more than 3 % (24 experts of 640 x 5376, 186 rows each 77.6 against
// 50.5 us; 32 of 384 x 5632 gated after Zipf 82 and 55); now 6 of 1000 others are, the worst 1.14 times.
float grouped_direct_many_estimate_us(int total_rows, int N, int K, int num_experts, bool gate, int* shape) {
    *shape = gate ? 2 : 3;
    const float passes = static_cast<float>(total_rows) / 64.0f + 0.6f * static_cast<float>(num_experts);
    const int columns = (N + 63) / 64;
    const float per_cu = passes * static_cast<float>((columns + kXcds - 1) / kXcds) * static_cast<float>(kXcds) / static_cast<float>(num_cus());
    const float ktiles = static_cast<float>(K / BK);
    return (per_cu > 0.8f ? per_cu + 0.5f : 1.0f) * (gate ? 4.5f + 0.345f * ktiles : 3.1f + 0.225f * ktiles);
}

int gemm_nt_direct(const GemmArgs& p, int fmt, int epi, int scale_mode, int shape, hipStream_t st) {
    if (epi == EPI_SILU_GATE) return fmt == 0 ? launch_gate<false>(p, scale_mode, shape, st) : CF_ERR_UNSUPPORTED;
    if (scale_mode == SCALE_BLOCK) return launch_plain<0, true, false>(p, epi, scale_mode, shape, st);
    return fmt == 1 ? launch_plain<1, false, false>(p, epi, scale_mode, shape, st)
         : fmt == 0 ? launch_plain<0, false, false>(p, epi, scale_mode, shape, st) : CF_ERR_UNSUPPORTED;
}
int grouped_gemm_nt_direct(const GemmArgs& p, int fmt, int epi, int shape, hipStream_t st) {
    if (epi == EPI_SILU_GATE) return fmt == 0 ? launch_gate<true>(p, SCALE_ROWCOL, shape, st) : CF_ERR_UNSUPPORTED;
    return fmt == 1 ? launch_plain<1, false, true>(p, epi, SCALE_ROWCOL, shape, st)
                    : launch_plain<0, false, true>(p, epi, SCALE_ROWCOL, shape, st);
}

}  // namespace cf
