// What the FP8 GEMM sources (gemm.hip, gemm_duo.hip, gemm_direct.hip) share: the arguments of a launch, the order tiles are
// walked in, small device helpers.
#pragma once
#include "internal.hpp"

#include <type_traits>

namespace cf {

enum { EPI_NONE = 0, EPI_BIAS = 1, EPI_SILU_GATE = 2, EPI_ACCUM_F32 = 3, EPI_ACCUM_BF16 = 4, EPI_STORE_F32 = 5 };
enum { SCALE_TENSOR = 0, SCALE_ROWCOL = 1, SCALE_BLOCK = 2, SCALE_ROW = 3 };   // SCALE_ROW: sa per row, sb one scalar (ring kernel)

constexpr int BM = 256, BN = 256, BK = 128;       // tile of the persistent kernels; BK is every kernel's K-tile
constexpr int kXcds = 8;
constexpr int kMapWords = 5;                      // words per entry of the row-tile table (build_tile_map), an entry being BM rows

struct GemmArgs {
    int M, N, K;                 // N = output columns
    const uint8_t* A; int lda;   // activations [M,K]
    const uint8_t* B; int ldb;   // weights [N,K] (gate weights for EPI_SILU_GATE)
    const uint8_t* B2;           // up weights [N,K] for EPI_SILU_GATE
    const float* sa;             // descale of A: [1] or [M]
    const float* sb;             // descale of B: [1] or [N]
    const float* sb2;            // descale of B2
    const uint16_t* bias;        // bf16 [N] for EPI_BIAS
    uint16_t* C; int ldc;        // bf16 [M,N]
    float* Cf;                   // fp32 [M,N] for EPI_ACCUM_F32 (C += product)
    int tiles_m, tiles_n;
    int force_staged;            // take the register-staged kernel even when the ring kernel applies
    int duo;                     // 1: the two-workgroups-per-CU kernel where it applies, 2: the same without the stagger, 0: where its estimate is lowest
    int small;                   // 1 + the tile shape of the small-tile kernel a caller asks for, 0: where its estimate is lowest
    int half;                    // take the half-tile kernel where it applies
    int ring;                    // keep the persistent kernels where a smaller-tile kernel's estimate is lower
    int mfma32;                  // keep k_gemm_nt_ring (the 32 x 32 x 64 MFMA shape) where k_gemm_nt_ring16 would apply
    int edge;                    // 256, 128: take the kernel of that tile edge of gemm_block.hip or gemm_accum.hip where it applies
    // grouped (per-expert) form, ring and small-tile kernels; all null / 0 for a dense GEMM
    const int* tile_map;         // [0] = number of row tiles, then kMapWords words per row tile: expert, its first row, end row, first tile, tiles
    int map_entries;             // small-tile kernel: row tiles the table has room for (tiles_m may be several times that: workgroups that share an entry)
    const int* a_row_index;      // compact row r reads A row (and its descale) a_row_index[r]; null = r
    int a_rows;                  // rows of the A buffer (= M without a row index)
    long long b_expert_stride;   // bytes between the weight matrices of consecutive experts
    int sb_expert_stride;        // elements between the channel descales of consecutive experts
    // term-split form (ring kernel, MX instantiation only): A's K axis is `K / b_k_period` terms laid side by side,
    // term t = the residual of the terms before it scaled by 16^t; every term multiplies the same b_k_period
    // columns of B, and the matrix cores scale its products by 2^(-4 t)
    int b_k_period;
};

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// Tile t of the walk order -> (tile_m, tile_n): patches of 8 (M) x tiles_n, row tiles varying fastest, so that
// 32 consecutive tiles form an 8 x 4 patch whose operands an XCD's L2 can hold.
__device__ __forceinline__ void tile_coords(int t, int tiles_m, int tiles_n, int& tm, int& tn) {
    constexpr int GM = 8;
    const int group = t / (GM * tiles_n);
    const int first_m = group * GM;
    const int gm = min(GM, tiles_m - first_m);
    const int in_group = t - group * GM * tiles_n;
    tm = first_m + in_group % gm;
    tn = in_group / gm;
}
__device__ __forceinline__ int swz(int row) { return (row ^ ((row >> 3) & 3)) & 7; }

// SiLU gate for the fused epilogue: x * 1/(1 + 2^(-x*log2 e)) on the hardware exp2 and reciprocal
// (1 ulp each).  The stand-alone swiglu kernel keeps the correctly-rounded divide and the
// reproducible expf; the two differ by at most one bf16 ulp of the product.
__device__ __forceinline__ float fast_silu(float x) {
    const float e = __builtin_amdgcn_exp2f(-1.44269504f * x);
    return x * __builtin_amdgcn_rcpf(1.0f + e);
}

inline int num_cus() {
    static int n = [] {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) != hipSuccess) return 256;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) return 256;
        return v;
    }();
    return n;
}
// Workgroups of a persistent launch over `total` tiles, at most `most`: a multiple of 8, which the tile walk needs to keep
// "position % 8 = XCD", rounded UP while there is room.  (Rounded down, 44 tiles ran on 40 workgroups, four of which then
// had two tiles: 44 us instead of 22 for 256 x 2 x 5632 x 2048.)  A workgroup without a tile returns at once.
inline int persistent_grid(int total, int most) {
    if (total < kXcds) return total;
    const int up = (total + kXcds - 1) / kXcds * kXcds;
    return up <= most ? up : most / kXcds * kXcds;
}

// Whether a row of C begins inside a 128-byte line, so that neighbouring tiles write parts of the same lines.
inline bool c_lines_shared(const GemmArgs& p, int elem_bytes) { return static_cast<long long>(p.ldc) * elem_bytes % 128 != 0; }

// gemm_direct.hip: whether it takes a problem (at all; with a tile shape), the time of its best tile shape and which one that is,
// the launches (dense; grouped over a row-tile table)
bool direct_ok(const GemmArgs& p, int fmt, int epi, int scale_mode);
bool direct_takes(const GemmArgs& p, int epi, int scale_mode, int shape);
float direct_estimate_us(const GemmArgs& p, int epi, int scale_mode, int* shape);
float grouped_direct_estimate_us(int total_rows, int N, int K, int num_experts, bool gate, int* shape);
float grouped_direct_many_estimate_us(int total_rows, int N, int K, int num_experts, bool gate, int* shape);
int gemm_nt_direct(const GemmArgs& p, int fmt, int epi, int scale_mode, int shape, hipStream_t st);
int grouped_gemm_nt_direct(const GemmArgs& p, int fmt, int epi, int shape, hipStream_t st);
// gemm_half.hip: whether it takes a problem, its time, the launch
bool half_ok(const GemmArgs& p, int fmt, int epi, int scale_mode);
float half_estimate_us(const GemmArgs& p, int epi, bool shared);
int gemm_nt_half(const GemmArgs& p, int fmt, int epi, int scale_mode, hipStream_t st);
// gemm_duo.hip: whether it takes a problem, its time, the launch
bool duo_ok(const GemmArgs& p, int fmt, int epi, int scale_mode);
float duo_estimate_us(const GemmArgs& p, int epi);
int gemm_nt_duo(GemmArgs p, int fmt, int epi, int scale_mode, hipStream_t st);
// gemm_block.hip (block scales on 256 x 256 tiles): whether it takes a problem, its time, the launch
bool block_wide_ok(const GemmArgs& p);
float block_wide_estimate_us(const GemmArgs& p);
int gemm_nt_block_wide(GemmArgs p, hipStream_t st);
bool block_slim_ok(const GemmArgs& p);
float block_slim_estimate_us(const GemmArgs& p);
int gemm_nt_block_slim(GemmArgs p, hipStream_t st);
// gemm_accum.hip
bool accum_wide_ok(const GemmArgs& p, int fmt, int epi, int scale_mode);
float accum_wide_estimate_us(const GemmArgs& p);
int gemm_nt_accum_wide(GemmArgs p, hipStream_t st);

}  // namespace cf
