"""The block-scaled GEMM on 256 x 256 tiles: the fewest K-tiles it takes and odd and even counts after them, rows that end inside
a tile, a wavefront's part and a 16-row block, one tile per workgroup and several, rows of C beyond N."""
import ctypes

import numpy as np
import pytest
import torch

import oracle_lib as orc
from gpu_util import bf16_bits, case, dev_arr, stream

pytestmark = pytest.mark.gpu
BLOCK, BLOCK_WIDE, FLAG = 2, 6, 4096


# sizes whose 128 x 256 tiles need more rounds over 256 CUs than the 256 x 256 ones by half or more, which is where the latter are chosen;
# asked for here, so that the test does not hang on the estimates
@pytest.mark.parametrize("M,N,K,pad", [
    (255, 33024, 384, 0), (257, 22016, 512, 8), (129, 33024, 640, 0),
    (1000, 8448, 1024, 8),          # 4 row tiles, the last one 232 rows
    (2100, 8192, 384, 0),           # 288 tiles: some workgroups take two, others one
    (2561, 16384, 512, 0),          # 704 tiles, three a workgroup; one row in the last row tile
])
def test_block_scales_on_wide_tiles(cf, dev, M, N, K, pad):
    case(f"block-scaled gemm, wide tiles {M}x{N}x{K} ldc N + {pad}")
    kernel = ctypes.c_int(-1)
    cf.cf_fp8_gemm_route(M, N, K, 0, 0, BLOCK, 0, N + pad, FLAG, ctypes.byref(kernel))
    assert kernel.value == BLOCK_WIDE
    rng = np.random.default_rng(M + N + K)
    A = orc.quantize_e4m3(orc.bf16_from_f32(rng.standard_normal((M, K)).astype(np.float32)), np.float32(100.0))
    B = orc.quantize_e4m3(orc.bf16_from_f32(rng.standard_normal((N, K)).astype(np.float32)), np.float32(100.0))
    sa = (2.0 ** rng.uniform(-8, 2, (M, K // 128))).astype(np.float32)
    sb = (2.0 ** rng.uniform(-8, 2, (N // 128, K // 128))).astype(np.float32)
    C = torch.full((M, N + pad), -7.0, dtype=torch.bfloat16, device=dev)
    cf.cf_fp8_gemm_nt_bf16_ex(M, N, K, dev_arr(A, dev), K, 0, dev_arr(sa, dev), dev_arr(B, dev), K, dev_arr(sb, dev), BLOCK, 0, None, None,
                              None, C, N + pad, FLAG, stream())
    got = orc.bf16_to_f32(bf16_bits(C))
    assert (got[:, N:] == -7.0).all()
    rows = np.unique(np.concatenate([np.arange(min(M, 48)), np.arange(max(M - 48, 0), M), rng.integers(0, M, 32)]))
    ref, absdot = orc.gemm_nt_ref(A[rows], B, sa[rows], sb, scale_mode=BLOCK)
    orc.assert_gemm_close(got[rows, :N], ref, absdot, what=f"wide block {M}x{N}x{K}")
