"""Weight gradients over a K that is no multiple of 128, on 256 x 256 tiles: last K-tiles of 16 to 112 bytes after
odd and even counts of whole ones, one tile per workgroup, two for some, three and six for all, rows and columns that end inside a
tile, rows of C that do not begin at lines."""
import ctypes

import numpy as np
import pytest
import torch

import oracle_lib as orc
from gpu_util import case, dev_arr, stream

pytestmark = pytest.mark.gpu
TENSOR, ACCUM_F32, DUO, ACCUM_WIDE = 0, 3, 4, 8
F_DUO, F_WIDE = 4, 4096


# sizes at which two workgroups of 128 x 128 tiles per CU are estimated to take longer; both are asked for here, so that the test does
# not hang on the estimates
@pytest.mark.parametrize("M,N,K,pad", [
    (3841, 4092, 2704, 4),          # 256 tiles; one row in the last row tile, 252 columns in the last column tile
    (4096, 4000, 2992, 0),          # the last column tile 160 columns
    (3900, 4064, 2864, 32),
    (7100, 4096, 1520, 32),         # 448 tiles: some workgroups take two, others one
    (7037, 4092, 2512, 8),          # rows of C off the lines
    (12200, 4096, 1504, 0),         # 768, three a workgroup
    (12200, 8192, 1232, 0),         # 1536 tiles, six a workgroup
])
def test_ragged_k_on_wide_tiles(cf, dev, M, N, K, pad):
    case(f"wgrad accumulate, wide tiles {M}x{N}x{K} ldc N + {pad}")
    kernel = ctypes.c_int(-1)
    for flag, which in ((F_WIDE, ACCUM_WIDE), (F_DUO, DUO)):
        cf.cf_fp8_gemm_route(M, N, K, 0, 1, TENSOR, ACCUM_F32, N + pad, flag, ctypes.byref(kernel))
        assert kernel.value == which
    rng = np.random.default_rng(M + N + K)
    A = orc.quantize_e4m3(orc.bf16_from_f32(rng.standard_normal((M, K), dtype=np.float32)), np.float32(100.0))
    B = orc.quantize_e5m2(orc.bf16_from_f32(rng.standard_normal((N, K), dtype=np.float32)), np.float32(1000.0))
    sa, sb = np.float32([0.01]), np.float32([3e-5])
    C = torch.randn(M, N + pad, device=dev, generator=torch.Generator(device=dev).manual_seed(K)) * 0.01
    held = C.clone()
    cf.cf_fp8_gemm_nt_accum_f32_ex(M, N, K, dev_arr(A, dev), K, 0, dev_arr(sa, dev), dev_arr(B, dev), K, 1, dev_arr(sb, dev), C, N + pad, F_WIDE,
                                   stream())
    assert torch.equal(C[:, N:], held[:, N:])
    rows = np.unique(np.concatenate([np.arange(32), np.arange(M - 32, M), rng.integers(0, M, 32)]))
    at = torch.from_numpy(rows).to(dev)
    got, before = C[at][:, :N].cpu().numpy().astype(np.float64), held[at][:, :N].cpu().numpy().astype(np.float64)
    ref, absdot = orc.gemm_nt_ref(A[rows], B, sa, sb, b_e5m2=True)
    want = before + ref
    assert np.all(np.abs(got - want) <= orc.ACC_MFMA * absdot + 2.0 ** -22 * (np.abs(want) + np.abs(before)))
    # every other element: against the 128 x 128 tiles, whose sums differ in their order alone
    other = held.clone()
    cf.cf_fp8_gemm_nt_accum_f32_ex(M, N, K, dev_arr(A, dev), K, 0, dev_arr(sa, dev), dev_arr(B, dev), K, 1, dev_arr(sb, dev), other, N + pad, F_DUO,
                                   stream())
    bound = 2 * orc.ACC_MFMA * float(absdot.max()) * 2 + 2.0 ** -20 * float(C.abs().max())      # (absdot of other rows: at most twice the largest seen)
    assert float((C - other).abs().max()) <= bound


@pytest.mark.parametrize("M,N,K,pad_a,pad_b,pad_c", [
    (300, 516, 272, 16, 0, 4),                # three K-tiles, the fewest it takes
    (256, 252, 400, 112, 48, 0),              # one tile
    (4353, 4100, 1296, 48, 16, 12),           # 306 tiles; rows that begin off the lines in all three
    (3000, 2048, 16400, 0, 32, 0),            # many K-tiles
])
def test_ragged_k_with_rows_further_apart(cf, dev, M, N, K, pad_a, pad_b, pad_c):
    """Bytes between the end of a row's K and the next row are NaN (E4M3) and infinite (E5M2): none of them may be multiplied."""
    case(f"wgrad accumulate, wide tiles {M}x{N}x{K} lda K + {pad_a} ldb K + {pad_b} ldc N + {pad_c}")
    g = torch.Generator(device=dev).manual_seed(K)
    A = torch.full((M, K + pad_a), 0x7f, dtype=torch.uint8, device=dev)
    B = torch.full((N, K + pad_b), 0x7c, dtype=torch.uint8, device=dev)
    A[:, :K] = (torch.randn(M, K, device=dev, generator=g) * 100.0).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn).view(torch.uint8)
    B[:, :K] = (torch.randn(N, K, device=dev, generator=g) * 1000.0).to(torch.float8_e5m2).view(torch.uint8)
    sa, sb = np.float32([0.01]), np.float32([3e-5])
    C = torch.randn(M, N + pad_c, device=dev, generator=g) * 0.01
    held = C.clone()
    kernel = ctypes.c_int(-1)
    cf.cf_fp8_gemm_route(M, N, K, 0, 1, TENSOR, ACCUM_F32, N + pad_c, F_WIDE, ctypes.byref(kernel))
    assert kernel.value == ACCUM_WIDE
    cf.cf_fp8_gemm_nt_accum_f32_ex(M, N, K, A, K + pad_a, 0, dev_arr(sa, dev), B, K + pad_b, 1, dev_arr(sb, dev), C, N + pad_c, F_WIDE, stream())
    assert torch.equal(C[:, N:], held[:, N:])
    rng = np.random.default_rng(K)
    rows = np.unique(np.concatenate([np.arange(18), np.arange(M - 18, M), rng.integers(0, M, 16)]))
    at = torch.from_numpy(rows).to(dev)
    got, before = C[at][:, :N].cpu().numpy().astype(np.float64), held[at][:, :N].cpu().numpy().astype(np.float64)
    ref, absdot = orc.gemm_nt_ref(A[at][:, :K].cpu().numpy(), B[:, :K].cpu().numpy(), sa, sb, b_e5m2=True)
    want = before + ref
    assert np.all(np.abs(got - want) <= orc.ACC_MFMA * absdot + 2.0 ** -22 * (np.abs(want) + np.abs(before)))
    assert bool(torch.isfinite(C).all())
