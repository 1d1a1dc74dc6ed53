"""The three persistent block-scaled kernels beside one another, each asked for: K up to the 256 scale groups they take (the scales of a
weight block come in passes of 64 groups), a copy stream that is a whole tile ahead, several tiles a workgroup, rows of the operands further
apart than K with NaN bytes between them."""
import ctypes

import numpy as np
import pytest
import torch

import oracle_lib as orc
from gpu_util import bf16_bits, case, dev_arr, stream

pytestmark = pytest.mark.gpu
BLOCK = 2
RING, WIDE, SLIM = (2, 32), (6, 4096), (7, 8192)          # kernel number, flag


def operand(rows, K, pad, dev, seed):
    """Quantized normal values, as the tolerance assumes (an MFMA aligns its products to the largest of them), the padding all NaN."""
    g = torch.Generator(device=dev).manual_seed(seed)
    t = torch.full((rows, K + pad), 0x7f, dtype=torch.uint8, device=dev)
    t[:, :K] = (torch.randn(rows, K, device=dev, generator=g) * 100.0).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn).view(torch.uint8)
    return t


@pytest.mark.parametrize("M,N,K,pad_a,pad_b,kernels", [
    (4353, 3840, 384, 0, 0, (RING, WIDE)),                   # 270 tiles of 256 x 256, some workgroups two
    (2049, 4224, 512, 0, 0, (SLIM,)),                        # four K-tiles, as many as the ring has stages; 561 tiles, two or three a workgroup
    (2049, 4352, 640, 128, 16, (RING, WIDE, SLIM)),          # five
    (4353, 3840, 1152, 16, 256, (RING, WIDE, SLIM)),         # five tiles of 128 x 128 for some
    (257, 256, 8320, 0, 0, (RING, WIDE, SLIM)),              # 65 groups
    (4353, 3840, 8320, 48, 0, (RING, WIDE, SLIM)),
    (300, 768, 16384 + 128, 0, 32, (RING, WIDE, SLIM)),      # 129 groups
    (4353, 3840, 32768, 0, 0, (RING, WIDE, SLIM)),           # 256 groups
    (1100, 8576, 32768, 16, 16, (SLIM,)),                    # 603 tiles
])
def test_block_scaled_kernels_side_by_side(cf, dev, M, N, K, pad_a, pad_b, kernels):
    case(f"block-scaled kernels {M}x{N}x{K} lda K + {pad_a} ldb K + {pad_b}")
    rng = np.random.default_rng(M + N + K)
    A, B = operand(M, K, pad_a, dev, 1), operand(N, K, pad_b, dev, 2)
    sa = (2.0 ** rng.uniform(-8, 2, (M, K // 128))).astype(np.float32)
    sb = (2.0 ** rng.uniform(-8, 2, (N // 128, K // 128))).astype(np.float32)
    d_sa, d_sb = dev_arr(sa, dev), dev_arr(sb, dev)
    # rows and columns at the edges of tiles and wavefronts' parts, all the others against the other kernels
    rows = np.unique(np.concatenate([np.arange(18), np.arange(M - 18, M), rng.integers(0, M, 16)]))
    blocks = sorted({0, 1, N // 256, N // 128 - 1})
    cols = np.concatenate([np.arange(128 * b, 128 * b + 128) for b in blocks])
    ref, absdot = orc.gemm_nt_ref(A[dev_arr(rows, dev)][:, :K].cpu().numpy(), B[dev_arr(cols, dev)][:, :K].cpu().numpy(), sa[rows], sb[blocks],
                                  scale_mode=BLOCK)
    outs = {}
    for number, flag in kernels:
        kernel = ctypes.c_int(-1)
        cf.cf_fp8_gemm_route(M, N, K, 0, 0, BLOCK, 0, N + 8, flag, ctypes.byref(kernel))
        assert kernel.value == number
        C = torch.full((M, N + 8), -7.0, dtype=torch.bfloat16, device=dev)
        cf.cf_fp8_gemm_nt_bf16_ex(M, N, K, A, K + pad_a, 0, d_sa, B, K + pad_b, d_sb, BLOCK, 0, None, None, None, C, N + 8, flag, stream())
        assert bool((C[:, N:] == -7.0).all())
        got = orc.bf16_to_f32(bf16_bits(C[dev_arr(rows, dev)][:, dev_arr(cols, dev)]))
        orc.assert_gemm_close(got, ref, absdot, what=f"kernel {number}")
        outs[number] = C
    # each folds a scale group's products into its sums in the order of K, and these values' products add without rounding: the same bits
    first = outs[kernels[0][0]]
    assert all(torch.equal(first.view(torch.int16), c.view(torch.int16)) for c in outs.values())


@pytest.mark.parametrize("M,N,K", [(1000, 768, 2048), (2049, 4352, 8320)])
def test_block_scaled_kernels_on_values_of_every_exponent(cf, dev, M, N, K):
    """An MFMA rounds here: the two kernels that take a scale group in one still have the same bits, the third neighbouring ones."""
    case(f"block-scaled kernels, every exponent {M}x{N}x{K}")
    g = torch.Generator(device=dev).manual_seed(K)

    def fp8(*shape):
        t = torch.randint(0, 256, shape, dtype=torch.uint8, device=dev, generator=g)
        return torch.where((t & 0x7f) == 0x7f, 0x3c, t)

    A, B = fp8(M, K), fp8(N, K)
    sa, sb = torch.rand(M, K // 128, device=dev, generator=g) + 0.5, torch.rand(N // 128, K // 128, device=dev, generator=g) + 0.5
    outs = {}
    for number, flag in (RING, WIDE, SLIM):
        outs[number] = C = torch.empty((M, N), dtype=torch.bfloat16, device=dev)
        cf.cf_fp8_gemm_nt_bf16_ex(M, N, K, A, K, 0, sa, B, K, sb, BLOCK, 0, None, None, None, C, N, flag, stream())
    assert torch.equal(outs[6].view(torch.int16), outs[7].view(torch.int16))
    # of 768,000 outputs 36 differed, of 8,917,248 539, each by a rounding to bf16
    assert int((outs[2].view(torch.int16) != outs[6].view(torch.int16)).sum()) <= M * N // 1000
    assert float((outs[2].float() - outs[6].float()).norm() / outs[6].float().norm()) <= 1e-4
