"""GPU parity of the 128 x 128-tile FP8 GEMM with two workgroups per CU (gemm_duo.hip) beyond the forms that
test_gpu_gemm.py compares bit by bit: any scale mode, E5M2 activations, bias, N and K that end inside a tile, and the
accumulating forms."""
import numpy as np
import pytest
import torch

import oracle_lib as orc
from gpu_util import case
from test_gpu_gemm import EPI_BIAS, EPI_NONE, PER_TENSOR, ROW_COL, rand_fp8, run_accum, run_gemm

pytestmark = pytest.mark.gpu

DUO_IN_STEP = 12


# a last K-tile of 16, 80 and 112 bytes; two K-tiles with the second one cut; N that ends 8 columns into a tile; more tiles
# than workgroups (2816 x 3208: 22 x 26 tiles)
@pytest.mark.parametrize("M,N,K", [(128, 128, 144), (300, 264, 208), (257, 392, 624), (1, 136, 2000), (2816, 3208, 272), (130, 256, 512)])
@pytest.mark.parametrize("kind", ["tensor", "e5m2_rows", "bias"])
def test_duo_forms(cf, dev, M, N, K, kind):
    case(f"duo gemm {M}x{N}x{K} {kind}")
    rng = np.random.default_rng(M + N + K)
    A, sa = rand_fp8(rng, (M, K), e5m2=kind == "e5m2_rows")
    B, sb = rand_fp8(rng, (N, K), sigma=0.02)
    mode = ROW_COL if kind == "e5m2_rows" else PER_TENSOR
    if mode == ROW_COL:
        sa, sb = (sa * rng.uniform(0.5, 2, M)).astype(np.float32), (sb * rng.uniform(0.5, 2, N)).astype(np.float32)
    kw = dict(mode=mode, a_e5m2=kind == "e5m2_rows", flags=DUO_IN_STEP, ldc=N + 8)
    got = run_gemm(cf, dev, A, B, sa, sb, **kw)
    assert np.isnan(got[:, N:]).all()
    rows = np.unique(np.concatenate([np.arange(0, M, max(1, M // 60)), [M - 1]]))
    ref, absdot = orc.gemm_nt_ref(A[rows], B, np.atleast_1d(sa)[rows] if mode else np.atleast_1d(sa), np.atleast_1d(sb), scale_mode=mode,
                                  a_e5m2=kind == "e5m2_rows")
    orc.assert_gemm_close(got[rows][:, :N], ref, absdot, what=f"{M}x{N}x{K}")
    if kind == "bias":                           # added to the bf16 result
        bias = orc.bf16_from_f32(rng.standard_normal(N).astype(np.float32))
        biased = run_gemm(cf, dev, A, B, sa, sb, epi=EPI_BIAS, bias=bias, **kw)
        want = orc.bf16_to_f32(orc.bf16_from_f32((got[:, :N] + orc.bf16_to_f32(bias)).astype(np.float32)))
        assert np.array_equal(biased[:, :N], want)


@pytest.mark.parametrize("M,N,K", [(128, 128, 144), (300, 260, 208), (257, 388, 2000), (2000, 4100, 272), (130, 256, 512)])
@pytest.mark.parametrize("bf16_out", [False, True])
def test_duo_accumulate(cf, dev, M, N, K, bf16_out):
    case(f"duo wgrad accumulate {M}x{N}x{K} bf16={bf16_out}")
    rng = np.random.default_rng(M + N + K)
    Xt, sx = rand_fp8(rng, (M, K))
    dYt, sy = rand_fp8(rng, (N, K), e5m2=True, sigma=1e-3)
    C0 = rng.standard_normal((M, N + 4)) * 1e-3
    got = run_accum(cf, dev, Xt, dYt, sx, sy, C0, a_e5m2=False, b_e5m2=True, bf16_out=bf16_out, flags=DUO_IN_STEP, ldc=N + 4)
    held = C0.astype(np.float32).astype(np.float64)
    if bf16_out:
        held = orc.bf16_to_f32(orc.bf16_from_f32(C0.astype(np.float32))).astype(np.float64)
    assert np.array_equal(got[:, N:], held[:, N:])                     # columns beyond N: untouched
    rows = np.unique(np.concatenate([np.arange(0, M, max(1, M // 60)), [M - 1]]))
    ref, absdot = orc.gemm_nt_ref(Xt[rows], dYt, [sx], [sy], b_e5m2=True)
    want, mine = held[rows][:, :N] + ref, got[rows][:, :N]
    if bf16_out:
        assert np.all(np.abs(mine - want) <= 1.01 * orc.bf16_ulp(want) / 2 + orc.ACC_MFMA * absdot)
    else:
        assert np.all(np.abs(mine - want) <= orc.ACC_MFMA * absdot + 2.0 ** -22 * (np.abs(want) + np.abs(held[rows][:, :N])))
