"""GPU parity of the half-tile FP8 GEMM (gemm_half.hip) where its tiles, its pipeline and its epilogues have their edges."""
import numpy as np
import pytest

import oracle_lib as orc
from gpu_util import case
from test_gpu_gemm import EPI_BIAS, EPI_SILU, PER_TENSOR, ROW_COL, rand_fp8, run_gemm

pytestmark = pytest.mark.gpu

HALF = 128


# 256 x 128 and 128 x 256 tiles (whichever are fewer); a last K-tile of 16, 80 and 112 bytes, two and three K-tiles (the pipeline
# has four); N that ends 8 columns into a tile; more tiles than the card has CUs, so that workgroups go on from one to the next: 2816 x
# 3208 is 11 x 26 of 256 x 128 (and as many of the other), 640 x 14344 5 x 57 of 128 x 256 (339 of the other)
@pytest.mark.parametrize("M,N,K", [(256, 128, 144), (128, 256, 256), (300, 264, 208), (257, 392, 624), (1, 136, 2000), (2816, 3208, 384),
                                   (640, 14344, 384), (130, 8, 512)])
@pytest.mark.parametrize("kind", ["tensor", "rows", "e5m2", "e5m2_rows", "bias", "bias_rows", "e5m2_bias_rows"])
def test_half_forms(cf, dev, M, N, K, kind):
    case(f"half-tile gemm {M}x{N}x{K} {kind}")
    rng = np.random.default_rng(M + N + K)
    e5m2 = kind.startswith("e5m2")
    A, sa = rand_fp8(rng, (M, K), e5m2=e5m2)
    B, sb = rand_fp8(rng, (N, K), sigma=0.02)
    mode = ROW_COL if kind.endswith("rows") else PER_TENSOR
    if mode == ROW_COL:
        sa, sb = (sa * rng.uniform(0.5, 2, M)).astype(np.float32), (sb * rng.uniform(0.5, 2, N)).astype(np.float32)
    kw = dict(mode=mode, a_e5m2=e5m2, flags=HALF, ldc=N + 8)
    got = run_gemm(cf, dev, A, B, sa, sb, **kw)
    assert np.isnan(got[:, N:]).all()
    rows = np.unique(np.concatenate([np.arange(0, M, max(1, M // 60)), [M - 1]]))
    ref, absdot = orc.gemm_nt_ref(A[rows], B, np.atleast_1d(sa)[rows] if mode else np.atleast_1d(sa), np.atleast_1d(sb), scale_mode=mode,
                                  a_e5m2=e5m2)
    orc.assert_gemm_close(got[rows][:, :N], ref, absdot, what=f"{M}x{N}x{K}")
    if "bias" in kind:                           # added to the bf16 result
        bias = orc.bf16_from_f32(rng.standard_normal(N).astype(np.float32))
        biased = run_gemm(cf, dev, A, B, sa, sb, epi=EPI_BIAS, bias=bias, **kw)
        want = orc.bf16_to_f32(orc.bf16_from_f32((got[:, :N] + orc.bf16_to_f32(bias)).astype(np.float32)))
        assert np.array_equal(biased[:, :N], want)


# the gate's own tiles: 128 x 128 outputs; N that ends 8 columns into one and into a wavefront's half of one; several tiles per workgroup
@pytest.mark.parametrize("M,N,K", [(128, 128, 256), (300, 136, 400), (1, 8, 144), (257, 200, 272), (2200, 2312, 384)])
@pytest.mark.parametrize("mode", [PER_TENSOR, ROW_COL])
def test_half_silu_gate(cf, dev, M, N, K, mode):
    case(f"half-tile silu gate {M}x{N}x{K} mode {mode}")
    rng = np.random.default_rng(M + N + K)
    X, sx = rand_fp8(rng, (M, K))
    G, sg = rand_fp8(rng, (N, K), sigma=0.05)
    U, su = rand_fp8(rng, (N, K), sigma=0.05)
    if mode == ROW_COL:
        sx, sg, su = ((s * rng.uniform(0.5, 2, n)).astype(np.float32) for s, n in ((sx, M), (sg, N), (su, N)))
    got = run_gemm(cf, dev, X, G, sx, sg, mode=mode, epi=EPI_SILU, B2=U, sb2=su, flags=HALF, ldc=N + 8)
    assert np.isnan(got[:, N:]).all()
    # the two plain products of the same kernel sum K in the same order; the fused sigmoid is within an fp32 ulp or two, which moves
    # a product at a rounding boundary to the neighbouring bf16 value
    gate, up = (run_gemm(cf, dev, X, W, sx, sw, mode=mode, flags=HALF) for W, sw in ((G, sg), (U, su)))
    want = orc.bf16_to_f32(orc.swiglu_forward(orc.bf16_from_f32(gate.astype(np.float32)), orc.bf16_from_f32(up.astype(np.float32)))).astype(np.float64)
    assert np.all(np.abs(got[:, :N] - want) <= orc.bf16_ulp(want)) and (got[:, :N] != want).mean() < 0.01
