"""GPU parity of the small-tile FP8 GEMM (gemm_direct.hip: K split over a workgroup's wavefronts, operands copied per
wavefront) at the edges of its tile shapes, and of the persistent kernels where CF_GEMM_FLAG_RING keeps them."""
import ctypes

import numpy as np
import pytest
import torch

import oracle_lib as orc
from gpu_util import bf16_bits, case, dev_arr, host, stream
from test_gpu_gemm import EPI_BIAS, EPI_NONE, EPI_SILU, PER_TENSOR, ROW_COL, rand_fp8, run_gemm, silu_ref

pytestmark = pytest.mark.gpu

BLOCK, RING, SMALL = 2, 32, 64
KERNEL_SMALL = 16


def runs_shape(cf, M, N, K, mode, epi, shape, a_e5m2=0):
    """Flags that ask for a tile shape, checked to get it."""
    k, flags = ctypes.c_int(-1), SMALL | shape << 8
    cf.cf_fp8_gemm_route(M, N, K, a_e5m2, 0, mode, epi, N + 8, flags, ctypes.byref(k))
    assert k.value == KERNEL_SMALL + shape
    return flags


def pick_rows(M, at_most=40):
    edges = [0, 15, 16, 31, 32, 63, 64, 127, 128, M - 1]
    some = np.random.default_rng(M).choice(M, min(M, at_most), replace=False)
    return np.unique(np.concatenate([some, [r for r in edges if r < M]]))


# every tile shape by its number: rows and columns that end inside a tile of each (150 = 9 x 16 + 6 = 2 x 64 + 22 = 128 + 22), five
# whole K-tiles (one wavefront has two) and 16 bytes; a single row and K-tile
@pytest.mark.parametrize("M,N,K", [(150, 200, 656), (1, 8, 128), (257, 392, 1152)])
@pytest.mark.parametrize("shape", range(6))
@pytest.mark.parametrize("kind", ["tensor", "rows_bias", "e5m2"])
def test_every_tile_shape(cf, dev, M, N, K, shape, kind):
    case(f"small-tile gemm shape {shape} {M}x{N}x{K} {kind}")
    e5m2, mode = kind == "e5m2", ROW_COL if kind == "rows_bias" else PER_TENSOR
    rng = np.random.default_rng(M + N + K + shape)
    A, sa = rand_fp8(rng, (M, K), e5m2=e5m2)
    B, sb = rand_fp8(rng, (N, K), sigma=0.02)
    if mode:
        sa, sb = (sa * rng.uniform(0.5, 2, M)).astype(np.float32), (sb * rng.uniform(0.5, 2, N)).astype(np.float32)
    flags = runs_shape(cf, M, N, K, mode, EPI_NONE, shape, int(e5m2))
    got = run_gemm(cf, dev, A, B, sa, sb, mode=mode, a_e5m2=e5m2, ldc=N + 8, flags=flags)
    assert np.isnan(got[:, N:]).all()
    ref, absdot = orc.gemm_nt_ref(A, B, np.atleast_1d(sa), np.atleast_1d(sb), scale_mode=mode, a_e5m2=e5m2)
    orc.assert_gemm_close(got[:, :N], ref, absdot, what=f"shape {shape} {M}x{N}x{K}")
    if kind == "rows_bias":                      # added to the bf16 result
        bias = orc.bf16_from_f32(rng.standard_normal(N).astype(np.float32))
        biased = run_gemm(cf, dev, A, B, sa, sb, mode=mode, epi=EPI_BIAS, bias=bias, ldc=N + 8, flags=flags)
        want = orc.bf16_to_f32(orc.bf16_from_f32((got[:, :N] + orc.bf16_to_f32(bias)).astype(np.float32)))
        assert np.array_equal(biased[:, :N], want)


@pytest.mark.parametrize("M,N,K", [(150, 200, 656), (257, 392, 1152)])
@pytest.mark.parametrize("shape", range(4))
@pytest.mark.parametrize("mode", [PER_TENSOR, ROW_COL])
def test_every_tile_shape_silu_gate(cf, dev, M, N, K, shape, mode):
    case(f"small-tile gemm silu-gate shape {shape} {M}x{N}x{K} mode={mode}")
    rng = np.random.default_rng(M + N + shape)
    A, sa = rand_fp8(rng, (M, K))
    G, sg = rand_fp8(rng, (N, K), sigma=0.02)
    U, su = rand_fp8(rng, (N, K), sigma=0.02)
    if mode:
        sa = (sa * rng.uniform(0.5, 2, M)).astype(np.float32)
        sg, su = (sg * rng.uniform(0.5, 2, N)).astype(np.float32), (su * rng.uniform(0.5, 2, N)).astype(np.float32)
    got = run_gemm(cf, dev, A, G, sa, sg, mode=mode, epi=EPI_SILU, B2=U, sb2=su, ldc=N + 8,
                   flags=runs_shape(cf, M, N, K, mode, EPI_SILU, shape))
    assert np.isnan(got[:, N:]).all()
    gref, _ = orc.gemm_nt_ref(A, G, np.atleast_1d(sa), np.atleast_1d(sg), scale_mode=mode, want_abs=False)
    uref, _ = orc.gemm_nt_ref(A, U, np.atleast_1d(sa), np.atleast_1d(su), scale_mode=mode, want_abs=False)
    exact = silu_ref(gref, uref)
    assert np.sqrt(((got[:, :N] - exact) ** 2).sum() / (exact ** 2).sum()) <= 4e-3      # three bf16 roundings


# the last: 112 groups of scales along K, the most LDS
@pytest.mark.parametrize("M,N,K", [(150, 200, 656), (1, 136, 128), (70, 136, 14336)])
@pytest.mark.parametrize("shape", range(4))
def test_every_tile_shape_block_scales(cf, dev, M, N, K, shape):
    case(f"small-tile gemm block scales shape {shape} {M}x{N}x{K}")
    rng = np.random.default_rng(M + K + shape)
    A, _ = rand_fp8(rng, (M, K))
    B, _ = rand_fp8(rng, (N, K), sigma=0.02)
    sa = rng.uniform(0.5, 2, (M, -(-K // 128))).astype(np.float32)
    sb = rng.uniform(0.5, 2, (-(-N // 128), -(-K // 128))).astype(np.float32)
    got = run_gemm(cf, dev, A, B, sa, sb, mode=BLOCK, ldc=N + 8, flags=runs_shape(cf, M, N, K, BLOCK, EPI_NONE, shape))
    assert np.isnan(got[:, N:]).all()
    ref, absdot = orc.gemm_nt_ref(A, B, sa, sb, scale_mode=BLOCK)
    orc.assert_gemm_close(got[:, :N], ref, absdot, what=f"block shape {shape} {M}x{N}x{K}")


# What the sizes choose.  One row; one 16-row tile and its neighbours; a K of one tile, of fewer K-tiles than wavefronts, with a
# last K-tile of 16 and of 112 bytes; columns that end inside a 16-column block, at an odd count
SHAPES = [(1, 40, 128), (16, 64, 256), (17, 33, 144), (15, 16, 624), (33, 520, 1264), (64, 1032, 512), (130, 1000, 400), (300, 2000, 528),
          (700, 2304, 1040), (1000, 4080, 4112)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("kind", ["tensor", "rows_bias", "e5m2"])
def test_small_tiles(cf, dev, M, N, K, kind):
    case(f"small-tile gemm {M}x{N}x{K} {kind}")
    rng = np.random.default_rng(M + N + K)
    A, sa = rand_fp8(rng, (M, K), e5m2=kind == "e5m2")
    B, sb = rand_fp8(rng, (N, K), sigma=0.02)
    mode, kw, bias = PER_TENSOR, {}, None
    if kind == "rows_bias":
        mode = ROW_COL
        sa = (sa * rng.uniform(0.5, 2, M)).astype(np.float32)
        sb = (sb * rng.uniform(0.5, 2, N)).astype(np.float32)
        bias = orc.bf16_from_f32(rng.standard_normal(N).astype(np.float32))
    pad = 3 if N % 2 else 8                      # an odd row stride of C: element stores; otherwise 8-byte stores
    got = run_gemm(cf, dev, A, B, sa, sb, mode=mode, a_e5m2=kind == "e5m2", ldc=N + pad,
                   epi=EPI_BIAS if bias is not None else EPI_NONE, bias=bias)
    assert np.isnan(got[:, N:]).all() and not np.isnan(got[:, :N]).any()
    r = pick_rows(M)
    ref, absdot = orc.gemm_nt_ref(A[r], B, np.atleast_1d(sa)[r] if mode else np.atleast_1d(sa), np.atleast_1d(sb), scale_mode=mode,
                                  a_e5m2=kind == "e5m2")
    if bias is not None:                         # bias is added to the bf16 result: one more rounding, of a larger value
        plain = run_gemm(cf, dev, A, B, sa, sb, mode=mode)
        orc.assert_gemm_close(plain[r], ref, absdot, what=f"{M}x{N}x{K}")
        want = orc.bf16_to_f32(orc.bf16_from_f32((plain + orc.bf16_to_f32(bias)).astype(np.float32)))
        assert np.array_equal(got[:, :N], want)
    else:
        orc.assert_gemm_close(got[r][:, :N], ref, absdot, what=f"{M}x{N}x{K}")


@pytest.mark.parametrize("M,N,K", [(1, 40, 128), (16, 128, 272), (31, 200, 656), (60, 1408, 400), (130, 3000, 1040)])
def test_small_tiles_silu_gate(cf, dev, M, N, K):
    case(f"small-tile gemm silu-gate {M}x{N}x{K}")
    rng = np.random.default_rng(M + N)
    A, sa = rand_fp8(rng, (M, K))
    G, sg = rand_fp8(rng, (N, K), sigma=0.02)
    U, su = rand_fp8(rng, (N, K), sigma=0.02)
    sa = (sa * rng.uniform(0.5, 2, M)).astype(np.float32)
    sg, su = (sg * rng.uniform(0.5, 2, N)).astype(np.float32), (su * rng.uniform(0.5, 2, N)).astype(np.float32)
    got = run_gemm(cf, dev, A, G, sa, sg, mode=ROW_COL, epi=EPI_SILU, B2=U, sb2=su, ldc=N + 8)
    assert np.isnan(got[:, N:]).all()
    gref, _ = orc.gemm_nt_ref(A, G, sa, sg, scale_mode=1, want_abs=False)
    uref, _ = orc.gemm_nt_ref(A, U, sa, su, scale_mode=1, want_abs=False)
    exact = silu_ref(gref, uref)
    rel = np.sqrt(((got[:, :N] - exact) ** 2).sum() / (exact ** 2).sum())
    assert rel <= 4e-3, rel                      # three bf16 roundings, as in the fused test of the large kernel


@pytest.mark.parametrize("M,N,K", [(1, 100, 128), (16, 256, 1000 // 16 * 16), (40, 520, 896), (100, 1000, 1152), (300, 2048, 640)])
def test_small_tiles_block_scales(cf, dev, M, N, K):
    case(f"small-tile gemm block scales {M}x{N}x{K}")
    rng = np.random.default_rng(M + K)
    A, _ = rand_fp8(rng, (M, K))
    B, _ = rand_fp8(rng, (N, K), sigma=0.02)
    kb, nb = -(-K // 128), -(-N // 128)
    sa = rng.uniform(0.5, 2, (M, kb)).astype(np.float32)
    sb = rng.uniform(0.5, 2, (nb, kb)).astype(np.float32)
    got = run_gemm(cf, dev, A, B, sa, sb, mode=BLOCK, ldc=N + 8)
    assert np.isnan(got[:, N:]).all()
    ref, absdot = orc.gemm_nt_ref(A, B, sa, sb, scale_mode=BLOCK)
    orc.assert_gemm_close(got[:, :N], ref, absdot, what=f"block {M}x{N}x{K}")


def check_grouped(cf, dev, counts, N, K, gate):
    E = len(counts)
    offsets = np.concatenate([[0], np.cumsum(counts)[:-1]]).astype(np.int32)
    total = int(counts.sum())
    case(f"small-tile grouped gemm total={total} N={N} gate={gate}")
    assert total <= 40 * E
    rng = np.random.default_rng(total)
    rows = 50
    A, sa = rand_fp8(rng, (rows, K))
    sa = (sa * rng.uniform(0.5, 2, rows)).astype(np.float32)
    B, sb = rand_fp8(rng, (E * N, K), sigma=0.02)
    U, su = rand_fp8(rng, (E * N, K), sigma=0.02)
    sb, su = (sb * rng.uniform(0.5, 2, E * N)).astype(np.float32), (su * rng.uniform(0.5, 2, E * N)).astype(np.float32)
    index = rng.integers(0, rows, total).astype(np.int32)
    d = lambda a: dev_arr(a, dev)
    sz = ctypes.c_size_t(0)
    assert cf.raw_cf_fp8_grouped_gemm_workspace_bytes(total, E, ctypes.byref(sz)) == 0
    ws = torch.empty(sz.value, dtype=torch.uint8, device=dev)
    C = torch.full((total + 1, N), float("nan"), dtype=torch.bfloat16, device=dev)
    cf.cf_fp8_grouped_gemm_nt_bf16_ex(total, N, K, E, d(counts), d(offsets), d(A), rows, K, d(index), d(sa), d(B), d(sb), ROW_COL,
                                      EPI_SILU if gate else EPI_NONE, d(U) if gate else None, d(su) if gate else None, C, N, ws,
                                      sz.value, stream())
    torch.cuda.synchronize()
    got = orc.bf16_to_f32(bf16_bits(C)).astype(np.float64)
    assert np.isnan(got[total]).all()
    for e in range(E):
        if counts[e] == 0:
            continue
        i = index[offsets[e]:offsets[e] + counts[e]]
        w = slice(e * N, (e + 1) * N)
        ref, absdot = orc.gemm_nt_ref(A[i], B[w], sa[i], sb[w], scale_mode=1)
        mine = got[offsets[e]:offsets[e] + counts[e]]
        if gate:
            uref, _ = orc.gemm_nt_ref(A[i], U[w], sa[i], su[w], scale_mode=1, want_abs=False)
            exact = silu_ref(ref, uref)
            assert np.sqrt(((mine - exact) ** 2).sum() / (exact ** 2).sum()) <= 4e-3, e
        else:
            orc.assert_gemm_close(mine, ref, absdot, what=f"expert {e}")


# counts times `scale`: 16-row tiles, then 32- and 64-row ones; the plain form takes 64 columns instead of 16 or 32 per workgroup
# where there are many
@pytest.mark.parametrize("gate,scale,N", [(False, 1, 128), (False, 1, 256), (False, 1, 520), (False, 2, 256), (False, 2, 1000), (False, 3, 256),
                                          (True, 1, 256), (True, 3, 256)])
def test_small_tiles_grouped(cf, dev, gate, scale, N):
    """Experts without rows, with one row, with a tile and a row more, and with rows in two entries of the row-tile table."""
    check_grouped(cf, dev, np.array([0, 1, 16, 17, 33, 130, 0, 3] + [0] * 16, np.int32) * scale, N, 384, gate)


# the same number of workgroups whatever the counts: all rows on one expert (one entry and several), on the first and the last,
# on just under and just over half of the experts, and no entry to spare
@pytest.mark.parametrize("rows", [{7: 90}, {0: 300}, {23: 600}, {0: 1, 23: 257}, {i: 17 for i in range(11)}, {i: 35 for i in range(13)},
                                  {i: 20 for i in range(23)}, {i: 33 for i in range(24)}])
@pytest.mark.parametrize("gate", [False, True])
def test_small_tiles_grouped_skewed(cf, dev, rows, gate):
    counts = np.zeros(24, np.int32)
    for e, n in rows.items():
        counts[e] = n
    check_grouped(cf, dev, counts, 256, 256, gate)


@pytest.mark.parametrize("M,N,K", [(300, 512, 512), (770, 256, 384), (1024, 1024, 256), (300, 264, 512), (512, 1000, 384), (256, 8, 256),
                                   (300, 11 * 256, 256)])
@pytest.mark.parametrize("mode", [PER_TENSOR, ROW_COL, BLOCK])
def test_ring_flag_keeps_the_persistent_kernels(cf, dev, M, N, K, mode):
    """The last shape has 22 tiles: a grid rounded up to 24 workgroups, two of them without a tile."""
    case(f"ring gemm {M}x{N}x{K} mode={mode}")
    rng = np.random.default_rng(M + N + K)
    A, sa = rand_fp8(rng, (M, K))
    B, sb = rand_fp8(rng, (N, K), sigma=0.02)
    if mode == ROW_COL:
        sa, sb = (sa * rng.uniform(0.5, 2, M)).astype(np.float32), (sb * rng.uniform(0.5, 2, N)).astype(np.float32)
    if mode == BLOCK:
        sa = (sa * rng.uniform(0.5, 2, (M, -(-K // 128)))).astype(np.float32)
        sb = (sb * rng.uniform(0.5, 2, (-(-N // 128), -(-K // 128)))).astype(np.float32)
    got = run_gemm(cf, dev, A, B, sa, sb, mode=mode, flags=RING)
    ref, absdot = orc.gemm_nt_ref(A, B, np.atleast_1d(sa), np.atleast_1d(sb), scale_mode=mode)
    orc.assert_gemm_close(got, ref, absdot, what=f"ring {M}x{N}x{K}")
