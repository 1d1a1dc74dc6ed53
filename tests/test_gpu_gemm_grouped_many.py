"""The grouped FP8 GEMM between 40 and 256 rows an expert, where few experts are walked in 64-row passes that run side by side: balanced and skewed
counts, passes that end one row early and late, entries of the row-tile table with fewer and with more workgroups than passes."""
import ctypes

import numpy as np
import pytest
import torch

import oracle_lib as orc
from gpu_util import bf16_bits, case, dev_arr, stream
from test_gpu_gemm import EPI_NONE, EPI_SILU, ROW_COL, rand_fp8, silu_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [
    [41] * 8, [64] * 8, [65, 63, 128, 129, 1, 0, 64, 33], [256] * 8, [255, 257, 0, 513, 1, 320, 64, 128],
    [0, 0, 0, 0, 0, 0, 0, 330], [2048, 0, 0, 0, 0, 0, 0, 0], [300, 0, 0, 40], [81], [256],
])
@pytest.mark.parametrize("gate", [False, True])
def test_grouped_passes(cf, dev, counts, gate):
    counts = np.array(counts, np.int32)
    E, N, K, rows, total = len(counts), 256, 384, 50, int(sum(counts))
    case(f"grouped gemm in passes counts={list(counts)} gate={gate}")
    assert 40 * E < total <= 256 * E
    offsets = np.concatenate([[0], np.cumsum(counts)[:-1]]).astype(np.int32)
    rng = np.random.default_rng(total)
    A, sa = rand_fp8(rng, (rows, K))
    sa = (sa * rng.uniform(0.5, 2, rows)).astype(np.float32)
    B, sb = rand_fp8(rng, (E * N, K), sigma=0.02)
    U, su = rand_fp8(rng, (E * N, K), sigma=0.02)
    sb, su = (sb * rng.uniform(0.5, 2, E * N)).astype(np.float32), (su * rng.uniform(0.5, 2, E * N)).astype(np.float32)
    index = rng.integers(0, rows, total).astype(np.int32)
    d = lambda a: dev_arr(a, dev)
    sz = ctypes.c_size_t(0)
    assert cf.raw_cf_fp8_grouped_gemm_workspace_bytes(total, E, ctypes.byref(sz)) == 0
    ws = torch.full((sz.value + 64,), 0x7f, dtype=torch.uint8, device=dev)
    C = torch.full((total + 1, N), float("nan"), dtype=torch.bfloat16, device=dev)
    cf.cf_fp8_grouped_gemm_nt_bf16_ex(total, N, K, E, d(counts), d(offsets), d(A), rows, K, d(index), d(sa), d(B), d(sb), ROW_COL,
                                      EPI_SILU if gate else EPI_NONE, d(U) if gate else None, d(su) if gate else None, C, N, ws,
                                      sz.value, stream())
    assert bool((ws[sz.value:] == 0x7f).all())
    got = orc.bf16_to_f32(bf16_bits(C)).astype(np.float64)
    assert np.isnan(got[total]).all()
    for e in np.flatnonzero(counts):
        i = index[offsets[e]:offsets[e] + counts[e]]
        w = slice(e * N, (e + 1) * N)
        ref, absdot = orc.gemm_nt_ref(A[i], B[w], sa[i], sb[w], scale_mode=1)
        mine = got[offsets[e]:offsets[e] + counts[e]]
        if gate:                                   # the bar of the other grouped tests of this epilogue
            uref, _ = orc.gemm_nt_ref(A[i], U[w], sa[i], su[w], scale_mode=1, want_abs=False)
            exact = silu_ref(ref, uref)
            assert np.sqrt(((mine - exact) ** 2).sum() / (exact ** 2).sum()) <= 4e-3, e
        else:
            orc.assert_gemm_close(mine, ref, absdot, what=f"expert {e}")


RING, PASSES = 32, 64 | 3 << 8          # flags of the dense form: the persistent kernel, the small tiles of 64 x 64


# times with passes and on the ring kernel
@pytest.mark.parametrize("E,N,K,per,kernel", [
    (24, 640, 5376, 186, RING),          # 77.6, 50.5: three passes an expert, and the first XCDs have most of them
    (32, 256, 4864, 239, RING),          # 59.3, 45.6
    (8, 1024, 2048, 64, PASSES),         # 10.1, 25.3
    (8, 1024, 2048, 250, PASSES),        # 19.9, 25.5
])
def test_which_kernel_takes_the_experts(cf, dev, E, N, K, per, kernel):
    """The two sum K in different orders, which shows where values of every exponent meet: an expert's rows have the bits of the dense product
    on the kernel that the grouped one took, and not all of the other one's."""
    case(f"grouped gemm, kernel of {E} experts {N}x{K} rows {per}")
    g = torch.Generator(device=dev).manual_seed(E + N)

    def fp8(*shape):
        t = torch.randint(0, 256, shape, dtype=torch.uint8, device=dev, generator=g)
        return torch.where((t & 0x7f) == 0x7f, 0x3c, t)

    total = E * per
    A, B = fp8(total, K), fp8(E, N, K)
    sa, sb = torch.rand(total, device=dev, generator=g) + 0.5, torch.rand(E, N, device=dev, generator=g) + 0.5
    counts = torch.full((E,), per, dtype=torch.int32, device=dev)
    offsets = torch.arange(E, dtype=torch.int32, device=dev) * per
    sz = ctypes.c_size_t(0)
    assert cf.raw_cf_fp8_grouped_gemm_workspace_bytes(total, E, ctypes.byref(sz)) == 0
    ws = torch.empty(sz.value, dtype=torch.uint8, device=dev)
    C = torch.empty((total, N), dtype=torch.bfloat16, device=dev)
    cf.cf_fp8_grouped_gemm_nt_bf16_ex(total, N, K, E, counts, offsets, A, total, K, None, sa, B, sb, ROW_COL, EPI_NONE, None, None, C, N, ws,
                                      sz.value, stream())
    for flag in (RING, PASSES):
        D = torch.empty_like(C)
        for e in range(E):
            rows = slice(e * per, (e + 1) * per)
            cf.cf_fp8_gemm_nt_bf16_ex(per, N, K, A[rows], K, 0, sa[rows].clone(), B[e], K, sb[e], ROW_COL, EPI_NONE, None, None, None, D[rows], N,
                                      flag, stream())
        assert torch.equal(C.view(torch.int16), D.view(torch.int16)) == (flag == kernel)
