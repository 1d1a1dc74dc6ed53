"""GPU parity: the weight-gradient kernel of gemm_bf16_duo.hip where its tiles, steps and rules have their edges, on small
integers: every product and partial sum is exact in fp32, so the result must match a float64 matmul to the bit (bf16: its one
rounding)."""
import pytest
import torch

from gpu_util import case, stream

pytestmark = pytest.mark.gpu


def ints(g, *shape):
    return torch.randint(-4, 5, shape, generator=g).to(torch.bfloat16)


def padded(x, ld):
    out = torch.full((*x.shape[:-1], ld), float("nan"), dtype=x.dtype)
    out[..., :x.shape[-1]] = x
    return out


# tiles of 256 x 128 and of 128 x 256 (whichever are fewer), one column short of and beyond them; K around the steps of 32, the
# pairs of steps and the shortest pipeline of four; the last size is as large as what is streamed, but its rows begin off the lines;
# the two of 289 tiles have one tile per workgroup and two workgroups on some CUs: turns of eight steps, the last one short, and none;
# and 512 x 136 is as many tiles either way
@pytest.mark.parametrize("M,N,K", [(256, 128, 1), (128, 256, 31), (264, 120, 33), (120, 264, 64), (248, 136, 65), (8, 8, 127), (512, 384, 129),
                                   (384, 512, 200), (2048, 2056, 96), (5128, 5192, 40),
                                   (2056, 4104, 709), (4104, 2056, 100), (512, 136, 100)])
@pytest.mark.parametrize("f32", [True, False])
def test_wgrad_edges(cf, dev, M, N, K, f32):
    case(f"bf16 wgrad {M}x{N}x{K} f32 {f32}")
    g = torch.Generator().manual_seed(M + N + K)
    A, B = ints(g, K, M), ints(g, K, N)
    C0 = ints(g, M, N).to(torch.float32 if f32 else torch.bfloat16)
    lda, ldb, ldc = M + 8, N + 16, N + 4
    C = padded(C0, ldc).to(dev)
    call = cf.cf_gemm_bf16_tn_accum_f32 if f32 else cf.cf_gemm_bf16_tn_accum_bf16
    call(M, N, K, padded(A, lda).to(dev), lda, padded(B, ldb).to(dev), ldb, C, ldc, stream())
    want = (C0.double() + A.double().T @ B.double()).to(C0.dtype)
    got = C.cpu()
    assert torch.equal(got[:, :N], want)
    assert torch.isnan(got[:, N:]).all()           # the row padding of C is left alone


# operands so large that one workgroup of 256 x 256 per CU takes them: beyond 1.6 GB in several rounds of tiles, one column short of and
# beyond tiles, K one short of and beyond the pairs of 64; and in a single round of the smaller tiles
@pytest.mark.parametrize("M,N,K,f32", [(8200, 4088, 22527, True), (4104, 8184, 22529, False), (1136, 9976, 28203, True), (9976, 1136, 28292, False)])
def test_wgrad_large_operands(cf, dev, M, N, K, f32):
    case(f"bf16 wgrad {M}x{N}x{K} f32 {f32}, large operands")
    tiles = min(-(-M // 256) * -(-N // 128), -(-M // 128) * -(-N // 256))
    assert 2 * (M + N) * K > (600e6 if 256 < tiles <= 512 else 1600e6 / -(-tiles // 512))
    g = torch.Generator(device=dev).manual_seed(M)
    A, B = (torch.randint(-4, 5, (K, n + 8), generator=g, device=dev).to(torch.bfloat16) for n in (M, N))
    A[:, M:], B[:, N:] = float("nan"), float("nan")
    dt = torch.float32 if f32 else torch.bfloat16
    C = torch.full((M, N + 8), float("nan"), dtype=dt, device=dev)
    C0 = torch.randint(-4, 5, (M, N), generator=g, device=dev).to(dt)
    C[:, :N] = C0
    call = cf.cf_gemm_bf16_tn_accum_f32 if f32 else cf.cf_gemm_bf16_tn_accum_bf16
    call(M, N, K, A, M + 8, B, N + 8, C, N + 8, stream())
    # sums of at most 16 x 28292 in magnitude: exact in fp32 on either side
    want = (C0.float() + A[:, :M].float().T.contiguous() @ B[:, :N].float()).to(dt)
    assert torch.equal(C[:, :N], want) and torch.isnan(C[:, N:]).all()


# C larger than what is left to the caches: streamed where its rows begin at 128-byte lines, not where C itself begins off one
@pytest.mark.parametrize("M,N,ldc,f32", [(5000, 5168, 5184, True), (10008, 5168, 5184, False)])
@pytest.mark.parametrize("off", [0, 4])
def test_wgrad_large_c(cf, dev, M, N, ldc, f32, off):
    case(f"bf16 wgrad {M}x{N}, C of more than 96 MiB, f32 {f32} off {off}")
    dt = torch.float32 if f32 else torch.bfloat16
    assert ldc * dt.itemsize % 128 == 0 and M * ldc * dt.itemsize > 96 << 20
    g = torch.Generator().manual_seed(M + off)
    A, B = ints(g, 40, M).to(dev), ints(g, 40, N).to(dev)
    buf = torch.full((M * ldc + 64,), float("nan"), dtype=dt, device=dev)
    C = buf[off:off + M * ldc].view(M, ldc)
    C0 = torch.randint(-4, 5, (M, N), device=dev, generator=torch.Generator(device=dev).manual_seed(M)).to(dt)
    C[:, :N] = C0
    call = cf.cf_gemm_bf16_tn_accum_f32 if f32 else cf.cf_gemm_bf16_tn_accum_bf16
    call(M, N, 40, A, M, B, N, C, ldc, stream())
    want = (C0.double() + A.double().T.contiguous() @ B.double()).to(dt)
    assert torch.equal(C[:, :N], want)
    assert torch.isnan(C[:, N:]).all() and torch.isnan(buf[:off]).all() and torch.isnan(buf[off + M * ldc:]).all()


# rows per expert from none to several tiles' worth of steps; experts whose rows of tiles (6 and 11) end in a partial patch of four.
# The last two have at least 176 tiles for an XCD's 64 workgroups, so that each walks several: of 256 x 128 and of 128 x 256 (fp32: streamed).
SEVERAL = [40, 3, 64, 0, 65, 33, 1, 96, 31, 32, 70, 2, 129, 0, 17, 50]
@pytest.mark.parametrize("M,N,counts", [(264, 136, [0, 1, 63, 64, 65, 0, 129, 300, 5]), (136, 264, [40, 0, 0, 7]), (512, 136, [9, 0, 130, 3]),
                                        (1408, 1024, [70, 0, 33, 1, 0, 64, 97, 128, 3, 200, 0, 32]),
                                        (1416, 2056, SEVERAL), (1288, 2048, SEVERAL)])
@pytest.mark.parametrize("f32", [True, False])
def test_grouped_wgrad_edges(cf, dev, M, N, counts, f32):
    case(f"grouped bf16 wgrad {M}x{N} {counts} f32 {f32}")
    g = torch.Generator().manual_seed(sum(counts) + M)
    R, E = sum(counts), len(counts)
    A, B = ints(g, R, M), ints(g, R, N)
    C0 = ints(g, E, M, N).to(torch.float32 if f32 else torch.bfloat16)
    C0[counts.index(0)] = -0.0                      # an expert without rows keeps its bits
    offsets = [sum(counts[:e]) for e in range(E)]
    C = C0.to(dev)
    call = cf.cf_moe_grouped_gemm_bf16_tn_accum_f32 if f32 else cf.cf_moe_grouped_gemm_bf16_tn_accum_bf16
    call(M, N, R, E, torch.tensor(counts, dtype=torch.int32, device=dev), torch.tensor(offsets, dtype=torch.int32, device=dev),
         A.to(dev), M, B.to(dev), N, C, stream())
    got = C.cpu()
    for e, (o, n) in enumerate(zip(offsets, counts)):
        want = (C0[e].double() + A[o:o + n].double().T @ B[o:o + n].double()).to(C0.dtype) if n else C0[e]
        assert torch.equal(got[e], want), f"expert {e}"
        assert n or torch.equal(torch.signbit(got[e]), torch.signbit(want))


# rows so far apart that 32 bits do not hold the offset of a k row beyond the last: row 16 of one with 2^27 elements a row, row 8 of
# 2^28, row 9 of nearly that (which would land in row 1).  A wrapped row would be added a second time.
@pytest.mark.parametrize("K,ld", [(1, 1 << 27), (2, 1 << 28), (3, (1 << 28) - 8)])
@pytest.mark.parametrize("M,N", [(136, 264), (264, 120)])
def test_wgrad_row_stride(cf, dev, K, ld, M, N):
    case(f"bf16 wgrad {M}x{N}x{K}, {ld} elements a row")
    g = torch.Generator().manual_seed(M + K)
    A, B = ints(g, K, M), ints(g, K, N)

    def far(x):
        buf = torch.zeros((K - 1) * ld + x.shape[1], dtype=torch.bfloat16, device=dev)
        for k in range(K): buf[k * ld:k * ld + x.shape[1]] = x[k].to(dev)
        return buf
    a, b = far(A), far(B)
    want = (A.double().T @ B.double()).float()
    C = torch.zeros(M, N, device=dev)
    cf.cf_gemm_bf16_tn_accum_f32(M, N, K, a, ld, b, ld, C, N, stream())
    assert torch.equal(C.cpu(), want)
    if K > 1:                           # an expert per row
        C = torch.zeros(K, M, N, device=dev)
        counts, offsets = torch.ones(K, dtype=torch.int32, device=dev), torch.arange(K, dtype=torch.int32, device=dev)
        cf.cf_moe_grouped_gemm_bf16_tn_accum_f32(M, N, K, K, counts, offsets, a, ld, b, ld, C, stream())
        assert torch.equal(C.cpu(), (A.double()[:, :, None] * B.double()[:, None, :]).float())
