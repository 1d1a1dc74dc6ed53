"""Which kernel a dense FP8 GEMM runs on (cf_fp8_gemm_route; decided on the host).  Times are microseconds on one MI355X from
captured graphs, weights from HBM; each case names the two kernels between which the choice lies."""
import ctypes

import pytest

NAIVE, STAGED, RING, RING16, DUO, HALF, BLOCK_WIDE, BLOCK_SLIM, ACCUM_WIDE, SMALL = 0, 1, 2, 3, 4, 5, 6, 7, 8, 16
TENSOR, ROW_COL, BLOCK = 0, 1, 2
PLAIN, BIAS, GATE, ACCUM_F32, ACCUM_BF16 = range(5)
F_NAIVE, F_STAGED, F_DUO, F_MFMA32, F_RING, F_SMALL, F_HALF, F_WIDE, F_SLIM = 1, 2, 4, 16, 32, 64, 128, 4096, 8192


def route(cf, M, N, K, mode=TENSOR, epi=PLAIN, flags=0, pad=0, a_e5m2=0):
    k = ctypes.c_int(-1)
    cf.cf_fp8_gemm_route(M, N, K, a_e5m2, int(epi >= ACCUM_F32), mode, epi, N + pad, flags, ctypes.byref(k))
    return k.value


def test_flags_name_kernels(cf):
    assert route(cf, 512, 512, 512, flags=F_NAIVE) == NAIVE == route(cf, 512, 512, 40)
    assert route(cf, 512, 512, 512, flags=F_STAGED) == STAGED
    assert route(cf, 512, 512, 512, flags=F_RING) == RING16 and route(cf, 512, 512, 640, flags=F_RING) == RING
    assert route(cf, 512, 512, 512, flags=F_MFMA32) == RING
    assert route(cf, 512, 512, 512, flags=F_RING, mode=BLOCK) == RING
    assert route(cf, 512, 512, 512, flags=F_DUO) == DUO == route(cf, 512, 512, 512, flags=F_DUO, epi=ACCUM_BF16)
    for shape in range(6):
        assert route(cf, 512, 512, 512, flags=F_SMALL | shape << 8) == SMALL + shape
    assert route(cf, 512, 512, 512, flags=F_WIDE, mode=BLOCK) == BLOCK_WIDE and route(cf, 512, 640, 512, flags=F_SLIM, mode=BLOCK) == BLOCK_SLIM
    assert route(cf, 512, 512, 528, flags=F_WIDE, epi=ACCUM_F32) == ACCUM_WIDE
    assert route(cf, 14336, 4096, 2000, flags=F_DUO, epi=ACCUM_F32) == DUO and route(cf, 4096, 7168, 7168, flags=F_RING, mode=BLOCK) == RING
    # what a kernel does not take falls to the persistent or the staged one
    assert route(cf, 512, 512, 256, flags=F_WIDE, mode=BLOCK) == STAGED == route(cf, 512, 640, 512, flags=F_WIDE, mode=BLOCK)
    assert route(cf, 512, 512, 384, flags=F_SLIM, mode=BLOCK) == RING == route(cf, 512, 512, 512, flags=F_WIDE, epi=ACCUM_F32)
    assert route(cf, 512, 512, 512, flags=F_WIDE) == RING16 == route(cf, 512, 512, 512, flags=F_SLIM)
    assert route(cf, 512, 516, 512, flags=F_DUO) == STAGED
    assert route(cf, 512, 512, 512, flags=F_SMALL | 4 << 8, epi=GATE) == RING16
    assert route(cf, 512, 512, 512, flags=F_SMALL, epi=ACCUM_F32) == RING
    assert route(cf, 512, 512, 112, flags=F_SMALL) == STAGED


def test_estimates_ask_what_the_launch_asks(cf):
    """The persistent kernels' rate is assumed where they are launched, and only there."""
    # rows of C a multiple of 4 and not of 8: the accumulating ring takes them (306 us; two workgroups per CU 369)
    assert route(cf, 4096, 14336, 4096, epi=ACCUM_F32, pad=4) == RING
    assert route(cf, 4096, 14336, 4096, epi=ACCUM_BF16, pad=4) == RING
    # block scales with K of two K-tiles: the register-staged kernel (9.6 us against 4.4), priced as such
    assert route(cf, 1000, 512, 256, mode=BLOCK) >= SMALL


# ring (or register-staged, where N is no multiple of 256) against two workgroups per CU
@pytest.mark.parametrize("M,N,K,pad,epi,kernel", [
    (4096, 4096, 256, 0, ACCUM_BF16, RING),          # 21.8, 29.2
    (4096, 14336, 512, 0, ACCUM_BF16, RING),         # 74.2, 85.6
    (4096, 14336, 256, 0, ACCUM_BF16, RING),         # 64.1, 79.9
    (4096, 14336, 512, 4, ACCUM_F32, RING),          # 191, 222: rows of C that do not begin at a line
    (4100, 5636, 256, 0, ACCUM_F32, DUO),            # 116 (register-staged), 94
    (1024, 4096, 1024, 0, ACCUM_F32, DUO),           # 24.1, 13.5: 64 tiles
    (14336, 4096, 2000, 0, ACCUM_F32, ACCUM_WIDE),   # 262, 188 and, on 256 x 256 tiles, 164: K no multiple of 128
    (14336, 4096, 512 + 16, 0, ACCUM_F32, DUO),      # few K-tiles
    (14336, 4100, 1488, 0, ACCUM_F32, DUO),          # 209, 256 x 256 tiles 222: rows of C off the lines
    (10620, 3072, 800, 0, ACCUM_F32, DUO),           # 64.4, 70.7: two rounds, nearly full
    (10023, 4864, 928, 0, ACCUM_F32, DUO),           # 98.6, 104.8: three
    (14336, 4096, 1488, 0, ACCUM_F32, ACCUM_WIDE),   # 152, 144: three and a half
    (5120, 4096, 8176, 0, ACCUM_F32, DUO),           # 198, 210: a quarter of the second round filled
    (14336, 4096, 8192, 0, ACCUM_F32, RING),         # 389, 431
])
def test_accumulating_kernel(cf, M, N, K, pad, epi, kernel):
    assert route(cf, M, N, K, epi=epi, pad=pad) == kernel


# times of the tile shapes 32x32, 64x32, 64x64 and of the persistent kernels (128 x 256 tiles, and the one named)
@pytest.mark.parametrize("M,N,K,kernel", [
    (3000, 512, 4096, (BLOCK_SLIM,)),                # 34.3, 42.7, 29.1, 36.9, 27.0
    (3000, 512, 2048, (BLOCK_SLIM,)),                # 18.5, 22.7, 17.5, 16.3, 11.9
    (6000, 1000, 7168, (STAGED,)),                   # 197, 227, 137, 103 (register-staged)
    (4096, 1000, 2000, (STAGED,)),                   # 56.6, 70.0, 44.1, 35.6 (register-staged)
    (100, 1000, 4096, (SMALL + 1,)),                 # 16x16 8.3; 6.7, 8.9, 11.5, 55.5 (register-staged)
    (1024, 128, 7168, (SMALL + 1,)),                 # 16x16 12.5; 10.7, 15.5, 16.6, 97.4
    (1000, 512, 4096, (SMALL + 1, SMALL + 2)),       # 11.7, 12.1, 13.7, 28.6
    (4096, 7168, 7168, (BLOCK_WIDE,)),               # 210, 186
    (2560, 7168, 7168, (RING,)),                     # 154, 256 x 256 tiles 169: 1.1 rounds of those
    (3000, 7168, 2048, (RING,)),                     # 48.2, 256 x 256 tiles 54.5: few K-tiles
    (3500, 7168, 2048, (BLOCK_WIDE,)),               # 63.0, 54.2
    (2892, 11008, 640, (RING,)),                     # 27.7, 34.9
    (512, 7168, 7168, (BLOCK_SLIM,)),                # with the quantize 59.7, 43.3
    (700, 7168, 7168, (RING,)),                      # with the quantize 61.1, 128 x 128 tiles 70.7
])
def test_block_scaled_kernel(cf, M, N, K, kernel):
    assert route(cf, M, N, K, mode=BLOCK) in kernel


# 256 x 128-output persistent tiles against 128 x 64-output ones, two workgroups per CU
@pytest.mark.parametrize("M,N,K,kernel", [
    (512, 14336, 1024, RING16),                      # 20.8, 26.0: a round and three quarters of the smaller tiles
    (1024, 7168, 1024, RING16),                      # 20.1, 24.5
    (700, 7168, 2048, RING16),                       # 28.0, 32.7
    (1000, 896, 1024, DUO),                          # 56 tiles instead of 28
    (1500, 4096, 1024, DUO),                         # 19.1, 16.5
    (8192, 14336, 4096, RING16),
])
def test_silu_gate_kernel(cf, M, N, K, kernel):
    assert route(cf, M, N, K, mode=ROW_COL, epi=GATE) == kernel


# half tiles against the kernel that was the fastest of the others (two workgroups per CU, 128 x 128 small tiles, 256 x 256 tiles)
@pytest.mark.parametrize("M,N,K,epi,kernel", [
    (2048, 4096, 50304, PLAIN, HALF),                # 317 us, small tiles 361: 256 half tiles
    (2048, 4096, 14336, PLAIN, HALF),                # 90.8, two per CU 102.6
    (1000, 4096, 14336, PLAIN, SMALL + 5),           # 71.8, small tiles 52.8: 128 half tiles
    (4000, 2048, 32000, PLAIN, HALF),                # 189, small tiles 302
    (257, 14336, 4096, PLAIN, DUO),                  # 27.0, two per CU 24.9
    (8192, 4096, 14336, PLAIN, RING16),              # 346, 256 x 256 tiles 294
    (700, 14336, 4096, GATE, HALF),                  # 79.3, 256 x 256 tiles 88.7: 336 of those are one and a third rounds
    (8192, 14336, 4096, GATE, RING16),               # 733, 653
    (2665, 15960, 1584, PLAIN, DUO),                 # 104.8, two per CU 87.9: rows of K that share lines
    (1092, 9432, 3696, PLAIN, DUO),                  # 67.2, 57.2
    (869, 5808, 5072, PLAIN, HALF),                  # 40.7, 47.0: a part of a round
    (1348, 8352, 13296, GATE, HALF),                 # 297, small tiles 622
])
def test_half_tiles(cf, M, N, K, epi, kernel):
    assert route(cf, M, N, K, mode=ROW_COL, epi=epi) == kernel
    assert route(cf, M, N, K, mode=ROW_COL, epi=epi, flags=F_HALF) == HALF


def test_block_scales_shape_without_the_lds_for_its_scales(cf):
    """Groups of scales along K lie in LDS beside the operands: a 64 x 64 tile has room for 125 of them."""
    assert route(cf, 64, 4096, 16000, mode=BLOCK, flags=F_SMALL | 3 << 8) == SMALL + 3
    assert route(cf, 64, 4096, 16384, mode=BLOCK, flags=F_SMALL | 3 << 8) == RING
    assert SMALL <= route(cf, 64, 4096, 16384, mode=BLOCK) < SMALL + 3


def test_route_refuses_what_the_entry_points_refuse(cf):
    k = ctypes.c_int(-1)
    ask = lambda M, N, K, a, b, mode, epi, ldc: cf.raw_cf_fp8_gemm_route(M, N, K, a, b, mode, epi, ldc, 0, ctypes.byref(k))
    assert ask(64, 256, 256, 0, 0, BLOCK, BIAS, 256) == -2 and ask(64, 256, 256, 1, 0, BLOCK, PLAIN, 256) == -2
    assert ask(64, 256, 256, 0, 1, TENSOR, PLAIN, 256) == -2 and ask(64, 256, 256, 0, 1, ROW_COL, ACCUM_F32, 256) == -2
    assert ask(64, 256, 256, 0, 0, TENSOR, 5, 256) == -1 and ask(64, 256, 256, 0, 0, 3, PLAIN, 256) == -1
    assert ask(64, 256, 256, 0, 0, TENSOR, PLAIN, 255) == -1 and ask(0, 256, 256, 0, 0, TENSOR, PLAIN, 256) == -1
    assert k.value == -1
