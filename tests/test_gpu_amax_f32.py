"""cf_fp8_amax_f32 on both sides of the lines between its launch shapes, the largest magnitude at places where a pass over the tensor can
go wrong (first, last, last whole vector, remainder), NaN ignored.  A maximum is exact, so no tolerance."""
import pytest
import torch

from gpu_util import case, stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("n", [1, 3, (256 << 10) - 1, 256 << 10, (256 << 10) + 3, (1 << 20) + 5, (8 << 20) + 4100, 32 << 20, (32 << 20) + 1])
def test_amax_f32_launch_shapes(cf, dev, n, off):
    case(f"amax f32 n={n} off={off}")
    buf = torch.randn(n + off + 8, device=dev, generator=torch.Generator(device=dev).manual_seed(n))
    buf[:off] = 1e30; buf[off + n:] = 1e30                                 # what lies outside must not count
    x = buf[off:off + n]
    out = torch.full((1,), 7e20, device=dev)
    cf.cf_fp8_amax_f32(x, n, out, stream())
    assert float(out) == float(x.abs().max())
    for k, at in enumerate({0, n - 1, n // 4 * 4 - 1, max(n - 5, 0), n // 2} if n > 4 else {n - 1}):
        x[at] = -100.0 - k
        cf.cf_fp8_amax_f32(x, n, out, stream())
        assert float(out) == 100.0 + k, at
    if n > 3:
        x[1] = float("nan")
        cf.cf_fp8_amax_f32(x, n, out, stream())
        assert float(out) == float(torch.nan_to_num(x, nan=0.0).abs().max())
