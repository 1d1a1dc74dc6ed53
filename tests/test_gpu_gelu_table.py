"""The forms that look GELU up in a table held in LDS (2^-18 <= |x| < 16, closed forms beside it) against the direct forms:
every bf16 value, on both sides of each line between the forms.  Same bits, so no tolerance.  That the direct forms are right is pinned
against the oracle in test_gpu_moe_grouped.py and test_gpu_moe_slots.py."""
import numpy as np
import pytest
import torch

from gpu_util import case, dev_arr, stream

pytestmark = pytest.mark.gpu


def values(n, dev, finite):
    """All bf16 values in turn, the rows full of non-finite ones made finite if asked."""
    x = torch.arange(n, device=dev, dtype=torch.int64).remainder(65536).to(torch.int32).to(torch.int16).view(torch.bfloat16).clone()
    # neighbours from all over the range, so that one row mixes table and direct values
    x = x[torch.randperm(n, device=dev, generator=torch.Generator(device=dev).manual_seed(n))]
    if finite: x = torch.where(x.float().abs() <= 3e38, x, torch.zeros_like(x))
    return x


@pytest.mark.parametrize("rows,K", [(1490, 1408), (1489, 1408), (2048, 1024), (4200, 512), (33000, 64), (1024, 2048), (1100, 2032), (6097, 2064),
                                    (6096, 2064), (3072, 4096), (3073, 4080)])
def test_rows_every_value(cf, dev, rows, K):
    case(f"gelu + per-row quantize, table against gelu_forward then quantize, rows={rows} K={K}")
    for finite in (False, True):
        x = values(rows * K, dev, finite).reshape(rows, K)
        x[::3] *= 2.0 ** -20 if finite else 1.0                            # rows whose largest value is small
        q = torch.full((rows, K), 0xEE, dtype=torch.uint8, device=dev); s = torch.zeros(rows, device=dev); d = torch.zeros(rows, device=dev)
        cf.cf_gelu_quantize_rows_e4m3(x, rows, K, q, s, d, stream())
        y = torch.empty_like(x); q2 = torch.zeros_like(q); s2 = torch.zeros_like(s); d2 = torch.zeros_like(d)
        cf.cf_gelu_forward_bf16(x, y, rows * K, stream())
        cf.cf_fp8_quantize_rows(y, rows, K, 0, q2, s2, d2, stream())
        torch.cuda.synchronize()
        assert torch.equal(q, q2)
        assert torch.equal(s.view(torch.int32), s2.view(torch.int32)) and torch.equal(d.view(torch.int32), d2.view(torch.int32))


@pytest.mark.parametrize("E,K,bound,recompute", [(8, 1408, 3100, 0), (1, 1408, 3100, 0), (64, 1408, 3100, 1), (100, 512, 8300, 0),
                                                 (7, 4096, 1100, 0), (100, 1408, 18000, 0), (64, 2048, 24600, 0), (300, 1408, 24000, 0),
                                                 (64, 2048, 24500, 1), (200, 1408, 3100, 0)])
@pytest.mark.parametrize("e5m2", [0, 1])
def test_grouped_every_value(cf, dev, E, K, bound, recompute, e5m2):
    """total_rows is an upper bound, so the same routing runs through the direct form (tight) and the table form (bound)."""
    case(f"grouped GELU quantize E={E} K={K} bound={bound} recompute={recompute} e5m2={e5m2}")
    total = min(2900, (4 << 20) // K - 8)
    assert total * K < (4 << 20) <= bound * K
    rng = np.random.default_rng(E * K)
    cut = np.sort(rng.integers(0, total + 1, E - 1)); counts = np.diff(np.concatenate([[0], cut, [total]])).astype(np.int32)
    if E > 2: counts[1] += counts[0]; counts[0] = 0                        # an expert without rows
    offsets = np.concatenate([[0], np.cumsum(counts)[:-1]]).astype(np.int32)
    x = values(bound * K, dev, True).reshape(bound, K)
    hist = 4
    stride = cf.raw_cf_act_slot_state_words(hist)
    init = torch.zeros((E, stride), dtype=torch.float32, device=dev)
    init[:, 1] = 50.0; init[:, 2] = 0.02; init[:, 3] = 50.0; init[:, 4] = 0.02; init[:, 16] = 6.0
    init.view(torch.int32)[:, 8] = 1; init.view(torch.int32)[:, 9] = 1
    got = []
    for rows in (total, bound):
        st = init.clone(); out = torch.full((bound, K), 0xEE, dtype=torch.uint8, device=dev); rd = torch.full((bound,), -1.0, device=dev)
        for _ in range(2):
            cf.cf_moe_grouped_quantize_delayed(x, out, K, E, dev_arr(counts, dev), dev_arr(offsets, dev), rows, st, stride, hist, e5m2, 1,
                                               recompute, rd, stream())
        torch.cuda.synchronize()
        got.append((out, rd, st))
    (o1, r1, s1), (o2, r2, s2) = got
    assert torch.equal(o1, o2) and torch.equal(r1, r2) and torch.equal(s1.view(torch.int32), s2.view(torch.int32))
    assert bool((o2[total:] == 0xEE).all()) and bool((r2[total:] == -1.0).all())
