"""Routing's lane exchanges and the offsets' scan, bit for bit against the oracle: the largest score in every lane of the wavefront in
turn, expert counts at the edges of its 16- and 32-lane groups, ties across them, the type's lowest value; expert counts around the
64 that the scan takes at a time."""
import numpy as np
import pytest
import torch

import oracle_lib as orc
from gpu_util import case, dev_arr, host, stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E", [1, 2, 4, 8, 15, 16, 17, 31, 32, 33, 48, 63, 64])
def test_topk_every_lane(cf, dev, E):
    case(f"top-k, the largest score in every lane, E={E}")
    rng = np.random.default_rng(E)
    x = rng.standard_normal((2 * E + 3, E)).astype(np.float32)
    for e in range(E):
        x[e, e] = 9.0                                   # lane e alone
        x[E + e] = -1.0; x[E + e, [e, (e + E // 2) % E]] = 2.0      # two equal ones, half the lanes apart
    x[2 * E] = np.finfo(np.float32).min; x[2 * E + 1] = 0.0; x[2 * E + 2, ::2] = np.finfo(np.float32).min
    for k in (1, 2, 6):
        d = torch.from_numpy(x.copy()).to(dev); rs = torch.empty(len(x), device=dev); sv = torch.empty(x.shape, device=dev)
        cf.cf_moe_topk_route_f32(d, len(x), E, k, stream(), rs, sv, 1)
        torch.cuda.synchronize()
        want = orc.moe_topk_route(x, k, True, want_saves=True)
        for got, w in zip((d, rs, sv), want): assert np.array_equal(host(got).view(np.uint32), w.view(np.uint32))


@pytest.mark.parametrize("E", [1, 63, 64, 65, 127, 128, 129, 1000, 2048])
def test_offsets(cf, dev, E):
    case(f"expert offsets E={E}")
    counts = np.random.default_rng(E).integers(0, 1000, E).astype(np.int32); counts[::5] = 0
    off = torch.full((E + 1,), -9, dtype=torch.int32, device=dev)
    cf.cf_moe_expert_offsets_from_counts(dev_arr(counts, dev), off, E, stream())
    torch.cuda.synchronize()
    assert np.array_equal(host(off)[:E], orc.moe_expert_offsets(counts)) and host(off)[E] == -9
