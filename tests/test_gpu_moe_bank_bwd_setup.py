"""The GELU bank's backward: what its first launch derives from the routing, under row offsets in any order, with gaps, overlaps and
ranges that end beyond the compact buffers; and the one pass that leaves GELU output and quantized bytes, against the two calls it
stands for."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_util import bf16_bits, case, dev_arr, dev_bf16, host, stream
from test_gpu_moe_bank_bwd import NAMES

pytestmark = pytest.mark.gpu


def run(cf, dev, rows, E, H, Ie, counts, offsets, total, seed=1):
    g = torch.Generator(device=dev).manual_seed(seed)
    lists = torch.zeros(E, rows, dtype=torch.int32, device=dev)
    for e, n in enumerate(counts):
        lists[e, :n] = torch.randperm(rows, generator=g, device=dev)[:n].sort().values.int()
    offs, size = (ctypes.c_size_t * len(NAMES))(), ctypes.c_size_t(0)
    cf.cf_moe_grouped_gelu_backward_workspace(rows, total, E, H, Ie, offs, ctypes.byref(size))
    ws = torch.full((size.value,), 0xA7, dtype=torch.uint8, device=dev)
    ws[offs[NAMES.index("PRE")]:] = 0           # no NaN patterns in rows that no expert has
    bf = lambda *s: torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)
    f8 = lambda *s: bf(*s).to(torch.float8_e4m3fn).view(torch.uint8)
    one = lambda v: torch.tensor([v], device=dev)
    words = int(cf.raw_cf_act_slot_state_words(4))
    slots = torch.zeros(E, words, device=dev)
    slots[:, 1:5] = torch.tensor([90.0, 1 / 90.0, 110.0, 1 / 110.0], device=dev)
    c, o = dev_arr(np.array(counts, np.int32), dev), dev_arr(np.array(offsets, np.int32), dev)
    d_rw = torch.full((rows, E), float("nan"), device=dev)
    cf.cf_moe_grouped_gelu_backward_fp8_slots(
        bf(rows, H), f8(rows, H), one(0.01), 0, bf(rows, H), torch.rand(rows, E, generator=g, device=dev), c, o, lists, f8(E, Ie, H), one(0.5),
        f8(E, H, Ie), one(0.25), bf(E, Ie, H), bf(E, H, Ie), d_rw, bf(E, Ie, H), bf(E, H, Ie), bf(rows, H), rows, H, Ie, E, total, slots, words,
        4, 0, ws, size.value, stream())
    torch.cuda.synchronize()

    def grab(name, dtype, *shape):
        n = int(np.prod(shape)) * torch.empty(0, dtype=dtype).element_size()
        return ws[offs[NAMES.index(name)]:][:n].view(dtype).view(*shape)

    return grab, host(lists), host(d_rw), (c, o, slots, words)


@pytest.mark.parametrize("rows,E,counts,offsets,total", [
    (300, 5, [70, 0, 30, 100, 5], [0, 70, 70, 100, 200], 205),              # back to back, one expert without rows
    (300, 5, [70, 20, 30, 100, 5], [130, 110, 80, 210, 3], 333),            # any order, gaps before, between and behind
    (300, 4, [70, 20, 60, 300], [0, 60, 40, 250], 300),                     # overlapping ranges; the last one cut at the buffers' end
    (300, 3, [10, 0, 0], [290, 0, 5], 320),                                 # zeros before the only range and behind it
    (64, 3, [0, 0, 0], [0, 0, 0], 64),                                      # nothing but zeros
    (9000, 2, [9000, 8000], [9100, 100], 18500),                            # several workgroups to an expert
    (40, 300, [1] * 40 + [0] * 260, list(range(39, -1, -1)) + [0] * 260, 64),        # more experts than a workgroup has lanes
])
def test_index_of_any_offsets(cf, dev, rows, E, counts, offsets, total):
    case(f"bank backward setup {rows} rows, {E} experts, total {total}")
    grab, lists, d_rw, _ = run(cf, dev, rows, E, 256, 256, counts, offsets, total)
    got = host(grab("INDEX", torch.int32, total))
    allowed = [set() for _ in range(total)]                 # where ranges overlap either entry will do
    for e, (n, o) in enumerate(zip(counts, offsets)):
        for s in range(max(0, min(n, total - o))):
            allowed[o + s].add(int(lists[e, s]))
    assert all(int(v) in (a or {0}) for v, a in zip(got, allowed))
    selected = np.zeros((rows, E), bool)
    for e, (n, o) in enumerate(zip(counts, offsets)):
        selected[lists[e, :max(0, min(n, total - o))], e] = True
    assert (d_rw[~selected] == 0).all()
    assert (host(grab("HIDDEN_DESCALE", torch.float32, rows)) == np.float32(0.01)).all()
    assert (host(grab("IN_DESCALE", torch.float32, E * 256)) == 0.5).all() and (host(grab("OUT_DESCALE", torch.float32, E * 256)) == 0.25).all()


@pytest.mark.parametrize("E,per,Ie", [(5, 60, 256), (64, 70, 1408), (64, 400, 1408)])     # plain passes, table dealt out, table in equal runs
def test_gelu_and_recompute_quantize_in_one_pass(cf, dev, E, per, Ie):
    case(f"bank backward gelu + quantize {E} experts x {per} x {Ie}")
    rng = np.random.default_rng(E)
    counts = [max(1, per + int(d)) for d in rng.integers(-9, 10, E)]
    offsets = np.concatenate([[0], np.cumsum(counts)[:-1]]).tolist()
    total, rows = int(sum(counts)), max(counts) + 7
    grab, _, _, (c, o, slots, words) = run(cf, dev, rows, E, 256, Ie, counts, offsets, total)
    pre = grab("PRE", torch.bfloat16, total, Ie).clone()
    post, q, rd = torch.empty_like(pre), torch.empty(total, Ie, dtype=torch.uint8, device=dev), torch.empty(total, device=dev)
    cf.cf_gelu_forward_bf16(pre, post, pre.numel(), stream())
    cf.cf_moe_grouped_quantize_delayed(post, q, Ie, E, c, o, total, slots, words, 4, 0, 0, 1, rd, stream())
    torch.cuda.synchronize()
    assert torch.equal(post.view(torch.int16), grab("POST", torch.int16, total, Ie))
    assert torch.equal(q, grab("POSTQ", torch.uint8, total, Ie))
    assert torch.equal(rd, grab("POST_DESCALE", torch.float32, total))
