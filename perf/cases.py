"""The calls that a trainer or a server built on this library makes, over the sizes it makes them at.

Eight kinds of work, each one pass through the public entry points of `Lib` (include/cf_fp8.h):

  linear       one FP8 linear layer on fp32 activations: per-tensor amax, scale, quantize, GEMM with bias
  mlp          the gated MLP forward with per-token / per-channel scales, from one token (decode) to a training batch
  block        a linear layer with 1x128 / 128x128 block scales
  mlp_backward the down projection's backward under delayed scaling: quantize dY, dX, dW, and the weight's refresh
  head         one chunk of the loss head: projection onto the vocabulary, cross-entropy, dX and dW
  moe          a routed SwiGLU expert layer: norm, routing, permute, expert bank, unpermute
  moe_train    the GELU expert bank with per-expert activation slots, forward and backward
  moe_drop_in  the GELU expert bank under the reference's own argument list (no workspace)
"""
import ctypes
import importlib

import torch

cf = importlib.import_module("__graft_entry__").load_package().lib()
DEV = torch.device("cuda:0")

E4M3_MAX, E5M2_MAX = 448.0, 57344.0
PER_TENSOR, ROW_COL, BLOCK_128 = 0, 1, 2
EPI_NONE, EPI_BIAS, EPI_SILU_GATE = 0, 1, 2
HISTORY = 16            # delayed-scaling history of a dense call site
SLOT_HISTORY = 8        # and of an expert's activation slot


def listed():
    return [
        # A small layer on its own: every launch counts.
        {"name": "linear_512", "kind": "linear", "tokens": 512, "k": 1024, "n": 1024},
        # Decode: a small batch of sequences, one token each, against a Llama-sized MLP.
        {"name": "mlp_decode_16", "kind": "mlp", "tokens": 16, "h": 4096, "i": 14336},
        # Prefill of a prompt whose length is a multiple of nothing.
        {"name": "mlp_prefill_1000", "kind": "mlp", "tokens": 1000, "h": 4096, "i": 14336},
        # A training batch through the same MLP: the library's headline shape.
        {"name": "mlp_train_8192", "kind": "mlp", "tokens": 8192, "h": 4096, "i": 14336},
        # Block-scaled layer at training size.
        {"name": "block_4096", "kind": "block", "tokens": 4096, "k": 7168, "n": 7168},
        # Backward of the down projection: a short batch (a token count that is no multiple of a GEMM's K step) ...
        {"name": "mlp_backward_2000", "kind": "mlp_backward", "tokens": 2000, "h": 4096, "i": 14336},
        # ... and the batch of mlp_train_8192.
        {"name": "mlp_backward_8192", "kind": "mlp_backward", "tokens": 8192, "h": 4096, "i": 14336},
        # One chunk of the loss head, padded GPT-2 vocabulary.
        {"name": "head_2048", "kind": "head", "tokens": 2048, "h": 4096, "v": 50304},
        # Routed experts at decode: a handful of rows per expert, every expert's weights touched.
        {"name": "moe_decode_64", "kind": "moe", "tokens": 64, "h": 2048, "i": 1408, "experts": 64, "top_k": 6},
        # Routed experts over a training batch.
        {"name": "moe_train_16384", "kind": "moe", "tokens": 16384, "h": 2048, "i": 1408, "experts": 64, "top_k": 6},
        # GELU experts of a training step, forward then backward.
        {"name": "moe_gelu_step_4096", "kind": "moe_train", "tokens": 4096, "h": 2048, "i": 1408, "experts": 64, "top_k": 6},
        # The reference trainer's own call of the expert bank.
        {"name": "moe_drop_in_2048", "kind": "moe_drop_in", "tokens": 2048, "h": 2048, "i": 1408, "experts": 64, "top_k": 6},
    ]


def _log_size(rng, lo, hi, multiple=1):
    n = int(round(lo * (hi / lo) ** rng.random()))
    return max(lo, min(hi, n // multiple * multiple if multiple > 1 else n))


def draw(rng):
    kind = rng.choice(["linear", "mlp", "mlp", "block", "mlp_backward", "head", "moe", "moe_train", "moe_drop_in"])
    if kind == "linear":
        return {"kind": kind, "tokens": _log_size(rng, 16, 4096), "k": rng.choice([512, 1024, 2048, 4096]),
                "n": rng.choice([512, 1024, 2048, 4096])}
    if kind == "mlp":
        h, i = rng.choice([(1024, 4096), (2048, 5632), (4096, 14336), (4096, 14336)])
        return {"kind": kind, "tokens": _log_size(rng, 1, 8192), "h": h, "i": i}
    if kind == "block":
        k, n = rng.choice([(2048, 7168), (4096, 4096), (7168, 2048), (7168, 7168)])
        return {"kind": kind, "tokens": _log_size(rng, 16, 4096), "k": k, "n": n}
    if kind == "mlp_backward":      # the FP8 weight gradient takes token counts that are multiples of 16
        h, i = rng.choice([(1024, 4096), (2048, 5632), (4096, 14336)])
        return {"kind": kind, "tokens": _log_size(rng, 256, 8192, 16), "h": h, "i": i}
    if kind == "head":
        v = rng.choice([32000, 50304, 128256])
        return {"kind": kind, "tokens": _log_size(rng, 128, 2048 if v < 60000 else 768, 8), "h": rng.choice([1024, 2048, 4096]), "v": v}
    h, i, e, k = rng.choice([(2048, 1408, 64, 6), (2048, 1408, 64, 6), (1024, 2048, 8, 2)])
    most = {"moe": 16384, "moe_train": 4096, "moe_drop_in": 2048}[kind]
    return {"kind": kind, "tokens": _log_size(rng, 16 if kind != "moe_train" else 256, most), "h": h, "i": i, "experts": e, "top_k": k}


# ---- inputs -------------------------------------------------------------------------------------------------------

class State:
    pass


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _normal(g, *shape, sigma=1.0, dtype=torch.bfloat16):
    return torch.randn(*shape, device=DEV, generator=g, dtype=torch.float32).mul_(sigma).to(dtype)


def _activations(g, rows, cols):
    """N(0,1) with one element in a thousand at +-40, as FFN activations have them."""
    x = torch.randn(rows, cols, device=DEV, generator=g, dtype=torch.float32)
    hit = torch.rand(rows, cols, device=DEV, generator=g) < 1e-3
    return torch.where(hit, torch.copysign(torch.full_like(x, 40.0), x), x).to(torch.bfloat16)


def _u8(*shape):
    return torch.empty(*shape, dtype=torch.uint8, device=DEV)


def _f32(*shape):
    return torch.empty(*shape, dtype=torch.float32, device=DEV)


def _bf16(*shape):
    return torch.empty(*shape, dtype=torch.bfloat16, device=DEV)


def _one(value=0.0):
    return torch.full((1,), float(value), dtype=torch.float32, device=DEV)


def _int(*shape):
    return torch.zeros(*shape, dtype=torch.int32, device=DEV)


def _channel_weight(g, rows, cols):
    """An E4M3 weight [rows, cols] with one descale per output channel."""
    q, s, d = _u8(rows, cols), _f32(rows), _f32(rows)
    cf.cf_fp8_quantize_rows(_normal(g, rows, cols, sigma=0.02), rows, cols, 0, q, s, d, _stream())
    return q, d


def _tensor_weight(w):
    """E4M3 bytes and device descale of a bf16 tensor under one scale."""
    amax, s, d, q = _one(), _one(), _one(), _u8(*w.shape)
    cf.cf_fp8_amax_bf16(w, w.numel(), amax, _stream())
    cf.cf_fp8_scale_from_amax(amax, E4M3_MAX, s, d, _stream())
    cf.cf_fp8_quantize_e4m3(w, q, s, w.numel(), _stream())
    return q, d


def _workspace(size_fn, *args):
    n = ctypes.c_size_t(0)
    size_fn(*args, ctypes.byref(n))
    return _u8(n.value), n.value       # torch's device allocations are 512-byte aligned


class Delayed:
    """Device state of one delayed-scaling call site in steady state."""

    def __init__(self, amax, fp8_max):
        self.amax = _one()
        self.scale, self.descale = _one(fp8_max / amax), _one(amax / fp8_max)
        self.scale_snap, self.descale_snap = _one(), _one()
        self.history = torch.full((HISTORY,), float(amax), dtype=torch.float32, device=DEV)
        self.cursor, self.count = _int(1), torch.full((1,), HISTORY, dtype=torch.int32, device=DEV)
        self.running, self.arrived = _one(), _int(1)

    def quantize(self, x, out, is_e5m2, st):
        cf.cf_fp8_quantize_delayed_step(x, out, x.numel(), is_e5m2, self.amax, self.scale, self.descale, self.scale_snap,
                                        self.descale_snap, self.history, HISTORY, self.cursor, self.count, self.running,
                                        self.arrived, st)


def _routing(s, g, T, E, k):
    """Route weights and row lists of random logits, and the buffers that hold them."""
    s.logits = torch.randn(T, E, device=DEV, generator=g)
    s.route = s.logits.clone()
    s.counts, s.offsets, s.rows = _int(E), _int(E), _int(E * T)


def _route(s, c, st):
    T, E, k = c["tokens"], c["experts"], c["top_k"]
    s.route.copy_(s.logits)            # the router's projection writes its scores here; top-k works in place
    cf.cf_moe_topk_route_f32(s.route, T, E, k, st, None, None, 1)
    cf.cf_moe_build_expert_row_lists(s.route, s.counts, s.rows, T, E, st)
    cf.cf_moe_expert_offsets_from_counts(s.counts, s.offsets, E, st)


def prepare(case, seed):
    s = State()
    s.case = c = dict(case)
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    globals()["_prepare_" + c["kind"]](s, c, g)
    return s


def run(state):
    return globals()["_run_" + state.case["kind"]](state, state.case, _stream())


# ---- one linear layer on fp32 activations ---------------------------------------------------------------------------

def _prepare_linear(s, c, g):
    M, K, N = c["tokens"], c["k"], c["n"]
    s.x = torch.randn(M, K, device=DEV, generator=g)
    s.w, s.wd = _tensor_weight(_normal(g, N, K, sigma=0.02))
    s.bias = _normal(g, N, sigma=0.02)
    s.amax, s.scale, s.descale = _one(), _one(), _one()
    s.xq, s.y = _u8(M, K), _bf16(M, N)


def _run_linear(s, c, st):
    M, K, N = c["tokens"], c["k"], c["n"]
    cf.cf_fp8_amax_f32(s.x, M * K, s.amax, st)
    cf.cf_fp8_scale_from_amax(s.amax, E4M3_MAX, s.scale, s.descale, st)
    cf.cf_fp8_quantize_f32_e4m3(s.x, s.xq, s.scale, M * K, st)
    cf.cf_fp8_gemm_nt_bf16_ex(M, N, K, s.xq, K, 0, s.descale, s.w, K, s.wd, PER_TENSOR, EPI_BIAS, s.bias, None, None, s.y, N, 0, st)
    return s.xq, s.descale, s.y


# ---- gated MLP ----------------------------------------------------------------------------------------------------------

def _prepare_mlp(s, c, g):
    M, H, I = c["tokens"], c["h"], c["i"]
    s.x = _activations(g, M, H)
    s.gate, s.gate_d = _channel_weight(g, I, H)
    s.up, s.up_d = _channel_weight(g, I, H)
    s.down, s.down_d = _channel_weight(g, H, I)
    s.xq, s.xs, s.xd = _u8(M, H), _f32(M), _f32(M)
    s.h = _bf16(M, I)
    s.hq, s.hs, s.hd = _u8(M, I), _f32(M), _f32(M)
    s.y = _bf16(M, H)


def _run_mlp(s, c, st):
    M, H, I = c["tokens"], c["h"], c["i"]
    cf.cf_fp8_quantize_rows(s.x, M, H, 0, s.xq, s.xs, s.xd, st)
    cf.cf_fp8_gemm_nt_bf16_ex(M, I, H, s.xq, H, 0, s.xd, s.gate, H, s.gate_d, ROW_COL, EPI_SILU_GATE, None, s.up, s.up_d, s.h, I, 0, st)
    cf.cf_fp8_quantize_rows(s.h, M, I, 0, s.hq, s.hs, s.hd, st)
    cf.cf_fp8_gemm_nt_bf16_ex(M, H, I, s.hq, I, 0, s.hd, s.down, I, s.down_d, ROW_COL, EPI_NONE, None, None, None, s.y, H, 0, st)
    return s.xq, s.xd, s.h, s.y


# ---- block-scaled linear layer ------------------------------------------------------------------------------------------

def _prepare_block(s, c, g):
    M, K, N = c["tokens"], c["k"], c["n"]
    s.x = _normal(g, M, K)
    s.w, ws, s.wd = _u8(N, K), _f32(N // 128, K // 128), _f32(N // 128, K // 128)
    cf.cf_fp8_quantize_block_128x128(_normal(g, N, K, sigma=0.02), N, K, s.w, ws, s.wd, _stream())
    s.xq, s.xs, s.xd, s.y = _u8(M, K), _f32(M, K // 128), _f32(M, K // 128), _bf16(M, N)


def _run_block(s, c, st):
    M, K, N = c["tokens"], c["k"], c["n"]
    cf.cf_fp8_quantize_block_1x128(s.x, M, K, s.xq, s.xs, s.xd, st)
    cf.cf_fp8_gemm_nt_bf16_ex(M, N, K, s.xq, K, 0, s.xd, s.w, K, s.wd, BLOCK_128, EPI_NONE, None, None, None, s.y, N, 0, st)
    return s.xq, s.xd, s.y


# ---- backward of a projection [tokens, i] -> [tokens, h] ---------------------------------------------------------------

def _prepare_mlp_backward(s, c, g):
    M, H, I = c["tokens"], c["h"], c["i"]
    s.dy = _normal(g, M, H, sigma=1e-3)
    s.site = Delayed(6e-3, E5M2_MAX)
    s.act = _normal(g, M, I)                                    # the projection's input, kept by the forward pass
    s.act_scale, s.act_d = _one(E4M3_MAX / 6.0), _one(6.0 / E4M3_MAX)
    s.w = _normal(g, H, I, sigma=0.02)                          # [out, in]
    s.amax, s.ws, s.wd = _one(), _one(), _one()
    s.fwd8, s.bwd8 = _u8(H, I), _u8(I, H)
    cf.cf_fp8_refresh_weight(s.w, s.fwd8, s.bwd8, s.amax, s.ws, s.wd, I, H, 1, 1, _stream())
    s.dyq, s.dyq_t = _u8(M, H), _u8(H, M)
    s.act8, s.act8_t = _u8(M, I), _u8(I, M)
    s.dx = _bf16(M, I)
    s.dw = torch.zeros(I, H, dtype=torch.float32, device=DEV)   # accumulated over micro-steps


def _run_mlp_backward(s, c, st):
    M, H, I = c["tokens"], c["h"], c["i"]
    cf.cf_fp8_quant_and_transpose_e4m3(s.act, s.act8, s.act8_t, s.act_scale, M, I, st)
    s.site.quantize(s.dy, s.dyq, 1, st)
    cf.cf_transpose_u8(s.dyq, s.dyq_t, M, H, st)
    cf.cf_fp8_gemm_tn_accum_f32(I, H, M, s.act8_t, s.act_d, s.dyq_t, s.site.descale_snap, s.dw, H, st)
    cf.cf_fp8_gemm_nt_bf16(M, I, H, s.dyq, H, 1, s.site.descale_snap, s.bwd8, s.wd, s.dx, I, st)
    cf.cf_fp8_refresh_weight(s.w, s.fwd8, s.bwd8, s.amax, s.ws, s.wd, I, H, 1, 1, st)     # after the optimizer's step
    return s.dx, s.dw, s.dyq_t, s.act8_t, s.fwd8, s.bwd8, s.wd, s.site.scale


# ---- loss head ----------------------------------------------------------------------------------------------------------

def _prepare_head(s, c, g):
    M, H, V = c["tokens"], c["h"], c["v"]
    s.x = _normal(g, M, H)
    w = _normal(g, V, H, sigma=0.02)
    amax, ws, s.wd = _one(), _one(), _one()
    s.fwd8, s.bwd8 = _u8(V, H), _u8(H, V)
    cf.cf_fp8_refresh_weight(w, s.fwd8, s.bwd8, amax, ws, s.wd, H, V, 1, 1, _stream())
    s.labels = torch.randint(0, V, (M,), device=DEV, generator=g, dtype=torch.int32)
    s.labels[::9] = -100                                        # ignored positions
    s.valid, s.loss = _int(1), _one()
    s.site = Delayed(6.0, E4M3_MAX)
    s.xq, s.logits, s.grad, s.grad8 = _u8(M, H), _bf16(M, V), _bf16(M, V), _u8(M, V)
    s.gscale, s.gd, s.gamax = _one(E5M2_MAX * M / 2.0), _one(2.0 / (E5M2_MAX * M)), _one()
    s.dx = _bf16(M, H)
    s.dw = torch.zeros(V, H, dtype=torch.float32, device=DEV)   # accumulated over the chunks of a step


def _run_head(s, c, st):
    M, H, V = c["tokens"], c["h"], c["v"]
    s.valid.zero_()
    s.loss.zero_()
    s.gamax.zero_()
    s.site.quantize(s.x, s.xq, 0, st)
    cf.cf_fp8_gemm_nt_bf16(M, V, H, s.xq, H, 0, s.site.descale_snap, s.fwd8, s.wd, s.logits, V, st)
    cf.cf_cross_entropy_count_valid(s.labels, M, s.valid, st)
    cf.cf_cross_entropy_fwd_bwd_chunk_quant_e5m2(s.logits, s.labels, s.loss, s.grad, s.grad8, s.gscale, s.gamax, M, V, s.valid, st)
    cf.cf_gemm_bf16_tn_accum_f32(V, H, M, s.grad, V, s.x, H, s.dw, H, st)
    cf.cf_fp8_gemm_nt_bf16(M, H, V, s.grad8, V, 1, s.gd, s.bwd8, s.wd, s.dx, H, st)
    return s.loss, s.logits, s.grad, s.gamax, s.dx, s.dw


# ---- routed SwiGLU experts --------------------------------------------------------------------------------------------

def _prepare_moe(s, c, g):
    T, H, I, E, k = (c[n] for n in ("tokens", "h", "i", "experts", "top_k"))
    s.x = _activations(g, T, H)
    s.gamma = (1.0 + 0.1 * torch.randn(H, device=DEV, generator=g)).to(torch.bfloat16)
    _routing(s, g, T, E, k)
    s.gate, s.gate_d = _channel_weight(g, E * I, H)
    s.up, s.up_d = _channel_weight(g, E * I, H)
    s.down, s.down_d = _channel_weight(g, E * H, I)
    s.xq, s.xs, s.xd = _u8(T, H), _f32(T), _f32(T)
    s.mixed = _bf16(T, H)
    s.ws, s.ws_bytes = _workspace(cf.cf_moe_grouped_swiglu_workspace_bytes, T * k, E, H, I)


def _run_moe(s, c, st):
    T, H, I, E, k = (c[n] for n in ("tokens", "h", "i", "experts", "top_k"))
    cf.cf_rmsnorm_clip_quantize_rows(s.x, s.gamma, T, H, 1e-6, 0.0, 0, None, None, s.xq, s.xs, s.xd, st)
    _route(s, c, st)
    s.mixed.zero_()
    cf.cf_moe_grouped_swiglu_forward_fp8(s.xq, s.xd, s.route, s.counts, s.offsets, s.rows, s.gate, s.gate_d, s.up, s.up_d,
                                         s.down, s.down_d, s.mixed, T, H, I, E, T * k, s.ws, s.ws_bytes, st)
    return s.xq, s.xd, s.route, s.counts, s.mixed


# ---- GELU experts: training step, and the call of the reference trainer -------------------------------------------------

def _gelu_bank(s, c, g):
    T, H, I, E, k = (c[n] for n in ("tokens", "h", "i", "experts", "top_k"))
    s.hidden = _normal(g, T, H)
    s.hq, s.hd = _tensor_weight(s.hidden)
    _routing(s, g, T, E, k)
    _route(s, c, _stream())
    s.fc_in, s.fc_out = _normal(g, E * I, H, sigma=0.02), _normal(g, E * H, I, sigma=0.02)
    s.fc_in8, s.fc_in_d = _tensor_weight(s.fc_in)
    s.fc_out8, s.fc_out_d = _tensor_weight(s.fc_out)
    s.mixed = _bf16(T, H)


def _prepare_moe_train(s, c, g):
    T, H, I, E, k = (c[n] for n in ("tokens", "h", "i", "experts", "top_k"))
    _gelu_bank(s, c, g)
    s.words = int(cf.raw_cf_act_slot_state_words(SLOT_HISTORY))
    s.bank = torch.zeros(E, s.words, dtype=torch.float32, device=DEV)
    s.bank[:, 1], s.bank[:, 3] = E4M3_MAX / 4.0, E4M3_MAX / 4.0
    s.bank[:, 2], s.bank[:, 4] = 4.0 / E4M3_MAX, 4.0 / E4M3_MAX
    s.fws, s.fws_bytes = _workspace(cf.cf_moe_grouped_gelu_workspace_bytes, T, T * k, E, H, I)
    s.bws, s.bws_bytes = _workspace(cf.cf_moe_grouped_gelu_backward_workspace, T, T * k, E, H, I, None)
    s.d_mixed = _normal(g, T, H, sigma=0.01)
    s.d_route, s.d_hidden = _f32(T, E), _bf16(T, H)
    s.g_in, s.g_out = torch.zeros_like(s.fc_in), torch.zeros_like(s.fc_out)     # accumulated over micro-steps


def _run_moe_train(s, c, st):
    T, H, I, E, k = (c[n] for n in ("tokens", "h", "i", "experts", "top_k"))
    s.mixed.zero_()
    cf.cf_moe_grouped_gelu_forward_fp8_slots(s.hq, s.hd, 0, s.route, s.counts, s.offsets, s.rows, s.fc_in8, s.fc_in_d,
                                             s.fc_out8, s.fc_out_d, s.mixed, T, H, I, E, T * k, s.bank, s.words, SLOT_HISTORY,
                                             0, 0, s.fws, s.fws_bytes, st)
    s.d_hidden.zero_()
    cf.cf_moe_grouped_gelu_backward_fp8_slots(s.d_mixed, s.hq, s.hd, 0, s.hidden, s.route, s.counts, s.offsets, s.rows,
                                              s.fc_in8, s.fc_in_d, s.fc_out8, s.fc_out_d, s.fc_in, s.fc_out, s.d_route,
                                              s.g_in, s.g_out, s.d_hidden, T, H, I, E, T * k, s.bank, s.words, SLOT_HISTORY,
                                              0, s.bws, s.bws_bytes, st)
    return s.mixed, s.d_route, s.d_hidden, s.g_in, s.g_out, s.bank[:, 1:5]


def _prepare_moe_drop_in(s, c, g):
    _gelu_bank(s, c, g)
    s.fc_in = s.fc_out = None


def _run_moe_drop_in(s, c, st):
    T, H, I, E, k = (c[n] for n in ("tokens", "h", "i", "experts", "top_k"))
    s.mixed.zero_()
    cf.cf_moe_grouped_expert_forward_fp8(s.hq, s.hd, 0, s.route, s.counts, s.offsets, s.rows, s.fc_in8, s.fc_in_d, s.fc_out8,
                                         s.fc_out_d, s.mixed, T, H, I, E, T * k, st)
    return s.mixed


# ---- what a pass cannot do without ----------------------------------------------------------------------------------------

def work(case):
    c, kind = case, case["kind"]
    M = c["tokens"]
    if kind == "linear":        # x fp32, its bytes written and read, w, y
        K, N = c["k"], c["n"]
        return {"bytes": 4 * M * K + M * K + N * K + 2 * M * N, "flops": 2 * M * K * N}
    if kind == "mlp":           # x, q(x), three weights, h, y
        H, I = c["h"], c["i"]
        return {"bytes": 3 * M * H + 3 * H * I + 2 * M * I + 2 * M * H, "flops": 6 * M * H * I}
    if kind == "block":
        K, N = c["k"], c["n"]
        return {"bytes": 3 * M * K + K * N + 2 * M * N, "flops": 2 * M * K * N}
    if kind == "mlp_backward":  # dy, q(dy) twice, act, its bytes twice, dx, dw read and written; w and its bytes twice
        H, I = c["h"], c["i"]
        return {"bytes": 4 * M * H + 4 * M * I + 2 * M * I + 8 * H * I + 4 * H * I, "flops": 4 * M * H * I}
    if kind == "head":          # x, head twice, logits and gradient, dx, dw read and written
        H, V = c["h"], c["v"]
        return {"bytes": 5 * M * H + 2 * V * H + 5 * M * V + 8 * V * H, "flops": 6 * M * H * V}
    H, I, E, k = c["h"], c["i"], c["experts"], c["top_k"]
    R = M * k
    used = E * (1.0 - (1.0 - k / E) ** M)      # experts that some token selects, in expectation
    if kind == "moe":
        return {"bytes": 3 * M * H + 8 * M * E + 3 * used * H * I + 2 * M * H, "flops": 6 * R * H * I}
    if kind == "moe_drop_in":
        return {"bytes": M * H + 4 * M * E + 2 * used * H * I + 2 * M * H, "flops": 4 * R * H * I}
    # forward and recompute on E4M3 weights, bf16 weights, gradients read and written
    return {"bytes": 9 * M * H + 8 * M * E + 2 * used * H * I + 4 * used * H * I + 8 * used * H * I, "flops": (4 + 4 + 8) * R * H * I}


def tolerance(case):
    """Four times what a path differs from itself when the same inputs come with their contracted dimensions in another
    order.  One GEMM rounds to bf16 a little differently here and there; where its result is quantized again (mlp, moe,
    the GELU banks) a value at a rounding boundary, or a row's maximum, moves by a whole fp8 step.  Bytes, indices and
    scales made from inputs alone do not move at all."""
    return {
        "linear": {"rel": 1e-3, "max": 0.05},
        "mlp": {"rel": 1.3e-2, "max": 0.4},
        "block": {"rel": 1e-3, "max": 0.04},
        "mlp_backward": {"rel": 1e-3, "max": 0.04},
        "head": {"rel": 2.5e-3, "max": 0.07},
        "moe": {"rel": 1.6e-2, "max": 0.3},
        "moe_train": {"rel": 8e-3, "max": 0.3},
        "moe_drop_in": {"rel": 1.3e-2, "max": 0.1},
    }[case["kind"]]
