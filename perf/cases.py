"""Timed cases of the transformer op set: what a program built on this library has it do on one MI355X.

The families, each with the range of sizes it stands for:

  gpt2         forward of the GPT-2-small-shaped decoder (logits and argmax), one short prompt to a full batch
  encoder      pre-LN transformer stack on resident activations, launch-bound at the small end
  sdpa         attention over whole sequences (prefill): causal or full, one or several query heads per K/V head
  decode       attention of one to four new tokens per sequence against a long padded K/V cache (grouped heads, masked)
  attn_step    training step of a pre-LN attention sublayer: forward, then every gradient
  head_step    training step of the LM head: logits, cross-entropy, gradients of the hidden states and of the table
  int8         dynamic-quantised int8 linear layer, from one token to a large batch
  row_ops      softmax, LayerNorm, RMSNorm, GELU and bias + residual over one activation tensor
  linear_f64   LayerNorm + linear training step in float64, the reference's default type
  host         three host-slice calls in a row, the way a CPU dispatcher hands single ops over

Tensors are torch tensors on the GPU, handed to the library as typed pointers; weights, descriptors, output buffers and
workspaces are made once in `prepare`, as a program would keep them, and a pass is the library calls alone.
"""
import math

import numpy as np
import torch

from frankentorch_amd import device, fused, kernel_hip
from frankentorch_amd.core import TensorMeta

F32, F64 = torch.float32, torch.float64
_NP = {torch.float32: np.float32, torch.float64: np.float64, torch.int64: np.int64, torch.int8: np.int8, torch.uint8: np.uint8}


class Tensor:
    """A torch tensor in the shape the device tier takes its operands: an address, a numpy dtype, a size."""

    def __init__(self, t):
        self.t = t
        self.ptr = t.data_ptr()
        self.dtype = np.dtype(_NP[t.dtype])
        self.size = t.numel()
        self.nbytes = t.numel() * t.element_size()


class _Maker:
    """Seeded inputs: one generator per state, on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(1000003 * int(seed) + 17)

    def normal(self, shape, std=1.0, mean=0.0, dtype=F32):
        t = torch.randn(shape, generator=self.g, device="cuda", dtype=dtype)
        return t if std == 1.0 and mean == 0.0 else t.mul_(std).add_(mean)

    def ids(self, n, below):
        return torch.randint(0, below, (n,), generator=self.g, device="cuda", dtype=torch.int64)


def _empty(shape, dtype=F32):
    return Tensor(torch.empty(shape, device="cuda", dtype=dtype))


# ---- the cases -------------------------------------------------------------------------------------------------------

GPT2 = dict(vocab=50257, max_pos=1024, d=768, heads=12, ffn=3072, layers=12)


def listed():
    return [
        # a full batch of full-length sequences through the decoder: evaluation, scoring, prefill (the largest case)
        dict(name="gpt2_b8_s1024", kind="gpt2", batch=8, seq=1024),
        # one short prompt: the first token of an interactive session; the weights are read once for 37 tokens
        dict(name="gpt2_b1_s37", kind="gpt2", batch=1, seq=37),
        # one 128-token transformer block of width 256 (the smallest case: seven launches of a few microseconds)
        dict(name="block_b1_s128_d256", kind="encoder", batch=1, seq=128, d=256, layers=1, tanh=False),
        # long-context causal attention at head size 128
        dict(name="sdpa_causal_b4_h32_s2048_d128", kind="sdpa", batch=4, hq=32, group=1, seq_q=2048, seq_k=2048, d=128, causal=True),
        # one token per sequence, 16 sequences, 32 query heads on 8 K/V heads, a cache padded to 3967 positions
        dict(name="decode_b16_hq32_hkv8_k3967", kind="decode", batch=16, hq=32, group=4, seq_q=1, seq_k=3967, d=128),
        # fine-tuning an attention sublayer of width 768 on three sequences of a ragged length
        dict(name="attn_step_b3_s777_d768", kind="attn_step", batch=3, seq=777, d=768, hd=64),
        # training the LM head over the GPT-2 vocabulary: rows that are no multiple of a 128-bit vector
        dict(name="head_step_2048x50257x768", kind="head_step", rows=2048, vocab=50257, d=768),
        # quantised linear layer on a large batch of tokens
        dict(name="int8_8192x4096x4096", kind="int8", m=8192, k=4096, n=4096),
        # the same weights for the 13 tokens of a decode step: bound by reading them
        dict(name="int8_13x4096x11008", kind="int8", m=13, k=4096, n=11008),
        # the five row ops on one large activation tensor
        dict(name="row_ops_8192x4096", kind="row_ops", rows=8192, cols=4096, f64=False),
        # float64 training step of LayerNorm + linear, odd batch
        dict(name="linear_f64_1021x1024x1000", kind="linear_f64", rows=1021, d_in=1024, d_out=1000),
        # LayerNorm, linear and GELU called one by one on host arrays
        dict(name="host_1031x768x3072", kind="host", rows=1031, d_in=768, d_out=3072),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["gpt2", "encoder", "sdpa", "decode", "attn_step", "head_step", "int8", "row_ops", "linear_f64", "host"])
    if kind == "gpt2":
        batch = rng.randint(1, 8)
        return dict(kind=kind, batch=batch, seq=_log(rng, 1, 1024))
    if kind == "encoder":
        d = rng.choice([256, 384, 512, 768])
        return dict(kind=kind, batch=rng.randint(1, 8), seq=_log(rng, 16, 512), d=d, layers=rng.randint(1, 4), tanh=rng.random() < 0.5)
    if kind == "sdpa":
        seq = _log(rng, 128, 2048)
        return dict(kind=kind, batch=rng.randint(1, 4), hq=rng.choice([8, 12, 16, 32]), group=rng.choice([1, 1, 4]),
                    seq_q=seq, seq_k=seq if rng.random() < 0.7 else _log(rng, 128, 2048), d=rng.choice([64, 128]), causal=rng.random() < 0.6)
    if kind == "decode":
        return dict(kind=kind, batch=_log(rng, 1, 32), hq=32, group=rng.choice([1, 4, 8]), seq_q=rng.choice([1, 1, 1, 2, 4]),
                    seq_k=_log(rng, 256, 4096), d=rng.choice([64, 128]))
    if kind == "attn_step":
        return dict(kind=kind, batch=rng.randint(1, 6), seq=_log(rng, 64, 1024), d=rng.choice([256, 512, 768, 1024]), hd=rng.choice([64, 64, 128]))
    if kind == "head_step":
        return dict(kind=kind, rows=_log(rng, 64, 4096), vocab=_log(rng, 1000, 50257), d=64 * rng.randint(4, 16))
    if kind == "int8":
        return dict(kind=kind, m=_log(rng, 1, 8192), k=64 * _log(rng, 12, 172), n=_log(rng, 768, 11008))
    if kind == "row_ops":
        f64 = rng.random() < 0.3
        return dict(kind=kind, rows=_log(rng, 16, 8192), cols=_log(rng, 64, 2048 if f64 else 8192), f64=f64)
    if kind == "linear_f64":
        return dict(kind=kind, rows=_log(rng, 32, 2048), d_in=_log(rng, 128, 2048), d_out=_log(rng, 128, 2048))
    return dict(kind=kind, rows=_log(rng, 32, 2048), d_in=64 * rng.randint(4, 16), d_out=64 * rng.randint(4, 48))


# ---- gpt2 and encoder ------------------------------------------------------------------------------------------------


def _layer(mk, d, ffn):
    w = lambda *s: mk.normal(s, 0.02).cpu().numpy()
    near1 = lambda n: mk.normal((n,), 0.1, 1.0).cpu().numpy()
    return {"ln1_w": near1(d), "ln1_b": w(d), "wq": w(d, d), "bq": w(d), "wk": w(d, d), "bk": w(d), "wv": w(d, d), "bv": w(d),
            "wo": w(d, d), "bo": w(d), "ln2_w": near1(d), "ln2_b": w(d), "w1": w(ffn, d), "b1": w(ffn), "w2": w(d, ffn), "b2": w(d)}


def _prepare_gpt2(case, mk):
    c = GPT2
    tokens = case["batch"] * case["seq"]
    wte, wpe = mk.normal((c["vocab"], c["d"]), 0.02).cpu().numpy(), mk.normal((c["max_pos"], c["d"]), 0.01).cpu().numpy()
    layers = [_layer(mk, c["d"], c["ffn"]) for _ in range(c["layers"])]
    model = fused.Gpt2Hip(wte, wpe, layers, mk.normal((c["d"],), 0.1, 1.0).cpu().numpy(), mk.normal((c["d"],), 0.02).cpu().numpy(),
                          c["heads"], 1e-5, gelu_tanh=True)
    ids = Tensor(mk.ids(tokens, c["vocab"]).to(F64))
    return dict(model=model, ids=ids, logits=_empty((tokens, c["vocab"])), best=_empty((tokens,)))


def _run_gpt2(case, s):
    s["model"].forward_dev(s["ids"], case["batch"], case["seq"], s["logits"], s["best"])
    return s["logits"].t, s["best"].t.view(torch.int32)  # the token ids are whole numbers held in float32


def _block_flops(batch, seq, d, ffn, causal=True):
    tokens = batch * seq
    pairs = seq * (seq + 1) // 2 if causal else seq * seq
    return 2 * tokens * d * (4 * d + 2 * ffn) + 4 * batch * d * pairs


def _work_gpt2(case):
    c = GPT2
    tokens = case["batch"] * case["seq"]
    flops = c["layers"] * _block_flops(case["batch"], case["seq"], c["d"], c["ffn"]) + 2 * tokens * c["d"] * c["vocab"]
    weights = c["layers"] * (4 * c["d"] ** 2 + 2 * c["d"] * c["ffn"] + 9 * c["d"] + c["ffn"]) + c["vocab"] * c["d"]
    return {"bytes": 4 * (weights + min(case["seq"], c["max_pos"]) * c["d"]) + 8 * tokens + 4 * tokens * (c["vocab"] + 1), "flops": flops}


def _prepare_encoder(case, mk):
    d = case["d"]
    tokens = case["batch"] * case["seq"]
    enc = fused.EncoderHip(d, d // 64, 4 * d, [_layer(mk, d, 4 * d) for _ in range(case["layers"])], 1e-5, causal=True, gelu_tanh=case["tanh"])
    return dict(enc=enc, x=Tensor(mk.normal((tokens, d))), out=_empty((tokens, d)))


def _run_encoder(case, s):
    s["enc"].forward_dev(s["x"], s["out"], case["batch"], case["seq"])
    return s["out"].t


def _work_encoder(case):
    d, n = case["d"], case["layers"]
    tokens = case["batch"] * case["seq"]
    return {"bytes": 4 * (n * (12 * d * d + 13 * d) + 2 * tokens * d), "flops": n * _block_flops(case["batch"], case["seq"], d, 4 * d)}


# ---- attention -------------------------------------------------------------------------------------------------------


def _prepare_sdpa(case, mk):
    b, hq, hkv, d = case["batch"], case["hq"], case["hq"] // case["group"], case["d"]
    q, k, v = mk.normal((b, hq, case["seq_q"], d)), mk.normal((b, hkv, case["seq_k"], d)), mk.normal((b, hkv, case["seq_k"], d))
    desc = device.sdpa_desc_gqa(b, hq, hkv, case["seq_q"], case["seq_k"], d, d, case["causal"])
    return dict(desc=desc, q=Tensor(q), k=Tensor(k), v=Tensor(v), out=_empty((b, hq, case["seq_q"], d)))


def _run_sdpa(case, s):
    device.sdpa_forward(s["desc"], device.default_scale(case["d"]), s["q"], s["k"], s["v"], s["out"])
    return s["out"].t


def _work_sdpa(case):
    sq, sk, d = case["seq_q"], case["seq_k"], case["d"]
    pairs = sum(min(i + 1, sk) for i in range(sq)) if case.get("causal") else sq * sk
    heads = case["batch"] * case["hq"]
    return {"bytes": 4 * d * (2 * heads * sq + 2 * heads // case["group"] * sk), "flops": 4 * d * heads * pairs}


def _prepare_decode(case, mk):
    s = _prepare_sdpa(dict(case, causal=False), mk)
    b, sq, sk = case["batch"], case["seq_q"], case["seq_k"]
    # each sequence has its own length; the padding behind it and the later ones of the new tokens are hidden
    length = torch.randint(max(sq, sk // 2), sk + 1, (b,), generator=mk.g, device="cuda")
    seen = length[:, None] - sq + 1 + torch.arange(sq, device="cuda")
    hidden = torch.arange(sk, device="cuda") >= seen[:, :, None]
    mask = torch.zeros(hidden.shape, device="cuda").masked_fill_(hidden, float("-inf"))
    s["mask"] = Tensor(mask[:, None].expand(b, case["hq"], sq, sk).contiguous())
    return s


def _run_decode(case, s):
    device.sdpa_forward_masked(s["desc"], device.default_scale(case["d"]), s["q"], s["k"], s["v"], s["mask"], case["seq_q"] * case["seq_k"], s["out"])
    return s["out"].t


def _work_decode(case):
    w = _work_sdpa(case)
    return {"bytes": w["bytes"] + 4 * case["batch"] * case["hq"] * case["seq_q"] * case["seq_k"], "flops": w["flops"]}


# ---- training step of an attention sublayer: y = x + Wo . attention(LN(x)) ----------------------------------------------


def _prepare_attn_step(case, mk):
    b, seq, d, hd = case["batch"], case["seq"], case["d"], case["hd"]
    t, h = b * seq, d // hd
    s = {n: Tensor(mk.normal((d, d), 0.02)) for n in ("wq", "wk", "wv", "wo")}
    s.update({n: Tensor(mk.normal((d,), 0.02)) for n in ("bq", "bk", "bv", "bo", "beta")})
    s.update(gamma=Tensor(mk.normal((d,), 0.1, 1.0)), x=Tensor(mk.normal((t, d))), dy=Tensor(mk.normal((t, d), 0.1)))
    for n in ("h", "lin", "qh", "kh", "vh", "ctxh", "ctx", "y", "dctx", "dctxh", "dqh", "dkh", "dvh", "dtok", "dh", "dh2", "dx0", "dx"):
        s[n] = _empty((t, d))
    for n in ("q", "k", "v", "o"):
        s["dw" + n], s["db" + n] = _empty((d, d)), _empty((d,))
    s["dgamma"], s["dbeta"] = _empty((d,)), _empty((d,))
    s["desc"] = device.sdpa_desc_contiguous(b * h, seq, seq, hd, hd, True)
    s["lin_bias"] = device.gemm_desc(t, d, d, trans_b=True, epilogue=device.EPI_BIAS)
    s["lin_bias_res"] = device.gemm_desc(t, d, d, trans_b=True, epilogue=device.EPI_BIAS | device.EPI_RESIDUAL)
    # the first backward calls size the workspaces the program keeps
    s["ws_lin"] = device.linear_backward(s["dy"], s["x"], s["wo"], s["dctx"], s["dwo"], s["dbo"], t, d, d)
    s["ws_ln"] = device.layer_norm_backward(s["dy"], s["x"], s["gamma"], s["dx0"], s["dgamma"], s["dbeta"], t, d, 1e-5)
    s["ws_sdpa"] = device.sdpa_backward(s["x"], s["x"], s["x"], s["dy"], b * h, seq, seq, hd, hd, device.default_scale(hd), True, s["dqh"], s["dkh"], s["dvh"])
    return s


def _run_attn_step(case, s):
    b, seq, d, hd = case["batch"], case["seq"], case["d"], case["hd"]
    t, h, scale = b * seq, d // hd, device.default_scale(hd)
    device.layer_norm(s["x"], s["gamma"], s["beta"], s["h"], t, d, 1e-5)
    for n in ("q", "k", "v"):
        device.gemm(s["lin_bias"], s["h"], s["w" + n], s["lin"], s["b" + n])
        device.permute_0213(s["lin"], s[n + "h"], b, seq, h, hd)
    device.sdpa_forward(s["desc"], scale, s["qh"], s["kh"], s["vh"], s["ctxh"])
    device.permute_0213(s["ctxh"], s["ctx"], b, h, seq, hd)
    device.gemm(s["lin_bias_res"], s["ctx"], s["wo"], s["y"], s["bo"], s["x"])
    # backward
    device.linear_backward(s["dy"], s["ctx"], s["wo"], s["dctx"], s["dwo"], s["dbo"], t, d, d, workspace=s["ws_lin"])
    device.permute_0213(s["dctx"], s["dctxh"], b, seq, h, hd)
    device.sdpa_backward(s["qh"], s["kh"], s["vh"], s["dctxh"], b * h, seq, seq, hd, hd, scale, True, s["dqh"], s["dkh"], s["dvh"], workspace=s["ws_sdpa"])
    for i, n in enumerate(("q", "k", "v")):
        device.permute_0213(s["d" + n + "h"], s["dtok"], b, h, seq, hd)
        device.linear_backward(s["dtok"], s["h"], s["w" + n], s["dh2"] if i else s["dh"], s["dw" + n], s["db" + n], t, d, d, workspace=s["ws_lin"])
        if i:
            device.add(s["dh"], s["dh2"], s["dh"], t * d)
    device.layer_norm_backward(s["dh"], s["x"], s["gamma"], s["dx0"], s["dgamma"], s["dbeta"], t, d, 1e-5, workspace=s["ws_ln"])
    device.add(s["dx0"], s["dy"], s["dx"], t * d)
    return {n: s[n].t for n in ("y", "dx", "dwq", "dwk", "dwv", "dwo", "dbq", "dbv", "dbo", "dgamma", "dbeta")}


def _work_attn_step(case):
    b, seq, d = case["batch"], case["seq"], case["d"]
    t = b * seq
    return {"bytes": 4 * (4 * t * d + 8 * d * d + 12 * d), "flops": 4 * 6 * t * d * d + (4 + 10) * b * d * (seq * (seq + 1) // 2)}


# ---- training step of the LM head ----------------------------------------------------------------------------------------


def _prepare_head_step(case, mk):
    rows, vocab, d = case["rows"], case["vocab"], case["d"]
    s = dict(x=Tensor(mk.normal((rows, d))), w=Tensor(mk.normal((vocab, d), 0.02)), target=Tensor(mk.ids(rows, vocab)),
             dloss=Tensor(torch.full((rows,), 1.0 / rows, device="cuda")), logits=_empty((rows, vocab)), loss=_empty((rows,)),
             dlogits=_empty((rows, vocab)), dx=_empty((rows, d)), dw=_empty((vocab, d)), desc=device.gemm_desc(rows, vocab, d, trans_b=True))
    s["ws"] = _empty((4,))  # a bias gradient would need one; without it the workspace is not touched
    return s


def _run_head_step(case, s):
    rows, vocab, d = case["rows"], case["vocab"], case["d"]
    device.gemm(s["desc"], s["x"], s["w"], s["logits"])
    device.cross_entropy_forward(s["logits"], s["target"], rows, vocab, s["loss"])
    device.cross_entropy_backward(s["logits"], s["target"], s["dloss"], rows, vocab, s["dlogits"])
    device.linear_backward(s["dlogits"], s["x"], s["w"], s["dx"], s["dw"], None, rows, d, vocab, workspace=s["ws"])
    return s["loss"].t, s["dx"].t, s["dw"].t


def _work_head_step(case):
    rows, vocab, d = case["rows"], case["vocab"], case["d"]
    return {"bytes": 4 * (2 * rows * d + 2 * vocab * d + 2 * rows) + 8 * rows, "flops": 6 * rows * vocab * d}


# ---- int8 linear -----------------------------------------------------------------------------------------------------------


def _prepare_int8(case, mk):
    m, k, n = case["m"], case["k"], case["n"]
    s = dict(x=Tensor(mk.normal((m, k), 3.0)), wq=_empty((n, k), torch.int8), ws=_empty((n,)), bias=Tensor(mk.normal((n,))), out=_empty((m, n)))
    device.quantize_rows_i8(Tensor(mk.normal((n, k), 0.5)), n, k, s["wq"], s["ws"])
    device.synchronize()
    s["work"] = Tensor(torch.empty(max(16, device.linear_int8_workspace_bytes(m, k)), device="cuda", dtype=torch.uint8))
    return s


def _run_int8(case, s):
    device.linear_int8_dynamic(s["x"], case["m"], case["k"], s["wq"], s["ws"], case["n"], s["bias"], s["out"], workspace=s["work"])
    return s["out"].t


def _work_int8(case):
    m, k, n = case["m"], case["k"], case["n"]
    return {"bytes": 4 * m * k + n * k + 8 * n + 4 * m * n, "flops": 2 * m * k * n}


# ---- row ops ---------------------------------------------------------------------------------------------------------------


def _prepare_row_ops(case, mk):
    rows, cols, dt = case["rows"], case["cols"], F64 if case["f64"] else F32
    s = dict(x=Tensor(mk.normal((rows, cols), dtype=dt)), res=Tensor(mk.normal((rows, cols), dtype=dt)), gamma=Tensor(mk.normal((cols,), 0.1, 1.0, dtype=dt)),
             beta=Tensor(mk.normal((cols,), 0.1, dtype=dt)), bias=Tensor(mk.normal((cols,), 0.1, dtype=dt)))
    s["y"] = [_empty((rows, cols), dt) for _ in range(5)]
    return s


def _run_row_ops(case, s):
    rows, cols, y = case["rows"], case["cols"], s["y"]
    device.softmax_lastdim(s["x"], y[0], rows, cols)
    device.layer_norm(s["x"], s["gamma"], s["beta"], y[1], rows, cols, 1e-5)
    device.rms_norm(s["x"], s["gamma"], y[2], rows, cols, 1e-6)
    device.gelu(s["x"], y[3], rows * cols)
    device.bias_residual_add(s["x"], s["bias"], s["res"], y[4], rows, cols)
    return [t.t for t in y]


def _work_row_ops(case):
    size = 8 if case["f64"] else 4  # five independent calls: each reads its own inputs (6 tensors in all) and writes its output
    return {"bytes": size * (11 * case["rows"] * case["cols"] + 4 * case["cols"]), "flops": 40 * case["rows"] * case["cols"]}


# ---- float64 training step: y = LN(x) . W^T + b ---------------------------------------------------------------------------------


def _prepare_linear_f64(case, mk):
    r, i, o = case["rows"], case["d_in"], case["d_out"]
    n = lambda shape, std=1.0, mean=0.0: Tensor(mk.normal(shape, std, mean, F64))
    s = dict(x=n((r, i)), gamma=n((i,), 0.1, 1.0), beta=n((i,), 0.1), w=n((o, i), 0.05), b=n((o,), 0.1), dy=n((r, o)))
    for name, shape in (("h", (r, i)), ("y", (r, o)), ("dh", (r, i)), ("dw", (o, i)), ("db", (o,)), ("dx", (r, i)), ("dgamma", (i,)), ("dbeta", (i,))):
        s[name] = _empty(shape, F64)
    s["desc"] = device.gemm_desc(r, o, i, trans_b=True, epilogue=device.EPI_BIAS)
    s["ws_lin"] = device.linear_backward(s["dy"], s["x"], s["w"], s["dh"], s["dw"], s["db"], r, i, o)
    s["ws_ln"] = device.layer_norm_backward(s["x"], s["x"], s["gamma"], s["dx"], s["dgamma"], s["dbeta"], r, i, 1e-5)
    return s


def _run_linear_f64(case, s):
    r, i, o = case["rows"], case["d_in"], case["d_out"]
    device.layer_norm(s["x"], s["gamma"], s["beta"], s["h"], r, i, 1e-5)
    device.gemm(s["desc"], s["h"], s["w"], s["y"], s["b"])
    device.linear_backward(s["dy"], s["h"], s["w"], s["dh"], s["dw"], s["db"], r, i, o, workspace=s["ws_lin"])
    device.layer_norm_backward(s["dh"], s["x"], s["gamma"], s["dx"], s["dgamma"], s["dbeta"], r, i, 1e-5, workspace=s["ws_ln"])
    return {n: s[n].t for n in ("y", "dx", "dw", "db", "dgamma", "dbeta")}


def _work_linear_f64(case):
    r, i, o = case["rows"], case["d_in"], case["d_out"]
    return {"bytes": 8 * (2 * r * i + 2 * r * o + 2 * i * o + 4 * i + 2 * o), "flops": 6 * r * i * o}


# ---- host slices -------------------------------------------------------------------------------------------------------------


def _prepare_host(case, mk):
    r, i, o = case["rows"], case["d_in"], case["d_out"]
    n = lambda shape, std=1.0, mean=0.0: mk.normal(shape, std, mean).cpu().numpy().reshape(-1)
    return dict(x=n((r, i)), gamma=n((i,), 0.1, 1.0), beta=n((i,), 0.1), w=n((o, i), 0.02), b=n((o,), 0.02), meta=TensorMeta.from_shape((r, o)))


def _run_host(case, s):
    r, i, o = case["rows"], case["d_in"], case["d_out"]
    h = kernel_hip.layer_norm_forward_f32(s["x"], s["gamma"], s["beta"], r, i, 1e-5)
    y = kernel_hip.linear_tensor_f32(h, s["w"], s["b"], r, i, o)
    return kernel_hip.gelu_tensor_contiguous_f32(y, s["meta"])


def _work_host(case):
    r, i, o = case["rows"], case["d_in"], case["d_out"]
    return {"bytes": 4 * (2 * r * i + 2 * i + r * i + o * i + o + r * o + 2 * r * o), "flops": 2 * r * i * o}


# ---- entry points ------------------------------------------------------------------------------------------------------------

_PREPARE = {"gpt2": _prepare_gpt2, "encoder": _prepare_encoder, "sdpa": _prepare_sdpa, "decode": _prepare_decode, "attn_step": _prepare_attn_step,
            "head_step": _prepare_head_step, "int8": _prepare_int8, "row_ops": _prepare_row_ops, "linear_f64": _prepare_linear_f64, "host": _prepare_host}
_RUN = {"gpt2": _run_gpt2, "encoder": _run_encoder, "sdpa": _run_sdpa, "decode": _run_decode, "attn_step": _run_attn_step, "head_step": _run_head_step,
        "int8": _run_int8, "row_ops": _run_row_ops, "linear_f64": _run_linear_f64, "host": _run_host}
_WORK = {"gpt2": _work_gpt2, "encoder": _work_encoder, "sdpa": _work_sdpa, "decode": _work_decode, "attn_step": _work_attn_step,
         "head_step": _work_head_step, "int8": _work_int8, "row_ops": _work_row_ops, "linear_f64": _work_linear_f64, "host": _work_host}

# Largest relative error (2-norm) and largest single difference of another correct implementation at the same precision: about
# four times what the families show against the same computation in float64 over their ranges of sizes. float32 sums of 50000
# terms are the widest (head_step); a token id may differ where two logits are closer than the logits' own error.
_TOLERANCE = {
    "gpt2": {"rel": 4.5e-6, "max": 3e-5, "differ": 2e-3},
    "encoder": {"rel": 1.2e-6, "max": 7e-6},
    "sdpa": {"rel": 2e-6, "max": 6e-5},
    "decode": {"rel": 4e-6, "max": 2.5e-5},
    "attn_step": {"rel": 4e-6, "max": 2.5e-5},
    "head_step": {"rel": 7e-6, "max": 1.2e-4},
    "int8": "exact",
    "row_ops": {"rel": 3.5e-7, "max": 2e-6},
    "row_ops_f64": {"rel": 1e-15, "max": 5e-15},
    "linear_f64": {"rel": 6e-15, "max": 4e-14},
    "host": {"rel": 2e-6, "max": 2e-5},
}


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, _Maker(seed))
    torch.cuda.synchronize()
    state["case"] = case
    return state


def run(state):
    case = state["case"]
    return _RUN[case["kind"]](case, state)


def work(case):
    return _WORK[case["kind"]](case)


def tolerance(case):
    return _TOLERANCE["row_ops_f64" if case.get("f64") else case["kind"]]
