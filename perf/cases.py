"""The calls whose speed this repository looks after, as a program that uses it makes them.

A case is a dict of plain values: its `kind` names one of the paths below, the rest are sizes and
options. `listed()` has the standing ones, `draw(rng)` gives others of the same ranges.

  linear   one weight-only projection, `w4a16_matmul` or `w8a16_matmul`, called eagerly: from one
           decode row (the smallest call there is) to the rows of a long prompt.
  mlp      the MLP halves of a few decoder layers at decode rows, through the runner's backend
           (norm -> gate_up -> activation -> down), replayed as one hipGraph as a decode loop does;
           consecutive layers have weights of their own, so they come from HBM.
  attend   the attention block of a prompt on the tiled KV cache (`prefill_attention`), with or
           without positions already in the cache (a continued conversation, a chunk of a prompt).
  decode   one token through a whole model (`QwenRunner`), a hipGraph replay, at some depth of its
           cache; logits come back.
  prompt   a whole prompt through a model, eagerly, as prompts of any length arrive; logits and the
           filled cache come back.
  convert  a weight into the packed format or back (`quantize_rtn`, `quantize_fp8`, `dequantize`,
           `dequantize_fp8`): what loading or exporting a checkpoint does for every projection.
  rows     the normalisation and the activation of a prompt's rows (`rmsnorm` with its residual,
           `swiglu_fused`).

Widths are those of the repository's configurations (hidden 1536 with 8960, 4096 with 14336) or
generic multiples of the int4 group.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path
from types import SimpleNamespace as Bag

import torch

PKG = Path(__file__).resolve().parent.parent / "llm-decode-kernels_amd"
if str(PKG) not in sys.path:
    sys.path.insert(0, str(PKG))

GROUP = 128
HEAD_DIM = 128
EPS = 1e-6
THETA = 1_000_000.0
VOCAB = 151936

# The most a drawn case may cost, as (bytes or flops / 50), the larger: the largest listed case's.
COST_CAP = 2 * 2048 * 14336 * 4096 / 50


# ------------------------------------------------------------------------------------ the cases
def listed() -> list[dict]:
    return [
        # the attention output projection of one decoded token: latency and the launch itself
        dict(name="linear_o_1row", kind="linear", fmt="int4", rows=1, n=1536, k=1536, bias=False),
        # a short prompt or a speculative batch, rows that divide no tile, with a bias
        dict(name="linear_100rows", kind="linear", fmt="int4", rows=100, n=14336, k=4096, bias=True),
        # a long prompt's up projection in int4: the largest product
        dict(name="linear_2048rows", kind="linear", fmt="int4", rows=2048, n=14336, k=4096, bias=False),
        # a prompt's down projection in e4m3, ragged rows, long K
        dict(name="linear_fp8_777rows", kind="linear", fmt="fp8", rows=777, n=4096, k=14336, bias=False),
        # single-stream decoding of the small model
        dict(name="mlp_1row", kind="mlp", fmt="int4", rows=1, hidden=1536, inter=8960, layers=8),
        # batched decoding of the 8B widths in e4m3, an odd batch
        dict(name="mlp_fp8_13rows", kind="mlp", fmt="fp8", rows=13, hidden=4096, inter=14336, layers=3),
        # the attention of a prompt of a few thousand tokens
        dict(name="attend_3000", kind="attend", tokens=3000, start=0, heads=12, kv=2),
        # one token deep in a long context, the whole model
        dict(name="decode_6000", kind="decode", fmt="int4", layers=8, hidden=1536, inter=8960, heads=12,
             kv=2, pos=6000, max_len=8192),
        # a page of text in, the whole model, e4m3 weights
        dict(name="prompt_fp8_511", kind="prompt", fmt="fp8", layers=4, hidden=1536, inter=8960, heads=12,
             kv=2, tokens=511, max_len=1024),
        # packing one 8B projection while loading a checkpoint
        dict(name="quantize_int4", kind="convert", fmt="int4", back=False, n=14336, k=4096, dtype="float16"),
        # e4m3 weights back to bf16, an odd number of channels
        dict(name="dequantize_fp8_odd", kind="convert", fmt="fp8", back=True, n=1533, k=8960,
             dtype="bfloat16"),
        # the elementwise half of a prompt layer, ragged rows
        dict(name="rows_1999", kind="rows", rows=1999, hidden=1536, inter=8960),
    ]


def _log(rng, lo, hi, step=1) -> int:
    """An integer spread over the logarithm of lo..hi, a multiple of `step`."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(-(-lo // step) * step, min(int(round(v / step)) * step, hi // step * step))


def draw(rng) -> dict:
    while True:
        case = _draw(rng)
        w = work(case)
        if max(w["bytes"], w["flops"] / 50) <= COST_CAP:
            return case


def _draw(rng) -> dict:
    kind = rng.choice(["linear", "linear", "mlp", "attend", "decode", "prompt", "convert", "rows"])
    fmt = rng.choice(["int4", "fp8"])
    if kind == "linear":
        return dict(kind=kind, fmt=fmt, rows=_log(rng, 1, 4096), n=_log(rng, 256, 17920, 4),
                    k=_log(rng, 512, 14336, GROUP), bias=rng.random() < 0.5)
    if kind == "mlp":
        return dict(kind=kind, fmt=fmt, rows=_log(rng, 1, 16), hidden=_log(rng, 1024, 4096, GROUP),
                    inter=_log(rng, 2816, 14336, GROUP), layers=rng.randint(2, 6))
    if kind == "attend":
        heads, kv = rng.choice([(12, 2), (32, 8), (16, 16), (28, 4)])
        tokens = _log(rng, 17, 6000)
        start = rng.choice([0, 0, _log(rng, 1, 4000)])
        return dict(kind=kind, tokens=tokens, start=start, heads=heads, kv=kv)
    if kind in ("decode", "prompt"):
        hidden, inter, heads, kv = rng.choice([(1536, 8960, 12, 2), (1024, 2816, 8, 2), (2048, 5632, 16, 4)])
        size = dict(kind=kind, fmt=fmt, layers=rng.randint(2, 6), hidden=hidden, inter=inter, heads=heads, kv=kv)
        if kind == "decode":
            pos = _log(rng, 32, 16000)
            return dict(size, pos=pos, max_len=-(-(pos + rng.randint(32, 2 * pos)) // 32) * 32)
        tokens = _log(rng, 17, 2048)
        return dict(size, tokens=tokens, max_len=-(-(tokens + rng.randint(32, 1024)) // 32) * 32)
    if kind == "convert":
        back = rng.random() < 0.5
        dtype = "float16" if back and fmt == "int4" else rng.choice(["float16", "bfloat16", "float32"])
        return dict(kind=kind, fmt=fmt, back=back, n=_log(rng, 256, 17920), k=_log(rng, 512, 14336, GROUP),
                    dtype=dtype)
    return dict(kind=kind, rows=_log(rng, 1, 4096), hidden=_log(rng, 512, 8192, 8),
                inter=_log(rng, 1024, 14336, 8))


# ------------------------------------------------------------------------------------- the inputs
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape, std: float = 1.0, dtype=torch.float16) -> torch.Tensor:
    return (torch.randn(*shape, generator=g, device="cuda") * std).to(dtype)


def _weight(g, n, k, dtype=torch.float16) -> torch.Tensor:
    """A projection's [n, k] weight, as initialisation leaves it."""
    return _normal(g, n, k, std=0.02, dtype=dtype)


def _rtn(w):
    """Round-to-nearest asymmetric int4 of w [n, k] in plain torch: (q int32 [k, n], scales and
    zeros [k / GROUP, n] in w's dtype)."""
    n, k = w.shape
    f = w.t().contiguous().float().view(k // GROUP, GROUP, n)
    lo, hi = f.amin(1), f.amax(1)
    scale = ((hi - lo) / torch.full_like(hi, 15.0)).clamp_min(1e-6)  # by a tensor: a true division
    zero = torch.round(-lo / scale).clamp(0, 15)
    q = torch.round(f / scale[:, None] + zero[:, None]).clamp(0, 15)
    return q.view(k, n).to(torch.int32), scale.to(w.dtype), zero.to(w.dtype)


def _pack(q):
    """q int32 [k, n] in 0..15 -> int32 [k / 8, n], value i of a word in bits 4i .. 4i + 3."""
    q = q.view(q.shape[0] // 8, 8, q.shape[1])
    word = q[:, 0].clone()
    for i in range(1, 8):
        word |= q[:, i] << (4 * i)
    return word


def _e4m3(w):
    """Per-channel absmax e4m3 of w [n, k] in plain torch: (wq [k, n], scale [n] in w's dtype)."""
    f = w.float()
    top = f.abs().amax(1)
    scale = (top / torch.full_like(top, 448.0)).clamp_min(1e-12)  # by a tensor: a true division
    wq = (f / scale[:, None]).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return wq.t().contiguous(), scale.to(w.dtype)


def _quantized(w, fmt):
    """What a loaded checkpoint holds for w: the packed tensors of the format."""
    if fmt == "int4":
        q, s, z = _rtn(w)
        return _pack(q), s, z
    return _e4m3(w)


def _dense(w, fmt) -> torch.Tensor:
    """The float64 [n, k] weight that the quantized form of w stands for."""
    if fmt == "int4":
        q, s, z = _rtn(w)
        s, z = (t.double().repeat_interleave(GROUP, 0) for t in (s, z))
        return ((q.double() - z) * s).t()
    wq, s = _e4m3(w)
    return wq.float().double().t() * s.double()[:, None]


def _backend(fmt):
    from kernels.e2e.model import make_backend

    return make_backend("ours" if fmt == "int4" else "ours_fp8")


def _captured(body):
    """(graph, outputs) of body() on a side stream after two eager calls, as a decode loop is
    captured."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            body()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode="thread_local"):
        out = body()
    torch.cuda.synchronize()
    return graph, out


def _inv_freq() -> torch.Tensor:
    return 1.0 / (THETA ** (torch.arange(0, HEAD_DIM, 2, device="cuda", dtype=torch.float) / HEAD_DIM))


def _linear_inputs(case, seed):
    g = _gen(seed)
    n, k = case["n"], case["k"]
    w = _weight(g, n, k)
    x = _normal(g, case["rows"], k)
    b = _normal(g, n, std=0.1) if case["bias"] else None
    return w, x, b


def _mlp_inputs(case, seed):
    g = _gen(seed)
    h, i = case["hidden"], case["inter"]
    layers = [((1 + _normal(g, h, std=0.1)), _weight(g, 2 * i, h), _weight(g, h, i))
              for _ in range(case["layers"])]
    return _normal(g, 1, case["rows"], h), _normal(g, 1, case["rows"], h), layers


def _attend_inputs(case, seed):
    g = _gen(seed)
    t, start, heads, kv = (case[f] for f in ("tokens", "start", "heads", "kv"))
    max_len = -(-(start + t) // 32) * 32
    qkv = _normal(g, 1, t, (heads + 2 * kv) * HEAD_DIM)
    k = torch.zeros(kv, max_len, HEAD_DIM, device="cuda", dtype=torch.float16)
    v = torch.zeros_like(k)
    k[:, :start] = _normal(g, kv, start, HEAD_DIM)
    v[:, :start] = _normal(g, kv, start, HEAD_DIM)
    return qkv, k, v, max_len


def _model_inputs(case, seed):
    """A decoder's weights (HF names and shapes) from the seed, and the generator after them."""
    g = _gen(seed)
    h, i, heads, kv = (case[f] for f in ("hidden", "inter", "heads", "kv"))

    def lin(n, k, bias=False):
        return Bag(weight=_weight(g, n, k), bias=_normal(g, n, std=0.02) if bias else None)

    def norm():
        return Bag(weight=1 + _normal(g, h, std=0.1))

    blocks = [Bag(input_layernorm=norm(), post_attention_layernorm=norm(),
                  self_attn=Bag(q_proj=lin(heads * HEAD_DIM, h, True), k_proj=lin(kv * HEAD_DIM, h, True),
                                v_proj=lin(kv * HEAD_DIM, h, True), o_proj=lin(h, heads * HEAD_DIM)),
                  mlp=Bag(gate_proj=lin(i, h), up_proj=lin(i, h), down_proj=lin(h, i)))
              for _ in range(case["layers"])]
    embed = Bag(weight=_weight(g, VOCAB, h))
    cfg = Bag(num_attention_heads=heads, num_key_value_heads=kv, head_dim=HEAD_DIM, hidden_size=h,
              rms_norm_eps=EPS, rope_theta=THETA)
    model = Bag(config=cfg, lm_head=Bag(weight=embed.weight, bias=None),
                model=Bag(embed_tokens=embed, layers=blocks, norm=norm()))
    return model, g


def _decode_inputs(case, seed):
    """The model, the token, and the roped keys and values already in the cache."""
    model, g = _model_inputs(case, seed)
    token = torch.randint(0, VOCAB, (1, 1), device="cuda", generator=g)
    shape = (case["layers"], case["kv"], case["max_len"], HEAD_DIM)
    return model, token, _normal(g, *shape, std=0.8), _normal(g, *shape, std=0.8)


def _prompt_inputs(case, seed):
    model, g = _model_inputs(case, seed)
    return model, torch.randint(0, VOCAB, (1, case["tokens"]), device="cuda", generator=g)


def _rows_inputs(case, seed):
    g = _gen(seed)
    m, h = case["rows"], case["hidden"]
    return (_normal(g, m, h), _normal(g, m, h), 1 + _normal(g, h, std=0.1),
            _normal(g, m, 2 * case["inter"]))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        w, x, b = _linear_inputs(case, seed)
        return Bag(case=case, x=x, bias=b, packed=_quantized(w, case["fmt"]))
    if kind == "mlp":
        from kernels.e2e.model import Linear

        x, residual, layers = _mlp_inputs(case, seed)
        be = _backend(case["fmt"])

        def pack(w):
            p = _quantized(w, case["fmt"])
            return Linear(qweight=p[0], scales=p[1], zeros=p[2] if len(p) == 3 else None)

        layers = [(ln, pack(up), pack(down)) for ln, up, down in layers]

        def body():
            h, r = x, residual
            for ln, up, down in layers:
                gate_up, r = be.norm_linear(h, ln, EPS, r, up)
                h = be.act_linear(gate_up, down)
            return h, r

        graph, out = _captured(body)
        return Bag(case=case, graph=graph, out=out, keep=(x, residual, layers))
    if kind == "attend":
        from kernels.attention import k_to_tiles, vt_to_tiles

        qkv, k, v, max_len = _attend_inputs(case, seed)
        pos = torch.arange(case["start"], case["start"] + case["tokens"], device="cuda")
        return Bag(case=case, qkv=qkv, pos=pos, inv_freq=_inv_freq(), k=k_to_tiles(k).contiguous(),
                   vt=vt_to_tiles(v).contiguous())
    if kind == "decode":
        from kernels.attention import k_to_tiles, vt_to_tiles
        from kernels.e2e.model import QwenRunner

        model, token, k, v = _decode_inputs(case, seed)
        runner = QwenRunner(model, _backend(case["fmt"]), max_len=case["max_len"])
        runner.k_cache.copy_(k_to_tiles(k)[:, None])
        runner.vt_cache.copy_(vt_to_tiles(v)[:, None])
        pos = torch.tensor([case["pos"]], device="cuda")
        graph, logits = _captured(lambda: runner.forward(token, pos))
        return Bag(case=case, graph=graph, out=logits, keep=(runner, token, pos))
    if kind == "prompt":
        from kernels.e2e.model import QwenRunner

        model, ids = _prompt_inputs(case, seed)
        runner = QwenRunner(model, _backend(case["fmt"]), max_len=case["max_len"])
        return Bag(case=case, runner=runner, ids=ids, pos=torch.arange(case["tokens"], device="cuda"))
    if kind == "convert":
        w = _weight(_gen(seed), case["n"], case["k"], getattr(torch, case["dtype"]))
        return Bag(case=case, given=_quantized(w, case["fmt"]) if case["back"] else (w,))
    x, residual, weight, gate_up = _rows_inputs(case, seed)
    return Bag(case=case, x=x, residual=residual, weight=weight, gate_up=gate_up)


# --------------------------------------------------------------------------------------- the pass
def run(s):
    case, kind = s.case, s.case["kind"]
    if kind == "linear":
        from kernels.fp8 import w8a16_matmul
        from kernels.w4a16 import w4a16_matmul

        if case["fmt"] == "int4":
            return w4a16_matmul(s.x, *s.packed, bias=s.bias)
        return w8a16_matmul(s.x, *s.packed, bias=s.bias)
    if kind in ("mlp", "decode"):
        s.graph.replay()
        return s.out
    if kind == "attend":
        from kernels.attention import prefill_attention

        out = prefill_attention(s.qkv, s.pos, s.inv_freq, s.k, s.vt, case["heads"], case["kv"],
                                HEAD_DIM ** -0.5)
        return out, s.k, s.vt
    if kind == "prompt":
        logits = s.runner.forward(s.ids, s.pos)
        return logits, s.runner.k_cache, s.runner.vt_cache
    if kind == "convert":
        from kernels.fp8 import dequantize_fp8, quantize_fp8
        from kernels.quant import dequantize, quantize_rtn

        if case["fmt"] == "int4":
            return dequantize(*s.given) if case["back"] else quantize_rtn(*s.given)
        if case["back"]:
            return dequantize_fp8(*s.given)
        wq, scale = quantize_fp8(*s.given)
        return wq.view(torch.uint8), scale
    from kernels.rmsnorm import rmsnorm
    from kernels.swiglu import swiglu_fused

    return *rmsnorm(s.x, s.weight, EPS, residual=s.residual), swiglu_fused(s.gate_up)


# ------------------------------------------------------------------------------ what it has to do
def _weight_bytes(n, k, fmt) -> int:
    return n * k // 2 + 4 * (k // GROUP) * n if fmt == "int4" else n * k + 2 * n


def _layer(case) -> tuple[int, int]:
    """(weight bytes, weight elements) of one decoder layer's projections."""
    h, i, q, kv = case["hidden"], case["inter"], case["heads"] * HEAD_DIM, case["kv"] * HEAD_DIM
    shapes = [(q + 2 * kv, h), (h, q), (2 * i, h), (h, i)]
    return sum(_weight_bytes(n, k, case["fmt"]) for n, k in shapes), sum(n * k for n, k in shapes)


def work(case) -> dict:
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["rows"], case["n"], case["k"]
        return dict(bytes=_weight_bytes(n, k, case["fmt"]) + 2 * m * (k + n), flops=2 * m * n * k)
    if kind == "mlp":
        m, h, i, n = case["rows"], case["hidden"], case["inter"], case["layers"]
        per = _weight_bytes(2 * i, h, case["fmt"]) + _weight_bytes(h, i, case["fmt"]) + 2 * h
        return dict(bytes=n * per + 8 * m * h, flops=n * 6 * m * h * i)
    if kind == "attend":
        t, start, heads, kv = (case[f] for f in ("tokens", "start", "heads", "kv"))
        seen = t * start + t * (t + 1) // 2
        return dict(bytes=2 * HEAD_DIM * (t * (2 * heads + 2 * kv) + 2 * kv * (start + t)),
                    flops=4 * HEAD_DIM * heads * seen)
    if kind in ("decode", "prompt"):
        wb, we = _layer(case)
        n, h, heads, kv = case["layers"], case["hidden"], case["heads"], case["kv"]
        if kind == "decode":
            t, seen, held = 1, case["pos"] + 1, case["pos"]
        else:
            t = case["tokens"]
            seen, held = t * (t + 1) // 2, t
        return dict(bytes=n * (wb + 4 * HEAD_DIM * kv * held) + 2 * VOCAB * (h + 1) + 2 * t * h,
                    flops=n * (2 * t * we + 4 * HEAD_DIM * heads * seen) + 2 * VOCAB * h)
    if kind == "convert":
        n, k = case["n"], case["k"]
        size = 4 if case["dtype"] == "float32" else 2
        packed = n * k // 2 + 2 * size * (k // GROUP) * n if case["fmt"] == "int4" else n * k + size * n
        return dict(bytes=n * k * size + packed, flops=2 * n * k)
    m, h, i = case["rows"], case["hidden"], case["inter"]
    return dict(bytes=m * (8 * h + 6 * i) + 2 * h, flops=m * (6 * h + 8 * i))


def tolerance(case):
    return TOLERANCE[case["kind"]]


# About four times what the path differs by from `exact`, which has none of its fp16 roundings:
# measured rel / max 2.1e-4..2.8e-4 / 1.2e-3 (linear), 1.7e-3 / 6.5e-3 (mlp), 4.6e-4 / 6.7e-3
# (attend), 2.5e-3 / 1.2e-2 (decode), 2.1e-3 / 9.5e-3 (prompt), 3.7e-4 / 1.3e-3 (rows).
TOLERANCE = {
    "linear": dict(rel=1.2e-3, max=5e-3),
    "mlp": dict(rel=7e-3, max=2.6e-2),
    "attend": dict(rel=1.8e-3, max=2.7e-2),
    "decode": dict(rel=1e-2, max=5e-2),
    "prompt": dict(rel=8.5e-3, max=4e-2),
    "convert": "exact",
    "rows": dict(rel=1.5e-3, max=5e-3),
}


# ------------------------------------------------------------------------------- in 64 bits, plain
def _norm64(h, w):
    return w.double() * (h * torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS))


def _silu_mul64(gate_up):
    gate, up = gate_up.chunk(2, -1)
    return torch.nn.functional.silu(gate) * up


def _rope64(x, pos):
    """x [..., T, HEAD_DIM] at positions pos [T] (rotate_half pairs)."""
    ang = (pos[:, None].float() * _inv_freq()[None, :]).double()
    c, s = torch.cat((ang, ang), -1).cos(), torch.cat((ang, ang), -1).sin()
    half = HEAD_DIM // 2
    return x * c + torch.cat((-x[..., half:], x[..., :half]), -1) * s


def _attention64(q, k, v, pos):
    """q [heads, T, d], k and v [kv, L, d]: token t sees the positions 0 .. pos[t]."""
    group = q.shape[0] // k.shape[0]
    out = torch.empty_like(q)
    for t0 in range(0, q.shape[1], 1024):
        p = pos[t0:t0 + 1024]
        n = int(p.max()) + 1
        hidden = torch.arange(n, device=q.device)[None, :] > p[:, None]
        for h in range(q.shape[0]):
            kh, vh = k[h // group, :n], v[h // group, :n]
            a = (q[h, t0:t0 + 1024] @ kh.t()) * HEAD_DIM ** -0.5
            out[h, t0:t0 + 1024] = torch.softmax(a.masked_fill(hidden, float("-inf")), -1) @ vh
    return out


def _block64(qkv, pos, heads, kv, k_cache, v_cache):
    """qkv [T, ...] -> the attention output [T, heads * d], the caches [kv, L, d] updated at pos."""
    t = qkv.shape[0]
    q, k, v = (x.reshape(t, -1, HEAD_DIM).transpose(0, 1)
               for x in qkv.split([heads * HEAD_DIM, kv * HEAD_DIM, kv * HEAD_DIM], -1))
    k_cache[:, pos], v_cache[:, pos] = _rope64(k, pos), v
    out = _attention64(_rope64(q, pos), k_cache, v_cache, pos)
    return out.transpose(0, 1).reshape(t, heads * HEAD_DIM)


def _model64(case, model, ids, pos, k_cache, v_cache):
    fmt, heads, kv = case["fmt"], case["heads"], case["kv"]

    def lin(x, *mods):
        y = x @ _dense(torch.cat([m.weight for m in mods]), fmt).t()
        return y if mods[0].bias is None else y + torch.cat([m.bias for m in mods]).double()

    h = model.model.embed_tokens.weight[ids[0]].double()
    for i, b in enumerate(model.model.layers):
        a = b.self_attn
        qkv = lin(_norm64(h, b.input_layernorm.weight), a.q_proj, a.k_proj, a.v_proj)
        h = h + lin(_block64(qkv, pos, heads, kv, k_cache[i], v_cache[i]), a.o_proj)
        gate_up = lin(_norm64(h, b.post_attention_layernorm.weight), b.mlp.gate_proj, b.mlp.up_proj)
        h = h + lin(_silu_mul64(gate_up), b.mlp.down_proj)
    last = _norm64(h[-1:], model.model.norm.weight)
    return (last @ model.lm_head.weight.double().t())[None]


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        w, x, b = _linear_inputs(case, seed)
        y = x.double() @ _dense(w, case["fmt"]).t()
        return y if b is None else y + b.double()
    if kind == "mlp":
        x, residual, layers = _mlp_inputs(case, seed)
        h, r = x.double(), residual.double()
        for ln, up, down in layers:
            r = h + r
            h = _silu_mul64(_norm64(r, ln) @ _dense(up, case["fmt"]).t()) @ _dense(down, case["fmt"]).t()
        return h, r
    if kind == "attend":
        qkv, k, v, _ = _attend_inputs(case, seed)
        pos = torch.arange(case["start"], case["start"] + case["tokens"], device="cuda")
        out = _block64(qkv[0].double(), pos, case["heads"], case["kv"], k.double(), v.double())
        return out[None], None, None
    if kind == "decode":
        model, token, k, v = _decode_inputs(case, seed)
        return _model64(case, model, token, torch.tensor([case["pos"]], device="cuda"), k.double(), v.double())
    if kind == "prompt":
        model, ids = _prompt_inputs(case, seed)
        k = torch.zeros(case["layers"], case["kv"], case["tokens"], HEAD_DIM, device="cuda", dtype=torch.float64)
        pos = torch.arange(case["tokens"], device="cuda")
        return _model64(case, model, ids, pos, k, torch.zeros_like(k)), None, None
    if kind == "convert":
        w = _weight(_gen(seed), case["n"], case["k"], getattr(torch, case["dtype"]))
        if case["back"]:
            return _dense(w, case["fmt"])
        if case["fmt"] == "int4":
            _, s, z = _rtn(w)
            return None, s.double(), z.double()
        return None, _e4m3(w)[1].double()
    x, residual, weight, gate_up = _rows_inputs(case, seed)
    h = x.double() + residual.double()
    return _norm64(h, weight), h, _silu_mul64(gate_up.double())
