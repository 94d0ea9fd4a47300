"""The workloads this library's speed is judged on, and how each is set up and called.

Every case is one call (or, for the MLP, one short chain of calls) of registered operators
through operator_find(...)->func, the way a C program or a ctypes binding calls them: the
function pointers, the slot arrays and the params structs are made once, a pass is the
calls alone.  Tensors are torch's, on its current (null) stream.

Kinds and what they stand for:
  decode   MHA_Decode: one new token per sequence through the projections, the cache
           append, attention over the cache and the output projection.
  ragged   the decode attention core over sequences of different lengths.
  prefill  MHA_Fused: whole prompts (or encoder inputs) through attention with its
           projections; "mixed" is the operator with FP32 buffers and FP16 arithmetic.
  mlp      LayerNorm, the up projection and the down projection of a feed-forward block
           (the activation between them is not one of this library's operators).
"""

from __future__ import annotations

import ctypes
import math
from ctypes import POINTER, c_void_p

import torch

import cudaforge_amd as cf


# ------------------------------------------------------------------------- the cases ---

def listed():
    return [
        # The smallest decode step: GPT-2-small shape, FP32, one sequence half-way through
        # a 512-position cache; four short launches.
        dict(name="decode_f32_b1", kind="decode", dtype="f32", B=1, H=12, H_kv=12, d=64, T=257, cap=512, rope=False),
        # A few FP16 sequences of a GPT-2-medium-shaped model at an uneven length.
        dict(name="decode_f16_b6", kind="decode", dtype="f16", B=6, H=16, H_kv=16, d=64, T=777, cap=1024, rope=False),
        # A full serving batch of a Llama-3-8B-shaped layer, GQA and RoPE, cache of 4096.
        dict(name="decode_rope_f16_b16", kind="decode", dtype="f16", B=16, H=32, H_kv=8, d=128, T=4096, cap=4096,
             rope=True),
        # Long-context serving: four sequences of very different lengths.
        dict(name="ragged_f16_b4", kind="ragged", dtype="f16", B=4, H=32, H_kv=8, d=128, cap=32768, lens=404),
        # The smallest prefill: eight tokens through FP32 buffers.
        dict(name="prefill_mixed_b1_s8", kind="prefill", dtype="mixed", B=1, S=8, H=12, H_kv=12, d=64, causal=False,
             residual=True),
        # A batch of prompts whose length is what the tokenizer gave.
        dict(name="prefill_f16_b3_s197", kind="prefill", dtype="f16", B=3, S=197, H=12, H_kv=12, d=64, causal=True,
             residual=True),
        # An encoder batch, BERT-base.
        dict(name="prefill_f16_b8_s512", kind="prefill", dtype="f16", B=8, S=512, H=12, H_kv=12, d=64, causal=False,
             residual=True),
        # A causal batch, GPT-2-medium.
        dict(name="prefill_f16_b4_s1024", kind="prefill", dtype="f16", B=4, S=1024, H=16, H_kv=16, d=64, causal=True,
             residual=False),
        # A long prompt of a Llama-3-8B-shaped layer (GQA, head size 128); the largest work.
        dict(name="prefill_f16_b1_s2048", kind="prefill", dtype="f16", B=1, S=2048, H=32, H_kv=8, d=128, causal=True,
             residual=False),
        # The encoder batch in full FP32.
        dict(name="prefill_f32_b8_s512", kind="prefill", dtype="f32", B=8, S=512, H=12, H_kv=12, d=64, causal=False,
             residual=True),
        # The feed-forward block of that encoder batch, weights (in, out).
        dict(name="mlp_f16_n4096", kind="mlp", dtype="f16", N=4096, D=768, F=3072, tb=False),
        # The feed-forward block of a decode step, weights (out, in) as linear layers are
        # commonly exported (transpose_b).
        dict(name="mlp_f16_n16", kind="mlp", dtype="f16", N=16, D=4096, F=14336, tb=True),
    ]


# Head layouts the repository's configurations name (GPT-2 small / BERT-base, GPT-2 medium,
# Llama-3-8B) and a grouped one in between.
_HEADS = [(12, 12, 64), (16, 16, 64), (16, 4, 128), (32, 8, 128)]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "ragged", "prefill", "prefill", "prefill", "mlp", "mlp"])
    if kind == "decode":
        H, H_kv, d = rng.choice(_HEADS)
        dtype = rng.choice(["f16", "f16", "f32"])
        B = _log_int(rng, 1, 16 if dtype == "f16" else 8)
        T = _log_int(rng, 16, 4096 if d == 128 else 2048)
        return dict(kind=kind, dtype=dtype, B=B, H=H, H_kv=H_kv, d=d, T=T, cap=-(-T // 256) * 256,
                    rope=rng.random() < 0.5)
    if kind == "ragged":
        H, H_kv, d = rng.choice([(16, 16, 64), (16, 4, 128), (32, 8, 128)])
        B = _log_int(rng, 2, 32)
        cap = _log_int(rng, 512, min(32768, (131072 if H_kv * d <= 1024 else 65536) // B))
        return dict(kind=kind, dtype="f16", B=B, H=H, H_kv=H_kv, d=d, cap=cap, lens=rng.randrange(1, 1 << 30))
    if kind == "prefill":
        H, H_kv, d = rng.choice(_HEADS)
        dtype = rng.choice(["f16", "f16", "f16", "f32", "mixed"])
        # Tokens so that no draw does more than the largest listed case of its precision.
        most = {768: 8192, 1024: 6144, 2048: 3072, 4096: 2048}[H * d]
        if dtype == "f32":
            most = {768: 4096, 1024: 2560, 2048: 768, 4096: 192}[H * d]
        S = _log_int(rng, 8, min(most, 2048))
        if rng.random() < 0.4:
            S = max(8, S // 8 * 8)
        B = _log_int(rng, 1, max(1, min(16, most // S)))
        return dict(kind=kind, dtype=dtype, B=B, S=S, H=H, H_kv=H_kv, d=d, causal=rng.random() < 0.5,
                    residual=rng.random() < 0.5)
    dtype = rng.choice(["f16", "f16", "f16", "f32"])
    D, F = rng.choice([(768, 3072), (1024, 4096), (4096, 14336)])
    N = _log_int(rng, 1, (8192 if D <= 1024 else 512) // (1 if dtype == "f16" else 4))
    return dict(kind="mlp", dtype=dtype, N=N, D=D, F=F, tb=rng.random() < 0.5)


# ---------------------------------------------------------------------- inputs, state ---

def _torch_dtype(case):
    return torch.float16 if case["dtype"] == "f16" else torch.float32


def _lengths(case):
    """The attended lengths of a ragged case: uniform in [cap / 32, cap], the case's own."""
    g = torch.Generator().manual_seed(case["lens"])
    return [int(x) for x in torch.randint(max(1, case["cap"] // 32), case["cap"] + 1, (case["B"],), generator=g)]


def _inputs(case, seed):
    """The case's input tensors by name: activations and caches N(0, 1), weights and biases
    N(0, 0.02), LayerNorm gain about 1, in the order given and from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = _torch_dtype(case)

    def mk(*shape, std=1.0, mean=0.0):
        t = torch.randn(shape, dtype=dt, device="cuda", generator=g)
        return t if std == 1.0 and mean == 0.0 else t.mul_(std).add_(mean)

    if case["kind"] == "mlp":
        N, D, F = case["N"], case["D"], case["F"]
        up, down = ((F, D), (D, F)) if case["tb"] else ((D, F), (F, D))
        return dict(x=mk(N, D), gamma=mk(D, std=0.1, mean=1.0), beta=mk(D, std=0.02), w1=mk(*up, std=0.02),
                    b1=mk(F, std=0.02), w2=mk(*down, std=0.02), b2=mk(D, std=0.02))
    B, H, H_kv, d = case["B"], case["H"], case["H_kv"], case["d"]
    D, kvd = H * d, H_kv * d
    if case["kind"] == "ragged":
        return dict(q=mk(B, H, d), k=mk(B, case["cap"], H_kv, d), v=mk(B, case["cap"], H_kv, d))
    t = dict(x=mk(B, case.get("S", 1), D))
    if case["kind"] == "decode":
        t.update(k=mk(B, case["cap"], H_kv, d), v=mk(B, case["cap"], H_kv, d))
    elif case["residual"]:
        t.update(r=mk(B, case["S"], D))
    for n, w in (("q", D), ("k", kvd), ("v", kvd), ("o", D)):
        t["w" + n] = mk(D, w, std=0.02)
        t["b" + n] = mk(w, std=0.02)
    return t


_ready = []


def _call(name, inputs, outputs, params):
    """One operator call, ready to make: (function, inputs, outputs, params, stream)."""
    if not _ready:
        cf.init_gpu(0)
        _ready.append(True)
    ins = (c_void_p * len(inputs))(*[None if t is None else t.data_ptr() for t in inputs])
    outs = (c_void_p * len(outputs))(*[t.data_ptr() for t in outputs])
    return (cf.find_op(name).func, ctypes.cast(ins, POINTER(c_void_p)), ctypes.cast(outs, POINTER(c_void_p)),
            ctypes.cast(ctypes.pointer(params), c_void_p), None)


def prepare(case, seed):
    t = _inputs(case, seed)
    dt = _torch_dtype(case)
    e = "f16" if case["dtype"] == "f16" else "f32"
    if case["kind"] == "mlp":
        N, D, F = case["N"], case["D"], case["F"]
        h, u, y = (torch.empty((N, w), dtype=dt, device="cuda") for w in (D, F, D))
        mm = "matmul_%s_cuda" % e
        calls = [_call("layernorm_%s_cuda" % e, [t["x"], t["gamma"], t["beta"]], [h], cf.LayerNormParams(N, D, 1e-5)),
                 _call(mm, [h, t["w1"], t["b1"]], [u], cf.MatmulParams(N, F, D, False, case["tb"], 1, 0, 0, 0, 0)),
                 _call(mm, [u, t["w2"], t["b2"]], [y], cf.MatmulParams(N, D, F, False, case["tb"], 1, 0, 0, 0, 0))]
        return dict(t, calls=calls, out=dict(h=h, u=u, y=y))
    B, H, H_kv, d = case["B"], case["H"], case["H_kv"], case["d"]
    D, scale = H * d, 1.0 / math.sqrt(d)
    if case["kind"] == "ragged":
        lens = torch.tensor([n - 1 for n in _lengths(case)], dtype=torch.int32, device="cuda")
        o = torch.empty((B, H, d), dtype=dt, device="cuda")
        p = cf.MhaDecodeParams(B, D, H, H_kv, d, scale, -1, case["cap"])
        return dict(t, lens=lens, calls=[_call("mha_decode_attn_%s_cuda" % e, [t["q"], t["k"], t["v"], lens], [o], p)],
                    out=dict(o=o))
    y = torch.empty_like(t["x"])
    weights = [t[k] for k in ("wq", "bq", "wk", "bk", "wv", "bv", "wo", "bo")]
    if case["kind"] == "decode":
        p = cf.MhaDecodeParams(B, D, H, H_kv, d, scale, case["T"] - 1, case["cap"])
        name = "mha_decode_%s_cuda" % e
        if case["rope"]:
            p, name = cf.MhaDecodeRopeParams(p, 10000.0, 0), "mha_decode_rope_%s_cuda" % e
        # The caches are updated in place, as in a decode loop.
        return dict(t, calls=[_call(name, [t["x"], t["k"], t["v"]] + weights, [y, t["k"], t["v"]], p)],
                    out=dict(y=y, k=t["k"], v=t["v"]))
    p = cf.MhaFusedParams(B, case["S"], D, H, H_kv, d, scale, case["residual"], case["causal"])
    name = {"f16": "mha_fused_f16io_cuda", "f32": "mha_fused_f32_cuda", "mixed": "mha_fused_f16_cuda"}[case["dtype"]]
    return dict(t, calls=[_call(name, [t["x"], t.get("r")] + weights, [y], p)], out=dict(y=y))


def run(state):
    for func, ins, outs, params, stream in state["calls"]:
        rc = func(ins, outs, params, stream)
        if rc != 0:
            raise RuntimeError("operator returned %d" % rc)
    return state["out"]


# --------------------------------------------------------------- what a pass has to do ---

def work(case):
    es = 2 if case["dtype"] == "f16" else 4
    if case["kind"] == "mlp":
        N, D, F = case["N"], case["D"], case["F"]
        return dict(bytes=es * (2 * D * F + 3 * D + F + 3 * N * D + N * F), flops=4 * N * D * F)
    B, H, H_kv, d = case["B"], case["H"], case["H_kv"], case["d"]
    D, kvd = H * d, H_kv * d
    if case["kind"] == "ragged":
        n = sum(_lengths(case))
        return dict(bytes=es * (2 * n * kvd + 2 * B * D) + 4 * B, flops=4 * n * D)
    weights = 2 * D * D + 2 * D * kvd + 2 * D + 2 * kvd
    if case["kind"] == "decode":
        return dict(bytes=es * (2 * B * case["T"] * kvd + weights + 2 * B * D),
                    flops=2 * B * (2 * D * D + 2 * D * kvd) + 4 * B * case["T"] * D)
    S = case["S"]
    pairs = S * (S + 1) // 2 if case["causal"] else S * S
    return dict(bytes=es * (weights + (3 if case["residual"] else 2) * B * S * D),
                flops=2 * B * S * (2 * D * D + 2 * D * kvd) + 4 * B * pairs * D)


def tolerance(case):
    """About four times what a correct implementation at the same precision is off by.  With
    FP16 storage that is the rounding of intermediates and results (measured 2.1e-4 to
    5.5e-4 against 64 bits), with FP32 the order of the sums over K of 768 to 14336
    (measured 1.6e-7 on the smallest, growing with K)."""
    return dict(rel=3e-6) if case["dtype"] == "f32" else dict(rel=2e-3)


# ------------------------------------------------------------------ the same in 64 bits ---

def _rotate(x, pos, base=10000.0):
    d = x.shape[-1]
    i = torch.arange(d // 2, dtype=torch.float64, device=x.device)
    a = pos / base ** (2.0 * i / d)
    c, s = torch.cos(a), torch.sin(a)
    y = torch.empty_like(x)
    y[..., 0::2] = x[..., 0::2] * c - x[..., 1::2] * s
    y[..., 1::2] = x[..., 0::2] * s + x[..., 1::2] * c
    return y


def _attend(q, k, v, scale, causal):
    """softmax(q k^T scale) v: q (H, n, d), k and v (H_kv, T, d), query head h of group h / (H / H_kv)."""
    g = q.shape[0] // k.shape[0]
    out = torch.empty_like(q)
    for h in range(q.shape[0]):
        s = torch.mm(q[h], k[h // g].t().contiguous()) * scale
        if causal:
            s = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), -math.inf)
        out[h] = torch.mm(torch.softmax(s, -1), v[h // g])
    return out


def exact(case, seed):
    t = {k: v.double() for k, v in _inputs(case, seed).items()}
    if case["kind"] == "mlp":
        h = torch.nn.functional.layer_norm(t["x"], (case["D"],), t["gamma"], t["beta"], 1e-5)
        w1, w2 = (t["w1"].t(), t["w2"].t()) if case["tb"] else (t["w1"], t["w2"])
        u = h @ w1 + t["b1"]
        return dict(h=h, u=u, y=u @ w2 + t["b2"])
    B, H, H_kv, d = case["B"], case["H"], case["H_kv"], case["d"]
    scale = 1.0 / math.sqrt(d)
    if case["kind"] == "ragged":
        o = torch.empty_like(t["q"])
        for b, n in enumerate(_lengths(case)):
            k, v = (t[x][b, :n].transpose(0, 1).contiguous() for x in "kv")
            o[b] = _attend(t["q"][b].unsqueeze(1), k, v, scale, False)[:, 0]
        return dict(o=o)
    n = case.get("S", 1)
    q, k, v = ((t["x"] @ t["w" + c] + t["b" + c]).view(B, n, -1, d) for c in "qkv")
    if case["kind"] == "decode":
        T = case["T"]
        if case["rope"]:
            q, k = _rotate(q, T - 1), _rotate(k, T - 1)
        t["k"][:, T - 1], t["v"][:, T - 1] = k[:, 0], v[:, 0]
        k, v = t["k"][:, :T], t["v"][:, :T]
    o = torch.empty_like(q)
    for b in range(B):
        hq, hk, hv = (x[b].transpose(0, 1).contiguous() for x in (q, k, v))
        o[b] = _attend(hq, hk, hv, scale, case.get("causal", False)).transpose(0, 1)
    y = o.reshape(B, n, H * d) @ t["wo"] + t["bo"]
    if "r" in t:
        y = y + t["r"]
    return dict(y=y, k=t["k"], v=t["v"]) if case["kind"] == "decode" else dict(y=y)
