"""The workloads that this library's performance is judged by, one pass of
each through the public entry points.

`listed()` holds the fixed cases, `draw(rng)` more of the same ranges;
`prepare` makes a case's inputs (and the layer object a program keeps) on the
GPU from a seed, `run` is one pass over them, `work` the bytes and operations
a pass cannot do without, `tolerance` how far another correct implementation
may be off, and `exact` the same result in 64 bits from plain torch.

The families:

  decode   one decode step over a paged cache: the fresh token appended and
           attended (attention_decode_paged_append);
  contig   decode attention over a contiguous cache (attention_decode);
  prefill  attention over a fresh sequence (attention_prefill);
  gemm     W8A8 GEMM with per-channel scales (qgemm_perchannel);
  norm     RMSNorm -> int8 quantize -> W8A8 GEMM (rmsnorm_qgemm);
  mlp      a prompt's W8A8 MLP block: rmsnorm_quant with the residual, gate/up
           GEMM + SwiGLU + quantize, down GEMM;
  layer    one whole W8A8 decode layer (DecodeLayer.forward);
  sample   the step after the LM head (decode_step_batched).
"""

import math
import random

import numpy as np
import torch

import fusedtok_amd as ft

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
BYTES = {"f32": 4, "bf16": 2, "f16": 2}
DEV = "cuda"
EPS, THETA = 1e-5, 500000.0

# (hidden, q heads, kv heads, head dim, mlp width) of the decode layers drawn
LAYERS = ((4096, 32, 8, 128, 14336), (2048, 32, 8, 64, 8192), (1024, 16, 4, 64, 2816))


def listed():
    return [
        # The smallest call: a small model's step at a handful of short
        # conversations, where latency and launches are all there is.
        dict(name="decode_small", kind="decode", dtype="bf16", b=4, hq=32, hkv=8, d=64, page=16,
             lo=128, hi=1024, lens_seed=3),
        # The serving step: 32 conversations of very different length.
        dict(name="decode_ragged", kind="decode", dtype="bf16", b=32, hq=32, hkv=8, d=128, page=16,
             lo=512, hi=32768, lens_seed=2026),
        # Float32 caches (the entry points' default type for numpy callers):
        # one long conversation.
        dict(name="contig_f32", kind="contig", dtype="f32", b=1, hq=32, hkv=8, d=128, t=16384),
        # A 4096-token prompt.
        dict(name="prefill_bf16", kind="prefill", dtype="bf16", b=1, hq=32, hkv=8, d=128, s=4096,
             causal=True),
        # The same in float32, a prompt of no round length.
        dict(name="prefill_f32", kind="prefill", dtype="f32", b=1, hq=32, hkv=8, d=128, s=1500,
             causal=True),
        # A prompt-sized projection of a large model.
        dict(name="gemm_large", kind="gemm", m=4096, n=28672, k=8192, out="bf16"),
        # A projection for more rows than a decode batch and fewer than a
        # prompt: a large batch, a short prompt, a few speculated tokens a row.
        dict(name="gemm_mid", kind="gemm", m=150, n=14336, k=4096, out="bf16"),
        # The decode-sized norm + projection, eight conversations.
        dict(name="norm_gemm", kind="norm", m=8, n=11008, k=4096, dtype="f16"),
        # The MLP block over a 1000-token prompt.
        dict(name="mlp_prompt", kind="mlp", m=1000, hidden=4096, inter=14336, dtype="bf16"),
        # A whole layer of a serving batch: 64 conversations at 8192 tokens.
        dict(name="layer_batch64", kind="layer", dtype="bf16", shape=0, b=64, lo=8192, hi=8192,
             lens_seed=4),
        # A whole layer of a small model at a small batch, short contexts.
        dict(name="layer_small", kind="layer", dtype="bf16", shape=1, b=6, lo=100, hi=2000,
             lens_seed=5),
        # Sampling: 64 rows of a 128k vocabulary, 64 past ids a row.
        dict(name="sample_batch64", kind="sample", rows=64, vocab=128256, ids=64, penalty=1.2,
             p=0.9, temperature=0.8),
    ]


def _log(rng, lo, hi):
    """An int in [lo, hi], uniform in its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "contig", "prefill", "prefill", "gemm", "gemm", "norm",
                       "mlp", "layer", "layer", "sample"])
    if kind in ("decode", "contig"):
        hkv = rng.choice([1, 2, 4, 8, 16])
        c = dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "f16", "f32"]), hkv=hkv,
                 hq=hkv * rng.choice([1, 2, 4, 8]), d=rng.choice([64, 128, 128]))
        # about 2 GB of K and V at most
        room = int(2e9 / (2 * hkv * c["d"] * BYTES[c["dtype"]]))
        c["b"] = _log(rng, 1, 64)
        top = max(64, min(32768, room // c["b"]))
        if kind == "contig":
            return dict(c, t=_log(rng, 64, top))
        hi = _log(rng, 64, top)
        return dict(c, page=rng.choice([16, 16, 32, 64]), hi=hi, lo=rng.randint(1, hi),
                    lens_seed=rng.randrange(1 << 20))
    if kind == "prefill":
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        hkv = rng.choice([2, 4, 8])
        c = dict(kind=kind, dtype=dtype, hkv=hkv, hq=hkv * rng.choice([1, 2, 4]),
                 d=rng.choice([64, 128]), causal=rng.random() < 0.75)
        c["s"] = _log(rng, 16, 1500 if dtype == "f32" else 4096)
        c["b"] = rng.randint(1, max(1, min(8, (1500 if dtype == "f32" else 4096) // c["s"])))
        return c
    if kind == "gemm":
        return dict(kind=kind, m=_log(rng, 1, 4096), n=8 * _log(rng, 128, 3584),
                    k=64 * _log(rng, 8, 128), out=rng.choice(["bf16", "f16", "f32"]))
    if kind == "norm":
        return dict(kind=kind, m=_log(rng, 1, 64), n=8 * _log(rng, 128, 3584),
                    k=64 * _log(rng, 8, 64), dtype=rng.choice(["bf16", "f16"]))
    if kind == "mlp":
        hidden, _, _, _, inter = rng.choice(LAYERS)
        return dict(kind=kind, m=_log(rng, 65, 2048), hidden=hidden, inter=inter,
                    dtype=rng.choice(["bf16", "f16"]))
    if kind == "layer":
        b = _log(rng, 1, 64)
        hi = _log(rng, 64, 8192)
        return dict(kind=kind, dtype=rng.choice(["bf16", "f16"]), shape=rng.randrange(3), b=b,
                    hi=hi, lo=rng.randint(1, hi), lens_seed=rng.randrange(1 << 20))
    return dict(kind=kind, rows=_log(rng, 1, 64), vocab=_log(rng, 32000, 152000),
                ids=rng.randint(1, 256), penalty=rng.choice([1.0, 1.1, 1.2]),
                p=rng.choice([0.5, 0.9, 0.95]), temperature=rng.choice([0.7, 0.8, 1.0]))


def _lens(c):
    r = random.Random(c["lens_seed"])
    return [r.randint(c["lo"], c["hi"]) for _ in range(c["b"])]


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(gen, shape, dtype):
    return torch.randn(shape, generator=gen, device=DEV, dtype=dtype)


def _codes(gen, rows, cols):
    return torch.randint(-127, 128, (rows, cols), generator=gen, device=DEV, dtype=torch.int8)


def _scales(gen, n, k=None):
    """Per-channel weight scales; for K inputs, such that inputs of unit
    variance give outputs of about that (a model's activations), else in
    [1e-3, 1e-2]."""
    r = torch.rand(n, generator=gen, device=DEV)
    return r * 9e-3 + 1e-3 if k is None else (r + 0.5) / (73.0 * math.sqrt(k))


def _norm_weight(gen, n):
    return torch.rand(n, generator=gen, device=DEV) + 0.5


def _paged(c, gen, hkv, d, page, dtype):
    """Pools of twice the pages in use, permuted tables and the lengths."""
    lens = _lens(c)
    pages = [(n + 1 + page - 1) // page for n in lens]
    pool = 2 * sum(pages)
    perm = torch.randperm(pool, generator=gen, device=DEV).to(torch.int32)
    table = torch.zeros((c["b"], max(pages)), dtype=torch.int32, device=DEV)
    at = 0
    for i, n in enumerate(pages):
        table[i, :n] = perm[at:at + n]
        at += n
    return dict(k_pool=_randn(gen, (pool, hkv, page, d), dtype),
                v_pool=_randn(gen, (pool, hkv, page, d), dtype), table=table,
                lens=torch.tensor(lens, dtype=torch.int32, device=DEV))


def _layer_dims(c):
    return LAYERS[c["shape"]]


def _weights(c, gen):
    hidden, hq, hkv, d, inter = _layer_dims(c)
    nqkv = (hq + 2 * hkv) * d
    return dict(norm1=_norm_weight(gen, hidden), norm2=_norm_weight(gen, hidden),
                w_qkv=_codes(gen, nqkv, hidden), s_qkv=_scales(gen, nqkv, hidden),
                w_o=_codes(gen, hidden, hq * d), s_o=_scales(gen, hidden, hq * d),
                w_gu=_codes(gen, 2 * inter, hidden), s_gu=_scales(gen, 2 * inter, hidden),
                w_down=_codes(gen, hidden, inter), s_down=_scales(gen, hidden, inter))


def _inputs(c, seed):
    gen, kind = _gen(seed), c["kind"]
    dt = DTYPES.get(c.get("dtype"))
    if kind == "decode":
        s = _paged(c, gen, c["hkv"], c["d"], c["page"], dt)
        return dict(s, q=_randn(gen, (c["b"], c["hq"], c["d"]), dt),
                    k_new=_randn(gen, (c["b"], c["hkv"], c["d"]), dt),
                    v_new=_randn(gen, (c["b"], c["hkv"], c["d"]), dt))
    if kind == "contig":
        cache = (c["b"], c["hkv"], c["t"], c["d"])
        return dict(q=_randn(gen, (c["b"], c["hq"], c["d"]), dt), k=_randn(gen, cache, dt),
                    v=_randn(gen, cache, dt))
    if kind == "prefill":
        rows = (c["b"], c["hkv"], c["s"], c["d"])
        return dict(q=_randn(gen, (c["b"], c["hq"], c["s"], c["d"]), dt),
                    k=_randn(gen, rows, dt), v=_randn(gen, rows, dt))
    if kind == "gemm":
        return dict(a=_codes(gen, c["m"], c["k"]), sa=0.0123, w=_codes(gen, c["n"], c["k"]),
                    sw=_scales(gen, c["n"]))
    if kind == "norm":
        return dict(x=_randn(gen, (c["m"], c["k"]), dt), norm=_norm_weight(gen, c["k"]),
                    w=_codes(gen, c["n"], c["k"]), sw=_scales(gen, c["n"]))
    if kind == "mlp":
        m, hidden, inter = c["m"], c["hidden"], c["inter"]
        return dict(x=_randn(gen, (m, hidden), dt), res=_randn(gen, (m, hidden), dt),
                    norm=_norm_weight(gen, hidden), w_gu=_codes(gen, 2 * inter, hidden),
                    s_gu=_scales(gen, 2 * inter, hidden), w_down=_codes(gen, hidden, inter),
                    s_down=_scales(gen, hidden, inter))
    if kind == "layer":
        hidden, _, hkv, d, _ = _layer_dims(c)
        s = _paged(c, gen, hkv, d, 16, dt)
        return dict(s, w=_weights(c, gen), x=_randn(gen, (c["b"], hidden), dt))
    rng = np.random.default_rng(seed)
    return dict(logits=2.0 * _randn(gen, (c["rows"], c["vocab"]), torch.float32),
                ids=rng.integers(0, c["vocab"], (c["rows"], c["ids"])),
                seeds=rng.integers(0, 1 << 40, c["rows"]))


def prepare(case, seed):
    s = dict(_inputs(case, seed), case=case)
    if case["kind"] == "layer":
        _, hq, hkv, _, _ = _layer_dims(case)
        s["layer"] = ft.DecodeLayer(q_heads=hq, kv_heads=hkv, page=16, max_batch=case["b"],
                                    dtype=DTYPES[case["dtype"]], eps=EPS, theta=THETA, neox=True,
                                    **s["w"])
    return s


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "decode":
        out = ft.attention_decode_paged_append(s["q"], s["k_pool"], s["v_pool"], s["table"],
                                               s["k_new"], s["v_new"], s["lens"])
        return dict(out=out, k_pool=s["k_pool"], v_pool=s["v_pool"])
    if kind == "contig":
        return ft.attention_decode(s["q"], s["k"], s["v"])
    if kind == "prefill":
        return ft.attention_prefill(s["q"], s["k"], s["v"], c["causal"])
    if kind == "gemm":
        return ft.qgemm_perchannel(s["a"], s["sa"], s["w"], s["sw"], out_dtype=DTYPES[c["out"]])
    if kind == "norm":
        y, q, scale = ft.rmsnorm_qgemm(s["x"], s["norm"], s["w"], s["sw"], eps=EPS,
                                       out_dtype=DTYPES[c["dtype"]])
        return dict(y=y, q=q, scale=scale)
    if kind == "mlp":
        dt = DTYPES[c["dtype"]]
        q1, s1 = ft.rmsnorm_quant(s["x"], s["norm"], residual=s["res"], eps=EPS, device_scale=True)
        h, q2, s2 = ft.qgemm_swiglu_quant(q1, s1, s["w_gu"], s["s_gu"], out_dtype=dt,
                                          device_scale=True)
        y = ft.qgemm_perchannel(q2, s2, s["w_down"], s["s_down"], out_dtype=dt)
        return dict(q1=q1, s1=s1, h=h, q2=q2, s2=s2, y=y)
    if kind == "layer":
        y = s["layer"].forward(s["x"], s["k_pool"], s["v_pool"], s["table"], s["lens"])
        return dict(y=y, k_pool=s["k_pool"], v_pool=s["v_pool"])
    return ft.decode_step_batched(s["logits"], s["ids"], c["penalty"], p=c["p"],
                                  temperature=c["temperature"], seeds=s["seeds"], device_out=True)


def _attn_work(c, tokens, hq, hkv, d, size):
    """K and V of `tokens` cache rows read, q read, the output written."""
    return (2 * tokens * hkv * d * size + 2 * c["b"] * hq * d * size, 4 * tokens * hq * d)


def work(case):
    c, kind = case, case["kind"]
    e = BYTES.get(c.get("dtype"), 2)
    if kind == "decode":
        lens = _lens(c)
        nb, fl = _attn_work(c, sum(lens) + c["b"], c["hq"], c["hkv"], c["d"], e)
        # the fresh rows are written too; one table entry a page
        nb += 2 * c["b"] * c["hkv"] * c["d"] * e + 4 * sum(n // c["page"] + 1 for n in lens)
        return dict(bytes=nb, flops=fl)
    if kind == "contig":
        nb, fl = _attn_work(c, c["b"] * c["t"], c["hq"], c["hkv"], c["d"], e)
        return dict(bytes=nb, flops=fl)
    if kind == "prefill":
        b, hq, hkv, s, d = c["b"], c["hq"], c["hkv"], c["s"], c["d"]
        pairs = s * (s + 1) // 2 if c["causal"] else s * s
        return dict(bytes=2 * b * (hq + hkv) * s * d * e, flops=4 * b * hq * pairs * d)
    if kind == "gemm":
        m, n, k = c["m"], c["n"], c["k"]
        return dict(bytes=m * k + n * k + 4 * n + m * n * BYTES[c["out"]], flops=2 * m * n * k)
    if kind == "norm":
        m, n, k = c["m"], c["n"], c["k"]
        return dict(bytes=n * k + 4 * n + 4 * k + m * k * (e + 1) + m * n * e, flops=2 * m * n * k)
    if kind == "mlp":
        m, hidden, inter = c["m"], c["hidden"], c["inter"]
        nb = (3 * inter * hidden + 4 * (2 * inter + 2 * hidden) + m * hidden * (3 * e + 1)
              + m * inter * (2 * e + 1))
        return dict(bytes=nb, flops=6 * m * inter * hidden)
    if kind == "layer":
        hidden, hq, hkv, d, inter = _layer_dims(c)
        wn = (hq + 2 * hkv) * d * hidden + hq * d * hidden + 3 * inter * hidden
        nb, fl = _attn_work(c, sum(_lens(c)) + c["b"], hq, hkv, d, e)
        nb += wn + 2 * c["b"] * hidden * e
        return dict(bytes=nb, flops=fl + 2 * c["b"] * wn)
    return dict(bytes=4 * c["rows"] * c["vocab"], flops=4 * c["rows"] * c["vocab"])


def tolerance(case):
    kind = case["kind"]
    if kind in ("gemm", "sample"):
        return "exact"  # whole-number sums and one rounding; tokens
    if kind in ("decode", "contig", "prefill"):
        # float32: another order of the sums (4e-7 off the 64-bit result);
        # 16 bits: the output's rounding (1.7e-3 off for bf16)
        return dict(rel=dict(f32=3e-6, bf16=6e-3, f16=8e-4)[case["dtype"]])
    # int8 codes move by one where a sum's last bit decides, and 16-bit
    # activations are rounded from sums that differ by that (a layer whose
    # attention sums in another order: 3.2e-3 off)
    return dict(rel=1.2e-2, differ=2e-3)


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _attend(q, k, v):
    """q [Hq, D] over k, v [Hkv, T, D], float64."""
    hkv, d = k.shape[0], k.shape[2]
    qg = q.double().reshape(hkv, -1, d)
    out = [torch.softmax(qg[h] @ k[h].double().t() / math.sqrt(d), -1) @ v[h].double()
           for h in range(hkv)]
    return torch.cat(out)


def _rows_of(pool, table_row, n):
    """The first n cache rows [Hkv, n, D] behind one row of the table."""
    page = pool.shape[2]
    blk = pool[table_row[: (n + page - 1) // page].long()]
    return blk.transpose(0, 1).reshape(pool.shape[1], -1, pool.shape[3])[:, :n]


def _paged_attention(s, q, k_new, v_new):
    """Each sequence's attention over its cached rows and the fresh one."""
    out = []
    for i, n in enumerate(s["lens"].tolist()):
        k = torch.cat([_rows_of(s["k_pool"], s["table"][i], n).double(), k_new[i][:, None]], 1)
        v = torch.cat([_rows_of(s["v_pool"], s["table"][i], n).double(), v_new[i][:, None]], 1)
        out.append(_attend(q[i], k, v))
    return torch.stack(out)


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _quant(x):
    scale = x.abs().max() / 127
    return torch.clamp(torch.round(x / scale), -127, 127), scale


def _linear(q, scale, w, sw):
    return (q @ w.double().t()) * (scale * sw.double())


def _swiglu(h, inter):
    g, u = h[:, :inter], h[:, inter:]
    return g / (1 + torch.exp(-g)) * u


def _rope(x, pos, d):
    """x [B, heads, D] turned to positions pos [B], halves (j, j + D/2)."""
    j = torch.arange(d // 2, device=DEV, dtype=torch.float64)
    ang = pos.double()[:, None] * THETA ** (-2 * j / d)
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    a, b = x[..., : d // 2], x[..., d // 2:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "sample":
        return None
    s = _inputs(case, seed)
    if kind == "decode":
        out = _paged_attention(s, s["q"], s["k_new"].double(), s["v_new"].double())
        return dict(out=out, k_pool=None, v_pool=None)
    if kind == "contig":
        return torch.stack([_attend(s["q"][i], s["k"][i], s["v"][i]) for i in range(c["b"])])
    if kind == "prefill":
        g = c["hq"] // c["hkv"]
        out = torch.empty(s["q"].shape, dtype=torch.float64, device=DEV)
        for i in range(c["b"]):
            for h in range(c["hq"]):
                sc = s["q"][i, h].double() @ s["k"][i, h // g].double().t() / math.sqrt(c["d"])
                if c["causal"]:
                    sc.masked_fill_(torch.ones_like(sc, dtype=torch.bool).triu(1), -math.inf)
                out[i, h] = torch.softmax(sc, -1) @ s["v"][i, h // g].double()
        return out
    if kind == "gemm":
        return _linear(s["a"].double(), s["sa"], s["w"], s["sw"])
    if kind == "norm":
        q, scale = _quant(_norm(s["x"].double(), s["norm"]))
        return dict(y=_linear(q, scale, s["w"], s["sw"]), q=None, scale=scale.reshape(1))
    if kind == "mlp":
        q1, s1 = _quant(_norm(s["x"].double() + s["res"].double(), s["norm"]))
        h = _linear(q1, s1, s["w_gu"], s["s_gu"])
        q2, s2 = _quant(_swiglu(h, c["inter"]))
        return dict(q1=None, s1=s1.reshape(1), h=h, q2=None, s2=s2.reshape(1),
                    y=_linear(q2, s2, s["w_down"], s["s_down"]))
    _, hq, hkv, d, inter = _layer_dims(c)
    w, x, b = s["w"], s["x"].double(), c["b"]
    qkv = _linear(*_quant(_norm(x, w["norm1"])), w["w_qkv"], w["s_qkv"]).reshape(b, -1, d)
    q = _rope(qkv[:, :hq], s["lens"], d)
    k = _rope(qkv[:, hq:hq + hkv], s["lens"], d)
    att = _paged_attention(s, q, k, qkv[:, hq + hkv:]).reshape(b, hq * d)
    r = x + _linear(*_quant(att), w["w_o"], w["s_o"])
    h = _linear(*_quant(_norm(r, w["norm2"])), w["w_gu"], w["s_gu"])
    y = r + _linear(*_quant(_swiglu(h, inter)), w["w_down"], w["s_down"])
    return dict(y=y, k_pool=None, v_pool=None)
