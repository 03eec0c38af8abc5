"""The work that a program built on this package has it do, as cases that can
be timed and compared: linear layers from one token to long prompts, batched
products, attention over prompts and over KV caches, the sampling tail, an MLP
block, and two whole calls of the decoder.

Sizes are those of the benchmark's workloads (a 64 x 768 x 3072 fp32 product, a
4096 x 11008 decode projection, 4096^3, 4096-token attention, the Llama-style 1B
decoder: width 2048, 32 query and 8 KV heads of 64, MLP width 5632, 32000
tokens) and generic ones between and around them: batches and prompts have any
length, so rows and keys are odd as often as even."""
import math

import torch

import kuillm_amd  # noqa: F401  (registers the package's operators)
from kuillm_amd import ops
from kuillm_amd.decoder import LlamaDecoder, LlamaShape

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
ITEM = {"bf16": 2, "f16": 2, "f32": 4}
LLAMA = dict(vocab=32000, d=2048, ffn=5632, layers=16, hq=32, hkv=8)
CAPACITY = 640          # the decoder's KV cache: a 512-token prompt and 128 tokens
TOP_P = 0.9
# the largest listed case: 512 tokens through the decoder
MOST_FLOPS = 8.5e11
MOST_BYTES = 1.7e9


def listed():
    return [
        # an fp32 layer of a small model (MLP up projection, 64 tokens): the smallest call
        dict(name="linear_f32_64", kind="linear", m=64, k=768, n=3072, dtype="f32", layout="kn", bias=True),
        # a decode projection for a batch of 16, the weight stored [in, out]
        dict(name="linear_decode_16", kind="linear", m=16, k=4096, n=11008, dtype="bf16", layout="kn", bias=False),
        # a layer with a bias over a short prompt of a narrow model, an nn.Linear weight
        dict(name="linear_prompt_203", kind="linear", m=203, k=896, n=4864, dtype="bf16", layout="nk", bias=True),
        # a wide layer over a long prompt
        dict(name="linear_4096", kind="linear", m=4096, k=4096, n=4096, dtype="bf16", layout="kn", bias=True),
        # the MLP half of a decoder layer over a 500-token prompt: norm, gate|up, SwiGLU, down
        dict(name="mlp_500", kind="mlp", m=500, d=2048, ffn=5632, dtype="bf16"),
        # eager attention's second product, probabilities times values, for a ragged prompt
        dict(name="bmm_probs_777", kind="bmm", b=32, m=777, k=777, n=128, dtype="bf16", layout="kn"),
        # attention over a long prompt
        dict(name="attn_prompt_4096", kind="attn", batch=1, hq=32, hkv=32, s=4096, hd=128, dtype="bf16", mask="causal"),
        # attention over a left-padded batch of prompts, with the additive mask that a batch needs
        dict(name="attn_padded_4x600", kind="attn", batch=4, hq=32, hkv=8, s=600, hd=64, dtype="bf16", mask="padded"),
        # one new token for each of 16 sequences with long caches of their own lengths
        dict(name="attn_cache_16x4000", kind="cache", batch=16, hq=32, hkv=8, s=4000, hd=128, dtype="bf16"),
        # the sampling tail for a batch of 8: top-p filter, softmax, draw
        dict(name="sample_8", kind="sample", m=8, vocab=32000),
        # a whole prompt through the decoder
        dict(name="decoder_prompt_512", kind="prompt", batch=1, t=512, dtype="bf16"),
        # one decode step of the whole decoder for a batch of 8, its graph replayed
        dict(name="decoder_step_8", kind="step", batch=8, t=512, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer width: mostly multiples of 64, some of 8."""
    step = rng.choice((64, 64, 64, 8))
    return max(step, _log(rng, lo, hi) // step * step)


def draw(rng):
    while True:
        kind = rng.choice(("linear", "linear", "linear", "mlp", "bmm", "attn", "attn", "cache", "sample", "prompt", "step"))
        dtype = rng.choice(("bf16", "bf16", "bf16", "f16"))
        if kind == "linear":
            dtype = rng.choice(("bf16", "bf16", "bf16", "f16", "f32"))
            case = dict(kind=kind, m=_log(rng, 1, 8192), k=_width(rng, 512, 8192), n=_width(rng, 512, 16384),
                        dtype=dtype, layout=rng.choice(("nk", "nk", "kn")), bias=rng.random() < 0.5)
        elif kind == "mlp":
            d = _width(rng, 512, 4096)
            case = dict(kind=kind, m=_log(rng, 65, 4096), d=d, ffn=_width(rng, 2 * d, 4 * d), dtype=dtype)
        elif kind == "bmm":
            # scores (head dim inside, keys out) or probabilities times values (keys inside)
            b, m, s, hd = rng.choice((8, 16, 32, 64)), _log(rng, 16, 2048), _log(rng, 16, 2048), rng.choice((64, 128))
            case = (dict(kind=kind, b=b, m=m, k=hd, n=s, dtype=dtype, layout="nk") if rng.random() < 0.5 else
                    dict(kind=kind, b=b, m=m, k=s, n=hd, dtype=dtype, layout="kn"))
        elif kind == "attn":
            hq = rng.choice((8, 14, 16, 32, 40))
            batch = rng.choice((1, 1, 2, 4, 8))
            case = dict(kind=kind, batch=batch, hq=hq, hkv=rng.choice([h for h in (2, 8, hq) if hq % h == 0]),
                        s=_log(rng, 17, 4096), hd=rng.choice((64, 128)), dtype=dtype,
                        mask=rng.choice(("causal", "causal", "full", "padded")) if batch > 1 else rng.choice(("causal", "full")))
        elif kind == "cache":
            # a serving batch: at least 512 query rows
            hq = rng.choice((8, 14, 16, 32, 40))
            case = dict(kind=kind, batch=_log(rng, -(-512 // hq), 96), hq=hq, hkv=rng.choice([h for h in (2, 8, hq) if hq % h == 0]),
                        s=_log(rng, 100, 16384), hd=rng.choice((64, 128)), dtype=dtype)
        elif kind == "sample":
            case = dict(kind=kind, m=_log(rng, 1, 64), vocab=rng.choice((32000, rng.randrange(8000, 32769))))
        elif kind == "prompt":
            batch = rng.choice((1, 1, 2, 4))
            case = dict(kind=kind, batch=batch, t=_log(rng, 17, 512 // batch), dtype="bf16")
        else:
            case = dict(kind=kind, batch=rng.choice((1, 2, 4, 8, 16, 32, 64)), t=_log(rng, 17, 512), dtype="bf16")
        w = work(case)
        # fp32 products have no 16-bit matrix rate to use
        flops = w["flops"] * (8 if case.get("dtype") == "f32" else 1)
        if flops <= MOST_FLOPS and w["bytes"] <= MOST_BYTES:
            return case


# ------------------------------------------------------------------ inputs

def _randn(g, shape, dtype, std=1.0):
    return (torch.randn(shape, device=DEV, generator=g) * std).to(dtype)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _llama_state(g, dtype):
    c = LLAMA
    d, hd = c["d"], c["d"] // c["hq"]
    st = {"model.embed_tokens.weight": _randn(g, (c["vocab"], d), dtype),
          "lm_head.weight": _randn(g, (c["vocab"], d), dtype, 0.02),
          "model.norm.weight": (1 + 0.1 * torch.randn(d, device=DEV, generator=g)).to(dtype)}
    for i in range(c["layers"]):
        p = f"model.layers.{i}."
        st[p + "self_attn.q_proj.weight"] = _randn(g, (d, d), dtype, 0.02)
        st[p + "self_attn.k_proj.weight"] = _randn(g, (c["hkv"] * hd, d), dtype, 0.02)
        st[p + "self_attn.v_proj.weight"] = _randn(g, (c["hkv"] * hd, d), dtype, 0.02)
        st[p + "self_attn.o_proj.weight"] = _randn(g, (d, d), dtype, 0.02)
        st[p + "mlp.gate_proj.weight"] = _randn(g, (c["ffn"], d), dtype, 0.02)
        st[p + "mlp.up_proj.weight"] = _randn(g, (c["ffn"], d), dtype, 0.02)
        st[p + "mlp.down_proj.weight"] = _randn(g, (d, c["ffn"]), dtype, 0.02)
        st[p + "input_layernorm.weight"] = (1 + 0.1 * torch.randn(d, device=DEV, generator=g)).to(dtype)
        st[p + "post_attention_layernorm.weight"] = (1 + 0.1 * torch.randn(d, device=DEV, generator=g)).to(dtype)
    return st


def _padding_mask(batch, s, lengths, dtype):
    """Additive causal mask of a left-padded batch, [batch, 1, s, s]: -inf on
    later keys and on padding; a padding query attends everywhere, as no row
    may be empty."""
    key = torch.arange(s, device=DEV)
    visible = (key[None, :] <= key[:, None])[None] & (key[None, None, :] >= (s - lengths)[:, None, None])
    visible |= ~visible.any(-1, keepdim=True)
    return torch.zeros(batch, 1, s, s, device=DEV).masked_fill(~visible[:, None], -math.inf).to(dtype)


def _lengths(g, batch, s):
    return torch.randint(max(1, s // 2), s + 1, (batch,), device=DEV, generator=g)


def _inputs(case, seed):
    """The tensors of a case, without any of this package's objects."""
    g, kind = _gen(seed), case["kind"]
    dt = DTYPES[case.get("dtype", "f32")]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        W = _randn(g, (n, k) if case["layout"] == "nk" else (k, n), dt, 0.02)
        return dict(x=_randn(g, (m, k), dt), W=W, bias=_randn(g, (n,), dt, 0.02) if case["bias"] else None)
    if kind == "mlp":
        m, d, f = case["m"], case["d"], case["ffn"]
        return dict(x=_randn(g, (m, d), dt), res=_randn(g, (m, d), dt),
                    norm=(1 + 0.1 * torch.randn(d, device=DEV, generator=g)).to(dt),
                    wgu=_randn(g, (2 * f, d), dt, 0.02), wd=_randn(g, (d, f), dt, 0.02))
    if kind == "bmm":
        b, m, k, n = case["b"], case["m"], case["k"], case["n"]
        if case["layout"] == "nk":
            return dict(A=_randn(g, (b, m, k), dt), B=_randn(g, (b, n, k), dt))
        A = torch.softmax(2 * torch.randn(b, m, k, device=DEV, generator=g), -1).to(dt)
        return dict(A=A, B=_randn(g, (b, k, n), dt))
    if kind == "attn":
        n, s, hd = case["batch"], case["s"], case["hd"]
        # projections' layout [batch, tokens, heads, head dim]
        q, k, v = (_randn(g, (n, s, h, hd), dt) for h in (case["hq"], case["hkv"], case["hkv"]))
        bias = _padding_mask(n, s, _lengths(g, n, s), dt) if case["mask"] == "padded" else None
        return dict(q=q, k=k, v=v, bias=bias)
    if kind == "cache":
        n, s, hd = case["batch"], case["s"], case["hd"]
        return dict(q=_randn(g, (n, case["hq"], 1, hd), dt), k=_randn(g, (n, case["hkv"], s, hd), dt),
                    v=_randn(g, (n, case["hkv"], s, hd), dt), len=_cache_lengths(case, seed))
    if kind == "sample":
        # logits with a few likely tokens, as a trained head gives
        return dict(scores=4 * torch.randn(case["m"], case["vocab"], device=DEV, generator=g),
                    u=torch.rand(case["m"], 1, device=DEV, generator=g))
    if kind in ("prompt", "step"):
        n = case["batch"]
        return dict(state=_llama_state(g, dt),
                    prompt=torch.randint(0, LLAMA["vocab"], (n, case["t"]), device=DEV, generator=g),
                    tok=torch.randint(0, LLAMA["vocab"], (n,), device=DEV, generator=g))
    raise ValueError(kind)


def _cache_lengths(case, seed):
    """Keys of each sequence: the longest fills the cache."""
    if case["batch"] == 1:
        return torch.tensor([case["s"]], dtype=torch.int32, device=DEV)
    lens = _lengths(_gen(seed + 1), case["batch"], case["s"])
    lens[0] = case["s"]
    return lens.to(torch.int32)


def prepare(case, seed):
    i, kind = _inputs(case, seed), case["kind"]
    i["case"] = case
    if kind == "bmm" and case["layout"] == "nk":
        i["B"] = i["B"].transpose(1, 2)         # keys as q k^T takes them
    elif kind == "attn":
        for name in "qkv":
            i[name] = i[name].transpose(1, 2)
    elif kind in ("prompt", "step"):
        # the prompt fills the cache; a step is for the token after it
        cap = CAPACITY
        dec = LlamaDecoder(LlamaShape(**LLAMA), i.pop("state"), capacity=cap, batch=case["batch"], device=DEV)
        i["dec"] = dec
        if kind == "step":
            t = case["t"]
            dec.prefill(i["prompt"])
            i["at"] = torch.tensor([[t] * case["batch"], [t + 1] * case["batch"]], dtype=torch.int32, device=DEV)
            dec.capture()
    return i


# -------------------------------------------------------------------- runs

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        x, W, bias = state["x"], state["W"], state["bias"]
        if case["layout"] == "nk":
            return ops.linear(x, W, bias)
        return ops.mm(x, W) if bias is None else ops.addmm(bias, x, W)
    if kind == "mlp":
        res = torch.empty_like(state["x"])
        h = ops.rmsnorm(state["x"], state["norm"], 1e-5, residual=state["res"], res_out=res)
        return ops.linear(ops.silu_mul(ops.linear(h, state["wgu"])), state["wd"]), res
    if kind == "bmm":
        return ops.bmm(state["A"], state["B"])
    if kind == "attn":
        return ops.sdpa(state["q"], state["k"], state["v"], is_causal=case["mask"] == "causal", bias=state["bias"])
    if kind == "cache":
        return ops.sdpa_decode(state["q"], state["k"], state["v"], kv_len=state["len"], return_lse=True)
    if kind == "sample":
        probs = ops.softmax(ops.top_p_filter(state["scores"], TOP_P))
        return probs, ops.multinomial(probs, 1, uniforms=state["u"], check=False)
    dec = state["dec"]
    if kind == "prompt":
        logits, _ = dec.prefill(state["prompt"])
        return logits, dec.kcache, dec.vcache
    # a program that picks its own tokens: the token in, one step, its logits out
    dec.tok.copy_(state["tok"])
    dec.step_state.copy_(state["at"])
    dec.graph.replay()
    return dec.graph_logits, dec.kcache, dec.vcache


# -------------------------------------------------------------------- work

def work(case):
    kind = case["kind"]
    e = ITEM[case.get("dtype", "f32")]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": e * (m * k + k * n + m * n + (n if case["bias"] else 0)), "flops": 2 * m * k * n}
    if kind == "mlp":
        m, d, f = case["m"], case["d"], case["ffn"]
        return {"bytes": e * (3 * d * f + 4 * m * d + d), "flops": 6 * m * d * f}
    if kind == "bmm":
        b, m, k, n = case["b"], case["m"], case["k"], case["n"]
        return {"bytes": e * b * (m * k + k * n + m * n), "flops": 2 * b * m * k * n}
    if kind == "attn":
        n, hq, hkv, s, hd = (case[x] for x in ("batch", "hq", "hkv", "s", "hd"))
        bias = e * n * s * s if case["mask"] == "padded" else 0
        return {"bytes": 2 * e * n * s * hd * (hq + hkv) + 4 * n * hq * s + bias,
                "flops": 4 * n * hq * s * s * hd * (0.5 if case["mask"] != "full" else 1)}
    if kind == "cache":
        n, hq, hkv, s, hd = (case[x] for x in ("batch", "hq", "hkv", "s", "hd"))
        keys = s if n == 1 else 0.75 * n * s    # lengths are spread over s / 2 .. s
        return {"bytes": 2 * e * keys * hkv * hd + 2 * e * n * hq * hd, "flops": 4 * keys * hq * hd}
    if kind == "sample":
        return {"bytes": 8 * case["m"] * case["vocab"], "flops": 0}
    c = LLAMA
    d, f, hd = c["d"], c["ffn"], c["d"] // c["hq"]
    layer = d * (c["hq"] + 2 * c["hkv"]) * hd + d * d + 3 * d * f
    n, t = case["batch"], case["t"]
    kv = 2 * c["layers"] * c["hkv"] * hd * 2    # bytes of K and V per token
    weights = 2 * (c["layers"] * layer + c["vocab"] * d)
    if kind == "prompt":
        flops = 2 * n * t * c["layers"] * layer + 2 * n * c["vocab"] * d + c["layers"] * 2 * n * c["hq"] * t * t * hd
        return {"bytes": weights + n * t * (kv + 2 * d) + 2 * n * c["vocab"], "flops": flops}
    return {"bytes": weights + n * (t + 1) * kv + 2 * n * (c["vocab"] + d),
            "flops": 2 * n * (c["layers"] * layer + c["vocab"] * d)}


def tolerance(case):
    kind = case["kind"]
    if case.get("dtype") == "f32":
        return {"rel": 1e-5}                    # fp32 products, summed in another order
    if kind == "sample":
        return {"rel": 1e-5}                    # fp32 probabilities; the draws are the same
    if kind in ("linear", "bmm"):
        return {"rel": 4e-3}                    # one rounding of an fp32 sum to 16 bits
    if kind in ("attn", "cache"):
        return {"rel": 8e-3}                    # probabilities and the result rounded to 16 bits
    if kind == "mlp":
        return {"rel": 1.5e-2}                  # four roundings to 16 bits, 6e-3 from the 64-bit result
    return {"rel": 3e-2}                        # 16 layers of such roundings, 2e-2 from the 64-bit result


# ------------------------------------------------------------------- exact

def _norm64(x, w, eps=1e-5):
    return w.double() * (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps))


def _attention64(q, k, v, scale, bias=None, causal_from=None):
    """One sequence: q [hq, l, hd], k / v [hkv, s, hd], head by head; query i
    sees keys j <= causal_from + i."""
    rep, outs, lses = q.shape[0] // k.shape[0], [], []
    for h in range(q.shape[0]):
        z = q[h].double() @ k[h // rep].double().t().contiguous() * scale
        if bias is not None:
            z = z + bias.double()
        if causal_from is not None:
            l, s = z.shape
            z = z.masked_fill(torch.arange(s, device=DEV)[None] > causal_from + torch.arange(l, device=DEV)[:, None],
                              -math.inf)
        lses.append(torch.logsumexp(z, -1))
        outs.append(torch.softmax(z, -1) @ v[h // rep].double())
    return torch.stack(outs), torch.stack(lses)


def _rotate64(x, pos, theta=10000.0):
    """Split-half rotary embedding of x [heads, t, hd] at positions pos [t]."""
    hd = x.shape[-1]
    inv = 1.0 / theta ** (torch.arange(0, hd, 2, device=DEV, dtype=torch.float64) / hd)
    a = pos.double()[:, None] * inv
    c, s = torch.cat([a.cos()] * 2, -1), torch.cat([a.sin()] * 2, -1)
    return x * c + torch.cat([-x[..., hd // 2:], x[..., :hd // 2]], -1) * s


def _decoder64(state, tokens, cap):
    """(logits after the last token, K, V [layers, n, hkv, cap, hd]) in 64 bits."""
    c = LLAMA
    hd = c["d"] // c["hq"]
    n, t = tokens.shape
    kc = torch.zeros(c["layers"], n, c["hkv"], cap, hd, dtype=torch.float64, device=DEV)
    vc = torch.zeros_like(kc)
    h = state["model.embed_tokens.weight"][tokens].double()
    pos = torch.arange(t, device=DEV)

    def lin(x, name):
        return x @ state[name].double().t().contiguous()

    def heads(x, k):
        return x.view(n, t, k, hd).transpose(1, 2)

    for i in range(c["layers"]):
        p = f"model.layers.{i}."
        x = _norm64(h, state[p + "input_layernorm.weight"])
        q = _rotate64(heads(lin(x, p + "self_attn.q_proj.weight"), c["hq"]), pos)
        k = _rotate64(heads(lin(x, p + "self_attn.k_proj.weight"), c["hkv"]), pos)
        v = heads(lin(x, p + "self_attn.v_proj.weight"), c["hkv"])
        kc[i, :, :, :t], vc[i, :, :, :t] = k, v
        o = torch.stack([_attention64(q[b], k[b], v[b], hd ** -0.5, causal_from=0)[0] for b in range(n)])
        h = h + lin(o.transpose(1, 2).reshape(n, t, -1), p + "self_attn.o_proj.weight")
        x = _norm64(h, state[p + "post_attention_layernorm.weight"])
        x = torch.nn.functional.silu(lin(x, p + "mlp.gate_proj.weight")) * lin(x, p + "mlp.up_proj.weight")
        h = h + lin(x, p + "mlp.down_proj.weight")
    return lin(_norm64(h[:, -1], state["model.norm.weight"]), "lm_head.weight"), kc, vc


def exact(case, seed):
    i, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        W = i["W"].t().contiguous() if case["layout"] == "nk" else i["W"]
        y = i["x"].double() @ W.double()
        return y if i["bias"] is None else y + i["bias"].double()
    if kind == "mlp":
        f = case["ffn"]
        res = i["x"].double() + i["res"].double()
        z = _norm64(res, i["norm"]) @ i["wgu"].double().t().contiguous()
        return (torch.nn.functional.silu(z[:, :f]) * z[:, f:]) @ i["wd"].double().t().contiguous(), res
    if kind == "bmm":
        B = i["B"].transpose(1, 2).contiguous() if case["layout"] == "nk" else i["B"]
        return torch.stack([a.double() @ b.double() for a, b in zip(i["A"], B)])
    if kind == "attn":
        got = []
        for b in range(case["batch"]):
            bias = None if i["bias"] is None else i["bias"][b, 0]
            got.append(_attention64(i["q"][b].transpose(0, 1), i["k"][b].transpose(0, 1), i["v"][b].transpose(0, 1),
                                    case["hd"] ** -0.5, bias, 0 if case["mask"] == "causal" else None))
        return torch.stack([o for o, _ in got]), torch.stack([x for _, x in got])
    if kind == "cache":
        got = []
        for b, s in enumerate(i["len"].tolist()):
            got.append(_attention64(i["q"][b], i["k"][b, :, :s], i["v"][b, :, :s], case["hd"] ** -0.5))
        return torch.stack([o for o, _ in got]), torch.stack([x for _, x in got])
    if kind == "sample":
        x = i["scores"].double()
        z, at = x.sort(-1)
        drop = torch.softmax(z, -1).cumsum(-1) <= 1 - TOP_P
        drop[:, -1] = False
        kept = x.masked_fill(torch.zeros_like(drop).scatter(1, at, drop), -math.inf)
        return torch.softmax(kept, -1), None
    tokens = i["prompt"] if kind == "prompt" else torch.cat([i["prompt"], i["tok"][:, None]], 1)
    if tokens.numel() > 8 * 513:
        return None
    return _decoder64(i["state"], tokens, CAPACITY)
