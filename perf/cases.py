"""The work a user of this package has it do, as cases that can be timed and checked.

Kinds of case, each through a public entry point:

  linear    an `LRSLinear` forward: y = x·Bᵀ·Aᵀ + x·Sᵀ + b
  nm        the same with a 2:4 S
  group     an `LRSLinearGroup` forward: linears that read the same x (q,k,v or gate,up)
  chain     a `PreparedChain` step: a layer's projections q,k,v | o | gate,up | down
  op        torch.ops.ssalaad.tilelang_bsr_addmm_inplace_dense_ on a given `out`
  step      a `DecodeEngine` step of a small model: one new token per sequence
  compress  the compression loop's block projection and the encoding of its result

Weights, structures and inputs are drawn from the seed on the GPU, with the
distributions of the package's own benchmark: x ~ N(0, 1), factors and blocks
~ N(0, 0.02), blocks placed uniformly or with Zipf(1.2) row counts.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "s-salaad_amd"))

import ssalaad_amd  # noqa: E402
from ssalaad_amd.bundle import build_model_from_config  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SCALE = 0.02


# ------------------------------------------------------------------ cases --
def listed():
    return [
        # the smallest projection: 512 wide, fp32, one short sequence
        dict(name="linear_512_fp32_256t", kind="linear", dtype="fp32", tokens=256, n=512, m=512,
             r=128, p=32, q=32, density=0.5, zipf=False, bias=True),
        # a 60M model's gate projection over a batch of 8 sequences of 256 (fp32)
        dict(name="linear_60m_gate_fp32_2048t", kind="linear", dtype="fp32", tokens=2048, n=1376,
             m=512, r=128, p=32, q=32, density=0.5, zipf=False, bias=False),
        # serving one sequence: a 7B feed-forward projection on one token
        dict(name="linear_7b_ffn_1t", kind="linear", dtype="bf16", tokens=1, n=11008, m=4096,
             r=256, p=64, q=64, density=0.5, zipf=False, bias=False),
        # a short prompt (or a batch of verification tokens) through a 7B down projection
        dict(name="linear_7b_down_256t", kind="linear", dtype="bf16", tokens=256, n=4096, m=11008,
             r=256, p=64, q=64, density=0.3, zipf=False, bias=False),
        # prefill of a long prompt through a 7B feed-forward projection
        dict(name="linear_7b_ffn_2048t", kind="linear", dtype="bf16", tokens=2048, n=11008,
             m=4096, r=256, p=64, q=64, density=0.5, zipf=False, bias=False),
        # prefill with a skewed structure of small blocks
        dict(name="linear_zipf16_2048t", kind="linear", dtype="bf16", tokens=2048, n=4096,
             m=11008, r=128, p=16, q=16, density=0.5, zipf=True, bias=False),
        # prefill of a ragged prompt through a 2:4 projection
        dict(name="nm_4096_1000t", kind="nm", dtype="fp16", tokens=1000, n=4096, m=4096, r=256,
             bias=True),
        # prefill through a 1B layer's gate and up (5461 features, not a multiple of the block)
        dict(name="group_1b_gate_up_2048t", kind="group", dtype="bf16", tokens=2048, m=2048,
             n=5461, n2=5461, n3=0, r=256, p=32, density=0.5),
        # batched decode: a 1B layer's seven projections for 16 sequences
        dict(name="chain_1b_layer_16t", kind="chain", dtype="bf16", tokens=16, hidden=2048,
             ffn=5461, r=256, p=32, density=0.5),
        # the in-place op at a ragged token count
        dict(name="op_2048_5461_300t", kind="op", dtype="bf16", tokens=300, n=2048, m=5472, p=32,
             q=32, density=0.5, zipf=False),
        # batched serving: a whole decode step (attention over about 1000 cached tokens, norms,
        # projections, LM head) of a model with 1B-wide layers, cut to four of them
        dict(name="step_1b_4layers_16seq", kind="step", dtype="bf16", tokens=16, hidden=2048,
             ffn=5461, heads=16, kv_heads=16, layers=4, vocab=32000, context=1024, r=256, p=32,
             density=0.5),
        # one round of the compression loop on a 7B matrix
        dict(name="compress_7b_ffn_64", kind="compress", dtype="fp32", n=11008, m=4096, p=64,
             q=64, density=0.5),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi, p):
    """A feature count: mostly a multiple of the block, sometimes any number."""
    v = _log_int(rng, lo, hi)
    return max(p, v if rng.random() < 0.25 else v // p * p)


def _tokens(rng):
    """Decode batches, short prompts and long ones."""
    return rng.choice([1, 16, 256, 2048, _log_int(rng, 1, 64), _log_int(rng, 65, 600),
                       _log_int(rng, 256, 2048)])


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        # at most the largest listed case's work, and its time: fp32 runs at a
        # sixteenth of the 16-bit rate and small blocks at about a third
        slow = (16.0 if c["dtype"] == "fp32" and c["kind"] != "compress" else
                3.0 if c.get("p", 64) < 32 and c["kind"] != "compress" else 1.5)
        if w["flops"] * slow <= 1.5e11 and w["bytes"] <= 7e8:
            return c


def _draw(rng):
    kind = rng.choice(["linear"] * 6 + ["group", "group", "nm", "chain", "op", "step", "compress"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
    p = rng.choice([16, 32, 32, 64, 64])
    q = p if rng.random() < 0.9 else rng.choice([16, 32, 64])
    density = round(rng.uniform(0.1, 0.9), 2)
    if kind == "linear":
        hi = 2048 if dtype == "fp32" else 11008
        return dict(kind=kind, dtype=dtype, tokens=_tokens(rng), n=_width(rng, 512, hi, p),
                    m=_width(rng, 512, hi, q), r=rng.choice([64, 100, 128, 256, 256]), p=p, q=q,
                    density=density, zipf=rng.random() < 0.3, bias=rng.random() < 0.5)
    if kind == "nm":
        return dict(kind=kind, dtype=rng.choice(["bf16", "fp16"]), tokens=_tokens(rng),
                    n=_width(rng, 1024, 11008, 32), m=_log_int(rng, 1024, 8192) // 4 * 4,
                    r=rng.choice([64, 128, 256]), bias=rng.random() < 0.5)
    if kind == "group":
        n = _width(rng, 1024, 11008, p)
        three = rng.random() < 0.5
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "fp16"]), tokens=_tokens(rng),
                    m=_width(rng, 1024, 4096, p), n=n, n2=_width(rng, 512, 4096, p) if three else n,
                    n3=_width(rng, 512, 4096, p) if three else 0, r=rng.choice([64, 128, 256]),
                    p=p, density=density)
    if kind == "chain":
        hidden = rng.choice([1024, 2048, 2560, 4096])
        return dict(kind=kind, dtype=rng.choice(["bf16", "fp16"]), tokens=_log_int(rng, 1, 64),
                    hidden=hidden, ffn=_width(rng, 2 * hidden, 3 * hidden, p),
                    r=rng.choice([64, 128, 256]), p=p, density=density)
    if kind == "op":
        hi = 2048 if dtype == "fp32" else 11008
        return dict(kind=kind, dtype=dtype, tokens=_tokens(rng),
                    n=max(p, _log_int(rng, 512, hi) // p * p),
                    m=max(q, _log_int(rng, 512, hi) // q * q), p=p, q=q, density=density,
                    zipf=rng.random() < 0.3)
    if kind == "step":
        hd = rng.choice([64, 128])
        heads = rng.choice([8, 16, 24, 32]) if hd == 64 else rng.choice([8, 16])
        return dict(kind=kind, dtype=rng.choice(["bf16", "fp16"]), tokens=_log_int(rng, 1, 16),
                    hidden=heads * hd, ffn=_width(rng, 2 * heads * hd, 3 * heads * hd, 32),
                    heads=heads, kv_heads=rng.choice([heads, heads // 4]), layers=rng.randint(2, 4),
                    vocab=_log_int(rng, 8000, 32000), context=_log_int(rng, 128, 1500),
                    r=rng.choice([64, 128, 256]), p=rng.choice([16, 32, 64]), density=density)
    return dict(kind=kind, dtype=rng.choice(["fp32", "bf16"]),
                n=max(p, _log_int(rng, 512, 11008) // p * p),
                m=max(q, _log_int(rng, 512, 8192) // q * q), p=p, q=q, density=density)


# ----------------------------------------------------------------- inputs --
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(gen, *shape, dtype=torch.float32, scale=1.0):
    return (torch.randn(*shape, generator=gen, device="cuda") * scale).to(dtype)


def _counts_zipf(NB, NBK, density, gen):
    """Blocks per block-row ∝ rank^-1.2 over a random order of the rows, at most
    NBK each, density·NB·NBK in all."""
    target = int(round(density * NB * NBK))
    w = torch.arange(1, NB + 1, dtype=torch.float64) ** -1.2
    w = w[torch.randperm(NB, generator=gen, device="cuda").cpu()]
    lo, hi = 0.0, float(NBK) / float(w.min())
    for _ in range(60):  # the scale at which the capped rows hold the target
        mid = (lo + hi) / 2
        lo, hi = (mid, hi) if float((w * mid).clamp(max=NBK).sum()) < target else (lo, mid)
    c = (w * hi).clamp(max=NBK).floor().long()
    free = (c < NBK).nonzero().flatten()
    c[free[: max(0, target - int(c.sum()))]] += 1
    return c


def _blocks(gen, n, m, p, q, density, zipf, dtype):
    """(crow, col, values (nnz, p, q)) over ⌈n/p⌉ × ⌈m/q⌉ blocks, zero past n and m."""
    NB, NBK = -(-n // p), -(-m // q)
    if zipf:
        counts = _counts_zipf(NB, NBK, density, gen).cuda()
        order = torch.rand(NB, NBK, generator=gen, device="cuda").argsort(1).argsort(1)
        keep = order < counts[:, None]
    else:
        k = int(round(density * NB * NBK))
        keep = torch.zeros(NB * NBK, dtype=torch.bool, device="cuda")
        keep[torch.randperm(NB * NBK, generator=gen, device="cuda")[:k]] = True
        keep = keep.view(NB, NBK)
    rows, cols = keep.nonzero(as_tuple=True)
    crow = torch.zeros(NB + 1, dtype=torch.int64, device="cuda")
    crow[1:] = keep.sum(1).cumsum(0)
    vals = _randn(gen, rows.numel(), p, q, dtype=dtype, scale=SCALE)
    if n % p:
        vals[rows == NB - 1, n - (NB - 1) * p:, :] = 0
    if m % q:
        vals[cols == NBK - 1, :, m - (NBK - 1) * q:] = 0
    return crow, cols, vals


def _parts(gen, n, m, r, p, q, density, zipf, bias, dtype):
    return dict(n=n, m=m, p=p, q=q, A=_randn(gen, n, r, dtype=dtype, scale=SCALE),
                B=_randn(gen, r, m, dtype=dtype, scale=SCALE),
                S=_blocks(gen, n, m, p, q, density, zipf, dtype),
                bias=_randn(gen, n, dtype=dtype, scale=SCALE) if bias else None)


def _module(w):
    crow, col, vals = w["S"]
    S = torch.sparse_bsr_tensor(crow, col, vals, size=((crow.numel() - 1) * w["p"],
                                                       -(-w["m"] // w["q"]) * w["q"]),
                                check_invariants=False)
    return ssalaad_amd.LRSLinear(w["A"], w["B"], S, in_features=w["m"], out_features=w["n"],
                                 bias=w["bias"], block_p=w["p"], block_q=w["q"])


def _dense(w):
    """S of the parts, as float64 [n, m]."""
    crow, col, vals = w["S"]
    NB, NBK = crow.numel() - 1, -(-w["m"] // w["q"])
    S = torch.zeros(NB, NBK, w["p"], w["q"], dtype=torch.float64, device="cuda")
    rows = torch.repeat_interleave(torch.arange(NB, device="cuda"), crow[1:] - crow[:-1])
    S[rows, col] = vals.double()
    return S.permute(0, 2, 1, 3).reshape(NB * w["p"], NBK * w["q"])[: w["n"], : w["m"]]


def _linear64(x, w):
    y = (x @ w["B"].double().T) @ w["A"].double().T + x @ (_dense(w) if "S" in w else w["D"].double()).T
    return y if w["bias"] is None else y + w["bias"].double()


def _layer_shapes(c, q_rows, kv_rows):
    h, f = c["hidden"], c["ffn"]
    return [(q_rows, h), (kv_rows, h), (kv_rows, h), (h, q_rows), (f, h), (f, h), (h, f)]


def _inputs(c, seed):
    """Everything of the case that the seed draws, as plain tensors."""
    g, dt, kind = _gen(seed), DTYPES[c["dtype"]], c["kind"]
    if kind == "linear":
        w = _parts(g, c["n"], c["m"], c["r"], c["p"], c["q"], c["density"], c["zipf"], c["bias"], dt)
        return dict(x=_randn(g, c["tokens"], c["m"], dtype=dt), w=[w])
    if kind == "group":
        ns = [v for v in (c["n"], c["n2"], c["n3"]) if v]
        return dict(x=_randn(g, c["tokens"], c["m"], dtype=dt),
                    w=[_parts(g, n, c["m"], c["r"], c["p"], c["p"], c["density"], False, False, dt)
                       for n in ns])
    if kind == "nm":
        n, m = c["n"], c["m"]
        D = _randn(g, n, m // 4, 4, scale=SCALE)
        top = D.abs().topk(2, dim=-1).indices
        D = torch.zeros_like(D).scatter(-1, top, D.gather(-1, top)).view(n, m).to(dt)
        w = dict(n=n, m=m, A=_randn(g, n, c["r"], dtype=dt, scale=SCALE),
                 B=_randn(g, c["r"], m, dtype=dt, scale=SCALE), D=D,
                 bias=_randn(g, n, dtype=dt, scale=SCALE) if c["bias"] else None)
        return dict(x=_randn(g, c["tokens"], m, dtype=dt), w=[w])
    if kind == "chain":
        return dict(x=_randn(g, c["tokens"], c["hidden"], dtype=dt),
                    w=[_parts(g, n, m, c["r"], c["p"], c["p"], c["density"], False, False, dt)
                       for n, m in _layer_shapes(c, c["hidden"], c["hidden"])])
    if kind == "op":
        crow, col, vals = _blocks(g, c["n"], c["m"], c["p"], c["q"], c["density"], c["zipf"], dt)
        return dict(x=_randn(g, c["tokens"], c["m"], dtype=dt), S=(crow, col, vals),
                    out=_randn(g, c["tokens"], c["n"], dtype=dt))
    if kind == "step":
        hd = c["hidden"] // c["heads"]
        ctx, L, B = c["context"], c["layers"], c["tokens"]
        kv = (L, B, c["kv_heads"], ctx, hd)
        return dict(layers=[[_parts(g, n, m, c["r"], c["p"], c["p"], c["density"], False, False, dt)
                             for n, m in _layer_shapes(c, c["hidden"], c["kv_heads"] * hd)]
                            for _ in range(L)],
                    norms=[1 + _randn(g, c["hidden"], scale=0.1).to(dt) for _ in range(2 * L + 1)],
                    embed=_randn(g, c["vocab"], c["hidden"], dtype=dt),
                    head=_randn(g, c["vocab"], c["hidden"], dtype=dt, scale=SCALE),
                    k=_randn(g, *kv, dtype=dt), v=_randn(g, *kv, dtype=dt),
                    tokens=torch.randint(0, c["vocab"], (B,), generator=g, device="cuda"),
                    positions=torch.randint(ctx * 15 // 16, ctx, (B,), generator=g,
                                            device="cuda").cpu().tolist())
    # block norms of a weight matrix differ from block to block
    n, m, p, q = c["n"], c["m"], c["p"], c["q"]
    s = _randn(g, n // p, 1, m // q, 1, scale=0.5).exp() * SCALE
    return dict(R=(_randn(g, n // p, p, m // q, q) * s).view(n, m).to(dt),
                keep=int(round(c["density"] * (n // p) * (m // q))))


_PROJ = ("q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj")


def _engine(c, inp):
    dt = DTYPES[c["dtype"]]
    cfg = {"model_type": "llama", "hidden_size": c["hidden"], "intermediate_size": c["ffn"],
           "num_hidden_layers": c["layers"], "num_attention_heads": c["heads"],
           "num_key_value_heads": c["kv_heads"], "head_dim": c["hidden"] // c["heads"],
           "vocab_size": c["vocab"], "max_position_embeddings": c["context"],
           "rms_norm_eps": 1e-5, "rope_theta": 500000.0, "hidden_act": "silu",
           "tie_word_embeddings": False}
    with torch.device("meta"):
        model = build_model_from_config(cfg, attn_implementation="sdpa")
    for layer, ws in zip(model.model.layers, inp["layers"]):
        for i, name in enumerate(_PROJ):
            setattr(layer.self_attn if i < 4 else layer.mlp, name, _module(ws[i]))
    model = model._apply(lambda t: torch.empty_like(t, device="cuda") if t.is_meta else t).to(dt)
    model.model.rotary_emb = type(model.model.rotary_emb)(config=model.config, device="cuda")
    with torch.no_grad():
        model.model.embed_tokens.weight.copy_(inp["embed"])
        model.lm_head.weight.copy_(inp["head"])
        norms = [n for l in model.model.layers for n in (l.input_layernorm, l.post_attention_layernorm)]
        for mod, w in zip(norms + [model.model.norm], inp["norms"]):
            mod.weight.copy_(w)
    eng = ssalaad_amd.DecodeEngine(model.eval(), max_batch=c["tokens"], max_context=c["context"])
    eng.k_cache.copy_(inp["k"])
    eng.v_cache.copy_(inp["v"])
    return eng


def prepare(case, seed):
    inp, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        return dict(kind=kind, mod=_module(inp["w"][0]), x=inp["x"])
    if kind == "nm":
        w = inp["w"][0]
        mod = ssalaad_amd.LRSLinear(w["A"], w["B"], w["D"], in_features=w["m"], out_features=w["n"],
                                    bias=w["bias"], nm_n=2, nm_m=4)
        return dict(kind=kind, mod=mod, x=inp["x"])
    if kind == "group":
        return dict(kind=kind, mod=ssalaad_amd.LRSLinearGroup(*map(_module, inp["w"])), x=inp["x"])
    if kind == "chain":
        q, k, v, o, gate, up, down = map(_module, inp["w"])
        chain = ssalaad_amd.LRSLinearChain([[q, k, v], [o], [gate, up], [down]],
                                           sources=[q, o, gate])
        x = inp["x"]
        return dict(kind=kind, chain=chain.prepare(x), x=x)
    if kind == "op":
        crow, col, vals = inp["S"]
        counts = crow[1:] - crow[:-1]
        return dict(kind=kind, x=inp["x"], out=inp["out"], crow=crow.to(torch.int32),
                    col=col.to(torch.int32), vals=vals.transpose(1, 2).contiguous(),
                    active=counts.nonzero().flatten().to(torch.int32))
    if kind == "step":
        return dict(kind=kind, eng=_engine(case, inp), tokens=inp["tokens"],
                    positions=inp["positions"])
    return dict(kind=kind, R=inp["R"], keep=inp["keep"], p=case["p"], q=case["q"])


def run(state):
    kind = state["kind"]
    if kind in ("linear", "nm", "group"):
        return state["mod"](state["x"])
    if kind == "chain":
        return state["chain"].run()
    if kind == "op":
        out = state["out"].clone()  # the op adds in place: each pass starts from the same out
        torch.ops.ssalaad.tilelang_bsr_addmm_inplace_dense_(
            out, state["x"], state["crow"], state["col"], state["vals"], state["active"])
        return out
    if kind == "step":
        return state["eng"].step(state["tokens"], state["positions"])
    S = ssalaad_amd.project_S(state["R"], state["keep"], state["p"], state["q"])
    return (S,) + tuple(ssalaad_amd.encode_for_kernels(S, state["p"], state["q"]))


# ------------------------------------------------------------------- work --
def _linear_work(n, m, r, p, q, density, e):
    """Weight bytes and multiply-adds per token of one linear."""
    NB, NBK = -(-n // p), -(-m // q)
    nnz = int(round(density * NB * NBK))
    return (e * (r * (n + m) + nnz * p * q) + 4 * (nnz + 2 * NB + 1),
            r * (n + m) + nnz * p * q)


def work(case):
    c, kind = case, case["kind"]
    e = 4 if c["dtype"] == "fp32" else 2
    if kind == "compress":
        n, m, p, q = c["n"], c["m"], c["p"], c["q"]
        kept = int(round(c["density"] * (n // p) * (m // q)))
        # R read, S written, then S read and the kept blocks written
        return {"bytes": (e + 4 + 4) * n * m + 4 * kept * (p * q + 1), "flops": 2.0 * n * m}
    M = c["tokens"]
    if kind == "nm":
        n, m, r = c["n"], c["m"], c["r"]
        return {"bytes": e * (M * (n + m) + r * (n + m) + n * m // 2) + n * m // 8
                + (e * n if c["bias"] else 0),
                "flops": 2.0 * M * (r * (n + m) + n * m // 2)}
    if kind == "op":
        NB, NBK = c["n"] // c["p"], c["m"] // c["q"]
        nnz = int(round(c["density"] * NB * NBK))
        # the copy of out that a pass starts from is read and written too
        return {"bytes": e * (M * (c["m"] + 4 * c["n"]) + nnz * c["p"] * c["q"]) + 4 * (nnz + 2 * NB),
                "flops": 2.0 * M * nnz * c["p"] * c["q"]}
    if kind == "linear":
        shapes, q = [(c["n"], c["m"])], c["q"]
        io = M * (c["n"] + c["m"])
    elif kind == "group":
        shapes, q = [(n, c["m"]) for n in (c["n"], c["n2"], c["n3"]) if n], c["p"]
        io = M * (c["m"] + sum(n for n, _ in shapes))
    else:
        heads = (c["kv_heads"] * (c["hidden"] // c["heads"])) if kind == "step" else c["hidden"]
        shapes, q = _layer_shapes(c, c["hidden"], heads) * c.get("layers", 1), c["p"]
        io = M * sum(n for n, _ in shapes) + M * c["hidden"]
    each = [_linear_work(n, m, c["r"], c["p"], q, c["density"], e) for n, m in shapes]
    b, f = sum(x for x, _ in each) + e * io, 2.0 * M * sum(x for _, x in each)
    if kind == "linear" and c["bias"]:
        b += e * c["n"]
    if kind == "step":
        kv = c["layers"] * M * c["kv_heads"] * (c["hidden"] // c["heads"]) * c["context"]
        b += e * (2 * kv + c["vocab"] * (c["hidden"] + M))
        f += 4.0 * kv * (c["heads"] // c["kv_heads"]) + 2.0 * M * c["vocab"] * c["hidden"]
    return {"bytes": b, "flops": f}


# ------------------------------------------------------------ correctness --
def tolerance(case):
    """About four times the error each kind shows against 64-bit sums: linears,
    groups and the op 1.8e-3 in bf16, 2.2e-4 in fp16 and 4e-7 in fp32; a chain's
    last stage 3.6e-3 and a decode step's logits 6.8e-3 in bf16."""
    if case["kind"] == "compress":
        return "exact"
    if case["dtype"] == "fp32":
        return {"rel": 2.5e-6, "max": 2.5e-5}
    bf = 8 if case["dtype"] == "bf16" else 1
    if case["kind"] == "chain":
        return {"rel": 1.9e-3 * bf, "max": 1.5e-2 * bf}
    if case["kind"] == "step":
        return {"rel": 3.4e-3 * bf, "max": 2.5e-2 * bf}
    return {"rel": 9e-4 * bf, "max": 8e-3 * bf}


def _step64(c, inp):
    hd, H, KH = c["hidden"] // c["heads"], c["heads"], c["kv_heads"]
    B, pos = c["tokens"], torch.tensor(inp["positions"], device="cuda")

    def norm(x, w):
        return x * (x.square().mean(-1, keepdim=True) + 1e-5).rsqrt() * w.double()

    inv = 500000.0 ** (-torch.arange(0, hd, 2, device="cuda").double() / hd)
    ang = pos.double()[:, None] * inv
    cos, sin = (torch.cat([f(ang)] * 2, -1)[:, None] for f in (torch.cos, torch.sin))

    def rope(x):
        a, b = x.chunk(2, -1)
        return x * cos + torch.cat([-b, a], -1) * sin

    h = inp["embed"][inp["tokens"]].double()
    for i, ws in enumerate(inp["layers"]):
        x = norm(h, inp["norms"][2 * i])
        q = rope(_linear64(x, ws[0]).view(B, H, hd))
        k = rope(_linear64(x, ws[1]).view(B, KH, hd))
        v = _linear64(x, ws[2]).view(B, KH, hd)
        att = []
        for b in range(B):
            n = inp["positions"][b]
            ks = torch.cat([inp["k"][i, b, :, :n].double(), k[b][:, None]], 1)
            vs = torch.cat([inp["v"][i, b, :, :n].double(), v[b][:, None]], 1)
            ks, vs = (t.repeat_interleave(H // KH, 0) for t in (ks, vs))
            s = (ks * q[b][:, None]).sum(-1) * hd ** -0.5
            att.append((s.softmax(-1)[..., None] * vs).sum(1).reshape(-1))
        h = h + _linear64(torch.stack(att), ws[3])
        x = norm(h, inp["norms"][2 * i + 1])
        g = _linear64(x, ws[4])
        h = h + _linear64(g * torch.sigmoid(g) * _linear64(x, ws[5]), ws[6])
    return norm(h, inp["norms"][-1]) @ inp["head"].double().T


def exact(case, seed):
    inp, kind = _inputs(case, seed), case["kind"]
    if kind in ("linear", "nm"):
        return _linear64(inp["x"].double(), inp["w"][0])
    if kind == "group":
        return tuple(_linear64(inp["x"].double(), w) for w in inp["w"])
    if kind == "chain":
        x, ws = inp["x"].double(), inp["w"]
        qkv = tuple(_linear64(x, w) for w in ws[:3])
        o = _linear64(qkv[0], ws[3])
        gu = tuple(_linear64(o, w) for w in ws[4:6])
        return qkv, (o,), gu, (_linear64(gu[0], ws[6]),)
    if kind == "op":
        w = dict(S=inp["S"], n=case["n"], m=case["m"], p=case["p"], q=case["q"])
        return inp["out"].double() + inp["x"].double() @ _dense(w).T
    if kind == "step":
        return _step64(case, inp)
    # the projection in 64 bits; the encoding of it has no rounding at all
    n, m, p, q = case["n"], case["m"], case["p"], case["q"]
    R = inp["R"].double().view(n // p, p, m // q, q)
    kept = R.square().sum((1, 3)).flatten().topk(inp["keep"]).indices
    mask = torch.zeros((n // p) * (m // q), dtype=torch.bool, device="cuda")
    mask[kept] = True
    return ((R * mask.view(n // p, 1, m // q, 1)).view(n, m), None, None, None, None)
