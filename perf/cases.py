"""The work that users of this package have it do, as measurable cases: attention training steps (causal and
non-causal), whole attention blocks, and recurrent inference, through the public entry points."""
import math
from types import SimpleNamespace

import torch
import torch.nn.functional as F

import cottention_transformer_amd as ct
from cottention_transformer_amd.modules import BertCosAttention, GPTCosAttention

DEV = "cuda:0"
_DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}

# Elements of one (B,H,N,D) tensor up to which cases are drawn, per path and type: those of the largest listed case of
# that path and type, so that a drawn case costs no more than the listed ones.
_MOST = {"bf16": 1 << 27, "fp16": 1 << 27, "autocast": 1 << 24, "fp32": 1 << 22, "wide": 1 << 22, "noncausal": 1 << 24,
         "noncausal32": 1 << 22}


def _attention(name, path, b, h, n, dk, dv, dtype):
    c = {"path": path, "B": b, "H": h, "N": n, "Dk": dk, "Dv": dv, "dtype": dtype}
    return dict(c, name=name) if name else c


def _block(name, path, b, s, e, h, masked):
    c = {"path": path, "B": b, "S": s, "E": e, "H": h, "masked": masked}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a training step of the attention operator, forward and gradients: the reference's CPU-runnable size, all latency
        _attention("causal_small_fp32", "causal", 1, 2, 128, 64, 64, "fp32"),
        # one short sequence of odd length, fp16 (the length of the reference's timing script)
        _attention("causal_1023_fp16", "causal", 1, 12, 1023, 64, 64, "fp16"),
        # the headline: a batch of GPT-300M-shaped sequences
        _attention("causal_gpt300m_bf16", "causal", 8, 16, 2048, 64, 64, "bf16"),
        # the same step as the reference's trainer makes it: fp32 tensors under autocast, forward in bf16, gradients in fp32
        _attention("causal_gpt300m_autocast", "causal", 8, 16, 2048, 64, 64, "autocast"),
        # GPT-1.2B-shaped heads over a long context: the largest tensors
        _attention("causal_65536_bf16", "causal", 1, 16, 65536, 128, 128, "bf16"),
        # the same heads in fp32, a medium sequence
        _attention("causal_2048_d128_fp32", "causal", 1, 16, 2048, 128, 128, "fp32"),
        # 16 heads of a 4096-wide model at S = 1024, a point of the reference's published width sweep
        _attention("causal_d256_bf16", "causal", 1, 16, 1024, 256, 256, "bf16"),
        # BERT-style non-causal step
        _attention("noncausal_bert_bf16", "noncausal", 32, 12, 512, 64, 64, "bf16"),
        # a whole causal attention block of a training step under bf16 autocast, padded batch
        _block("gpt_block", "gpt_block", 8, 2048, 1024, 16, True),
        # a whole BERT self-attention block of a training step under bf16 autocast, padded batch
        _block("bert_block", "bert_block", 32, 512, 768, 12, True),
        # one recurrent step of a large serving batch
        {"name": "decode_batch256", "path": "decode", "B": 256, "H": 16, "D": 128, "dtype": "bf16"},
        # one user's generation through a GPT-1.2B-shaped block: a prompt, then tokens one by one
        {"name": "generate_batch1", "path": "generate", "B": 1, "P": 1000, "T": 16, "E": 2048, "H": 16},
    ]


def _spread(rng, lo, hi):
    """An integer between lo and hi, evenly over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _fit(rng, most, h, d, lo, hi):
    """(B, N) with N between lo and hi over the logarithm and B*H*N*D within `most` elements."""
    n = _spread(rng, lo, max(lo, min(hi, most // (h * d))))
    return _spread(rng, 1, max(1, min(64, most // (h * d * n)))), n


def draw(rng):
    kind = rng.choice(["causal16"] * 5 + ["autocast", "fp32", "fp32", "wide", "wide", "noncausal", "noncausal",
                                          "gpt_block", "bert_block", "decode", "generate"])
    h = rng.choice([2, 4, 8, 12, 16, 16, 20, 32])
    d = rng.choice([32, 48, 64, 64, 64, 80, 96, 128, 128])
    dv = d if rng.random() < 0.8 else rng.choice([32, 64, 128])
    if kind == "causal16":
        b, n = _fit(rng, _MOST["bf16"], h, max(d, dv), 63, 65536)
        return _attention(None, "causal", b, h, n, d, dv, rng.choice(["bf16", "bf16", "fp16"]))
    if kind in ("autocast", "fp32"):
        b, n = _fit(rng, _MOST[kind], h, max(d, dv), 63, 8192)
        return _attention(None, "causal", b, h, n, d, dv, kind)
    if kind == "wide":
        d = rng.choice([160, 192, 224, 256, 256])
        h = rng.choice([2, 4, 8, 12, 16])
        b, n = _fit(rng, _MOST["wide"], h, d, 63, 4096)
        return _attention(None, "causal", b, h, n, d, d, rng.choice(["bf16", "bf16", "fp16"]))
    if kind == "noncausal":
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        b, n = _fit(rng, _MOST["noncausal32" if dtype == "fp32" else "noncausal"], h, max(d, dv), 31, 8192)
        return _attention(None, "noncausal", b, h, n, d, dv, dtype)
    if kind in ("gpt_block", "bert_block"):
        e, h = rng.choice([(512, 8), (768, 12), (1024, 16), (1024, 8), (2048, 16)])
        s = _spread(rng, 65, 2048)
        b = _spread(rng, 1, max(1, min(32, (1 << 24) // (s * e) * 1024 // e)))
        return _block(None, kind, b, s, e, h, rng.random() < 0.5)
    if kind == "decode":
        d = rng.choice([64, 64, 128, 128])
        return {"path": "decode", "B": _spread(rng, 1, (1 << 26) // (h * d * d) if h * d * d * 256 > 1 << 26 else 256), "H": h,
                "D": d, "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"])}
    e, h = rng.choice([(768, 12), (1024, 16), (2048, 16)])
    return {"path": "generate", "B": _spread(rng, 1, 8), "P": _spread(rng, 17, 1000), "T": _spread(rng, 4, 16), "E": e, "H": h}


def _rotary_dim(case):
    return min(64, case["E"] // case["H"])


def _lengths(g, b, s):
    """Keep mask of a padded batch: every sequence at least half full."""
    lengths = torch.randint((s + 1) // 2, s + 1, (b, 1), generator=g, device=DEV)
    return torch.arange(s, device=DEV)[None, :] < lengths


def _module(cls, config, seed):
    torch.manual_seed(seed)
    with torch.device(DEV):
        m = cls(config)
        with torch.no_grad():
            m.norm_const.copy_(torch.linspace(-1.0, 1.0, config.num_attention_heads).reshape(1, -1, 1, 1))
    return m


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    randn = lambda *shape, **kw: torch.randn(*shape, generator=g, device=DEV, **kw)
    path = case["path"]
    if path in ("causal", "noncausal"):
        b, h, n, dk, dv = (case[x] for x in ("B", "H", "N", "Dk", "Dv"))
        dtype = _DTYPES.get(case["dtype"], torch.float32)
        out_dtype = torch.bfloat16 if case["dtype"] == "autocast" else dtype
        q, k = (F.normalize(randn(b, h, n, dk), dim=-1).to(dtype).requires_grad_(True) for _ in range(2))
        v = randn(b, h, n, dv).to(dtype).requires_grad_(True)
        return {"case": case, "qkv": (q, k, v), "grad": randn(b, h, n, dv).to(out_dtype)}
    if path in ("gpt_block", "bert_block"):
        b, s, e, h = (case[x] for x in ("B", "S", "E", "H"))
        config = SimpleNamespace(hidden_size=e, num_attention_heads=h, max_position_embeddings=2048, rotary_dim=_rotary_dim(case),
                                 attn_pdrop=0.0, resid_pdrop=0.0, attention_probs_dropout_prob=0.0)
        m = _module(GPTCosAttention if path == "gpt_block" else BertCosAttention, config, seed)
        mask = None
        if case["masked"]:  # as the surrounding model hands it over: 0 at real tokens, a large negative number at padding
            mask = torch.where(_lengths(g, b, s), 0.0, torch.finfo(torch.float32).min)[:, None, None, :]
        kw = {"attention_mask": mask}
        if path == "gpt_block":
            kw["position_ids"] = torch.arange(s, device=DEV)[None, :]
        return {"case": case, "module": m, "hidden": randn(b, s, e).requires_grad_(True), "kw": kw, "params": list(m.parameters()),
                "grad": randn(b, s, e).to(torch.bfloat16)}
    if path == "decode":
        b, h, d = case["B"], case["H"], case["D"]
        dtype = _DTYPES[case["dtype"]]
        q, k = (F.normalize(randn(b, h, d), dim=-1).to(dtype) for _ in range(2))
        return {"case": case, "state": 0.1 * randn(b, h, d, d), "q": q, "k": k, "v": randn(b, h, d).to(dtype)}
    b, p, t, e, h = (case[x] for x in ("B", "P", "T", "E", "H"))
    config = SimpleNamespace(hidden_size=e, num_attention_heads=h, max_position_embeddings=2048, rotary_dim=_rotary_dim(case),
                             attn_pdrop=0.0, resid_pdrop=0.0, fast_inference=True)
    m = _module(GPTCosAttention, config, seed).to(torch.bfloat16).eval()
    return {"case": case, "module": m, "prompt": randn(b, p, e).to(torch.bfloat16), "tokens": randn(t, b, 1, e).to(torch.bfloat16)}


def run(state):
    case = state["case"]
    path = case["path"]
    if path in ("causal", "noncausal"):
        op = ct.CustomAttention if path == "causal" else ct.NonCausalAttention
        if case["dtype"] == "autocast":
            with torch.autocast("cuda", dtype=torch.bfloat16):
                out = op.apply(*state["qkv"])
        else:
            out = op.apply(*state["qkv"])
        return (out.detach(), *torch.autograd.grad(out, state["qkv"], state["grad"]))
    if path in ("gpt_block", "bert_block"):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            out = state["module"](state["hidden"], **state["kw"])[0]
        return (out.detach(), *torch.autograd.grad(out, [state["hidden"], *state["params"]], state["grad"]))
    if path == "decode":
        return ct.decode_step(state["state"], state["q"], state["k"], state["v"]), state["state"]
    m = state["module"]
    m.reset_state()
    with torch.no_grad():
        outs = [m(state["prompt"])[0]]
        outs += [m(token)[0] for token in state["tokens"]]
    return (torch.cat(outs, dim=1), m.state)


def work(case):
    """Each input read and each output written once; the multiplications of the definition, two operations each."""
    path = case["path"]
    if path in ("causal", "noncausal"):
        units = case["B"] * case["H"] * case["N"]
        size = 2 if case["dtype"] in ("bf16", "fp16") else 4
        grad = 2 if case["dtype"] == "autocast" else size
        dk, dv = case["Dk"], case["Dv"]
        # in: q, k, v, d_o; out: o, dq, dk, dv.  Forward: state update and read-out; gradients: two states, three read-outs
        return {"bytes": units * (size * (4 * dk + 2 * dv) + grad * 2 * dv), "flops": 14 * units * dk * dv}
    if path in ("gpt_block", "bert_block"):
        rows, e = case["B"] * case["S"], case["E"]
        mats = 4 if path == "gpt_block" else 3
        # fp32 hidden states and parameters in, their gradients out; the bf16 output and its gradient
        return {"bytes": rows * e * (4 + 4 + 2 + 2) + 8 * mats * e * e,
                "flops": 3 * mats * 2 * rows * e * e + 14 * rows * e * (e // case["H"])}
    if path == "decode":
        heads, d = case["B"] * case["H"], case["D"]
        return {"bytes": heads * (8 * d * d + 4 * d * (4 if case["dtype"] == "fp32" else 2)), "flops": 4 * heads * d * d}
    rows, e = case["B"] * (case["P"] + case["T"]), case["E"]
    state = case["B"] * e * (e // case["H"])
    # the weights are needed once for the prompt and once for each token, which follows from the one before
    return {"bytes": 2 * 2 * rows * e + (1 + case["T"]) * 4 * 2 * e * e + case["T"] * 8 * state + 4 * state,
            "flops": 4 * 2 * rows * e * e + 4 * rows * e * (e // case["H"])}


def tolerance(case):
    """About four times the largest relative error against the same path in 64 bits: 6.3e-6 in fp32, 3.0e-4 in fp16, 2.4e-3 in
    bf16, and 6.4e-3 through a block's chain of bf16 products (bias gradients, sums over all rows, up to 1e-2)."""
    dtype = case.get("dtype", "bf16")
    if case["path"] in ("gpt_block", "bert_block", "generate"):
        return {"rel": 2.5e-2}
    return {"rel": {"fp32": 2.5e-5, "fp16": 1.2e-3}.get(dtype, 1e-2)}
