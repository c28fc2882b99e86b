"""The calls this framework is timed on: the drop-in module's forward and the
single layers under it (projection, feed-forward block, attention, residual
add + LayerNorm), each through its public entry point.

``listed()`` names the cases, ``draw(rng)`` gives one more of the same ranges,
``prepare`` makes what a program holds before the call, ``run`` is one pass,
``work`` the bytes and operations a pass cannot do without, ``tolerance`` the
difference another correct implementation at the same precision may show and
``exact`` the result in 64 bits from plain torch.
"""

import math
import os
import random
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "tiktok-techjam-2026_amd"))

from tjkernels import TransformerConfig, UserOptimizedTransformer, ops  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
WEIGHT_STD = 0.02
EPS = 1e-5


def listed():
    return [
        # Batch inference of the headline configuration (4 layers, d 1024,
        # S 2048) over prompts of different lengths.
        dict(name="model-bf16", kind="model", dtype="bf16", layers=4, d=1024, heads=16, ffn=4096, batch=4, seq=2048,
             min_len=1024, causal=True),
        # One short sequence through a small model: latency of a single
        # interactive request.
        dict(name="model-short-fp16", kind="model", dtype="fp16", layers=4, d=512, heads=8, ffn=2048, batch=1, seq=128,
             min_len=0, causal=True),
        # One layer of an fp32 model (the plan that holds the 1e-4 budget) on
        # a ragged batch.
        dict(name="block-fp32", kind="model", dtype="fp32", layers=1, d=512, heads=8, ffn=2048, batch=4, seq=512,
             min_len=128, causal=True),
        # The packed QKV projection of the headline model over the valid
        # tokens of a ragged batch.
        dict(name="qkv-bf16", kind="proj", dtype="bf16", rows=5430, k=1024, n=3072),
        # The headline model's feed-forward block over the same tokens, added
        # into the residual.
        dict(name="mlp-bf16", kind="mlp", dtype="bf16", rows=5430, d=1024, f=4096),
        # The feed-forward block of the wide model (d 2048), the largest
        # contraction in use.
        dict(name="mlp-wide-bf16", kind="mlp", dtype="bf16", rows=8192, d=2048, f=8192),
        # The small model's feed-forward block on one short sequence.
        dict(name="mlp-short-fp16", kind="mlp", dtype="fp16", rows=128, d=512, f=2048),
        # A feed-forward block whose widths are no multiple of the matrix
        # tile, on an odd number of tokens.
        dict(name="mlp-odd-fp16", kind="mlp", dtype="fp16", rows=2443, d=1000, f=2600),
        # Causal attention over packed prompts of different lengths.
        dict(name="attn-packed-bf16", kind="attn", dtype="bf16", layout="packed", batch=4, seq=2048, heads=16, hd=64,
             min_len=1024, causal=True),
        # Causal attention of the wide model: long full sequences, head
        # dimension 128.
        dict(name="attn-long-bf16", kind="attn", dtype="bf16", layout="padded", batch=2, seq=4096, heads=16, hd=128,
             min_len=0, causal=True),
        # Bidirectional encoder attention with an arbitrary (non-prefix) mask
        # of valid tokens.
        dict(name="attn-masked-fp16", kind="attn", dtype="fp16", layout="masked", batch=8, seq=512, heads=12, hd=64,
             min_len=0, causal=False),
        # The residual add + LayerNorm between two blocks of the wide model.
        dict(name="norm-bf16", kind="norm", dtype="bf16", rows=8192, d=2048),
    ]


# ------------------------------------------------------------------ drawing

def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A feature width: mostly whole matrix tiles, now and then not."""
    w = _log(rng, lo, hi)
    step = 64 if rng.random() < 0.7 else 8
    return max(step, (w + step // 2) // step * step)


def _draw_model(rng):
    hd = rng.choice([32, 64, 64, 128])
    heads = max(1, _log(rng, 128, 1024) // hd)
    batch = _log(rng, 1, 16)
    seq = max(16, min(2048, _log(rng, 16, 8192) // batch))
    return dict(kind="model", dtype=rng.choice(["bf16", "fp16", "fp32"]), layers=rng.randint(1, 4), d=heads * hd,
                heads=heads, ffn=heads * hd * rng.choice([1, 2, 4]), batch=batch, seq=seq,
                min_len=rng.choice([0, max(1, seq // 2), 1]), causal=rng.random() < 0.8)


def _draw_proj(rng):
    return dict(kind="proj", dtype=rng.choice(["bf16", "fp16", "fp32"]), rows=_log(rng, 16, 16384),
                k=_width(rng, 128, 4096), n=_width(rng, 128, 8192))


def _draw_mlp(rng):
    return dict(kind="mlp", dtype=rng.choice(["bf16", "fp16"]), rows=_log(rng, 16, 16384), d=_width(rng, 128, 2048),
                f=_width(rng, 256, 8192))


def _draw_attn(rng):
    layout = rng.choice(["packed", "padded", "masked"])
    batch, hd = _log(rng, 1, 16), rng.choice([32, 64, 64, 96, 128])
    seq = _log(rng, 64, 8192)
    return dict(kind="attn", dtype=rng.choice(["bf16", "fp16"]), layout=layout, batch=batch, seq=seq,
                heads=_log(rng, 2, 16), hd=hd, min_len=max(1, seq // rng.choice([2, 8])) if layout == "packed" else 0,
                causal=rng.random() < 0.6)


def _draw_norm(rng):
    return dict(kind="norm", dtype=rng.choice(["bf16", "fp16"]), rows=_log(rng, 64, 32768), d=_width(rng, 128, 4096))


def _cost(case):
    """Rough seconds of a pass, to keep a drawn case below the largest listed one."""
    w = work(case)
    rate = 60e12 if case["dtype"] == "fp32" else 250e12 if case["kind"] == "attn" else 500e12
    return w["flops"] / rate + w["bytes"] / 2e12


def draw(rng):
    kind = rng.choice([_draw_model, _draw_proj, _draw_mlp, _draw_attn, _draw_attn, _draw_norm])
    while True:
        case = kind(rng)
        if _cost(case) <= 0.7e-3:
            return case


# ------------------------------------------------------------------- inputs

def _lengths(case, seed):
    """Sequence lengths spread evenly over [min_len, seq], in an order of the
    seed's; all of them ``seq`` without a min_len."""
    b, s, lo = case["batch"], case["seq"], case["min_len"]
    if not lo:
        return [s] * b
    out = [lo + int((i + 0.5) / b * (s - lo + 1)) for i in range(b)]
    random.Random(seed).shuffle(out)
    return out


class _Random:
    """Normal values on the GPU from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=self.g, device="cuda") * std).to(dtype)

    def keep(self, *shape, share):
        return torch.rand(*shape, generator=self.g, device="cuda") < share


def _model_weights(case, rng):
    """fp32 state_dict of the module, its matrices rounded to the case's dtype."""
    d, f, dt = case["d"], case["ffn"], DTYPES[case["dtype"]]

    def mat(*shape):
        return rng.normal(*shape, std=WEIGHT_STD, dtype=dt).float()

    sd = {}
    for i in range(case["layers"]):
        p = "layers.%d." % i
        for norm in ("norm1", "norm2"):
            sd[p + norm + ".weight"] = (1 + mat(d)).to(dt).float()
            sd[p + norm + ".bias"] = mat(d)
        for name in ("q_proj", "k_proj", "v_proj", "out_proj"):
            sd[p + "attention.%s.weight" % name] = mat(d, d)
            sd[p + "attention.%s.bias" % name] = mat(d)
        sd[p + "ffn_in.weight"], sd[p + "ffn_in.bias"] = mat(f, d), mat(f)
        sd[p + "ffn_out.weight"], sd[p + "ffn_out.bias"] = mat(d, f), mat(d)
    sd["final_norm.weight"], sd["final_norm.bias"] = (1 + mat(d)).to(dt).float(), mat(d)
    return sd


def _inputs(case, seed):
    """The tensors a pass reads, before anything of the framework is made."""
    rng, kind, dt = _Random(seed), case["kind"], DTYPES[case["dtype"]]
    t = {}
    if kind == "model":
        b, s = case["batch"], case["seq"]
        t["weights"] = _model_weights(case, rng)
        lengths = torch.tensor(_lengths(case, seed), device="cuda")
        t["mask"] = torch.arange(s, device="cuda")[None, :] < lengths[:, None]
        t["x"] = (rng.normal(b, s, case["d"]) * t["mask"][..., None]).to(dt)
        t["lengths"] = lengths
    elif kind == "proj":
        t["h"] = rng.normal(case["rows"], case["k"], dtype=dt)
        t["w"] = rng.normal(case["n"], case["k"], std=WEIGHT_STD, dtype=dt)
        t["b"] = rng.normal(case["n"], std=WEIGHT_STD, dtype=dt)
    elif kind == "mlp":
        m, d, f = case["rows"], case["d"], case["f"]
        t["h"] = rng.normal(m, d, dtype=dt)
        t["w1"], t["b1"] = rng.normal(f, d, std=WEIGHT_STD, dtype=dt), rng.normal(f, std=WEIGHT_STD, dtype=dt)
        t["w2"], t["b2"] = rng.normal(d, f, std=WEIGHT_STD, dtype=dt), rng.normal(d, std=WEIGHT_STD, dtype=dt)
        t["res"] = rng.normal(m, d)
    elif kind == "attn":
        b, s, h, hd = case["batch"], case["seq"], case["heads"], case["hd"]
        if case["layout"] == "packed":
            lengths = _lengths(case, seed)
            cu = [0]
            for n in lengths:
                cu.append(cu[-1] + n)
            t["cu"] = torch.tensor(cu, dtype=torch.int32, device="cuda")
            t["lengths"] = lengths
            t["qkv"] = rng.normal(cu[-1], 3, h, hd, dtype=dt)
        else:
            t["qkv"] = rng.normal(b, s, 3, h, hd, dtype=dt)
            if case["layout"] == "masked":
                t["mask"] = rng.keep(b, s, share=0.75)
    else:
        m, d = case["rows"], case["d"]
        t["res"], t["delta"] = rng.normal(m, d), rng.normal(m, d, std=0.5, dtype=dt)
        t["gamma"], t["beta"] = 1 + rng.normal(d, std=WEIGHT_STD), rng.normal(d, std=WEIGHT_STD)
    return t


def prepare(case, seed):
    t, kind, dt = _inputs(case, seed), case["kind"], DTYPES[case["dtype"]]
    state = {"kind": kind, "case": case}
    if kind == "model":
        cfg = TransformerConfig(batch_size=case["batch"], seq_len=case["seq"], d_model=case["d"],
                                num_heads=case["heads"], ffn_dim=case["ffn"], num_layers=case["layers"],
                                causal=case["causal"])
        with torch.device("meta"):
            module = UserOptimizedTransformer(cfg)
        module = module.to_empty(device="cuda")
        module.load_state_dict(t.pop("weights"), strict=True)
        state["module"] = module.to(dtype=dt).eval()
        state["x"] = t["x"]
        state["mask"] = t["mask"] if case["min_len"] else None
        return state
    state.update(t)
    # the activations a layer writes are buffers that a program keeps
    if kind == "proj":
        state["out"] = torch.empty(case["rows"], case["n"], dtype=dt, device="cuda")
    elif kind == "mlp":
        state["mid"] = torch.empty(case["rows"], case["f"], dtype=dt, device="cuda")
    elif kind == "attn":
        rows = t["qkv"].shape[0] if case["layout"] == "packed" else case["batch"] * case["seq"]
        state["out"] = torch.empty(rows, case["heads"] * case["hd"], dtype=dt, device="cuda")
        if case["layout"] == "packed":
            state["longest"] = max(t["lengths"])
    elif kind == "norm":
        state["out"] = torch.empty(case["rows"], case["d"], dtype=dt, device="cuda")
    return state


def run(state):
    s, kind = state, state["kind"]
    if kind == "model":
        with torch.inference_mode():
            return s["module"](s["x"], s["mask"])
    if kind == "proj":
        return ops.gemm(s["h"], s["w"], s["b"], s["out"], ops.EPI_BIAS)
    if kind == "mlp":
        ops.gemm(s["h"], s["w1"], s["b1"], s["mid"], ops.EPI_BIAS_GELU)
        return ops.gemm(s["mid"], s["w2"], s["b2"], s["res"], ops.EPI_BIAS_RESIDUAL)
    if kind == "attn":
        c = s["case"]
        if c["layout"] == "packed":
            return ops.flash_attention(s["qkv"], s["out"], causal=c["causal"], cu_seqlens=s["cu"],
                                       max_seqlen=s["longest"])
        return ops.flash_attention(s["qkv"], s["out"], causal=c["causal"], key_mask=s.get("mask"))
    ops.add_layernorm(s["res"], s["delta"], s["gamma"], s["beta"], EPS, s["out"], res_out=s["res"])
    return [s["out"], s["res"]]


# --------------------------------------------------------------------- work

def _pairs(lengths, causal):
    return sum(n * (n + 1) // 2 if causal else n * n for n in lengths)


def work(case):
    kind, es = case["kind"], 4 if case["dtype"] == "fp32" else 2
    if kind == "model":
        d, f, n = case["d"], case["ffn"], case["layers"]
        lengths = _lengths(case, 0)
        t = sum(lengths)
        flops = n * (8.0 * t * d * d + 4.0 * t * d * f + 4.0 * d * _pairs(lengths, case["causal"]))
        weights = n * (4 * d * d + 2 * d * f + 9 * d + f) + 2 * d
        return {"bytes": es * (weights + t * d + case["batch"] * case["seq"] * d), "flops": flops}
    if kind == "proj":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": es * (m * k + n * k + n + m * n), "flops": 2.0 * m * n * k}
    if kind == "mlp":
        m, d, f = case["rows"], case["d"], case["f"]
        return {"bytes": es * (m * d + 2 * d * f + d + f) + 8 * m * d, "flops": 4.0 * m * d * f}
    if kind == "attn":
        lengths = _lengths(case, 0)
        d = case["heads"] * case["hd"]
        mask = case["batch"] * case["seq"] if case["layout"] == "masked" else 0
        return {"bytes": es * 4 * sum(lengths) * d + mask, "flops": 4.0 * d * _pairs(lengths, case["causal"])}
    m, d = case["rows"], case["d"]
    return {"bytes": m * d * (8 + 2 * es) + 8 * d, "flops": 8.0 * m * d}


# ------------------------------------------------------------------ results

def tolerance(case):
    # about four times the error measured against exact() (bf16 2.5e-3 for a
    # model and 1.7e-3 to 2.0e-3 for a layer, fp16 3e-4, fp32 2.5e-7; sums of
    # 4096 fp32 products in another order differ by more than 512 do)
    if case["dtype"] == "fp32":
        return {"rel": 5e-6}
    if case["dtype"] == "fp16":
        return {"rel": 1.2e-3}
    return {"rel": 1e-2 if case["kind"] == "model" else 8e-3}


def _attend(q, k, v, causal, keep=None):
    """softmax(q k^T / sqrt(hd)) v over [H, L, hd]; a row without a key is 0."""
    n = q.shape[1]
    s = torch.matmul(q, k.transpose(1, 2)) * q.shape[2] ** -0.5
    hide = torch.zeros(n, n, dtype=torch.bool, device=q.device)
    if causal:
        hide |= torch.ones_like(hide).triu(1)
    if keep is not None:
        hide |= ~keep[None, :]
    p = torch.softmax(s.masked_fill_(hide, float("-inf")), dim=-1).nan_to_num_(0.0)
    return torch.matmul(p, v)


def _exact_model(case, t):
    d, h = case["d"], case["heads"]
    w = {k: v.double() for k, v in t["weights"].items()}
    out = torch.zeros(t["x"].shape, dtype=torch.float64, device="cuda")
    for b, n in enumerate(t["lengths"].tolist()):
        x = t["x"][b, :n].double()
        for i in range(case["layers"]):
            p = "layers.%d." % i
            y = F.layer_norm(x, (d,), w[p + "norm1.weight"], w[p + "norm1.bias"], EPS)
            q, k, v = (F.linear(y, w[p + "attention.%s.weight" % m], w[p + "attention.%s.bias" % m])
                       .view(n, h, d // h).transpose(0, 1) for m in ("q_proj", "k_proj", "v_proj"))
            ctx = _attend(q, k, v, case["causal"]).transpose(0, 1).reshape(n, d)
            x = x + F.linear(ctx, w[p + "attention.out_proj.weight"], w[p + "attention.out_proj.bias"])
            y = F.layer_norm(x, (d,), w[p + "norm2.weight"], w[p + "norm2.bias"], EPS)
            y = F.gelu(F.linear(y, w[p + "ffn_in.weight"], w[p + "ffn_in.bias"]))
            x = x + F.linear(y, w[p + "ffn_out.weight"], w[p + "ffn_out.bias"])
        out[b, :n] = F.layer_norm(x, (d,), w["final_norm.weight"], w["final_norm.bias"], EPS)
    return out


def _exact_attn(case, t):
    h, hd = case["heads"], case["hd"]
    packed = case["layout"] == "packed"
    lengths = t["lengths"] if packed else [case["seq"]] * case["batch"]
    rows = t["qkv"] if packed else t["qkv"].reshape(-1, 3, h, hd)
    out = torch.empty(rows.shape[0], h * hd, dtype=torch.float64, device="cuda")
    at = 0
    for b, n in enumerate(lengths):
        keep = t["mask"][b] if "mask" in t else None
        for j in range(h):  # one head at a time: the scores are n x n
            q, k, v = (rows[at:at + n, c, j].double().unsqueeze(0) for c in range(3))
            out[at:at + n, j * hd:(j + 1) * hd] = _attend(q, k, v, case["causal"], keep)[0]
        at += n
    return out


def exact(case, seed):
    kind, t = case["kind"], _inputs(case, seed)
    if kind == "model":
        return _exact_model(case, t)
    if kind == "proj":
        return F.linear(t["h"].double(), t["w"].double(), t["b"].double())
    if kind == "mlp":
        mid = F.gelu(F.linear(t["h"].double(), t["w1"].double(), t["b1"].double()))
        return t["res"].double() + F.linear(mid, t["w2"].double(), t["b2"].double())
    if kind == "attn":
        return _exact_attn(case, t)
    x = t["res"].double() + t["delta"].double()
    return [F.layer_norm(x, (case["d"],), t["gamma"].double(), t["beta"].double(), EPS), x]
