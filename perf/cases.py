"""The work a user of this framework has it do, as a list of measurable cases.

A pass is one mixture-of-experts layer on one batch of tokens, as a serving
engine calls it: the router's logits go through the configuration's top-k
(softmax, or sigmoid scores with a correction bias and grouped selection), and
``XpuFusedMoe.apply`` runs the chosen experts.  The sizes are those of the
benchmark configurations in ``vllm_xpu_kernels/workloads.py``, whole or as one
rank of an expert- or tensor-parallel deployment holds them; token counts run
from one (a single decode) to 8192 (the largest prefill batch measured there),
odd ones included.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "vllm-xpu-kernels_amd"))

DEV = "cuda"

# hidden, intermediate, experts, top-k, router, activation, biases, router skew
SHAPES = {
    "tiny": (512, 1024, 8, 2, "softmax", "silu", False, 0.0),
    "qwen3-30b-a3b": (2048, 768, 128, 8, "softmax", "silu", False, 0.0),
    "qwen3-235b-a22b": (4096, 1536, 128, 8, "softmax", "silu", False, 0.5225),
    "deepseek-v3": (7168, 2048, 256, 8, "grouped", "silu", False, 0.0),
    "gpt-oss-20b": (2880, 2880, 32, 4, "softmax", "swigluoai", True, 0.0),
}
GROUPS, TOP_GROUPS, ROUTED_SCALE = 8, 4, 2.5  # the grouped router's


def _case(shape, recipe, tokens, dtype="bf16", ep=1, tp=1, prequant=False, name=None):
    c = {"shape": shape, "recipe": recipe, "tokens": tokens, "dtype": dtype, "ep": ep, "tp": tp,
         "prequant": prequant}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one user's decode step: latency, and the launches of a layer
        _case("gpt-oss-20b", "mxfp4", 1, name="mxfp4_decode_1"),
        _case("deepseek-v3", "fp8block", 1, name="fp8_decode_1"),
        # small decode batches: a few slots per expert, most experts active
        _case("qwen3-30b-a3b", "bf16", 24, name="bf16_decode_24"),
        _case("qwen3-30b-a3b", "int4", 61, dtype="fp16", name="int4_decode_61"),
        _case("deepseek-v3", "fp8block", 64, name="fp8_decode_64"),
        # continuous batching at full load: all weights read once, 16 slots
        # per expert or so
        _case("gpt-oss-20b", "mxfp4", 128, name="mxfp4_decode_128"),
        _case("qwen3-30b-a3b", "bf16", 250, name="bf16_decode_250"),
        # one rank of eight in expert parallelism: 32 of 256 experts, tokens
        # of all ranks, already quantised by the dispatch that sent them
        _case("deepseek-v3", "fp8block", 1003, ep=8, prequant=True, name="fp8_ep_rank_1003"),
        # prefill chunks; the second with a skewed router
        _case("qwen3-30b-a3b", "bf16", 3001, name="bf16_prefill_3001"),
        _case("qwen3-235b-a22b", "fp8block", 2048, name="fp8_prefill_2048_skewed"),
        _case("gpt-oss-20b", "mxfp4", 4096, name="mxfp4_prefill_4096"),
        # the largest batch of the benchmark
        _case("deepseek-v3", "fp8block", 8192, name="fp8_prefill_8192"),
    ]


def draw(rng):
    shape, recipe = rng.choice([
        ("tiny", "bf16"), ("qwen3-30b-a3b", "bf16"), ("qwen3-30b-a3b", "bf16"),
        ("qwen3-30b-a3b", "int4"), ("qwen3-235b-a22b", "fp8block"),
        ("deepseek-v3", "fp8block"), ("deepseek-v3", "fp8block"), ("deepseek-v3", "mxfp8"),
        ("deepseek-v3", "fp8"), ("gpt-oss-20b", "mxfp4"), ("gpt-oss-20b", "mxfp4")])
    # 16-bit matrix instructions on the largest shape: a quarter of the tokens
    # costs what the largest listed case does
    tokens = int(round(math.exp(rng.uniform(0.0, math.log(2048 if recipe == "fp8" else 8192)))))
    dtype = "fp16" if recipe in ("bf16", "int4", "mxfp4", "fp8") and rng.random() < 0.3 else "bf16"
    ep = tp = 1
    split = rng.random()
    if split < 0.25 and shape != "tiny":
        ep = rng.choice([2, 4, 8])
    elif split < 0.5:
        # fp8 block scales need an intermediate size % 128, int4 groups too
        tp = rng.choice({"tiny": [2, 4], "qwen3-30b-a3b": [2], "qwen3-235b-a22b": [2, 4],
                         "deepseek-v3": [2, 4, 8], "gpt-oss-20b": [2]}[shape])
    prequant = recipe == "fp8block" and rng.random() < 0.3
    return _case(shape, recipe, tokens, dtype, ep, tp, prequant)


def _sizes(case):
    H, I, E, k, router, act, bias, tau = SHAPES[case["shape"]]
    return H, I // case["tp"], E, E // case["ep"], k, router, act, bias, tau


def _dtype(case):
    return torch.float16 if case["dtype"] == "fp16" else torch.bfloat16


# ------------------------------------------------------------------ weights
# Normal weights of standard deviation 0.02, in each recipe's storage form.

def _fp8_block(w):
    """[e, N, K] -> e4m3 and a scale per 128 x 128 block."""
    e, N, K = w.shape
    b = w.view(e, N // 128, 128, K // 128, 128)
    s = (b.abs().amax((2, 4)) / 448.0).clamp(min=1e-6)
    return (b / s[:, :, None, :, None]).view(e, N, K).to(torch.float8_e4m3fn), s


def _pow2_scale(w, top):
    """Per 32 along K: the least power of two that brings w within top; (w / it, its e8m0 code)."""
    b = w.view(*w.shape[:-1], -1, 32)
    e = torch.ceil(torch.log2(b.abs().amax(-1, keepdim=True).clamp(min=1e-30) / top)).clamp(-127, 127)
    return b * torch.exp2(-e), (e + 127).squeeze(-1).to(torch.uint8)


def _e2m1(v):
    m = v.abs()
    c = torch.zeros_like(m, dtype=torch.uint8)
    for bound in (0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0):
        c += (m > bound).to(torch.uint8)
    return c | ((v < 0).to(torch.uint8) << 3)


def _pairs(codes):
    return codes[..., 0::2] | (codes[..., 1::2] << 4)


def _matrices(case, gen, E, N, K):
    """One weight of every expert in the layout the layer's constructor takes, and its scales."""
    recipe = case["recipe"]
    if recipe == "bf16":
        w = torch.randn(E, K, N, generator=gen, device=DEV, dtype=_dtype(case))
        return w.mul_(0.02), None
    ws, ss = [], []
    step = max(1, (1 << 28) // (N * K))
    for e0 in range(0, E, step):
        w = torch.randn(min(step, E - e0), N, K, generator=gen, device=DEV).mul_(0.02)
        if recipe == "fp8block":
            q, s = _fp8_block(w)
        elif recipe == "fp8":
            s = w.abs().amax((1, 2)) / 448.0
            q = (w / s[:, None, None]).to(torch.float8_e4m3fn).transpose(1, 2).contiguous()
        elif recipe == "mxfp8":
            v, s = _pow2_scale(w, 448.0)
            q = v.view(w.shape).to(torch.float8_e4m3fn).transpose(1, 2).contiguous()
            s = s.transpose(1, 2).contiguous()
        elif recipe == "mxfp4":
            v, s = _pow2_scale(w, 6.0)
            q = _pairs(_e2m1(v.view(w.shape)))
        else:  # int4: unsigned codes with zero point 8, a 16-bit scale per 128
            g = w.view(w.shape[0], N, K // 128, 128)
            s = (g.abs().amax(-1) / 7.0).to(_dtype(case))
            q = torch.round(g / s.float().unsqueeze(-1)).clamp(-8, 7) + 8
            q = _pairs(q.to(torch.uint8).view(w.shape))
        ws.append(q)
        ss.append(s)
    q = torch.cat(ws)
    return q.view(torch.float4_e2m1fn_x2) if recipe == "mxfp4" else q, torch.cat(ss)


def _weights(case, seed):
    H, I, _, El, _, _, _, bias, _ = _sizes(case)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(1000003 * seed + 1)
    w13, s13 = _matrices(case, gen, El, 2 * I, H)
    w2, s2 = _matrices(case, gen, El, H, I)
    b13 = b2 = None
    if bias:
        b13 = torch.randn(El, 2 * I, generator=gen, device=DEV, dtype=_dtype(case)) * 0.01
        b2 = torch.randn(El, H, generator=gen, device=DEV, dtype=_dtype(case)) * 0.01
    return w13, s13, b13, w2, s2, b2


def _tokens(case, seed):
    """Activations, router logits (skewed towards some experts where the shape says so), correction bias."""
    H, _, E, _, _, router, _, _, tau = _sizes(case)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(1000003 * seed + 2)
    T = case["tokens"]
    x = torch.randn(T, H, generator=gen, device=DEV).to(_dtype(case))
    logits = torch.randn(T, E, generator=gen, device=DEV)
    if tau:
        rank = torch.randperm(E, generator=gen, device=DEV) + 1
        logits += tau * torch.log_softmax(-1.1 * torch.log(rank.float()), 0)
    corr = torch.randn(E, generator=gen, device=DEV) * 0.01 if router == "grouped" else None
    return x, logits, corr


def _quant_rows(x):
    """e4m3 with a scale per 1 x 128, as a dispatch between ranks sends the tokens."""
    g = x.float().view(x.shape[0], -1, 128)
    s = (g.abs().amax(-1) / 448.0).clamp(min=1.0 / (448.0 * 512.0))
    return (g / s.unsqueeze(-1)).clamp(-448, 448).view(x.shape).to(torch.float8_e4m3fn), s


def prepare(case, seed):
    from vllm_xpu_kernels.fused_moe_interface import XpuFusedMoe
    _, _, _, El, k, _, act, _, _ = _sizes(case)
    w13, s13, b13, w2, s2, b2 = _weights(case, seed)
    moe = XpuFusedMoe(w13, s13, b13, w2, s2, b2, k, act, El, ep_rank=case["ep"] // 2,
                      ep_size=case["ep"])
    x, logits, corr = _tokens(case, seed)
    state = {"case": case, "moe": moe, "x": x, "logits": logits, "corr": corr, "scale": None,
             "out_dtype": x.dtype}
    if case["prequant"]:
        state["x"], state["scale"] = _quant_rows(x)
    return state


def run(state):
    from vllm_xpu_kernels import ops
    case, x = state["case"], state["x"]
    k = SHAPES[case["shape"]][3]
    if state["corr"] is None:
        w, ids, _ = ops.topk_softmax(state["logits"], k, True)
    else:
        w, ids = ops.fused_grouped_topk(state["logits"], k, True, state["corr"], GROUPS,
                                        TOP_GROUPS, "sigmoid", ROUTED_SCALE)
    out = torch.empty(x.shape, dtype=state["out_dtype"], device=x.device)
    state["moe"].apply(out, x, w, ids, a1q_scale=state["scale"])
    return {"out": out, "weights": w, "ids": ids}


def work(case):
    """Weights of the experts that a uniform router reaches, tokens and logits read once, the output and the
    routing written once; two multiplications and additions per weight and routed token."""
    H, I, E, El, k, _, _, bias, _ = _sizes(case)
    T = case["tokens"]
    active = El * (1.0 - (1.0 - k / E) ** T)
    n = 3 * H * I
    per = {"bf16": 2 * n, "fp8block": n + n / 4096, "fp8": n, "mxfp8": n + n / 32,
           "mxfp4": n / 2 + n / 32, "int4": n / 2 + 2 * n / 128}[case["recipe"]]
    per += 2 * (2 * I + H) if bias else 0
    row_in = H + H / 32 if case["prequant"] else 2 * H
    return {"bytes": active * per + T * (row_in + 2 * H + 4 * E + 8 * k),
            "flops": 6.0 * T * k / case["ep"] * H * I}


def tolerance(case):
    """16-bit outputs of fp32 sums, rounded to 16 bits twice on the way (w13's output, the activation): sums in
    another order measured 1e-4 apart.  The fp8 recipes round the activation between the two products to e4m3
    again, so that another order moves some values by one of its steps (1/16): 8e-4 apart."""
    if case["recipe"] in ("fp8block", "mxfp8"):
        return {"rel": 1e-2}
    return {"rel": 1e-3 if case["dtype"] == "fp16" else 5e-3}


# ------------------------------------------------------- the same in 64 bits

def _e4m3(v):
    return v.clamp(-448, 448).float().to(torch.float8_e4m3fn).double()


def _between(recipe, a):
    """The quantisation that the recipe applies to a GEMM's input, and its value."""
    if recipe == "fp8block":
        g = a.view(a.shape[0], -1, 128)
        s = (g.abs().amax(-1, keepdim=True) / 448.0).clamp(min=1.0 / (448.0 * 512.0))
        return (_e4m3(g / s) * s).view(a.shape)
    if recipe == "mxfp8":
        g = a.view(a.shape[0], -1, 32)
        s = torch.exp2(torch.ceil(torch.log2(g.abs().amax(-1, keepdim=True).clamp(min=1e-10) / 448.0)))
        return (_e4m3(g / s) * s).view(a.shape)
    return a


def _value(case, q, s, K):
    """One expert's weight [N, K] in 64 bits."""
    recipe = case["recipe"]
    if recipe == "bf16":
        return q.double().t()
    if recipe == "fp8":
        return q.double().t() * s.double()
    if recipe == "mxfp8":
        return (q.double().t().reshape(-1, K // 32, 32) *
                torch.exp2(s.double().t() - 127).unsqueeze(-1)).reshape(-1, K)
    if recipe == "fp8block":
        return q.double() * s.double().repeat_interleave(128, 0).repeat_interleave(128, 1)
    u = q.view(torch.uint8)
    c = torch.stack((u & 15, u >> 4), -1).view(u.shape[0], K)
    if recipe == "int4":
        return (c.double() - 8) * s.double().repeat_interleave(K // s.shape[1], 1)
    grid = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6], dtype=torch.float64, device=u.device)
    v = torch.where(c > 7, -grid[(c & 7).long()], grid[(c & 7).long()])
    return v * torch.exp2(s.double() - 127).repeat_interleave(32, 1)


def exact(case, seed):
    H, I, E, El, k, router, act, _, _ = _sizes(case)
    w13, s13, b13, w2, s2, b2 = _weights(case, seed)
    x, logits, corr = _tokens(case, seed)
    T = case["tokens"]
    if router == "softmax":
        w, ids = torch.softmax(logits.double(), -1).topk(k, -1)
        w = w / w.sum(-1, keepdim=True)
    else:
        score = torch.sigmoid(logits.double())
        pick = score + corr.double()
        groups = pick.view(T, GROUPS, -1).topk(2, -1).values.sum(-1).topk(TOP_GROUPS, -1).indices
        keep = torch.zeros(T, GROUPS, dtype=torch.bool, device=DEV).scatter_(1, groups, True)
        ids = pick.masked_fill(~keep.repeat_interleave(E // GROUPS, 1), -math.inf).topk(k, -1).indices
        w = score.gather(1, ids)
        w = w / w.sum(-1, keepdim=True) * ROUTED_SCALE
    if case["prequant"]:
        q, s = _quant_rows(x)
        a = (q.double().view(T, -1, 128) * s.double().unsqueeze(-1)).view(T, H)
    else:
        a = _between(case["recipe"], x.double())
    out = torch.zeros(T, H, dtype=torch.float64, device=DEV)
    first = case["ep"] // 2 * El
    for e in range(El):
        t, j = (ids == first + e).nonzero(as_tuple=True)
        if not t.numel():
            continue
        g = a[t] @ _value(case, w13[e], None if s13 is None else s13[e], H).t()
        g = g if b13 is None else g + b13[e].double()
        if act == "swigluoai":
            gate, up = g[:, 0::2].clamp(max=7.0), g[:, 1::2].clamp(-7.0, 7.0)
            g = (up + 1) * gate * torch.sigmoid(1.702 * gate)
        else:
            g = torch.nn.functional.silu(g[:, :I]) * g[:, I:]
        y = _between(case["recipe"], g.contiguous()) @ _value(case, w2[e], None if s2 is None else s2[e], I).t()
        y = y if b2 is None else y + b2[e].double()
        out.index_add_(0, t, y * w[t, j].unsqueeze(1))
    return {"out": out, "weights": w, "ids": None}
