"""GPU parity of the SMALL family (moe_gemm_mid.hip) against the oracle at the
edges of its blocks and of its operands: 16- to 128-slot blocks filled to one
slot, to one less and one more than a tile, K that ends inside a 128-value
stage, column remainders, row-major and K-blocked weights, every int4 group
size, scales on addresses that do not allow whole-word loads.

Bars: the 16-bit type's rounding of an output (bf16 2^-8, fp16 2^-11 of it)
twice over, plus the fp32 accumulation of K <= 512 products: rtol = atol =
1e-2; layers the bar of test_gpu_gemm_fused.py."""
import dataclasses

import pytest
import torch

from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu

# rows per expert: averages (per active expert) of 6, 18, 43, 70 and 99, which take
# blocks of 16, 32, 64, 96 and 128 slots where the recipe has them
ROWS = [[17, 0, 3], [16, 33, 5], [64, 65, 1], [95, 97, 20], [128, 129, 40]]


def _int4(w, group, dt):
    """[N, K] -> two's-complement nibbles [N, K/2], scales [N, K/group], value."""
    N, K = w.shape
    s = (w.view(N, K // group, group).abs().amax(-1) / 7).to(dt)
    v = torch.round(w / s.float().repeat_interleave(group, 1)).clamp(-8, 7)
    c = (v.to(torch.int32) & 15).to(torch.uint8)
    return c[:, 0::2] | (c[:, 1::2] << 4), s, (v * s.float().repeat_interleave(group, 1)).to(dt)


@pytest.mark.parametrize("rows", ROWS, ids=lambda r: "-".join(map(str, r)))
@pytest.mark.parametrize("recipe,N,K,dt", [
    ("bf16", 72, 136, torch.bfloat16), ("bf16", 264, 512, torch.float16),
    ("fp8block", 256, 384, torch.bfloat16), ("mxfp4", 72, 160, torch.float16),
    ("mxfp4", 264, 256, torch.bfloat16), ("fp8", 72, 160, torch.bfloat16),
    ("int4-32", 72, 160, torch.bfloat16), ("int4-64", 264, 192, torch.float16),
    ("int4-128", 72, 256, torch.float16), ("int4-256", 72, 512, torch.bfloat16)])
def test_grouped_gemm_small_blocks(dev, recipe, N, K, dt, rows):
    from vllm_xpu_kernels import ops
    print(f"small blocks: {recipe} N={N} K={K} {dt} rows={rows}", flush=True)
    g = torch.Generator().manual_seed(N + K)
    E, M = len(rows), sum(rows)
    a = torch.randn(M, K, generator=g).to(dt)
    w = torch.randn(E, N, K, generator=g) * 0.05
    rpe = torch.tensor(rows, dtype=torch.int32, device=dev)
    d = torch.empty(M, N, dtype=dt, device=dev)
    if recipe == "bf16":
        w = w.to(dt)
        b, s, val = w.transpose(1, 2).contiguous(), None, w.float()
    elif recipe == "fp8block":
        b, s = O.fp8_block_quant_weight(w)
        val = None
    elif recipe == "fp8":
        s = w.abs().amax((1, 2)) / 448
        q = (w / s[:, None, None]).to(torch.float8_e4m3fn)
        b, val = q.transpose(1, 2).contiguous(), q.float() * s[:, None, None]
    elif recipe == "mxfp4":
        q, s = zip(*(O.to_mxfp4(w[e]) for e in range(E)))
        b, s = torch.stack(q), torch.stack(s)
        val = torch.stack([O.dequant_mxfp4(b[e], s[e]) for e in range(E)])
    else:
        q, s, val = (torch.stack(t) for t in zip(*(_int4(w[e], int(recipe[5:]), dt) for e in range(E))))
        b, val = q.view(torch.int8), val.float()
    ops.cutlass_grouped_gemm(a.to(dev), b.to(dev), None if s is None else s.to(dev), None, d, rpe,
                             N, K, E)
    if val is None:
        ref = O.grouped_gemm("fp8block", a, b, s, None, rows).float()
    else:
        ref = torch.cat([a[sum(rows[:e]):sum(rows[:e + 1])].float() @ val[e].t() for e in range(E)])
    torch.testing.assert_close(d.cpu().float(), ref, rtol=1e-2, atol=1e-2)


def _layer_ref(cfg, w, x, tw, ti, dt):
    """The layer's oracle on the reference-layout weights."""
    act = cfg.activation
    c = lambda t: None if t is None else t.cpu()  # noqa: E731
    if cfg.recipe == "int4":
        deq = lambda q, s: torch.stack([  # noqa: E731
            ((torch.stack((q[e] & 15, q[e] >> 4), -1).view(q.shape[1], -1).float() - 8) *
             s[e].float().repeat_interleave(128, 1)).to(dt) for e in range(q.shape[0])])
        return O.fused_moe("bf16", x, deq(w[0].cpu(), w[1].cpu()), None, None,
                           deq(w[3].cpu(), w[4].cpu()), None, None, tw, ti, activation=act)
    return O.fused_moe(cfg.recipe, x, w[0].cpu().view(torch.uint8), c(w[1]), c(w[2]),
                       w[3].cpu().view(torch.uint8), c(w[4]), c(w[5]), tw, ti, activation=act)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("T", [5, 12, 30, 50])
@pytest.mark.parametrize("recipe,dt", [("mxfp4", torch.bfloat16), ("int4", torch.float16),
                                       ("int4", torch.bfloat16)])
def test_layer_packed_weights_scale_alignment(dev, recipe, dt, T, offset):
    """K-blocked 4-bit layers (blocks of 16 to 64 slots) with the scales at an
    aligned address and one element past it, prepared in place."""
    from vllm_xpu_kernels import workloads as W
    from vllm_xpu_kernels.fused_moe_interface import XpuFusedMoe
    print(f"scale alignment: {recipe} {dt} T={T} offset={offset}", flush=True)
    cfg = dataclasses.replace(W.config("C5" if recipe == "mxfp4" else "C2"), recipe=recipe,
                              hidden=256, inter=384, experts=4, topk=4 if T > 30 else 2)
    m = W.make_weights(cfg, dev)
    args = list(m.layer_args(copy=True))
    if recipe == "int4":
        args[1], args[4] = args[1].to(dt), args[4].to(dt)
    ref_args = [None if t is None else t.clone() for t in args]
    for i in (1, 4):
        flat = torch.empty(args[i].numel() + offset, dtype=args[i].dtype, device=dev)
        flat[offset:] = args[i].reshape(-1)
        args[i] = flat[offset:].view(args[i].shape)
    moe = XpuFusedMoe(*args, cfg.topk, cfg.activation, cfg.experts)
    x = W.make_activations(cfg, T, dev).to(dt)
    tw, ti = W.route(cfg, W.make_router_logits(cfg, T, dev))
    out = torch.empty_like(x)
    moe.apply(out, x, tw, ti)
    ref = _layer_ref(cfg, ref_args, x.cpu(), tw.cpu(), ti.cpu(), dt)
    torch.testing.assert_close(out.cpu().float(), ref.float(), rtol=2e-2, atol=2e-2)


def test_noalloc_takes_smaller_blocks(dev):
    """A layer whose preferred 32-slot blocks pad its activation beyond the
    static scratch (93 MB) runs 16-slot blocks there (60 MB), bit-identical
    to the caller-workspace entry's 32-slot blocks."""
    from test_zz_no_alloc import _run_pair
    from vllm_xpu_kernels import workloads as W
    from vllm_xpu_kernels.fused_moe_interface import XpuFusedMoe
    cfg = dataclasses.replace(W.config("C2"), hidden=256, inter=4096, experts=256)
    w = W.make_weights(cfg, dev)
    moe = XpuFusedMoe(*w.layer_args(), cfg.topk, cfg.activation, cfg.experts)
    _run_pair(cfg, 400, dev, moe, w, seed=3)
