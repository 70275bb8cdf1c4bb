"""GPU parity of the 320-slot e4m3 / e2m1 kernel (moe_gemm_wide8p.hip) with
the valid slot tiles of a block split over two wave halves: every count of
tiles per half from 1 to 10, at the edges of the 16-slot tiles and of the
halves, over one, two and three K stages (the two weight slots in turn).

Bars: grouped GEMM, a bf16 output's rounding (2^-8 of it) twice over plus the
fp32 accumulation of K <= 384 products: rtol = atol = 1e-2; layers, which
re-quantise the activation between the GEMMs, the bar of
test_gpu_layer_cases.py."""
import pytest
import torch

from oracle import moe_oracle as O
from test_gpu_layer_cases import _close_fp8, _layer_cls, _W

pytestmark = pytest.mark.gpu

# rows per expert: 1..10 tiles per half with their last tile full, short of
# one row and holding one row; 321 leaves a block of one row
ROWS = [1, 16, 17, 33, 64, 65, 96, 97, 128, 129, 161, 192, 193, 224, 225, 256, 257, 288, 289,
        319, 320, 321]


@pytest.mark.parametrize("K", [128, 256, 384])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_grouped_gemm_tiles_per_half(dev, K, dt):
    from vllm_xpu_kernels import ops
    print(f"wide8p: K={K} {dt}", flush=True)
    g = torch.Generator().manual_seed(K)
    E, M, N = len(ROWS), sum(ROWS), 384
    a = torch.randn(M, K, generator=g).to(dt)
    q, s = O.fp8_block_quant_weight(torch.randn(E, N, K, generator=g) * 0.02)
    d = torch.empty(M, N, dtype=dt, device=dev)
    ops.cutlass_grouped_gemm(a.to(dev), q.to(dev), s.to(dev), None, d,
                             torch.tensor(ROWS, dtype=torch.int32, device=dev), N, K, E)
    ref = O.grouped_gemm("fp8block", a, q, s, None, ROWS)
    torch.testing.assert_close(d.cpu().float(), ref.float(), rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("recipe", ["fp8block", "mxfp8", "mxfp4"])
def test_layer_tiles_per_half(dev, recipe):
    """Both epilogues; mxfp4 with e2m1 tokens, K and N with a tail of half a
    256-value stage."""
    print(f"wide8p layer: {recipe}", flush=True)
    W = _W()
    g = torch.Generator().manual_seed(5)
    E, T, H, I = len(ROWS), sum(ROWS), 384, 384
    w13 = torch.randn(E, 2 * I, H, generator=g) / 16
    w2 = torch.randn(E, H, I, generator=g) / 16
    quant = {"fp8block": W.fp8_block_quant, "mxfp8": W.mxfp8_quant, "mxfp4": W.mxfp4_quant}[recipe]
    (q13, s13), (q2, s2) = quant(w13), quant(w2)
    lay = ora = (q13, s13, None, q2, s2, None)
    if recipe == "mxfp8":
        lay = tuple(None if t is None else t.transpose(1, 2).contiguous() for t in ora)
    elif recipe == "mxfp4":
        lay = (q13.view(torch.float4_e2m1fn_x2), s13, None, q2.view(torch.float4_e2m1fn_x2), s2,
               None)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(ROWS))
    ti = ids[torch.randperm(T, generator=g)].view(T, 1)
    tw = torch.rand(T, 1, generator=g)
    x, xs = torch.randn(T, H, generator=g).to(torch.bfloat16) / 4, None
    moe = _layer_cls()(*[None if t is None else t.to(dev) for t in lay], 1, "silu", E)
    out = torch.empty(T, H, dtype=torch.bfloat16, device=dev)
    if recipe == "mxfp4":
        x, xs = O.to_mxfp4(x.float())
        moe.apply(out, x.to(dev).view(torch.float4_e2m1fn_x2), tw.to(dev), ti.to(dev),
                  a1q_scale=xs.to(dev))
    else:
        moe.apply(out, x.to(dev), tw.to(dev), ti.to(dev))
    ref = O.fused_moe(recipe, x, *ora, tw, ti, a1q_scale=xs)
    _close_fp8(out.cpu(), ref)


def test_layer_in_short_scratch(dev):
    """56 slots per expert: 320-slot blocks pad the activation beyond the
    static 64 MiB scratch of the allocation-free entry, which then runs
    64-slot blocks; both against each other to the fp8 layer bar."""
    import ctypes
    import dataclasses

    from vllm_xpu_kernels import capi
    from vllm_xpu_kernels import workloads as W
    cfg, T = dataclasses.replace(W.config("C2"), recipe="fp8block"), 900
    print(f"wide8p short scratch: {cfg.name} {cfg.recipe} T={T}", flush=True)
    w = W.make_weights(cfg, dev)
    moe = _layer_cls()(*w.layer_args(), cfg.topk, cfg.activation, cfg.experts)
    x = W.make_activations(cfg, T, dev, seed=3)
    tw, ti = W.route(cfg, W.make_router_logits(cfg, T, dev, seed=4), None)
    ref, out = torch.empty_like(x), torch.full_like(x, float("nan"))
    moe.apply(ref, x, tw, ti)
    a = capi.fused_args(moe, out, x, tw, ti)
    assert capi.workspace_for(a, dev).numel() > 64 << 20
    capi.lib.mi355moe_fused_moe_noalloc.argtypes = [ctypes.POINTER(capi.FusedMoeArgs),
                                                    ctypes.c_void_p]
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = capi.lib.mi355moe_fused_moe_noalloc(ctypes.byref(a), stream)
    assert rc == 0, capi.lib.mi355moe_last_error()
    _close_fp8(out.cpu(), ref.cpu())
