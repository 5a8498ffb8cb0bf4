"""MXFP4 on the prefill kernels that convert in registers: every tile height,
row-major and tiled weights, scale bytes in 16-byte pieces (reductions of a
multiple of four groups) and one by one, split reductions, SwiGLU with biases,
scale bytes 0 and 255, against the oracle and the streaming kernels."""

import pytest
import torch

from flaggems_sglang import _lib
from flaggems_sglang import quant as Q
from oracle import fused_moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _ids(counts, k=2):
    flat = torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts))
    return flat.view(k, -1).t().contiguous().to(torch.int32)


def _rel(a, b):
    # exact weights on both sides: rows differ by bf16 rounding flips only
    return float(((a - b).norm(dim=1) / b.norm(dim=1).clamp_min(1e-20)).max())


def _problem(counts, K, N, seed=0):
    ids = _ids(counts)
    d = O.make_inputs(ids.shape[0], K, N, len(counts), 2, wscale=0.05, seed=seed)
    return d, ids, Q.quantize_mxfp4(d["w13"]), Q.quantize_mxfp4(d["w2"])


COUNTS = {32: [33, 31, 1, 33, 32, 0, 30, 16], 64: [65, 1, 64, 63, 0, 33, 64, 62],
          128: [129, 127, 1, 128, 0, 130, 100, 65]}


@pytest.mark.parametrize("K,N", [(128, 7168), (512, 7296), (640, 7168), (384, 8192)])
@pytest.mark.parametrize("bm", sorted(COUNTS))
def test_heights(bm, K, N):
    import flaggems_sglang

    d, ids, (q1, s1), (q2, s2) = _problem(COUNTS[bm], K, N)
    M = ids.shape[0]
    assert _lib.lib().fmoe_fused_block_m(_lib.W_MXFP4, M, 2, 8, 0, K, N) == bm
    assert _lib.lib().fmoe_fused_block_m(_lib.W_MXFP4_TILED, M, 2, 8, 0, K, N) == bm

    def call(tiled, path):
        a, b = q1.to(DEV), q2.to(DEV)
        if tiled:
            a, b = Q.tile_mxfp4(a), Q.tile_mxfp4(b)
        return flaggems_sglang.fused_experts(
            d["x"].to(DEV), a, b, d["topk_weights"].to(DEV), ids.to(DEV), path=path, use_mxfp4_w4a16=True,
            w1_scale=s1.to(DEV), w2_scale=s2.to(DEV)).float().cpu()

    out = call(False, 0)
    assert torch.equal(out, call(True, 0))  # the layout changes addresses only
    assert _rel(out, call(True, 2)) < 1e-2
    ref = O.fused_experts_mxfp4(d["x"], q1, s1, q2, s2, d["topk_weights"], ids).float()
    assert _rel(out, ref) < 1e-2


@pytest.mark.parametrize("bm", sorted(COUNTS))
def test_bias_swiglu(bm):
    """The bias entry at each height that the rule picks."""
    import flaggems_sglang
    from types import SimpleNamespace

    K, N = 256, 7168
    d, ids, (q1, s1), (q2, s2) = _problem(COUNTS[bm], K, N, seed=3)
    g = torch.Generator().manual_seed(4)
    b13, b2 = torch.randn(8, 2 * N, generator=g) * 0.1, torch.randn(8, K, generator=g) * 0.1
    tw = d["topk_weights"].to(DEV)
    rd, gi, si = flaggems_sglang.ops.fused_moe._standard_topk_to_triton_kernels(tw, ids.to(DEV), 8)
    pc = [SimpleNamespace(weight_scale=s.to(DEV).transpose(1, 2)) for s in (s1, s2)]
    out = flaggems_sglang.triton_kernel_fused_experts_with_bias(
        d["x"].to(DEV), q1.to(DEV).transpose(1, 2), pc[0], b13.to(DEV), q2.to(DEV).transpose(1, 2), pc[1],
        b2.to(DEV), rd, gi, si, gemm1_alpha=1.702, gemm1_clamp_limit=7.0).float().cpu()
    assert bm in rd.expt_data.block_pid_map
    ref = O.fused_experts_bias(d["x"], O.mxfp4_dequant(q1, s1), b13, O.mxfp4_dequant(q2, s2), b2,
                               d["topk_weights"], ids, alpha=1.702, limit=7.0).float()
    assert _rel(out, ref) < 1e-2


@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("bm,counts", [(32, [17, 1, 32, 2]), (64, [33, 65, 1, 33]), (128, [129, 3, 66, 2])])
def test_split_inside_a_scale_piece(bm, counts, tiled):
    """GEMM2 reductions of 20 groups in two parts: the second starts at group 10,
    inside a 16-byte piece of scale bytes (groups 8 to 11)."""
    import ctypes

    import flaggems_sglang

    K, N, E = 256, 2560, 24
    d, ids, (q1, s1), (q2, s2) = _problem(counts * 6, K, N, seed=7)
    M = ids.shape[0]
    L, wt = _lib.lib(), _lib.W_MXFP4_TILED if tiled else _lib.W_MXFP4
    assert L.fmoe_fused_block_m(wt, M, 2, E, 0, K, N) == bm
    r = _lib.Routing(None, None, None, None, None, None, None, M, 2, E, bm, L.fmoe_max_tiles(2 * M, E))
    assert L.fmoe_gemm2_splits(wt, K, N, ctypes.byref(r), 0) == 2
    a, b = q1.to(DEV), q2.to(DEV)
    if tiled:
        a, b = Q.tile_mxfp4(a), Q.tile_mxfp4(b)
    out = flaggems_sglang.fused_experts(d["x"].to(DEV), a, b, d["topk_weights"].to(DEV), ids.to(DEV),
                                        use_mxfp4_w4a16=True, w1_scale=s1.to(DEV), w2_scale=s2.to(DEV)).float().cpu()
    assert _rel(out, O.fused_experts_mxfp4(d["x"], q1, s1, q2, s2, d["topk_weights"], ids).float()) < 1e-2


def test_scale_bytes_0_and_255():
    """2^-127 and NaN scales: the outputs of the streaming kernels, NaN for NaN."""
    import flaggems_sglang

    d, ids, (q1, s1), (q2, s2) = _problem(COUNTS[32], 512, 7168, seed=5)
    s1 = s1.clone()
    s1[0] = 0       # expert 0: gate and up vanish
    s2 = s2.clone()
    s2[3, 5, 2] = 255  # expert 3: one NaN block in output column 5
    args = (d["x"].to(DEV), q1.to(DEV), q2.to(DEV), d["topk_weights"].to(DEV), ids.to(DEV))
    kw = dict(use_mxfp4_w4a16=True, w1_scale=s1.to(DEV), w2_scale=s2.to(DEV))
    out = flaggems_sglang.fused_experts(*args, **kw).float().cpu()
    dec = flaggems_sglang.fused_experts(*args, path=2, **kw).float().cpu()
    assert torch.equal(out.isnan(), dec.isnan()) and out.isnan().any()
    assert _rel(out.nan_to_num(0.0), dec.nan_to_num(0.0)) < 1e-2


@pytest.mark.parametrize("M", [0, 1, 5, 40, 300, 520])
@pytest.mark.parametrize("on_input,rsf", [(False, None), (True, 2.5)])
def test_hook_one_call_equals_stages(M, on_input, rsf):
    """The hook's MXFP4 bias layer (one C call up to 255 slots per expert: streaming
    to M=40, 128-row tiles at M=300; the stages above) against the bias entry on
    prepared routing, bit-identical, and against the oracle."""
    from types import SimpleNamespace

    import flaggems_sglang
    from flaggems_sglang.ops import fused_moe as F

    K, N, E, k = 256, 3328, 4, 2
    assert _lib.lib().fmoe_fused_block_m(_lib.W_MXFP4, M, k, E, 0, K, N) == (128 if M >= 300 else 16)
    d = O.make_inputs(max(M, 1), K, N, E, k, wscale=0.05)
    x, tw, ti = (d[n][:M].to(DEV) for n in ("x", "topk_weights", "topk_ids"))
    (q1, s1), (q2, s2) = Q.quantize_mxfp4(d["w13"].to(DEV)), Q.quantize_mxfp4(d["w2"].to(DEV))
    g = torch.Generator().manual_seed(9)
    b13, b2 = (torch.randn(E, n, generator=g).mul(0.1).to(DEV) for n in (2 * N, K))
    layer = torch.nn.Module()
    for name, t in (("w13_weight", q1), ("w13_weight_scale", s1), ("w2_weight", q2), ("w2_weight_scale", s2),
                    ("w13_weight_bias", b13), ("w2_weight_bias", b2)):
        layer.register_parameter(name, torch.nn.Parameter(t, requires_grad=False))
    cfg = SimpleNamespace(num_experts=E, no_combine=False, activation="silu", apply_router_weight_on_input=on_input,
                          routed_scaling_factor=rsf, gemm1_alpha=1.702, gemm1_clamp_limit=7.0)
    out = F.fused_moe_flagos(SimpleNamespace(runner=SimpleNamespace(config=cfg)), layer, SimpleNamespace(
        hidden_states=x, topk_output=SimpleNamespace(topk_weights=tw, topk_ids=ti))).hidden_states
    if M == 0:
        assert out.shape == (0, K)
        return
    rd, gi, si = F._standard_topk_to_triton_kernels(tw, ti, E)
    pc = [SimpleNamespace(weight_scale=s.transpose(1, 2)) for s in (s1, s2)]
    ref = flaggems_sglang.triton_kernel_fused_experts_with_bias(
        x, q1.transpose(1, 2), pc[0], b13, q2.transpose(1, 2), pc[1], b2, rd, gi, si,
        apply_router_weight_on_input=on_input, gemm1_alpha=1.702, gemm1_clamp_limit=7.0)
    if rsf is not None:
        ref.mul_(rsf)
    assert torch.equal(out, ref)
    orc = O.fused_experts_bias(x.cpu(), O.mxfp4_dequant(q1.cpu(), s1.cpu()), b13.cpu(),
                               O.mxfp4_dequant(q2.cpu(), s2.cpu()), b2.cpu(), tw.cpu(), ti.cpu(), alpha=1.702, limit=7.0,
                               apply_router_weight_on_input=on_input).float()
    assert _rel(out.float().cpu(), orc * (1.0 if rsf is None else rsf)) < 1e-2


def test_unaligned_scales():
    """Scale bytes that do not start at a multiple of 16 (a view into a larger
    buffer): the streaming kernels' result, whole call, bias entry and per-slot rows."""
    from types import SimpleNamespace

    import flaggems_sglang

    d, ids, (q1, s1), (q2, s2) = _problem(COUNTS[32], 512, 7168, seed=6)

    def view(s, off):
        buf = torch.empty(s.numel() + 16, dtype=torch.uint8, device=DEV)
        v = buf[off:off + s.numel()].view(s.shape)
        assert v.data_ptr() % 16 == off
        return v.copy_(s)

    x, a, b, tw, ti = d["x"].to(DEV), q1.to(DEV), q2.to(DEV), d["topk_weights"].to(DEV), ids.to(DEV)
    z13, z2 = torch.zeros(8, 2 * 7168, device=DEV), torch.zeros(8, 512, device=DEV)

    def calls(off, path):
        kw = dict(use_mxfp4_w4a16=True, w1_scale=view(s1, off), w2_scale=view(s2, off), path=path)
        rd, gi, si = flaggems_sglang.ops.fused_moe._standard_topk_to_triton_kernels(tw, ti, 8)
        pc = [SimpleNamespace(weight_scale=kw[n].transpose(1, 2)) for n in ("w1_scale", "w2_scale")]
        bias = flaggems_sglang.triton_kernel_fused_experts_with_bias(
            x, a.transpose(1, 2), pc[0], z13, b.transpose(1, 2), pc[1], z2, rd, gi, si)
        return (flaggems_sglang.fused_experts(x, a, b, tw, ti, **kw),
                flaggems_sglang.fused_experts(x, a, b, tw, ti, no_combine=True, **kw), bias)

    odd, even = calls(1, 0), calls(0, 2)
    for o, e in zip(odd[:2], even[:2]):
        assert torch.equal(o, e)
    assert _rel(odd[2].float().cpu(), calls(0, 0)[2].float().cpu()) < 1e-2
