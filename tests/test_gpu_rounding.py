"""fp32 -> bf16 rounding of the result rows on the GPU: every exponent with the
mantissas around the rounding midpoint, both signs, denormals, infinities and
NaN, through the top-k sum of one slot per token, against torch's conversion
(bit for bit; a NaN stays a NaN).  And the SiLU quotient at the ends of its
range through the stage-level GEMM1."""

import pytest
import torch

from flaggems_sglang import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


def test_moe_sum_rounds_as_torch():
    exps = torch.arange(256, dtype=torch.int64).view(-1, 1, 1) << 23
    man = torch.tensor([0, 1, 0x7fff, 0x8000, 0x8001, 0xffff, 0x10000, 0x17fff, 0x18000, 0x18001,
                        0x7effff, 0x7f7fff, 0x7f8000, 0x7f8001, 0x7fffff, 0x400000]).view(1, -1, 1)
    sign = (torch.arange(2, dtype=torch.int64) << 31).view(1, 1, -1)
    bits = (exps | man | sign).reshape(-1)
    y = torch.where(bits >= 2 ** 31, bits - 2 ** 32, bits).to(torch.int32).view(torch.float32)
    K = 64
    y = y.view(-1, K).to(DEV)
    M = y.shape[0]
    gi = torch.arange(M, dtype=torch.int32, device=DEV)
    out = torch.empty(M, K, dtype=torch.bfloat16, device=DEV)
    _lib.check(_lib.lib().fmoe_moe_sum(y.data_ptr(), 1, gi.data_ptr(), M, 1, K, 1.0, out.data_ptr(),
                                       _lib.stream_of(y)), "moe_sum")
    ref = (y + 0.0).to(torch.bfloat16)  # the sum starts from +0
    nan = ref.isnan()
    assert torch.equal(out.isnan(), nan)
    assert torch.equal(out[~nan].view(torch.int16), ref[~nan].view(torch.int16))


@pytest.mark.parametrize("M", [16, 406])  # the streaming kernels; 256-row tiles
def test_silu_quotient_range(M):
    """Gates from far below exp's overflow (quotient -0) to far above (the
    gate itself), up = 1: one expert whose gate rows pick x's first element."""
    import flaggems_sglang

    K = N = 128
    gates = torch.cat([torch.linspace(-130, 130, 261), torch.linspace(-9, 9, 145)])
    x = torch.zeros(M, K)
    x[:, 0] = gates[:: gates.numel() // M][:M]
    x[:, 1] = 1.0
    x = x.to(torch.bfloat16)
    w13 = torch.zeros(1, 2 * N, K)
    w13[:, :N, 0] = 1.0   # gate = x[0]
    w13[:, N:, 1] = 1.0   # up = x[1] = 1
    w2 = torch.eye(K).view(1, K, N)
    out = flaggems_sglang.fused_experts(
        x.to(DEV), w13.to(torch.bfloat16).to(DEV), w2.to(torch.bfloat16).to(DEV),
        torch.ones(M, 1, device=DEV), torch.zeros(M, 1, dtype=torch.int32, device=DEV))
    g = x[:, :1].double()
    ref = (g / (1.0 + torch.exp(-g))).float()
    # one bf16 rounding (half an ulp: 2^-8 of the value); __expf's relative error grows with |g| (below
    # 130 * 2^-24 + 2^-22, far under 2^-12); quotients below 1e-35 may flush
    torch.testing.assert_close(out.float().cpu(), ref.expand(M, K), rtol=2.0 ** -8 + 2.0 ** -12, atol=1e-35)


@pytest.mark.parametrize("act", ["silu", "swiglu"])
@pytest.mark.parametrize("M", [16, 406])  # the streaming kernels; 256-row tiles
def test_small_quotients_survive(act, M):
    """Gates whose sigmoid denominator lies above 2^126, where its reciprocal is
    denormal: the quotient (about 1e-37) is a normal number, and a large up
    value makes it visible in the output."""
    import ctypes

    K = N = 128
    g = torch.tensor([-88.5, -88.0, -87.5, -87.0, -86.5, -86.0, -85.0, -80.0]).repeat(-(-M // 8))[:M]
    x = torch.zeros(M, K)
    x[:, 0], x[:, 1] = g, 2.0 ** 60
    w13 = torch.zeros(1, 2 * N, K)
    gate, up = (slice(0, N), slice(N, None)) if act == "silu" else (slice(0, None, 2), slice(1, None, 2))
    w13[:, gate, 0], w13[:, up, 1] = 1.0, 2.0 ** 40
    x, w13, w2 = (t.to(torch.bfloat16).to(DEV) for t in (x, w13, torch.eye(K).view(1, K, N)))
    out = torch.empty(M, K, dtype=torch.bfloat16, device=DEV)
    tw, ids = torch.ones(M, 1, device=DEV), torch.zeros(M, 1, dtype=torch.int32, device=DEV)
    a = _lib.FusedArgs()
    a.wtype, a.x, a.M, a.K, a.N, a.E, a.top_k = _lib.W_BF16, x.data_ptr(), M, K, N, 1, 1
    a.w13, a.w2, a.group_size, a.topk_weights, a.topk_ids = w13.data_ptr(), w2.data_ptr(), 128, tw.data_ptr(), ids.data_ptr()
    a.routed_scaling_factor, a.out, a.alpha = 1.0, out.data_ptr(), 1.0
    a.activation = _lib.ACT_SILU if act == "silu" else _lib.ACT_SWIGLU
    n = _lib.lib().fmoe_fused_experts_workspace_bytes(ctypes.byref(a))
    ws = torch.empty(n, dtype=torch.uint8, device=DEV)
    a.workspace, a.workspace_bytes = ws.data_ptr(), n
    _lib.check(_lib.lib().fmoe_fused_experts(ctypes.byref(a), _lib.stream_of(x)), "fused_experts")
    d = g.double().view(-1, 1)
    ref = (d / (1.0 + torch.exp(-d)) * (2.0 ** 100 + (act == "swiglu"))).float()
    # the bound of test_silu_quotient_range, without its absolute part
    torch.testing.assert_close(out.float().cpu(), ref.expand(M, K), rtol=2.0 ** -8 + 2.0 ** -12, atol=0)
