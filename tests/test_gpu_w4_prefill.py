"""int4 batches of 81 to 255 slots per expert (the prefill kernels that unpack
nibbles in registers), against the dequantizing oracle and the streaming
kernels: row-major and tiled weights, reductions of 1 to 5 groups in either
GEMM (fewer and more than the ring's depth), partial and one-row tiles, an
empty expert, a half-filled last output tile, GELU, weight on the input, routed
scaling, an expert map.  Layers are just above the size from which these
kernels run; every call's route is asserted."""

import ctypes

import pytest
import torch

from flaggems_sglang import quant as Q
from oracle import fused_moe_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _ids(counts, k):
    flat = torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts))
    return flat.view(k, -1).t().contiguous().to(torch.int32)


def _unpacks(M, K, N, E, k, n_global=0):
    """Whether a path 0 call leaves the streaming kernels (whose workspace, with
    its split planes and without copies of x, is another)."""
    from flaggems_sglang import _lib

    some = ctypes.create_string_buffer(16)
    a = _lib.FusedArgs()
    a.wtype, a.M, a.K, a.N, a.E, a.top_k, a.group_size = _lib.W_INT4, M, K, N, E, k, 128
    a.x = a.w13 = a.w2 = 4096  # aligned operands (a query without any covers both routes)
    if n_global:
        a.expert_map, a.n_global = ctypes.addressof(some), n_global
    sizes = []
    for a.path in (0, 2):
        sizes.append(_lib.lib().fmoe_fused_experts_workspace_bytes(ctypes.byref(a)))
    return sizes[0] != sizes[1] and M * k < 256 * E


def _run(d, ids, tiled, path, **kw):
    import flaggems_sglang

    if path == 0:
        E, _, K = d["w13"].shape
        assert _unpacks(*ids.shape[:1], K, d["w2"].shape[2], E, ids.shape[1], kw.get("global_num_experts", 0))

    q1, s1, z1 = Q.quantize_int4_group(d["w13"].to(DEV))
    q2, s2, z2 = Q.quantize_int4_group(d["w2"].to(DEV))
    w = (Q.tile_int4(q1), Q.tile_int4(q2)) if tiled else (q1, q2)
    out = flaggems_sglang.fused_experts(d["x"].to(DEV), *w, d["topk_weights"].to(DEV), ids.to(DEV), path=path,
                                        use_int4_w4a16=True, w1_scale=s1, w2_scale=s2, w1_zp=z1, w2_zp=z2, **kw)
    return out.float().cpu(), (q1, s1, z1, q2, s2, z2)


def _rel(a, b):
    # bf16 activations and results: both sides round at the same two points, so
    # rows differ by rounding flips only (2^-9 of a value each); a wrong scale,
    # zero or row shows as tens of percent of the row
    return float(((a - b).norm(dim=1) / b.norm(dim=1).clamp_min(1e-20)).max())


COUNTS = [[129, 129, 257, 1], [128, 0, 256, 128], [100, 155, 85, 100]]


@pytest.mark.parametrize("E,K,N,pattern", [(4, 640, 13184, 0), (4, 640, 13184, 1), (4, 640, 13184, 2), (4, 128, 65664, 0),
                                           (8, 384, 11008, 0), (20, 2688, 640, 0), (20, 2688, 640, 1),
                                           (20, 2688, 640, 2), (33, 2688, 384, 0), (98, 2816, 128, 2)])
def test_matches_oracle(E, K, N, pattern):
    k = 2
    counts = (COUNTS[pattern] * E)[:E]
    counts[0] += sum(counts) % k
    ids = _ids(counts, k)
    d = O.make_inputs(ids.shape[0], K, N, len(counts), k, wscale=0.05)
    ref = None
    for tiled in (False, True):
        out, q = _run(d, ids, tiled, 0)
        if ref is None:
            ref = O.fused_experts_w4a16(d["x"], *[t.cpu() for t in q], d["topk_weights"], ids).float()
            first = out
        assert _rel(out, ref) < 1e-2
        assert torch.equal(out, first)  # the layout changes addresses only
    dec, _ = _run(d, ids, True, 2)
    assert _rel(out, dec) < 1e-2


@pytest.mark.parametrize("kw", [dict(activation="gelu"), dict(apply_router_weight_on_input=True),
                                dict(routed_scaling_factor=2.5)])
def test_options_match_streaming_kernels(kw):
    ids = _ids([130, 90, 200, 60], 2)
    d = O.make_inputs(ids.shape[0], 640, 13184, 4, 2, wscale=0.05)
    out, _ = _run(d, ids, True, 0, **kw)
    dec, _ = _run(d, ids, True, 2, **kw)
    assert _rel(out, dec) < 1e-2


def test_expert_map():
    """8 global experts, 4 of them here: about half of every token's choices drop."""
    ids = _ids([110, 100, 120, 90] * 2, 2)
    emap = torch.tensor([-1, 2, -1, 0, 1, -1, 3, -1], dtype=torch.int32)
    d = O.make_inputs(ids.shape[0], 640, 13184, 4, 2, wscale=0.05)
    kw = dict(expert_map=emap.to(DEV), global_num_experts=8)
    out, _ = _run(d, ids, True, 0, **kw)
    dec, _ = _run(d, ids, True, 2, **kw)
    live = dec.norm(dim=1) > 0
    assert torch.equal(out[~live], dec[~live])
    assert _rel(out[live], dec[live]) < 1e-2


def test_graph_replay_and_tail_split():
    """A reduction long enough for GEMM2's tail split, captured and replayed
    between eager calls: bit-identical every time."""
    ids = _ids([100, 90, 85, 95], 2)
    assert _unpacks(ids.shape[0], 256, 32896, 4, 2)
    d = O.make_inputs(ids.shape[0], 256, 32896, 4, 2, wscale=0.02)
    q1, s1, z1 = Q.quantize_int4_group(d["w13"].to(DEV))
    q2, s2, z2 = Q.quantize_int4_group(d["w2"].to(DEV))
    t1, t2 = Q.tile_int4(q1), Q.tile_int4(q2)
    x, tw, ti = d["x"].to(DEV), d["topk_weights"].to(DEV), ids.to(DEV)

    import flaggems_sglang

    def call(path=0):
        return flaggems_sglang.fused_experts(x, t1, t2, tw, ti, path=path, use_int4_w4a16=True, w1_scale=s1,
                                             w2_scale=s2, w1_zp=z1, w2_zp=z2)

    eager = call()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        call()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            out = call()
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        assert torch.equal(call(), eager)
    assert _rel(eager.float().cpu(), call(2).float().cpu()) < 1e-2


def test_no_allocation_entry_takes_what_it_took():
    """A batch whose prefill workspace (tail-split parts) is above the
    library's scratch: the no-allocation entry runs the streaming kernels."""
    import flaggems_sglang
    from flaggems_sglang import _lib

    L = _lib.lib()
    M, K, N, E, k = 1300, 4352, 4096, 32, 2
    g = torch.Generator(device=DEV).manual_seed(1)

    def weight(R, C):
        q = torch.randint(0, 256, (E, R // 16, C // 128, 1024), device=DEV, generator=g).to(torch.uint8)
        s = (0.002 + 0.001 * torch.rand(E, C // 128, R, device=DEV, generator=g)).to(torch.float16)
        return q, s, torch.full((E, C // 128, R // 2), 0x77, dtype=torch.uint8, device=DEV)

    (q1, s1, z1), (q2, s2, z2) = weight(2 * N, K), weight(K, N)
    x = torch.randn(M, K, device=DEV, generator=g).to(torch.bfloat16)
    tw, ti = flaggems_sglang.topk_softmax(torch.randn(M, E, device=DEV, generator=g), k)
    out = torch.empty_like(x)
    a = _lib.FusedArgs()
    a.wtype, a.x, a.M, a.K, a.N, a.E, a.top_k = _lib.W_INT4_TILED, x.data_ptr(), M, K, N, E, k
    a.w13, a.w2, a.w13_scale, a.w2_scale = q1.data_ptr(), q2.data_ptr(), s1.data_ptr(), s2.data_ptr()
    a.w13_zero, a.w2_zero, a.group_size = z1.data_ptr(), z2.data_ptr(), 128
    a.topk_weights, a.topk_ids, a.routed_scaling_factor = tw.data_ptr(), ti.data_ptr(), 1.0
    a.out = out.data_ptr()
    assert L.fmoe_fused_experts_workspace_bytes(ctypes.byref(a)) > 64 << 20
    a.path = 2
    assert 0 < L.fmoe_fused_experts_workspace_bytes(ctypes.byref(a)) <= 64 << 20
    a.path = 0
    _lib.check(L.fmoe_fused_experts_noalloc(ctypes.byref(a), _lib.stream_of(x)), "noalloc")
    ref = flaggems_sglang.fused_experts(x, q1, q2, tw, ti, path=2, use_int4_w4a16=True, w1_scale=s1, w2_scale=s2,
                                        w1_zp=z1, w2_zp=z2)
    assert torch.equal(out, ref)


def test_size_rule():
    """Small layers keep the streaming kernels: g1 = E N / 128 up to 96, or
    E K N below 2^25."""
    for (E, K, N), unpacks in (((8, 4096, 1792), True), ((8, 8192, 1024), False), ((4, 640, 13184), True),
                               ((4, 640, 13056), False), ((97, 2816, 128), True), ((96, 2816, 128), False)):
        assert _unpacks(50 * E, K, N, E, 2) == unpacks
