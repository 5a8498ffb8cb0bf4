"""Prefill launches at the bound of their grid: routings in which every expert
ends in a tile of one row make exactly (slots + E (block_m - 1)) / block_m
tiles, the most that a batch can have, for each tile height -- over reduction
lengths of 1 to 10 ring stages (fewer than the ring's depth, odd and even)."""

import pytest
import torch

from oracle import fused_moe_oracle as O
from test_gpu_fused_moe import _close

pytestmark = pytest.mark.gpu
DEV = "cuda"
E, k = 8, 2

COUNTS = {  # tile height -> slots per expert, each 1 modulo the height
    32: [33, 33] + [1] * 6,
    64: [65, 65, 65] + [1] * 5,
    128: [129, 129, 129] + [1] * 5,
    160: [161] * 6 + [1, 1],
    256: [257] * 8,
}


def _ids(counts):
    flat = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    M = flat.numel() // 2
    return torch.stack((flat[:M], flat[M:]), dim=1).to(torch.int32)


@pytest.mark.parametrize("K,N", [(128, 128), (256, 384), (384, 256), (640, 128), (128, 640)])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("bm", sorted(COUNTS))
def test_every_expert_ends_in_a_one_row_tile(bm, fp8, K, N):
    import flaggems_sglang
    from flaggems_sglang import _lib
    from flaggems_sglang import quant as Q

    if fp8 and bm in (32, 256):
        pytest.skip(f"no {bm}-row fp8 tiles")
    counts = COUNTS[bm]
    ids = _ids(counts)
    M = ids.shape[0]
    assert sum((c + bm - 1) // bm for c in counts) == (M * k + E * (bm - 1)) // bm
    assert _lib.lib().fmoe_fused_block_m(_lib.W_FP8 if fp8 else _lib.W_BF16, M, k, E, 1, K, N) == bm
    d = O.make_inputs(M, K, N, E, k, wscale=0.05, seed=bm)
    tw = d["topk_weights"]
    args = (d["x"].to(DEV),)
    if fp8:
        q1, s1 = Q.quantize_fp8_block(d["w13"])
        q2, s2 = Q.quantize_fp8_block(d["w2"])
        out = flaggems_sglang.fused_experts(*args, q1.to(DEV), q2.to(DEV), tw.to(DEV), ids.to(DEV), path=1,
                                            use_fp8_w8a8=True, block_shape=[128, 128], w1_scale=s1.to(DEV),
                                            w2_scale=s2.to(DEV))
        ref = O.fused_experts_fp8(d["x"], q1, s1, q2, s2, tw, ids)
        # row by row, by norm: both sides round the activation to e4m3, and one
        # code flipped by another summation order moves an element by up to
        # 2^-3 of its largest term (seen: 0.11 rms on 1 of 1e5 elements), a row of
        # N terms by 2^-3 / sqrt(N) (N = 128: 1.1%) of its norm per flip;
        # a row from a missing or misplaced tile is off by its whole norm
        err = (out.float().cpu() - ref.float()).norm(dim=1) / ref.float().norm(dim=1)
        assert float(err.max()) < 5e-2
    else:
        out = flaggems_sglang.fused_experts(*args, d["w13"].to(DEV), d["w2"].to(DEV), tw.to(DEV), ids.to(DEV), path=1)
        _close(out, O.fused_experts(d["x"], d["w13"], d["w2"], tw, ids), 2e-2)
