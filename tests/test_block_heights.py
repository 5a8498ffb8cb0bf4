"""Tile heights that the library picks at both sides of each line (host only)."""

import pytest

from flaggems_sglang import _lib


def _bm(wt, M, k, E, K=8192, N=16384, path=0):
    return _lib.lib().fmoe_fused_block_m(wt, M, k, E, path, K, N)


@pytest.mark.parametrize("M,bm", [(1, 16), (80, 16), (81, 32), (183, 32), (184, 64), (391, 64), (392, 128),
                                  (2047, 160), (2048, 256)])
def test_bf16_by_mean(M, bm):
    assert _bm(_lib.W_BF16, M, 1, 8) == bm


@pytest.mark.parametrize("M,bm", [(24, 16), (25, 64), (319, 64), (320, 128)])
def test_fp8_by_mean(M, bm):
    assert _bm(_lib.W_FP8, 32 * M, 1, 256, K=7168, N=2048) == bm


@pytest.mark.parametrize("wt,E,K,N,line", [
    (_lib.W_BF16, 8, 4096, 14336, 10), (_lib.W_BF16, 8, 4096, 7168, 13), (_lib.W_BF16, 8, 4096, 1792, 13),
    (_lib.W_BF16, 64, 1280, 3072, 10), (_lib.W_BF16, 128, 2048, 768, 10), (_lib.W_BF16, 8, 2048, 896, 13),
    (_lib.W_BF16, 8, 2048, 768, 16), (_lib.W_BF16, 8, 8192, 512, 16),
    (_lib.W_FP8, 256, 7168, 2048, 3), (_lib.W_FP8, 64, 1280, 3072, 3), (_lib.W_FP8, 128, 2048, 768, 3),
    (_lib.W_FP8, 32, 7168, 2048, 3), (_lib.W_FP8, 256, 1024, 512, 13), (_lib.W_FP8, 40, 4096, 2048, 13),
    (_lib.W_FP8, 8, 4096, 14336, 13), (_lib.W_FP8, 8, 4096, 1792, 13), (_lib.W_FP8, 4, 4096, 8192, 16),
    (_lib.W_FP8, 8, 4096, 1536, 16)])
def test_streaming_line_by_workgroups(wt, E, K, N, line):
    """The last streaming mean and the first prefill one, by what the layer's
    prefill tiles would make of the chip."""
    assert _bm(wt, line * E, 1, E, K=K, N=N) == 16
    assert _bm(wt, line * E + 1, 1, E, K=K, N=N) in (32, 64)
    assert _bm(wt, line * E, 1, E, K=K, N=N, path=1) in (32, 64)
    assert _lib.lib().fmoe_choose_block_m(wt, 13 * E, 1, E, 0) == 16


def test_small_4bit_layers_stream():
    """Up to 96 GEMM1 workgroups of 256 weight rows."""
    for wt in (_lib.W_MXFP4, _lib.W_MXFP4_TILED):
        assert _bm(wt, 8 * 200, 1, 8, K=8192, N=1536) == 16
        assert _bm(wt, 8 * 200, 1, 8, K=8192, N=1664) == 128


@pytest.mark.parametrize("wt,N,stream", [(_lib.W_MXFP4, 7168, 1), (_lib.W_MXFP4_TILED, 7168, 3),
                                         (_lib.W_MXFP4, 7040, 24), (_lib.W_MXFP4_TILED, 7040, 36)])
def test_mxfp4_by_width_and_layout(wt, N, stream):
    assert _bm(wt, 8 * stream, 1, 8, N=N) == 16
    nxt = 32 if stream < 22 else (64 if stream < 48 else 128)
    assert _bm(wt, 8 * (stream + 1), 1, 8, N=N) == nxt
    assert _bm(wt, 8 * 49, 1, 8, N=N) == 128
    for path in (1, 2):
        assert _bm(wt, 8 * 49, 1, 8, N=N, path=path) == 16
    assert _lib.lib().fmoe_choose_block_m(wt, 8 * 49, 1, 8, 0) == 16


def test_int4_routing_stays_at_16():
    for M in (1, 100, 700, 5000):
        assert _bm(_lib.W_INT4, M, 2, 8) == 16 and _bm(_lib.W_INT4_TILED, M, 2, 8) == 16


@pytest.mark.parametrize("K,N", [(6144, 32768), (16512, 2048), (2048, 16512)])
def test_fp8_layers_above_the_staged_scales_stream(K, N):
    """The prefill kernels hold the scales of reductions up to 16384; larger
    layers stream up to 16 slots per expert, as the size-free choice does."""
    for M in (1, 13, 16, 64):
        assert _bm(_lib.W_FP8, M, 2, 8, K=K, N=N) == 16
        assert _lib.lib().fmoe_choose_block_m(_lib.W_FP8, M, 2, 8, 0) == 16
    assert _bm(_lib.W_FP8, 65, 2, 8, K=K, N=N) == 64
    assert _bm(_lib.W_FP8, 13, 2, 8, K=16384, N=16384) == 64
    assert _bm(_lib.W_FP8, 12, 2, 8, K=16384, N=16384) == 16


@pytest.mark.parametrize("wt,M,bm", [
    # 32 of 256 experts, top-8; slots per expert: M / 32 at the even share, M / 4 at the largest load
    (_lib.W_FP8, 64, 16), (_lib.W_FP8, 65, 64), (_lib.W_FP8, 159, 64), (_lib.W_FP8, 160, 128),
    (_lib.W_FP8, 512, 160), (_lib.W_FP8, 547, 128), (_lib.W_FP8, 1001, 128), (_lib.W_FP8, 2048, 160),
    (_lib.W_BF16, 64, 16), (_lib.W_BF16, 65, 32), (_lib.W_BF16, 192, 64), (_lib.W_BF16, 256, 128),
    (_lib.W_BF16, 546, 160), (_lib.W_BF16, 547, 128), (_lib.W_BF16, 2048, 160), (_lib.W_BF16, 4096, 256),
    # MXFP4: streaming while the even share is (512 GEMM1 workgroups here: 1 slot), then M / 16
    (_lib.W_MXFP4, 32, 16), (_lib.W_MXFP4, 33, 32), (_lib.W_MXFP4, 367, 32), (_lib.W_MXFP4, 368, 64),
    (_lib.W_MXFP4, 783, 64), (_lib.W_MXFP4, 784, 128)])
def test_expert_parallel_heights(wt, M, bm):
    L = _lib.lib()
    assert L.fmoe_fused_block_m_ep(wt, M, 8, 32, 256, 0, 7168, 2048) == bm
    assert L.fmoe_fused_block_m_ep(wt, M, 8, 32, 0, 0, 7168, 2048) == L.fmoe_fused_block_m(wt, M, 8, 32, 0, 7168, 2048)


@pytest.mark.parametrize("wt", [_lib.W_BF16, _lib.W_FP8, _lib.W_MXFP4, _lib.W_MXFP4_TILED])
@pytest.mark.parametrize("E,n_global,k", [(32, 256, 8), (4, 256, 8), (16, 128, 8), (4, 8, 2), (1, 64, 4)])
def test_expert_parallel_never_streams_a_full_load(wt, E, n_global, k):
    """Tokens dispatched to the rank can fill every choice: whatever the even
    share is, batches of more than 16 such slots per expert (MXFP4: 48) run on
    prefill tiles, bf16 and fp8 ones of 128 rows or more once the full load needs
    two tiles."""
    mx = wt in (_lib.W_MXFP4, _lib.W_MXFP4_TILED)
    N = 12928 // E // 128 * 128 + 128 if mx else 2048  # more than 96 GEMM1 workgroups
    for M in range(1, 3000, 7):
        bm = _lib.lib().fmoe_fused_block_m_ep(wt, M, k, E, n_global, 0, 2048, N)
        if M * k > (48 if mx else 16) * min(E, M * k):
            assert bm > 16
        if not mx and M * k > 160 * E:
            assert bm >= 128
