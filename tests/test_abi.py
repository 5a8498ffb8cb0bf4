"""CPU checks of the C-ABI boundary: libfmoe.so loads, exports every function
``include/fmoe.h`` declares (and ctypes binds exactly those), and the
host-only entry points (sizes, argument validation) behave.  No kernel is
launched: argument errors are detected before any HIP call."""

import ctypes
import os
import re

import pytest

from flaggems_sglang import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "fmoe.h")


def _declared():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(fmoe_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_expected_entries():
    names = _declared()
    for n in ("fmoe_align", "fmoe_gemm1", "fmoe_gemm2", "fmoe_moe_sum", "fmoe_fused_experts",
              "fmoe_topk_softmax", "fmoe_grouped_topk", "fmoe_quant_fp8_group"):
        assert n in names


def test_library_exports_every_declared_symbol():
    lib = ctypes.CDLL(_lib.LIB_PATH)
    for n in _declared():
        assert hasattr(lib, n), n
    assert sorted(_lib.EXPORTED) == _declared()


def test_host_queries():
    L = _lib.lib()
    assert L.fmoe_abi_version() == 2
    assert L.fmoe_status_string(2) == b"not supported"
    assert L.fmoe_max_tiles(8, 256) == 8
    assert L.fmoe_max_tiles(65536, 256) == 255 + (65536 - 256 + 1 + 15) // 16
    assert L.fmoe_sorted_ids_len(128, 8, 16) == 128 + 8 * 15
    assert L.fmoe_choose_block_m(_lib.W_INT4, 4096, 2, 8, 0) == 16
    assert L.fmoe_choose_block_m(_lib.W_BF16, 1, 2, 8, 0) == 16
    assert L.fmoe_choose_block_m(_lib.W_BF16, 4096, 2, 8, 0) == 256
    assert L.fmoe_choose_block_m(_lib.W_BF16, 1024, 8, 128, 0) == 128
    assert L.fmoe_choose_block_m(_lib.W_BF16, 400, 8, 128, 0) == 64
    # fp8: 160-row tiles where the mean + 2 sd load per expert needs fewer of
    # them than of 128-row tiles (DSV3 M=4096: 128 +- 11 slots per expert)
    assert L.fmoe_choose_block_m(_lib.W_FP8, 4096, 8, 256, 0) == 160
    assert L.fmoe_choose_block_m(_lib.W_FP8, 8192, 8, 256, 0) == 160
    assert L.fmoe_choose_block_m(_lib.W_FP8, 3072, 8, 256, 0) == 128
    assert L.fmoe_choose_block_m(_lib.W_FP8, 6400, 8, 256, 0) == 128
    # the fused path's choice: fp8 160-row tiles only while K, N <= 8192
    assert L.fmoe_fused_block_m(_lib.W_FP8, 4096, 8, 256, 0, 7168, 2048) == 160
    assert L.fmoe_fused_block_m(_lib.W_FP8, 4096, 8, 256, 0, 8448, 2048) == 128
    assert L.fmoe_fused_block_m(_lib.W_FP8, 4096, 8, 256, 0, 7168, 8320) == 128
    assert L.fmoe_fused_block_m(_lib.W_BF16, 1024, 8, 64, 0, 16384, 16384) == 160


def test_argument_errors_map_to_reference_convention():
    L = _lib.lib()
    st = L.fmoe_topk_softmax(None, 4, 8, 0, 1, None, None, None)
    assert st == _lib.FMOE_ERR_INVALID
    with pytest.raises(ValueError, match="topk_softmax"):
        _lib.check(st, "topk_softmax")
    ao = _lib.AlignOut()
    st = L.fmoe_align(None, None, 4, 2, 8, 48, ctypes.byref(ao), None, 0, None)
    assert st == _lib.FMOE_ERR_UNSUPPORTED
    with pytest.raises(AssertionError, match="is not supported"):
        _lib.check(st, "align")
    fa = _lib.FusedArgs()
    fa.wtype, fa.M, fa.K, fa.N, fa.E, fa.top_k = 0, 4, 100, 256, 8, 2
    assert L.fmoe_fused_experts_workspace_bytes(ctypes.byref(fa)) == 0
    assert L.fmoe_fused_experts(ctypes.byref(fa), None) == _lib.FMOE_ERR_UNSUPPORTED
    fa.K = 128
    assert L.fmoe_fused_experts_workspace_bytes(ctypes.byref(fa)) > 0
    assert L.fmoe_fused_experts(ctypes.byref(fa), None) == _lib.FMOE_ERR_INVALID  # null pointers
    # int4 weights take SiLU / GELU only (no SWIGLU row pairing)
    fa.wtype, fa.group_size, fa.activation = _lib.W_INT4_TILED, 128, _lib.ACT_SWIGLU
    assert L.fmoe_fused_experts_workspace_bytes(ctypes.byref(fa)) == 0
    assert L.fmoe_fused_experts(ctypes.byref(fa), None) == _lib.FMOE_ERR_UNSUPPORTED
    assert b"SWIGLU" in L.fmoe_last_error()
    fa.activation = _lib.ACT_SILU
    assert L.fmoe_fused_experts_workspace_bytes(ctypes.byref(fa)) > 0


@pytest.mark.parametrize("M", [1, 16, 100, 700, 1100])  # one launch, streaming, unpacking, bf16 copies
@pytest.mark.parametrize("wt,fields", [
    (_lib.W_FP8, ("w13_scale", "w2_scale")),
    (_lib.W_MXFP4, ("w13_scale", "w2_scale")), (_lib.W_MXFP4_TILED, ("w13_scale", "w2_scale")),
    (_lib.W_INT4, ("w13_scale", "w2_scale", "w13_zero", "w2_zero")),
    (_lib.W_INT4_TILED, ("w13_scale", "w2_scale", "w13_zero", "w2_zero"))])
def test_null_scales_and_zeros_are_refused(wt, fields, M):
    """Every route of the whole-path call, before anything is launched: the
    other pointers are host memory, which no kernel may see."""
    L = _lib.lib()
    buf = ctypes.create_string_buffer(64)
    host = ctypes.addressof(buf)
    for missing in fields:
        a = _lib.FusedArgs()
        a.wtype, a.M, a.K, a.N, a.E, a.top_k, a.group_size = wt, M, 256, 256, 8, 2, 128
        a.x = a.w13 = a.w2 = a.topk_weights = a.topk_ids = a.out = host
        for f in fields:
            setattr(a, f, None if f == missing else host)
        # no workspace: a library without the check stops there, short of a launch
        assert L.fmoe_fused_experts(ctypes.byref(a), None) == _lib.FMOE_ERR_INVALID, missing
        assert b"need" in L.fmoe_last_error()


@pytest.mark.parametrize("wt,M,K,N,E,k,path,n_global", [
    (_lib.W_BF16, 256, 7168, 2048, 32, 8, 0, 256), (_lib.W_BF16, 300, 7168, 2048, 32, 8, 0, 256),
    (_lib.W_BF16, 320, 7168, 2048, 32, 8, 0, 256),  # a rank of eight
    (_lib.W_BF16, 300, 7168, 2048, 256, 8, 1, 0), (_lib.W_FP8, 400, 7168, 2048, 256, 8, 1, 0),  # up to 16 slots, path 1
    (_lib.W_INT4, 250, 7168, 128, 256, 8, 2, 0), (_lib.W_MXFP4, 250, 7168, 256, 32, 8, 0, 0),
    (_lib.W_FP8, 250, 7168, 2048, 256, 8, 0, 0)])
def test_noalloc_takes_what_fits_some_layout(wt, M, K, N, E, k, path, n_global):
    """Calls whose preferred layout is above the library's scratch, or close to
    it, but whose streaming kernels or bf16 rows fit: not refused for their size
    (with null pointers they end at the pointer check; without a device before it)."""
    L = _lib.lib()
    some = ctypes.create_string_buffer(16)
    a = _lib.FusedArgs()
    a.wtype, a.M, a.K, a.N, a.E, a.top_k, a.group_size, a.path = wt, M, K, N, E, k, 128, path
    if n_global:
        a.expert_map, a.n_global = ctypes.addressof(some), n_global
    assert L.fmoe_fused_experts_noalloc(ctypes.byref(a), None) in (_lib.FMOE_ERR_INVALID, _lib.FMOE_ERR_HIP)
    a.M = 40 * M
    assert L.fmoe_fused_experts_noalloc(ctypes.byref(a), None) == _lib.FMOE_ERR_UNSUPPORTED


@pytest.mark.parametrize("wt,M,fields", [
    (_lib.W_BF16, 56, ("x", "w13", "w2")), (_lib.W_FP8, 56, ("w13", "w2")),
    (_lib.W_INT4, 400, ("w13", "w2")), (_lib.W_MXFP4, 400, ("x", "w13", "w2", "w13_scale", "w2_scale"))])
def test_unaligned_operands_stream(wt, M, fields):
    """Operands that the prefill kernels' 16-byte DMA cannot fetch take the
    streaming kernels, as the whole range of those calls once did; a size query
    without pointers covers both."""
    L = _lib.lib()

    def size(path=0, **ptrs):
        a = _lib.FusedArgs()
        a.wtype, a.M, a.K, a.N, a.E, a.top_k, a.group_size, a.path = wt, M, 4096, 7168, 8, 2, 128, path
        for f in ("x", "w13", "w2", "w13_scale", "w2_scale", "w13_zero", "w2_zero"):
            setattr(a, f, ptrs.get(f, ptrs.get("all")))
        return L.fmoe_fused_experts_workspace_bytes(ctypes.byref(a))

    prefill, stream = size(all=4096), size(path=2, all=4096)
    assert prefill != stream
    for f in fields:
        assert size(all=4096, **{f: 4096 + 8}) == stream
    assert size() == max(prefill, stream)
    if wt == _lib.W_INT4:
        assert size(all=4096, w13_zero=4096 + 4) == prefill and size(all=4096, w2_scale=4096 + 2) == stream
