"""C-ABI checks that need no GPU: the library loads, exports every symbol declared in
include/tlmi355x.h, and rejects bad arguments before touching HIP (error paths modelled on the
reference's ValueError / status-code conventions, cython_wrapper.pyx:76-79, 130-150 and
main_template.cpp:15-31, 64-67)."""
import ctypes
import os
import re

import pytest

from conftest import ROOT

from tilelang.jit.adapter.mi355x import lib

HEADER = os.path.join(ROOT, "include", "tlmi355x.h")


def declared_symbols():
    src = open(HEADER).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    return sorted(set(re.findall(r"\b(tlm_[a-z0-9_]+)\s*\(", src)))


def test_header_declares_entry_points():
    syms = declared_symbols()
    for s in ("tlm_init", "tlm_last_error", "tlm_rmsnorm", "tlm_gemm", "tlm_rope", "tlm_swiglu",
              "tlm_flash_attn_fwd", "tlm_mla_decode", "tlm_mla_workspace_bytes",
              "tlm_paged_gather", "tlm_kv_append_fp8", "tlm_cast", "tlm_flash_attn_fwd_ex",
              "tlm_gemm_fp8", "tlm_sigmoid", "tlm_gather_rows", "tlm_topk", "tlm_row_reduce",
              "tlm_flash_attn_varlen_fwd", "tlm_flash_attn_bhsd_fwd"):
        assert s in syms


def test_library_exports_every_declared_symbol():
    L = lib.load()
    missing = [s for s in declared_symbols() if not hasattr(L, s)]
    assert not missing, f"libtlmi355x.so lacks {missing}"
    # and the ctypes table covers them all
    assert set(declared_symbols()) <= set(lib.EXPORTED)


def test_version():
    assert lib.load().tlm_version() >= 100


def _err():
    return lib.load().tlm_last_error().decode()


def test_rmsnorm_rejects_null_and_dtype():
    L = lib.load()
    assert L.tlm_rmsnorm(None, None, None, 4, 4, 1e-6, lib.F16, None) == -1
    assert "null" in _err()
    p = ctypes.c_void_p(0x1000)
    assert L.tlm_rmsnorm(p, None, p, 4, 4, 1e-6, lib.F8E4M3, None) == -2
    assert "dtype" in _err()
    # fp32 rows need 4-byte alignment
    assert L.tlm_rmsnorm(ctypes.c_void_p(0x1002), None, p, 4, 4, 1e-6, lib.F32, None) == -1
    assert L.tlm_rmsnorm(p, None, p, -1, 4, 1e-6, lib.F16, None) == -1
    assert L.tlm_rmsnorm(ctypes.c_void_p(0x1001), None, p, 4, 4, 1e-6, lib.F16, None) == -1
    assert "aligned" in _err()
    assert L.tlm_rmsnorm(p, None, p, 4, 4, -1.0, lib.F16, None) == -1


def test_swiglu_rope_validation():
    L = lib.load()
    p = ctypes.c_void_p(0x1000)
    assert L.tlm_swiglu(p, None, p, 8, lib.BF16, None) == -1
    assert L.tlm_swiglu(p, p, p, -8, lib.BF16, None) == -1
    assert L.tlm_swiglu(p, p, p, 8, lib.F8E4M3, None) == -2
    # zero-size is a successful no-op that never reaches HIP
    assert L.tlm_swiglu(p, p, p, 0, lib.BF16, None) == 0
    assert L.tlm_swiglu(p, p, p, 0, lib.F32, None) == 0
    assert L.tlm_swiglu(ctypes.c_void_p(0x1002), p, p, 8, lib.F32, None) == -1
    assert L.tlm_rope(p, p, p, p, p, None, 4, 2, 2, 128, lib.BF16, None) == -1  # k_out missing
    assert L.tlm_rope(p, None, p, p, p, None, 4, 2, 0, 127, lib.BF16, None) == -1  # odd dim
    assert L.tlm_rope(p, None, p, p, p, None, 0, 2, 0, 128, lib.BF16, None) == 0
    assert L.tlm_rope(p, None, p, p, p, None, 0, 2, 0, 128, lib.F32, None) == 0
    assert L.tlm_rope(p, None, p, p, p, None, 4, 2, 0, 128, lib.F8E4M3, None) == -2


def test_gemm_fp8_validation():
    L = lib.load()
    p = ctypes.c_void_p(0x1000)
    assert L.tlm_gemm_fp8(None, p, p, 16, 16, 16, lib.F8E4M3, lib.F32, 1, None) == -1
    assert L.tlm_gemm_fp8(p, p, p, 16, 16, 16, lib.F16, lib.F32, 1, None) == -2
    assert L.tlm_gemm_fp8(p, p, p, 16, 16, 16, lib.F8E4M3, lib.F8E5M2, 1, None) == -2
    assert L.tlm_gemm_fp8(p, p, p, 16, 16, 16, lib.F8E4M3, lib.F32, 2, None) == -1
    assert L.tlm_gemm_fp8(p, p, p, 0, 16, 16, lib.F8E5M2, lib.F8E5M2, 1, None) == 0


def test_ppl_ops_validation():
    L = lib.load()
    p = ctypes.c_void_p(0x1000)
    assert L.tlm_sigmoid(None, p, 8, lib.F32, None) == -1
    assert L.tlm_sigmoid(p, p, 8, lib.I32, None) == -2
    assert L.tlm_sigmoid(p, p, 0, lib.F32, None) == 0
    assert L.tlm_gather_rows(p, 10, 256, None, 4, p, None) == -1
    assert L.tlm_gather_rows(p, 10, 3, p, 4, p, None) == -1  # odd row bytes
    assert L.tlm_gather_rows(p, 10, 256, p, 0, p, None) == 0
    assert L.tlm_topk(p, 100, 101, 1, lib.F32, p, p, None) == -1  # k > length
    assert L.tlm_topk(p, 100, 8, 1, lib.F16, p, p, None) == -2
    assert L.tlm_topk(p, 16385, 8, 1, lib.F32, p, p, None) == -2  # one-workgroup limit
    assert "limit" in _err()
    assert L.tlm_topk(p, 0, 0, 1, lib.U32, p, p, None) == 0
    assert L.tlm_row_reduce(p, p, 4, 4, 7, lib.F16, lib.F16, None) == -1  # unknown op
    assert L.tlm_row_reduce(p, p, 4, 4, lib.REDUCE_MAX, lib.I32, lib.F16, None) == -2
    assert L.tlm_row_reduce(p, p, 0, 4, lib.REDUCE_SUM, lib.F16, lib.F32, None) == 0


def test_cast_validation():
    L = lib.load()
    p = ctypes.c_void_p(0x1000)
    assert L.tlm_cast(None, lib.F32, p, lib.F16, 8, None) == -1
    assert L.tlm_cast(p, lib.F32, p, lib.F16, -1, None) == -1
    assert L.tlm_cast(p, lib.F16, p, lib.BF16, 8, None) == -2  # 16-bit <-> 16-bit
    assert L.tlm_cast(p, lib.F32, p, lib.F32, 8, None) == -2
    assert L.tlm_cast(ctypes.c_void_p(0x1002), lib.F32, p, lib.F16, 8, None) == -1
    assert L.tlm_cast(p, lib.BF16, p, lib.F32, 0, None) == 0


@pytest.mark.parametrize("args,code", [
    # null pointers
    ((None, None, None, 16, 16, 16, lib.F16, lib.F16, 0), -1),
    # bad in dtype (fp32 operands are cast to 16-bit tiles by the caller, tlm_cast)
    ((0x1000, 0x1000, 0x1000, 16, 16, 16, lib.F32, lib.F16, 0), -2),
    # bad trans flag
    ((0x1000, 0x1000, 0x1000, 16, 16, 16, lib.F16, lib.F16, 2), -1),
    # negative size
    ((0x1000, 0x1000, 0x1000, -1, 16, 16, lib.F16, lib.F16, 0), -1),
])
def test_gemm_validation(args, code):
    L = lib.load()
    a = [ctypes.c_void_p(x) if isinstance(x, int) and i < 3 else x for i, x in enumerate(args)]
    assert L.tlm_gemm(*a, None) == code


def test_flash_attn_validation():
    L = lib.load()
    p = ctypes.c_void_p(0x1000)
    assert L.tlm_flash_attn_fwd(None, p, p, p, 1, 16, 1, 128, 0, 0.1, lib.BF16, None) == -1
    assert L.tlm_flash_attn_fwd(p, p, p, p, 1, 16, 1, 100, 0, 0.1, lib.BF16, None) == -2  # D % 8
    assert L.tlm_flash_attn_fwd(p, p, p, p, 1, 16, 1, 264, 0, 0.1, lib.BF16, None) == -2  # > 256
    assert L.tlm_flash_attn_fwd(p, p, p, p, 1, 16, 1, 128, 0, 0.1, lib.F8E4M3, None) == -2
    # fp32 attention takes head dims that are multiples of 4 and an fp32 output only
    assert L.tlm_flash_attn_fwd(p, p, p, p, 1, 16, 1, 22, 0, 0.1, lib.F32, None) == -2
    assert L.tlm_flash_attn_fwd_ex(p, p, p, p, 1, 16, 1, 1, 20, 0, 0.1, lib.F32, lib.BF16,
                                   None) == -2
    assert L.tlm_flash_attn_fwd(p, p, p, p, 1, 0, 1, 128, 0, 0.1, lib.BF16, None) == 0
    assert L.tlm_flash_attn_fwd(p, p, p, p, 1, 0, 1, 8, 0, 0.1, lib.BF16, None) == 0
    ex = L.tlm_flash_attn_fwd_ex
    assert ex(p, p, p, p, 1, 0, 1, 1, 8, 0, 0.1, lib.F16, lib.F32, None) == 0
    assert ex(p, p, p, p, 1, 16, 1, 1, 8, 0, 0.1, lib.F16, lib.BF16, None) == -2
    assert ex(p, p, p, p, 1, 0, 1, 1, 8, 0, 0.1, lib.F32, lib.F32, None) == 0  # fp32: valid
    assert ex(p, p, p, p, 1, 16, 8, 3, 128, 0, 0.1, lib.BF16, lib.BF16, None) == -1  # 8 % 3
    assert ex(p, p, p, p, 1, 16, 8, 0, 128, 0, 0.1, lib.BF16, lib.BF16, None) == -1
    assert ex(p, p, p, p, 1, 0, 8, 2, 128, 0, 0.1, lib.BF16, lib.BF16, None) == 0
    vl = L.tlm_flash_attn_varlen_fwd
    cu = ctypes.c_void_p(0x2000)
    # q, k, v, o, cu_q, cu_k, B, max_seqlen_q, total_q, total_k, H, H_kv, D, causal, scale, ...
    # (only rejected or empty calls: a valid one would launch on the fake pointers)
    assert vl(p, p, p, p, None, cu, 2, 64, 100, 90, 8, 2, 128, 0, 0.1, lib.F16, lib.F16,
              None) == -1
    assert vl(p, p, p, p, ctypes.c_void_p(0x2002), cu, 2, 64, 100, 90, 8, 2, 128, 0, 0.1,
              lib.F16, lib.F16, None) == -1  # cu_seqlens alignment
    assert vl(p, p, p, p, cu, cu, -1, 64, 100, 90, 8, 2, 128, 0, 0.1, lib.F16, lib.F16,
              None) == -1
    assert vl(p, p, p, p, cu, cu, 2, 64, 2 ** 31, 90, 8, 2, 128, 0, 0.1, lib.F16, lib.F16,
              None) == -1  # total rows beyond int32
    assert vl(p, p, p, p, cu, cu, 2, 64, 100, 90, 8, 3, 128, 0, 0.1, lib.F16, lib.F16,
              None) == -1  # 8 % 3
    assert vl(p, p, p, p, cu, cu, 2, 64, 100, 90, 8, 2, 100, 0, 0.1, lib.F16, lib.F16,
              None) == -2  # D % 8
    assert vl(p, p, p, p, cu, cu, 2, 64, 100, 90, 8, 2, 128, 0, 0.1, lib.F8E5M2, lib.F32,
              None) == -2
    assert vl(p, p, p, p, cu, cu, 2, 64, 100, 90, 8, 2, 128, 0, -1.0, lib.F16, lib.F16,
              None) == -1
    # nothing to do: no sequences, no queries, no rows
    assert vl(p, p, p, p, cu, cu, 0, 64, 100, 90, 8, 2, 128, 0, 0.1, lib.F16, lib.F16, None) == 0
    assert vl(p, p, p, p, cu, cu, 2, 0, 100, 90, 8, 2, 128, 0, 0.1, lib.F16, lib.F16, None) == 0
    assert vl(p, p, p, p, cu, cu, 2, 64, 0, 90, 8, 2, 128, 0, 0.1, lib.F16, lib.F16, None) == 0
    bh = L.tlm_flash_attn_bhsd_fwd
    # q, k, v, o, B, H, H_kv, S_q, S_kv, D, causal, scale, in, out, stream (rejected or empty only)
    assert bh(None, p, p, p, 1, 8, 2, 64, 80, 128, 0, 0.1, lib.F16, lib.F16, None) == -1
    assert bh(p, p, p, p, 1, 8, 3, 64, 80, 128, 0, 0.1, lib.F16, lib.F16, None) == -1  # 8 % 3
    assert bh(p, p, p, p, 1, 8, 2, -1, 80, 128, 0, 0.1, lib.F16, lib.F16, None) == -1
    assert bh(p, p, p, p, 1, 8, 2, 64, 2 ** 25, 128, 0, 0.1, lib.F16, lib.F16, None) == -1
    assert bh(p, p, p, p, 1, 8, 2, 64, 80, 260, 0, 0.1, lib.F16, lib.F16, None) == -2
    assert bh(p, p, p, p, 1, 8, 2, 64, 80, 128, 0, 0.1, lib.F16, lib.BF16, None) == -2
    assert bh(p, p, p, p, 1, 8, 2, 64, 80, 128, 1, 0.0, lib.F16, lib.F16, None) == -1
    assert bh(p, p, p, p, 0, 8, 2, 64, 80, 128, 0, 0.1, lib.F16, lib.F16, None) == 0
    assert bh(p, p, p, p, 1, 8, 2, 0, 80, 128, 0, 0.1, lib.F16, lib.F16, None) == 0


def test_splitkv_attention_validation_and_workspace():
    L = lib.load()
    p = ctypes.c_void_p(0x1000)
    wsb = L.tlm_flash_attn_splitkv_workspace_bytes
    # example_mha_inference.py defaults: B 1, 128 queries, 8192 keys, 32 heads, D 128, 4 splits:
    # 128 workgroups before the key parts, so each split is cut in two (fp32 O and lse per part)
    assert wsb(1, 128, 8192, 32, 128, 4) == 1 * 128 * 32 * 4 * 2 * 129 * 4
    assert wsb(1, 128, 8190, 32, 128, 4) == 0  # S_kv not a multiple of num_split
    assert wsb(1, 128, 8192, 32, 128, 17) == 0
    f = L.tlm_flash_attn_splitkv_fwd
    # q, k, v, glse, o_partial, o, ws, ws_bytes, B, S_q, S_kv, H, H_kv, D, ns, scale, dtype, stream
    big = 1 << 30
    assert f(p, p, p, None, p, p, p, big, 1, 128, 8192, 32, 32, 128, 4, 0.1, lib.F16, None) == -1
    assert f(p, p, p, p, p, p, p, big, 1, 128, 8190, 32, 32, 128, 4, 0.1, lib.F16, None) == -1
    assert f(p, p, p, p, p, p, p, big, 1, 128, 8192, 32, 32, 128, 17, 0.1, lib.F16, None) == -2
    assert f(p, p, p, p, p, p, p, big, 1, 128, 8192, 32, 32, 128, 4, 0.1, lib.F32, None) == -2
    assert f(p, p, p, p, p, p, p, big, 1, 128, 8192, 32, 3, 128, 4, 0.1, lib.F16, None) == -1
    assert f(p, p, p, p, p, p, p, 64, 1, 128, 8192, 32, 32, 128, 4, 0.1, lib.F16, None) == -4
    assert "workspace" in _err()
    assert f(p, p, p, p, p, p, p, 0, 0, 128, 8192, 32, 32, 128, 4, 0.1, lib.F16, None) == 0


def test_mla_validation_and_workspace():
    L = lib.load()
    ws = L.tlm_mla_workspace_bytes(64, 128, 512, 4)
    assert ws >= 64 * 128 * 4 * (512 + 1) * 4
    p = ctypes.c_void_p(0x1000)
    # workspace too small
    rc = L.tlm_mla_decode(p, p, 576, 576, p, p, 576, 576, 1000, p, p, p, p, 16, 2, 128, 512, 64,
                          64, 4, 2, 0.07, None, lib.BF16, lib.F8E4M3, lib.BF16, None)
    assert rc == -4 and "workspace" in _err()
    # head dims beyond the generic kernel's (dv <= 1024, dpe <= 256)
    rc = L.tlm_mla_decode(p, p, 2048, 576, p, p, 2048, 576, 1000, p, p, p, p, 1 << 30, 2, 128,
                          2048, 64, 64, 4, 2, 0.07, None, lib.BF16, lib.F8E4M3, lib.BF16, None)
    assert rc == -2
    rc = L.tlm_mla_decode(p, p, 576, 576, p, p, 576, 576, 1000, p, p, p, p, 1 << 30, 2, 128, 512,
                          512, 64, 4, 2, 0.07, None, lib.BF16, lib.F8E4M3, lib.BF16, None)
    assert rc == -2
    # misaligned (odd) pointer for 16-bit Q
    rc = L.tlm_mla_decode(ctypes.c_void_p(0x1001), p, 576, 576, p, p, 576, 576, 1000, p, p, p, p,
                          1 << 30, 2, 128, 512, 64, 64, 4, 2, 0.07, None, lib.BF16, lib.F8E4M3,
                          lib.BF16, None)
    assert rc == -1
    # null block table
    rc = L.tlm_mla_decode(p, p, 576, 576, p, p, 576, 576, 1000, None, p, p, p, 1 << 30, 2, 128,
                          512, 64, 64, 4, 2, 0.07, None, lib.BF16, lib.F8E4M3, lib.BF16, None)
    assert rc == -1
    # fp16 KV with bf16 Q is not a kernel combination
    rc = L.tlm_mla_decode(p, p, 576, 576, p, p, 576, 576, 1000, p, p, p, p, 1 << 30, 2, 128,
                          512, 64, 64, 4, 2, 0.07, None, lib.BF16, lib.F16, lib.BF16, None)
    assert rc == -2
    # max_pages * page beyond the int32 token range
    rc = L.tlm_mla_decode(p, p, 576, 576, p, p, 576, 576, 1000, p, p, p, p, 1 << 62, 2, 128,
                          512, 64, 1 << 20, 1 << 20, 1, 0.07, None, lib.BF16, lib.F8E4M3,
                          lib.BF16, None)
    assert rc == -1


def test_mla_decode_ex_validation():
    L = lib.load()
    p = ctypes.c_void_p(0x1000)
    bt = ctypes.c_void_p(0x2000)
    f = L.tlm_mla_decode_ex
    # q, q_pe, qs, qpes, kv, k_pe, kvs, kpes, rows, bt, sl, o, ws, ws_bytes, B, Hq, dv, dpe, page,
    # max_pages, ns, scale, kv_scale, q_dt, kv_dt, o_dt, glse, o_partial, part_block, p_dt, stream
    args = [p, p, 576, 576, p, p, 576, 576, 1024, bt, bt, p, p, 1 << 30, 2, 64, 512, 64, 64, 8,
            4, 0.1, None, lib.F16, lib.F16, lib.F16]
    assert f(*args, p, None, 64, lib.F16, None) == -1       # o_partial missing
    assert f(*args, p, p, 0, lib.F16, None) == -1           # part_block
    assert f(*args, p, p, 64, lib.F8E4M3, None) == -1       # partial dtype
    assert f(*args, ctypes.c_void_p(0x1001), p, 64, lib.F16, None) == -1  # glse alignment
    a2 = list(args)
    a2[16] = 510  # dv not a multiple of 4
    a2[2] = a2[6] = 574
    assert f(*a2, p, p, 64, lib.F16, None) == -2
    a0 = list(args)
    a0[14] = 0   # no sequences: nothing to do
    assert f(*a0, p, p, 64, lib.F16, None) == 0


def test_mla_noalloc_validation():
    """The allocation-free entry point validates like tlm_mla_decode and rejects, before any HIP
    call, a request whose scratch need exceeds the library's array."""
    L = lib.load()
    assert L.tlm_mla_scratch_bytes() == 128 << 20
    p = ctypes.c_void_p(0x1000)

    def call(B=64, Hq=128, dv=512, splits=4, bt=p, kv_dt=lib.F8E4M3, page=64):
        return L.tlm_mla_decode_noalloc(p, p, 576, 576, p, p, 576, 576, 1 << 20, bt, p, p, B, Hq,
                                        dv, 64, page, 128, splits, 0.07, None, lib.BF16, kv_dt,
                                        lib.BF16, None)
    assert call(bt=None) == -1
    assert call(dv=2048) == -2
    assert call(kv_dt=lib.F16) == -2  # fp16 KV with bf16 Q
    # the FP8 config with 64 splits needs far more than the scratch
    assert call(splits=64) == -4 and "scratch" in _err()
    # fp8 pages of 16 tokens take the split path, whose 16 splits x 64 sequences need 269 MB
    assert call(page=16, splits=16) == -4 and "scratch" in _err()
    # bf16 KV (split path, 4 splits x 4096 sequences) as well
    assert L.tlm_mla_decode_noalloc(p, p, 576, 576, p, p, 576, 576, 1 << 20, p, p, p, 4096, 128,
                                    512, 64, 64, 128, 4, 0.07, None, lib.BF16, lib.BF16,
                                    lib.BF16, None) == -4
    assert call(B=0) == 0
    # the config's FP8 path fits the scratch at the benchmark's 4 splits (the size check passes;
    # without a GPU the call fails after it), not at 5
    assert call(splits=5) == -4 and "scratch" in _err()
    assert call(splits=4) != -4


def test_paged_gather_validation():
    L = lib.load()
    p = ctypes.c_void_p(0x1000)
    assert L.tlm_paged_gather(None, 576, 10, p, p, p, p, 1, 64, 4, None) == -1
    assert L.tlm_paged_gather(p, 0, 10, p, p, p, p, 1, 64, 4, None) == -1
    assert L.tlm_paged_gather(p, 576, 10, p, p, p, p, 0, 64, 4, None) == 0


def test_init_without_gpu_reports_error():
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is visible")
    L = lib.load()
    assert L.tlm_init(0) != 0
    assert _err()
    assert L.tlm_init(-1) == -1


def test_kv_append_validation():
    L = lib.load()
    p = ctypes.c_void_p(0x1000)
    args = lambda x=p, dt=lib.BF16, D=576, B=2, T=3, ks=576: (
        x, 576 * 3, 576, dt, p, p, p, 4, 64, p, ks, 100, B, T, D, p, None)
    assert L.tlm_kv_append_fp8(*args(x=None)) == -1
    assert L.tlm_kv_append_fp8(*args(dt=lib.F32)) == -2
    assert L.tlm_kv_append_fp8(*args(D=570, ks=576)) == -2
    assert L.tlm_kv_append_fp8(*args(ks=100)) == -1  # kv row stride smaller than D
    assert L.tlm_kv_append_fp8(*args(B=0)) == 0


def test_elementwise_validation():
    L = lib.load()
    P, I = ctypes.c_void_p, ctypes.c_int
    p = P(0x1000)
    ins = (P * 1)(p)
    dts = (I * 1)(lib.F32)
    bc = (I * 1)(lib.EW_FULL)
    outs = (P * 1)(p)
    odt = (I * 1)(lib.F32)
    cf = (ctypes.c_float * 1)(1.0)

    def run(code, n_in=1, bcast=bc, rows=4, cols=4, n_const=1):
        cw = (ctypes.c_int32 * len(code))(*code)
        return L.tlm_elementwise(ins, dts, bcast, n_in, outs, odt, 1, cw, len(code), cf, n_const,
                                 rows, cols, None)
    load0, store0 = lib.EW_LOAD, lib.EW_STORE
    assert run([load0, store0], rows=0) == 0
    assert run([load0 | 1 << 20, store0]) == -1          # input 1 of 1
    assert run([lib.EW_CONST | 1 << 20, store0]) == -1    # constant 1 of 1
    assert run([load0, store0 | 1 << 20]) == -1          # output 1 of 1
    assert run([load0 | 8 << 8, store0]) == -1           # slot 8 of 8
    assert run([11, store0]) == -1                       # no such opcode
    assert run([lib.EW_ROUND | 7 << 20, store0]) == -1    # rounding to a non-float dtype
    assert run([load0, store0], bcast=(I * 1)(9)) == -1  # broadcast kind
    assert run([]) == -1
    assert run([load0] * 65) == -1


def test_mla_h16_ranges_fit_the_cus():
    """A decode workgroup holds a CU's whole LDS: the ranges times the blocks of 64 heads are at most the 256 CUs
    (the rest would start when the first end), and their partial rows fit the workspace."""
    L = lib.load()
    for hq in range(64, 4097, 64):
        for B in (1, 2, 8, 60, 300, 4096):
            for ns in (1, 4, 64):
                ws = L.tlm_mla_workspace_bytes(B, hq, 512, ns)
                G = L.tlm_mla_h16_ranges(B, hq, ws)
                assert G == 1 or G * (hq // 64) <= 256, (hq, B, ns, G)
                assert (G - 1 + min(B, G - 1)) * hq * 513 * 4 <= ws
            assert L.tlm_mla_h16_ranges(B, hq, 0) == 1
    assert L.tlm_mla_h16_ranges(8, 128, 1 << 30) == 128
    assert L.tlm_mla_h16_ranges(8, 192, 1 << 30) == 85
