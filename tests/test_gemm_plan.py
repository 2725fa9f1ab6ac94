"""Which kernel, tile and split a GEMM call takes (tlm_gemm_plan: host only, no GPU needed)."""
import ctypes

import pytest

from tilelang.jit.adapter.mi355x import lib

PER_THREAD = 2  # hipStreamPerThread

# Calls that reach every tile, whole and split, with remainders in M, N and K, with one row tile and with
# several: (call, M, N, K, tile rows, tile columns, split). nn / nt: 16-bit row-major B / B^T; fp8: B^T;
# dual: tlm_gemm_swiglu (N columns of each of its two matrices). test_gpu_gemm_tile.py runs them.
TILE_CASES = [
    ("nn", 1, 72, 72, 32, 64, False), ("nn", 1, 72, 776, 32, 64, True),
    ("nn", 1, 16392, 72, 32, 128, False), ("nn", 1, 3080, 2056, 32, 128, True),
    ("nn", 33, 72, 72, 64, 64, False), ("nn", 33, 72, 520, 64, 64, True),
    ("nn", 65, 72, 72, 64, 64, False), ("nn", 65, 72, 1032, 64, 64, True),
    ("nn", 33, 16392, 264, 128, 128, False), ("nn", 129, 12296, 136, 128, 128, False),
    ("nn", 65, 8200, 1032, 128, 128, True), ("nn", 200, 4104, 1032, 128, 128, True),
    ("nn", 129, 16392, 136, 256, 128, False), ("nn", 257, 12296, 136, 256, 128, False),
    ("nn", 1025, 12296, 136, 256, 256, False),
    ("nt", 1, 77, 72, 32, 64, False), ("nt", 17, 77, 776, 32, 64, True),
    ("nt", 33, 77, 72, 64, 64, False), ("nt", 33, 77, 520, 64, 64, True),
    ("nt", 65, 77, 72, 64, 64, False), ("nt", 65, 77, 1032, 64, 64, True),
    ("nt", 33, 16397, 264, 128, 128, False), ("nt", 129, 12301, 136, 128, 128, False),
    ("nt", 65, 8205, 1032, 128, 128, True), ("nt", 200, 4109, 1032, 128, 128, True),
    ("nt", 129, 16397, 136, 256, 128, False), ("nt", 257, 12301, 136, 256, 128, False),
    ("nt", 1025, 12301, 136, 256, 256, False),
    ("fp8", 1, 72, 80, 32, 64, False), ("fp8", 1, 72, 2064, 32, 64, True),
    ("fp8", 17, 72, 80, 32, 64, False), ("fp8", 20, 72, 2064, 32, 64, True),
    ("fp8", 33, 72, 80, 64, 64, False), ("fp8", 33, 72, 2064, 64, 64, True),
    ("fp8", 65, 72, 80, 64, 64, False), ("fp8", 65, 72, 2064, 64, 64, True),
    ("fp8", 200, 28680, 80, 128, 128, False), ("fp8", 65, 3080, 8208, 128, 128, True),
    ("fp8", 3000, 72, 8208, 128, 128, True), ("fp8", 1025, 12296, 144, 256, 128, False),
    ("fp8", 129, 16392, 4112, 256, 256, False),
    ("dual", 1, 39, 72, 32, 128, False), ("dual", 1, 39, 776, 32, 128, True),
    ("dual", 33, 39, 72, 64, 64, False), ("dual", 33, 39, 520, 64, 64, True),
    ("dual", 65, 39, 72, 64, 64, False), ("dual", 65, 39, 1032, 64, 64, True),
    ("dual", 33, 8199, 264, 128, 128, False), ("dual", 129, 6151, 136, 128, 128, False),
    ("dual", 65, 4103, 1032, 128, 128, True), ("dual", 200, 2055, 1032, 128, 128, True),
    ("dual", 129, 8199, 136, 256, 128, False), ("dual", 257, 6151, 136, 256, 128, False),
]
# the kernel of one decode step (16 rows, row-major B from 32 MB): K % 16 == 8, ragged strips, uneven ranges
SKINNY_CASES = [(1, 4104, 4104), (5, 4104, 8200), (16, 14344, 1176), (16, 2056, 8200), (3, 16392, 1032),
                (16, 6152, 4104)]


def plan(M, N, K, dt=lib.F16, trans_b=True, dual=False, stream=None, captured=False):
    out = [ctypes.c_int() for _ in range(3)]
    lib.call("tlm_gemm_plan", M, N, K, dt, int(trans_b), int(dual), stream, int(captured),
             *(ctypes.byref(v) for v in out))
    return tuple(v.value for v in out)


@pytest.mark.parametrize("call,M,N,K,rows,cols,split", TILE_CASES)
def test_tile_cases_take_their_tile(call, M, N, K, rows, cols, split):
    for dt in (lib.F8E4M3, lib.F8E5M2) if call == "fp8" else (lib.F16, lib.BF16):
        r, c, ns = plan(M, N, K, dt, trans_b=call != "nn", dual=call == "dual")
        assert (r, c, ns > 1) == (rows, cols, split)


def test_tile_cases_cover_every_tile():
    """Every (tile, split or not) that any call of a grid of shapes takes is among the cases."""
    seen = {(c[0], *c[4:]) for c in TILE_CASES}
    for M in (1, 16, 17, 33, 64, 65, 128, 200, 257, 500, 1000, 2048, 4096):
        for N in (72, 520, 1032, 2056, 4104, 8200, 14336, 28680):
            for K in (72, 264, 1032, 2064, 4096, 8208, 14336):
                for call in ("nn", "nt", "fp8", "dual"):
                    if call == "fp8" and K % 16:
                        continue
                    r, c, ns = plan(M, N, K, lib.F8E4M3 if call == "fp8" else lib.F16,
                                    trans_b=call != "nn", dual=call == "dual")
                    if (r, c) == (16, 128) or (call == "dual" and c == 256):
                        continue  # the decode kernel, or three calls
                    assert (call, r, c, ns > 1) in seen, (call, M, N, K, r, c, ns)


@pytest.mark.parametrize("M,N,K", SKINNY_CASES)
def test_skinny_cases_take_the_decode_kernel(M, N, K):
    assert plan(M, N, K, trans_b=False)[:2] == (16, 128)


SPLIT_CALLS = [dict(M=16, N=14336, K=4096, trans_b=False), dict(M=16, N=4096, K=14336, trans_b=False),
               dict(M=16, N=4096, K=4096, trans_b=False), dict(M=16, N=4096, K=14336),
               dict(M=64, N=1024, K=4096, dt=lib.BF16), dict(M=500, N=4096, K=4096, trans_b=False),
               dict(M=16, N=4096, K=4096, dt=lib.F8E4M3), dict(M=64, N=2048, K=7168, dual=True)]


@pytest.mark.parametrize("call", SPLIT_CALLS)
def test_per_thread_stream_never_splits(call):
    """hipStreamPerThread is one handle for a stream of every thread: a workspace slot kept by the handle would be
    shared by calls that overlap."""
    assert plan(**call)[2] > 1
    assert plan(**call, stream=0x1000)[2] > 1
    assert plan(**call, stream=PER_THREAD)[2] == 1
    assert plan(**call, stream=PER_THREAD, captured=True)[2] == 1


def test_plan_rejects_bad_arguments():
    L = lib.load()
    v = ctypes.byref(ctypes.c_int())
    assert L.tlm_gemm_plan(1, 8, 8, lib.F16, 0, 0, None, 0, None, v, v) == -1
    assert L.tlm_gemm_plan(0, 8, 8, lib.F16, 0, 0, None, 0, v, v, v) == -1
    assert L.tlm_gemm_plan(1, 8, 8, lib.F32, 0, 0, None, 0, v, v, v) == -2
    assert L.tlm_gemm_plan(1, 8, 8, lib.F16, 0, 1, None, 0, v, v, v) == -2
    assert plan(4, 64, 60) == (0, 0, 1)


def test_captured_calls_that_may_keep_the_streams_workspace():
    """Two graphs captured on one stream may be replayed side by side unless they hold a call that keeps the
    stream's workspace: 16 rows or fewer of 16 bits, B^T of up to 8,192 columns (128 strips of 64) and row-major
    B of up to 16,384 (128 strips of 128) or more than 2,048 of k. No other call splits inside a capture."""
    for M in (1, 16):
        for K in (64, 256, 480, 512, 2048, 2056, 4096, 7168, 14336, 28672):
            for N in (64, 1000, 4096, 8192, 8200, 9000, 10496, 12288, 16384, 16392, 20480, 28672):
                for dt in (lib.F16, lib.BF16):
                    if N > 8192 or K <= 480:
                        assert plan(M, N, K, dt, captured=True)[2] == 1, (M, N, K)
                    if N > 16384 and K <= 2048:
                        assert plan(M, N, K, dt, trans_b=False, captured=True)[2] == 1, (M, N, K)
                assert plan(M, N, K, lib.F8E4M3, captured=True)[2] == 1
                assert plan(M, N, K, lib.BF16, dual=True, captured=True)[2] == 1
                for rows in (17, 64, 500):
                    for tb in (False, True):
                        assert plan(rows, N, K, trans_b=tb, captured=True)[2] == 1
    # those that kept it still split
    assert plan(16, 4096, 14336, captured=True)[2] > 1
    assert plan(16, 14336, 4096, trans_b=False, captured=True)[2] > 1
    assert plan(16, 4096, 4096, trans_b=False, captured=True)[2] > 1


@pytest.mark.parametrize("M", [1, 17, 32, 64, 100, 300])
@pytest.mark.parametrize("dt", [lib.F16, lib.F8E4M3])
def test_no_grid_above_the_launch_limit(M, dt):
    """A launch counts its threads in 32 bits; very wide calls that 256 x 256 tiles (or one thread per output)
    cover within it do not take smaller tiles that exceed it."""
    for N in (1 << 28, 1 << 29, (1 << 29) + 4096, 600_000_000, 1 << 30):
        for K in (16, 64, 128, 256, 512):
            rows, cols, ns = plan(M, N, K, dt)
            if 0 < rows and (rows, cols) != (256, 256):
                assert -(-M // rows) * -(-N // cols) * ns * 512 < 1 << 32, (N, K, rows, cols)
