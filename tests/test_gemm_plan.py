"""Which kernel, tile and split a GEMM call takes (tlm_gemm_plan: host only, no GPU needed)."""
import ctypes

import pytest

from tilelang.jit.adapter.mi355x import lib

PER_THREAD = 2  # hipStreamPerThread


def plan(M, N, K, dt=lib.F16, trans_b=True, dual=False, stream=None, captured=False):
    out = [ctypes.c_int() for _ in range(3)]
    lib.call("tlm_gemm_plan", M, N, K, dt, int(trans_b), int(dual), stream, int(captured),
             *(ctypes.byref(v) for v in out))
    return tuple(v.value for v in out)


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
