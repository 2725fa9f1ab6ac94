"""GPU parity of the tiles between one decode step and a whole prompt batch (tlm_gemm_tile.h): every tile, whole
and split over K, with remainders on each axis (TILE_CASES, whose tiles test_gemm_plan.py asserts), and a list of
mixed shapes, against the fp64 product of the same inputs.

Tolerance: fp32 sums of K products with |partial sums| <= s err by at most K ulp(s) / 2; here the
relative 2-norm error stays below 4 sqrt(K) 2^-24, plus half an ulp of the output type (2^-9 bf16,
2^-12 fp16). fp8 above 16 rows: the fp8 matrix instruction drops low bits of its sums (measured 1.3e-5).
"""
import subprocess
import sys

import pytest
import torch

from conftest import PKG
from test_gemm_plan import SKINNY_CASES, TILE_CASES
from tilelang.jit.adapter.mi355x import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
ULP = {torch.float32: 0.0, torch.float16: 2.0 ** -12, torch.bfloat16: 2.0 ** -9}


def _rel(c, exp):
    return float((c.double() - exp).norm() / exp.norm())


def _run(M, N, K, dt, out, trans_b, seed=0, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed + M + N + K)
    a = torch.randn(M, K, generator=g, device=DEV).to(dt)
    b = torch.randn(*((N, K) if trans_b else (K, N)), generator=g, device=DEV).to(dt)
    c = torch.full((M, N), float("nan"), device=DEV).to(out)
    ops.gemm(a, b, c, trans_b=trans_b)
    bd = b.double()
    return c, a.double() @ (bd.T if trans_b else bd)


def _swiglu(M, N, K, dt, shift=0):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g, device=DEV).to(dt)
    bg, bu = ((torch.randn(N * K + 1, generator=g, device=DEV) * K ** -0.5).to(dt)[shift:shift + N * K].view(N, K)
              for _ in range(2))
    h = torch.full((M, N), float("nan"), dtype=dt, device=DEV)
    ops.gemm_swiglu(a, bg, bu, h)
    gate, up = a.double() @ bg.double().T, a.double() @ bu.double().T
    assert _rel(h, up * gate * torch.sigmoid(gate)) < 3 * ULP[dt]


OUTS = {"nn": [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32)],
        "nt": [(torch.float16, torch.float16), (torch.bfloat16, torch.float32)],
        "fp8": [(torch.float8_e4m3fn, torch.float32), (torch.float8_e5m2, torch.float32)],
        "dual": [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16)]}


@pytest.mark.parametrize("call,M,N,K,rows,cols,split", TILE_CASES)
def test_every_tile(call, M, N, K, rows, cols, split):
    for dt, out in OUTS[call]:
        if call == "dual":
            _swiglu(M, N, K, dt)
            continue
        c, exp = _run(M, N, K, dt, out, call != "nn")
        low_bits = 5e-5 if call == "fp8" and M > 16 else 0
        assert _rel(c, exp) < 4 * K ** 0.5 * 2.0 ** -24 + ULP[out] + low_bits


@pytest.mark.parametrize("M,N,K", SKINNY_CASES)
def test_decode_kernel(M, N, K):
    """One decode step on 32 MB of row-major B or more."""
    for dt, out in OUTS["nn"]:
        c, exp = _run(M, N, K, dt, out, False)
        assert _rel(c, exp) < 4 * K ** 0.5 * 2.0 ** -24 + ULP[out]


SHAPES = [(17, 64, 64), (32, 136, 200), (33, 64, 4096), (64, 2048, 1000), (65, 520, 2048),
          (128, 128, 7168), (129, 1032, 776), (200, 4096, 264), (257, 640, 4096), (500, 4096, 1024),
          (1000, 1024, 520), (1025, 4096, 128), (1, 2048, 2048), (16, 520, 72), (5, 28672, 256)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("dt,out,trans_b", [(torch.bfloat16, torch.bfloat16, False),
                                            (torch.float16, torch.float32, True),
                                            (torch.float16, torch.float16, True),
                                            (torch.bfloat16, torch.float32, False)])
def test_gemm_tiles(M, N, K, dt, out, trans_b):
    c, exp = _run(M, N, K, dt, out, trans_b)
    assert _rel(c, exp) < 4 * K ** 0.5 * 2.0 ** -24 + ULP[out]


@pytest.mark.parametrize("M,N,K", [(20, 77, 64), (70, 1001, 520), (130, 131, 2056)])
def test_gemm_tiles_bt_any_column_count(M, N, K):
    """B^T takes any N: the last columns leave as single values."""
    for out in (torch.float16, torch.float32):
        c, exp = _run(M, N, K, torch.float16, out, True)
        assert _rel(c, exp) < 4 * K ** 0.5 * 2.0 ** -24 + ULP[out]


@pytest.mark.parametrize("M,N,K", [(1, 512, 4096), (16, 1000, 528), (17, 64, 128), (64, 2048, 2000),
                                   (65, 520, 1024), (300, 1040, 784), (512, 4096, 512)])
@pytest.mark.parametrize("dt", [torch.float8_e4m3fn, torch.float8_e5m2])
def test_gemm_fp8_tiles(M, N, K, dt):
    """16 rows or fewer are multiplied as fp16: fp32 sums, no low bits dropped."""
    c, exp = _run(M, N, K, dt, torch.float32, True)
    assert _rel(c, exp) < 4 * K ** 0.5 * 2.0 ** -24 + (0 if M <= 16 else 5e-5)


def test_gemm_fp8_few_rows_keep_specials():
    """inf, NaN and subnormals of both formats through the fp16 product."""
    for dt in (torch.float8_e4m3fn, torch.float8_e5m2):
        a = torch.eye(16, 256, device=DEV).to(dt)
        codes = torch.arange(256, dtype=torch.uint8, device=DEV).view(1, 256).repeat(64, 1)
        b = torch.zeros(64, 256, dtype=dt, device=DEV)
        for i in range(16):  # column k of B^T holds 64 consecutive codes, one k per row of A
            b.view(torch.uint8)[:, i] = codes[0, (16 * torch.arange(64, device=DEV) + i) % 256]
        c = torch.empty(16, 64, device=DEV)
        ops.gemm(a, b, c, trans_b=True)
        exp = b.float()[:, :16].T
        finite = torch.isfinite(b.float()).all(1)  # 0 * inf = NaN in a row with a special
        assert torch.equal(c[:, finite], exp[:, finite])
        assert not torch.isfinite(c[:, ~finite]).any()


def test_gemm_split_tiles_repeat_and_replay():
    """A split call gives the same bits again, with other calls between; captured, it runs unsplit, so two graphs
    of one capture stream may replay at the same time on two streams."""
    g = torch.Generator(device=DEV).manual_seed(3)
    a = [torch.randn(64, 4096, generator=g, device=DEV).half() for _ in range(2)]
    b = torch.randn(1024, 4096, generator=g, device=DEV).half()
    eager = []
    for x in a:
        for _ in range(2):
            c = torch.empty(64, 1024, device=DEV)
            ops.gemm(x, b, c, trans_b=True)
            eager.append(c)
            ops.gemm(x[:20], b[:200], torch.empty(20, 200, device=DEV), trans_b=True)
    assert torch.equal(eager[0], eager[1]) and torch.equal(eager[2], eager[3])
    side = torch.cuda.Stream()
    outs, graphs = [torch.zeros(64, 1024, device=DEV) for _ in a], []
    side.wait_stream(torch.cuda.current_stream())
    for x, c in zip(a, outs):
        gr = torch.cuda.CUDAGraph()
        with torch.cuda.graph(gr, stream=side):
            ops.gemm(x, b, c, trans_b=True)
        graphs.append(gr)
    streams = [torch.cuda.Stream() for _ in a]
    torch.cuda.synchronize()
    for _ in range(3):
        for gr, st in zip(graphs, streams):
            with torch.cuda.stream(st):
                gr.replay()
        torch.cuda.synchronize()
        for c, e in zip(outs, (eager[0], eager[2])):
            assert _rel(c, e.double()) < 4 * 64 * 2.0 ** -24
        for c in outs:
            c.zero_()
        torch.cuda.synchronize()


@pytest.mark.parametrize("M,N,K", [(1, 64, 72), (16, 2048, 1024), (33, 1000, 520), (64, 2048, 7168),
                                   (100, 76, 256), (129, 1408, 2048), (520, 520, 264), (4, 64, 60),
                                   (4096, 4096, 128)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_gemm_swiglu(M, N, K, dt):
    """up * silu(gate) of two products, each rounded to the dtype first; K 60 and a weight that is not
    16-byte aligned run as three calls. Three roundings of half an ulp each."""
    for shift in (0, 1) if M <= 33 else (0,):
        _swiglu(M, N, K, dt, shift)


DECODE_SLOTS = """
import torch
from tilelang.jit.adapter.mi355x import ops
g = torch.Generator(device="cuda").manual_seed(5)
x = torch.randn(64, 4096, generator=g, device="cuda").half()
w = torch.randn(2048, 4096, generator=g, device="cuda").half()
streams = [torch.cuda.Stream() for _ in range(4)]
torch.cuda.synchronize()
for st in streams:  # split calls of 64 rows own a workspace each
    with torch.cuda.stream(st):
        ops.gemm(x, w, torch.empty(64, 2048, device="cuda"), trans_b=True)
torch.cuda.synchronize()
res = []
for i in range(6):
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        res.append(ops.gemm(x[:16], w, torch.empty(16, 2048, device="cuda"), trans_b=True))
    streams.append(st)  # kept: a handle is not used again
torch.cuda.synchronize()
print("EQUAL", [bool(torch.equal(r, res[0])) for r in res])
"""


def test_decode_calls_keep_their_workspaces_beside_larger_calls():
    """Streams that run split calls of more than 16 rows take none of the four slots of decode steps: four further
    streams still split them (the bits of one call), the streams after those run unsplit (others)."""
    r = subprocess.run([sys.executable, "-c", DECODE_SLOTS], capture_output=True, text=True, timeout=100,
                       cwd=PKG)
    assert r.returncode == 0, r.stderr[-2000:]
    assert "EQUAL [True, True, True, True, False, False]" in r.stdout, r.stdout
