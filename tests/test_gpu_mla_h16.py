"""GPU parity of the balanced MLA decode over a 16-bit cache: sequences shorter and longer than a 32-token tile,
empty ones, several ranges per sequence and several sequences per range, page sizes on both sides of a tile,
head blocks, workspaces that hold few slots, scores of -inf, and score jumps that move the running maximum.

Reference: fp64 attention over the gathered rows. Tolerance: P is rounded to the 16-bit type (2^-9
bf16, 2^-12 fp16 relative per weight) and the output once: 2-norm error within two such ulps.
"""
import pytest
import torch

from tilelang.jit.adapter.mi355x import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
DV, DPE = 512, 64


def _case(lens, H, page, dt, seed=0, ns=4, fused=True, jump=None, bad_page=False, edit=None, ws_bytes=None):
    g = torch.Generator(device=DEV).manual_seed(seed + sum(lens) + H)
    B = len(lens)
    pages = max(1, -(-max(lens) // page))
    rows = torch.randn(B * pages * page, DV + DPE, generator=g, device=DEV).to(dt)
    if jump is not None:  # a few tokens far above the rest
        rows[jump::97] *= 8
    table = torch.randperm(B * pages, generator=g, device=DEV).view(B, pages).to(torch.int32)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    q = torch.randn(B, H, DV + DPE, generator=g, device=DEV).to(dt)
    scale = (DV + DPE) ** -0.5
    at = torch.arange(pages * page, device=DEV)
    exp = torch.zeros(B, H, DV, dtype=torch.float64, device=DEV)
    if edit is not None:  # edit(cache rows of the sequence's tokens, queries of the sequence)
        for b, n in enumerate(lens):
            row = table[b].long()[at[:n] // page] * page + at[:n] % page
            own = rows[row]
            edit(own, q[b])
            rows[row] = own
    if bad_page:
        table[0, 0] = B * pages + 7
    for b, n in enumerate(lens):
        if n:
            row = table[b].long()[at[:n] // page] * page + at[:n] % page
            ok = row < rows.shape[0]
            kv = rows[row * ok].double() * ok[:, None]
            exp[b] = torch.softmax(q[b].double() @ kv.T * scale, 1) @ kv[:, :DV]
    kv, kpe = rows[:, :DV], rows[:, DV:]
    if not fused:
        kv, kpe = kv.contiguous(), kpe.contiguous()
    out = torch.full((B, H, DV), float("nan"), dtype=dt, device=DEV)
    ws = torch.empty(ws_bytes or ops.mla_workspace_bytes(B, H, DV, ns), dtype=torch.uint8, device=DEV)
    ops.mla_decode(q[..., :DV], q[..., DV:], kv, kpe, table, sl, out, ws, page, ns, scale)
    return out, exp


def _check(out, exp, lens, dt):
    tol = 2 * (2.0 ** -9 if dt == torch.bfloat16 else 2.0 ** -12)
    for b, n in enumerate(lens):
        if n == 0:
            assert torch.equal(out[b], torch.zeros_like(out[b]))
        else:
            assert float((out[b].double() - exp[b]).norm() / exp[b].norm()) < tol, (b, n)


@pytest.mark.parametrize("lens", [[1], [64], [65, 0, 63], [3000], [500, 4000, 1, 128, 0, 2000, 77, 640],
                                  [33] * 40, [0, 0, 5], [1300] * 16,
                                  [31, 32, 33, 511, 512, 513, 16384]])
@pytest.mark.parametrize("H,page,dt", [(128, 64, torch.bfloat16), (64, 16, torch.float16),
                                       (192, 100, torch.bfloat16), (256, 128, torch.float16)])
def test_lengths_and_heads(lens, H, page, dt):
    out, exp = _case(lens, H, page, dt)
    _check(out, exp, lens, dt)


@pytest.mark.parametrize("ns", [1, 2, 16, 64])
@pytest.mark.parametrize("lens", [[700, 90, 2000], [900], [300] * 20])
def test_workspace_sizes(ns, lens):
    """num_split only sizes the workspace, and with it the number of ranges: fewer and more than sequences."""
    for dt in (torch.bfloat16, torch.float16):
        out, exp = _case(lens, 128, 64, dt, ns=ns, fused=False)
        _check(out, exp, lens, dt)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_score_jumps(dt):
    """Tiles far above the running maximum of the ones before them go through the rescale."""
    lens = [1000, 64, 300]
    for jump in (0, 50, 96):
        out, exp = _case(lens, 128, 64, dt, jump=jump, ns=2)
        _check(out, exp, lens, dt)


def test_rows_outside_the_pool_read_as_zeros():
    lens = [200, 150]
    out, exp = _case(lens, 128, 64, torch.bfloat16, bad_page=True)
    _check(out, exp, lens, torch.bfloat16)


@pytest.mark.parametrize("B,H", [(65, 128), (300, 192), (1100, 64)])
def test_large_batches(B, H):
    """The combine takes several heads per wave; empty, whole and cut sequences among them."""
    lens = [(37 * b) % 90 for b in range(B)]
    lens[B // 2] = 1500
    out, exp = _case(lens, H, 16, torch.bfloat16, ns=1)
    _check(out, exp, lens, torch.bfloat16)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("mask", ["-inf", "lowest"])
@pytest.mark.parametrize("lens", [[20000, 100, 3000], [400] * 150])
def test_masked_prefix(lens, mask, dt):
    """Tokens masked through a rope dimension: the first tiles of a sequence score -inf for every head, or the
    type's lowest value times q (-inf in bf16) for every head or one. The others score about 0, or 150
    below it, or one of them far above the rest. Pieces of several tiles, cut sequences and whole ones."""
    value = float("-inf") if mask == "-inf" else torch.finfo(dt).min
    scale = (DV + DPE) ** -0.5
    for masked in (40, 320):
        for heads in (slice(None), slice(5, 6)) if mask == "lowest" else (slice(None),):
            for level, jump in ((0, 0), (-150, 0), (0, 24)):
                def edit(own, q):
                    n = own.shape[0]
                    if n <= masked:
                        return
                    own[:, DV] = 0
                    own[:masked, DV] = value
                    q[:, DV] = 0
                    q[heads, DV] = 16
                    own[:, DV + 1] = level
                    own[n - 3, DV + 1] = level + jump
                    q[:, DV + 1] = 1 / scale
                out, exp = _case(lens, 128, 64, dt, edit=edit)
                _check(out, exp, lens, dt)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("at", [0, 33, 100, 15000])
def test_largest_weight_is_exact(at, dt):
    """A token 2^34 above the rest wherever it stands in its piece: its weight is 1 and the output is its row, to
    the others' 2^-20."""
    lens = [20000] * 2

    def edit(own, q):
        own[:, DV] = 0
        own[at, DV] = 24  # e^24 ahead of scores of about randn
        q[:, DV] = (DV + DPE) ** 0.5
    out, exp = _case(lens, 128, 64, dt, edit=edit)
    err = float((out.double() - exp).norm() / exp.norm())
    assert err < 2.0 ** -14, err


@pytest.mark.parametrize("lens,H,ns", [([5000], 64, 64), ([7000], 192, 64), ([900, 2000], 64, 16)])
def test_result_does_not_depend_on_a_larger_workspace(lens, H, ns):
    """The ranges follow from the call, so a workspace that an earlier, larger call left behind gives the same
    bits."""
    need = ops.mla_workspace_bytes(len(lens), H, DV, ns)
    runs = [_case(lens, H, 64, torch.bfloat16, ns=ns, ws_bytes=b)[0] for b in (need, 2 * need, 128 << 20)]
    assert torch.equal(runs[1], runs[0]) and torch.equal(runs[2], runs[0])
