"""GPU parity of the D 128 attention kernel's tilings: 128-query workgroups (one or a pair of
causal tiles) and 256-query pairs, at sequence lengths on both sides of a query tile, a 64-key tile
and the choices between them, against fp64 softmax attention.

Tolerance: P is rounded to the 16-bit type before P V (relative 2^-9 bf16, 2^-12 fp16 per weight,
averaged over the keys) and the output once more: 2-norm error within two such ulps.
"""
import pytest
import torch

from tilelang.jit.adapter.mi355x import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _exact(q, k, v, scale, causal):
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    off = k.shape[1] - q.shape[1]
    for b in range(q.shape[0]):
        for h in range(q.shape[2]):
            kh, vh = (x[b, :, h // (q.shape[2] // x.shape[2])].double() for x in (k, v))
            s = q[b, :, h].double() @ kh.T * scale
            if causal:
                s.masked_fill_(torch.ones_like(s, dtype=torch.bool).triu_(1 + off), -torch.inf)
            out[b, :, h] = torch.softmax(s, 1).nan_to_num(0.0) @ vh
    return out


def _check(o, exp, dt):
    assert float((o.double() - exp).norm() / exp.norm()) < 2 * (2.0 ** -9 if dt == torch.bfloat16 else
                                                              2.0 ** -12)


@pytest.mark.parametrize("S,H,Hkv", [(1, 8, 8), (16, 8, 2), (127, 16, 4), (128, 8, 8), (129, 32, 8),
                                     (300, 64, 4), (513, 8, 1), (1111, 32, 8), (1030, 16, 16)])
@pytest.mark.parametrize("causal", [True, False])
def test_short_sequences(S, H, Hkv, causal):
    g = torch.Generator(device=DEV).manual_seed(S + H)
    for dt in (torch.bfloat16, torch.float16):
        q, k, v = (torch.randn(1, S, n, 128, generator=g, device=DEV).to(dt) for n in (H, Hkv, Hkv))
        o = torch.full_like(q, float("nan"))
        ops.flash_attn_fwd(q, k, v, o, causal, 128 ** -0.5)
        _check(o, _exact(q, k, v, 128 ** -0.5, causal), dt)


@pytest.mark.parametrize("Sq,Sk", [(100, 900), (257, 300), (300, 257), (700, 1500)])
def test_causal_offsets_head_major(Sq, Sk):
    """Causal with more (or fewer) keys than queries, score jumps that send tiles through the redo."""
    g = torch.Generator(device=DEV).manual_seed(Sq + Sk)
    q = torch.randn(2, 4, Sq, 128, generator=g, device=DEV).half()
    k = torch.randn(2, 4, Sk, 128, generator=g, device=DEV).half()
    k[:, :, Sk // 2:] *= 6
    v = torch.randn(2, 4, Sk, 128, generator=g, device=DEV).half()
    o = torch.full_like(q, float("nan"))
    ops.flash_attn_bhsd_fwd(q, k, v, o, True, 128 ** -0.5)
    exp = _exact(*(x.transpose(1, 2) for x in (q, k, v)), 128 ** -0.5, True).transpose(1, 2)
    _check(o, exp, torch.float16)


def test_ragged_batch_of_short_sequences():
    lens = [1, 130, 64, 0, 257, 16]
    g = torch.Generator(device=DEV).manual_seed(9)
    cu = torch.tensor([0] + lens, dtype=torch.int32).cumsum(0).to(torch.int32).to(DEV)
    q, k, v = (torch.randn(sum(lens), n, 128, generator=g, device=DEV).bfloat16() for n in (8, 2, 2))
    for causal in (False, True):
        o = torch.full_like(q, float("nan"))
        ops.flash_attn_varlen_fwd(q, k, v, cu, cu, max(lens), o, causal, 128 ** -0.5)
        at = 0
        for n in lens:
            if n:
                r = slice(at, at + n)
                _check(o[r], _exact(q[None, r], k[None, r], v[None, r], 128 ** -0.5, causal)[0],
                       torch.bfloat16)
            at += n


@pytest.mark.parametrize("B,H,Sq,Skv,ns", [(2, 8, 1, 512, 2), (2, 8, 16, 2048, 4), (2, 8, 128, 1024, 1),
                                           (2, 8, 129, 512, 2), (2, 8, 200, 4096, 8), (3, 3, 40, 2000, 5),
                                           (1, 1, 128, 4096, 1), (1, 5, 300, 1280, 4),
                                           (4, 32, 64, 2304, 1), (4, 32, 1, 2200, 1)])
def test_split_inference(B, H, Sq, Skv, ns):
    """Short query blocks over a key split, parts on both sides of 1,024 keys; fp32 parts merged, lse and partials
    stored in fp16."""
    g = torch.Generator(device=DEV).manual_seed(Sq + Skv)
    q = torch.randn(B, Sq, H, 128, generator=g, device=DEV).half()
    k, v = (torch.randn(B, Skv, H, 128, generator=g, device=DEV).half() for _ in range(2))
    lse = torch.empty(B, H, ns, Sq, dtype=torch.float16, device=DEV)
    part = torch.empty(B, Sq, H, ns, 128, dtype=torch.float16, device=DEV)
    o = torch.empty_like(q)
    ws = torch.empty(ops.flash_attn_splitkv_workspace_bytes(B, Sq, Skv, H, 128, ns),
                     dtype=torch.uint8, device=DEV)
    ops.flash_attn_splitkv_fwd(q, k, v, lse, part, o, ns, 128 ** -0.5, ws)
    per = Skv // ns
    for s in range(ns):
        exp = _exact(q, k[:, s * per:(s + 1) * per], v[:, s * per:(s + 1) * per], 128 ** -0.5, False)
        _check(part[:, :, :, s], exp, torch.float16)
    # the weights 2^lse carry lse's fp16 rounding: half an ulp of ~16 is 2^-7 ln 2 = 0.5%
    exp = _exact(q, k, v, 128 ** -0.5, False)
    assert float((o.double() - exp).norm() / exp.norm()) < 6e-3
