"""Performance cases: the work that programs built on this framework hand to it, each as one call of a
kernel that ``tilelang.compile`` returned, with every parameter passed (outputs written in place).

A case is a dict of plain values; ``kind`` names the program family. The families are those a
transformer layer is made of (norm, RoPE, dense projections, the gated MLP, attention in
prefill, attention over a long cache, latent-attention decode), at the token counts of one
decode step, of a chunk of a prompt, and of whole prompts. Dense weights are randn / sqrt(K) and
activations randn, as a normalised layer sees them.
"""
import functools
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "tilelang-tpu_amd"))

import tilelang  # noqa: E402
from tilelang.testing import programs  # noqa: E402

DT = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32,
      "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
SIZE = {"float16": 2, "bfloat16": 2, "float32": 4, "e4m3": 1, "e5m2": 1}
EPS = 1e-6
DV, DPE, PAGE = 512, 64, 64  # latent and rope dims of the cache rows, tokens per page


def listed():
    return [
        # one decode step of 16 sequences: the smallest call, launch and host cost
        dict(name="rmsnorm_decode", kind="rmsnorm", dtype="float16", rows=16, cols=4096),
        # q and k of a 2,000-token chunk, grouped-query heads
        dict(name="rope_chunk", kind="rope", dtype="bfloat16", tokens=2000, hq=32, hk=8, dim=128),
        # a projection in one decode step: the weight stream is everything
        dict(name="gemm_decode", kind="gemm", dtype="float16", M=16, N=14336, K=4096, trans_b=False),
        # the same layer for a ragged chunk of prompt tokens
        dict(name="gemm_chunk", kind="gemm", dtype="bfloat16", M=500, N=4096, K=4096, trans_b=False),
        # a whole prompt batch (the benchmark's headline size)
        dict(name="gemm_prefill", kind="gemm", dtype="float16", M=4096, N=4096, K=4096,
             trans_b=False),
        # quantised projection of a chunk, fp32 result
        dict(name="gemm_fp8_chunk", kind="gemm_fp8", dtype="e4m3", out="float32", M=512, N=4096,
             K=4096),
        # gated MLP (gate, up, SwiGLU, down) of a decode batch at the MLP program's sizes
        dict(name="mlp_decode", kind="mlp", dtype="bfloat16", M=64, hidden=7168, inter=2048),
        # one prompt of odd length, causal, four query heads per K/V head
        dict(name="fa_prompt", kind="fa", dtype="bfloat16", B=1, S=1111, H=32, groups=4, D=128,
             causal=True),
        # a batch of prompts of unequal length without padding: the largest call
        dict(name="fa_ragged_batch", kind="fa_varlen", dtype="float16", B=16, lo=538, hi=3789, H=32,
             groups=1, D=128),
        # a block of queries over a long cache, split over its keys (the inference example's size)
        dict(name="fa_inference", kind="fa_split", dtype="float16", B=1, Sq=128, Skv=8192, H=32,
             D=128, splits=4),
        # latent attention decode, 16-bit paged cache, a few sequences in flight
        dict(name="mla_decode_bf16", kind="mla", dtype="bfloat16", kv="bfloat16", B=8, lo=500,
             hi=4000, H=128),
        # the same over an fp8 cache at a full serving batch
        dict(name="mla_decode_fp8", kind="mla", dtype="bfloat16", kv="e4m3", B=64, lo=1024, hi=8192,
             H=128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rmsnorm", "rope", "gemm", "gemm", "gemm", "gemm_fp8", "mlp", "fa", "fa",
                       "fa_varlen", "fa_split", "mla", "mla"])
    h16 = rng.choice(["float16", "bfloat16"])
    if kind == "rmsnorm":
        return dict(kind=kind, dtype=rng.choice([h16, h16, "float32"]), rows=_log(rng, 1, 8192),
                    cols=rng.choice([1000, 2048, 4096, 5120, 7168, 8192]))
    if kind == "rope":
        hq, hk = rng.choice([(32, 32), (32, 8), (64, 8), (16, 2)])
        return dict(kind=kind, dtype=h16, tokens=_log(rng, 1, 8192), hq=hq, hk=hk,
                    dim=rng.choice([64, 128]))
    if kind in ("gemm", "gemm_fp8"):
        step = 8 if kind == "gemm" else 16
        while True:  # any token count, layer widths a multiple of the vector width
            M = _log(rng, 1, 4096)
            N, K = (step * (_log(rng, 512, 14336) // step) for _ in range(2))
            if M * N * K <= 4096 ** 3:
                break
        if kind == "gemm":
            return dict(kind=kind, dtype=h16, M=M, N=N, K=K, trans_b=rng.random() < 0.5)
        dt = rng.choice(["e4m3", "e4m3", "e5m2"])
        return dict(kind=kind, dtype=dt, out=rng.choice(["float32", "bfloat16"]), M=M, N=N, K=K)
    if kind == "mlp":
        hidden, inter = rng.choice([(7168, 2048), (2048, 1408), (4096, 11008)])
        return dict(kind=kind, dtype="bfloat16", M=_log(rng, 1, 1024), hidden=hidden, inter=inter)
    if kind == "fa":
        H, groups = rng.choice([(32, 1), (32, 4), (64, 16), (16, 1)])
        return dict(kind=kind, dtype=h16, B=rng.choice([1, 1, 2, 4]), S=_log(rng, 64, 4096), H=H,
                    groups=groups, D=rng.choice([128, 128, 64]), causal=rng.random() < 0.75)
    if kind == "fa_varlen":
        hi = _log(rng, 64, 3789)
        return dict(kind=kind, dtype=h16, B=rng.randint(2, 16), lo=rng.randint(1, hi), hi=hi, H=32,
                    groups=rng.choice([1, 4]), D=128)
    if kind == "fa_split":
        splits = rng.choice([1, 2, 4, 8])
        return dict(kind=kind, dtype=h16, B=rng.choice([1, 2, 4]), Sq=_log(rng, 1, 256),
                    Skv=64 * splits * _log(rng, 4, 128 // splits), H=32, D=128, splits=splits)
    hi = _log(rng, 128, 8192)
    kv = rng.choice(["e4m3", h16])
    return dict(kind=kind, dtype=h16, kv=kv, B=_log(rng, 1, 64 if kv == "e4m3" else 16),
                lo=rng.randint(1, hi), hi=hi, H=rng.choice([64, 128]))


def _lens(c):
    """The batch's sequence lengths, spread evenly over lo .. hi (their order comes with the seed)."""
    n = c["B"]
    return [c["hi"] - (c["hi"] - c["lo"]) * i // max(1, n - 1) for i in range(n)]


def _slots(c):
    """Tokens a sequence's page table can hold."""
    return -(-c["hi"] // PAGE) * PAGE


@functools.lru_cache(maxsize=None)
def _kernel(items):
    c = dict(items)
    k, dt = c["kind"], c["dtype"]
    if k == "rmsnorm":
        f = programs.rms_norm(c["rows"], c["cols"], 1, dt, eps=EPS, with_weight=True)
    elif k == "rope":
        f = programs.rope_qk(c["tokens"], c["hq"], c["hk"], c["dim"], dtype=dt)
    elif k == "gemm":
        f = programs.matmul(c["M"], c["N"], c["K"], 128, 128, 64, dtype=dt, out_dtype=dt,
                            trans_b=c["trans_b"])
    elif k == "gemm_fp8":
        f = programs.matmul_fp8(c["M"], c["N"], c["K"], dtype=c["dtype"] + "_float8",
                                out_dtype=c["out"])
    elif k == "mlp":
        f = programs.deepseek_mlp(64, c["hidden"], c["inter"], c["M"], c["hidden"], c["inter"], dt)
    elif k == "fa":
        f = programs.flashattn_gqa(c["B"], c["H"], c["S"], c["D"], c["causal"], groups=c["groups"],
                                   dtype=dt)
    elif k == "fa_varlen":
        n = sum(_lens(c))
        f = programs.flashattn_varlen(c["B"], n, n, c["H"], c["D"], groups=c["groups"], dtype=dt)
    elif k == "fa_split":
        f = programs.mha_inference(c["B"], c["H"], c["Sq"], c["Skv"], c["D"],
                                   num_split=c["splits"], dtype=dt)
    else:
        kv = {"e4m3": "float8_e4m3"}.get(c["kv"], c["kv"])
        f = programs.mla_decode(c["B"], c["H"], 1, _slots(c), DV, DPE, PAGE, 64, 1, PAGE, dtype=dt,
                                kv_dtype=kv)
    return tilelang.compile(f, target="mi355x")


def _inputs(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def randn(*shape, scale=1.0, dtype=None):
        return torch.randn(*shape, generator=g, device="cuda").mul_(scale).to(dtype or DT[c["dtype"]])

    def perm(n):
        return torch.randperm(n, generator=g, device="cuda")

    k = c["kind"]
    if k == "rmsnorm":
        return dict(x=randn(c["rows"], c["cols"]), w=1 + randn(c["cols"], scale=0.1))
    if k == "rope":
        t, d = c["tokens"], c["dim"]
        inv = 10000.0 ** (-torch.arange(0, d, 2, device="cuda", dtype=torch.float64) / d)
        a = torch.arange(t, device="cuda", dtype=torch.float64)[:, None] * inv
        a = a.repeat_interleave(2, dim=1)
        return dict(q=randn(t, c["hq"], d), k=randn(t, c["hk"], d), cos=a.cos().to(DT[c["dtype"]]),
                    sin=a.sin().to(DT[c["dtype"]]))
    if k == "gemm":
        shape = (c["N"], c["K"]) if c["trans_b"] else (c["K"], c["N"])
        return dict(a=randn(c["M"], c["K"]), b=randn(*shape, scale=c["K"] ** -0.5))
    if k == "gemm_fp8":
        return dict(a=randn(c["M"], c["K"]), b=randn(c["N"], c["K"]))
    if k == "mlp":
        h, i = c["hidden"], c["inter"]
        return dict(x=randn(c["M"], h), wg=randn(i, h, scale=h ** -0.5),
                    wu=randn(i, h, scale=h ** -0.5), wd=randn(h, i, scale=i ** -0.5))
    if k == "fa":
        kv = (c["B"], c["S"], c["H"] // c["groups"], c["D"])
        return dict(q=randn(c["B"], c["S"], c["H"], c["D"]), k=randn(*kv), v=randn(*kv))
    if k == "fa_varlen":
        lens = torch.tensor(_lens(c), device="cuda")[perm(c["B"])]
        cu = torch.nn.functional.pad(lens.cumsum(0), (1, 0)).to(torch.int32)
        kv = (sum(_lens(c)), c["H"] // c["groups"], c["D"])
        return dict(q=randn(sum(_lens(c)), c["H"], c["D"]), k=randn(*kv), v=randn(*kv), cu=cu)
    if k == "fa_split":
        kv = (c["B"], c["Skv"], c["H"], c["D"])
        return dict(q=randn(c["B"], c["Sq"], c["H"], c["D"]), k=randn(*kv), v=randn(*kv))
    # paged latent cache: fused 576-wide rows, pages handed out in random order
    B, pages = c["B"], _slots(c) // PAGE
    lens = torch.tensor(_lens(c), device="cuda", dtype=torch.int32)[perm(B)]
    table = perm(B * pages).view(B, pages).to(torch.int32)
    fp8 = c["kv"] == "e4m3"
    scale = 5.0 / 448.0
    rows = randn(B * pages * PAGE, DV + DPE, scale=1 / scale if fp8 else 1.0, dtype=torch.bfloat16)
    rows = (rows.clamp_(-448, 448) if fp8 else rows).to(DT[c["kv"]])
    d = dict(q=randn(B, c["H"], DV + DPE), kv=rows, table=table, lens=lens)
    if fp8:
        d["kv_scale"] = torch.tensor([scale], device="cuda")
    return d


def prepare(case, seed):
    c = {k: v for k, v in case.items() if k != "name"}
    t = _inputs(c, seed)
    k, dt = c["kind"], DT[c["dtype"]]

    def new(*shape, dtype=dt):
        return torch.empty(*shape, dtype=dtype, device="cuda")

    if k == "rmsnorm":
        out = [torch.empty_like(t["x"])]
        args = [t["x"], t["w"], *out]
    elif k == "rope":
        out = [torch.empty_like(t["q"]), torch.empty_like(t["k"])]
        args = [t["q"], t["k"], t["cos"], t["sin"], *out]
    elif k == "gemm":
        out = [new(c["M"], c["N"])]
        args = [t["a"], t["b"], *out]
    elif k == "gemm_fp8":
        out = [new(c["M"], c["N"], dtype=DT[c["out"]])]
        args = [t["a"], t["b"], *out]
    elif k == "mlp":
        out = [torch.empty_like(t["x"])]
        args = [*out, t["x"], t["wg"], t["wu"], t["wd"]]
    elif k == "fa":
        out = [torch.empty_like(t["q"])]
        args = [t["q"], t["k"], t["v"], *out]
    elif k == "fa_varlen":
        out = [torch.empty_like(t["q"])]
        args = [t["q"], t["k"], t["v"], t["cu"], t["cu"], c["hi"], *out]
    elif k == "fa_split":
        B, Sq, H, D, ns = c["B"], c["Sq"], c["H"], c["D"], c["splits"]
        out = [new(B, H, ns, Sq), new(B, Sq, H, ns, D), new(B, Sq, H, D)]
        args = [t["q"], t["k"], t["v"], *out]
    else:
        B, H = c["B"], c["H"]
        fp8 = c["kv"] == "e4m3"
        pdt = torch.float32 if fp8 else dt
        rows = t["kv"].unsqueeze(1)
        out = [new(B, H, DV)]
        # the one-split program's partials are parameters that it does not need to keep
        args = [t["q"][..., :DV], t["q"][..., DV:], rows[..., :DV], rows[..., DV:], t["table"],
                t["lens"], new(B, H, 1, dtype=pdt), new(B, H, 1, DV, dtype=pdt), *out]
        if fp8:
            args.append(t["kv_scale"])
    return dict(kernel=_kernel(tuple(sorted(c.items()))), args=args, out=out)


def run(state):
    state["kernel"](*state["args"])
    return state["out"]


def work(case):
    c, k = case, case["kind"]
    es = SIZE[c["dtype"]]
    if k == "rmsnorm":
        n = c["rows"] * c["cols"]
        return {"bytes": es * (2 * n + c["cols"]), "flops": 4 * n}
    if k == "rope":
        n = c["tokens"] * (c["hq"] + c["hk"]) * c["dim"]
        return {"bytes": es * (2 * n + 2 * c["tokens"] * c["dim"]), "flops": 3 * n}
    if k in ("gemm", "gemm_fp8"):
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": es * (M * K + N * K) + SIZE[c.get("out", c["dtype"])] * M * N,
                "flops": 2 * M * N * K}
    if k == "mlp":
        M, h, i = c["M"], c["hidden"], c["inter"]
        return {"bytes": es * (3 * h * i + 2 * M * h), "flops": 6 * M * h * i + 5 * M * i}
    if k == "fa":
        B, S, H, D = c["B"], c["S"], c["H"], c["D"]
        pairs = S * (S + 1) // 2 if c["causal"] else S * S
        return {"bytes": es * B * S * D * 2 * (H + H // c["groups"]), "flops": 4 * B * H * D * pairs}
    if k == "fa_varlen":
        n, H, D = sum(_lens(c)), c["H"], c["D"]
        return {"bytes": es * n * D * 2 * (H + H // c["groups"]),
                "flops": 4 * H * D * sum(x * x for x in _lens(c))}
    if k == "fa_split":
        B, Sq, Skv, H, D, ns = (c[x] for x in ("B", "Sq", "Skv", "H", "D", "splits"))
        return {"bytes": es * B * H * (D * (2 * Sq + 2 * Skv + Sq * ns) + ns * Sq),
                "flops": 4 * B * H * Sq * Skv * D}
    n, B, H = sum(_lens(c)), c["B"], c["H"]
    return {"bytes": SIZE[c["kv"]] * n * (DV + DPE) + es * B * H * (2 * DV + DPE)
            + 4 * B * (_slots(c) // PAGE + 1), "flops": 2 * n * H * (2 * DV + DPE)}


def tolerance(case):
    k, dt = case["kind"], case["dtype"]
    if k == "gemm_fp8" and case["out"] == "float32":
        # the fp8 products' sums are 1.3e-5 off the 64-bit ones at K 4096
        return {"rel": 5e-5}
    if k == "fa_split":
        # the program stores log2 sum-exps of ~13 in 16 bits and weighs its partials by them: 1.4e-3 off
        # the 64-bit attention in fp16
        return {"rel": 5e-3 if dt == "float16" else 0.03}
    if k == "mla" and case["kv"] == "e4m3":
        # weights rounded to 8 bits on both sides, as the fp8 decode does
        return {"rel": 0.03, "max": 0.6}
    if dt == "float32":
        return {"rel": 1e-6}
    return {"rel": 8e-3 if dt == "bfloat16" or case.get("out") == "bfloat16" else 1e-3}


def _attend(q, k, v, scale, causal=False):
    """softmax(scale q k^T) v per head in float64; q [n, H, D], k, v [m, Hk, D]: (out, log2 sum-exp)."""
    H, groups = q.shape[1], q.shape[1] // k.shape[1]
    out = torch.empty(q.shape[0], H, v.shape[2], dtype=torch.float64, device=q.device)
    lse = torch.empty(H, q.shape[0], dtype=torch.float64, device=q.device)
    for h in range(H):
        s = q[:, h].double() @ k[:, h // groups].double().T
        s *= scale
        if causal:
            s.masked_fill_(torch.ones_like(s, dtype=torch.bool).triu_(1), -math.inf)
        lse[h] = s.logsumexp(1)
        out[:, h] = (s - lse[h][:, None]).exp_() @ v[:, h // groups].double()
    return out, lse / math.log(2.0)


def exact(case, seed):
    c = {k: v for k, v in case.items() if k != "name"}
    t, k = _inputs(c, seed), c["kind"]
    if k == "rmsnorm":
        x = t["x"].double()
        return [x * (x.square().mean(1, keepdim=True) + EPS).rsqrt() * t["w"].double()]
    if k == "rope":
        cos, sin = t["cos"].double()[:, None], t["sin"].double()[:, None]

        def turn(x):
            x = x.double()
            y = torch.stack((-x[..., 1::2], x[..., ::2]), -1).flatten(-2)
            return x * cos + y * sin

        return [turn(t["q"]), turn(t["k"])]
    if k in ("gemm", "gemm_fp8"):
        b = t["b"].double()
        return [t["a"].double() @ (b if k == "gemm" and not c["trans_b"] else b.T)]
    if k == "mlp":
        x = t["x"].double()
        gate, up = x @ t["wg"].double().T, x @ t["wu"].double().T
        return [(gate * torch.sigmoid(gate) * up) @ t["wd"].double().T]
    if k == "fa":
        return [torch.stack([_attend(t["q"][b], t["k"][b], t["v"][b], c["D"] ** -0.5, c["causal"])[0]
                             for b in range(c["B"])])]
    if k == "fa_varlen":
        cu = t["cu"].tolist()
        return [torch.cat([_attend(t["q"][a:b], t["k"][a:b], t["v"][a:b], c["D"] ** -0.5)[0]
                           for a, b in zip(cu, cu[1:])])]
    if k == "fa_split":
        B, ns, per = c["B"], c["splits"], c["Skv"] // c["splits"]
        scale = c["D"] ** -0.5
        part = [[_attend(t["q"][b], t["k"][b, s * per:(s + 1) * per], t["v"][b, s * per:(s + 1) * per],
                         scale) for s in range(ns)] for b in range(B)]
        glse = torch.stack([torch.stack([p[1] for p in row], 1) for row in part])
        partial = torch.stack([torch.stack([p[0] for p in row], 2) for row in part])
        full = torch.stack([_attend(t["q"][b], t["k"][b], t["v"][b], scale)[0] for b in range(B)])
        return [glse, partial, full]
    out = []
    s = t["kv_scale"].double() if "kv_scale" in t else 1.0
    at = torch.arange(_slots(c), device="cuda")
    for b, n in enumerate(t["lens"].tolist()):
        row = t["table"][b].long()[at[:n] // PAGE] * PAGE + at[:n] % PAGE
        kv = t["kv"][row].double() * s
        p = torch.softmax(t["q"][b].double() @ kv.T * (DV + DPE) ** -0.5, 1)
        out.append(p @ kv[:, :DV])
    return [torch.stack(out)]
