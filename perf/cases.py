"""The attention work a user of this package has it do, as timed cases.

Each case is one pass through a public entry point (`hip_sdpa` with autograd or forward-mode AD, `hip_sdpa_hvp`,
`GraphedSDPAHVP`, `sdpa_custom`), at the sizes of this repository's configurations and tests and at odd ones
between them. A case is a dict of plain values:

  kind    "train"      forward and (dQ, dK, dV) by autograd, as one layer of a training step
          "infer"      forward only, under no_grad
          "jvp"        forward and the tangent of O, by forward-mode AD
          "hvp"        H v of 0.5 ||O - target||^2 straight from the kernels (`hip_sdpa_hvp`)
          "hvp_weight" H v of <W, O>, the same entry point
          "hvp_graph"  H v of <W, O> through autograd, captured once and replayed with new vectors
          "probs"      the fused scores + softmax backend, P V in PyTorch
  dtype, B, H, T (queries), M (keys), D (head dim), causal
  std     standard deviation of Q, K, V: 0.5 and 1 give spread-out rows, 2 the peaked rows of trained attention
  packed  Q, K, V are views of one packed projection (B, T, 3, H, D), as a model's attention layer has them
"""

from __future__ import annotations

import math

import torch
import torch.autograd.forward_ad as fwAD

from theria_amd.attention.custom import sdpa_custom
from theria_amd.autograd import GraphedSDPAHVP
from theria_amd.autograd.hip_sdpa import hip_sdpa, hip_sdpa_hvp

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
# Units of D flops per visible (query, key) pair: the products each direction needs, S = Q K^T formed once per
# kernel pass that the path has by its interface (the scores are never kept between forward and backward).
_UNITS = {"train": 14, "infer": 4, "jvp": 14, "hvp": 38, "hvp_weight": 28, "hvp_graph": 38, "probs": 4}


def _case(name, kind, dtype, B, H, T, M, D, causal=False, std=1.0, packed=False):
    c = {"kind": kind, "dtype": dtype, "B": B, "H": H, "T": T, "M": M, "D": D, "causal": causal, "std": std,
         "packed": packed}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the smallest call: the CPU-reference configuration's HVP, a unit-test-sized probe; launches and latency
        _case("tiny_hvp_fp32", "hvp_weight", "fp32", 2, 2, 16, 16, 8),
        # full MAML's attention: 16 tasks x 25 support sequences, 4 heads of 16, in float32, differentiated twice
        _case("maml_graph_fp32", "hvp_graph", "fp32", 400, 4, 64, 64, 16),
        # the headline training shape
        _case("train_bf16", "train", "bf16", 4, 16, 2048, 2048, 64),
        # cross attention of ragged lengths with peaked rows, float16, a head dim between the kernels' sizes
        _case("train_ragged_fp16", "train", "fp16", 3, 7, 1030, 777, 80, std=2.0),
        # an ordinary float32 training layer on a packed projection, odd length
        _case("train_fp32", "train", "fp32", 2, 16, 1000, 1000, 64, packed=True),
        # the longest sequence: causal, head dim 128
        _case("long_causal_bf16", "train", "bf16", 1, 32, 8192, 8192, 128, causal=True, std=0.5),
        # few queries against a long context: the forward alone
        _case("infer_few_queries_bf16", "infer", "bf16", 1, 16, 100, 6000, 128),
        # directional derivative of a layer at training size
        _case("jvp_bf16", "jvp", "bf16", 4, 16, 2048, 2048, 64),
        # curvature probes (HVP of the quadratic loss) at the second-order configuration, both precisions
        _case("hvp_bf16", "hvp", "bf16", 8, 8, 512, 512, 64),
        _case("hvp_fp32", "hvp", "fp32", 8, 8, 512, 512, 64),
        # the same of a causal layer with large heads
        _case("hvp_d128_bf16", "hvp", "bf16", 2, 8, 1024, 1024, 128, causal=True),
        # the partial-fusion backend, which returns through materialised probabilities
        _case("probs_bf16", "probs", "bf16", 2, 8, 1500, 1500, 64),
    ]


_LARGEST = 14 * 128 * 32 * 8192 * 8193 // 2  # flops of long_causal_bf16, the largest listed case


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges, costing at most what the largest listed case does."""
    while True:
        kind = rng.choice(["train", "train", "train", "infer", "jvp", "hvp", "hvp", "hvp_weight", "hvp_graph", "probs"])
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32", "fp32"])
        if kind == "probs":
            dtype = rng.choice(["bf16", "fp16"])
        D = rng.choice([8, 16, 20, 32, 40, 48, 64, 64, 64, 80, 96, 128, 128])
        B, H = _log_int(rng, 1, 512), rng.choice([1, 2, 4, 7, 8, 16, 32])
        T = _log_int(rng, 16, 8192)
        if kind == "infer" and rng.random() < 0.5:
            T = _log_int(rng, 1, 128)
        M = T if rng.random() < 0.6 else _log_int(rng, 16, 8192)
        causal = M == T and kind != "probs" and rng.random() < 0.5
        std = rng.choice([0.5, 1.0, 1.0, 2.0])
        packed = M == T and rng.random() < 0.4 and kind not in ("probs", "hvp_graph")
        c = _case(None, kind, dtype, B, H, T, M, D, causal, std, packed)
        pairs = B * H * T * M
        # float32 products run at a sixteenth of the 16-bit rate: the largest case's time, not only its flops
        cost = work(c)["flops"] * (8 if dtype == "fp32" else 1) * (2 if kind.startswith("hvp") else 1)
        if 2 ** 14 <= pairs <= 2 ** 30 and cost <= _LARGEST and B * H * max(T, M) * D <= 2 ** 26:
            return c


def _pairs(c):
    T, M = c["T"], c["M"]
    if not c["causal"]:
        per_head = T * M
    else:
        n = min(T, M)
        per_head = n * (n + 1) // 2 + max(0, T - M) * M
    return c["B"] * c["H"] * per_head


def work(case):
    c = case
    es = 4 if c["dtype"] == "fp32" else 2
    bh, rows_q, rows_k = c["B"] * c["H"], c["T"] * c["D"] * es, c["M"] * c["D"] * es
    # (query-side tensors, key-side tensors) read or written once
    nq, nk = {"train": (4, 4), "infer": (2, 2), "jvp": (4, 4), "hvp": (4, 6), "hvp_weight": (4, 6),
              "hvp_graph": (4, 6), "probs": (2, 2)}[c["kind"]]
    nbytes = bh * (nq * rows_q + nk * rows_k)
    if c["kind"] == "probs":
        nbytes += 4 * _pairs(c) * 2  # the float32 probabilities, written by one step and read by the next
    return {"bytes": nbytes, "flops": _UNITS[c["kind"]] * c["D"] * _pairs(c)}


def _inputs(c, seed, dev="cuda:0"):
    """The case's tensors: q, k, v and what its kind takes beside them, from the seed alone."""
    gen = torch.Generator(device=dev).manual_seed(seed)
    dt, B, H, T, M, D = _DTYPES[c["dtype"]], c["B"], c["H"], c["T"], c["M"], c["D"]

    def rand(rows, std=1.0):
        return (torch.randn(B, H, rows, D, generator=gen, device=dev) * std).to(dt)

    if c["packed"]:
        qkv = (torch.randn(B, T, 3, H, D, generator=gen, device=dev) * c["std"]).to(dt)
        q, k, v = qkv.permute(2, 0, 3, 1, 4)
    else:
        q, k, v = rand(T, c["std"]), rand(M, c["std"]), rand(M, c["std"])
    x = {"q": q, "k": k, "v": v}
    if c["kind"] == "train":
        x["do"] = rand(T)
    elif c["kind"] == "jvp":
        x.update(tq=rand(T, 0.1), tk=rand(M, 0.1), tv=rand(M, 0.1))
    elif c["kind"].startswith("hvp"):
        x.update(w=rand(T), vq=rand(T), vk=rand(M), vv=rand(M))
    return x


def prepare(case, seed):
    x = _inputs(case, seed)
    state = {"case": case, **x}
    if case["kind"] == "train":
        for n in ("q", "k", "v"):
            state[n] = x[n].detach().requires_grad_(True)
    elif case["kind"] == "hvp_graph":
        state["graph"] = GraphedSDPAHVP(x["q"], x["k"], x["v"], x["vq"], x["vk"], x["vv"], weight=x["w"],
                                        causal=case["causal"])
    return state


def run(state):
    c, kind = state["case"], state["case"]["kind"]
    q, k, v, causal = state["q"], state["k"], state["v"], state["case"]["causal"]
    if kind == "train":
        o = hip_sdpa(q, k, v, causal=causal)
        return (o, *torch.autograd.grad(o, (q, k, v), state["do"]))
    if kind == "infer":
        with torch.no_grad():
            return hip_sdpa(q, k, v, causal=causal)
    if kind == "jvp":
        with fwAD.dual_level():
            duals = [fwAD.make_dual(a, t) for a, t in ((q, state["tq"]), (k, state["tk"]), (v, state["tv"]))]
            return tuple(fwAD.unpack_dual(hip_sdpa(*duals, causal=causal)))
    if kind == "hvp":
        return hip_sdpa_hvp(q, k, v, state["vq"], state["vk"], state["vv"], target=state["w"], causal=causal)
    if kind == "hvp_weight":
        return hip_sdpa_hvp(q, k, v, state["vq"], state["vk"], state["vv"], weight=state["w"], causal=causal)
    if kind == "hvp_graph":
        return state["graph"](vq=state["vq"], vk=state["vk"], vv=state["vv"])
    if kind == "probs":
        return sdpa_custom(q, k, v, backend="triton_qk_softmax")
    raise ValueError(f"unknown kind {c['kind']}")


def tolerance(case):
    # about four times the largest error against exact() over the listed cases and sixty drawn ones (relative error
    # of one output: float32 1.4e-6, of an HVP 3.0e-6; float16 4.2e-4; bfloat16 3.4e-3)
    if case["dtype"] == "fp32":
        return {"rel": 1.2e-5 if case["kind"].startswith("hvp") else 6e-6}
    return {"rel": 1.7e-3 if case["dtype"] == "fp16" else 1.4e-2}


# ---------------------------------------------------------------------------------------------------
# the same outputs in plain float64 torch
# ---------------------------------------------------------------------------------------------------
def _probs64(q, k, scale, causal):
    s = torch.matmul(q, k.transpose(-2, -1)) * scale
    if causal:
        s.masked_fill_(~torch.ones(s.shape[-2:], dtype=torch.bool, device=s.device).tril(), -math.inf)
    return torch.softmax(s, dim=-1)


def _backward64(p, q, k, v, do, scale):
    dp = torch.matmul(do, v.transpose(-2, -1))
    ds = p * (dp - (p * dp).sum(-1, keepdim=True))
    return scale * torch.matmul(ds, k), scale * torch.matmul(ds.transpose(-2, -1), q), torch.matmul(p.transpose(-2, -1), do)


def _tangent64(p, q, k, v, tq, tk, tv, scale):
    g = scale * (torch.matmul(tq, k.transpose(-2, -1)) + torch.matmul(q, tk.transpose(-2, -1)))
    pg = p * (g - (p * g).sum(-1, keepdim=True))
    return torch.matmul(pg, v) + torch.matmul(p, tv)


def _double_backward64(p, q, k, v, do, gq, gk, gv, scale):
    """Gradient with respect to q, k, v (do held fixed) of <gq, dQ> + <gk, dK> + <gv, dV>."""
    dp = torch.matmul(do, v.transpose(-2, -1))
    z = (p * dp).sum(-1, keepdim=True)
    gam = scale * (torch.matmul(gq, k.transpose(-2, -1)) + torch.matmul(q, gk.transpose(-2, -1)))  # cotangent of dS
    r = (p * gam).sum(-1, keepdim=True)
    g_dp = p * (gam - r)
    # dS = p (dp - z) and dV = p^T do: cotangent of p, then through the softmax
    g_p = (gam - r) * dp - z * gam + torch.matmul(do, gv.transpose(-2, -1))
    g_s = p * (g_p - (p * g_p).sum(-1, keepdim=True))
    ds = p * (dp - z)
    hq = scale * (torch.matmul(g_s, k) + torch.matmul(ds, gk))
    hk = scale * (torch.matmul(g_s.transpose(-2, -1), q) + torch.matmul(ds.transpose(-2, -1), gq))
    return hq, hk, torch.matmul(g_dp.transpose(-2, -1), do)


def exact(case, seed):
    c, kind = case, case["kind"]
    x = _inputs(c, seed)
    B, H, T, M, D = c["B"], c["H"], c["T"], c["M"], c["D"]
    flat = {n: t.reshape(B * H, -1, D) for n, t in x.items()}
    scale = 1.0 / math.sqrt(D)
    step = max(1, 2 ** 25 // (T * M))  # heads at a time: a few (T, M) float64 matrices each
    parts = []
    for i in range(0, B * H, step):
        t = {n: a[i:i + step].double() for n, a in flat.items()}
        q, k, v = t["q"], t["k"], t["v"]
        p = _probs64(q, k, scale, c["causal"])
        o = torch.matmul(p, v)
        if kind == "train":
            parts.append((o, *_backward64(p, q, k, v, t["do"], scale)))
        elif kind in ("infer", "probs"):
            parts.append((o,))
        elif kind == "jvp":
            parts.append((o, _tangent64(p, q, k, v, t["tq"], t["tk"], t["tv"], scale)))
        elif kind == "hvp":
            h = _double_backward64(p, q, k, v, o - t["w"], t["vq"], t["vk"], t["vv"], scale)
            jv = _tangent64(p, q, k, v, t["vq"], t["vk"], t["vv"], scale)
            parts.append(tuple(a + b for a, b in zip(h, _backward64(p, q, k, v, jv, scale))))
        else:
            parts.append(_double_backward64(p, q, k, v, t["w"], t["vq"], t["vk"], t["vv"], scale))
    outs = tuple(torch.cat(col).reshape(B, H, -1, D) for col in zip(*parts))
    return outs[0] if kind in ("infer", "probs") else outs
