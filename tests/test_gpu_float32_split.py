"""float32 products formed on the bfloat16 matrix pipe from three-term splits (MfmaX3): operands of 2^-20 to 2^20 in one
row, the largest float32 and infinities against operands of either residual sign, and tile and k-chunk edges.

Bound: S = sum of D products, the split keeping each to 2^-24 (2^-21 where both operands are large) and the accumulator
rounding at most once per term: |S - S64| <= (D + 8) 2^-24 sum |q| |k|, float32's own bound for a sum of D terms in any
order."""

import math

import pytest
import torch

from oracle import sdpa_oracle as O
from theria_amd import _ops
from theria_amd.attention.scores import triton_qk

pytestmark = pytest.mark.gpu

# k chunks of 16, subtiles of 32, tiles of 64 and blocks of 128 rows: one below, at and above
SHAPES = [(1, 1, 1), (31, 33, 15), (32, 32, 16), (33, 64, 17), (128, 65, 32), (129, 63, 33), (64, 130, 64), (70, 40, 100),
          (33, 31, 127), (130, 129, 128)]


@pytest.mark.parametrize("T,M,D", SHAPES)
def test_scores_of_operands_over_many_magnitudes(T, M, D):
    print(f"float32 split scores T{T} M{M} D{D}", flush=True)
    g = torch.Generator().manual_seed(T * 1000 + M * 10 + D)

    def wide(rows):  # magnitudes 2^-20 .. 2^20 within every row
        return torch.randn(1, 2, rows, D, generator=g) * torch.exp2(torch.randint(-20, 21, (1, 2, rows, D), generator=g).float())

    q, k = wide(T), wide(M)
    s = triton_qk(q.cuda(), k.cuda()).double().cpu()
    ref = q.double() @ k.double().transpose(-2, -1)
    bound = (D + 8) * 2.0**-24 * (q.double().abs() @ k.double().abs().transpose(-2, -1))
    assert ((s - ref).abs() <= bound).all(), float(((s - ref).abs() / bound).max())


@pytest.mark.parametrize("D", [16, 64, 128])
def test_largest_values_and_infinities(D):
    """The lowest float32 and -infinity in a key mask it (its scores are far below the others), the largest one in
    V stays finite in O, and an infinite V reaches O's column and no other, as in float32."""
    print(f"float32 split extremes D{D}", flush=True)
    g = torch.Generator().manual_seed(D)
    q = torch.rand(1, 1, 40, D, generator=g) + 0.5  # positive: every score of a masked key is negative
    k, v = (torch.randn(1, 1, 70, D, generator=g) for _ in range(2))
    big = torch.finfo(torch.float32).max
    k[0, 0, 3, 0] = -big
    k[0, 0, 68, 1] = -float("inf")
    v[0, 0, 5, 2] = big
    v[0, 0, 7, 4] = float("inf")
    o = _ops.fwd(q.cuda(), k.cuda(), v.cuda(), D**-0.5, False)[0].cpu()
    keep = [j for j in range(70) if j not in (3, 68)]
    p = torch.softmax(q.double() @ k[:, :, keep].double().transpose(-2, -1) * D**-0.5, -1)
    ref = p @ v[:, :, keep].double()
    assert torch.isinf(o[..., 4]).all() and (o[..., 4] > 0).all()
    cols = [d for d in range(D) if d not in (2, 4)]
    torch.testing.assert_close(o[..., cols].double(), ref[..., cols], rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(o[..., 2].double(), ref[..., 2], rtol=1e-4, atol=0.0)  # P of one key, scaled by 3.4e38


@pytest.mark.parametrize("D", [64, 80, 128])
@pytest.mark.parametrize("T,M,causal", [(20, 90, False), (130, 130, True)])
def test_jvp_rounds_as_the_forward(T, M, causal, D, hip_device):
    """Scores of up to ~20: lse and the JVP's scores round alike, so the tangent is no worse than PyTorch's float32
    formula with its own softmax (bar: 1.5 times its error against float64; the kernel measured ~0.9 times, and 1.4 times
    lse's rounding more when its scores were rounded in another order)."""
    print(f"float32 split jvp T{T} M{M} D{D} causal={causal}", flush=True)
    g = torch.Generator().manual_seed(D + T)
    q, tq = (torch.randn(2, 4, T, D, generator=g) * s for s in (2.0, 1.0))
    k, tk, v, tv = (torch.randn(2, 4, M, D, generator=g) * s for s in (2.0, 1.0, 1.0, 1.0))
    mask = torch.ones(T, M, dtype=torch.bool).triu(1) if causal else torch.zeros(T, M, dtype=torch.bool)

    def plain(dt):
        a, b, c, ta, tb, tc = (t.to(dt) for t in (q, k, v, tq, tk, tv))
        p = torch.softmax((a @ b.mT * D**-0.5).masked_fill(mask, -float("inf")), -1)
        ds = p * ((ta @ b.mT + a @ tb.mT) * D**-0.5)
        return (ds - p * ds.sum(-1, keepdim=True)) @ c + p @ tc

    dev = [t.to(hip_device) for t in (q, k, v, tq, tk, tv)]
    o, lse = _ops.fwd(*dev[:3], D**-0.5, causal)[:2]
    got = _ops.jvp(*dev[:3], o, lse, *dev[3:], D**-0.5, causal).cpu()
    ref = plain(torch.float64)
    err, bar = (float((t.double() - ref).norm() / ref.norm()) for t in (got, plain(torch.float32)))
    assert err <= 1.5 * bar, (err, bar)


@pytest.mark.parametrize("D", [72, 96, 128])
@pytest.mark.parametrize("T,M,causal", [(100, 1, False), (100, 100, True)])
def test_one_visible_key_gives_no_curvature(T, M, causal, D, hip_device):
    """A row that sees one key has P = 1 whatever its scores: its G_Q is 0 exactly where the row statistics, the row
    kernel and the column kernel form S and dP by the same products, in the same order of rounding."""
    print(f"float32 split one key T{T} M{M} D{D} causal={causal}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(D + M)
    q, do, tq = (torch.randn(1, 2, T, D, generator=g, device=hip_device) for _ in range(3))
    k, v, tk, tv = (torch.randn(1, 2, M, D, generator=g, device=hip_device) for _ in range(4))
    o, lse = _ops.fwd(q, k, v, D**-0.5, causal)[:2]
    gq = _ops.bwd_bwd(q, k, v, o, do, lse, None, tq, tk, tv, D**-0.5, causal)[0]
    assert (gq[:, :, 0 if causal else slice(None)] == 0).all()


def masked_inputs(T, M, D, mask):
    """Standard normal inputs, q's first element 1002.5 (its bfloat16 is 1004: the residual has the other sign) or 800; keys
    3, M / 2 and M - 1 masked by `mask` in that element. Every other key has 0 there."""
    g = torch.Generator().manual_seed(T + D)
    q, do = (torch.randn(2, 2, T, D, generator=g) for _ in range(2))
    k, v, tk, tv = (torch.randn(2, 2, M, D, generator=g) for _ in range(4))
    q[..., 0] = torch.where(torch.arange(T) % 2 == 0, 1002.5, 800.0)
    k[..., 0] = 0.0
    gone = [3, M // 2, M - 1]
    k[:, :, gone, 0] = mask
    return q, k, v, do, tk, tv, [j for j in range(M) if j not in gone], gone


@pytest.mark.parametrize("mask", [-float("inf"), float(torch.finfo(torch.float32).min), -1e37], ids=["inf", "lowest", "1e37"])
@pytest.mark.parametrize("T,M,D", [(40, 50, 16), (64, 64, 64), (160, 150, 16), (128, 150, 64), (96, 90, 80), (160, 150, 128)])
def test_keys_masked_by_value(T, M, D, mask, hip_device):
    """Scores below the lowest float32 are -infinity, whatever the products' terms overflow to, in every kernel: the keys
    are gone from O, the tangent and the gradients (1e-5 of the float64 results without them)."""
    print(f"float32 split masked keys T{T} M{M} D{D} {mask}", flush=True)
    q, k, v, do, tk, tv, keep, gone = masked_inputs(T, M, D, mask)
    scale = D**-0.5
    dq_, dk_, dv_, ddo, dtk, dtv = (t.to(hip_device) for t in (q, k, v, do, tk, tv))
    k0, v0, tk0, tv0 = (t[:, :, keep] for t in (k, v, tk, tv))
    cols = slice(1, None) if math.isinf(mask) else slice(None)  # (0 times infinity in dQ's and G_Q's first column)

    def close(got, ref, what):
        got = got.double().cpu()
        assert torch.isfinite(got).all(), what
        tol = 1e-5 * max(1.0, float(ref.abs().max()))
        torch.testing.assert_close(got, ref, rtol=1e-5, atol=tol, msg=lambda m: f"{what}: {m}")

    s = triton_qk(dq_, dk_)
    assert (s[..., gone] == -float("inf")).all() or mask == -1e37
    o, lse = _ops.fwd(dq_, dk_, dv_, scale, False)[:2]
    close(o, O.forward(q, k0, v0, scale, False)[0], "O")
    gq, gk, gv = _ops.bwd(dq_, dk_, dv_, o, lse, ddo, scale, False)[:3]
    rq, rk, rv = O.backward(q, k0, v0, do, scale, False)
    close(gq[..., cols], rq[..., cols], "dQ")
    for name, x, r in (("dK", gk, rk), ("dV", gv, rv)):
        close(x[:, :, keep], r, name)
        close(x[:, :, gone], torch.zeros_like(r[:, :, :3]), name + " of the masked keys")
    t = _ops.jvp(dq_, dk_, dv_, o, lse, None, dtk, dtv, scale, False)
    close(t, O.jvp(q, k0, v0, None, tk0, tv0, scale, False), "tangent")
    hq, hk, hv, hdo = _ops.bwd_bwd(dq_, dk_, dv_, o, ddo, lse, None, None, dtk, dtv, scale, False)
    Hq, Hk, Hv, Hdo = O.double_backward(q, k0, v0, do, torch.zeros_like(q), tk0, tv0, scale, False)
    close(hq[..., cols], Hq[..., cols], "G_Q")
    close(hdo, Hdo, "G_dO")
    for name, x, r in (("G_K", hk, Hk), ("G_V", hv, Hv)):
        close(x[:, :, keep], r, name)
