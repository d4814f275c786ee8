"""The one-workgroup backward and double backward (at most 64 queries and 64 keys): every entry point against the
float64 oracle at the edges of their 32-row subtiles and head dims, on strided and broadcast operands, and the
backward against the general dQ and dK/dV kernels on the same inputs. Bars: tests/bars.py."""

import pytest
import torch

import bars
from test_gpu_parity import _check_all_entry_points, make
from theria_amd import _ops

pytestmark = pytest.mark.gpu

F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16
# one below, at and above a subtile; the largest small problem; the first sizes past it
SIZES = [(1, 1), (1, 64), (64, 1), (31, 33), (32, 32), (33, 31), (63, 64), (64, 64), (64, 65), (65, 64)]
DIMS = [3, 16, 17, 32, 33, 64, 72, 128]  # DP = 16, 32, 64 and (16-bit) 128, odd ones on element-wise loads


@pytest.mark.parametrize("dt", [F32, F16, BF16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("D", DIMS)
def test_small_problems_match_oracle(D, dt, hip_device):
    for i, (T, M) in enumerate(SIZES):
        causal = (i + D) % 2 == 1
        print(f"[small] {dt} T{T} M{M} D{D} causal={causal}", flush=True)
        _check_all_entry_points((dt, 2, 1 + i % 2, T, M, D, causal), hip_device, seed=500 + i)


@pytest.mark.parametrize("dt", [F32, BF16], ids=["fp32", "bf16"])
@pytest.mark.parametrize("D", [16, 24, 64])
def test_small_problems_on_strided_views(D, dt, hip_device):
    """Views of a packed projection (row stride 3 H D), and a dO one element past an aligned base shared by every head:
    the same results, bit for bit, as on contiguous copies."""
    B, H, T = 3, 2, 50
    print(f"[small strided] {dt} D{D}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(D)

    def rand(*shape):
        return torch.randn(*shape, generator=g, device=hip_device).to(dt)

    q, k, v = rand(B, T, 3, H, D).permute(2, 0, 3, 1, 4)
    tq, tk, tv = rand(B, T, 3, H, D).permute(2, 0, 3, 1, 4)
    do = rand(T * D + 1)[1:].view(1, 1, T, D).expand(B, H, T, D)
    for causal in (False, True):
        got = []
        for ts in ((q, k, v, do, tq, tk, tv), [t.contiguous() for t in (q, k, v, do, tq, tk, tv)]):
            o, lse = _ops.fwd(*ts[:3], D**-0.5, causal)[:2]
            got.append([o, lse, *_ops.bwd(*ts[:3], o, lse, ts[3], D**-0.5, causal),
                        *_ops.bwd_bwd(*ts[:3], o, ts[3], lse, None, *ts[4:], D**-0.5, causal)])
        assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("std", [1.0, 3.0])
@pytest.mark.parametrize("dt,D", [(F32, 16), (F32, 64), (F16, 48), (BF16, 64), (BF16, 128)])
def test_small_backward_equals_general_kernels(dt, D, std, hip_device):
    """theria_sdpa_bwd at 60 x 45 against theria_sdpa_bwd_dq + _dkdv (always the general kernels), with O in the input
    dtype and in float32; std 3 has rows flagged peaked, where both form the row term from P and dP. float32: both
    sum the same float32 products in another order (1e-5); 16-bit: half a unit of the output dtype each, and the
    general kernels' single 16-bit P and dS terms on rows not flagged (the 16-bit bar)."""
    B, H, T, M = 2, 3, 60, 45
    print(f"[small vs general] {dt} D{D} std{std}", flush=True)
    (q, _), (k, _) = make((B, H, T, D), dt, hip_device, 1, std), make((B, H, M, D), dt, hip_device, 2, std)
    (v, _), (do, _) = make((B, H, M, D), dt, hip_device, 3), make((B, H, T, D), dt, hip_device, 4)
    scale = D**-0.5
    for causal in (False, True):
        for o_f32 in (False, True):
            o, lse = _ops.fwd(q, k, v, scale, causal, out_fp32=o_f32)[:2]
            got = _ops.bwd(q, k, v, o, lse, do, scale, causal)
            dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
            delta = torch.empty_like(lse)
            prob = _ops._problem(q, k, scale, causal)
            _ops.bwd_dq(prob, q, k, v, o, o_f32, do, lse, delta, dq)
            _ops.bwd_dkdv(prob, q, k, v, do, lse, delta, dk, dv)
            for name, a, b in zip(("dQ", "dK", "dV", "delta"), got, (dq, dk, dv, delta)):
                bars.close(a, b.double().cpu(), what=f"{name} causal={causal} o_f32={o_f32}", **bars.tol(dt))
            only_dv = _ops.bwd(q, k, v, o, lse, do, scale, causal, need_dq=False, need_dk=False)
            assert only_dv[0] is None and only_dv[1] is None
            assert torch.equal(only_dv[2], got[2]) and torch.equal(only_dv[3], got[3])


@pytest.mark.parametrize("dt", [F32, F16, BF16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("T,M", [(50, 40), (70, 40)], ids=["small", "general"])
def test_nan_key_reaches_the_rows_that_see_it(T, M, dt, hip_device):
    """A NaN in one key, no cotangent of dQ (so that it enters the double backward through P alone): every row that sees
    the key is NaN throughout, the causal rows before it are as without it."""
    print(f"[small nan] {dt} T{T} M{M}", flush=True)
    D, key = 16, 20
    g = torch.Generator(device=hip_device).manual_seed(3)
    q, do = (torch.randn(2, 2, T, D, generator=g, device=hip_device).to(dt) for _ in range(2))
    k, v, tk, tv = (torch.randn(2, 2, M, D, generator=g, device=hip_device).to(dt) for _ in range(4))
    bad = k.clone()
    bad[:, :, key, 5] = float("nan")
    for causal in (False, True):
        outs = []
        for kk in (bad, k):
            o, lse = _ops.fwd(q, kk, v, D**-0.5, causal)[:2]
            outs.append(_ops.bwd_bwd(q, kk, v, o, do, lse, None, None, tk, tv, D**-0.5, causal))
        first = key if causal else 0
        for i in (0, 3):  # G_Q, G_dO
            assert torch.isnan(outs[0][i][:, :, first:]).all()
            cols = [d for d in range(D) if i == 3 or d != 5]  # (0 times NaN in that column of G_Q)
            assert torch.equal(outs[0][i][:, :, :first, cols], outs[1][i][:, :, :first, cols])


@pytest.mark.parametrize("dt", [F32, F16, BF16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("T,M", [(50, 40), (96, 40)], ids=["small", "general"])
def test_rows_without_a_visible_score(T, M, dt, hip_device):
    """Every score is -infinity: P = 0, so nothing but the columns that meet an infinite key element (0 times infinity)
    is anything but 0."""
    print(f"[small masked rows] {dt} T{T} M{M}", flush=True)
    D = 16
    g = torch.Generator(device=hip_device).manual_seed(4)
    q, do = (torch.randn(2, 2, T, D, generator=g, device=hip_device).to(dt) for _ in range(2))
    k, v, tk, tv = (torch.randn(2, 2, M, D, generator=g, device=hip_device).to(dt) for _ in range(4))
    q[..., 0] = 1.0
    k[..., 0] = -float("inf")
    for causal in (False, True):
        o, lse = _ops.fwd(q, k, v, D**-0.5, causal)[:2]
        assert (o == 0).all() and (lse == -float("inf")).all()
        dq, dk, dv = _ops.bwd(q, k, v, o, lse, do, D**-0.5, causal)[:3]
        gq, gk, gv, gdo = _ops.bwd_bwd(q, k, v, o, do, lse, None, None, tk, tv, D**-0.5, causal)
        for name, x in (("dQ", dq[..., 1:]), ("dK", dk), ("dV", dv), ("G_Q", gq[..., 1:]), ("G_K", gk), ("G_V", gv),
                        ("G_dO", gdo)):
            assert (x == 0).all(), name
