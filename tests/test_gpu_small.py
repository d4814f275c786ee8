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
            if dt == F32:  # the general entry forms dO . O from a given O: take the row term the combined one wrote
                delta.copy_(got[3])
                _ops.bwd_dq(prob, q, k, v, None, False, do, lse, delta, dq)
            else:
                _ops.bwd_dq(prob, q, k, v, o, o_f32, do, lse, delta, dq)
            _ops.bwd_dkdv(prob, q, k, v, do, lse, delta, dk, dv)
            for name, a, b in zip(("dQ", "dK", "dV", "delta"), got, (dq, dk, dv, delta)):
                bars.close(a, b.double().cpu(), what=f"{name} causal={causal} o_f32={o_f32}", **bars.tol(dt))
            only_dv = _ops.bwd(q, k, v, o, lse, do, scale, causal, need_dq=False, need_dk=False)
            assert only_dv[0] is None and only_dv[1] is None
            assert torch.equal(only_dv[2], got[2]) and torch.equal(only_dv[3], got[3])
