"""The split second-order kernels above head dim 64 (computed at 128): the JVP with two key groups and with one (256 or
more 128-query blocks), the key-split row and query-split column kernels of the double backward, at the edges of their
32-row subtiles and 64- or 128-row blocks, against the float64 oracle (bars: tests/bars.py)."""

import pytest
import torch

import bars
from oracle import sdpa_oracle as O
from test_gpu_parity import _check_all_entry_points, make
from theria_amd import _ops

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16


@pytest.mark.parametrize("dt,D", [(BF16, 72), (F16, 96), (BF16, 128)])
def test_second_order_of_large_heads_matches_oracle(dt, D, hip_device):
    for i, (T, M) in enumerate([(65, 63), (64, 65), (1, 129), (129, 1), (127, 32), (128, 128), (200, 33), (97, 300)]):
        for causal in (False, True):
            print(f"[split 128] {dt} T{T} M{M} D{D} causal={causal}", flush=True)
            _check_all_entry_points((dt, 1, 2, T, M, D, causal), hip_device, seed=700 + i)


@pytest.mark.parametrize("std", [1.0, 3.0])
@pytest.mark.parametrize("T,M,causal", [(65, 65, True), (70, 33, False), (130, 64, False), (129, 129, True)])
def test_jvp_of_many_blocks(T, M, causal, std, hip_device):
    """256 (batch, head) pairs: one key group per workgroup; every tangent, one of them, and head dims below 128."""
    for D in (80, 128):
        print(f"[split 128 jvp] T{T} M{M} D{D} causal={causal} std{std}", flush=True)
        (q, qc), (k, kc) = make((16, 16, T, D), BF16, hip_device, 1, std), make((16, 16, M, D), BF16, hip_device, 2, std)
        (v, vc), (tq, tqc) = make((16, 16, M, D), BF16, hip_device, 3), make((16, 16, T, D), BF16, hip_device, 4)
        (tk, tkc), (tv, tvc) = (make((16, 16, M, D), BF16, hip_device, 5 + i) for i in range(2))
        s = D**-0.5
        o, lse = _ops.fwd(q, k, v, s, causal)[:2]
        for ts, tcs in (((tq, tk, tv), (tqc, tkc, tvc)), ((None, tk, None), (None, tkc, None))):
            got = _ops.jvp(q, k, v, o, lse, *ts, s, causal)
            bars.close(got, O.jvp(qc, kc, vc, *tcs, s, causal), what=f"JVP D{D}", **bars.tol(BF16))


@pytest.mark.parametrize("D", [80, 128])
def test_large_heads_on_strided_views(D, hip_device):
    """Packed-projection views (row stride 3 H D): the same results as on contiguous copies, bit for bit."""
    B, H, T = 2, 2, 150
    print(f"[split 128 strided] D{D}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(D)
    q, k, v = torch.randn(B, T, 3, H, D, generator=g, device=hip_device).to(BF16).permute(2, 0, 3, 1, 4)
    tq, tk, tv = torch.randn(B, T, 3, H, D, generator=g, device=hip_device).to(BF16).permute(2, 0, 3, 1, 4)
    do = torch.randn(B, T, H, D, generator=g, device=hip_device).to(BF16).transpose(1, 2)
    got = []
    for ts in ((q, k, v, do, tq, tk, tv), [t.contiguous() for t in (q, k, v, do, tq, tk, tv)]):
        o, lse = _ops.fwd(*ts[:3], D**-0.5, True)[:2]
        got.append([_ops.jvp(*ts[:3], o, lse, *ts[4:], D**-0.5, True),
                    *_ops.bwd_bwd(*ts[:3], o, ts[3], lse, None, *ts[4:], D**-0.5, True)])
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("D", [96, 128])
@pytest.mark.parametrize("T", [130, 600])
def test_causal_dq_of_small_and_large_grids(T, D, hip_device):
    """A causal grid of at most one workgroup per CU takes the peaked and common query blocks in one launch, a larger one
    in two: the same head gives the same gradients bit for bit alone and as one of 160."""
    print(f"[causal dq grids] T{T} D{D}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(T + D)
    q, k, v, do = (torch.randn(1, 1, T, D, generator=g, device=hip_device).to(BF16) for _ in range(4))
    one = [q, k, v, do]
    many = [t.expand(1, 160, T, D) for t in one]
    got = []
    for ts in (one, many):
        o, lse = _ops.fwd(*ts[:3], D**-0.5, True)[:2]
        got.append(_ops.bwd(*ts[:3], o, lse, ts[3], D**-0.5, True))
    for a, b in zip(*got):
        assert torch.equal(a[0, 0], b[0, 0]) and torch.equal(a[0, 0], b[0, 159])


def rounding(x, dt):
    """2-norm error of rounding a float64 tensor to dt, relative to it."""
    return float((x.to(dt).double() - x).norm() / x.norm())


@pytest.mark.parametrize("std", [0.5, 1.0])
@pytest.mark.parametrize("dt,D", [(BF16, 72), (BF16, 128), (F16, 96)])
def test_jvp_error_is_the_rounding_of_its_output(dt, D, std, hip_device):
    """Spread-out rows, few (two key groups) and many (one) blocks: P o G and P enter their products as two 16-bit terms,
    2^-16 of the cancelling terms, so that of the tangents of Q and K only the output's own rounding shows (bar: 1.05
    times it; one 16-bit term each gave 1.4 times)."""
    for B, H, causal in ((1, 4, False), (1, 4, True), (16, 8, False)):
        T, M = 200, 300
        print(f"[split 128 jvp rounding] {dt} B{B}H{H} D{D} std{std} causal={causal}", flush=True)
        g = torch.Generator().manual_seed(D + B)
        q, tq = (torch.randn(B, H, T, D, generator=g).mul(x).to(dt) for x in (std, 1.0))
        k, tk, v = (torch.randn(B, H, M, D, generator=g).mul(x).to(dt) for x in (std, 1.0, 1.0))
        dev = [t.to(hip_device) for t in (q, k, v)]
        o, lse = _ops.fwd(*dev, D**-0.5, causal)[:2]
        got = _ops.jvp(*dev, o, lse, tq.to(hip_device), tk.to(hip_device), None, D**-0.5, causal).cpu().double()
        ref = O.jvp(q, k, v, tq, tk, None, D**-0.5, causal)
        err = float((got - ref).norm() / ref.norm())
        print(f"    error {err:.3e}, rounding {rounding(ref, dt):.3e}", flush=True)
        assert err <= 1.05 * rounding(ref, dt)


@pytest.mark.parametrize("std", [0.5, 1.0])
@pytest.mark.parametrize("dt,D", [(BF16, 72), (BF16, 128), (F16, 96)])
def test_double_backward_of_dout_error_is_the_rounding_of_its_output(dt, D, std, hip_device):
    """G_dO of the key-split row kernel, whose first pass also sums z and t from the same products: as the JVP above."""
    T, M = 200, 300
    for causal in (False, True):
        print(f"[split 128 G_dO rounding] {dt} D{D} std{std} causal={causal}", flush=True)
        g = torch.Generator().manual_seed(D)
        q, tq = (torch.randn(2, 3, T, D, generator=g).mul(x).to(dt) for x in (std, 1.0))
        k, tk, v = (torch.randn(2, 3, M, D, generator=g).mul(x).to(dt) for x in (std, 1.0, 1.0))
        do = torch.randn(2, 3, T, D, generator=g).to(dt)
        dq, dk, dv, ddo, dtq, dtk = (t.to(hip_device) for t in (q, k, v, do, tq, tk))
        o, lse = _ops.fwd(dq, dk, dv, D**-0.5, causal)[:2]
        got = _ops.bwd_bwd(dq, dk, dv, o, ddo, lse, None, dtq, dtk, None, D**-0.5, causal)[3].cpu().double()
        ref = O.jvp(q, k, v, tq, tk, None, D**-0.5, causal)
        err = float((got - ref).norm() / ref.norm())
        print(f"    error {err:.3e}, rounding {rounding(ref, dt):.3e}", flush=True)
        assert err <= 1.05 * rounding(ref, dt)
