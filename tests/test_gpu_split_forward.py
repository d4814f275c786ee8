"""The forward whose keys are split over workgroups (few query blocks against many keys): O, lse and the reference's
statistics against the same problem run whole (theria_sdpa_fwd, which has no workspace) and against float64.

Both forms are held to the bars of tests/bars.py against float64, and so to twice them against each other (the general
kernel and the pipelined one round P against different offsets, so 16-bit results of the two are not one unit apart)."""

import ctypes

import pytest
import torch

import bars
from oracle import sdpa_oracle as O
from theria_amd import _lib, _ops

pytestmark = pytest.mark.gpu

F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16
# T around the 128-query block, M at the first split size and one key past / short of whole tiles, every padded head dim,
# head dims on the general kernel (33, 20) and the pipelined one; (B, H) up to the largest split grid of the type
CASES = [
    (BF16, 1, 16, 100, 1300, 128), (BF16, 1, 1, 1, 1280, 64), (BF16, 2, 3, 129, 1281, 64), (BF16, 1, 2, 257, 1999, 32),
    (BF16, 2, 2, 130, 577, 96), (BF16, 1, 64, 128, 512, 72), (F16, 1, 2, 200, 1290, 40), (F16, 3, 1, 31, 1400, 20),
    (F16, 1, 1, 60, 5000, 8), (F32, 1, 4, 300, 512, 32), (F32, 2, 2, 64, 577, 33), (F32, 1, 1, 1, 4159, 64),
    (F32, 1, 128, 100, 512, 16), (F32, 1, 2, 200, 639, 128),
]


def whole(q, k, v, scale, o_f32):
    """theria_sdpa_fwd: no workspace, so never split."""
    lib = _lib.load()
    o = torch.empty(q.shape, dtype=F32 if o_f32 else q.dtype, device=q.device)
    lse, m, l = (torch.empty(q.shape[:3], device=q.device) for _ in range(3))
    prob = _ops._problem(q, k, scale, False)
    rc = lib.theria_sdpa_fwd(ctypes.byref(prob), _ops._tv(q), _ops._tv(k), _ops._tv(v), _ops._tv(o), int(o_f32),
                             lse.data_ptr(), m.data_ptr(), l.data_ptr(), _ops._stream(q.device))
    assert rc == 0
    return o, lse, m, l


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{str(c[0])[6:]}-B{c[1]}H{c[2]}T{c[3]}M{c[4]}D{c[5]}")
@pytest.mark.parametrize("std", [1.0, 3.0])
def test_split_forward_equals_whole(case, std, hip_device):
    dt, B, H, T, M, D = case
    print(f"[split forward] {case} std{std}", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(M + D)
    # views of one buffer (rows of 2 H D), as a packed projection has them; peaked rows at std 3
    kv = torch.randn(B, M, 2, H, D, generator=g, device=hip_device)
    kv[:, :, 0] *= std
    kv = kv.to(dt)
    k, v = kv.permute(2, 0, 3, 1, 4)
    q = (torch.randn(B, H, T, D, generator=g, device=hip_device) * std).to(dt)
    scale = D**-0.5
    assert _lib.load().theria_sdpa_fwd_ws_floats(ctypes.byref(_ops._problem(q, k, scale, False))) > 0
    ref = O.forward(q.double().cpu(), k.double().cpu(), v.double().cpu(), scale, False)[0]
    tol = bars.tol(dt)
    if dt == F32 and std > 1:  # peaked float32 rows: what float32 arithmetic itself reaches (its PyTorch error, doubled)
        f32 = torch.softmax(q.cpu() @ k.cpu().transpose(-2, -1) * scale, -1) @ v.cpu()
        tol["atol"] = max(tol["atol"], 2 * float((f32.double() - ref).abs().max()))
    for o_f32 in (False, True):
        got = _ops.fwd(q, k, v, scale, False, out_fp32=o_f32, stats=True)
        want = whole(q, k, v, scale, o_f32)
        bars.close(got[0], ref, what="O", **tol)
        bars.close(want[0], ref, what="O (whole)", **tol)
        bars.close(got[0], want[0].double().cpu(), what="O against whole", **{n: 2 * x for n, x in tol.items()})
        # lse: the flag bit moves it by one unit in the last place, 16-bit row sums are of 16-bit P
        stat = dict(rtol=1e-5, atol=1e-5) if dt == F32 else dict(rtol=4e-3, atol=4e-3)
        bars.close(got[1], want[1].double().cpu(), what="lse", **stat)
        bars.close(got[2], want[2].double().cpu(), what="m", rtol=1e-5, atol=1e-5)
        bars.close(got[3], want[3].double().cpu(), what="l", **stat)
        if dt != F32:  # every row whose largest probability exceeds 1/4 is flagged
            pmax = O.probs(q.double().cpu(), k.double().cpu(), scale, False).amax(-1)
            flagged = (got[1].cpu().view(torch.int32) & 1).bool()
            assert not ((pmax > 0.25 * (1 + 1e-2)) & ~flagged).any()
        else:
            assert torch.isfinite(got[1]).all()


def test_split_forward_with_masked_keys(hip_device):
    """Keys of -infinity scores in every part, whole parts of them, and rows that see none (O = 0, lse = -inf)."""
    print("[split forward masked keys]", flush=True)
    g = torch.Generator(device=hip_device).manual_seed(5)
    q = torch.rand(1, 2, 70, 64, generator=g, device=hip_device) + 0.5
    k = torch.randn(1, 2, 1024, 64, generator=g, device=hip_device)
    v = torch.randn(1, 2, 1024, 64, generator=g, device=hip_device)
    k[:, :, 100:700, 0] = -float("inf")
    k[:, 1, :, 0] = -float("inf")
    got = _ops.fwd(q, k, v, 0.125, False, stats=True)
    want = whole(q, k, v, 0.125, False)
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5)
    assert (got[0][:, 1] == 0).all() and (got[1][:, 1] == -float("inf")).all()


@pytest.mark.parametrize("dt", [F16, BF16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("T,D", [(1, 64), (65, 96), (100, 128), (128, 40), (60, 20)])
def test_split_forward_sums_rows_in_float32(T, D, dt, hip_device):
    """At most 128 queries: lse and the row sum are sums of float32 P, as they are unsplit, also where later keys' scores
    are far above the first tiles' (float16 then moves the offset before a P leaves its range: 13 nats a tile). Bounds:
    1e-5 for the sum of M float32 terms; in l's exponentials also the roundings of a score of size |S|: scale log2(e) (two),
    the dot product (two), its product with that, the maximum in the log2 domain and back, and their difference, each
    at most 2^-24 |S|: 8 of them. Rounded P gave 1e-4."""
    M, scale = 1500, D**-0.5
    print(f"[split forward row sums] {dt} T{T} D{D}", flush=True)
    g = torch.Generator().manual_seed(T + D)
    for std, rise in ((0.5, 0.0), (2.0, 0.0), (0.5, 300.0)):
        q, k, v = (torch.randn(1, 3, n, D, generator=g) for n in (T, M, M))
        q, k = q * std, k * std
        if rise:  # scores climb by `rise` over the keys along one direction
            q[..., 0] = 1.0
            k[..., 0] = torch.linspace(0.0, rise / scale, M)
        q, k, v = (t.to(dt) for t in (q, k, v))
        assert _lib.load().theria_sdpa_fwd_ws_floats(ctypes.byref(_ops._problem(q, k, scale, False))) > 0
        S = (q.double() @ k.double().transpose(-2, -1)) * scale
        m = S.amax(-1)
        l = torch.exp(S - m[..., None]).sum(-1)
        got = _ops.fwd(*(t.to(hip_device) for t in (q, k, v)), scale, False, stats=True)
        bars.close(got[0], torch.softmax(S, -1) @ v.double(), what="O", **bars.tol(dt))
        bars.close(got[1], m + torch.log(l), what="lse", rtol=1e-5, atol=1e-5)
        bars.close(got[2], m, what="m", rtol=1e-5, atol=1e-5)
        bars.close(got[3], l, what="l", rtol=1e-5 + 8 * 2.0**-24 * float(S.abs().max()), atol=0.0)
