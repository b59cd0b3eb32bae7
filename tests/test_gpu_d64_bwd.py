"""d_qk = d_v = 64 backward on the key-major scheme (the atomics' results are
the other implementation at the same precision) and its dispatch.

Tolerance: both round P and dS to bf16 (2^-9 relative each, random signs) and
the result to bf16, so the two differ by well under 2^-8 of the gradient's
norm."""
import pytest
import torch

import ops_amd
from oracle.sfa_oracle import sfa_backward as ref_backward

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(B, S, Skv, G, Hkv, K, seed, repeats=False):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(s, generator=g, device=DEV).bfloat16()
    q, k, v, do = rnd(B, S, G * Hkv, 64), rnd(B, Skv, Hkv, 64), rnd(B, Skv, Hkv, 64), rnd(B, S, G * Hkv, 64)
    # distinct keys per row in random order, some dropped, the first row empty
    idx = torch.rand((B, S, Hkv, Skv), generator=g, device=DEV).argsort(-1)[..., :K].to(torch.int32)
    idx[torch.rand(idx.shape, generator=g, device=DEV) < 0.1] = -1
    idx[0, 0] = -1
    if repeats:
        idx[:, 5, :, 3] = idx[:, 5, :, 7]
    return q, k, v, do, idx


def _rel(a, b):
    return float((a.double().cpu() - b.double().cpu()).norm() / b.double().cpu().norm())


# query blocks of 128 / G queries: partial last blocks (S odd), key blocks of 128: partial last, several chunks (G = 64)
@pytest.mark.parametrize("G,Hkv,S,Skv,K", [(16, 1, 1025, 1100, 1024), (64, 1, 515, 700, 600), (32, 2, 600, 900, 520),
                                           (128, 1, 253, 1000, 1000), (1, 8, 1100, 1100, 256), (8, 4, 1030, 513, 512)])
def test_against_atomics_and_oracle(G, Hkv, S, Skv, K):
    q, k, v, do, idx = _inputs(2, S, Skv, G, Hkv, K, seed=S + G)
    sink = torch.linspace(-1.0, 1.0, G * Hkv, device=DEV)
    out, lse = ops_amd.sfa_forward(q, k, v, idx, attn_sink=sink)
    dlse = torch.randn(lse.shape, device=DEV)
    runs = {m: ops_amd.sfa_backward(q, k, v, idx, out, lse, do, attn_sink=sink, dlse=dlse, dkv_mode=m)
            for m in ("auto", "atomic")}
    for a, b in zip(runs["auto"], runs["atomic"]):
        assert _rel(a, b) < 2.0 ** -8
    again = ops_amd.sfa_backward(q, k, v, idx, out, lse, do, attn_sink=sink, dlse=dlse)
    for a, b in zip(runs["auto"], again):
        assert torch.equal(a, b)  # (the atomics' sums are not)
    runs = ops_amd.sfa_backward(q, k, v, idx, out, lse, do, attn_sink=sink)
    sub = slice(0, 40)  # dq of some queries against the oracle (its dk / dv would need all of them)
    ref = ref_backward(q[:, sub].cpu(), k.cpu(), v.cpu(), idx[:, sub].cpu(), out[:, sub].cpu(), lse[:, sub].cpu(),
                       do[:, sub].cpu(), sink=sink.cpu())
    assert _rel(runs[0][:, sub], ref[0]) < 1e-2


def test_repeated_keys_and_unread_rows():
    """A repeated key counts twice; key rows that nothing selects may hold
    anything."""
    q, k, v, do, idx = _inputs(2, 1024, 1500, 16, 2, 1030, seed=2, repeats=True)
    idx[(idx >= 1300) & (idx < 1400)] = -1
    k[:, 1300:1400] = float("nan")
    v[:, 1300:1400] = float("inf")
    out, lse = ops_amd.sfa_forward(q, k, v, idx)
    a = ops_amd.sfa_backward(q, k, v, idx, out, lse, do)
    b = ops_amd.sfa_backward(q, k, v, idx, out, lse, do, dkv_mode="atomic")
    for x, y in zip(a[:3], b[:3]):
        assert bool(torch.isfinite(x).all()) and _rel(x, y) < 2.0 ** -8


@pytest.mark.parametrize("G,Hkv,shared", [(16, 2, False), (64, 1, True), (1, 8, False)])
def test_rows_that_are_not_finite_reach_selected_keys_only(G, Hkv, shared):
    """Queries that select nothing may hold anything, and a NaN row reaches the
    keys that it selects and no others."""
    q, k, v, do, idx = _inputs(2, 1024, 1024, G, Hkv, 300, seed=4)
    if shared:
        v = k
    idx[0, 100:110] = -1
    q[0, 100:105] = float("nan")
    do[0, 103:110] = float("inf")
    q[1, 7, G - 1] = float("nan")  # one head of one kv head
    do[0, 640, 0, 5] = float("nan")
    out, lse = ops_amd.sfa_forward(q, k, v, idx)
    a = ops_amd.sfa_backward(q, k, v, idx, out, lse, do)[:3]
    b = ops_amd.sfa_backward(q, k, v, idx, out, lse, do, dkv_mode="atomic")[:3]
    for x, y in zip(a, b):
        ok = torch.isfinite(x)
        assert torch.equal(ok, torch.isfinite(y))
        assert _rel(torch.where(ok, x, 0.0), torch.where(ok, y, 0.0)) < 2.0 ** -8


def test_named_scheme_stays_refused():
    q, k, v, do, idx = _inputs(1, 256, 256, 16, 1, 64, seed=3)
    out, lse = ops_amd.sfa_forward(q, k, v, idx)
    with pytest.raises(RuntimeError):
        ops_amd.sfa_backward(q, k, v, idx, out, lse, do, dkv_mode="csr")
