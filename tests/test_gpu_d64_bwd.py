"""d_qk = d_v = 64 backward on the key-major scheme (the atomics' results are
the other implementation at the same precision) and its dispatch.

Tolerance: both round P and dS to bf16 (2^-9 relative each, random signs) and
the result to bf16, so the two differ by well under 2^-8 of the gradient's
norm."""
import pytest
import torch

import ops_amd
from oracle.sfa_oracle import sfa_backward as ref_backward
from oracle.sfa_oracle import sfa_forward as ref_forward

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


@pytest.mark.parametrize("what", ["plain", "repeats", "not finite", "unaligned dk"])
@pytest.mark.parametrize("G,Hkv,S,Skv,K", [(16, 2, 1030, 1100, 300), (64, 1, 515, 700, 600)])
def test_one_gradient_of_shared_rows(G, Hkv, S, Skv, K, what):
    """merge_kv: dK + dV of the shared rows in one sum, against the atomics'
    and against the separate gradients (each rounded to bf16 before they are
    added here: 2^-9 of a term more)."""
    q, k, _, do, idx = _inputs(2, S, Skv, G, Hkv, K, seed=S + K, repeats=what == "repeats")
    if what == "not finite":
        idx[0, 100:110] = -1
        q[0, 100:105] = float("nan")  # (a query that selects nothing may hold anything)
        q[1, 7, G - 1] = float("nan")
        do[0, 512, 0, 5] = float("inf")
        k[0, 3] = float("inf")  # (a key that few rows select)
        idx[idx == 3] = -1
        idx[0, 9, 0, 2] = 3
    out, lse = ops_amd.sfa_forward(q, k, k, idx)
    call = lambda **kw: ops_amd.sfa_backward(q, k, k, idx, out, lse, do, **kw)
    a, b = call(merge_kv=True), call(merge_kv=True, dkv_mode="atomic")
    dk = torch.full((2, Skv, Hkv, 67), 7.0, device=DEV, dtype=torch.bfloat16)
    if what == "unaligned dk":
        call(merge_kv=True, dk=dk[..., 1:65])
        assert torch.equal(dk[..., 1:65], a[1])
        assert bool((dk[..., :1] == 7.0).all()) and bool((dk[..., 65:] == 7.0).all())
    again = call(merge_kv=True)[1]
    assert a[2] is None and torch.equal(torch.nan_to_num(a[1]), torch.nan_to_num(again))  # (bitwise: not the atomics)
    for i in (0, 1):
        ok = torch.isfinite(a[i])
        assert torch.equal(ok, torch.isfinite(b[i])) and bool(ok.all()) == (what != "not finite")
        assert _rel(torch.where(ok, a[i], 0.0), torch.where(ok, b[i], 0.0)) < 2.0 ** -8
    _, dk2, dv2, _ = call()
    ok = torch.isfinite(a[1])
    both = dk2.float() + dv2.float()
    assert torch.equal(ok, torch.isfinite(both))
    assert _rel(torch.where(ok, a[1], 0.0), torch.where(ok, both, 0.0)) < 2.0 ** -7


def test_reference_signature_at_training_size():
    """One kv row for K and V under autograd, large enough for the key-major
    scheme (bitwise the same twice), against the oracle."""
    g = torch.Generator(device=DEV).manual_seed(12)
    S, B, H, K = 384, 2, 64, 200
    q = torch.randn((S, B, H, 64), generator=g, device=DEV).bfloat16().requires_grad_()
    kv = torch.randn((S, B, 64), generator=g, device=DEV).bfloat16().requires_grad_()
    sink = torch.randn(H, generator=g, device=DEV).requires_grad_()
    idx = torch.rand((S, B, S), generator=g, device=DEV).argsort(-1)[..., :K].int()
    do = torch.randn((S, B, H, 64), generator=g, device=DEV).bfloat16()
    runs = [torch.autograd.grad(ops_amd.SparseFlashAttentionTriton.apply(q, kv, sink, idx, 0.1), (q, kv, sink), do)
            for _ in range(2)]
    assert all(torch.equal(x, y) for x, y in zip(*runs))
    qb, kb = q.detach().transpose(0, 1).cpu(), kv.detach().transpose(0, 1).unsqueeze(2).cpu()
    ib, db, sb = idx.transpose(0, 1).unsqueeze(2).cpu(), do.transpose(0, 1).cpu(), sink.detach().cpu()
    o_ref, l_ref = ref_forward(qb, kb, kb, ib, 0.1, sink=sb)
    dq, dk, dv, ds = ref_backward(qb, kb, kb, ib, o_ref, l_ref, db, 0.1, sink=sb)
    for x, y in zip(runs[0], (dq.transpose(0, 1), (dk + dv)[:, :, 0].transpose(0, 1), ds)):
        assert _rel(x.detach(), y) < 1e-2


def test_named_scheme_stays_refused():
    q, k, v, do, idx = _inputs(1, 256, 256, 16, 1, 64, seed=3)
    out, lse = ops_amd.sfa_forward(q, k, v, idx)
    with pytest.raises(RuntimeError):
        ops_amd.sfa_backward(q, k, v, idx, out, lse, do, dkv_mode="csr")
