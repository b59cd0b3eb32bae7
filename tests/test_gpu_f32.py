"""float32 at head dims 64 and 128 (fp32 matrix instructions) against the
float64 oracle, forward and backward.

Tolerance: products are exact to fp32 and sums run over D <= 128 terms and K <=
600 slots, each term off by at most 2^-24 of the running sum: below 600 * 2^-24 =
3.6e-5 of the result's norm in the worst case of one sign, far less in fact."""
import pytest
import torch

import ops_amd
from ops_amd.workloads import page_kv
from oracle.sfa_oracle import sfa_backward as ref_backward
from oracle.sfa_oracle import sfa_forward as ref_forward

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = 3.6e-5


def _inputs(B, S, Skv, G, Hkv, D, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(s, generator=g, device=DEV)
    q, k, v, do = rnd(B, S, G * Hkv, D), rnd(B, Skv, Hkv, D), rnd(B, Skv, Hkv, D), rnd(B, S, G * Hkv, D)
    # repeats, padding and out-of-range ids in between, one masked row
    idx = torch.randint(-Skv // 8, Skv + Skv // 16, (B, S, Hkv, K), generator=g, device=DEV, dtype=torch.int32)
    idx[0, 1] = -1
    lens = torch.randint(max(1, Skv // 2), Skv + 1, (B,), generator=g, device=DEV, dtype=torch.int32)
    return q, k, v, do, idx, lens


def _rel(a, b):
    b = b.double()
    return float((a.double().cpu() - b).norm() / b.norm())


# edges of the 16-key tiles, of 4-slot steps, of the 64 slots loaded ahead, of the 256-slot windows and 16-head groups
@pytest.mark.parametrize("D,G,Hkv,K,shared", [
    (64, 1, 2, 1, False), (64, 4, 1, 15, True), (64, 5, 1, 64, False), (64, 16, 1, 65, True), (64, 17, 1, 255, True),
    (128, 2, 2, 16, False), (128, 16, 1, 257, True), (128, 40, 1, 30, False), (128, 7, 2, 600, False)])
def test_against_float64(D, G, Hkv, K, shared):
    q, k, v, do, idx, lens = _inputs(2, 9, 300, G, Hkv, D, K, seed=D + G + K)
    if shared:
        v = k
    sink = torch.linspace(-1.0, 2.0, G * Hkv, device=DEV) if K % 2 else None
    out, lse = ops_amd.sfa_forward(q, k, v, idx, kv_lens=lens, attn_sink=sink)
    c = [x.cpu() for x in (q, k, v, idx)]
    cs = dict(kv_lens=lens.cpu(), sink=None if sink is None else sink.cpu(), dtype=torch.float64)
    o_ref, l_ref = ref_forward(*c, **cs)
    assert _rel(out, o_ref) < TOL
    fin = torch.isfinite(l_ref)
    assert torch.equal(torch.isfinite(lse.cpu()), fin) and _rel(lse.cpu()[fin], l_ref[fin]) < TOL
    ref = ref_backward(*c, o_ref, l_ref, do.cpu().double(), **cs)
    got = ops_amd.sfa_backward(q, k, v, idx, out, lse, do, kv_lens=lens, attn_sink=sink, merge_kv=shared)
    if shared:
        ref = (ref[0], ref[1] + ref[2], None, ref[3])
    for a, b in zip(got, ref):
        if a is not None:
            assert _rel(a, b) < TOL


@pytest.mark.parametrize("D", [64, 128])
def test_error_is_no_larger_than_the_scalar_kernels(D):
    """Scores and dP are summed as trees over the dims, like the scalar kernels'
    lanes (rows that are not 16-byte aligned run on those): the error against
    float64 of out, dq and dk is at most theirs, up to the spread between two
    sets of independent roundings (a tenth; one running sum over the dims has
    1.2 and 1.6 times theirs at 64 and 128)."""
    q, k, v, do, idx, _ = _inputs(2, 64, 300, 16, 1, D, 128, seed=D)
    idx = torch.rand((2, 64, 1, 300), device=DEV).argsort(-1)[..., :128].int()
    odd = torch.empty((2, 300, 1, D + 1), device=DEV)[..., :D]
    odd.copy_(k)
    c = [x.cpu() for x in (q, k, k, idx)]
    o_ref, l_ref = ref_forward(*c, dtype=torch.float64)
    ref = ref_backward(*c, o_ref, l_ref, do.cpu().double(), dtype=torch.float64)
    err = []
    for kv in (k, odd):
        out, lse = ops_amd.sfa_forward(q, kv, kv, idx)
        dq, dk, _, _ = ops_amd.sfa_backward(q, kv, kv, idx, out, lse, do, merge_kv=True)
        err.append([_rel(out, o_ref), _rel(dq, ref[0]), _rel(dk, ref[1] + ref[2])])
    assert all(x <= 1.1 * y for x, y in zip(*err)), err


def test_gradient_strides_and_unaligned_rows():
    """Gradients go straight into the caller's tensors (any strides); rows that
    are not 16-byte aligned take the scalar kernels, with the same result."""
    q, k, v, do, idx, _ = _inputs(2, 20, 100, 8, 2, 64, 40, seed=3)
    out, lse = ops_amd.sfa_forward(q, k, v, idx)
    a = ops_amd.sfa_backward(q, k, v, idx, out, lse, do)
    dk = torch.full((100, 2, 2, 67), 7.0, device=DEV)
    dv = torch.full((2, 2, 100, 65), 7.0, device=DEV)
    b = ops_amd.sfa_backward(q, k, v, idx, out, lse, do, dk=dk.permute(1, 0, 2, 3)[..., :64],
                             dv=dv.permute(0, 2, 1, 3)[..., :64])
    assert all(_rel(x, y.cpu()) < TOL for x, y in zip(a[:3], b[:3]))
    assert bool((dk[..., 64:] == 7.0).all()) and bool((dv[..., 64:] == 7.0).all())
    odd = torch.randn((2, 100, 2, 65), device=DEV)[..., :64]
    odd.copy_(k)
    o2, l2 = ops_amd.sfa_forward(q, odd, v, idx)
    assert _rel(o2, out.cpu()) < TOL and torch.equal(torch.isfinite(l2), torch.isfinite(lse))
    c = ops_amd.sfa_backward(q, odd, v, idx, out, lse, do)
    assert all(_rel(x, y.cpu()) < TOL for x, y in zip(c[:3], a[:3]))


def test_infinite_rows_and_pages():
    q, k, v, _, idx, _ = _inputs(1, 3, 256, 16, 1, 64, 90, seed=4)
    kp, vp, bt = page_kv(k, v, 32, seed=1, spare_pages=2)
    a, b = ops_amd.sfa_forward(q, k, v, idx), ops_amd.sfa_forward_paged(q, kp, vp, bt, idx)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    # a selected row with infinite entries and a score of -inf is left out
    idx = idx.clamp(0, 254)
    drop = idx.clone()
    idx[..., 17] = 255
    drop[..., 17] = -1
    k[0, 255] = 0
    k[0, 255, 0, 3] = float("inf")
    v[0, 255] = float("inf")
    q[..., 3] = -1.0
    got, want = ops_amd.sfa_forward(q, k, v, idx)[0], ops_amd.sfa_forward(q, k, v, drop)[0]
    assert _rel(got, want.cpu()) < TOL


def test_pages_over_several_windows():
    """More than one 256-slot window, pages in between, one page unmapped."""
    q, k, v, _, idx, lens = _inputs(2, 5, 512, 20, 1, 128, 700, seed=8)
    kp, vp, bt = page_kv(k, v, 16, seed=1, spare_pages=2)
    bt[1, 4] = -1
    drop = idx.clone()
    drop[1][(drop[1] >= 64) & (drop[1] < 80)] = -1
    a = ops_amd.sfa_forward(q, k, v, drop, kv_lens=lens)
    b = ops_amd.sfa_forward_paged(q, kp, vp, bt, idx, kv_lens=lens)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    o_ref, _ = ref_forward(q.cpu(), k.cpu(), v.cpu(), drop.cpu(), kv_lens=lens.cpu(), dtype=torch.float64)
    assert _rel(b[0], o_ref) < TOL


@pytest.mark.parametrize("K", [8192, 8193])
def test_longest_rows_and_beyond(K):
    """8192 slots are the matrix kernels' longest rows, the scalar kernels take
    8193.  (Sums of 8192 terms of random sign: sqrt(8192) * 2^-24 = 5.4e-6.)"""
    q, k, v, do, idx, _ = _inputs(1, 2, 900, 4, 1, 64, K, seed=9)
    idx[0, 1] = torch.arange(K, device=DEV) % 1000 - 50
    out, lse = ops_amd.sfa_forward(q, k, v, idx)
    c = [x.cpu() for x in (q, k, v, idx)]
    o_ref, l_ref = ref_forward(*c, dtype=torch.float64)
    assert _rel(out, o_ref) < TOL and _rel(lse, l_ref) < TOL
    ref = ref_backward(*c, o_ref, l_ref, do.cpu().double(), dtype=torch.float64)
    for x, y in zip(ops_amd.sfa_backward(q, k, v, idx, out, lse, do)[:3], ref):
        assert _rel(x, y) < TOL


def test_rows_without_a_finite_score_have_no_gradient():
    """A query whose only selected key scores -inf has lse = -inf: its dq is 0
    and it adds nothing to dk / dv, whatever the key's rows hold."""
    q, k, v, do, idx, _ = _inputs(1, 4, 64, 8, 1, 64, 20, seed=6)
    idx = idx.clamp(0, 62)
    q[0, 2, :, 3] = -1.0
    k[0, 63] = 0
    k[0, 63, 0, 3] = float("inf")
    v[0, 63] = float("inf")
    idx[0, 2] = -1
    idx[0, 2, 0, 5] = 63
    out, lse = ops_amd.sfa_forward(q, k, v, idx)
    assert bool((lse[0, 2] == -float("inf")).all()) and bool((out[0, 2] == 0).all())
    dq, dk, dv, _ = ops_amd.sfa_backward(q, k, v, idx, out, lse, do)
    assert bool((dq[0, 2] == 0).all()) and all(bool(torch.isfinite(x).all()) for x in (dq, dk, dv))
