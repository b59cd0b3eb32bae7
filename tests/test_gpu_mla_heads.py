"""MLA rows (576 / 512) with up to 64 query heads, one rank of a head-parallel
group (``fwd_mla_g_kernel``), against the fp32 oracle.

Tolerance: the output is rounded to bf16 (half an ulp, 2^-8 of the value at
most once the fp32 sum differs too) and the products are summed in fp32, so a
sum of weights 1 over rows of magnitude up to ~5 is off by far less than 2^-14.
LSE is an fp32 sum of the score products: 1e-4 absolute."""
import pytest
import torch

import ops_amd
from ops_amd.workloads import page_kv
from oracle.sfa_oracle import sfa_forward as ref_forward

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(B, Sq, Skv, Hq, Hkv, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    q = torch.randn((B, Sq, Hq, 576), generator=g, device=DEV).bfloat16()
    kv = torch.randn((B, Skv, Hkv, 576), generator=g, device=DEV).bfloat16()
    # any order, padding and out-of-range ids in between, one masked row
    idx = torch.randint(-Skv // 8, Skv + Skv // 16, (B, Sq, Hkv, K), generator=g, device=DEV, dtype=torch.int32)
    idx[0, 0, 0] = -1
    lens = torch.randint(max(1, Skv // 2), Skv + 1, (B,), generator=g, device=DEV, dtype=torch.int32)
    return q, kv, idx, lens


def _check(out, lse, ref):
    o_ref, l_ref = ref
    out, lse = out.float().cpu(), lse.cpu()
    assert bool(((out - o_ref).abs() <= o_ref.abs() * 2.0 ** -8 + 2.0 ** -14).all())
    fin = torch.isfinite(l_ref)
    assert torch.equal(torch.isfinite(lse), fin)
    assert float((lse - l_ref)[fin].abs().max()) <= 1e-4


# tile edges (31 / 32 / 33), the 256-slot halves of the staged index ring (255 .. 257, 513, 2049), group edges
@pytest.mark.parametrize("G,Hkv,K,splits", [
    (1, 1, 1, 0), (5, 2, 31, 1), (16, 1, 32, 1), (16, 1, 33, 0), (16, 1, 255, 1), (16, 2, 257, 1), (16, 1, 513, 3),
    (17, 1, 256, 1), (32, 1, 2049, 1), (32, 2, 300, 8), (33, 1, 224, 1), (48, 1, 2049, 5), (64, 1, 700, 1),
    (64, 1, 96, 2), (16, 1, 2500, 64)])
def test_heads_and_slots(G, Hkv, K, splits):
    q, kv, idx, lens = _inputs(3, 3, 900, G * Hkv, Hkv, K, seed=G * 7 + K)
    sink = torch.linspace(-2.0, 3.0, G * Hkv, device=DEV) if K % 2 else None
    out = torch.full(q.shape[:3] + (512,), float("nan"), dtype=q.dtype, device=DEV)
    out, lse = ops_amd.sfa_forward(q, kv, kv[..., :512], idx, 0.05, kv_lens=lens, attn_sink=sink, num_splits=splits,
                                   out=out)
    ref = ref_forward(q.cpu(), kv.cpu(), kv[..., :512].cpu(), idx.cpu(), 0.05, kv_lens=lens.cpu(),
                      sink=None if sink is None else sink.cpu())
    _check(out, lse, ref)


@pytest.mark.parametrize("G,Sq,K,splits", [(16, 3, 600, 0), (32, 1, 2049, 4), (64, 2, 300, 1)])
def test_paged_is_contiguous(G, Sq, K, splits):
    q, kv, idx, lens = _inputs(4, Sq, 1024, G, 1, K, seed=G)
    kp, vp, bt = page_kv(kv, kv[..., :512], 64, seed=3, spare_pages=3)
    a = ops_amd.sfa_forward(q, kv, kv[..., :512], idx, 0.05, kv_lens=lens, num_splits=splits)
    b = ops_amd.sfa_forward_paged(q, kp, vp, bt, idx, 0.05, kv_lens=lens, num_splits=splits)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    bt[1, 3] = -1  # an unmapped page drops its slots
    drop = idx.clone()
    drop[1][(drop[1] >= 192) & (drop[1] < 256)] = -1
    a = ops_amd.sfa_forward(q, kv, kv[..., :512], drop, 0.05, kv_lens=lens, num_splits=splits)
    b = ops_amd.sfa_forward_paged(q, kp, vp, bt, idx, 0.05, kv_lens=lens, num_splits=splits)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


@pytest.mark.parametrize("splits", [1, 3])
def test_infinite_rows(splits):
    """A selected row with an infinite entry: heads whose score is -inf leave
    it out, heads whose score is +inf have no finite answer, as a scalar
    evaluation of the sum gives."""
    q, kv, idx, _ = _inputs(1, 2, 300, 16, 1, 96, seed=1)
    idx = idx.clamp(0, 298)
    idx[..., 40] = 299
    kv[0, 299] = 0
    kv[0, 299, 0, 7] = float("inf")
    q[..., 7] = torch.where(torch.arange(16, device=DEV) % 2 == 0, -1.0, 1.0)
    out, _ = ops_amd.sfa_forward(q, kv, kv[..., :512], idx, 0.05, num_splits=splits)
    kv[0, 299] = 0
    idx[..., 40] = -1
    o_ref, _ = ref_forward(q.cpu(), kv.cpu(), kv[..., :512].cpu(), idx.cpu(), 0.05)
    err = (out.float().cpu() - o_ref)[:, :, ::2].abs()
    assert bool((err <= o_ref[:, :, ::2].abs() * 2.0 ** -8 + 2.0 ** -14).all())
    assert bool(torch.isnan(out[:, :, 1::2]).all())


@pytest.mark.parametrize("sink", [None, 0.5, float("nan"), float("inf")])
@pytest.mark.parametrize("what", ["nan query", "inf query", "nan cache", "one nan key"])
@pytest.mark.parametrize("Hq", [16, 40, 128])
def test_rows_that_are_not_numbers_survive_the_merge(Hq, what, sink):
    """Whatever the split count, a row is NaN where the unsplit call's is, and
    has its log-sum-exp: also when no split has a finite sum (a NaN or infinite
    query, a cache of NaN).  (128 heads: 4 queries, the most that take this
    kernel.)"""
    q, kv, idx, _ = _inputs(2, 2, 300, Hq, 1, 200, seed=Hq)
    idx[0, 0, 0] = torch.arange(200, device=DEV)
    if what == "nan query":
        q[0, 1, 3, 575] = float("nan")
        q[1, 0, Hq - 1] = float("nan")
    elif what == "inf query":
        q[0, 1, 3, 575] = float("inf")
    elif what == "nan cache":
        kv[1] = float("nan")
    else:
        kv[0, 7, 0, 0] = float("nan")
    s = None if sink is None else torch.full((Hq,), sink, device=DEV)
    call = lambda n: ops_amd.sfa_forward(q, kv, kv[..., :512], idx, 0.05, attn_sink=s, num_splits=n)
    o_ref, l_ref = call(1)
    bad = torch.isnan(o_ref).any(-1)
    assert bool(bad.any()) and bool((l_ref[bad] == float("-inf")).all())
    for n in (0, 3, 64):
        out, lse = call(n)
        assert torch.equal(torch.isnan(out), torch.isnan(o_ref)), n
        ok = torch.isfinite(o_ref)
        assert float((out.float() - o_ref.float())[ok].abs().max()) <= 2.0 ** -7 * float(o_ref[ok].float().abs().max()), n
        assert torch.equal(torch.isfinite(lse), torch.isfinite(l_ref)) and not bool(torch.isnan(lse).any()), n
        fin = torch.isfinite(l_ref)
        assert not bool(fin.any()) or float((lse - l_ref)[fin].abs().max()) <= 1e-4, n


@pytest.mark.parametrize("B,Sq,Hq,K,splits", [(1, 256, 16, 2048, 1), (1, 128, 64, 1100, 1), (8, 1, 32, 1500, 0), (2, 1, 128, 1500, 0)])
def test_error_is_the_outputs_rounding(B, Sq, Hq, K, splits):
    """P in all its 24 bits: at most 6e-4 of the outputs are not the bf16 value
    nearest to the float64 result (an fp32 evaluation's own share, 2^-20 of the
    value against a bf16 step of 2^-8, is 2e-4 to 5e-4; P in 17 bits has 1.6e-3
    and more), and the LSE is off by less than 2^-24 of itself in the 2-norm."""
    q, kv, idx, _ = _inputs(B, Sq, 4096, Hq, 1, K, seed=K)
    idx[0, 0] = idx[0, Sq - 1] if Sq > 1 else torch.arange(K, device=DEV)
    idx = idx.clamp(min=-1, max=4095)
    out, lse = ops_amd.sfa_forward(q, kv, kv[..., :512], idx, 576 ** -0.5, num_splits=splits)
    off = n = 0
    el = torch.empty(lse.shape, dtype=torch.float64, device=DEV)
    for b in range(B):
        for t in range(Sq):
            ids = idx[b, t, 0].long()
            rows = kv[b, ids[ids >= 0], 0].double()
            s = (q[b, t].double() @ rows.T) * float(torch.tensor(576 ** -0.5, dtype=torch.float32))
            el[b, t] = torch.logsumexp(s, 1)
            o = torch.softmax(s, 1) @ rows[:, :512]
            off += int((out[b, t] != o.bfloat16()).sum())
            n += o.numel()
    assert off / n < 6e-4, off / n
    assert float((lse.double() - el).norm() / el.norm()) < 2.0 ** -24


def test_noalloc_splits_to_its_scratch():
    """The static scratch bounds the split count instead of refusing the call."""
    q, kv, idx, _ = _inputs(2, 100, 500, 64, 1, 300, seed=5)
    out = torch.empty(q.shape[:3] + (512,), dtype=q.dtype, device=DEV)
    lse = torch.empty(q.shape[:3], dtype=torch.float32, device=DEV)
    ops_amd.sfa_forward(q, kv, kv[..., :512], idx, 0.05, num_splits=8, out=out, lse=lse, noalloc=True)
    _check(out, lse, ref_forward(q.cpu(), kv.cpu(), kv[..., :512].cpu(), idx.cpu(), 0.05))


# 65..128 heads: up to 4 queries in groups of 16 heads (the last one partly empty), more on the 128-head kernel with 2
# to 8 splits of its own choice, each with its merge
@pytest.mark.parametrize("B,Sq,Hq,Hkv", [(1, 1, 128, 1), (2, 2, 100, 1), (1, 2, 144, 2), (5, 1, 128, 1), (33, 1, 72, 1),
                                         (37, 1, 128, 1), (43, 1, 128, 1), (52, 1, 80, 1), (86, 1, 128, 1)])
def test_few_queries_and_default_splits(B, Sq, Hq, Hkv):
    q, kv, idx, lens = _inputs(B, Sq, 600, Hq, Hkv, 520, seed=B)
    idx[0, 0, 0] = torch.arange(520, device=DEV)  # (not masked: it may be the only row)
    sink = torch.linspace(-2.0, 3.0, Hq, device=DEV)
    out = torch.full(q.shape[:3] + (512,), float("nan"), dtype=q.dtype, device=DEV)
    out, lse = ops_amd.sfa_forward(q, kv, kv[..., :512], idx, 0.05, kv_lens=lens, attn_sink=sink, out=out)
    o_ref, l_ref = ref_forward(q.cpu(), kv.cpu(), kv[..., :512].cpu(), idx.cpu(), 0.05, kv_lens=lens.cpu(),
                               sink=sink.cpu())
    if B * Sq * Hkv <= 4:
        _check(out, lse, (o_ref, l_ref))
    # the 128-head kernel rounds P and its partials to bf16 (2^-9 each, random signs over the slots)
    assert float((out.float().cpu() - o_ref).norm() / o_ref.norm()) < 2.0 ** -7
    fin = torch.isfinite(l_ref)
    assert torch.equal(torch.isfinite(lse.cpu()), fin) and float((lse.cpu() - l_ref)[fin].abs().max()) < 1e-3


# (more than 8 splits of the 128-head kernel's own choice: a long top-k, also for a few queries)
@pytest.mark.parametrize("B,K", [(5, 4200), (2, 8448), (9, 6145)])
def test_long_top_k_splits(B, K):
    q, kv, idx, lens = _inputs(B, 1, 2000, 128, 1, K, seed=K)
    idx[0, 0, 0] = torch.arange(K, device=DEV)
    out, lse = ops_amd.sfa_forward(q, kv, kv[..., :512], idx, 0.05, kv_lens=lens)
    o_ref, l_ref = ref_forward(q.cpu(), kv.cpu(), kv[..., :512].cpu(), idx.cpu(), 0.05, kv_lens=lens.cpu())
    assert float((out.float().cpu() - o_ref).norm() / o_ref.norm()) < 2.0 ** -7  # (P and partials in bf16, as above)
    assert float((lse.cpu() - l_ref).abs().max()) < 1e-3


@pytest.mark.parametrize("G,Sq", [(16, 1301), (24, 1024), (40, 1301)])
def test_many_queries(G, Sq):
    """Unsplit items placed in runs of 32 queries, then by eights, then singly
    (1301 = 1280 + 16 + 5), up to 32 heads on ascending rows: the sorted rows of
    the library equal rows sorted by the caller bitwise; sampled rows against
    the oracle; bitwise the same without allocation where the rows fit."""
    g = torch.Generator(device=DEV).manual_seed(G)
    Skv, K = 8200, 520
    q = torch.randn((1, Sq, G, 576), generator=g, device=DEV).bfloat16()
    kv = torch.randn((1, Skv, 1, 576), generator=g, device=DEV).bfloat16()
    idx = torch.stack([torch.randperm(Skv, generator=g, device=DEV)[:K] for _ in range(Sq)]).view(1, Sq, 1, K).int()
    idx[torch.rand(idx.shape, generator=g, device=DEV) < 0.05] = -1
    out = torch.full(q.shape[:3] + (512,), float("nan"), dtype=q.dtype, device=DEV)
    out, lse = ops_amd.sfa_forward(q, kv, kv[..., :512], idx, 0.05, out=out)
    rows = torch.cat([torch.arange(0, Sq, 97), torch.arange(Sq - 24, Sq)])
    ref = ref_forward(q[:, rows.to(DEV)].cpu(), kv.cpu(), kv[..., :512].cpu(), idx[:, rows.to(DEV)].cpu(), 0.05)
    _check(out[:, rows.to(DEV)], lse[:, rows.to(DEV)], ref)
    assert bool(torch.isfinite(out).all())
    if G <= 32:
        asc = torch.where(idx < 0, Skv, idx).sort(-1).values
        asc = torch.where(asc == Skv, -1, asc).int()
        o2, l2 = ops_amd.sfa_forward(q, kv, kv[..., :512], asc, 0.05, idx_sorted=True)
        assert torch.equal(out, o2) and torch.equal(lse, l2)
    o3, l3 = ops_amd.sfa_forward(q, kv, kv[..., :512], idx, 0.05, noalloc=True)
    assert torch.equal(out, o3) and torch.equal(lse, l3)


@pytest.mark.parametrize("G,Hkv,Sq,paged", [(16, 2, 520, False), (32, 1, 1024, True), (16, 2, 600, True)])
def test_ascending_rows_of_kv_heads_and_pages(G, Hkv, Sq, paged):
    """The library's ascending rows with two kv heads and over pages (one of
    them unmapped): bitwise those that the caller sorts, and on pages bitwise
    the contiguous call's."""
    q, kv, idx, lens = _inputs(1, Sq, 8192, G * Hkv, Hkv, 520, seed=Sq)
    idx = torch.stack([torch.randperm(8192 + 512, device=DEV)[:520] for _ in range(Sq * Hkv)]).view(1, Sq, Hkv, 520).int()
    call = lambda ids, **kw: ops_amd.sfa_forward(q, kv, kv[..., :512], ids, 0.05, kv_lens=lens, **kw)
    n = int(lens[0])
    if paged:
        kp, vp, bt = page_kv(kv, kv[..., :512], 64, seed=2, spare_pages=5)
        bt[0, 7] = -1
        out, lse = ops_amd.sfa_forward_paged(q, kp, vp, bt, idx, 0.05, kv_lens=lens)
        # (the unmapped page's slots keep their place in the ascending row: drop them there)
        key = torch.where(idx < n, idx, 8192)
        asc = key.sort(-1).values
        asc = torch.where((asc >= 448) & (asc < 512), -1, torch.where(asc == 8192, -1, asc)).int()
        ref = call(asc, idx_sorted=True)
    else:
        out, lse = call(idx)
        asc = torch.where(idx < n, idx, 8192).sort(-1).values
        ref = call(torch.where(asc == 8192, -1, asc).int(), idx_sorted=True)
    assert torch.equal(out, ref[0]) and torch.equal(lse, ref[1])
    o_ref, l_ref = ref_forward(q[:, ::97].cpu(), kv.cpu(), kv[..., :512].cpu(), (asc if paged else idx)[:, ::97].cpu(), 0.05,
                               kv_lens=lens.cpu())
    _check(out[:, ::97], lse[:, ::97], (o_ref, l_ref))
