"""The workgroup placement by kv head and XCD (d = 128, up to 16 heads per kv
head) is a permutation of the items: every head's rows equal, bitwise, those
of a call with that kv head alone."""
import pytest
import torch

import ops_amd

pytestmark = pytest.mark.gpu
DEV = "cuda"


# queries in whole rounds of runs, in runs and a remainder, in a remainder only; head counts with and without an XCD each
@pytest.mark.parametrize("B,S,Hkv", [(1, 256, 1), (2, 150, 2), (1, 77, 4), (2, 131, 8), (1, 100, 3), (1, 31, 8)])
def test_items_by_head(B, S, Hkv):
    g = torch.Generator(device=DEV).manual_seed(S)
    G, D, K = 4, 128, 64
    q, do = (torch.randn((B, S, G * Hkv, D), generator=g, device=DEV).bfloat16() for _ in range(2))
    k, v = (torch.randn((B, S, Hkv, D), generator=g, device=DEV).bfloat16() for _ in range(2))
    idx = torch.rand((B, S, Hkv, max(S, K)), generator=g, device=DEV).argsort(-1)[..., :K].int()  # (ids past S: invalid)
    out = torch.full_like(q, float("nan"))
    out, lse = ops_amd.sfa_forward(q, k, v, idx, out=out, num_splits=1)
    dq = ops_amd.sfa_backward(q, k, v, idx, out, lse, do)[0]
    for h in range(Hkv):
        hs = slice(h * G, (h + 1) * G)
        one = [x.contiguous() for x in (q[:, :, hs], k[:, :, h:h + 1], v[:, :, h:h + 1], idx[:, :, h:h + 1])]
        o1, l1 = ops_amd.sfa_forward(*one, num_splits=1)
        assert torch.equal(o1, out[:, :, hs]) and torch.equal(l1, lse[:, :, hs])
        assert torch.equal(ops_amd.sfa_backward(*one, o1, l1, do[:, :, hs].contiguous())[0], dq[:, :, hs])


def test_mla_ascending_rows_below_the_persistent_kernel():
    """128 heads, 1024 queries on 8192 keys: the library's ascending rows give
    bitwise what rows sorted by the caller give."""
    g = torch.Generator(device=DEV).manual_seed(0)
    q = torch.randn((1, 1024, 128, 576), generator=g, device=DEV).bfloat16()
    kv = torch.randn((1, 8192, 1, 576), generator=g, device=DEV).bfloat16()
    idx = torch.stack([torch.randperm(8192, generator=g, device=DEV)[:1024] for _ in range(1024)]).view(1, 1024, 1, 1024)
    a = ops_amd.sfa_forward(q, kv, kv[..., :512], idx.int())
    b = ops_amd.sfa_forward(q, kv, kv[..., :512], idx.sort(-1).values.int(), idx_sorted=True)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
