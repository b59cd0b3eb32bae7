"""The chunk length of the key-major dK/dV scheme follows the call's size (4 to
128 query blocks): sizes on both sides of each step and with a partial last
chunk, against the fp32-atomic scheme.

Tolerance: both round P, dS and the result to bf16 (2^-9 relative each, random
signs), so they differ by well under 2^-8 of the gradient's norm."""
import pytest
import torch

import ops_amd

pytestmark = pytest.mark.gpu
DEV = "cuda"


# (causal (key block, query block) pairs / 512: 0.3, 2.1, 5.9, 6.2, 23.8, 24.4, 192 and above; D, B, S, heads, kv heads, K)
@pytest.mark.parametrize("D,B,S,Hq,Hkv,K", [
    (128, 1, 300, 16, 1, 96), (128, 1, 1030, 16, 1, 200), (64, 1, 1700, 16, 1, 300), (128, 1, 1790, 16, 1, 130),
    (128, 1, 1750, 64, 1, 100), (128, 1, 1800, 128, 2, 70), (128, 1, 5025, 128, 1, 90),
    (128, 2, 8300, 64, 8, 130)])  # (the last: chunks of 64 blocks would take 1.2 GB of partials, so 128)
def test_chunks(D, B, S, Hq, Hkv, K):
    g = torch.Generator(device=DEV).manual_seed(S)
    q, do = (torch.randn((B, S, Hq, D), generator=g, device=DEV).bfloat16() for _ in range(2))
    k, v = (torch.randn((B, S, Hkv, D), generator=g, device=DEV).bfloat16() for _ in range(2))
    idx = torch.stack([torch.randperm(S, generator=g, device=DEV)[:K] for _ in range(64)]).to(torch.int32)
    idx = idx[torch.randint(0, 64, (B, S, Hkv), generator=g, device=DEV)]
    idx = torch.where(idx <= torch.arange(S, device=DEV)[None, :, None, None], idx, -1)  # causal, padding in between
    out, lse = ops_amd.sfa_forward(q, k, v, idx)
    a = ops_amd.sfa_backward(q, k, v, idx, out, lse, do)
    b = ops_amd.sfa_backward(q, k, v, idx, out, lse, do, dkv_mode="atomic")
    for x, y in zip(a[:3], b[:3]):
        assert float((x.double() - y.double()).norm() / y.double().norm()) < 2.0 ** -8
    again = ops_amd.sfa_backward(q, k, v, idx, out, lse, do)
    assert all(torch.equal(x, y) for x, y in zip(a[:3], again[:3]))
