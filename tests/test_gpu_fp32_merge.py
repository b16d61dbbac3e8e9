"""GPU: the gated merge in the fp32 selection kernels' epilogues against the two operators, bit for bit: each block size, ragged ends,
blocks in halves, more than 384 blocks of 64 (split values, and values that do not split), entries that are skipped, strided gates; tensors
that only the two operators take."""
import pytest
import torch

import speed3r_amd as s3r
from speed3r_amd.sparse_attn import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("b,h,n,kk,block", [(1, 1, 1, 1, 64), (2, 2, 200, 3, 64), (1, 16, 1041, 16, 64), (1, 64, 256, 4, 64), (1, 16, 1601, 16, 64), (2, 64, 250, 4, 64), (2, 3, 100, 2, 32), (2, 2, 203, 8, 16),
                                            (1, 2, 300, 2, 128)])
def test_merge_equals_the_two_operators(b, h, n, kk, block):
    g = torch.Generator(device=DEV).manual_seed(n)
    q, k, v = torch.randn((3, b, h, n, 64), generator=g, device=DEV).unbind(0)
    nb = -(-n // block)
    idx = torch.randint(-1, nb + 1, (b, h, nb, kk), generator=g, device=DEV, dtype=torch.int32)
    oc = torch.randn((b, h, nb, 64), generator=g, device=DEV)
    gate = torch.rand((b, n, h, 2), generator=g, device=DEV).permute(0, 2, 1, 3)
    want = s3r.gated_merge(oc, s3r.select_attn(q, k, v, idx, block), gate, block)
    got = ops._select_attn_merge(q, k, v, idx, oc, gate, block)
    assert got is not None and torch.equal(got, want)
    odd = torch.empty(oc.numel() + 1, device=DEV)[1:].view(oc.shape).copy_(oc)   # not at 16 bytes
    if block < 128:
        assert ops._select_attn_merge(q, k, v, idx, odd, gate, block) is None


@pytest.mark.parametrize("what,value", [("k", 2.0 ** 61), ("v", 2.0 ** 61), ("v", float("inf")), ("v", 1e-35)])
def test_merge_of_values_that_do_not_split(what, value):
    g = torch.Generator(device=DEV).manual_seed(4)
    t = dict(zip("qkv", torch.randn((3, 2, 100, 250, 64), generator=g, device=DEV).unbind(0)))
    t["q"][..., 5] = 0.0
    t[what][1, 7, 130, 5] = value
    idx = torch.randint(-1, 5, (2, 100, 4, 3), generator=g, device=DEV, dtype=torch.int32)
    idx[1, 7, :, 0] = 2
    oc = torch.randn((2, 100, 4, 64), generator=g, device=DEV)
    gate = torch.rand((2, 250, 100, 2), generator=g, device=DEV).permute(0, 2, 1, 3)
    o = s3r.select_attn(t["q"], t["k"], t["v"], idx, 64)
    got = ops._select_attn_merge(t["q"], t["k"], t["v"], idx, oc, gate, 64)
    assert bool(torch.isinf(o).any()) == (value == float("inf")) and not bool(torch.isnan(o).any())
    assert got is not None and torch.equal(got, s3r.gated_merge(oc, o, gate, 64))
