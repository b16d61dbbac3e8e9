"""GPU: the gated merge in the fp32 selection kernel's epilogue against the two operators, bit for bit: each block size, ragged ends,
blocks in halves, entries that are skipped, strided gates; tensors that only the two operators take."""
import pytest
import torch

import speed3r_amd as s3r
from speed3r_amd.sparse_attn import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("b,h,n,kk,block", [(1, 1, 1, 1, 64), (2, 2, 200, 3, 64), (1, 16, 1041, 16, 64), (1, 64, 256, 4, 64), (2, 3, 100, 2, 32), (2, 2, 203, 8, 16),
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
