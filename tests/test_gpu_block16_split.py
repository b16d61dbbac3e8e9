"""16-token blocks: the walk per half of a wave's 64 queries (lists that share little) at the sizes where it can go
wrong, against the oracle.  A wave takes it where the longer half's list is a small part of the union of its four lists;
the lists here draw the two halves' entries from disjoint ranges of blocks, which makes every such group take it."""
import pytest
import torch

import oracle
import speed3r_amd as s3r
from helpers import max_abs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _lists(n, h, k, n0, n1, seed, duplicates=False, last=False):
    """[1,h,nqb,k] lists: query blocks 0, 1 (2, 3) of a group name n0 (n1) distinct blocks of the lower (upper) part."""
    g = torch.Generator().manual_seed(seed)
    nqb = -(-n // 16)
    idx = torch.full((1, h, nqb, k), -1, dtype=torch.int32)
    for head in range(h):
        for grp in range(-(-nqb // 4)):
            for half, (lo, cnt) in enumerate(((0, n0), (nqb // 2, n1))):
                blocks = lo + torch.randperm(nqb // 2, generator=g)[:cnt].to(torch.int32)
                if half == 1 and last:
                    blocks[0] = nqb - 1                                   # the (ragged) block that ends the sequence
                for j, part in enumerate((blocks[:k], blocks[k:2 * k])):
                    m = 4 * grp + 2 * half + j
                    if m < nqb:
                        idx[0, head, m, :len(part)] = part
                        if duplicates and 0 < len(part) < k:
                            idx[0, head, m, -1] = part[0]
    return idx


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,k,n0,n1,extra", [
    (2048, 32, 64, 64, {}),                       # full lists, one tile per two blocks
    (2048, 32, 63, 1, {}),                        # an odd list beside a single block (too unequal for the split: one walk)
    (2048, 32, 33, 27, {}),                       # the shorter list ends first
    (4096, 64, 128, 127, {}),                     # the longest lists there are
    (96, 1, 2, 2, {}), (96, 1, 1, 1, {}),         # one tile per half
    (96, 2, 3, 3, {}),                            # two tiles, the second one half full
    (1033, 16, 20, 21, {"last": True}),           # ragged last block listed, group tail of one query block
    (1040, 16, 17, 12, {"duplicates": True}),     # blocks that count twice
    (1040, 16, 32, 0, {}),                        # a half that attends nothing (one walk)
])
def test_block16_lists_that_share_little_match_oracle(dtype, n, k, n0, n1, extra):
    h = 2
    g = torch.Generator().manual_seed(n + k)
    q, kk, v = ((torch.randn((1, h, n, 64), generator=g) * s).to(dtype) for s in (0.5, 0.5, 1.0))
    idx = _lists(n, h, k, n0, n1, 3 * n + k, **extra)
    o, lse = s3r.select_attn(q.to(DEV), kk.to(DEV), v.to(DEV), idx.to(DEV), 16, return_lse=True)
    want, lse_want = oracle.select_attention(q, kk, v, idx, 16, out_dtype=torch.float32, return_lse=True)
    assert max_abs(o, want) <= 2e-2                       # the bound of the operator's other parity tests at these inputs
    fin = torch.isfinite(lse_want)
    assert torch.equal(torch.isfinite(lse.cpu()), fin) and max_abs(lse.cpu()[fin], lse_want[fin]) <= 2e-3


@pytest.mark.parametrize("gain", [12.0, 2.0])
def test_block16_split_walk_handles_scores_far_above_the_reference(gain):
    """Blocks listed last line up with the queries: row sums beyond the bound, second walk with the running maximum."""
    n, h, k = 512, 2, 8
    g = torch.Generator().manual_seed(5)
    q = torch.randn((1, h, n, 64), generator=g).to(torch.bfloat16)
    kk = (torch.randn((1, h, n, 64), generator=g) * 0.01).to(torch.bfloat16)
    kk[:, :, 64:128] = (q[:, :, 0:64] * gain).to(torch.bfloat16)
    kk[:, :, 448:512] = (q[:, :, 0:64] * gain).to(torch.bfloat16)
    v = torch.randn((1, h, n, 64), generator=g).to(torch.bfloat16)
    idx = _lists(n, h, k, 12, 12, 9)
    idx[:, :, :2, 0] = torch.tensor([4, 5], dtype=torch.int32)
    idx[:, :, 2:4, 0] = torch.tensor([30, 31], dtype=torch.int32)
    o = s3r.select_attn(q.to(DEV), kk.to(DEV), v.to(DEV), idx.to(DEV), 16)
    assert torch.isfinite(o.float()).all()
    assert max_abs(o, oracle.select_attention(q, kk, v, idx, 16, out_dtype=torch.float32)) <= 2e-2
