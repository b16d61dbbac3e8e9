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


def _same_union_lists(n, h, k, seed, keep, last=False, duplicates=False):
    """Two sets of lists with the same union (2k blocks) per group of four query blocks and the same lists for half ``keep``
    of it.  Each half names 1.5k blocks in the first set; in the second the other half names the whole union, so that the
    group keeps to the common walk.  No two blocks of a union share a slot of the kernel's table, so that the order of the
    walk does not depend on which list names a block first."""
    g = torch.Generator().manual_seed(seed)
    nb, nqb = n // 16, -(-n // 16)
    slot = [(e * 0x9E3779B1 % 2 ** 32) >> 23 for e in range(nb)]
    lists = torch.full((2, 1, h, nqb, k), -1, dtype=torch.int32)
    for head in range(h):
        for grp in range(-(-nqb // 4)):
            by_slot = {slot[e]: e for e in torch.randperm(nb, generator=g).tolist()}
            union = torch.tensor(list(by_slot.values()), dtype=torch.int32)[:2 * k]
            named = {keep: (union[:3 * k // 2],) * 2, 1 - keep: (union[k // 2:], union)}
            for half, both in named.items():
                for which, blocks in enumerate(both):
                    blocks = blocks[torch.randperm(len(blocks), generator=torch.Generator().manual_seed(grp))]
                    parts = blocks[:k], torch.cat((blocks[k:], blocks[:k // 4 if len(blocks) < 2 * k else 0]))
                    for j, part in enumerate(parts):
                        m = 4 * grp + 2 * half + j
                        if m < nqb:
                            lists[which, 0, head, m, :len(part)] = part
                            if j == 1 and half == keep and last:
                                lists[which, 0, head, m, -1] = nqb - 1
                            if j == 1 and half == keep and duplicates:
                                lists[which, 0, head, m, -2] = part[0]
    return lists


@pytest.mark.parametrize("dtype,size", [(torch.bfloat16, 1.0), (torch.float16, 1.0), (torch.float16, 3.5), (torch.bfloat16, 9.0)])
@pytest.mark.parametrize("keep", [0, 1])
@pytest.mark.parametrize("n,k,extra", [(4096, 32, {}), (4105, 32, {"last": True}), (2048, 16, {"duplicates": True}), (8192, 64, {})])
def test_block16_result_does_not_depend_on_the_walk(dtype, size, keep, n, k, extra):
    """A half's queries get the same bits from the walk per half and from the common walk over the same union: the same
    order of additions, and each query's softmax reference from the same blocks.  ``size`` 3.5 and 9: row sums beyond the
    bound, the groups start over with the running maximum."""
    h = 2
    lists = _same_union_lists(n, h, k, n + keep, keep, **extra)
    g = torch.Generator().manual_seed(n + k)
    q, kk, v = ((torch.randn((1, h, n, 64), generator=g) * s).to(dtype).to(DEV) for s in (size, size, 1.0))
    (o, lse), (o_common, lse_common) = (s3r.select_attn(q, kk, v, idx.to(DEV), 16, return_lse=True) for idx in lists)
    rows = (torch.arange(n) // 32 % 2 == keep) & (torch.arange(n) < n // 64 * 64)    # of whole groups
    assert torch.equal(o[:, :, rows], o_common[:, :, rows])
    assert torch.equal(lse[:, :, rows], lse_common[:, :, rows])
