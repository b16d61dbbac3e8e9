"""GPU: key-block lists of every length at which their sort changes (one entry per lane, networks of 128, 256 and 512, the workgroup's
sort beyond), with repeated entries, against a stable sort on the host.  Whole numbers: equal."""
import pytest
import torch

from speed3r_amd.sparse_attn import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513])
def test_lists_of_length(n):
    gen = torch.Generator().manual_seed(n)
    nqb, k, nkb = 600, 4, 9
    idx = torch.full((2, 1, nqb * k), nkb, dtype=torch.int32)      # (beyond the last block: in no list)
    for b in range(2):                                              # block 3 n times, its neighbours once more and once less
        where = torch.randperm(nqb * k, generator=gen)
        idx[b, 0, where[:n]] = 3
        idx[b, 0, where[n:2 * n + 1]] = 4
        idx[b, 0, where[2 * n + 1:3 * n]] = 7
    idx = idx.view(2, 1, nqb, k)
    lists, off = (t.cpu() for t in ops.key_block_lists(idx.cuda(), nkb))
    for b in range(2):
        at = 0
        for j in range(nkb):
            want = (idx[b, 0] == j).nonzero()[:, 0]                 # row by row: ascending, a row once per entry
            assert off[b, 0, j] == at and torch.equal(lists[b, 0, at:at + len(want)].long(), want)
            at += len(want)
        assert off[b, 0, nkb] == at


# entries per head on both sides of the line between the kernels that make the lists; key blocks that the workgroups of a head share unevenly,
# fewer of them than workgroups, more heads than CUs; strided index rows, entries that are skipped; a workgroup's key blocks with one counter
# a thread and with more, up to the most that it takes (64 KB of counters) and one beyond; one head's many entries over the block counts that the
# two ways share
@pytest.mark.parametrize("bh,nqb,k,nkb", [(1, 4096, 32, 4096), (1, 4097, 32, 300), (3, 1000, 5, 1), (2, 777, 16, 3), (16, 130, 8, 131), (300, 20, 4, 20),
                                          (1, 50, 2, 70000), (2, 100, 64, 20000), (256, 40, 4, 1024), (256, 40, 4, 1025), (257, 40, 3, 2047),
                                          (128, 90, 7, 5000), (256, 90, 5, 16384), (256, 90, 5, 16385), (1, 6144, 16, 8192), (1, 6145, 16, 8192),
                                          (1, 6145, 16, 8193), (1, 6145, 16, 4096)])
def test_lists_of_heads(bh, nqb, k, nkb):
    gen = torch.Generator().manual_seed(nqb)
    wide = torch.randint(-2, nkb + 2, (1, bh, nqb, k + 3), generator=gen, dtype=torch.int32)
    wide = torch.where(torch.rand(wide.shape, generator=gen) < 0.2, wide.clamp(max=nkb // 3), wide)
    idx = wide.cuda()[..., :k]
    lists, off = (t.cpu()[0] for t in ops.key_block_lists(idx, nkb))
    for b in range(bh):
        e = wide[0, b, :, :k].reshape(-1).long()
        ok = (e >= 0) & (e < nkb)
        order = torch.sort(e[ok], stable=True)
        rows = torch.arange(nqb).repeat_interleave(k)[ok][order.indices]
        assert torch.equal(off[b].long(), torch.cat((torch.zeros(1, dtype=torch.long), torch.bincount(e[ok], minlength=nkb).cumsum(0))))
        assert torch.equal(lists[b, :len(rows)].long(), rows)
