"""16-token blocks: long walks, where a wave takes one, two and four query blocks (the number of (query block, head) pairs decides), against
the oracle.  The two halves of four neighbouring query blocks draw their lists from disjoint ranges of blocks: unions of up to 64, 128 and
256 distinct blocks a wave, which is all that its table and its list hold."""
from functools import lru_cache

import pytest
import torch

import oracle
import speed3r_amd as s3r
from helpers import max_abs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
PER_WAVE = {1: 1, 2: 5001, 4: 20001}   # query blocks a wave takes: fewest (query block, head) pairs


def _repeats(h, nqb, per_wave):
    """How often ``h`` heads are repeated so that a wave takes ``per_wave`` query blocks."""
    times = max(1, -(-PER_WAVE[per_wave] // (h * nqb)))
    pairs = times * h * nqb
    assert {1: pairs <= 5000, 2: 5000 < pairs <= 20000, 4: pairs > 20000}[per_wave]
    return times


def _attend(q, kk, v, idx, times):
    """Output and log-sum-exp of the first heads; their repetitions have the same bits, and so has the merge in the epilogue."""
    h, nqb = q.shape[1], idx.shape[2]
    q, kk, v, idx = (t.to(DEV).repeat(1, times, 1, 1) for t in (q, kk, v, idx))
    o, lse = s3r.select_attn(q, kk, v, idx, 16, return_lse=True)
    for t in (o, lse):
        assert torch.equal(t, t[:, :h].repeat(1, times, *[1] * (t.dim() - 2)))
    g = torch.Generator(device=DEV).manual_seed(1)
    oc = torch.randn((1, h * times, nqb, 64), generator=g, device=DEV).to(q.dtype)
    gate = torch.rand((1, h * times, q.shape[2], 2), generator=g, device=DEV).to(q.dtype)
    assert torch.equal(s3r.select_attn_merge(q, kk, v, idx, oc, gate, 16), s3r.gated_merge(oc, o, gate, 16))
    return o[:, :h], lse[:, :h]


def _matches(o, lse, want, lse_want):
    assert max_abs(o, want) <= 2e-2                       # the bound of the operator's other parity tests at these inputs
    fin = torch.isfinite(lse_want)
    assert torch.equal(torch.isfinite(lse.cpu()), fin) and max_abs(lse.cpu()[fin], lse_want[fin]) <= 2e-3


def _lists(n, h, k, n0, n1, seed, duplicates=False, last=False):
    """[1,h,nqb,k] lists: query blocks 0, 1 (2, 3) of four neighbours name n0 (n1) distinct blocks of the lower (upper) part."""
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


@lru_cache(maxsize=2)
def _case(dtype, n, k, n0, n1, extra):
    h = 2
    g = torch.Generator().manual_seed(n + k)
    q, kk, v = ((torch.randn((1, h, n, 64), generator=g) * s).to(dtype) for s in (0.5, 0.5, 1.0))
    idx = _lists(n, h, k, n0, n1, 3 * n + k, **dict(extra))
    return (q, kk, v, idx), oracle.select_attention(q, kk, v, idx, 16, out_dtype=torch.float32, return_lse=True)


@pytest.mark.parametrize("n,k,n0,n1,extra", [
    (2048, 32, 64, 64, ()),                             # full lists that share nothing: unions of 32, 64, 128
    (2048, 32, 63, 1, ()),                              # a list of one block beside full ones
    (2048, 32, 33, 27, ()),                             # the second list of a half is short, or empty
    (4096, 64, 128, 128, ()),                           # the longest unions there are: 64, 128, 256
    (96, 1, 2, 2, ()), (96, 1, 1, 1, ()),               # one entry
    (96, 2, 3, 3, ()),                                  # two
    (1033, 16, 20, 21, (("last", True),)),              # ragged last block listed, a group's tail of one query block
    (4105, 32, 64, 64, (("last", True),)),              # the same at the end of long unions
    (1040, 16, 17, 12, (("duplicates", True),)),        # blocks that count twice
    (4096, 64, 100, 90, (("duplicates", True),)),
    (1040, 16, 32, 0, ()),                              # a half that attends nothing
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("per_wave", PER_WAVE)
def test_block16_lists_that_share_little_match_oracle(per_wave, dtype, n, k, n0, n1, extra):
    inputs, want = _case(dtype, n, k, n0, n1, extra)
    _matches(*_attend(*inputs, _repeats(2, -(-n // 16), per_wave)), *want)


@pytest.mark.parametrize("per_wave", PER_WAVE)
def test_block16_unions_of_colliding_blocks(per_wave):
    """The union's table has 512 slots for (block * 0x9E3779B1 mod 2^32) / 2^23: blocks chosen so that four share a slot and the next
    slots are taken too, which takes chains of probes; 64 entries a list."""
    n, k, h = 16 * 2048, 64, 1
    nqb = n // 16
    by_slot = sorted(range(nqb), key=lambda e: (e * 0x9E3779B1 % 2 ** 32) >> 23)
    g = torch.Generator().manual_seed(8)
    idx = torch.empty((1, h, nqb, k), dtype=torch.int32)
    for grp in range(nqb // 4):
        at = (37 * grp) % (nqb - 256)
        blocks = torch.tensor(by_slot[at:at + 256], dtype=torch.int32)
        idx[0, 0, 4 * grp:4 * grp + 4] = blocks[torch.randperm(256, generator=g)].view(4, k)
    q, kk, v = ((torch.randn((1, h, n, 64), generator=g) * s).to(torch.bfloat16) for s in (0.5, 0.5, 1.0))
    o, lse = _attend(q, kk, v, idx, _repeats(h, nqb, per_wave))
    rows = slice(0, 16 * 256)                                             # (the first 64 groups on the host)
    part = torch.full_like(idx, -1)
    part[:, :, :256] = idx[:, :, :256]
    want, lse_want = oracle.select_attention(q, kk, v, part, 16, out_dtype=torch.float32, return_lse=True)
    _matches(o[:, :, rows], lse[:, :, rows], want[:, :, rows], lse_want[:, :, rows])


@pytest.mark.parametrize("gain", [12.0, 2.0])
@pytest.mark.parametrize("per_wave", PER_WAVE)
def test_block16_walk_handles_scores_far_above_the_reference(per_wave, gain):
    """Some blocks line up with the queries: row sums beyond the bound, second walk with the running maximum."""
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
    o, _ = _attend(q, kk, v, idx, _repeats(h, n // 16, per_wave))
    assert torch.isfinite(o.float()).all()
    assert max_abs(o, oracle.select_attention(q, kk, v, idx, 16, out_dtype=torch.float32)) <= 2e-2


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,k,extra", [(2048, 32, {}), (3205, 32, {"last": True}), (2048, 16, {"duplicates": True}), (2048, 64, {})])
def test_block16_result_does_not_depend_on_the_query_blocks_of_a_wave(dtype, n, k, extra):
    """A query block gets the same bits whichever others its wave walks with: the order of its blocks follows their slots in the
    table, of which so few blocks have one each, and so does the one that gives its softmax reference."""
    h, nqb = 2, -(-n // 16)
    slots = {(e * 0x9E3779B1 % 2 ** 32) >> 23 for e in range(nqb)}
    assert len(slots) == nqb
    idx = _lists(n, h, k, 3 * k // 2, 2 * k, n + k, **extra)
    g = torch.Generator().manual_seed(n + k)
    q, kk, v = ((torch.randn((1, h, n, 64), generator=g) * s).to(dtype) for s in (0.5, 0.5, 1.0))
    one, two, four = (_attend(q, kk, v, idx, _repeats(h, nqb, p)) for p in PER_WAVE)
    for other in (two, four):
        assert torch.equal(one[0], other[0]) and torch.equal(one[1], other[1])
