"""GPU: indices of the kernel that keeps its scores in LDS (up to 1216 keys) against the row-wise selection on the stored scores, bit
for bit, at the edges of its tiles, pieces and row groups, and on both sides of the rule that chooses it."""
import pytest
import torch

from speed3r_amd.sparse_attn import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _same(q, k, topk):
    got = ops.compressed_attn_topk(q, k, None, topk)[1]
    scores = ops.compressed_attn_topk(q, k, k, topk, return_scores=True, materialize_scores=True)[2]
    return got, ops.topk_rows(scores, topk), scores


# (batch, heads, rows, keys): tiles of 32 keys over eight waves, pieces of 256, groups of 16 rows, the last sizes of the kernel and
# the first beyond it (1217 keys; 97 groups x 16 heads)
SIZES = [(1, 1, 1, 1), (1, 2, 7, 5), (2, 3, 33, 31), (1, 2, 16, 32), (1, 2, 17, 33), (1, 2, 50, 255), (1, 2, 50, 257), (2, 2, 100, 512),
         (1, 3, 300, 769), (1, 2, 90, 1025), (1, 2, 1216, 1216), (1, 2, 64, 1217), (1, 16, 1536, 40), (1, 16, 1537, 40), (2, 16, 756, 756)]


@pytest.mark.parametrize("b,h,lq,lk", SIZES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_indices_match_the_selection_on_stored_scores(b, h, lq, lk, dtype):
    gen = torch.Generator(device=DEV).manual_seed(lq + lk)
    q = torch.randn(b, h, lq, 64, generator=gen, device=DEV).to(dtype)
    k = torch.randn(b, h, lk, 64, generator=gen, device=DEV).to(dtype)
    for topk in (1, 2, 4, 8, 16, 32):
        # random scores; few distinct ones (many ties); all equal; runs of near-equal ones, as the blocks of a frame have
        near = k[:, :, :1] + 1e-2 * k
        for qq, kk in ((q, k), (q.sign(), k.sign()), (q * 0, k), (q, near)):
            got, want, _ = _same(qq, kk, topk)
            assert torch.equal(got, want), topk


@pytest.mark.parametrize("topk,keys", [(1, 96), (2, 97), (4, 64), (4, 65), (8, 64), (8, 65), (16, 40), (16, 41), (4, 641), (8, 1025)])
def test_both_sides_of_the_rule(topk, keys):
    q, k = (torch.randn(1, 2, keys, 64, generator=torch.Generator(device=DEV).manual_seed(s), device=DEV).bfloat16() for s in (topk, keys))
    got, want, _ = _same(q, k, topk)
    assert torch.equal(got, want)


# still scenes: the same blocks in every frame, with a little of their own or none (equal scores), so that a query's best keys lie at
# one place of every frame: in few of the groups whose maxima bound the selection
@pytest.mark.parametrize("per,frames", [(64, 16), (64, 19), (16, 76), (256, 4), (96, 12), (1, 1216), (2, 300), (5, 240)])
@pytest.mark.parametrize("noise", [0.0, 0.1])
def test_still_scenes(per, frames, noise):
    gen = torch.Generator(device=DEV).manual_seed(per)
    randn = lambda *s: torch.randn(*s, generator=gen, device=DEV)
    x = (randn(1, 2, 1, per, 64) + noise * randn(1, 2, frames, per, 64)).reshape(1, 2, -1, 64)
    for dtype in (torch.bfloat16, torch.float16):
        q, k = x.to(dtype), (x + 0.1 * noise * randn(*x.shape)).to(dtype)
        for topk in (1, 8, 16, 32):
            for sign in (1, -1):   # scores above and below zero
                got, want, _ = _same(q, sign * k, topk)
                assert torch.equal(got, want), topk


def test_infinite_scores_and_strided_rows():
    q, k = torch.randn(1, 2, 40, 128, device=DEV).bfloat16(), torch.randn(1, 2, 100, 192, device=DEV).bfloat16()
    q, k = q[..., 64:], k[..., 64:128]                      # rows 128 and 192 values apart
    got, want, _ = _same(q, k, 16)
    assert torch.equal(got, want)
    q = torch.ones_like(q)
    k = k.clone()
    k[0, 0, 3] = 3e38                                        # +inf from the row's sum, and its negative
    k[0, 0, 50:90] = -3e38
    got, want, scores = _same(q, k, 32)
    assert scores.isinf().any() and torch.equal(got, want)


def test_nan_scores_are_never_chosen():
    q, k = torch.randn(1, 1, 20, 64, device=DEV).bfloat16(), torch.randn(1, 1, 70, 64, device=DEV).bfloat16()
    k[0, 0, 5:60] = float("nan")
    got = ops.compressed_attn_topk(q, k, None, 32)[1][0, 0]
    scores = ops.compressed_attn_topk(q, k, k, 32, return_scores=True, materialize_scores=True)[2][0, 0]
    order = torch.where(scores.isnan(), torch.full_like(scores, float("-inf")), scores).argsort(dim=1, descending=True, stable=True)
    assert torch.equal(got[:, :15].long(), order[:, :15])   # the 15 keys with a number, then the filler
    assert (got[:, 15:] == 69).all()
