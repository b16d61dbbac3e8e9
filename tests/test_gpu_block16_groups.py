"""GPU: selection attention with 16-token blocks where a wave takes one, two and four query blocks (the number of (query block, head)
pairs decides), against the oracle: ends of groups, ragged last blocks, blocks named twice, lists of one and of 64 entries."""
import pytest
import torch

import oracle
import speed3r_amd as s3r
from helpers import max_abs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# (heads, tokens, entries): 17 and 18 query blocks of 16 tokens; up to 5 000 pairs, up to 20 000, more
SIZES = [(3, 264, 5), (294, 265, 64), (295, 272, 1), (1111, 281, 32), (1112, 281, 32), (1180, 257, 7)]


def _inputs(h, n, k, dtype, seed, scale=0.5):
    g = torch.Generator().manual_seed(seed)
    q, kk, v = ((torch.randn((1, h, n, 64), generator=g) * s).to(dtype) for s in (scale, scale, 1.0))
    nb = -(-n // 16)
    idx = torch.randint(-1, nb + 1, (1, h, nb, k), generator=g, dtype=torch.int32)   # -1 and nb are skipped, blocks repeat
    idx[:, :, 2] = -1                                                               # a query block that attends nothing
    return q, kk, v, idx


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("h,n,k", SIZES)
def test_groups_match_the_oracle(dtype, h, n, k):
    q, kk, v, idx = _inputs(h, n, k, dtype, n + k)
    o, lse = s3r.select_attn(q.to(DEV), kk.to(DEV), v.to(DEV), idx.to(DEV), 16, return_lse=True)
    want, lse_want = oracle.select_attention(q, kk, v, idx, 16, out_dtype=torch.float32, return_lse=True)
    assert max_abs(o, want) <= 2e-2                       # the bound of the operator's other parity tests at these inputs
    fin = torch.isfinite(lse_want)
    assert torch.equal(torch.isfinite(lse.cpu()), fin) and max_abs(lse.cpu()[fin], lse_want[fin]) <= 2e-3


@pytest.mark.parametrize("h,n,k", SIZES)
def test_merge_has_the_bits_of_the_two_operators(h, n, k):
    q, kk, v, idx = (t.to(DEV) for t in _inputs(h, n, k, torch.bfloat16, n))
    g = torch.Generator(device=DEV).manual_seed(1)
    oc = torch.randn((1, h, idx.shape[2], 64), generator=g, device=DEV).bfloat16()
    gate = torch.rand((1, h, n, 2), generator=g, device=DEV).bfloat16()
    want = s3r.gated_merge(oc, s3r.select_attn(q, kk, v, idx, 16), gate, 16)
    assert torch.equal(s3r.select_attn_merge(q, kk, v, idx, oc, gate, 16), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("h", [2, 320, 1300])
def test_scores_far_above_the_first_block(dtype, h):
    """Blocks that line up with the queries come somewhere in the walk: sums beyond the bound start over with the running maximum."""
    n = 256
    g = torch.Generator().manual_seed(h)
    q, kk, v = (torch.randn((1, h, n, 64), generator=g).to(dtype) for _ in range(3))
    kk = (kk * 0.01).to(dtype)
    kk[:, :, 96:112] = (q[:, :, :16] * 12).to(dtype)
    idx = torch.stack([torch.randperm(16, generator=g)[:6] for _ in range(h * 16)]).view(1, h, 16, 6).to(torch.int32)
    idx[:, :, :, 3] = 6
    o = s3r.select_attn(q.to(DEV), kk.to(DEV), v.to(DEV), idx.to(DEV), 16)
    assert torch.isfinite(o.float()).all()
    # outputs of up to 5.5 (largest of 5 million normal values): half a step of bf16 there, 2^-6, and the probabilities' rounding,
    # 2^-9 relative, here and in the oracle, whose references differ: 0.0156 + 2 x 0.0107
    assert max_abs(o, oracle.select_attention(q, kk, v, idx, 16, out_dtype=torch.float32)) <= 3.7e-2
