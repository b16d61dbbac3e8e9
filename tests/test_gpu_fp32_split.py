"""The fp32 selection kernel where the last query blocks are computed in halves (up to 384 blocks in all), and its softmax reference, against
the oracle."""
import pytest
import torch

import oracle
import speed3r_amd as s3r
from helpers import max_abs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(q, k, v, idx, tol):
    o_ref, lse_ref = oracle.select_attention(q, k, v, idx, 64, out_dtype=torch.float32, return_lse=True)
    o, lse = s3r.select_attn(q.to(DEV), k.to(DEV), v.to(DEV), idx.to(DEV), 64, return_lse=True)
    assert max_abs(o, o_ref) <= tol
    fin = torch.isfinite(lse_ref)
    assert torch.equal(torch.isfinite(lse.cpu()), fin) and max_abs(lse.cpu()[fin], lse_ref[fin]) <= tol


# query blocks: 1, 128 (all in halves), 129 (none), 255, 256, 257, 384 (the last 128); 385 and 513, which go to the kernel of split values; last
# key blocks of 5, 17 and 64 keys
@pytest.mark.parametrize("h,n,kk", [(1, 40, 1), (64, 69, 2), (43, 145, 3), (85, 133, 2), (64, 256, 4), (257, 17, 1), (128, 133, 3), (77, 261, 2),
                                    (57, 517, 6)])
def test_blocks_in_halves_match_the_oracle(h, n, kk):
    """Bound: that of the operator's other fp32 tests, sums of a few hundred products of unit-variance terms."""
    g = torch.Generator().manual_seed(h * 1000 + n)
    q, k, v = (torch.randn((1, h, n, 64), generator=g) for _ in range(3))
    nb = -(-n // 64)
    idx = torch.randint(-1, nb + 1, (1, h, nb, kk), generator=g, dtype=torch.int32)   # -1 and nb are skipped, blocks repeat
    if h * nb > 1:
        idx[:, -1, -1] = -1                                                         # a block in halves (if any is) that attends nothing
    idx[:, 0, 0, 0] = 0
    _check(q, k, v, idx, 1e-5)


@pytest.mark.parametrize("step", [0.5, 3.0, 30.0])
def test_scores_that_rise_along_the_list(step):
    """Every listed block's scores lie ``step`` natural units above the ones before it: below and above what the reference lets
    pass.  Up to 6 * 30 units: a score's rounding, 2^-23 of it twice over (products and scale), moves the result by as much."""
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn((1, 40, 400, 64), generator=g) for _ in range(3))
    q[..., 0] = 8.0
    k[..., 0] = (torch.arange(400) // 64) * step
    idx = torch.arange(7, dtype=torch.int32).expand(1, 40, 7, 7).contiguous()
    _check(q, k, v, idx, 1e-5 + 4 * 6 * step * 2.0 ** -23)


@pytest.mark.parametrize("n,h", [(400, 40), (450, 32), (384, 47)])   # 280 query blocks (24 in halves), 256 (none), 282 (26, all of them full)
@pytest.mark.parametrize("dims", [slice(60, 61), slice(63, 64), slice(60, 64)])
def test_scores_that_rise_in_the_last_dimensions(dims, n, h):
    """The same, hundreds of units a block in the head dimensions that the last products of a score add: the reference of the softmax
    is read from finished sums.  A score is at most 6 * 400 units: its rounding, 2^-23 of it twice over, moves the result by as much."""
    g = torch.Generator().manual_seed(2)
    q, k, v = (torch.randn((1, h, n, 64), generator=g) for _ in range(3))
    width = dims.stop - dims.start
    q[..., dims] = 8.0
    k[..., dims] = (torch.arange(n) // 64)[:, None] * (400.0 / width)
    nb = -(-n // 64)
    order = torch.stack([torch.randperm(nb, generator=g) for _ in range(h * nb)]).view(1, h, nb, nb)   # (rising, falling and mixed)
    _check(q, k, v, order.int().contiguous(), 1e-5 + 4 * 2400 * 2.0 ** -23)
