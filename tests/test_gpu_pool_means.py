"""GPU: the means of q, k and v in one launch against one call each, bit for bit: every kernel of the pooling (blocks of one, two, four and
more loads a wave), ragged ends, strides of their own, three types."""
import pytest
import torch

import speed3r_amd as s3r
from speed3r_amd.sparse_attn import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,h,n,d,block", [(1, 1, 1, 64, 64), (2, 3, 130, 64, 16), (1, 2, 1041, 64, 64), (1, 2, 333, 64, 8), (1, 2, 200, 32, 32), (2, 2, 65, 128, 64)])
def test_means_of_three(dtype, b, h, n, d, block):
    gen = torch.Generator(device=DEV).manual_seed(n)
    packed = torch.randn((b, n, 3, h, d), generator=gen, device=DEV).to(dtype)
    q, k, v = packed.permute(2, 0, 3, 1, 4).unbind(0)
    for t in ((q, k, v), (q.contiguous(), k, v.flip(2)), (q[..., ::1], k.transpose(0, 1).contiguous().transpose(0, 1), v.contiguous())):
        for got, x in zip(ops._pool_means(*t, block), t):
            assert got.is_contiguous() and torch.equal(got, s3r.pool_mean(x, block))
