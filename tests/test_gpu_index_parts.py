"""GPU: indices where two waves share a row's keys (at most 512 workgroups of 64 rows), against the row-wise selection on the stored
scores, bit for bit: one tile (the second part has none), odd and even numbers of tiles, ragged ends, sampled first sweeps, the last
grid of these kernels and the first beyond it, equal scores, NaN.  And where no first sweep looks for a bound (one or two tiles), with
two waves to a row's keys, workgroups of two waves and of four."""
import pytest
import torch

from speed3r_amd import _lib
from speed3r_amd.sparse_attn import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("b,h,lq,lk,ks", [(1, 1, 1, 1, (1, 8)), (1, 2, 65, 40, (1, 4, 16)), (2, 2, 64, 64, (1, 2, 4, 8)), (1, 3, 130, 641, (1, 4)),
                                          (1, 2, 63, 1217, (1, 8, 32)), (1, 2, 1300, 1281, (2, 16, 32)), (2, 1, 100, 4096, (4, 32)),
                                          (1, 1, 200, 5003, (1, 16, 32)), (1, 16, 2016, 2016, (4, 32)), (1, 16, 2048, 1300, (8, 32)),
                                          (1, 16, 2049, 1300, (8, 32)), (1, 1, 40, 17000, (16,)),
                                          *((1, h, rows, keys, (1, 4, 8, 16, 32)) for h, rows in ((32, 1000), (16, 4164), (16, 6000))
                                            for keys in (30, 63, 64, 65, 128, 129))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_indices_match_the_selection_on_stored_scores(b, h, lq, lk, ks, dtype):
    gen = torch.Generator(device=DEV).manual_seed(lq + lk)
    q = torch.randn(b, h, lq, 64, generator=gen, device=DEV).to(dtype)
    k = torch.randn(b, h, lk, 64, generator=gen, device=DEV).to(dtype)
    alike = (0.8 * k[:, :, :1] + 0.05 * k).to(dtype)
    gone = k.clone()
    gone[:, :, ::7] = float("nan")
    for topk in ks:
        assert not _lib.lib().s3r_topk_in_lds(b * h, lq, lk, topk)
        # (with fewer numbers than slots the row-wise kernel names the NaNs, this one the last key)
        for qq, kk in ((q, k), (q.sign(), k.sign()), (q * 0, k), (q, alike), *([(q, gone)] if lk - -(-lk // 7) >= topk else [])):
            got = ops.compressed_attn_topk(qq, kk, None, topk)[1]
            scores = ops.compressed_attn_topk(qq, kk, k, topk, return_scores=True, materialize_scores=True)[2]
            assert torch.equal(got, ops.topk_rows(scores, topk)), topk
