"""The fp32 matrix-core attention kernel at the edges of its tiles, against the oracle (needs an MI355X)."""
import math

import pytest
import torch

import oracle
import speed3r_amd as s3r
from helpers import max_abs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n,block,kk", [(1, 16, 1), (15, 16, 3), (16, 16, 1), (17, 16, 64), (333, 16, 32), (31, 32, 2), (33, 32, 5),
                                        (97, 32, 64), (63, 64, 1), (64, 64, 2), (65, 64, 3), (96, 64, 4), (1041, 64, 16), (2081, 64, 64)])
def test_fp32_selection_at_tile_edges(n, block, kk):
    """Ragged ends on both sides of a 32-key stage and of a 16-row wave, skipped and repeated entries, a query block
    without a valid entry.  Bound: sums of at most 64 * block products of unit-variance terms in fp32 (1e-5)."""
    g = torch.Generator().manual_seed(n * 64 + kk)
    b, h = 2, 3
    q, k, v = (torch.randn((b, h, n, 64), generator=g) for _ in range(3))
    nb = -(-n // block)
    idx = torch.randint(-1, nb + 1, (b, h, nb, kk), generator=g, dtype=torch.int32)   # -1 and nb: skipped
    idx[:, 0, nb // 2] = -1
    o_ref, lse_ref = oracle.select_attention(q, k, v, idx, block, out_dtype=torch.float32, return_lse=True)
    o, lse = s3r.select_attn(q.to(DEV), k.to(DEV), v.to(DEV), idx.to(DEV), block, return_lse=True)
    assert max_abs(o, o_ref) <= 1e-5
    fin = torch.isfinite(lse_ref)
    assert torch.equal(torch.isfinite(lse.cpu()), fin) and max_abs(lse.cpu()[fin], lse_ref[fin]) <= 1e-5


@pytest.mark.parametrize("lq,lk", [(1, 1), (17, 15), (64, 33), (131, 131), (2100, 70)])
def test_fp32_compressed_scores_and_attention(lq, lk):
    """Single-wave and four-wave workgroups (2100 rows x 8 heads), ragged keys, strided inputs; scores to the rounding
    of 64 products (64 * 2^-24 of |q||k|), indices from exactly those scores."""
    g = torch.Generator().manual_seed(lq + lk)
    q = torch.randn((1, 8, lq, 64), generator=g)
    k, v = torch.randn((1, lk, 2, 8, 64), generator=g).permute(2, 0, 3, 1, 4).unbind(0)
    topk = 4
    o_ref, _, s_ref = oracle.compressed_attention(q, k, v, out_dtype=torch.float32)
    kd, vd = torch.stack((k, v), 0).permute(1, 3, 0, 2, 4).contiguous().to(DEV).permute(2, 0, 3, 1, 4).unbind(0)
    o, idx, s = s3r.compressed_attn_topk(q.to(DEV), kd, vd, topk, return_scores=True)
    room = q.norm(dim=-1)[..., None] * k.norm(dim=-1)[:, :, None, :]
    assert ((s.cpu() - s_ref).abs() <= 64 * 2.0 ** -24 * room).all()
    assert max_abs(o, o_ref) <= 1e-5
    assert torch.equal(idx, s3r.topk_rows(s, topk))
    o3 = s3r.compressed_attn_topk(q.to(DEV), kd, vd, topk, softmax_scale=3.0 / math.sqrt(64))[0]
    assert max_abs(o3, oracle.compressed_attention(q, k, v, softmax_scale=3.0 / math.sqrt(64), out_dtype=torch.float32)[0]) <= 3e-5


@pytest.mark.parametrize("lq,lk", [(64, 33), (131, 131), (1, 300)])
def test_fp32_scores_have_the_generic_kernels_bits(lq, lk):
    """The same tensors at addresses that are no multiples of 16 bytes go through the generic kernel."""
    g = torch.Generator().manual_seed(lq)
    q, k, v = (torch.randn((1, 3, n, 64), generator=g).to(DEV) for n in (lq, lk, lk))

    def off(t):
        return torch.empty(t.numel() + 1, device=DEV)[1:].view(t.shape).copy_(t)

    s = s3r.compressed_attn_topk(q, k, v, 1, return_scores=True)[2]
    assert torch.equal(s, s3r.compressed_attn_topk(off(q), off(k), off(v), 1, return_scores=True)[2])
