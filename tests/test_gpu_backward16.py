"""GPU: gradients of the selection attention with 16-token blocks at the sizes where its kernels can go wrong, against the closed
form in fp64 from the same inputs: odd and even numbers of steps, lists longer than a wave's 64 entries, groups of one query block,
ragged ends, blocks named twice, strided and far rows."""
import pytest
import torch

import oracle
from speed3r_amd.sparse_attn import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _reference(q, k, v, dout, idx):
    n, lk, dt = q.shape[2], k.shape[2], q.dtype
    q, k, v, dout = (t.cpu().double() for t in (q, k, v, dout))
    nkb = -(-lk // 16)
    mult = torch.zeros((*idx.shape[:3], nkb), dtype=torch.float64)
    ok = (idx >= 0) & (idx < nkb)
    mult.scatter_add_(3, idx.clamp(0, nkb - 1).long(), ok.double())
    w = mult.repeat_interleave(16, 2)[:, :, :n].repeat_interleave(16, 3)[..., :lk]
    s = (q @ k.transpose(-1, -2)) / 8
    p = w * torch.exp(s - s.masked_fill(w == 0, -float("inf")).amax(-1, keepdim=True).nan_to_num(neginf=0.0))
    p = p / p.sum(-1, keepdim=True).clamp_min(1e-300)
    dp = dout @ v.transpose(-1, -2)
    ds = p * (dp - (p * dp).sum(-1, keepdim=True)) / 8
    return ds @ k, ds.transpose(-1, -2) @ q, p.transpose(-1, -2) @ dout


def _check(q, k, v, idx, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    dout = torch.randn(q.shape, generator=g, device=DEV).to(q.dtype)
    o, lse = ops.select_attn(q, k, v, idx.to(DEV), 16, return_lse=True)
    got = ops.attn_bwd(q, k, v, o, dout, lse, idx.to(DEV), 16)
    # P and dS are rounded to the type before the products and the output before delta: relative errors of a few of its steps,
    # against the largest gradient, since a row of dS sums to zero; where a query attends to one key alone dS is the difference of
    # two equal sums of 64 products of size 1 in fp32, 64 x 2^-24 at most
    tol = (8e-3 if q.dtype == torch.bfloat16 else 1e-3) * 4
    for a, b in zip(got, _reference(q, k, v, dout, idx)):
        assert torch.isfinite(a).all() and (a.cpu().double() - b).abs().max() <= tol * b.abs().max() + 4e-6


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,kk", [(16, 1), (17, 1), (31, 2), (48, 3), (65, 5), (1024, 31), (1040, 32), (1041, 33), (1200, 64), (2500, 7)])
def test_sizes(dtype, n, kk):
    g = torch.Generator().manual_seed(n)
    nb = -(-n // 16)
    q, k, v = ((torch.randn((1, 2, n, 64), generator=g) * s).to(dtype).to(DEV) for s in (0.5, 0.5, 1.0))
    idx = torch.randint(-1, nb + 1, (1, 2, nb, kk), generator=g, dtype=torch.int32)   # -1 and nb are skipped, blocks repeat
    idx[:, 1, :, 0] = nb - 1                                                          # one list of every length: all query blocks
    idx[:, 0, 0] = -1                                                                 # and a query block that attends nothing
    _check(q, k, v, idx, n)


def test_strided_rows():
    g = torch.Generator().manual_seed(7)
    packed = torch.randn((2, 3, 333, 3, 64), generator=g).to(torch.bfloat16).to(DEV)   # rows 3 x 128 bytes apart
    idx = torch.randint(0, 21, (2, 3, 21, 9), generator=g, dtype=torch.int32)
    _check(0.5 * packed[:, :, :, 0], packed[:, :, :, 1], packed[:, :, :, 2], idx, 3)


def test_rows_beyond_4_gib_from_the_tensor_start():
    n, row = 4113, 1 << 19                                                             # a row per MB: 4.3 GB
    g = torch.Generator(device=DEV).manual_seed(1)
    far = torch.empty(n * row, dtype=torch.bfloat16, device=DEV).view(1, 1, n, row)[..., :64]
    far.copy_(torch.randn(far.shape, generator=g, device=DEV))
    q, k = (torch.randn(far.shape, generator=g, device=DEV).to(torch.bfloat16) * 0.5 for _ in range(2))
    nb = -(-n // 16)
    idx = torch.randint(0, nb, (1, 1, nb, 8), generator=torch.Generator().manual_seed(2), dtype=torch.int32)
    _check(q, k, far, idx, 5)
