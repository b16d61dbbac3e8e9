"""The 64-token backward kernels at the edges of their pipelines (needs an MI355X): one key tile, the ragged last one alone, first, last and
listed twice, query blocks with fewer than 16 rows, lists of odd length, strided inputs, other scales."""
import pytest
import torch

import speed3r_amd as s3r
from speed3r_amd.sparse_attn import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(got, want, room, unit, floor, what):
    """One factor of a product was rounded (``unit`` of it), sums and exponentials are fp32, the result is rounded once;
    ``floor``: fp32 roundings of what cancels, half the type's smallest step for each factor below its normal range."""
    bound = 1.05 * unit * room + 1.05 * unit * want.abs() + 2e-5 * room + floor + 1e-7
    worst = ((got.double().cpu() - want).abs() / bound).max().item()
    assert worst <= 1.0, (what, worst)


CASES = [
    (1, [[0]], 0.125), (15, [[0, 0]], 0.125), (17, [[0]], 0.3), (64, [[0]], 0.125), (64, [[0, 0, 0]], 0.125), (65, [[1], [0]], 0.125),
    (79, [[1, 1], [1, 0]], 0.125), (112, [[0, 1], [1, 0]], 1.0), (128, [[1], [0]], 0.125), (129, [[2, 0, 1], [1, 2, 2], [0, 0, 1]], 0.125),
    (200, [[3, 2, 1, 0], [-1, 3, -1, 2], [0, 1, 2, 9], [3, -1, -1, -1]], 0.07), (320, None, 0.125), (333, None, 0.125), (1090, None, 0.125),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,lists,scale", CASES)
def test_gradients_of_one_tile_more_or_less(dtype, n, lists, scale):
    _gradients(dtype, n, lists, scale, False)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,lists,scale", CASES)
def test_delta_from_the_output_on_the_way(dtype, n, lists, scale):
    _gradients(dtype, n, lists, scale, True)


def _gradients(dtype, n, lists, scale, inside):
    gen = torch.Generator().manual_seed(n)
    heads, nb = 2, -(-n // 64)
    wide = [torch.randn((1, n, heads, 72), generator=gen).mul_(0.6).to(dtype)[..., :64].permute(0, 2, 1, 3) for _ in range(4)]
    q, k, v, g = (t.to(DEV) for t in wide)                 # (strided rows, heads inside)
    idx = None if lists is None else torch.tensor(lists, dtype=torch.int32)[None, None].repeat(1, heads, 1, 1).to(DEV)
    if idx is None:
        o, _, lse = s3r.compressed_attn_topk(q, k, v, None, return_lse=True, softmax_scale=scale)
        times = torch.ones((nb, nb), dtype=torch.float64)
    else:
        o, lse = s3r.select_attn(q, k, v, idx, 64, return_lse=True, softmax_scale=scale)
        times = torch.stack([(torch.tensor(lists) == j).sum(1) for j in range(nb)], dim=1).double()   # how often a list names a block
    if inside:                                             # (a wider row stride for the output too)
        wide_o = torch.full((1, n, heads, 72), float("nan"), dtype=dtype, device=DEV)
        o = wide_o[..., :64].copy_(o.permute(0, 2, 1, 3)).permute(0, 2, 1, 3)
    delta = ops.attn_bwd_delta(o, g)
    dq, dk, dv = ops.attn_bwd(q, k, v, o, g, lse, idx, softmax_scale=scale, delta=None if inside else delta)

    qf, kf, vf, gf = (t.double() for t in wide)
    times = times.repeat_interleave(64, 0)[:n].repeat_interleave(64, 1)[:, :n]
    p = torch.exp(scale * (qf @ kf.transpose(-1, -2)) - lse.double().cpu()[..., None]) * times
    ds = scale * p * (gf @ vf.transpose(-1, -2) - delta.double().cpu()[..., None])
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    tiny = 0.0 if dtype == torch.bfloat16 else 2.0 ** -25
    # fp32 sums: 64 additions and the difference to delta, 66 roundings of 2^-24 of the largest term's size at most
    vague = 4e-6 * scale * p * (gf.abs() @ vf.abs().transpose(-1, -2) + delta.double().cpu().abs()[..., None])
    _check(dq, ds @ kf, ds.abs() @ kf.abs(), unit, vague @ kf.abs() + tiny * (times @ kf.abs()), "dq")
    _check(dk, ds.transpose(-1, -2) @ qf, ds.abs().transpose(-1, -2) @ qf.abs(), unit, vague.transpose(-1, -2) @ qf.abs() + tiny * (times.T @ qf.abs()), "dk")
    _check(dv, p.transpose(-1, -2) @ gf, p.transpose(-1, -2) @ gf.abs(), unit, tiny * (times.T @ gf.abs()), "dv")
