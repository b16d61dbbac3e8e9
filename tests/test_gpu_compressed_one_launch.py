"""GPU: attention output and log-sum-exp of the pooled tokens from the launch that also selects their blocks (up to 1216 keys), against
float64 at the edges of its steps of 64 keys and groups of 16 and 128 rows; views of a packed tensor, scores far apart, infinite values."""
import pytest
import torch

from speed3r_amd.sparse_attn import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
HALF = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}   # half a step of the type, relative to the value


def _reference(q, k, v):
    q, k, v = (t.double() for t in (q, k, v))
    s = (q @ k.transpose(-1, -2).contiguous()) / 8
    p = torch.softmax(s, -1)
    return p @ v, p @ v.abs(), torch.logsumexp(s, -1), (q.abs() @ k.abs().transpose(-1, -2).contiguous()).amax(-1) / 8


def _check(q, k, v, topk=32):
    o, idx, lse = ops.compressed_attn_topk(q, k, v, topk, return_lse=True)
    assert torch.equal(idx, ops.compressed_attn_topk(q, k, None, topk)[1])
    assert torch.equal(o, ops.compressed_attn_topk(q, k, v, topk)[0])
    want, room, want_lse, size = _reference(q, k, v)
    # a probability is rounded once to the type, the result once; a score's 64 products are summed in fp32, and an error of the score
    # is a relative one of the probability; exponentials and their sum in fp32
    score = (64 * 2.0 ** -24 * size).unsqueeze(-1)
    tol = HALF[q.dtype] * (room + want.abs()) * 1.01 + room * (2 * score + 2.0 ** -16) + 2.0 ** -24
    assert ((o.double() - want).abs() <= tol).all()
    assert ((lse.double() - want_lse).abs() <= score[..., 0] + 2.0 ** -20 * (want_lse.abs() + 8)).all()


@pytest.mark.parametrize("b,h,lq,lk", [(1, 1, 1, 1), (1, 2, 7, 5), (2, 3, 17, 63), (1, 2, 16, 64), (1, 2, 127, 65), (2, 2, 128, 126), (1, 3, 129, 129),
                                       (1, 2, 300, 256), (2, 1, 513, 511), (1, 2, 90, 1025), (1, 3, 1216, 1216)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_against_float64(b, h, lq, lk, dtype):
    gen = torch.Generator(device=DEV).manual_seed(lq + lk)
    packed = torch.randn(b, max(lq, lk), 3, h, 64, generator=gen, device=DEV).to(dtype)
    q, k, v = packed.permute(2, 0, 3, 1, 4).unbind(0)
    q, k, v = q[:, :, :lq], k[:, :, :lk], v[:, :, :lk]
    _check(q, k, v)
    _check(q.contiguous(), k.contiguous(), v.contiguous())
    _check((4 * q).contiguous(), (4 * k).contiguous(), v)      # scores up to some hundred apart
    _check(-k[:, :, :1].expand(b, h, lq, 64).contiguous(), k, v)


@pytest.mark.parametrize("lk", [5, 70, 128])
def test_values_that_are_not_finite(lk):
    q, k, v = torch.randn(3, 1, 1, lk, 64, generator=torch.Generator(device=DEV).manual_seed(lk), device=DEV).bfloat16().unbind(0)
    v[..., -1, 3] = float("inf")         # (the last row fills up a step)
    v[..., 0, 4] = float("-inf")
    q[..., 2, :] = float("nan")
    o = ops.compressed_attn_topk(q, k, v, 32)[0]
    keep = torch.arange(lk, device=DEV) != 2
    assert (o[..., keep, 3] == float("inf")).all() and (o[..., keep, 4] == float("-inf")).all()
    assert torch.isfinite(o[:, :, keep][..., 5:]).all() and torch.isnan(o[..., 2, :]).all()
