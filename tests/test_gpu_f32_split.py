"""fp32 selection attention in blocks of 64 on the 16-bit matrix instructions (needs an MI355X), more than 384 blocks: ragged last blocks, lists that repeat, skip or
lack entries, strided and odd-aligned queries, values that three bf16 parts do not hold."""
import pytest
import torch

import speed3r_amd as s3r

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _reference(q, k, v, idx, scale):
    """Output, log-sum-exp and an error bound of the output, in 64 bits on the CPU."""
    q, k, v, idx = (t.cpu().double() if t.is_floating_point() else t.cpu() for t in (q, k, v, idx))
    out, lse, bound = torch.zeros_like(q), torch.full(q.shape[:3], -float("inf"), dtype=torch.float64), torch.zeros_like(q)
    n = q.shape[2]
    for h in range(q.shape[1]):
        for i in range(idx.shape[2]):
            cols = [torch.arange(j * 64, min(n, j * 64 + 64)) for j in idx[0, h, i].tolist() if 0 <= j * 64 < n]
            if not cols:
                continue
            cols, rows = torch.cat(cols), slice(i * 64, min(n, i * 64 + 64))
            s = scale * q[0, h, rows] @ k[0, h, cols].T
            p = torch.softmax(s, -1)
            out[0, h, rows] = p @ v[0, h, cols]
            lse[0, h, rows] = torch.logsumexp(s, -1)
            # 64 + 16 roundings of 2^-24 in a score, as many in the exponent's product, then 40 in sums and quotient
            ds = 2.0 ** -24 * (80 * scale * q[0, h, rows].abs() @ k[0, h, cols].abs().T + 2 * s.abs()).amax(-1, keepdim=True)
            bound[0, h, rows] = (2 * ds + 40 * 2.0 ** -24) * (p @ v[0, h, cols].abs())
    return out, lse, bound


def _inputs(heads, n, seed, size=1.0):
    gen = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn((1, heads, n, 64), generator=gen).mul_(size).to(DEV) for _ in range(3))
    nb = -(-n // 64)
    idx = torch.randint(-1, nb + 1, (1, heads, nb, 5), generator=gen).int().to(DEV)   # (some skipped, some twice)
    return q, k, v, idx


@pytest.mark.parametrize("heads,n,scale", [(512, 1, 0.125), (512, 31, 0.125), (385, 33, 0.125), (512, 64, 1.0), (256, 65, 0.125), (171, 161, 0.3), (64, 512, 0.125)])
def test_against_64_bits(heads, n, scale):
    q, k, v, idx = _inputs(heads, n, n)
    idx[0, 0, 0] = -1                                                                 # nothing listed
    want, lse_want, bound = _reference(q, k, v, idx, scale)
    odd = torch.empty(heads * n * 65 + 1, device=DEV)[1:].view(1, n, heads, 65)[..., :64].copy_(q.permute(0, 2, 1, 3)).permute(0, 2, 1, 3)
    for query in (q, odd):
        o, lse = s3r.select_attn(query, k, v, idx, 64, scale, return_lse=True)
        assert ((o.double().cpu() - want).abs() <= bound + 1e-30).all()
        # as a whole: a score's sum rounds some 16 times by 2^-24 of its own size, 8 x scale, in either direction (two parts would give 3e-6 and more)
        assert bool((o.double().cpu() - want).norm() <= 2.0 ** -24 * (4 + 16 ** 0.5 * 8 * scale) * want.norm())
        far = torch.isinf(lse_want)
        assert torch.equal(torch.isinf(lse).cpu(), far) and ((lse.double().cpu() - lse_want).abs()[~far] <= 2e-5).all()


@pytest.mark.parametrize("what,value", [("k", 3.39e38), ("k", 1e-30), ("v", 1e-30), ("q", 1e-30), ("k", -float("inf")), ("v", float("inf")), ("q", float("nan")), ("v", float("nan"))])
def test_values_beyond_three_parts(what, value):
    t = dict(zip("qkvi", _inputs(256, 100, 3)))
    t["i"][0, :, 0] = torch.tensor([0, 1, 0, 1, 1], device=DEV)
    t["i"][0, 0, 1] = 0                                                               # (block 1's rows of head 0 do not see row 70)
    if abs(value) < 1:
        t[what].mul_(value)
    else:
        t[what][0, 0, 70, 5] = value
    if value == 3.39e38:
        t["q"][..., 5] = 2e-38                                                        # (finite scores)
    want, _, bound = _reference(t["q"], t["k"], t["v"], t["i"], 0.125)
    o = s3r.select_attn(t["q"], t["k"], t["v"], t["i"], 64).double().cpu()
    clean = torch.isfinite(want)
    assert torch.equal(torch.isfinite(o), clean) and torch.equal(torch.isinf(o), torch.isinf(want))
    bound = torch.nan_to_num(bound, nan=0.0, posinf=0.0)
    sure = clean & (bound > 0)
    assert ((o - want).abs()[sure] <= bound[sure] + 1e-44).all()


# A chain of fp32 products gives such a score -inf or a number that far down, and its key no weight; the products of parts have either sign.  Bound: 2^-24 for
# each of 64 roundings in the scores, which are at most 10, and of 40 in sums and quotient.  A key with any weight more would be 1e-2 of the result.
@pytest.mark.parametrize("size", [1e18, 1e19, 1e21, 1e25, 1e30])
@pytest.mark.parametrize("channels", [slice(5, 6), slice(8, 16), slice(0, 64)])
def test_scores_beyond_the_range(size, channels):
    q, k, v, idx = _inputs(256, 100, 5)
    idx[..., 0], idx[..., 1] = 0, 1
    q[..., channels], k[..., channels] = size, 0.0
    k[:, :, 70, channels] = -size                                                     # (one key far below the others, which are ordinary)
    want, lse_want, _ = _reference(q, k, v, idx, 0.125)
    o, lse = s3r.select_attn(q, k, v, idx, 64, 0.125, return_lse=True)
    assert bool((o.double().cpu() - want).norm() <= 4e-5 * want.norm()) and bool((lse.double().cpu() - lse_want).abs().max() <= 4e-5)


# Equal scores, so that only the values' parts and sums count: 80 sums of four products (the fp32 instructions'; split values have fewer) and the quotient round
# by 2^-24 of the sum of magnitudes.  Three bf16 parts of values of 1e-35 keep 18 bits, of 1e-36 14.
@pytest.mark.parametrize("size", [1.0, 1e-31, 1e-33, 1e-34, 1e-35, 1e-36, 1e-37])
def test_small_columns_beside_ordinary_ones(size):
    q, k, v, idx = _inputs(256, 100, 7)
    idx[..., 0] = 0
    q.zero_()
    v[..., [5, 40]] *= size
    v[:, :, 3], v[..., 41] = 0.0, 0.0
    want, _, _ = _reference(q, k, v, idx, 0.125)
    mags, _, _ = _reference(q, k, v.abs(), idx, 0.125)
    o = s3r.select_attn(q, k, v, idx, 64, 0.125).double().cpu()
    assert bool(((o - want).abs() <= 84 * 2.0 ** -24 * mags).all())


@pytest.mark.parametrize("heads", [128, 512])
def test_scales_that_bring_small_scores_back(heads):
    """Queries whose lowest bits three parts do not hold, keys as large, and the scale that makes a score of both (bound: of the 64-bit test)."""
    q, k, v, idx = _inputs(heads, 64, 11)
    q, k, scale = q * 2.0 ** -122, k * 2.0 ** 57, 2.0 ** 65
    want, lse_want, bound = _reference(q, k, v, idx, scale)
    o, lse = s3r.select_attn(q, k, v, idx, 64, scale, return_lse=True)
    far = torch.isinf(lse_want)
    assert bool(((o.double().cpu() - want).abs() <= bound).all()) and bool(((lse.double().cpu() - lse_want).abs()[~far] <= 2e-5).all())


def _whole_bound(score):
    """Of output and log-sum-exp: 1e-5, and the rounding of a score by 2^-24 of it with each of 64 products (a large one may come first), with
    the scale and in the exponent, twice for output and reference."""
    return 1e-5 + 2 * 66 * score * 2.0 ** -24


@pytest.mark.parametrize("step", [0.5, 3.0, 30.0])
@pytest.mark.parametrize("n,h", [(400, 60), (250, 128)])
def test_scores_that_rise_along_the_list(step, n, h):
    """Every listed block's scores lie ``step`` natural units above the ones before it: below and above what the reference lets pass."""
    gen, nb = torch.Generator().manual_seed(1), -(-n // 64)
    q, k, v = (torch.randn((1, h, n, 64), generator=gen) for _ in range(3))
    q[..., 0] = 8.0
    k[..., 0] = (torch.arange(n) // 64) * step
    idx = torch.arange(nb, dtype=torch.int32).expand(1, h, nb, nb).contiguous()
    want, lse_want, _ = _reference(q, k, v, idx, 0.125)
    o, lse = s3r.select_attn(*(t.to(DEV) for t in (q, k, v, idx)), 64, 0.125, return_lse=True)
    for got, exact in ((o, want), (lse, lse_want)):
        assert bool(((got.double().cpu() - exact).abs() <= _whole_bound((nb - 1) * step)).all())


@pytest.mark.parametrize("dims", [slice(0, 1), slice(31, 32), slice(32, 33), slice(60, 61), slice(63, 64), slice(60, 64)])
def test_scores_that_rise_in_some_dimensions(dims):
    """The same, hundreds of units a block in dimensions that the first or the last products of a score add, along lists in any order: the
    reference of the softmax is read from finished sums."""
    gen, n, h = torch.Generator().manual_seed(2), 450, 57
    q, k, v = (torch.randn((1, h, n, 64), generator=gen) for _ in range(3))
    width = dims.stop - dims.start
    q[..., dims] = 8.0
    k[..., dims] = (torch.arange(n) // 64)[:, None] * (400.0 / width)
    nb = -(-n // 64)
    idx = torch.stack([torch.randperm(nb, generator=gen) for _ in range(h * nb)]).view(1, h, nb, nb).int().contiguous()
    want, lse_want, _ = _reference(q, k, v, idx, 0.125)
    o, lse = s3r.select_attn(*(t.to(DEV) for t in (q, k, v, idx)), 64, 0.125, return_lse=True)
    for got, exact in ((o, want), (lse, lse_want)):
        assert bool(((got.double().cpu() - exact).abs() <= _whole_bound((nb - 1) * 400)).all())


def test_last_parts_of_values_count():
    """Equal scores, and values of which neighbours leave 2^-18 of each other.  Some 32 roundings of 2^-24 of a value or two in either direction
    against a sum of 64 such remainders: 0.7 %; values in two parts, off by up to 2^-18 themselves, would be off by most of it."""
    q, k, v, idx = _inputs(256, 128, 9)
    idx[...] = torch.tensor([0, 1, -1, -1, -1], device=DEV)
    q.zero_()
    v[:, :, 1::2] = -v[:, :, ::2] * (1 + 2.0 ** -18)
    want, _, _ = _reference(q, k, v, idx, 0.125)
    o = s3r.select_attn(q, k, v, idx, 64, 0.125).double().cpu()
    assert bool((o - want).norm() <= 0.03 * want.norm())
