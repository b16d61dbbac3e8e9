"""GPU: the index kernel whose first sweep samples the keys, against the row-wise selection on the stored scores, bit for bit: the
first size that samples, remainders of the sampled tiles, keys alike in runs and at one place of every period, far rows."""
import pytest
import torch

from speed3r_amd.sparse_attn import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(q, k, topk):
    got = ops.compressed_attn_topk(q, k, None, topk)[1]
    scores = ops.compressed_attn_topk(q, k, k, topk, return_scores=True, materialize_scores=True)[2]
    assert torch.equal(got, ops.topk_rows(scores, topk)), topk


# 64 tiles (4 033 to 4 096 keys) sample every second key, 240 tiles and more every tenth; one tile of 64 samples more or less
# (2 x 130 rows: workgroups of four waves; 16 x 4 164: of two)
@pytest.mark.parametrize("heads,rows,keys", [(2, 130, n) for n in (4032, 4033, 4096, 4097, 4608, 4610, 9215, 15361, 16001)]
                         + [(16, 4164, n) for n in (4032, 4033, 4610)])
def test_sizes_around_the_sampled_tiles(heads, rows, keys):
    gen = torch.Generator(device=DEV).manual_seed(keys)
    q, k = (torch.randn(1, heads, n, 64, generator=gen, device=DEV).bfloat16() for n in (rows, keys))
    for topk in (1, 4, 8, 16, 32):
        _check(q, k, topk)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("run,period", [(65, 4225), (1, 10), (1, 640), (640, 6400), (5000, 5000)])
def test_keys_alike_in_runs_and_periods(dtype, run, period):
    gen = torch.Generator(device=DEV).manual_seed(run + period)
    base = torch.randn(1, 2, period // run, 64, generator=gen, device=DEV).repeat_interleave(run, 2)
    base = base.repeat(1, 1, -(-6500 // base.shape[2]), 1)[:, :, :6500]
    for noise in (0.0, 0.05):
        k = (base + noise * torch.randn(base.shape, generator=gen, device=DEV)).to(dtype)
        for topk in (2, 16, 32):
            _check(k[:, :, ::47].contiguous(), k, topk)


def test_rows_too_far_apart_for_a_sampled_tile():
    """Row stride 3 MB: 64 rows ten apart would span 2^31 bytes and more; the sample gets denser."""
    far = torch.empty(4200 * 1_572_864, dtype=torch.bfloat16, device=DEV).view(1, 1, 4200, 1_572_864)
    k = far[..., :64]
    k.copy_(torch.randn(k.shape, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV))
    q = k[:, :, :70].contiguous()
    want = ops.compressed_attn_topk(q, k.contiguous(), None, 16)[1]
    assert torch.equal(ops.compressed_attn_topk(q, k, None, 16)[1], want)


@pytest.mark.parametrize("keys", [4032, 4100])   # without and with a sample
def test_one_key_seen_many_times(keys):
    """An expanded k (token stride 0): every score of a row is the same, the first blocks are the choice."""
    gen = torch.Generator(device=DEV).manual_seed(3)
    q, k = (torch.randn((1, 2, n, 64), generator=gen, device=DEV).bfloat16() for n in (130, 1))
    for topk in (1, 16):
        idx = ops.compressed_attn_topk(q, k.expand(1, 2, keys, 64), None, topk)[1]
        assert torch.equal(idx, torch.arange(topk, dtype=torch.int32, device=DEV).expand_as(idx))
        _check(q, k.expand(1, 2, keys, 64), topk)
