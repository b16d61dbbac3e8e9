"""GPU: the row-wise selection at the edges of its segments (256 and 1024 columns) and of what it ranks whole (32, 64), rows at 16 bytes and not, more candidates than lanes,
fewer columns than the list, against a stable sort: equal, since equal scores go lowest column first."""
import pytest
import torch

from speed3r_amd.sparse_attn import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("cols", [1, 3, 31, 32, 33, 40, 63, 64, 65, 131, 255, 256, 257, 1023, 1024, 1025, 4100])
@pytest.mark.parametrize("kk", [1, 16, 20, 64])
def test_rows_match_a_stable_sort(cols, kk):
    gen = torch.Generator(device=DEV).manual_seed(cols + kk)
    rows = torch.randn((37, cols), generator=gen, device=DEV)
    few = (2 * rows).round() + 0.5                       # many equal scores, none of them zero
    runs = torch.where(torch.arange(cols, device=DEV) % 256 < 5, rows + 50, rows)   # the best in few of the groups of columns
    low = torch.full_like(rows, -float("inf"))
    low[:, cols // 2] = 1.0
    for s in (rows, few, runs, torch.ones_like(rows), low):
        got = ops.topk_rows(s.contiguous(), kk)
        want = torch.sort(s, dim=1, descending=True, stable=True).indices[:, :kk].int()
        if cols < kk:
            want = torch.cat((want, want.new_full((37, kk - cols), cols - 1)), 1)
        assert torch.equal(got.view(want.shape), want)


@pytest.mark.parametrize("cols", [5, 32, 33, 64])
def test_every_order_of_special_values(cols):
    """The smallest and largest numbers, both zeros, infinities and NaNs rank by their bits (a NaN of either sign beyond the infinity of its sign)."""
    gen = torch.Generator(device=DEV).manual_seed(cols)
    special = torch.tensor([float("inf"), -float("inf"), 0.0, -0.0, 1e-45, -1e-45, 3e38, -3e38, float("nan"), 1.0], device=DEV)
    s = special[torch.randint(0, 10, (50, cols), generator=gen, device=DEV)]
    bits = s.view(torch.int32).long()
    key = torch.where(bits < 0, -(bits & 0x7fffffff) - 1, bits)
    for kk in (1, 8, cols):
        want = torch.sort(key, dim=1, descending=True, stable=True).indices[:, :kk].int()
        want = torch.cat((want, want.new_full((50, kk - want.shape[1]), cols - 1)), 1)
        assert torch.equal(ops.topk_rows(s.contiguous(), kk), want)
