"""Gradients of the layer's norm parameters as rows of one tensor: storage of their own, by no more launches than a copy each."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from speed3r_amd.sparse_attn import ops

F32, BF16 = torch.float32, torch.bfloat16


class Writes(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        if "select" not in func.name():
            self.seen.append(func.name())
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("dtypes,writes", [((F32,) * 4, 1), ((BF16,) * 4, 4), ((F32, None, F32, None), 1), ((F32, BF16, None, F32), 2),
                                           ((BF16, None, BF16, None), 2), ((None,) * 4, 0)])
def test_rows_become_tensors_of_their_own(dtypes, writes):
    rows = torch.randn(4, 64, generator=torch.Generator().manual_seed(1))
    with Writes() as mode:
        mode.seen = []
        got = ops._norm_grads(rows if any(dtypes) else None, [d and torch.empty(64, dtype=d) for d in dtypes][:4])
    seen = [n for n in mode.seen if "empty" not in n]
    assert len(seen) == writes, seen
    for g, d, row in zip(got, dtypes, rows):
        assert (g is None) == (d is None)
        if g is not None:
            assert torch.equal(g, row.to(d)) and g.untyped_storage().nbytes() == g.nbytes
    kept = [g for g in got if g is not None]
    assert len({g.untyped_storage().data_ptr() for g in kept} | {rows.untyped_storage().data_ptr()}) == len(kept) + 1
