"""Blocks of the model are called as modules wherever that does more than ``Block.forward`` (CPU)."""
from contextlib import nullcontext

import pytest
import torch
from torch import nn

from speed3r_amd.layers import RoPE2D
from speed3r_amd.model import Pi3SparseLike
from speed3r_amd.model.pi3_sparse_like import Block, DenseAttentionRope, run_blocks


class Shifted(Block):
    def forward(self, x, **kw):
        return super().forward(x, **kw) + 1.0


class Double(nn.Module):
    def forward(self, x, xpos=None, n_pos=None):
        return 2.0 * x


class Wrapper(nn.Module):
    """Forwards attributes to the module inside, as checkpoint wrappers do."""

    def __init__(self, inner):
        super().__init__()
        self.inner, self.calls = inner, 0

    def __getattr__(self, name):
        try:
            return super().__getattr__(name)
        except AttributeError:
            return getattr(self.inner, name)

    def forward(self, x, **kw):
        self.calls += 1
        return self.inner(x, **kw)


def _blocks(kind):
    torch.manual_seed(0)
    make = lambda cls: cls(32, 2, DenseAttentionRope, init_values=0.5, rope=RoPE2D(100.0))
    blocks = nn.ModuleList([make(Block) for _ in range(4)])
    if kind == "subclass":
        blocks[1] = make(Shifted)
    elif kind == "replaced":
        blocks[2].forward = lambda x, **kw: x + 1.0
    elif kind == "other":
        blocks[0], blocks[3] = Double(), Double()
    elif kind == "wrapper":
        blocks[1] = Wrapper(blocks[1])
    return blocks


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("kind", ["plain", "subclass", "replaced", "other", "wrapper"])
def test_blocks_in_sequence_are_the_modules_calls(kind, grad):
    blocks = _blocks(kind)
    x = torch.randn(2, 5, 32, requires_grad=grad)
    pos = torch.randint(0, 4, (2, 5, 2))
    norm = nn.LayerNorm(32)
    with nullcontext() if grad else torch.no_grad():
        got, normed = run_blocks(blocks, x, norm, xpos=pos, n_pos=5)
        want = x
        for blk in blocks:
            want = blk(want, xpos=pos, n_pos=5)
    assert torch.equal(got, want) and torch.equal(normed, norm(want))
    if kind == "wrapper":
        assert blocks[1].calls == 2


@pytest.mark.parametrize("grad", [False, True])
def test_every_kind_of_hook_fires_once_per_block(grad):
    blocks, seen = _blocks("plain"), []
    handles = [blocks[0].register_forward_hook(lambda m, i, o: seen.append("forward")),
               blocks[1].register_forward_pre_hook(lambda m, i: seen.append("pre")),
               nn.modules.module.register_module_forward_hook(lambda m, i, o: seen.append("global") if isinstance(m, Block) else None)]
    if grad:
        handles.append(blocks[2].register_full_backward_hook(lambda m, gi, go: seen.append("backward")))
    try:
        with nullcontext() if grad else torch.no_grad():
            x, _ = run_blocks(blocks, torch.randn(1, 3, 32, requires_grad=grad), None, xpos=torch.zeros((1, 3, 2), dtype=torch.int64))
        if grad:
            x.sum().backward()
    finally:
        for handle in handles:
            handle.remove()
    assert sorted(seen) == ["backward"] * grad + ["forward"] + ["global"] * 4 + ["pre"]


def test_decoder_takes_any_module_for_a_block():
    torch.manual_seed(0)
    m = Pi3SparseLike(dim=64, enc_depth=1, dec_depth=4, num_heads=2, head_depth=1, grid=(4, 4)).eval()
    for i in range(2):
        m.global_decoder[i] = Double()
    m.local_decoder[1] = Wrapper(m.local_decoder[1])
    with torch.no_grad():
        imgs = torch.rand(1, 2, 3, 56, 56)
        got = m(imgs, return_features=True)
        tokens = m.encoder(((imgs - m.image_mean) / m.image_std).reshape(2, 3, 56, 56))
        x = torch.cat((m.register_token.expand(2, -1, -1), tokens), dim=1)
        pos = m._positions(2, 4, 4, x.device)
        for i in range(2):
            x = local = m.local_decoder[i](x, xpos=pos, n_pos=5)
            x = 2.0 * x
    assert torch.equal(got["features"], torch.cat((local, x), dim=-1)) and m.local_decoder[1].calls == 2
