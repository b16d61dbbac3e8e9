"""The layer's training route against the same layer composed of torch modules (needs an MI355X)."""
import pytest
import torch
from torch import nn

from speed3r_amd.layers import RoPE2D, SparseFlashAttentionRope

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DIM, HEADS = 128, 2


class TorchRope(nn.Module):
    """RoPE2D as a module of another type: the layer composes torch expressions around it."""

    def __init__(self, rope):
        super().__init__()
        self.rope = rope

    def forward(self, tokens, positions):
        return self.rope(tokens, positions)


def _layer(rope, block_size=8, seed=0, dtype=torch.bfloat16, topk=4):
    torch.manual_seed(seed)
    m = SparseFlashAttentionRope(DIM, num_heads=HEADS, qkv_bias=True, qk_norm=True, rope=rope, block_size=block_size, topk=topk)
    with torch.no_grad():
        m.gate[0].weight.normal_(0, 0.05)
        for norm in (m.q_norm, m.k_norm):
            norm.weight.uniform_(0.5, 1.5)
            norm.bias.normal_(0, 0.1)
    return m.to(DEV, dtype)


def _step(m, x, pos, dout, **kw):
    """{name: tensor} of the output, the input's gradient and every parameter's."""
    x = x.detach().requires_grad_()
    out = m(x, xpos=pos, **kw)
    names, params = zip(*m.named_parameters())
    grads = torch.autograd.grad(out, (x, *params), dout, allow_unused=True)
    return {"out": out.detach(), "x": grads[0], **dict(zip(names, grads[1:]))}


def _inputs(n, b=1, high=40, seed=1, low=0, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    x, dout = (torch.randn((b, n, DIM), generator=g).to(DEV, dtype) for _ in range(2))
    return x, torch.randint(low, high, (b, n, 2), generator=g).to(DEV), dout


def _same(got, want):
    """Two 16-bit evaluations of the same sums: a chain of at most a dozen roundings to 2^-9, some of them of terms that
    cancel to a fifth: 5e-2 of the tensor's norm.  Positions that are off by one change it by more than a third."""
    assert got.keys() == want.keys()
    for k in want:
        assert got[k].dtype == want[k].dtype and got[k].shape == want[k].shape, k
        assert torch.isfinite(got[k]).all(), k
        diff, size = (got[k].double() - want[k].double()).norm(), want[k].double().norm()
        assert diff <= 5e-2 * size, (k, float(diff / size))


@pytest.mark.parametrize("block_size,n", [(8, 256), (8, 200), (4, 60)])
@pytest.mark.parametrize("n_pos", [None, 41, 8])
def test_training_rotates_by_every_position_whatever_the_tables(block_size, n, n_pos):
    """Positions beyond a rope module's ``max_positions`` and beyond a call's ``n_pos`` keep their own angles in training."""
    x, pos, dout = _inputs(n, high=41)
    got = _step(_layer(RoPE2D(100.0, max_positions=8), block_size), x, pos, dout, n_pos=n_pos)
    _same(got, _step(_layer(TorchRope(RoPE2D(100.0)), block_size), x, pos, dout))


class _ScaledRope(RoPE2D):
    def forward(self, tokens, positions):
        return super().forward(tokens, 2 * positions)


@pytest.mark.parametrize("what", ["q_norm hook", "k_norm pre-hook", "backward hook", "rope hook", "global hook", "rope subclass", "replaced forward"])
def test_training_calls_norms_and_rope_that_do_more_than_their_forward(what):
    """Hooks fire once for the tokens and once for the block means, and what they return counts."""
    x, pos, dout = _inputs(200)
    calls = []

    def scaled(mod, args, out):
        calls.append(1)
        return 0.5 * out

    def change(m):
        if what == "q_norm hook":
            return [m.q_norm.register_forward_hook(scaled)]
        if what == "k_norm pre-hook":
            return [m.k_norm.register_forward_pre_hook(lambda mod, args: (calls.append(1), (args[0] + 0.5,))[1])]
        if what == "backward hook":
            return [m.q_norm.register_full_backward_hook(lambda *a: calls.append(1))]
        if what == "rope hook":
            return [m.rope.register_forward_hook(scaled)]
        if what == "global hook":
            return [nn.modules.module.register_module_forward_hook(
                lambda mod, args, out: scaled(mod, args, out) if isinstance(mod, nn.LayerNorm) else None)]
        if what == "rope subclass":
            m.rope = TorchRope(_ScaledRope(100.0)) if isinstance(m.rope, TorchRope) else _ScaledRope(100.0)
        else:
            m.q_norm.forward = lambda t: nn.functional.layer_norm(t, (64,))
        return []

    results = []
    for rope in (RoPE2D(100.0), TorchRope(RoPE2D(100.0))):
        m = _layer(rope)
        calls.clear()
        handles = change(m)
        try:
            results.append((_step(m, x, pos, dout), len(calls)))
        finally:
            for handle in handles:
                handle.remove()
    (got, fired), (want, expected) = results
    assert fired == expected
    want, got = ({k: v for k, v in d.items() if v is not None} for d in (want, got))
    _same(got, want)


@pytest.mark.parametrize("shape", [(1, 200, 2), (3, 200, 2), (3, 1, 2), (1, 1, 2)])
def test_training_broadcasts_positions_over_the_batch(shape):
    x, _, dout = _inputs(200, b=3)
    pos = torch.randint(0, 40, shape, generator=torch.Generator().manual_seed(2)).to(DEV)
    _same(_step(_layer(RoPE2D(100.0)), x, pos, dout), _step(_layer(TorchRope(RoPE2D(100.0))), x, pos, dout))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.int32, torch.int16, torch.uint8])
@pytest.mark.parametrize("block_size", [8, 4])
def test_training_with_positions_of_any_type(dtype, block_size):
    """Fractional positions have their own angles (block means take the truncated mean, like the others)."""
    x, pos, dout = _inputs(200, high=30)
    pos = (pos.float() + 0.5).to(dtype) if dtype.is_floating_point else pos.to(dtype)
    _same(_step(_layer(RoPE2D(100.0), block_size, topk=16), x, pos, dout), _step(_layer(TorchRope(RoPE2D(100.0)), block_size, topk=16), x, pos, dout))


@pytest.mark.parametrize("block_size,low,high", [(8, -20, 20), (4, -90, -60), (8, -1, 1), (4, -3, 90)])
def test_training_with_positions_below_zero(block_size, low, high):
    x, pos, dout = _inputs(200, low=low, high=high)
    _same(_step(_layer(RoPE2D(100.0), block_size, topk=16), x, pos, dout), _step(_layer(TorchRope(RoPE2D(100.0)), block_size, topk=16), x, pos, dout))


def _flat_norms(m):
    """The norm parameters as views of one flat buffer, none of them at a multiple of 16 bytes."""
    flat = torch.cat([torch.zeros(1, dtype=m.q_norm.weight.dtype, device=DEV)] + [t.detach() for norm in (m.q_norm, m.k_norm) for t in (norm.weight, norm.bias)])
    views = flat[1:].split(64)
    for i, norm in enumerate((m.q_norm, m.k_norm)):
        norm.weight, norm.bias = nn.Parameter(views[2 * i]), nn.Parameter(views[2 * i + 1])
    assert all(t.data_ptr() % 16 for t in (*m.q_norm.parameters(), *m.k_norm.parameters()))
    return m


@pytest.mark.parametrize("norm_dtype", [torch.bfloat16, torch.float32])
def test_training_with_norm_parameters_off_a_16_byte_boundary(norm_dtype):
    x, pos, dout = _inputs(200)
    results = []
    for rope in (RoPE2D(100.0), TorchRope(RoPE2D(100.0))):
        m = _layer(rope)
        m.q_norm.to(norm_dtype), m.k_norm.to(norm_dtype)
        _flat_norms(m)
        if norm_dtype == torch.float32:
            with torch.autocast("cuda", dtype=torch.bfloat16):
                results.append(_step(m, x, pos, dout))
        else:
            results.append(_step(m, x, pos, dout))
    _same(*results)


def test_training_with_an_output_gradient_off_a_16_byte_boundary():
    x, pos, dout = _inputs(200)
    odd = torch.empty(dout.numel() + 1, dtype=dout.dtype, device=DEV)[1:].view(dout.shape).copy_(dout)
    results = []
    for grad in (odd, dout):
        m = _layer(RoPE2D(100.0))
        m.proj = nn.Identity()
        results.append(_step(m, x, pos, grad))
    assert all(torch.equal(results[0][k], results[1][k]) for k in results[1])


def test_training_of_the_gate_alone_runs_no_attention_backward(monkeypatch):
    """Nothing but the gate wants a gradient: the attention's is not computed, and the gate's is what it is in full
    training; a second derivative goes through it like through any product."""
    from speed3r_amd.sparse_attn import ops

    x, pos, dout = _inputs(200)
    want = _step(_layer(RoPE2D(100.0)), x, pos, dout)
    m = _layer(RoPE2D(100.0)).requires_grad_(False)
    m.gate.requires_grad_(True)
    ran = []
    for name in ("attn_bwd", "qkv_prepass_bwd", "key_block_lists"):
        real = getattr(ops, name)
        monkeypatch.setattr(ops, name, lambda *a, _real=real, _name=name, **kw: (ran.append(_name), _real(*a, **kw))[1])
    out = m(x, xpos=pos)
    params = list(m.gate.parameters())
    got = torch.autograd.grad(out, params, dout, create_graph=True)
    assert ran == []
    _same({"weight": got[0].detach(), "bias": got[1].detach(), "out": out.detach()},
          {"weight": want["gate.0.weight"], "bias": want["gate.0.bias"], "out": want["out"]})
    second = torch.autograd.grad(sum(g.float().square().sum() for g in got), params)
    assert all(torch.isfinite(t).all() and t.abs().max() > 0 for t in second)


@pytest.mark.parametrize("norm_dtype", [torch.bfloat16, torch.float32])
def test_norm_gradients_share_no_storage(norm_dtype):
    """Each gradient a tensor of its own, nothing of the kernels' workspace behind it."""
    x, pos, dout = _inputs(200)
    m = _layer(RoPE2D(100.0))
    m.q_norm.to(norm_dtype), m.k_norm.to(norm_dtype)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        out = m(x, xpos=pos)
    out.backward(dout)
    grads = [t.grad for norm in (m.q_norm, m.k_norm) for t in norm.parameters()]
    assert all(g.dtype == norm_dtype and g.untyped_storage().nbytes() == g.numel() * g.element_size() for g in grads)
    assert len({g.untyped_storage().data_ptr() for g in grads}) == 4


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("block_size,n,topk", [(8, 200, 2), (8, 256, 4), (4, 200, 8), (4, 250, 16)])
def test_mixed_precision_training_step(dtype, block_size, n, topk):
    """fp32 weights and inputs under autocast, two sequences, whole and ragged last blocks: every gradient in its
    parameter's type, against the composition of torch modules."""
    x, pos, dout = _inputs(n, b=2, dtype=torch.float32, high=30)
    results = []
    for rope in (RoPE2D(100.0), TorchRope(RoPE2D(100.0))):
        m = _layer(rope, block_size, dtype=torch.float32, topk=topk)
        m.keep_topk_idx = True
        with torch.autocast("cuda", dtype=dtype):
            results.append((_step(m, x, pos, dout.to(dtype)), m.last_topk_idx))
    (got, idx), (want, want_idx) = results
    assert (idx == want_idx).float().mean() >= 0.98   # (scores a rounding apart can change places)
    assert all(got[k].dtype == torch.float32 for k in got if k != "out") and got["out"].dtype == dtype
    _same(got, want)
