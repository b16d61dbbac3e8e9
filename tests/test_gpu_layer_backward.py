"""The layer's own backward kernels (gated merge; block means, qk-norm and RoPE of the packed projection) against autograd
through the torch expressions in fp64 (needs an MI355X)."""
import pytest
import torch

from speed3r_amd.layers import RoPE2D, SparseFlashAttentionRope, block_positions
from speed3r_amd.sparse_attn import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
STEP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _close(got, want, dtype, steps=0):
    """Within one rounding of the result; ``steps``: and that many rounding steps of the row's largest value."""
    want = want.double().cpu()
    room = want.abs() + (steps * want.abs().amax(-1, keepdim=True) if steps else 0.05 * want.pow(2).mean().sqrt())
    return bool(((got.double().cpu() - want).abs() <= STEP[dtype] * room + 1e-6).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,block", [(1, 16), (7, 64), (16, 16), (17, 16), (64, 64), (65, 64), (200, 16), (1041, 64)])
def test_merge_backward(dtype, n, block):
    b, h, nc = 2, 3, -(-n // block)
    g = torch.Generator().manual_seed(n + block)
    oc, os_, dout = (torch.randn(s, generator=g).to(dtype).to(DEV) for s in ((b, h, nc, 64), (b, h, n, 64), (b, n, h * 64)))
    gate = torch.rand((b, n, 2 * h), generator=g).to(dtype).to(DEV).view(b, n, h, 2).permute(0, 2, 1, 3)
    d_oc, d_os, d_gate, delta_c, delta_s = ops.gated_merge_bwd(dout, oc, os_, gate, block)
    co, so, gt = (t.double().requires_grad_() for t in (oc, os_, gate))
    out = gt[..., 0:1] * co[:, :, torch.arange(n, device=DEV) // block] + gt[..., 1:2] * so
    want = torch.autograd.grad(out.permute(0, 2, 1, 3).reshape(b, n, h * 64), (co, so, gt), dout.double())
    assert _close(d_oc, want[0], dtype) and _close(d_os, want[1], dtype) and _close(d_gate, want[2], dtype)
    for delta, d, o in ((delta_c, d_oc, oc), (delta_s, d_os, os_)):   # fp32 sums of 64 products of the rounded gradients
        ref = (d.double() * o.double())
        assert ((delta.double() - ref.sum(-1)).abs() <= 64 * 2.0 ** -24 * ref.abs().sum(-1) + 1e-12).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,block,norm,rot,high", [(1, 16, True, True, 5), (17, 16, True, True, 60), (65, 64, True, True, 300), (200, 16, False, True, 70),
                                                   (130, 64, True, False, 1), (1041, 64, True, True, 40), (5000, 16, True, True, 40)])
@pytest.mark.parametrize("fp32_norm", [False, True])
def test_projection_backward(dtype, n, block, norm, rot, high, fp32_norm):
    """``high`` > 64: positions beyond the default tables (angles evaluated in the kernel).  Positions int64 and int32."""
    b, h, nc = 2, 3, -(-n // block)
    g = torch.Generator().manual_seed(n + block + high)
    rnd = lambda *s: torch.randn(s, generator=g).to(dtype).to(DEV)
    qkv = rnd(b, n, 3 * h * 64)
    pos = torch.randint(0, high, (b, n, 2), generator=g).to(DEV) if rot else None
    if rot and block == 16:
        pos = pos.to(torch.int32)
    ldt = torch.float32 if fp32_norm else dtype
    ln = [((1 + 0.3 * torch.randn(64, generator=g)).to(ldt).to(DEV), (0.2 * torch.randn(64, generator=g)).to(ldt).to(DEV)) for _ in range(2)]
    q_ln, k_ln = ln if norm else (None, None)
    rope = RoPE2D(100.0)
    cos, sin, inv = rope.fused_tables(64, None, qkv.device, dtype) if rot else (None, None, None)
    fwd = ops.qkv_prepass(qkv, h, block, pos, cos, sin, q_ln, k_ln, 1e-6, pooled="final", keep_raw=True, inv_freq=inv)
    grads = [rnd(*t.shape) for t in fwd[:6]]
    d_qkv, d_norm = ops.qkv_prepass_bwd(qkv, h, block, pos, cos, sin, q_ln, k_ln, 1e-6, fwd[6:], grads, inv)

    x = qkv.double().requires_grad_()
    par = [t.double().requires_grad_() for pair in ln for t in pair]
    q, k, v = x.view(b, n, 3, h, 64).permute(2, 0, 3, 1, 4).unbind(0)
    blk = torch.arange(n, device=DEV) // block

    def pool(t, like=None):   # the kernels go on from the rounded mean; its gradient is the mean's
        s = torch.zeros((b, h, nc, 64), dtype=torch.float64, device=DEV).index_add(2, blk, t)
        m = s / torch.bincount(blk)[:, None]
        return m if like is None else m + (like.double() - m).detach()

    def angles(p):       # rounded to the tokens' dtype like their cosines and sines
        a = (p.float()[..., None] * rope.inv_freq(64, qkv.device)).to(dtype)
        return a.cos().double()[:, None], a.sin().double()[:, None]

    def norm_rot(t, which, p):
        if norm:
            t = torch.nn.functional.layer_norm(t, (64,), par[2 * which], par[2 * which + 1], 1e-6)
        if p is None:
            return t
        out = []
        for half in range(2):
            c, s = angles(p[..., half])
            a, e = t[..., 32 * half:32 * half + 16], t[..., 32 * half + 16:32 * half + 32]
            out += [a * c - e * s, e * c + a * s]
        return torch.cat(out, -1)

    pc = block_positions(pos, block) if rot else None
    raw_q, raw_k = fwd[6:] if norm else (None, None)
    outs = (norm_rot(q, 0, pos), norm_rot(k, 1, pos), v, norm_rot(pool(q, raw_q), 0, pc), norm_rot(pool(k, raw_k), 1, pc), pool(v))
    for got, want in zip(fwd[:6], outs):
        assert _close(got, want.detach(), dtype, steps=3)   # norm, two products, sum: half a step each, terms up to sqrt(2) of the row's maximum
    want = torch.autograd.grad(outs, [x, *(par if norm else [])], [t.double() for t in grads])
    assert _close(d_qkv, want[0], dtype)
    if norm:   # fp32 sums of n * h rows per batch
        for i in range(4):
            ref = want[1 + i]
            assert ((d_norm[i].double() - ref).abs() <= 1e-4 * ref.pow(2).mean().sqrt() + 1e-5 * (b * h * n) ** 0.5).all()
    else:
        assert d_norm is None


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,block,high", [(1, 64, 3), (33, 16, 40), (200, 64, 64), (333, 16, 500), (1041, 64, 40), (130, 256, 40)])
def test_finished_block_means_and_split_passes(dtype, n, block, high):
    """Block means normalised and rotated in the pass: the bits of pooling, ``block_positions`` and the norm + RoPE kernel
    with a table that covers every position; the pass in two launches gives the bits of one; int32 and int64 positions."""
    b, h = 2, 3
    g = torch.Generator().manual_seed(n + high)
    qkv = (torch.randn((b, n, 3 * h * 64), generator=g) * 0.7).to(dtype).to(DEV)
    pos = torch.randint(0, high, (b, n, 2), generator=g).to(DEV)
    ln = [((1 + 0.3 * torch.randn(64, generator=g)).to(dtype).to(DEV), (0.2 * torch.randn(64, generator=g)).to(dtype).to(DEV)) for _ in range(2)]
    rope = RoPE2D(100.0)
    cos, sin, inv = rope.fused_tables(64, None, qkv.device, dtype)
    full = rope.tables(64, high, qkv.device, dtype)
    got = ops.qkv_prepass(qkv, h, block, pos, cos, sin, *ln, 1e-6, pooled="final", inv_freq=inv)
    q, k, v = qkv.view(b, n, 3, h, 64).permute(2, 0, 3, 1, 4).unbind(0)
    raw = ops.pool_qkv_packed(qkv, h, block)
    pc = block_positions(pos, block)
    want = (*(ops.norm_rope(t, pos, *full, *l, 1e-6) for t, l in zip((q, k), ln)), v,
            *(ops.norm_rope(t, pc, *full, *l, 1e-6) for t, l in zip(raw, ln)), raw[2])
    for i, (a, w) in enumerate(zip(got, want)):
        assert torch.equal(a, w), i
    split = (*ops.qkv_prepass(qkv, h, 64, pos.to(torch.int32), cos, sin, *ln, 1e-6, pooled=None, inv_freq=inv),
             *ops.qkv_prepass(qkv, h, block, pos, cos, sin, *ln, 1e-6, tokens=False, pooled="final", inv_freq=inv))
    for a, w in zip(split, got):
        assert torch.equal(a, w)


def test_training_after_inference_mode():
    """Tables laid out, and positions made, in inference mode serve a training call (whose backward saves them)."""
    torch.manual_seed(0)
    layer = SparseFlashAttentionRope(128, num_heads=2, qkv_bias=True, qk_norm=True, rope=RoPE2D(100.0), block_size=8, topk=2).to(DEV, torch.bfloat16)
    x = torch.randn((1, 130, 128), device=DEV, dtype=torch.bfloat16)
    with torch.inference_mode():
        pos = torch.randint(0, 30, (1, 130, 2), device=DEV)
        layer(x, xpos=pos)
    got = torch.autograd.grad(layer(x, xpos=pos).float().square().sum(), list(layer.parameters()))
    layer.rope._tables.clear()
    want = torch.autograd.grad(layer(x, xpos=pos.clone()).float().square().sum(), list(layer.parameters()))
    assert all(torch.isfinite(g).all() for g in got)
    assert torch.equal(layer(x, xpos=pos), layer(x, xpos=pos.clone()))
    # two runs of the same kernels: the bits may differ only where a reduction's order does (one rounding of the result)
    assert all(_close(g, w, torch.bfloat16, steps=1) for g, w in zip(got, want))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,block,low,high", [(33, 16, -9, 0), (64, 16, -3, 4), (200, 64, -70, 0), (130, 64, -5, 70), (130, 256, -4, 2)])
@pytest.mark.parametrize("bound", [None, 3])
def test_positions_below_zero_take_the_first_table_row(dtype, n, block, low, high, bound):
    """Tokens' and block means' positions below zero, in one coordinate or both, are clamped like those beyond a bounded
    table: the bits of the norm + RoPE kernel, in one launch and in two (which holds no tables in LDS)."""
    b, h = 2, 3
    g = torch.Generator().manual_seed(n - low)
    qkv = (torch.randn((b, n, 3 * h * 64), generator=g) * 0.7).to(dtype).to(DEV)
    pos = torch.randint(low, high, (b, n, 2), generator=g)
    pos[0, :, 1] = pos[0, :, 1].abs()
    pos = pos.to(DEV)
    ln = [((1 + 0.3 * torch.randn(64, generator=g)).to(dtype).to(DEV), (0.2 * torch.randn(64, generator=g)).to(dtype).to(DEV)) for _ in range(2)]
    rope = RoPE2D(100.0)
    cos, sin, inv = rope.fused_tables(64, bound, qkv.device, dtype)
    full = rope.tables(64, bound or 128, qkv.device, dtype)
    q, k, v = qkv.view(b, n, 3, h, 64).permute(2, 0, 3, 1, 4).unbind(0)
    raw, pc = ops.pool_qkv_packed(qkv, h, block), block_positions(pos, block)
    want = (*(ops.norm_rope(t, pos, *full, *l, 1e-6) for t, l in zip((q, k), ln)), v,
            *(ops.norm_rope(t, pc, *full, *l, 1e-6) for t, l in zip(raw, ln)), raw[2])
    args = pos, cos, sin, *ln, 1e-6
    one = ops.qkv_prepass(qkv, h, block, *args, pooled="final", inv_freq=inv)
    two = (*ops.qkv_prepass(qkv, h, 64, *args, pooled=None, inv_freq=inv),
           *ops.qkv_prepass(qkv, h, block, *args, tokens=False, pooled="final", inv_freq=inv))
    for got in (one, two):
        for i, (a, w) in enumerate(zip(got, want)):
            assert torch.equal(a, w), i
