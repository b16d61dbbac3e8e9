"""GPU: the projection with norm, rotation and block means in its epilogue (``s3r_qkv_project``) against float64 on the same
rounded projection and against the pass over the projection, at the edges of tiles, blocks and tables."""
import pytest
import torch
import torch.nn.functional as F

from speed3r_amd import _lib
from speed3r_amd.layers import RoPE2D, SparseFlashAttentionRope
from speed3r_amd.sparse_attn import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(b, n, h, dtype, seed=0, spread=30):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    randn = lambda *s: torch.randn(*s, generator=gen, device=DEV)
    c = 64 * h
    x, w, bias = randn(b, n, c).to(dtype), (randn(3 * c, c) / c ** 0.5).to(dtype), randn(3 * c).to(dtype)
    pos = torch.randint(0, spread, (b, n, 2), generator=gen, device=DEV)
    ln = [(1 + 0.2 * randn(64)).to(dtype), (0.3 * randn(64)).to(dtype)], [(1 + 0.2 * randn(64)).to(dtype), None]
    return x, w, bias, pos, ln


def _rotate64(t, pos, cos, sin):
    """2-D rotation of [B,H,N,64] in float64 with the I/O type's tables."""
    out = []
    for half, p in ((t[..., :32], pos[..., 0]), (t[..., 32:], pos[..., 1])):
        cs, sn = (tab.double()[p][:, None] for tab in (cos, sin))
        a, b = half[..., :16], half[..., 16:]
        out += [a * cs - b * sn, b * cs + a * sn]
    return torch.cat(out, dim=-1)


def _want(x, w, bias, pos, ln, h, block, rope, rows, eps=1e-6):
    b, n, c = x.shape
    # the projection's own rounding: float64 products rounded once, which fp32 sums may round the other way
    qkv = (x.double() @ w.double().t() + (bias.double() if bias is not None else 0)).to(x.dtype)
    q, k, v = qkv.view(b, n, 3, h, 64).permute(2, 0, 3, 1, 4).unbind(0)
    cos, sin = rope.tables(64, rows, x.device, x.dtype)
    nc = -(-n // block)
    pad = nc * block - n
    cnt = torch.full((nc, 1), float(block), device=DEV, dtype=torch.float64)
    cnt[-1] -= pad

    def pool(t):
        return (F.pad(t.double(), (0, 0, 0, pad)).view(b, h, nc, block, 64).sum(3) / cnt).to(x.dtype)

    pos_c = (F.pad(pos, (0, 0, 0, pad)).view(b, nc, block, 2).sum(2) / cnt).long()

    def norm(t, p):
        return t.double() if p is None else F.layer_norm(t.double(), (64,), p[0].double(), None if p[1] is None else p[1].double(), eps)

    lq, lk = ln if ln is not None else (None, None)
    tok = [_rotate64(norm(q, lq), pos, cos, sin), _rotate64(norm(k, lk), pos, cos, sin), v.double()]
    return tok, [_rotate64(norm(pool(q), lq), pos_c, cos, sin), _rotate64(norm(pool(k), lk), pos_c, cos, sin), pool(v).double()]


# rows around the tiles of 128 and 256 tokens, ragged last blocks, several sequences with a tile across their border, several
# tiles per workgroup (the last two: the 256-wide tile)
@pytest.mark.parametrize("b,n,h,block", [(1, 1, 2, 64), (1, 65, 2, 16), (1, 127, 4, 64), (1, 300, 2, 16), (2, 320, 2, 64), (3, 272, 4, 16),
                                         (1, 2017, 16, 16), (2, 2560, 16, 16), (1, 16000, 6, 64), (1, 25212, 16, 64), (1, 24200, 16, 16)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_project_matches_float64(b, n, h, block, dtype):
    x, w, bias, pos, ln = _case(b, n, h, dtype, seed=n)
    rope = RoPE2D(100.0)
    cos, sin = rope.tables(64, 40, x.device, dtype)
    got = ops.qkv_project(x, w, bias, h, block, pos, cos, sin, *ln, 1e-6, pooled=True)
    tok, means = _want(x, w, bias, pos, ln, h, block, rope, 40)
    step = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
    for name, g, e in zip("q k v qc kc vc".split(), got, tok + means):
        assert g.shape == e.shape and g.is_contiguous()
        d = (g.double() - e).abs()
        # one rounding of the result, and where an fp32 sum rounded the projection (or a mean) the other way one step of one
        # value of the row, which norm (|w| <= 2, 1/std <= 2 here) and rotation spread to two values at most twofold each
        assert (d <= step * (0.5 * e.abs() + 8 * (1 + e.abs()))).all(), name
        # a rounding's error is spread evenly over a step: 0.29 of it; the means of q and k take three more (the norm, the two
        # products: together at most 2 more of the same size); flipped values are rare
        assert d.norm() <= (0.6 if name in ("qc", "kc") else 0.35) * step * e.norm(), name


@pytest.mark.parametrize("n", [700, 24200])
def test_project_without_means_or_norm_and_at_far_positions(n):
    """Positions beyond the staged rows, beyond the tables and below zero, as the pass over the projection takes them."""
    h = 16
    x, w, bias, pos, ln = _case(1, n, h, torch.bfloat16, seed=3)
    pos[0, 5] = torch.tensor([63, 64])
    pos[0, 37] = torch.tensor([65, 1])
    pos[0, 300:340, 0] = 150
    pos[0, n - 1] = torch.tensor([100000, 2])
    pos[0, 17] = torch.tensor([-3, 4])
    rope = RoPE2D(100.0)
    cos, sin, inv_freq = rope.fused_tables(64, None, x.device, x.dtype, bounded=True)
    qkv = ops.linear(x, w, bias)
    for q_ln, k_ln, block, pooled in ((*ln, 64, True), (*ln, 16, True), (*ln, 64, False), (None, None, 64, False)):
        for tables, freq in (((cos, sin), inv_freq), (rope.tables(64, 101, x.device, x.dtype), None), ((cos[:20], sin[:20]), inv_freq)):
            for p in (pos, pos.int()):
                got = ops.qkv_project(x, w, bias, h, block, p, *tables, q_ln, k_ln, 1e-6, pooled=pooled, inv_freq=freq)
                want = ops.qkv_prepass(qkv, h, block, p, *tables, q_ln, k_ln, 1e-6, pooled="final" if pooled else None, inv_freq=freq)
                assert torch.equal(got[2], want[2])
                for g, e in zip(got, want):
                    # a cos - b sin: the pass also rounds a, b and both products, each by up to 2^-8 of |a| or |b|, which are
                    # at most sqrt(2) of the row's largest result; the results themselves round once on either side
                    g, e = g.float(), e.float()
                    assert ((g - e).abs() <= 2.0 ** -8 * (4 * 1.42 * e.abs().amax(-1, keepdim=True) + 2 * e.abs())).all()
                    assert (g - e).norm() <= 4e-3 * e.norm()


# thin tiles of the gate: fewer tiles than XCDs, as many workgroups as tiles, a last round of tiles with idle workgroups, of the
# large and of the small tile
@pytest.mark.parametrize("n,h", [(1, 2), (130, 2), (2016, 16), (25212, 16), (65536, 2), (30000, 6), (21600, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_project_with_the_gate(n, h, dtype):
    x, w, bias, pos, ln = _case(1, n, h, dtype, seed=n)
    c = 64 * h
    gw, gb = (torch.randn(2 * h, c, device=DEV) / c ** 0.5).to(dtype), torch.randn(2 * h, device=DEV).to(dtype)
    cos, sin = RoPE2D(100.0).tables(64, 40, x.device, dtype)
    plain = ops.qkv_project(x, w, bias, h, 64, pos, cos, sin, *ln, 1e-6, pooled=True)
    step = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    rides = bool(_lib.lib().s3r_qkv_project_gate_rides(n, h))
    assert rides or n == 21600
    for b in (gb, None):
        got = ops.qkv_project(x, w, bias, h, 64, pos, cos, sin, *ln, 1e-6, pooled=True, gate=(gw, b))
        assert (got[6] is not None) == rides
        if not rides:
            continue
        assert all(torch.equal(a, e) for a, e in zip(got, plain))
        z = x.double() @ gw.double().t() + (b.double() if b is not None else 0)
        # half a step of the product (a whole one where fp32 sums round it the other way) through a slope of at most 1/4,
        # half a step of the result
        assert ((got[6].double() - z.sigmoid()).abs() <= step * (2 * z.abs() * 0.25 + z.sigmoid()) + 1e-6).all()
    assert ops.qkv_project(x, w, bias, h, 64, pos, cos, sin, *ln, 1e-6, pooled=True, gate=(gw[:3], None))[6] is None


def test_project_keeps_infinities_to_their_rows_and_blocks():
    x, w, bias, pos, ln = _case(1, 100, 2, torch.bfloat16)
    x[0, 99, 0] = float("inf")   # the last row, which the rows behind it repeat
    rope = RoPE2D(100.0)
    cos, sin = rope.tables(64, 40, x.device, x.dtype)
    got = ops.qkv_project(x, w, bias, 2, 16, pos, cos, sin, *ln, 1e-6, pooled=True)
    qkv = ops.linear(x, w, bias)
    want = ops.qkv_prepass(qkv, 2, 16, pos, cos, sin, *ln, 1e-6, pooled="final")
    for g, e in zip(got, want):
        assert torch.equal(g.isfinite(), e.isfinite()) and torch.equal(g.isnan(), e.isnan())


def test_project_refuses_what_it_is_not_built_for():
    rope = RoPE2D(100.0)
    cos, sin = rope.tables(64, 40, torch.device(DEV), torch.bfloat16)
    for b, n, h, block, kw in ((1, 64, 3, 64, {}), (1, 64, 2, 32, {}), (2, 200, 2, 64, {}), (2, 300, 2, 64, {})):
        x, w, bias, pos, ln = _case(b, n, h, torch.bfloat16)
        assert ops.qkv_project(x, w, bias, h, block, pos, cos, sin, *ln, 1e-6, pooled=True) is None
    x, w, bias, pos, ln = _case(1, 64, 2, torch.bfloat16)
    assert ops.qkv_project(x, w, bias, 2, 64, pos, cos, sin, None, None, pooled=True) is None
    assert ops.qkv_project(x, w, bias.float(), 2, 64, pos, cos, sin, *ln, 1e-6, pooled=True) is None


@pytest.mark.parametrize("heads,block_size,norm", [(3, 4, True), (4, 16, True), (4, 8, False), (4, 8, True)])
def test_layers_lay_out_tables_once(heads, block_size, norm):
    class Rope(RoPE2D):
        asked = 0

        def fused_tables(self, *args, **kwargs):
            self.asked += 1
            return super().fused_tables(*args, **kwargs)

    c, rope = 64 * heads, Rope(100.0)
    layer = SparseFlashAttentionRope(c, num_heads=heads, qk_norm=norm, rope=rope, block_size=block_size, topk=2).to(DEV, torch.bfloat16)
    with torch.no_grad():
        layer(torch.randn(1, 2048, c, device=DEV).bfloat16(), xpos=torch.randint(0, 30, (1, 2048, 2), device=DEV), n_pos=40)
    assert rope.asked == 1


# several sequences whose borders lie inside tiles of 128 and of 256 tokens (then with two heads a wave), at any row where there are no
# means; the sizes take the large tile where the second number says so
@pytest.mark.parametrize("b,n,h,pooled,block", [(3, 1041, 2, False, 64), (8, 1041, 16, False, 64), (5, 257, 2, False, 64), (2, 2576, 16, True, 16), (2, 2624, 16, True, 64),
                                                (3, 272, 2, True, 16)])
def test_project_across_the_borders_of_sequences(b, n, h, pooled, block):
    x, w, bias, pos, ln = _case(b, n, h, torch.bfloat16, seed=n)
    rope = RoPE2D(100.0)
    cos, sin, inv_freq = rope.fused_tables(64, None, x.device, x.dtype, bounded=True)
    near = pos.clone()
    for i in range(b):   # on both sides of a border: beyond the staged rows, beyond the tables, below zero
        pos[i, 0], pos[i, 1], pos[i, n - 1], pos[i, n - 2], pos[i, n // 2] = (torch.tensor(p) for p in ([70, 3], [5, 100000], [2, 90], [100001, 66], [-3, 4]))
    for p in (near, pos):
        got = ops.qkv_project(x, w, bias, h, block, p, cos, sin, *ln, 1e-6, pooled=pooled, inv_freq=inv_freq)
        for i in range(b):   # each sequence on its own: no border, the same sums
            one = ops.qkv_project(x[i:i + 1], w, bias, h, block, p[i:i + 1], cos, sin, *ln, 1e-6, pooled=pooled, inv_freq=inv_freq)
            assert all(torch.equal(g[i:i + 1], e) for g, e in zip(got, one))
    tok, means = _want(x, w, bias, near, ln, h, block, rope, 40)
    got = ops.qkv_project(x, w, bias, h, block, near, cos, sin, *ln, 1e-6, pooled=pooled, inv_freq=inv_freq)
    for name, g, e in zip("q k v qc kc vc".split(), got, tok + means):   # bounds: test_project_matches_float64
        assert ((g.double() - e).abs() <= 2.0 ** -7 * (0.5 * e.abs() + 8 * (1 + e.abs()))).all(), name


@pytest.mark.parametrize("b,n", [(1, 1100032), (2, 600064)])
def test_project_beyond_two_to_the_31(b, n):
    """x and every output beyond 2^31 bytes, all outputs together beyond 2^31 values: the same bits as pieces of it."""
    h, block = 16, 64
    x, w, bias, _, ln = _case(b, 64, h, torch.bfloat16)
    x = x.repeat(1, n // 64, 1).add_(torch.arange(n, device=DEV)[None, :, None] % 251 / 251)
    pos = torch.randint(0, 40, (b, n, 2), device=DEV)
    cos, sin = RoPE2D(100.0).tables(64, 40, x.device, x.dtype)
    got = ops.qkv_project(x, w, bias, h, block, pos, cos, sin, *ln, 1e-6, pooled=True)
    for i in range(b):
        for at in (0, n // 128 * 64, 2 ** 31 // 2048 - 128 if b == 1 else 2 ** 31 // 4096, n - 320):
            one = ops.qkv_project(x[i:i + 1, at:at + 320].contiguous(), w, bias, h, block, pos[i:i + 1, at:at + 320], cos, sin, *ln, 1e-6, pooled=True)
            for g, e in zip(got, one):
                part = g[i:i + 1, :, at:at + 320] if g.shape[2] == n else g[i:i + 1, :, at // block:(at + 320) // block]
                assert torch.equal(part, e), (i, at)
