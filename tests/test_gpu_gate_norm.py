"""The layer's gate and the residual sum with its norm as one pass each, against the torch expressions in fp64, at the edges of
their tiles."""
import pytest
import torch
import torch.nn.functional as F

from speed3r_amd.sparse_attn import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
UNIT = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}   # unit roundoff: half a step at a power of two


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,c,o,bias", [(1, 1024, 32, True), (16, 1024, 32, False), (17, 512, 16, True), (16399, 1024, 32, True),
                                           (33, 256, 8, True), (100, 768, 24, True), (2016, 1024, 2, True)])
def test_gate_matches_the_modules(dtype, rows, c, o, bias):
    g = torch.Generator(device=DEV).manual_seed(rows)
    x = torch.randn((1, rows, c), generator=g, device=DEV).to(dtype)
    w = (torch.randn((o, c), generator=g, device=DEV) * 0.05).to(dtype)
    b = torch.randn(o, generator=g, device=DEV).to(dtype) if bias else None
    got = ops.gate(x, w, b)
    lin = F.linear(x.double(), w.double(), b.double() if bias else None)
    # the product rounded to the type (through a slope of at most 1/4), the sigmoid rounded again; 1e-5 for the fp32 sums
    bound = 0.25 * UNIT[dtype] * lin.abs() + UNIT[dtype] * lin.sigmoid() * 1.01 + 1e-5
    assert got.shape == (1, rows, o) and ((got.double() - lin.sigmoid()).abs() <= bound).all()


def test_gate_has_no_kernel_for_other_forms():
    x = torch.zeros((4, 1024), dtype=torch.bfloat16, device=DEV)
    w = torch.zeros((32, 1024), dtype=torch.bfloat16, device=DEV)
    assert ops.gate(x.float(), w.float(), None) is None
    assert ops.gate(x, w.float(), None) is None
    assert ops.gate(x[:, :192], w[:, :192], None) is None
    assert ops.gate(x.t()[:256], w[:, :4], None) is None
    assert ops.gate(x, torch.zeros((34, 1024), dtype=torch.bfloat16, device=DEV), None) is None
    assert ops.gate(x[:0], w, None) is None
    assert ops.gate(x, w, w[0, :1]) is None   # (a bias that torch spreads over the outputs)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,c,gamma,bias", [(1, 1024, True, True), (5, 1024, False, True), (1023, 1024, True, False), (7, 8, True, True),
                                               (9, 520, False, True), (3, 2048, True, True)])
def test_residual_and_norm_match_the_two_steps(dtype, rows, c, gamma, bias):
    g = torch.Generator(device=DEV).manual_seed(rows + c)
    x, a = (torch.randn((rows, c), generator=g, device=DEV).to(dtype) for _ in range(2))
    w, b, gm = (torch.randn(c, generator=g, device=DEV).to(dtype) for _ in range(3))
    b, gm = b if bias else None, gm if gamma else None
    s, y = ops.add_layer_norm(x, a, gm, w, b, 1e-6)
    prod = a.double() * gm.double() if gamma else a.double()
    assert ((s.double() - (x.double() + prod)).abs() <= UNIT[dtype] * (x.double() + prod).abs() + 1e-6 * (1 + prod.abs())).all()
    assert torch.equal(y, ops.layer_norm(s, w, b, 1e-6))      # the norm of the rounded sum, bit for bit


def test_residual_and_norm_refuse_other_forms():
    x = torch.zeros((4, 64), dtype=torch.bfloat16, device=DEV)
    w = torch.zeros(64, dtype=torch.bfloat16, device=DEV)
    assert ops.add_layer_norm(x, x.float(), None, w, w, 1e-6) is None
    assert ops.add_layer_norm(x, x, None, w.float(), w.float(), 1e-6) is None
    assert ops.add_layer_norm(x.t().contiguous().t(), x, None, w, w, 1e-6) is None
    assert ops.add_layer_norm(x[:, :33], x[:, :33], None, w[:33], None, 1e-6) is None
