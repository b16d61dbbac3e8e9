"""GPU: linear layers (``s3r_linear``) against float64, at the edges of their tiles, and where the modules keep the call."""
import pytest
import torch
import torch.nn.functional as F
from torch import nn

from speed3r_amd.layers.sparse_attention import linear
from speed3r_amd.sparse_attn import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
ROWS = 1024   # the fewest that the layers hand to the kernel


# rows and outputs around the 128- and 256-wide tiles and the 16-row stores; two steps of K and more; several tiles per workgroup
@pytest.mark.parametrize("m,n,k", [(1, 8, 128), (127, 136, 128), (257, 264, 256), (1000, 200, 384), (6000, 1096, 128), (40000, 520, 128), (3000, 3072, 1024)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear_matches_float64(m, n, k, dtype):
    gen = torch.Generator(device=DEV).manual_seed(m + n)
    x = torch.randn(m, k, generator=gen, device=DEV).to(dtype)
    w = torch.randn(n, k, generator=gen, device=DEV).to(dtype)
    w[n // 2, 3] = 17.0   # (a product with one large weight lands in one column only)
    b = torch.randn(n, generator=gen, device=DEV).to(dtype)
    half = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11   # half a step of the type, of 8 or 11 binary digits, relative to the value
    for bias in (b, None):
        exact = x.double() @ w.double().t() + (bias.double() if bias is not None else 0.0)
        # half a step of the result, plus K fp32 roundings of the sum of magnitudes
        room = (x.double().abs() @ w.double().abs().t() + 10.0) * k * 2.0 ** -24
        for gelu in (False, True):
            want = F.gelu(exact) if gelu else exact
            got = ops.linear(x, w, bias, gelu)
            assert got.dtype == dtype and got.shape == (m, n)
            # GELU: slope at most 1.13; 1.5e-7 of |x| for the published error function, 2^-22 for the hardware's exp and reciprocal
            bound = half * want.abs() * (1 + half) + 1.13 * room + (exact.abs() * 4e-7 if gelu else 0.0) + 2.0 ** -25
            assert ((got.double() - want).abs() <= bound).all()


def test_gelu_of_infinities_and_nan():
    x, w = torch.ones(6, 128, device=DEV).bfloat16(), torch.ones(8, 128, device=DEV).bfloat16()
    x[1], x[2, 5], x[3, 5], x[4, 5], x[5] = 3e38, float("inf"), float("-inf"), float("nan"), -3e38   # (rows 1 and 5: infinite sums)
    want = F.gelu(F.linear(x, w))
    assert want[1:3].isposinf().all() and want[3:].isnan().all()
    got = ops.linear(x, w, None, gelu=True)
    assert torch.equal(got.isposinf(), want.isposinf()) and torch.equal(got.isnan(), want.isnan()) and torch.equal(got[0], want[0])


@torch.no_grad()
def test_linear_without_inputs():
    m, x = nn.Linear(0, 8, device=DEV, dtype=torch.bfloat16), torch.empty(5, 0, device=DEV, dtype=torch.bfloat16)
    assert torch.equal(linear(m, x), m(x)) and torch.equal(linear(m, x[:0]), m(x[:0]))


@torch.no_grad()
@pytest.mark.parametrize("rows,n,k,gelu,kernel", [(2016, 1024, 4096, False, False), (8064, 1024, 4096, False, True), (2016, 8192, 2048, False, False),
                                                  (2016, 8192, 2048, True, True), (400, 1536, 1536, True, False), (1024, 1024, 1024, False, True)])
def test_long_products_stay_with_the_library_where_it_is_faster(rows, n, k, gelu, kernel, monkeypatch):
    calls = []
    own = ops.linear
    monkeypatch.setattr(ops, "linear", lambda *a: (calls.append(1), own(*a))[1])
    m, x = nn.Linear(k, n, device=DEV, dtype=torch.bfloat16), torch.randn(rows, k, device=DEV, dtype=torch.bfloat16)
    out, want = linear(m, x, gelu), F.gelu(m(x)) if gelu else m(x)
    assert (len(calls) == 1) is kernel and torch.allclose(out.float(), want.float(), atol=2e-2, rtol=2e-2)
    assert torch.equal(linear(nn.Identity(), x), x)


def test_linear_beyond_two_to_the_31():
    """x beyond 2^31 bytes, y beyond 2^31 values: the same bits as pieces of it (which test_linear_matches_float64 checks)."""
    m, n, k = 1100001, 3072, 1024
    x, w, b = torch.randn(m, k, device=DEV, dtype=torch.bfloat16), torch.randn(n, k, device=DEV, dtype=torch.bfloat16), torch.randn(n, device=DEV, dtype=torch.bfloat16)
    y = ops.linear(x, w, b)
    for at in (0, 2 ** 31 // n - 100, 2 ** 31 // (2 * k) - 100, 2 ** 32 // (2 * n) - 100, m - 200):
        assert torch.equal(y[at:at + 200], ops.linear(x[at:at + 200], w, b)), at


def test_a_forward_put_in_the_place_of_linears_is_called(monkeypatch):
    m, x = nn.Linear(256, 128, device=DEV, dtype=torch.bfloat16), torch.randn(4096, 256, device=DEV, dtype=torch.bfloat16)
    own = nn.Linear.forward
    monkeypatch.setattr(nn.Linear, "forward", lambda self, t: own(self, t) + 1)
    for grad in (False, True):
        with torch.set_grad_enabled(grad):
            assert torch.equal(linear(m, x), m(x))


def test_linear_writes_inside_its_rows_only():
    x, w = torch.randn(300, 256, device=DEV).bfloat16(), torch.randn(264, 256, device=DEV).bfloat16()
    from speed3r_amd import _lib
    buf = torch.full((304, 320), 7.0, device=DEV, dtype=torch.bfloat16)
    rc = _lib.lib().s3r_linear(x.data_ptr(), w.data_ptr(), None, buf.data_ptr(), 300, 264, 256, 256, 256, 320, 0, _lib.S3R_BF16,
                               torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert (buf[300:] == 7.0).all() and (buf[:, 264:] == 7.0).all()
    assert torch.equal(buf[:300, :264], ops.linear(x, w, None))


def test_linear_keeps_hooked_modules_and_other_calls():
    x = torch.randn(ROWS, 256, device=DEV, dtype=torch.bfloat16)
    m = nn.Linear(256, 128, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        plain = linear(m, x)
        assert torch.allclose(plain.float(), m(x).float(), atol=2e-2, rtol=2e-2)
        m.register_forward_hook(lambda mod, args, out: out + 1)
        assert torch.equal(linear(m, x), m(x))
    m = nn.Linear(256, 128, device=DEV, dtype=torch.bfloat16)
    linear(m, x).sum().backward()                       # a gradient is wanted: the module's own graph
    assert m.weight.grad is not None
    with torch.no_grad():
        assert linear(nn.Linear(100, 128, device=DEV, dtype=torch.bfloat16), x[:, :100]).shape == (ROWS, 128)   # sizes without a kernel
        strided = torch.randn(ROWS, 512, device=DEV, dtype=torch.bfloat16)[:, ::2]
        assert torch.equal(linear(m, strided), m(strided))
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert linear(nn.Linear(256, 128, device=DEV), x).dtype == torch.bfloat16
        import torch.autograd.forward_ad as fwad
        with fwad.dual_level():
            out = linear(m, fwad.make_dual(x, torch.ones_like(x)))
            assert fwad.unpack_dual(out).tangent is not None
        assert torch.equal(torch.vmap(lambda row: linear(m, row))(x[:, None]), torch.vmap(lambda row: m(row))(x[:, None]))
