"""Gradients of linear layers' parameters (``s3r_linear_wgrad``) against float64 at the edges of their tiles and ranges of tokens, and
the calls that keep torch's own graph."""
import pytest
import torch
import torch.nn.functional as F
from torch import nn

from speed3r_amd.layers.sparse_attention import linear, linear_trains
from speed3r_amd.model.pi3_sparse_like import Mlp
from speed3r_amd.sparse_attn import ops

DEV = "cuda"
ROWS = 4096   # the fewest that the layers hand to the kernel


def test_function_has_the_gradients_of_linear():
    x, w, b = (torch.randn(s, dtype=torch.float64, requires_grad=True) for s in ((2, 3, 4), (5, 4), (5,)))
    assert torch.equal(ops._LinearFn.apply(x, w, b), F.linear(x, w, b))
    assert torch.autograd.gradcheck(ops._LinearFn.apply, (x, w, b), check_batched_grad=True)
    assert torch.autograd.gradgradcheck(ops._LinearFn.apply, (x, w, b))
    assert torch.autograd.gradcheck(lambda w: ops._LinearFn.apply(x.detach(), w, None), (w,))
    assert torch.autograd.gradcheck(lambda x, b: ops._LinearFn.apply(x, w.detach(), b), (x, b))


@pytest.mark.parametrize("lead", [(6,), (2, 3)])
@pytest.mark.parametrize("bias", [False, True])
def test_output_may_be_changed_in_place(lead, bias):
    x, w, b = (torch.randn(s, requires_grad=True) for s in ((*lead, 4), (5, 4), (5,)))
    wrt = (x, w, b) if bias else (x, w)
    got, want = (f(x, w, b if bias else None) for f in (ops.linear_autograd, F.linear))
    for out in (got, want):
        out.mul_(2.0)
        out[..., 1:3].add_(1.0)
    assert torch.equal(got, want)
    assert all(torch.equal(g, e) for g, e in zip(torch.autograd.grad(got.sum(), wrt), torch.autograd.grad(want.sum(), wrt)))


# rows below, at and beyond the pairs of steps; outputs and inputs around 16, 128 and 256; one range of tokens, and many
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,c", [(1, 8, 8), (127, 32, 1024), (128, 256, 256), (385, 264, 776), (1000, 32, 1024), (4097, 1032, 1032), (9000, 136, 520), (20161, 3072, 1024)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_wgrad_matches_float64(m, n, c, dtype):
    gen = torch.Generator(device=DEV).manual_seed(m + n)
    dy = torch.randn(m, n + 8, generator=gen, device=DEV).to(dtype)[:, :n]   # (rows of their own strides)
    x = torch.randn(m, c + 16, generator=gen, device=DEV).to(dtype)[:, 8:8 + c]
    bias = c > 768
    dw, db = ops.linear_wgrad(dy, x, bias)
    half = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11   # half a step of the type, relative to the value
    for got, a, b in ((dw, dy, x), (db, dy, torch.ones_like(x[:, :1]))) if bias else ((dw, dy, x),):
        want = a.double().t() @ b.double()
        room = (a.double().abs().t() @ b.double().abs()) * m * 2.0 ** -24   # a rounding of the sum of magnitudes per token
        assert got.dtype == dtype and got.is_contiguous()
        assert ((got.double() - want.view_as(got)).abs() <= half * want.abs().view_as(got) * (1 + half) + room.view_as(got) + 2.0 ** -25).all()
    assert torch.equal(dw, ops.linear_wgrad(dy, x, bias)[0])


# rows around the steps of 64 and the pairs of them, in one range and in many; around them, and in what the same workgroups worked on
# before, values that would show
@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 15, 63, 64, 65, 127, 129, 191, 193, 4100, 4159, 4161])
def test_wgrad_takes_its_rows_only(m):
    nan = float("nan")
    dy, x = (torch.full((m + 256, c), nan, device=DEV).bfloat16() for c in (136, 1032))
    dy[128:128 + m], x[128:128 + m] = torch.randn(m, 136, device=DEV).bfloat16(), torch.randn(m, 1032, device=DEV).bfloat16()
    ops.linear_wgrad(torch.full_like(dy, nan), torch.full_like(x, nan), True)
    a, b = dy[128:128 + m], x[128:128 + m]
    dw, db = ops.linear_wgrad(a, b, True)
    for got, t in ((dw, b), (db, torch.ones_like(b[:, :1]))):
        want, room = a.double().t() @ t.double(), (a.double().abs().t() @ t.double().abs()) * m * 2.0 ** -24
        # half a bf16 step of the value, a rounding of the sum of magnitudes per token
        assert ((got.double() - want.view_as(got)).abs() <= 2.0 ** -8 * want.abs().view_as(got) * (1 + 2.0 ** -8) + room.view_as(got) + 2.0 ** -25).all()


@pytest.mark.gpu
def test_wgrad_beyond_two_to_the_31():
    m, n, c = 1100001, 64, 1032   # x beyond 2^31 bytes
    gen = torch.Generator(device=DEV).manual_seed(0)
    dy, x = torch.randn(m, n, generator=gen, device=DEV, dtype=torch.bfloat16), torch.randn(m, c, generator=gen, device=DEV, dtype=torch.bfloat16)
    dw, db = ops.linear_wgrad(dy, x, True)
    want, mag = torch.zeros(n, c, device=DEV, dtype=torch.float64), torch.zeros(n, c, device=DEV, dtype=torch.float64)
    for a, b in zip(dy.split(100000), x.split(100000)):
        want += a.double().t() @ b.double()
        mag += a.double().abs().t() @ b.double().abs()
    # half a bf16 step of the value; an fp32 rounding of the sum of magnitudes per 16 tokens of one of 64 ranges, and per range (what a
    # tenth of the tokens adds is some 300)
    chain = (m / 64 / 16 + 64) * 2.0 ** -24
    assert ((dw.double() - want).abs() <= 2.0 ** -8 * want.abs() * 1.01 + chain * mag).all() and (chain * mag).max() < 100
    assert ((db.double() - dy.double().sum(0)).abs() <= 2.0 ** -8 * dy.double().sum(0).abs() * 1.01 + chain * dy.double().abs().sum(0)).all()


@pytest.mark.gpu
def test_wgrad_refuses_what_it_is_not_built_for():
    x, dy = torch.randn(256, 512, device=DEV).bfloat16(), torch.randn(256, 64, device=DEV).bfloat16()
    assert ops.linear_wgrad(dy, x, True) is None                       # sums of dY with few inputs
    assert ops.linear_wgrad(dy[:, :60], x, False) is None and ops.linear_wgrad(dy[:, 4:12], x, False) is None
    assert ops.linear_wgrad(dy.float(), x.float(), False) is None and ops.linear_wgrad(dy, x.half(), False) is None
    assert ops.linear_wgrad(dy, x.t().contiguous().t(), False) is None


@pytest.mark.gpu
@pytest.mark.parametrize("autocast", [False, True])
def test_layers_train_through_the_kernel(autocast):
    master = torch.float32 if autocast else torch.bfloat16
    m = nn.Linear(1024, 32, device=DEV, dtype=master)
    x = torch.randn(2, ROWS // 2 + 3, 1024, device=DEV, dtype=master, requires_grad=True)
    wrt = (x, m.weight, m.bias)
    dy = torch.randn(*x.shape[:2], 32, device=DEV).bfloat16()
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        assert linear_trains(m, x)
        got, want = linear(m, x), m(x)
    assert torch.equal(got, want) and type(got.grad_fn).__name__ == "_LinearFnBackward"
    a, b = (torch.autograd.grad(t, wrt, dy, retain_graph=True) for t in (got, want))
    assert torch.equal(a[0], b[0])
    for g, w, mag in zip(a[1:], b[1:], (dy.double().abs().flatten(0, 1).t() @ x.double().abs().flatten(0, 1), dy.double().abs().sum((0, 1)))):
        assert g.dtype == w.dtype == master
        # both within half a bf16 step of the value, and each within one fp32 rounding per token of the sum of magnitudes
        assert ((g.double() - w.double()).abs() <= 2.0 ** -7 * w.double().abs() + 2 * mag * x.shape[1] * 2 * 2.0 ** -24).all()
    second = torch.autograd.grad(got.float().square().sum(), m.weight, create_graph=True)[0]
    assert torch.autograd.grad(second.float().sum(), x)[0].shape == x.shape


@pytest.mark.gpu
def test_other_calls_keep_their_graph():
    x = torch.randn(ROWS, 256, device=DEV, dtype=torch.bfloat16)
    m = nn.Linear(256, 128, device=DEV, dtype=torch.bfloat16)
    assert linear_trains(m, x) and not linear_trains(m, x[1:]) and not linear_trains(m, x.cpu())
    with torch.no_grad():
        assert not linear_trains(m, x)
    assert torch.func.vmap(lambda t: torch.tensor(linear_trains(m, t)))(x[None]).logical_not().all()
    seen = []

    class Probe(torch.autograd.Function):   # what a backward is given where several gradients come at once
        forward = staticmethod(lambda ctx, t: t.clone())
        backward = staticmethod(lambda ctx, g: (seen.append(ops.ordinary(g)), g)[1])

    leaf = x.float().requires_grad_()
    torch.autograd.grad(Probe.apply(leaf), leaf, torch.ones(2, ROWS, 256, device=DEV), is_grads_batched=True)
    assert seen == [False]
    with torch.autograd.forward_ad.dual_level():
        assert not linear_trains(m, torch.autograd.forward_ad.make_dual(x, x))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not linear_trains(m, x.double())
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.to(DEV)):
        out = linear(m, x)
    out.sum().backward()
    assert m.weight.grad.shape == m.weight.shape
    m.register_full_backward_hook(lambda *a: None)
    assert not linear_trains(m, x)


@pytest.mark.gpu
def test_autocast_makes_one_copy_where_it_keeps_it():
    x = torch.randn(8, 8, device=DEV)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert ops.autocast_once(x).dtype == torch.bfloat16
        x.requires_grad_()
        assert ops.autocast_once(x).dtype == torch.bfloat16
        assert ops.autocast_once(x * 1.0).dtype == torch.float32   # two copies, whose gradients meet in fp32
    with torch.autocast("cuda", dtype=torch.bfloat16, cache_enabled=False):
        assert ops.autocast_once(x).dtype == torch.float32
    assert ops.autocast_once(x) is x


@pytest.mark.gpu
def test_calls_in_one_autocast_region_share_the_cast_weights():
    m, x = nn.Linear(1024, 32, device=DEV), torch.randn(2, 8, 1024, device=DEV)
    for cache in (True, False):
        kept, grads = [], []
        for f in (lambda t: ops.linear_autograd(t, m.weight, m.bias), m):
            saved = set()
            with torch.autocast("cuda", dtype=torch.bfloat16, cache_enabled=cache), torch.autograd.graph.saved_tensors_hooks(
                    lambda t: (saved.add(t.untyped_storage().data_ptr()) if t.shape[0] in (32, 1024) else None, t)[1], lambda t: t):
                out = sum(f(t.requires_grad_()).float().square().sum() for t in (x.clone(), x + 1))
                kept.append(len(saved))
            grads.append(torch.autograd.grad(out, (m.weight, m.bias)))
        assert kept == ([1, 1] if cache else [2, 2])
        for g, e in zip(*grads):   # (other sums of the same products: a rounding to bf16 of the value, twice)
            assert g.dtype == torch.float32 and (g - e).abs().max() <= 2.0 ** -7 * e.abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("c,bias", [(256, True), (256, False), (768, True), (776, True)])
def test_weights_of_few_inputs_train_through_the_kernel(c, bias, monkeypatch):
    calls = []
    kernel = ops.linear_wgrad
    monkeypatch.setattr(ops, "linear_wgrad", lambda *a: (calls.append(kernel(*a)), calls[-1])[1])
    m = nn.Linear(c, 64, bias=bias, device=DEV, dtype=torch.bfloat16)
    x, dy = torch.randn(ROWS, c, device=DEV).bfloat16(), torch.randn(ROWS, 64, device=DEV).bfloat16()
    wrt = tuple(m.parameters())
    got, want = torch.autograd.grad(linear(m, x), wrt, dy), torch.autograd.grad(m(x), wrt, dy)
    assert len(calls) == 1 and calls[0] is not None and calls[0][0] is got[0]
    mags = (dy.double().abs().t() @ x.double().abs(), dy.double().abs().sum(0))
    for g, w, mag in zip(got, want, mags):   # as above: half a bf16 step each, an fp32 rounding per token each
        assert ((g.double() - w.double()).abs() <= 2.0 ** -7 * w.double().abs() + 2 * mag * ROWS * 2.0 ** -24).all()


@pytest.mark.gpu
@pytest.mark.parametrize("n,c", [(60, 1024), (64, 100)])
def test_weights_without_a_kernel_keep_their_graph(n, c):
    assert not linear_trains(nn.Linear(c, n, device=DEV, dtype=torch.bfloat16), torch.randn(ROWS, c, device=DEV).bfloat16())


@pytest.mark.gpu
@pytest.mark.parametrize("rows,c,autocast,kernel", [(ROWS, 512, False, False), (16000, 512, False, True), (8320, 768, True, False), (12032, 768, True, True)])
def test_small_steps_keep_the_products_of_torch(rows, c, autocast, kernel, monkeypatch):
    calls = []
    own = ops.linear_autograd
    monkeypatch.setattr(ops, "linear_autograd", lambda *a: (calls.append(1), own(*a))[1])
    m = Mlp(c, 4 * c).to(DEV, torch.float32 if autocast else torch.bfloat16)
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        m(torch.randn(rows, c, device=DEV, dtype=m.fc1.weight.dtype)).float().sum().backward()
    assert len(calls) == (2 if kernel else 0) and all(p.grad is not None for p in m.parameters())


# one tile and less, ragged last tiles, both tile sizes; more inputs than the kernel is faster for, outputs, inputs, a type and a row stride that it does not
# take
@pytest.mark.gpu
@pytest.mark.parametrize("rows,n,k,dtype,kernel", [(1, 8, 128, torch.bfloat16, True), (4099, 136, 1024, torch.bfloat16, True), (8104, 3072, 1024, torch.float16, True),
                                                   (8104, 1024, 1024, torch.bfloat16, True), (4099, 1024, 2048, torch.bfloat16, False), (300, 60, 1024, torch.bfloat16, False), (300, 64, 200, torch.bfloat16, False),
                                                   (300, 64, 256, torch.float32, False)])
@pytest.mark.parametrize("bias", [True, False])
def test_forward_of_the_function(rows, n, k, dtype, kernel, bias, monkeypatch):
    own, calls = ops.linear, []
    monkeypatch.setattr(ops, "linear", lambda *a: (calls.append(own(*a)), calls[-1])[1])
    x, w, b = (torch.randn(s, device=DEV).to(dtype).requires_grad_() for s in ((rows, k), (n, k), (n,)))
    got = ops._LinearFn.apply(x, w, b if bias else None)
    assert (len(calls) == 1 and calls[0] is not None) == kernel and got.requires_grad
    want = x.double() @ w.double().t() + (b.double() if bias else 0)
    # half a step of the type, and an fp32 rounding for each of the products' sums
    mag = x.double().abs() @ w.double().abs().t() + b.double().abs()
    assert bool(((got.double() - want).abs() <= torch.finfo(dtype).eps / 2 * want.abs() + (k + 2) * 2.0 ** -24 * mag).all())
    strided = torch.randn(rows, 2, k, device=DEV, dtype=dtype)[:, 0]
    assert torch.equal(ops._LinearFn.apply(strided, w, None), F.linear(strided, w)) or rows == 1
