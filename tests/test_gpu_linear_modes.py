"""GPU: modes that are to see the torch operations see the products of the linear layers too, forward and backward."""
import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode
from torch.utils.flop_counter import FlopCounterMode

from speed3r_amd.model.pi3_sparse_like import Mlp
from speed3r_amd.sparse_attn import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
ROWS = 4096   # enough for the kernels of inference and of training


def _mlp(requires_grad=False):
    torch.manual_seed(0)
    m = Mlp(128, 256).to(DEV, torch.bfloat16).requires_grad_(requires_grad)
    return m, torch.randn(1, ROWS, 128, device=DEV, dtype=torch.bfloat16)


def test_a_traced_module_holds_its_products():
    m, x = _mlp()
    with torch.no_grad():
        graph = make_fx(m, tracing_mode="real")(x)
        other = torch.randn_like(x)
        want = m.fc2(torch.nn.functional.gelu(m.fc1(other)))
        assert torch.equal(graph(other), want)


def test_flops_of_forward_and_backward_are_counted():
    m, x = _mlp()
    flops = 2 * 2 * ROWS * 128 * 256
    with torch.no_grad(), FlopCounterMode(display=False) as count:
        m(x)
    assert count.get_total_flops() == flops
    w, b = (torch.randn(s, device=DEV, dtype=torch.bfloat16, requires_grad=True) for s in ((256, 1024), (256,)))
    out = ops.linear_autograd(torch.randn(ROWS, 1024, device=DEV, dtype=torch.bfloat16, requires_grad=True), w, b)
    with FlopCounterMode(display=False) as count:   # (a backward alone)
        out.backward(torch.randn_like(out))
    assert count.get_total_flops() == 2 * 2 * ROWS * 256 * 1024


def test_function_modes_see_the_products_and_a_device_context_is_none():
    class Seen(TorchFunctionMode):
        names = []

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.names.append(getattr(func, "__name__", ""))
            return func(*args, **(kwargs or {}))

    m, x = _mlp()
    with torch.no_grad(), Seen():
        m(x)
    assert Seen.names.count("linear") == 2
    with torch.device(DEV):
        assert ops.ordinary(x)
