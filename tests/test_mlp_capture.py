"""The model's MLP stays a module that scripting, symbolic tracing, compilation and export with a variable batch take."""
import pytest
import torch

from speed3r_amd.model.pi3_sparse_like import Mlp


def _mlp():
    torch.manual_seed(0)
    return Mlp(16, 32)


@pytest.mark.parametrize("grad", [True, False])
def test_scripting(grad):
    m, x = _mlp(), torch.randn(3, 5, 16)
    with torch.set_grad_enabled(grad):
        assert torch.equal(torch.jit.script(m)(x), m(x))


@pytest.mark.parametrize("grad", [True, False])
def test_symbolic_tracing(grad):
    m, x = _mlp(), torch.randn(3, 5, 16)
    with torch.set_grad_enabled(grad):
        assert torch.equal(torch.fx.symbolic_trace(m)(x), m(x))


@pytest.mark.parametrize("grad", [True, False])
def test_export_with_a_variable_batch(grad):
    m, x = _mlp(), torch.randn(3, 5, 16)
    with torch.set_grad_enabled(grad):
        program = torch.export.export(m, (x,), dynamic_shapes=({0: torch.export.Dim("b", min=2, max=100000)},))
        more = torch.randn(2000, 5, 16)
        assert torch.allclose(program.module()(more), m(more))


@pytest.mark.parametrize("grad", [True, False])
def test_one_compilation_for_few_and_many_rows(grad):
    torch._dynamo.reset()
    compiled = []

    def backend(graph, inputs):
        compiled.append(1)
        return graph

    m = torch.compile(_mlp(), backend=backend, fullgraph=True, dynamic=True)
    with torch.set_grad_enabled(grad):
        for rows in (3, 100, 3000):
            m(torch.randn(rows, 5, 16))
    assert len(compiled) == 1
