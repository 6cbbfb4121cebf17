"""CPU: the model's layers under torch's tracers.

RMSNorm, SwiGLU and the projections try their kernels first; a symbolic trace or
a script of them has to come out as the torch expressions."""
import pytest
import torch

from kerneldev_amd import _lib
from kerneldev_amd.gpt import Projection, RMSNorm, SwiGLU

LAYERS = [RMSNorm, lambda: SwiGLU(64, 128), lambda: Projection(64, 72)]


@pytest.mark.parametrize("make", LAYERS, ids=["norm", "swiglu", "projection"])
@pytest.mark.parametrize("how", ["fx", "script", "trace", "export"])
def test_layers_under_tracers(make, how):
    m, x = make(), torch.randn(2, 6, 64)
    if how == "fx":
        t = torch.fx.symbolic_trace(m)
        assert not any("native" in str(n.target) for n in t.graph.nodes)
    elif how == "script":
        t = torch.jit.script(m)
    elif how == "trace":
        t = torch.jit.trace(m, x)
    else:
        t = torch.export.export(m, (x,)).module()
    assert torch.equal(t(x), m(x))


def test_max_spans_on_the_cpu_needs_no_library(monkeypatch):
    from kerneldev_amd.span_head import max_spans

    monkeypatch.setattr(_lib, "native", lambda: pytest.fail("the GPU route was asked for"))
    assert max_spans(torch.tensor([[3, 3, 1], [3, 1, 1]])) == 2
