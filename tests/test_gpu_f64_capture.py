"""A float64 plan is whole when it is made: a call that runs per step (field
gradients) may be followed by a captured one of the same shape that runs
blocked, without any other call between them."""
import pytest
import torch

from tests.test_f64_plan import _model

pytestmark = pytest.mark.gpu


def test_capture_after_a_call_that_runs_per_step(cuda):
    model = _model(torch.float64).to(cuda)
    x = torch.randn(2, 90, dtype=torch.float64, device=cuda)
    model(x, output_fields=True).sum().backward()
    torch.cuda.synchronize()
    graph, y = torch.cuda.CUDAGraph(), None
    with torch.no_grad():
        model.cell.geom.c  # the geometry's own first call
        with torch.cuda.graph(graph):
            y = model(x)
    ref = None
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        with torch.no_grad():
            ref = model(x)
        assert torch.equal(y, ref)
    assert float(ref.abs().max()) > 0
