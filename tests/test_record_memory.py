"""Whole records and the memory they take: one per model at a time, whatever
the lengths, and calls whose record does not fit run with checkpoints."""
import weakref

import pytest
import torch

from tests.helpers import rel
from wavetorch_amd import (WaveCell, WaveGeometryFreeForm, WaveIntensityProbe, WaveRNN,
                           WaveSource, rnn)

pytestmark = pytest.mark.gpu


def _model(cuda, N=60):
    geom = WaveGeometryFreeForm((N, N - 8), 1.0, c0=1.0, c1=0.5, abs_N=8, abs_sig=1.0, abs_p=2,
                                rho="half")
    return WaveRNN(WaveCell(0.7, geom), WaveSource(N // 4, N // 2),
                   [WaveIntensityProbe(N - 16, N // 3), WaveIntensityProbe(N - 16, N // 2)]).to(cuda)


def _x(cuda, B, T):
    n = torch.arange(float(T))
    return torch.stack([torch.sin(0.3 * n + k) * torch.exp(-((n - 60) / 25) ** 2)
                        for k in range(B)]).to(cuda)


def _grad(model, y):
    model.zero_grad(set_to_none=True)
    y.sum().backward()
    return model.cell.geom.rho.grad.cpu().numpy()


class _Limit:
    """At most `nbytes` more device memory for torch than it holds now."""

    def __init__(self, cuda, nbytes):
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        total = torch.cuda.get_device_properties(cuda).total_memory
        self.fraction = (torch.cuda.memory_reserved(cuda) + nbytes) / total

    def __enter__(self):
        torch.cuda.set_per_process_memory_fraction(self.fraction)

    def __exit__(self, *exc):
        torch.cuda.set_per_process_memory_fraction(1.0)


def test_one_record_at_a_time_over_lengths(cuda):
    model = _model(cuda)
    x1, x2 = _x(cuda, 3, 150), _x(cuda, 2, 130)
    alone = _grad(model, model(x2))
    y1 = model(x1)
    y2 = model(x2)  # another length while y1's record waits
    model._plans.clear()
    y3 = model(x1)  # and with the waiting record's plan gone
    used = sorted((p.B, p.T, p.tuning["ck_every"]) for p in model._plans.values())
    assert (3, 150, 64) in used
    g1 = _grad(model, y1)
    assert rel(_grad(model, y2), alone) < 1e-5 and rel(_grad(model, y3), g1) < 1e-5
    model._plans.clear()
    y2 = model(x2)  # nothing waits any more
    y1 = model(x1)
    assert {(2, 130): 130, (3, 150): 64}.items() <= \
        {(p.B, p.T): p.tuning["ck_every"] for p in model._plans.values()}.items()
    assert torch.equal(y1, y3)


def test_retry_holds_nothing_of_the_failed_call(cuda, monkeypatch):
    model = _model(cuda)
    held = []

    class Loop:
        @staticmethod
        def apply(*args):
            if not held:
                saved = torch.empty(1 << 20, device=cuda)
                held.append(weakref.ref(saved))
                raise torch.cuda.OutOfMemoryError("out of memory")
            assert held[0]() is None
            return rnn_loop.apply(*args)

    rnn_loop = rnn.WaveLoop
    monkeypatch.setattr(rnn, "WaveLoop", Loop)
    assert torch.isfinite(model(_x(cuda, 2, 150))).all()


def test_record_that_leaves_no_room_for_the_backward(cuda):
    """The forward's own buffers would fit beside the record, the backward's
    would not: the call runs with checkpoints."""
    model, x = _model(cuda, 150), _x(cuda, 64, 150)
    p = model.plan(64, 150, x.device)
    assert p.tuning["ck_every"] == 150
    room = p.saved_bytes + p.temp_bytes_nograd + (12 << 20)
    assert room < p.saved_bytes + p.temp_bytes
    ref = _grad(model, model(x))
    with _Limit(cuda, room):
        y = model(x)
        g = _grad(model, y)
    assert rel(g, ref) < 1e-5
