"""Whole records and the memory they take: one per model at a time whatever the
lengths, and calls whose record does not fit run with checkpoints."""
import weakref

import numpy as np
import pytest
import torch

from tests.helpers import rel
from wavetorch_amd import (WaveCell, WaveGeometryFreeForm, WaveIntensityProbe, WaveRNN,
                           WaveSource, rnn)
from wavetorch_amd._loop import LoopConfig
from wavetorch_amd.batch import Instance, InstanceBatch

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


def test_batch_whose_record_does_not_fit(cuda):
    rng = np.random.default_rng(3)
    cfg = LoopConfig(Nx=200, Ny=200, dt=0.7, h=1.0, src_px=((20, 100, 0),), taps=((150, 90, 1),))
    insts = [Instance(cfg, torch.zeros(200, 200), T, 1.0) for T in (1500, 1200, 900, 600)]
    f = lambda a: torch.from_numpy(a.astype(np.float32)).to(cuda)
    cs = [f(rng.uniform(0.5, 1.0, (200, 200))) for _ in insts]
    xs = [f(rng.standard_normal(i.length)) for i in insts]
    ys = [f(rng.standard_normal((i.length, 1))) for i in insts]

    def run(bt):
        bt.set_inputs(cs, xs, ys)
        bt.fwd_adj()
        return [t.clone() for o in bt.outputs() for t in o]

    ref = run(InstanceBatch(insts, cuda, checkpoint_every=64))
    open_ = InstanceBatch(insts, cuda)
    assert open_.tuning[0]["ck_every"] == 1500
    del open_
    with _Limit(cuda, 400 << 20):  # the record takes 675 MB
        bt = InstanceBatch(insts, cuda)
        assert bt.tuning[0]["ck_every"] == 64
        out = run(bt)
    assert all(torch.equal(a, b) for a, b in zip(ref, out))
    with _Limit(cuda, 400 << 20):  # what the caller asked for is not changed
        with pytest.raises(torch.cuda.OutOfMemoryError):
            InstanceBatch(insts, cuda, checkpoint_every=1500)


def test_a_given_interval_needs_no_room_for_a_backward(cuda):
    """A forward at an interval that the caller named runs in the memory it
    needs itself, as there is nothing to fall back to."""
    model, x = _model(cuda, 150), _x(cuda, 64, 150)
    model.checkpoint_every = 150
    p = model.plan(64, 150, x.device)
    ref = model(x).detach()
    with _Limit(cuda, p.saved_bytes + p.temp_bytes_nograd + (12 << 20)):
        y = model(x)
    assert torch.equal(y, ref)
