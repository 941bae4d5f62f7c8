"""A search for a tuning runs the checkpoint interval that the tuned model's
calls take: left open, the one that the model chooses; given, the given one."""
import pytest
import torch

from wavetorch_amd import (WaveCell, WaveGeometryFreeForm, WaveIntensityProbe, WaveRNN,
                           WaveSource, autotune)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("native", [False, True])
@pytest.mark.parametrize("every", [None, 50])
def test_interval_of_a_tuned_model(every, native, cuda, monkeypatch):
    stored = {}
    monkeypatch.setattr(autotune, "_load", dict)
    monkeypatch.setattr(autotune, "_store", stored.update)
    geom = WaveGeometryFreeForm((60, 52), 1.0, c0=1.0, c1=0.5, abs_N=8, abs_sig=1.0, abs_p=2,
                                rho="half")
    model = WaveRNN(WaveCell(0.7, geom), WaveSource(16, 26),
                    [WaveIntensityProbe(44, 20)]).to(cuda)
    model.checkpoint_every = every
    x = torch.randn(3, 150, device=cuda)
    if native:
        best, _ = autotune.tune_native(model, x, reps=1, budget_s=1e-3)
    else:
        best = autotune.tune(model, x, steps=1, reps=1, budget_s=0.0)
    K = every or 150
    assert model._checkpoint_every == every
    run = model.plan(3, 150, x.device).tuning
    assert run["ck_every"] == K
    assert all(run[k] == v for k, v in best.items())
    assert list(stored) == [autotune.key(60, 52, 3, 150, K)]
