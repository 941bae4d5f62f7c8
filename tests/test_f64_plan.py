"""The plans of float64 models: no tiling of the float32 kernels' model reaches
them, so that the double-precision model chooses."""
import pytest
import torch

from wavetorch_amd import (WaveCell, WaveGeometryFreeForm, WaveIntensityProbe, WaveRNN,
                           WaveSource, rnn)


def _model(dtype):
    geom = WaveGeometryFreeForm((40, 34), 1.0, c0=1.0, c1=0.5, abs_N=6, abs_sig=1.0, abs_p=2,
                                rho="half")
    return WaveRNN(WaveCell(0.6, geom), WaveSource(10, 17),
                   [WaveIntensityProbe(30, 12)]).to(dtype)


@pytest.mark.parametrize("tuning", [None, dict(strips=2, tcols=2, tblock=8, nt=1024, cpt=6)])
def test_tiling_of_a_float64_plan(tuning, monkeypatch):
    asked = []

    class FakePlan:
        def __init__(self, cfg, B, T, cmax, device, tuning=None, group=0, waiting=None):
            asked.append(dict(tuning or {}))

        def bytes_rec_f64(self):
            return None

    monkeypatch.setattr(rnn, "Plan", FakePlan)
    model = _model(torch.float64)
    model.tuning = tuning
    assert model.cell.geom.b.dtype == torch.float64
    model.plan(2, 300, torch.device("cpu"), lean=True)
    assert asked == [dict(tuning or {}, ck_every=64)]
    # float32 of the same size: the float model's tiling unless one is given
    f32 = _model(torch.float32)
    f32.tuning = tuning
    f32.plan(2, 300, torch.device("cpu"), lean=True)
    assert asked[1].get("strips", 0) > 0
