"""A search for a tuning runs the checkpoint interval (and the span of its
gradient sums) that the tuned model's calls take: left open, the one that the
model chooses; given, the given one."""
import pytest
import torch

from wavetorch_amd import (WaveCell, WaveGeometryFreeForm, WaveIntensityProbe, WaveRNN,
                           WaveSource, _lib, autotune)

pytestmark = pytest.mark.gpu


class _Spy:
    """The library, noting the interval and span that a native search gets."""

    def __init__(self, lib, seen):
        self._lib, self._seen = lib, seen

    def __getattr__(self, name):
        f = getattr(self._lib, name)
        if not name.startswith("wt_autotune"):
            return f

        def call(*a):
            self._seen.add((a[4]._obj.ck_every, a[5] if name.endswith("group") else 0))
            return f(*a)
        return call


def _model(cuda, shape=(60, 52)):
    geom = WaveGeometryFreeForm(shape, 1.0, c0=1.0, c1=0.5, abs_N=8, abs_sig=1.0, abs_p=2,
                                rho="half")
    return WaveRNN(WaveCell(0.7, geom), WaveSource(16, 26), [WaveIntensityProbe(44, 20)]).to(cuda)


@pytest.mark.parametrize("native", [False, True])
@pytest.mark.parametrize("every", [None, 50])
def test_interval_of_a_tuned_model(every, native, cuda, monkeypatch):
    stored, seen = {}, set()
    monkeypatch.setattr(autotune, "_load", lambda: dict(stored))
    monkeypatch.setattr(autotune, "_store", stored.update)
    model = _model(cuda)
    model.checkpoint_every = every
    x = torch.randn(3, 150, device=cuda)
    if native:
        lib = _lib.lib()
        monkeypatch.setattr(_lib, "lib", lambda: _Spy(lib, seen))
        best, _ = autotune.tune_native(model, x, reps=1, budget_s=1e-3)
        monkeypatch.setattr(_lib, "lib", lambda: lib)
    else:
        plan = model.plan

        def spy(*a, **kw):
            p = plan(*a, **kw)
            seen.add((p.tuning["ck_every"], p.group))
            return p
        monkeypatch.setattr(model, "plan", spy)
        best = autotune.tune(model, x, steps=1, reps=1, budget_s=0.0)
    assert model._checkpoint_every == every
    run = model.plan(3, 150, x.device)
    assert seen == {(run.tuning["ck_every"], run.group)} == {(every, 0) if every else (150, 64)}
    assert all(run.tuning[k] == v for k, v in best.items())
    assert list(stored) == [autotune.key(60, 52, 3, 150, every or "auto", "gfx950")]
    assert autotune.lookup(60, 52, 3, 150) == (None if every else best)


@pytest.mark.parametrize("native", [False, True])
def test_search_after_a_tuning_that_does_not_fit(native, cuda, monkeypatch):
    """The tuning of another shape on the model, which no block holds here."""
    monkeypatch.setattr(autotune, "_load", dict)
    monkeypatch.setattr(autotune, "_store", lambda d: None)
    model = _model(cuda, (150, 120))
    model.tuning = dict(strips=1, tcols=1, tblock=8, nt=1024, cpt=4)
    x = torch.randn(2, 100, device=cuda)
    with pytest.raises(RuntimeError):
        model(x)
    if native:
        best, _ = autotune.tune_native(model, x, reps=1, budget_s=1e-3)
    else:
        best = autotune.tune(model, x, steps=1, reps=1, budget_s=0.0)
    assert model.tuning == best and torch.isfinite(model(x)).all()
