"""The launch-time model's tunings (``wt_plan_suggest``) on the host: every one
is a plan the library accepts, none is cheaper in workgroups than the chip
needs, and the adjoint keeps the default plan's depth at h = 1; on the device
a model's default call takes it and equals the library's default plan bit for
bit, forward and gradient."""
import math

import numpy as np
import pytest
import torch

from wavetorch_amd._loop import LoopConfig, Plan, WaveLoop, resolve, suggest

SHAPES = [(3, 3, 1, 5), (7, 300, 2, 40), (60, 57, 1, 300), (64, 64, 64, 65), (141, 123, 24, 1501),
          (500, 380, 1, 800), (1024, 1024, 1, 4000), (2000, 2000, 1, 100), (150, 150, 64, 3000)]


def _cfg(Nx, Ny, nl=False, h=1.0):
    return LoopConfig(Nx=Nx, Ny=Ny, dt=0.6 * h, h=h, src_px=((Nx // 4, Ny // 2, 0),),
                      taps=((Nx // 4 + Nx // 8, Ny // 2, 1),), sat_b0=0.5 if nl else 0.0,
                      sat_uth=0.3)


@pytest.mark.parametrize("nl", [False, True])
@pytest.mark.parametrize("Nx,Ny,B,T", SHAPES)
def test_suggested_tunings_are_plans(Nx, Ny, B, T, nl):
    cfg = _cfg(Nx, Ny, nl)
    for K, group in ((T, 64), (64, 0)):
        t = suggest(cfg, B, T, 1.0, K, group)
        got, _, _ = resolve(cfg, B, T, 1.0, t)
        assert got["plain"] == 0 and got["ck_every"] == min(K, T)
        assert {k: got[k] for k in t} == t  # taken as it is
        default, _, _ = resolve(cfg, B, T, 1.0, {"ck_every": group or K})
        assert t["a_tblock"] == default["a_tblock"]


def test_no_block_holds_it():
    """Several sources on one pixel: the per-step kernels, as by default."""
    cfg = LoopConfig(Nx=50, Ny=50, dt=0.6, h=1.0, src_px=((9, 9, 0), (9, 9, 1)),
                     taps=((20, 20, 1),))
    assert suggest(cfg, 2, 100, 1.0, 100, 64) == {"ck_every": 100}
    with pytest.raises(ValueError):
        suggest(_cfg(50, 50), 2, 100, 2.0, 100)  # CFL


@pytest.mark.gpu
@pytest.mark.parametrize("nl", [False, True])
@pytest.mark.parametrize("Nx,Ny,B,T", [(60, 57, 1, 130), (64, 64, 40, 65), (141, 123, 24, 100),
                                       (200, 190, 3, 90)])
def test_suggested_plan_equals_default(Nx, Ny, B, T, nl, cuda):
    cfg = _cfg(Nx, Ny, nl)
    rng = np.random.default_rng(1)
    src = {"x": rng.standard_normal((B, T)), "c": rng.uniform(0.5, 1.0, (Nx, Ny)),
           "b": np.zeros((Nx, Ny)), "rho": rng.uniform(0, 1, (Nx, Ny)),
           "w": rng.standard_normal((B, T, 1))}
    src = {k: torch.from_numpy(v.astype(np.float32)).to(cuda) for k, v in src.items()}
    out = []
    for plan in (Plan(cfg, B, T, 1.0, cuda, {"ck_every": 64}),
                 Plan(cfg, B, T, 1.0, cuda, suggest(cfg, B, T, 1.0, T, 64), 64)):
        print("case", plan.tuning, flush=True)
        x, c, rho = (src[k].clone().requires_grad_(True) for k in ("x", "c", "rho"))
        y = WaveLoop.apply(x, c, src["b"], rho if nl else None, plan, False, 1)
        (y * src["w"]).sum().backward()
        out.append([y.detach(), c.grad, x.grad] + ([rho.grad] if nl else []))
    assert math.isfinite(float(out[0][1].abs().sum())) and float(out[0][0].abs().max()) > 0
    for a, b in zip(*out):
        assert torch.equal(a, b)
