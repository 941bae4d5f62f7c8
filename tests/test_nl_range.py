"""The nonlinear cell outside the range of the blocked forward's quotients
(thresholds whose reciprocal is not a normal number, time steps near the end
of float32): the per-step kernels with the general division run there, probe
series bitwise equal to the fp32 oracle, NaN and infinities included."""
import numpy as np
import pytest
import torch

import oracle.c_oracle as co
from wavetorch_amd._loop import LoopConfig, Plan, WaveLoop, resolve, suggest

# uth, dt, b0 * dt and whether the blocked kernels take it
RANGE = [(0.3, 0.6, 0.5, True), (-0.3, 0.6, 0.5, True), (1e-20, 0.6, 0.5, True),
         (1e30, 0.6, 0.5, True), (0.3, 2e-17, 0.5, True), (0.3, 1e15, 0.5, True),
         (0.0, 0.6, 0.5, False), (1e-40, 0.6, 0.5, False), (1e-30, 0.6, 0.5, False),
         (3e38, 0.6, 0.5, False), (0.3, 9e-20, 0.5, False), (0.3, 1e19, 0.5, False),
         (0.3, 0.6, 1e20, False)]


def _cfg(uth, dt, b0):
    h = 1.0 if dt == 0.6 else dt / 0.6
    return LoopConfig(Nx=30, Ny=27, dt=dt, h=h, src_px=((7, 13, 0),),
                      taps=((20, 9, 0), (21, 15, 1)), sat_b0=b0 / dt, sat_uth=uth)


@pytest.mark.parametrize("uth,dt,b0,blocked", RANGE)
def test_plan(uth, dt, b0, blocked):
    cfg = _cfg(uth, dt, b0)
    for tun in (None, {"ck_every": 40}, suggest(cfg, 2, 40, 1.0, 40, 0)):
        assert resolve(cfg, 2, 40, 1.0, tun)[0]["plain"] == (0 if blocked else 1)
    if not blocked:  # the flat kernels divide: they take it at h = 1
        got = resolve(cfg, 2, 40, 1.0, {"kind": 1})[0]
        assert got["plain"] == (0 if cfg.h == 1.0 else 1)


@pytest.mark.gpu
@pytest.mark.parametrize("uth,dt,b0,blocked", RANGE)
def test_forward_equals_oracle(uth, dt, b0, blocked, cuda):
    cfg = _cfg(uth, dt, b0)
    print("case", cfg, flush=True)
    rng = np.random.default_rng(2)
    f = lambda a: a.astype(np.float32)
    x, c = f(0.3 * rng.standard_normal((2, 40))), f(rng.uniform(0.5, 1.0, (30, 27)))
    b, rho = f(rng.uniform(0, 0.1, (30, 27)) / dt), f(rng.uniform(0, 1, (30, 27)))
    yo, _ = co.forward(b, c, x, cfg.dt, cfg.h, cfg.src_px, cfg.taps,
                       nl=dict(sat_b0=cfg.sat_b0, sat_uth=uth, c_nl=0.0, rho=rho))
    plan = Plan(cfg, 2, 40, 1.0, cuda)
    with torch.no_grad():
        y = WaveLoop.apply(*(torch.from_numpy(a).to(cuda) for a in (x, c, b, rho)), plan, False, 1)
    assert np.array_equal(y.cpu().numpy(), yo, equal_nan=True)
