"""Temporally blocked float64 loop of the linear cell: forward bitwise equal
to the fp64 oracle (probe series and field snapshots), gradients within 1e-10
of its fp64 adjoint, for tilings with halos on every side, rows left over by
the rows per thread, one-step remainders, grid steps other than 1, a line
source across tiles and a clamped speed."""
import numpy as np
import pytest
import torch

import oracle.c_oracle as co
from tests.helpers import rel, small_problem
from wavetorch_amd._loop import LoopConfig, Plan, WaveLoop

pytestmark = pytest.mark.gpu

TUNINGS = {
    "auto": {},
    "R4": dict(strips=3, tcols=3, tblock=6, cpt=4, a_tblock=5, a_cpt=4, nt=1024),
    "R6-5": dict(strips=2, tcols=1, tblock=9, cpt=6, a_strips=1, a_tcols=2, a_tblock=8, a_cpt=5,
                 nt=1024),
    "R8": dict(strips=1, tcols=1, tblock=37, cpt=8, a_strips=4, a_tcols=3, a_tblock=2, a_cpt=5,
               nt=1024),
}


def _case(h, clamp, line):
    p = small_problem(Nx=43, Ny=38, T=73, amp=0.3, seed=4)
    p["h"], p["dt"] = h, 0.7 * h
    for k in ("b", "c", "x"):
        p[k] = p[k].astype(np.float64)
    if line:
        p["src"] = [[9, y, 0] for y in range(8, 30)]
    cfg = LoopConfig(Nx=43, Ny=38, dt=p["dt"], h=h, src_px=tuple(map(tuple, p["src"])),
                     taps=tuple(map(tuple, p["taps"])), c_clamp=(0.6, 0.9) if clamp else None)
    return p, cfg


@pytest.mark.parametrize("h,clamp,line", [(1.0, False, False), (1.4283556979968262, False, True),
                                          (1.0, True, True)])
@pytest.mark.parametrize("tun", sorted(TUNINGS))
def test_blocked_f64(tun, h, clamp, line, cuda):
    p, cfg = _case(h, clamp, line)
    plan = Plan(cfg, p["B"], p["T"], 1.0, cuda, TUNINGS[tun])
    print("case", tun, h, clamp, line, flush=True)
    assert plan.bytes_rec_f64() is not None
    x, c, b = (torch.from_numpy(p[k]).to(cuda).requires_grad_(k != "b") for k in ("x", "c", "b"))
    y = WaveLoop.apply(x, c, b, None, plan, False, 1)
    w = np.random.default_rng(6).standard_normal(y.shape)
    (y * torch.from_numpy(w).to(cuda)).sum().backward()
    nl = dict(rho=np.zeros_like(p["c"]), clamp=(0.6, 0.9)) if clamp else None
    yo, fo = co.forward(p["b"], p["c"], p["x"], p["dt"], h, p["src"], p["taps"], nl=nl,
                        fields=True, dtype=np.float64)
    assert np.array_equal(y.detach().cpu().numpy(), yo)
    g = co.adjoint(p["b"], p["c"], p["x"], p["dt"], h, p["src"], p["taps"], ybar=w, nl=nl)
    assert rel(c.grad.cpu().numpy(), g["gc"]) < 1e-10
    assert rel(x.grad.cpu().numpy(), g["gx"]) < 1e-10
    with torch.no_grad():
        f = WaveLoop.apply(x, c, b, None, plan, True, 1)
    assert np.array_equal(f.cpu().numpy(), fo)
