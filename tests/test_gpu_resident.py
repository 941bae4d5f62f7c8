"""Whole sweeps in one resident launch each, whose workgroups exchange halos
between chunks of steps: probe series and field snapshots bitwise equal to the
fp32 oracle, and gradients within rel 1e-4 of its
fp64 adjoint, for one tile, halos on every side, halos that reach past the
next tile, odd chunks and remainders, every rows-per-thread variant, and while
another stream keeps the device busy."""
import numpy as np
import pytest
import torch

import oracle.c_oracle as co
from tests.helpers import rel, small_problem
from wavetorch_amd._loop import LoopConfig, Plan, WaveLoop

pytestmark = pytest.mark.gpu

TUNINGS = {
    "one-tile": dict(strips=1, tcols=1, tblock=9, nt=1024, cpt=12),
    "3x3": dict(strips=3, tcols=3, tblock=7, nt=1024, cpt=4),
    "rows-only": dict(strips=5, tcols=1, tblock=4, nt=1024, cpt=8),
    "past-neighbours": dict(strips=8, tcols=6, tblock=12, nt=1024, cpt=6),
    "step-by-step": dict(strips=2, tcols=4, tblock=1, nt=1024, cpt=10),
    "512": dict(strips=2, tcols=2, tblock=37, nt=512, cpt=16),
}
# linear cell: adjoint tilings of the same kinds
A_TUNINGS = {
    "one-tile": dict(a_strips=1, a_tcols=1, a_tblock=9, a_nt=1024, a_cpt=10),
    "3x3": dict(a_strips=3, a_tcols=3, a_tblock=7, a_nt=1024, a_cpt=6),
    "rows-only": dict(a_strips=5, a_tcols=1, a_tblock=4, a_nt=1024, a_cpt=8),
    "past-neighbours": dict(a_strips=8, a_tcols=6, a_tblock=12, a_nt=1024, a_cpt=4),
    "step-by-step": dict(a_strips=2, a_tcols=4, a_tblock=1, a_nt=1024, a_cpt=10),
    "512": dict(a_strips=2, a_tcols=2, a_tblock=37, a_nt=512, a_cpt=16),
}
ADJ = dict(a_strips=2, a_tcols=2, a_tblock=5, a_nt=1024, a_cpt=4)
CASES = {"linear": (1.0, {}), "h": (1.4283556979968262, {}),
         "nonlinear": (1.0, dict(sat_b0=0.5, sat_uth=0.1 ** 0.5, c_nl=0.05, clamp=(0.55, 0.9)))}


def _setup(case, B=2):
    h, nl = CASES[case]
    p = small_problem(Nx=43, Ny=38, T=75, B=B, amp=0.3, seed=12)
    p["h"], p["dt"] = h, 0.6 * h
    p["rho"] = np.random.default_rng(3).uniform(0, 1, (p["Nx"], p["Ny"])).astype(np.float32)
    cfg = LoopConfig(Nx=p["Nx"], Ny=p["Ny"], dt=p["dt"], h=h, src_px=tuple(map(tuple, p["src"])),
                     taps=tuple(map(tuple, p["taps"])), sat_b0=nl.get("sat_b0", 0.0),
                     sat_uth=nl.get("sat_uth", 0.0), c_nl=nl.get("c_nl", 0.0),
                     c_clamp=nl.get("clamp"))
    return p, cfg, h, nl, dict(nl, rho=p["rho"]) if nl else None


@pytest.mark.parametrize("case", sorted(CASES))
@pytest.mark.parametrize("tun", sorted(TUNINGS))
def test_resident_forward(tun, case, cuda):
    p, cfg, h, nl, onl = _setup(case)
    plan = Plan(cfg, p["B"], p["T"], 1.0, cuda, {**TUNINGS[tun], **(ADJ if nl else A_TUNINGS[tun]),
                                                 "ck_every": p["T"]})
    print("case", tun, case, plan.tuning, flush=True)
    assert not plan.tuning["plain"] and plan.tuning["tblock"] == TUNINGS[tun]["tblock"]
    t = {k: torch.from_numpy(p[k]).to(cuda).requires_grad_(k != "b") for k in
         ("x", "c", "b", "rho")}
    rho = t["rho"] if nl else None
    yo, fo = co.forward(p["b"], p["c"], p["x"], p["dt"], h, p["src"], p["taps"], nl=onl,
                        fields=True)
    with torch.no_grad():
        y = WaveLoop.apply(t["x"], t["c"], t["b"], rho, plan, False, 1)
        f = WaveLoop.apply(t["x"], t["c"], t["b"], rho, plan, True, 1)
    assert np.array_equal(y.cpu().numpy(), yo)
    assert np.array_equal(f.cpu().numpy(), fo)
    y = WaveLoop.apply(t["x"], t["c"], t["b"], rho, plan, False, 1)
    assert np.array_equal(y.detach().cpu().numpy(), yo)
    w = np.random.default_rng(5).standard_normal(y.shape).astype(np.float32)
    (y * torch.from_numpy(w).to(cuda)).sum().backward()
    g = co.adjoint(p["b"], p["c"], p["x"], p["dt"], h, p["src"], p["taps"], ybar=w, nl=onl)
    assert rel(t["c"].grad.cpu().numpy(), g["gc"]) < 1e-4
    assert rel(t["x"].grad.cpu().numpy(), g["gx"]) < 1e-4


def test_resident_forward_beside_other_work(cuda):
    """Two streams with a workgroup for most CUs each, behind and beside a
    matrix product: workgroups start late and in parts."""
    p, cfg, h, nl, onl = _setup("linear", B=5)
    plans = [Plan(cfg, 5, p["T"], 1.0, cuda, dict(TUNINGS["past-neighbours"], ck_every=p["T"]))
             for _ in range(2)]
    t = [torch.from_numpy(p[k]).to(cuda) for k in ("x", "c", "b")]
    yo, _ = co.forward(p["b"], p["c"], p["x"], p["dt"], h, p["src"], p["taps"])
    m = torch.randn(4096, 4096, device=cuda)
    streams = [torch.cuda.Stream() for _ in plans]
    torch.cuda.synchronize()
    busy = m @ m
    out = []
    with torch.no_grad():
        for _ in range(4):
            for plan, s in zip(plans, streams):
                with torch.cuda.stream(s):
                    out.append(WaveLoop.apply(*t, None, plan, False, 1))
    torch.cuda.synchronize()
    assert torch.isfinite(busy).all()
    for y in out:
        assert np.array_equal(y.cpu().numpy(), yo)
