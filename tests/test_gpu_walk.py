"""How resident sweeps start and wait: one launch per sweep; the same bits when
only every n-th workgroup is started and the others' tiles are taken over,
forward and adjoint, float32 and float64, odd chunks and remainders; and NaN
for what a sweep has not computed when its waits are given up."""
import ctypes

import numpy as np
import pytest
import torch

import oracle.c_oracle as co
from tests.test_gpu_resident import A_TUNINGS, ADJ, TUNINGS, _setup
from wavetorch_amd import _lib
from wavetorch_amd._loop import Plan, WaveLoop

pytestmark = pytest.mark.gpu

TILED = sorted(t for t in TUNINGS if t != "one-tile")


def _plan(case, tun, cuda, rows=4):
    """A plan of 4 rows per thread (the adjoint: `rows`)."""
    p, cfg, h, nl, onl = _setup(case)
    tuning = {**TUNINGS[tun], **(ADJ if nl else A_TUNINGS[tun]), "ck_every": p["T"],
              "nt": 1024, "cpt": 4, "a_nt": 1024, "a_cpt": 4 if nl else rows}
    return p, nl, Plan(cfg, p["B"], p["T"], 1.0, cuda, tuning)


def _walk(plan, every, give_up=0):
    _lib.check(_lib.lib().wt_plan_walk(plan.handle, every, give_up), "wt_plan_walk")


def _run(p, nl, plan, cuda, dtype=torch.float32):
    """Probe series and fields without gradients, probe series with, and the
    gradients of c and x (and rho)."""
    t = {k: torch.from_numpy(p[k]).to(cuda, dtype).requires_grad_(k != "b")
         for k in ("x", "c", "b", "rho")}
    rho = t["rho"] if nl else None
    out = []
    with torch.no_grad():
        for fields in (False, True):
            out.append(WaveLoop.apply(t["x"], t["c"], t["b"], rho, plan, fields, 1))
    y = WaveLoop.apply(t["x"], t["c"], t["b"], rho, plan, False, 1)
    w = np.random.default_rng(5).standard_normal(y.shape)
    (y * torch.from_numpy(w).to(cuda, dtype)).sum().backward()
    torch.cuda.synchronize()
    return out + [y.detach(), t["c"].grad, t["x"].grad] + ([t["rho"].grad] if nl else [])


@pytest.mark.parametrize("tun", sorted(TUNINGS))
@pytest.mark.parametrize("case", ["linear", "nonlinear"])
def test_one_launch_per_sweep(case, tun, cuda):
    p, nl, plan = _plan(case, tun, cuda)
    L = _lib.lib()
    ms, n, cells = (ctypes.c_double * 3)(), (ctypes.c_int64 * 3)(), (ctypes.c_int64 * 3)()
    _lib.check(L.wt_profile(1), "wt_profile")
    try:
        _run(p, nl, plan, cuda)
        _lib.check(L.wt_profile_read(ms, n, cells), "wt_profile_read")
    finally:
        L.wt_profile(0)
    assert n[0] == 3 and n[1] == 0  # two forwards without gradients, one with
    assert (n[2] == 1) != nl        # the nonlinear adjoint keeps its launches
    assert cells[0] == 3 * p["B"] * p["Nx"] * p["Ny"] * p["T"]


@pytest.mark.parametrize("every,rows", [(2, 4), (3, 8), (1000, 4), (1000, 8)])
@pytest.mark.parametrize("tun", TILED)
@pytest.mark.parametrize("case", ["linear", "h", "nonlinear"])
def test_tiles_taken_over(case, tun, every, rows, cuda):
    p, nl, plan = _plan(case, tun, cuda, rows)
    ref = _run(p, nl, plan, cuda)
    print("case", case, tun, every, plan.tuning, flush=True)
    _walk(plan, every)  # 1000: one workgroup per sample
    out = _run(p, nl, plan, cuda)
    _walk(plan, 1)
    again = _run(p, nl, plan, cuda)
    assert torch.isfinite(ref[0]).all() and float(ref[3].abs().max()) > 0
    for a, b, c in zip(ref, out, again):
        assert torch.equal(a, b) and torch.equal(a, c)


@pytest.mark.parametrize("every", [2, 1000])
@pytest.mark.parametrize("tun", ["3x3", "rows-only", "past-neighbours", "step-by-step"])
@pytest.mark.parametrize("case", ["linear", "h"])
def test_tiles_taken_over_f64(case, tun, every, cuda):
    p, cfg, h, nl, onl = _setup(case)
    tuning = dict(TUNINGS[tun], cpt=4, ck_every=p["T"])
    plan = Plan(cfg, p["B"], p["T"], 1.0, cuda, tuning)
    ref = _run(p, nl, plan, cuda, torch.float64)
    print("case", case, tun, every, flush=True)
    _walk(plan, every)
    out = _run(p, nl, plan, cuda, torch.float64)
    yo, _ = co.forward(p["b"], p["c"], p["x"], p["dt"], h, p["src"], p["taps"], dtype=np.float64)
    assert np.array_equal(ref[0].cpu().numpy(), yo)
    for a, b in zip(ref, out):
        assert torch.equal(a, b)


@pytest.mark.parametrize("tun", TILED)
@pytest.mark.parametrize("case", ["linear", "nonlinear"])
def test_forward_given_up(case, tun, cuda):
    """Every wait ends at once: the first chunk's values stand, NaN for the
    rest of every probe series and every later field snapshot."""
    p, nl, plan = _plan(case, tun, cuda)
    n0 = plan.tuning["tblock"]
    t = {k: torch.from_numpy(p[k]).to(cuda) for k in ("x", "c", "b", "rho")}
    rho = t["rho"] if nl else None
    run = lambda fields, stride: WaveLoop.apply(t["x"], t["c"], t["b"], rho, plan, fields, stride)
    ref = [run(False, 1), run(True, 1), run(True, 5)]
    _walk(plan, 1, 1)
    y, f, f5 = run(False, 1), run(True, 1), run(True, 5)
    for a, r, k in ((y, ref[0], n0), (f, ref[1], n0), (f5, ref[2], n0 // 5)):
        assert torch.equal(a[:, :k], r[:, :k]) and torch.isnan(a[:, k:]).all()
    _walk(plan, 1)
    assert torch.equal(run(False, 1), ref[0])


@pytest.mark.parametrize("rows", [4, 8])
@pytest.mark.parametrize("tun", TILED)
def test_adjoint_given_up(tun, rows, cuda):
    """The gradient of c has a NaN for every tile, that of x a NaN for every
    step after the first chunk (the last steps)."""
    p, nl, plan = _plan("linear", tun, cuda, rows)
    k = plan.tuning["a_tblock"]
    grads = []
    for give_up in (0, 1):
        t = {q: torch.from_numpy(p[q]).to(cuda).requires_grad_(q != "b") for q in ("x", "c", "b")}
        _walk(plan, 1)
        y = WaveLoop.apply(t["x"], t["c"], t["b"], None, plan, False, 1)
        w = torch.from_numpy(np.random.default_rng(5).standard_normal(y.shape)).to(cuda, y.dtype)
        _walk(plan, 1, give_up)
        (y * w).sum().backward()
        grads.append((t["c"].grad, t["x"].grad))
    (gc, gx), (bc, bx) = grads
    tiles = plan.tuning["a_strips"] * plan.tuning["a_tcols"]
    assert int(torch.isnan(bc).sum()) == tiles and torch.isfinite(gc).all()
    assert torch.equal(bx[:, -k:], gx[:, -k:]) and torch.isnan(bx[:, :-k]).all()


@pytest.mark.parametrize("tun", TILED)
def test_forward_given_up_f64(tun, cuda):
    p, cfg, h, nl, onl = _setup("linear")
    plan = Plan(cfg, p["B"], p["T"], 1.0, cuda, dict(TUNINGS[tun], nt=1024, cpt=4,
                                                     ck_every=p["T"]))
    n0 = plan.tuning["tblock"]
    t = [torch.from_numpy(p[k]).to(cuda, torch.float64) for k in ("x", "c", "b")]
    run = lambda fields: WaveLoop.apply(*t, None, plan, fields, 1)
    ref = [run(False), run(True)]
    _walk(plan, 1, 1)
    for a, r in zip((run(False), run(True)), ref):
        assert torch.equal(a[:, :n0], r[:, :n0]) and torch.isnan(a[:, n0:]).all()


def test_arguments(cuda):
    _, _, plan = _plan("linear", "3x3", cuda)
    for every in (0, -1):
        with pytest.raises(ValueError):
            _walk(plan, every)
