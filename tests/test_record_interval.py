"""The checkpoint interval of a call that leaves it open: the rule on the
host, and on the device the plans that forwards take while an earlier
forward's whole record waits for its backward."""
import numpy as np
import pytest
import torch

import oracle.c_oracle as co
from tests.helpers import rel
from wavetorch_amd import (WaveCell, WaveGeometryFreeForm, WaveIntensityProbe, WaveRNN,
                           WaveSource)
from wavetorch_amd._loop import LoopConfig, auto_interval


@pytest.mark.parametrize("nonlinear", [False, True])
def test_auto_interval(nonlinear):
    cfg = LoopConfig(Nx=50, Ny=39, dt=0.6, h=1.0, src_px=((9, 9, 0),), taps=((20, 20, 1),),
                     c_nl=0.05 if nonlinear else 0.0)
    step = (8 if nonlinear else 4) * 3 * 50 * 40  # batch 3
    K = lambda T, steps: auto_interval(cfg, 3, T, steps * step, 64)
    assert K(1000, 1000) == 1000                  # fits whole
    assert K(1000, 999) == 500 and K(1001, 501) == 501
    assert K(1000, 334) == 334 and K(1000, 333) == 250 and K(1000, 250) == 250
    assert K(1000, 249) == 64                     # less than a quarter: not worth its memory
    assert K(64, 1) == 64 and K(10, 0) == 10      # no longer than the default interval
    assert K(100, 99) == 64                       # a half is shorter than the default


@pytest.mark.gpu
def test_forward_while_a_record_waits(cuda):
    geom = WaveGeometryFreeForm((60, 52), 1.0, c0=1.0, c1=0.5, abs_N=8, abs_sig=1.0, abs_p=2,
                                rho="half")
    model = WaveRNN(WaveCell(0.7, geom), WaveSource(16, 26),
                    [WaveIntensityProbe(44, 20), WaveIntensityProbe(44, 30)]).to(cuda)
    n = torch.arange(150.0)
    x = torch.stack([torch.sin(0.3 * n + k) * torch.exp(-((n - 60) / 25) ** 2)
                     for k in range(3)]).to(cuda)

    def grad(y):
        model.zero_grad(set_to_none=True)
        y.sum().backward()
        return geom.rho.grad.cpu().numpy()

    y1 = model(x)
    y2 = model(x)  # y1's record waits: checkpoints every 64 steps
    assert sorted(p.tuning["ck_every"] for p in model._plans.values()) == [64, 150]
    assert torch.equal(y1, y2)
    g2, g1 = grad(y2), grad(y1)
    assert rel(g1, g2) < 1e-5  # the same lambdas, summed over other launches
    y3 = model(x)              # nothing waits any more
    assert model.plan(3, 150, x.device).record_waits()
    assert rel(grad(y3), g1) == 0.0
    assert not model.plan(3, 150, x.device).record_waits()


@pytest.mark.gpu
@pytest.mark.parametrize("N,T", [(7, 300), (14, 257), (20, 1000)])
def test_launch_longer_than_its_block(N, T, cuda):
    """A small grid is one tile whose launches take up to 256 steps with 64
    or 128 threads: the staged input samples outnumber the threads."""
    geom = WaveGeometryFreeForm((N, N), 1.0, c0=1.0, c1=0.5, abs_N=2, abs_sig=1.0, abs_p=2,
                                rho="half")
    model = WaveRNN(WaveCell(0.7, geom), WaveSource(3, 3),
                    [WaveIntensityProbe(N - 3, N - 3)]).to(cuda)
    x = np.random.default_rng(N).standard_normal((2, T)).astype(np.float32)
    with torch.no_grad():
        y = model(torch.from_numpy(x).to(cuda)).cpu().numpy()
        c = geom.c.cpu().numpy()
    yo, _ = co.forward(geom.b.cpu().numpy(), c, x, 0.7, 1.0, [[3, 3, 0]], [[N - 3, N - 3, 1]])
    assert np.array_equal(y, yo)


@pytest.mark.gpu
def test_open_batch_equals_checkpointed(cuda):
    """A batch whose interval is left open records every step; its outputs and
    gradients are those of checkpoints every 64 steps, bit for bit (launches
    end at the same steps), also in several parts."""
    from wavetorch_amd.batch import Instance, InstanceBatch
    rng = np.random.default_rng(3)
    insts, cs, xs, ys = [], [], [], []
    for N, T in [(40, 150), (56, 131), (40, 70), (56, 64)]:
        cfg = LoopConfig(Nx=N, Ny=N, dt=0.7, h=1.0, taps=((N - 12, N // 2, 1),),
                         src_px=tuple((9, j, 0) for j in range(N // 4, 3 * N // 4)))
        insts.append(Instance(cfg, torch.zeros(N, N), T, 1.0))
        for lst, a in ((cs, rng.uniform(0.5, 1.0, (N, N))), (xs, rng.standard_normal(T)),
                       (ys, rng.standard_normal((T, 1)))):
            lst.append(torch.from_numpy(a.astype(np.float32)).to(cuda))
    ref = None
    for kw in (dict(checkpoint_every=64), {}, dict(tuning={"streams": 2})):
        bt = InstanceBatch(insts, cuda, **kw)
        print("case", kw, bt.tuning[0]["ck_every"], flush=True)
        assert bt.tuning[0]["ck_every"] == (64 if "checkpoint_every" in kw else 150)
        bt.set_inputs(cs, xs, ys)
        bt.fwd_adj()
        out = [t.clone() for o in bt.outputs() for t in o]
        ref = ref or out
        assert all(torch.equal(a, b) for a, b in zip(ref, out))
    assert float(ref[1].abs().max()) > 0
