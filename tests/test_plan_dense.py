"""Probe arrays that no block's tables hold: the plan says so at once instead of
after trying every tiling of the grid, and the per-step kernels take it."""
import time

import pytest

from wavetorch_amd._loop import LoopConfig, resolve, suggest

N = 300
ARRAYS = {
    # probe pixels, sources, whether a block holds them
    "sparse": ([(150 + 4 * k, 7 * k) for k in range(12)], [(75, 75, 0)], True),
    "line": ([(200, j) for j in range(16)], [(75, j, 0) for j in range(20, 270)], True),
    "block": ([(150 + k // 5, 7 * k % N) for k in range(40)], [(75, 75, 0)], False),
    "row": ([(200, j) for j in range(17)], [(75, 75, 0)], False),
    "edge": ([(0, j) for j in range(9)] + [(16, j) for j in range(8)], [(75, 75, 0)], False),
    "apart": ([(0, j) for j in range(9)] + [(290, j) for j in range(8)], [(75, 75, 0)], True),
    "shared": ([(150, 150)], [(75, 75, 0), (75, 75, 1)], False),
    "lines": ([(150, 150)], [(75 + k, j, 0) for k in range(2) for j in range(200)], False),
}


@pytest.mark.parametrize("name", sorted(ARRAYS))
def test_plan_of_a_probe_array(name):
    taps, src, holds = ARRAYS[name]
    cfg = LoopConfig(Nx=N, Ny=N, dt=0.6, h=1.0, src_px=tuple(src),
                     taps=tuple((x, y, 1) for x, y in taps))
    t0 = time.process_time()
    got, _, _ = resolve(cfg, 4, 500, 1.0, {"ck_every": 64})
    tun = suggest(cfg, 4, 500, 1.0, 500, 64)
    assert time.process_time() - t0 < 0.5
    assert got["plain"] == (0 if holds else 1)
    assert resolve(cfg, 4, 500, 1.0, tun)[0]["plain"] == got["plain"]
    # a block that was asked for is refused, not replaced
    if not holds:
        with pytest.raises(RuntimeError):
            resolve(cfg, 4, 500, 1.0, {"nt": 1024, "cpt": 8})
        with pytest.raises(RuntimeError):
            resolve(cfg, 4, 500, 1.0, {"strips": 9, "tcols": 9, "tblock": 16, "nt": 1024, "cpt": 4})
