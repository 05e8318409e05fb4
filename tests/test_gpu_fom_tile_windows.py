"""The window-tile FOM kernel with 2, 3 and 4 rows per wave (24-, 36- and 48-row
windows), overlapping in both directions, and one, two and four column blocks per
workgroup, a last group that is not full among them: the plan takes these on the
grids below (named by the planned steps per launch, which tell them apart). Every
value equals that of single steps (no FMA, the same expressions in the same order)."""
import numpy as np
import pytest

import shaw_amd
from tests.test_gpu_fom import LAYERED, say

pytestmark = pytest.mark.gpu

# (nr, nth, columns, precision), steps per launch of the plan; rows per wave, column
# blocks per workgroup
CASES = [((71, 259, 5, shaw_amd.FP64), 10),    # 2, 1
         ((60, 400, 5, shaw_amd.FP64), 16),    # 3, 1
         ((180, 500, 7, shaw_amd.FP64), 10),   # 3, 2
         ((160, 750, 13, shaw_amd.FP64), 8),   # 3, 4; seven blocks
         ((150, 1000, 1, shaw_amd.FP64), 16),  # 4, 1
         ((200, 500, 3, shaw_amd.FP64), 14),   # 4, 1
         ((85, 1000, 9, shaw_amd.FP64), 14),   # 4, 2; five blocks
         ((180, 700, 15, shaw_amd.FP64), 12),  # 4, 4
         ((180, 500, 7, shaw_amd.FP32), 6),    # 4, 1
         ((85, 1000, 9, shaw_amd.FP32), 8),    # 3, 2; five blocks
         ((160, 750, 13, shaw_amd.FP32), 8),   # 3, 4; seven blocks
         ((230, 700, 15, shaw_amd.FP32), 10)]  # 4, 4


@pytest.mark.parametrize("grid,steps", CASES)
def test_windows_equal_single_steps(grid, steps):
    nr, nth, m, precision = grid
    say(f"[gpu] window tiles {nr}x{nth} M={m} precision={precision}")
    rng = np.random.default_rng(nr * nth + m)
    app = shaw_amd.App.structured(nr, nth, LAYERED)
    src = rng.integers(0, nr, m) * nth + rng.integers(0, nth, m)
    recv = rng.integers(0, nr, 40) * nth + rng.integers(0, nth, 40)
    recv[3] = recv[0]
    runs = [1, steps, 2 * steps + 3]
    total = sum(runs)
    table = rng.standard_normal((total, m))
    state = [rng.standard_normal((n, m)) * 1e-3 for n in (app.nVp, app.nSp)]
    out = []
    for kw in ({}, dict(steps_per_launch=1)):
        fom = shaw_amd.Fom(app, m, 0.2, precision=precision, **kw)
        if not kw:
            shape = fom.launch_shape(100 * steps)
            assert shape == {"launches": 100, "steps_per_launch": steps, "segment": 0}
        fom.set_sources(src)
        fom.set_forcing(table)
        fom.set_receivers(recv, 3, total // 3)
        fom.set_state(*state)
        for n in runs:
            fom.advance(n)
        out.append((fom.seismogram(), *fom.state()))
        fom.close()
    for x, y in zip(*out):
        np.testing.assert_array_equal(x, y)
        assert np.isfinite(x).all() and np.abs(x).max() > 0


@pytest.mark.parametrize("precision", [shaw_amd.FP64, shaw_amd.FP32])
@pytest.mark.parametrize("nr,nth,m", [(49, 130, 2), (200, 500, 3), (230, 1000, 7), (400, 1200, 5), (160, 750, 13),
                                      (150, 900, 1)])
def test_short_launches_equal_single_steps(nr, nth, m, precision):
    """Advances by a few steps and snapshots every few: launches of 1 to 9 steps,
    by windows of their own or the marching kernels."""
    say(f"[gpu] short launches {nr}x{nth} M={m} precision={precision}")
    rng = np.random.default_rng(nr + nth + m)
    app = shaw_amd.App.structured(nr, nth, LAYERED)
    src = rng.integers(0, nr, m) * nth + rng.integers(0, nth, m)
    recv = rng.integers(0, nr, 20) * nth + rng.integers(0, nth, 20)
    runs = [1, 1, 2, 3, 4, 5, 6, 7, 8, 9]
    total = sum(runs) + 24
    table = rng.standard_normal((total, m))
    state = [rng.standard_normal((n, m)) * 1e-3 for n in (app.nVp, app.nSp)]
    out = []
    for kw in ({}, dict(steps_per_launch=1)):
        fom = shaw_amd.Fom(app, m, 0.2, precision=precision, **kw)
        if not kw:
            assert fom.launch_shape(5040)["segment"] == 0
        fom.set_sources(src)
        fom.set_forcing(table)
        fom.set_receivers(recv, 1, total)
        fom.set_state(*state)
        for n in runs:
            fom.advance(n)
        got = [fom.seismogram(), *fom.state()]
        fom.reset()
        fom.set_snapshots("vp", 5, [0], 4)
        fom.set_snapshots("sp", 2, [m - 1], 12)
        fom.advance(24)
        got += [fom.snapshots("vp"), fom.snapshots("sp"), *fom.state()]
        out.append(got)
        fom.close()
    for x, y in zip(*out):
        np.testing.assert_array_equal(x, y)
        assert np.isfinite(x).all() and np.abs(x).max() > 0
