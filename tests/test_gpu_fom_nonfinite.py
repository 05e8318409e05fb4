"""States with an infinite or undefined value (a run that has blown up): window
tiles spread it as single steps do, one point a step, and nothing crosses from
one side of a window to the other. Values that are finite in either run are so in
both and equal."""
import numpy as np
import pytest

import shaw_amd
from tests.test_gpu_fom import LAYERED, say

pytestmark = pytest.mark.gpu

# (nr, nth, columns), the point of the velocity that is not finite: the last lane
# of a window, the grid's ends, a window's last row, an inner point
CASES = [(37, 64, 1, (11, 63)), (37, 64, 2, (11, 0)), (21, 51, 1, (20, 50)), (24, 130, 2, (5, 63)),
         (49, 130, 1, (23, 62)), (85, 160, 3, (47, 159)), (85, 160, 1, (0, 63)), (60, 100, 2, (30, 40))]


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("precision", [shaw_amd.FP64, shaw_amd.FP32])
@pytest.mark.parametrize("nr,nth,m,point", CASES)
def test_tiles_spread_nonfinite_as_single_steps(nr, nth, m, point, precision, bad):
    say(f"[gpu] tile kernel {nr}x{nth} M={m} {bad} at {point} precision={precision}")
    rng = np.random.default_rng(nr + nth)
    app = shaw_amd.App.structured(nr, nth, LAYERED)
    vp, sp = rng.standard_normal((app.nVp, m)) * 1e-3, rng.standard_normal((app.nSp, m)) * 1e-3
    vp[point[0] * nth + point[1], m - 1] = bad
    out = []
    for kw in ({}, dict(steps_per_launch=1)):
        fom = shaw_amd.Fom(app, m, 0.5, precision=precision, **kw)
        if not kw:
            assert fom.launch_shape(10)["segment"] == 0  # window tiles
        fom.set_sources(np.arange(m) + nth)
        fom.set_forcing(np.zeros((12, m)))
        fom.set_receivers(np.arange((nr - 1) * nth, nr * nth), 1, 12)
        fom.set_state(vp, sp)
        fom.advance(12)
        out.append((fom.seismogram(), *fom.state()))
        fom.close()
    for x, y in zip(*out):
        np.testing.assert_array_equal(np.isfinite(x), np.isfinite(y))
        np.testing.assert_array_equal(x[np.isfinite(x)], y[np.isfinite(y)])
    assert not np.isfinite(out[0][1]).all()
    assert np.isfinite(out[0][1]).any()
