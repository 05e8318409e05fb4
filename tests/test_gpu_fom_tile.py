"""The window-tile FOM kernel (the default on grids whose states stay in the
last-level cache) at the edges of its windows: 64 points by 24 rows (taller ones
in test_gpu_fom_tile_windows.py), whole grids in one window of up to 48,
remainders of one point or row, one to five columns, split runs. Every output
equals the oracle's bit for bit (no FMA, the same expressions in the same order),
and FP32 states those of single FP32 steps."""
import numpy as np
import pytest

import oracle
import shaw_amd
from tests.test_gpu_fom import LAYERED, random_sources, say

pytestmark = pytest.mark.gpu

# (nr, nth, columns): one window; one row or point more than one; several
# windows whose last holds few rows and points
GRIDS = [(2, 3, 1), (24, 64, 1), (25, 64, 2), (24, 65, 3), (48, 64, 5), (49, 66, 1), (37, 113, 2), (85, 160, 4),
         (200, 161, 1), (71, 259, 5)]


def sources(rng, nr, nth, m):
    return rng.integers(0, nr, m) * nth + rng.integers(0, nth, m)


@pytest.mark.parametrize("nr,nth,m", GRIDS[1:])
def test_tiles_equal_oracle(nr, nth, m):
    say(f"[gpu] tile kernel {nr}x{nth} M={m}")
    rng = np.random.default_rng(nr * nth + m)
    app = shaw_amd.App.structured(nr, nth, LAYERED)
    ora = oracle.App("", LAYERED, structured=(nr, nth, 0.0, 180.0, 3480.0, 6371.0))
    src = random_sources(rng, m)
    rec = list(np.arange(0, 180, 11.5))
    a = shaw_amd.fom_run(app, 0.5, 75, src, m > 1, rec, 5, 25, 15)
    b = ora.fom_run(0.5, 75, src, m > 1, rec, 5, 25, 15)
    for key in b:
        np.testing.assert_array_equal(a[key], b[key], err_msg=key)


@pytest.mark.parametrize("precision", [shaw_amd.FP64, shaw_amd.FP32])
@pytest.mark.parametrize("nr,nth,m", GRIDS)
def test_tiles_equal_single_steps(nr, nth, m, precision):
    """Sources anywhere (halo rows and points included), receivers off the
    surface and twice on one point, runs of 1, 2, 17, 61 and 130 steps on
    one handle, a state set in between."""
    say(f"[gpu] tile kernel {nr}x{nth} M={m} precision={precision} against single steps")
    rng = np.random.default_rng(7 * nr + nth)
    app = shaw_amd.App.structured(nr, nth, LAYERED)
    src = sources(rng, nr, nth, m)
    recv = sources(rng, nr, nth, 9)
    recv[3] = recv[0]
    runs = [1, 2, 17, 61, 130]
    total = sum(runs)
    table = rng.standard_normal((total, m))
    state = [rng.standard_normal((n, m)) * 1e-3 for n in (app.nVp, app.nSp)]
    out = []
    for kw in ({}, dict(steps_per_launch=1)):
        fom = shaw_amd.Fom(app, m, 0.5, precision=precision, **kw)
        fom.set_sources(src)
        fom.set_forcing(table)
        fom.set_receivers(recv, 3, total // 3)
        for j, n in enumerate(runs):
            fom.advance(n)
            if j == 2:
                fom.set_state(*state)
        out.append((fom.seismogram(), *fom.state()))
        fom.close()
    for x, y in zip(*out):
        np.testing.assert_array_equal(x, y)
    assert np.abs(out[0][1]).max() > 0


@pytest.mark.parametrize("n,every", [(75, (5, 25, 15)), (33, (1, 0, 0)), (8, (2, 4, 8))])
def test_planned_packs_equal_oracle(n, every):
    """A grid on which the default options plan marching strips of their own
    pack length and segments: runs split evenly, up to snapshots too."""
    say(f"[gpu] planned packs n={n} every={every}")
    nr, nth, m = 200, 1000, 24
    rng = np.random.default_rng(n)
    app = shaw_amd.App.structured(nr, nth, LAYERED)
    fom = shaw_amd.Fom(app, m, 0.25)
    shape = fom.launch_shape(n)
    fom.close()
    assert shape["segment"] > 0 and 4 <= shape["steps_per_launch"] <= 7
    ora = oracle.App("", LAYERED, structured=(nr, nth, 0.0, 180.0, 3480.0, 6371.0))
    src = random_sources(rng, m, 600.0)
    rec = list(range(0, 180, 7))
    a = shaw_amd.fom_run(app, 0.25, n, src, True, rec, *every)
    b = ora.fom_run(0.25, n, src, True, rec, *every)
    for key in b:
        np.testing.assert_array_equal(a[key], b[key], err_msg=key)


def test_planned_packs_fp32_equal_single_steps():
    say("[gpu] planned packs FP32")
    nr, nth, m, n = 200, 1000, 24, 60
    rng = np.random.default_rng(3)
    app = shaw_amd.App.structured(nr, nth, LAYERED)
    src = random_sources(rng, m, 600.0)
    rec = list(range(0, 180, 7))
    a = shaw_amd.fom_run(app, 0.25, n, src, True, rec, 3, 20, 12, precision=shaw_amd.FP32)
    b = shaw_amd.fom_run(app, 0.25, n, src, True, rec, 3, 20, 12, precision=shaw_amd.FP32, steps_per_launch=1)
    for key in b:
        np.testing.assert_array_equal(a[key], b[key], err_msg=key)
