"""What the plan of a default handle's launches leaves to the options, the
autotuner and the byte counts."""
import time

import numpy as np
import pytest

import shaw_amd
from shaw_amd import workloads
from tests.test_gpu_fom import say

pytestmark = pytest.mark.gpu


def engine(nr, nth, m, steps, **kw):
    app = shaw_amd.App.structured(nr, nth, workloads.layered_material())
    fom = shaw_amd.Fom(app, m, 0.1, **kw)
    rng = np.random.default_rng(nr + m)
    fom.set_sources(rng.integers(0, nr, m) * nth + 1)
    fom.set_forcing(rng.standard_normal((steps, m)))
    return fom


@pytest.mark.parametrize("nr,nth,m", [(100, 300, 1), (200, 1000, 16)])
def test_graph_steps_are_replayed(nr, nth, m):
    """A graph length asked for is what runs: strips of the configured shape,
    whole chunks replayed, the same states as the planned launches."""
    say(f"[gpu] graph_steps {nr}x{nth} M={m}")
    out = []
    for kw in ({}, dict(graph_steps=-1), dict(graph_steps=96)):
        fom = engine(nr, nth, m, 250, **kw)
        shape, cfg = fom.launch_shape(96), fom.config()
        asked = kw.get("graph_steps", 0) > 0
        assert asked == (shape["steps_per_launch"] == cfg["steps_per_launch"] and shape["segment"] == cfg["segment"])
        for n in (100, 150):
            fom.advance(n)
        out.append(fom.state())
        fom.close()
    for other in out[1:]:
        for x, y in zip(out[0], other):
            np.testing.assert_array_equal(x, y)
    assert np.abs(out[0][0]).max() > 0


def test_autotune_keeps_window_tiles_near_the_tables_end():
    """Fewer steps left than a window tile takes: it is timed at those."""
    say("[gpu] autotune 21x51, 5 steps left")
    fom = engine(21, 51, 1, 50)
    fom.advance(45)
    before = fom.state()
    assert fom.launch_shape(5)["segment"] == 0
    ms = fom.autotune(3)
    assert ms > 0 and fom.launch_shape(5)["segment"] == 0
    for x, y in zip(before, fom.state()):
        np.testing.assert_array_equal(x, y)
    fom.close()


def test_autotune_is_not_slower_than_the_plan():
    """509 x 2051, 15 columns: the planned 85-row segments run in one round of the
    chip, the candidates' 64 rows in two and 128 rows with a third more work. What the
    tuner keeps takes no longer than the plan (5 % for the spread of a timing)."""
    say("[gpu] autotune 509x2051 M=15")
    fom = engine(509, 2051, 15, 3000)
    planned = fom.launch_shape(70)
    assert planned["segment"] not in (0, 64, 128)

    def ms():
        fom.reset()
        fom.advance(70)
        return min(fom.time(140)[0] for _ in range(5))

    before = ms()
    fom.autotune(3)
    after = ms()
    say(f"  plan {planned} {before:.3f} ms, tuned {fom.launch_shape(70)} {after:.3f} ms")
    assert after <= 1.05 * before
    fom.close()


@pytest.mark.parametrize("nr,nth,m", [(200, 1000, 1), (200, 1000, 24)])
@pytest.mark.parametrize("kw", [{}, dict(steps_per_launch=3), dict(kernel=shaw_amd.KERNEL_SPLIT)])
def test_bytes_per_step_are_of_the_launches_that_run(nr, nth, m, kw):
    say(f"[gpu] bytes per step {nr}x{nth} M={m} {kw}")
    fom = engine(nr, nth, m, 10, **kw)
    steps = fom.launch_shape(5040)["steps_per_launch"]  # a multiple of every planned length
    nvp, nsp = nr * nth, (nr - 1) * nth + nr * (nth - 1)
    passes = 3 if "kernel" in kw else 2
    want = 8.0 * (m * passes * (nvp + nsp) + 4 * nvp + 2 * nsp) / steps
    assert fom.bytes_per_step()[0] == pytest.approx(want, rel=1e-12)
    assert kw or m > 1 or steps != fom.config()["steps_per_launch"]  # window tiles
    fom.close()


def test_single_steps_are_not_slower_than_strips():
    """200 x 500, 3 columns: advances by one step, which long launches' windows take
    1.6 times as long for as the strips of explicit options (a quarter allowed for the
    spread of a timing)."""
    say("[gpu] single steps 200x500 M=3")
    best = {}
    for name, kw in (("default", {}), ("strips", dict(strip=64))):
        fom = engine(200, 500, 3, 2000, **kw)
        fom.advance(8)
        fom.sync()
        times = []
        for _ in range(5):
            t = time.perf_counter()
            for _ in range(200):
                fom.advance(1)
            fom.sync()
            times.append(time.perf_counter() - t)
        best[name] = min(times)
        fom.close()
    say(f"  us per step {({k: round(v * 5e3, 2) for k, v in best.items()})}")
    assert best["default"] <= 1.25 * best["strips"]
