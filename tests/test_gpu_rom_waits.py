"""Engines whose columns are shared among workgroups: waits that end without the
others. Groups that do not meet at a launch's start run unshared and give the
same values bit for bit, with the launches enqueued in a row or waited for one
by one; a value that does not come within a launch is an error, not a result. The
waits are set to nothing looked for in vain; every kernel ends normally."""
import numpy as np
import pytest

import shaw_amd

pytestmark = pytest.mark.gpu

CASES = [(384, 300, 40, shaw_amd.ROM_BF16X4, 0, 0), (500, 512, 17, shaw_amd.ROM_BF16X3, 5, 0),
         (384, 384, 640, shaw_amd.ROM_BF16X3, 5, 2), (512, 512, 100, shaw_amd.ROM_BF16X4, 5, 2),
         (256, 200, 60, shaw_amd.ROM_FP64, 0, 0), (384, 384, 300, shaw_amd.ROM_FP64, 0, 0),
         (512, 500, 250, shaw_amd.ROM_FP64, 0, 0)]


def engine(kv, ks, m, precision, macro, budget):
    rng = np.random.default_rng(kv + 3 * ks + m)
    arv = rng.standard_normal((kv, ks)) * (0.5 / np.sqrt(max(kv, ks)))
    rom = shaw_amd.Rom(arv, -arv.T.copy(), 0.2, precision, rng.standard_normal((7, kv)), max_cols=m, max_samples=60)
    if macro:
        rom.set_macro_steps(macro)
    if budget:
        rom.set_time_budget(budget)
    f = rng.standard_normal((300, m))
    f[100:] = 0.0
    horizons = [300 - 5 * (j % 7) for j in range(m)]
    return rom, rom.admit(rng.standard_normal((kv, m)), f, horizons, every=5)


def results(rom, slots):
    states = [rom.state(s) for s in slots[:3] + slots[-3:]]
    return rom.retire_many(slots, 60), states


@pytest.mark.parametrize("kv,ks,m,precision,macro,budget", CASES)
@pytest.mark.parametrize("waited", [False, True])
def test_groups_that_do_not_meet_run_unshared(kv, ks, m, precision, macro, budget, waited):
    print(f"[gpu] ROM waits kv={kv} ks={ks} M={m} precision={precision} macro={macro} waited={waited}", flush=True)
    out = []
    for tries in (None, 0):
        rom, slots = engine(kv, ks, m, precision, macro, budget)
        for j, n in enumerate((20, 60, 2, 90, 30, 98)):
            if tries is not None:  # by turns: nothing waited for, ordinary launches
                shaw_amd.debug_rom_waits(rom, tries if j % 3 != 1 else 1 << 24)
            rom.advance(n)
            if waited:
                rom.sync()
        out.append(results(rom, slots))
    for x, y in zip(out[0][0], out[1][0]):
        np.testing.assert_array_equal(x, y)
    for x, y in zip(out[0][1], out[1][1]):
        assert x[2] == y[2]
        np.testing.assert_array_equal(x[0], y[0])
        np.testing.assert_array_equal(x[1], y[1])
    assert max(np.abs(x).max() for x in out[0][0]) > 0


@pytest.mark.parametrize("kv,ks,m,precision", [(384, 300, 40, shaw_amd.ROM_BF16X4), (256, 256, 60, shaw_amd.ROM_FP64)])
def test_a_value_that_never_comes_is_an_error(kv, ks, m, precision):
    print(f"[gpu] ROM exchange lost kv={kv} M={m} precision={precision}", flush=True)
    rom, slots = engine(kv, ks, m, precision, 0, 0)
    shaw_amd.debug_rom_waits(rom, no_words=True)
    rom.advance(100)
    with pytest.raises(shaw_amd.ShawError, match="lost each other"):
        rom.sync()
    with pytest.raises(shaw_amd.ShawError, match="lost each other"):
        rom.state(slots[0])
    rom.close()


@pytest.mark.parametrize("tries", [100, 1 << 24])
def test_shared_engine_beside_a_long_launch(tries):
    """Another engine's launch holds most CUs for a tenth of a second: groups that
    cannot be placed wait for it, or give up early and run unshared after it."""
    print(f"[gpu] shared ROM beside a long launch, {tries} tries", flush=True)
    rng = np.random.default_rng(3)
    k, m = 512, 4000
    big = shaw_amd.Rom(rng.standard_normal((k, k)) * 0.01, rng.standard_normal((k, k)) * 0.01, 0.2, shaw_amd.ROM_FP64,
                       rng.standard_normal((2, k)), max_cols=m, max_samples=20)
    big.admit_signals(rng.standard_normal((k, m)), ["ricker"] * m, np.full(m, 20.0), np.full(m, 5.0), 2000, every=100)
    for kv, ks, cols, precision in ((384, 384, 640, shaw_amd.ROM_BF16X4), (512, 512, 128, shaw_amd.ROM_FP64)):
        out = []
        for beside in (False, True):
            rom, slots = engine(kv, ks, cols, precision, 0, 0)
            rom.sync()
            if beside:
                shaw_amd.debug_rom_waits(rom, tries)
                big.advance(800)
            for n in (100, 150, 50):
                rom.advance(n)
            out.append(results(rom, slots))
        for x, y in zip(out[0][0], out[1][0]):
            np.testing.assert_array_equal(x, y)
        for x, y in zip(out[0][1], out[1][1]):
            assert x[2] == y[2]
            np.testing.assert_array_equal(x[0], y[0])
            np.testing.assert_array_equal(x[1], y[1])
    big.sync()


@pytest.mark.parametrize("kv,ks,m,precision", [(384, 384, 40, shaw_amd.ROM_BF16X4), (512, 300, 20, shaw_amd.ROM_BF16X3),
                                               (256, 256, 20, shaw_amd.ROM_FP64), (384, 384, 300, shaw_amd.ROM_FP64)])
def test_nonfinite_columns_stay_their_own(kv, ks, m, precision):
    """A column that is infinite or undefined goes through the exchange as such and
    leaves the others alone, as in an engine that shares nothing."""
    print(f"[gpu] shared ROM with non-finite columns kv={kv} M={m} precision={precision}", flush=True)
    rng = np.random.default_rng(kv + m)
    arv = rng.standard_normal((kv, ks)) * (0.5 / np.sqrt(max(kv, ks)))
    rows, b, f = rng.standard_normal((3, kv)), rng.standard_normal((kv, m)), rng.standard_normal((60, m))
    f[7, 0], f[11, 5], f[13, 18] = np.nan, np.inf, -np.inf
    out = []
    for slots in (m, 2400):
        assert (shaw_amd.debug_rom_shape(precision, kv, ks, slots)[1] > 1) == (slots == m)
        rom = shaw_amd.Rom(arv, -arv.T.copy(), 0.2, precision, rows, max_cols=slots, max_samples=60)
        ids = rom.admit(b, f, [60] * m, every=1)
        rom.advance(60)
        states = [rom.state(s) for s in ids]
        out.append((rom.retire_many(ids, 60), states))
    for j, (x, y) in enumerate(zip(out[0][0], out[1][0])):
        np.testing.assert_array_equal(x, y)
        assert np.isfinite(x).all() == (j not in (0, 5, 18))
    for (v, s, _), (w, t, _) in zip(out[0][1], out[1][1]):
        np.testing.assert_array_equal(v, w)
        np.testing.assert_array_equal(s, t)
