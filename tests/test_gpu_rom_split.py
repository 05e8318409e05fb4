"""BF16 reduced-order engines of 257 to 512 modes share a tile of 16 columns
among several workgroups while the chip has room for them, and give it one
workgroup where it has not. Each row's sums run in the same order either way,
so an engine with few column slots must agree bit for bit with one of many on
the same problem: both sharing widths, a partly filled last group of eight
tiles, uneven horizons, split runs, more receivers than one row tile, macro
steps and a time budget."""
import numpy as np
import pytest

import shaw_amd

pytestmark = pytest.mark.gpu

# kv, ks, columns: eight row tiles a workgroup at the first sizes of a mode
# count, four at the last
SIZES = [(257, 300, 1), (384, 384, 640), (384, 290, 641), (290, 200, 1023), (380, 250, 1280), (400, 512, 17),
         (512, 512, 512), (500, 487, 513)]


def run(arv, ars, rows, b, f, horizons, precision, macro, cols, filler=0):
    rom = shaw_amd.Rom(arv, ars, 0.2, precision, rows, max_cols=cols, max_samples=f.shape[0] // 5)
    if macro:
        rom.set_macro_steps(5)
    if macro == 2:
        rom.set_time_budget(2)
    slots = rom.admit(b, f, horizons, every=5)
    if filler:
        rom.admit(np.ones((b.shape[0], filler)), np.zeros((f.shape[0], filler)), [f.shape[0]] * filler, every=5)
    for n in (1, 2, 7, 90, 200):
        rom.advance(n)
    states = [rom.state(s) for s in slots[:3] + slots[-3:]]
    return rom.retire_many(slots, f.shape[0] // 5), states


def compare(kv, ks, m, precision, macro, cols, filler=0):
    rng = np.random.default_rng(1000 * kv + ks + m)
    arv = rng.standard_normal((kv, ks)) * (0.5 / np.sqrt(max(kv, ks)))
    ars = -arv.T.copy()
    rows = rng.standard_normal((19, kv))
    b = rng.standard_normal((kv, m))
    f = rng.standard_normal((300, m))
    f[100:] = 0.0
    horizons = [300 - 5 * (j % 7) for j in range(m)]
    one = run(arv, ars, rows, b, f, horizons, precision, macro, m)
    two = run(arv, ars, rows, b, f, horizons, precision, macro, cols, filler)
    for x, y in zip(one[0], two[0]):
        np.testing.assert_array_equal(x, y)
    for x, y in zip(one[1], two[1]):
        assert x[2] == y[2]
        np.testing.assert_array_equal(x[0], y[0])
        np.testing.assert_array_equal(x[1], y[1])
    assert max(np.abs(x).max() for x in one[0]) > 0


@pytest.mark.parametrize("macro", [0, 1, 2])
@pytest.mark.parametrize("precision", [shaw_amd.ROM_BF16X3, shaw_amd.ROM_BF16X4])
@pytest.mark.parametrize("kv,ks,m", SIZES)
def test_shared_tile_equals_one_workgroup(kv, ks, m, precision, macro):
    print(f"[gpu] shared ROM tile kv={kv} ks={ks} M={m} precision={precision} macro={macro}", flush=True)
    compare(kv, ks, m, precision, macro, 2048)


# one set and two, at the most columns of each; the engine of many columns runs workgroups of sixteen (up to 256 modes,
# with enough of them active)
@pytest.mark.parametrize("kv,ks,m,cols,filler", [(193, 256, 1, 2400, 2100), (256, 256, 256, 2400, 2100),
                                                 (257, 384, 9, 2064, 0), (384, 384, 160, 2064, 0),
                                                 (384, 300, 320, 2064, 0),
                                                 (500, 487, 15, 2064, 0), (512, 512, 128, 2064, 0),
                                                 (512, 400, 256, 2064, 0)])
def test_shared_fp64_columns(kv, ks, m, cols, filler):
    print(f"[gpu] shared FP64 ROM columns kv={kv} ks={ks} M={m}", flush=True)
    compare(kv, ks, m, shaw_amd.ROM_FP64, 0, cols, filler)


def test_shared_engines_side_by_side():
    """Engines whose launches each want most of the chip, enqueued on their own
    streams without a wait between, give what each gives alone."""
    rng = np.random.default_rng(5)
    engines = []
    for kv, m, precision in ((384, 512, shaw_amd.ROM_BF16X4), (512, 128, shaw_amd.ROM_FP64), (500, 500, shaw_amd.ROM_BF16X3)):
        arv = rng.standard_normal((kv, kv)) * (0.5 / np.sqrt(kv))
        rows, b, f = rng.standard_normal((5, kv)), rng.standard_normal((kv, m)), rng.standard_normal((400, m))

        def engine():
            rom = shaw_amd.Rom(arv, -arv.T.copy(), 0.2, precision, rows, max_cols=m, max_samples=80)
            return rom, rom.admit(b, f, [400] * m, every=5)

        rom, slots = engine()
        rom.advance(400)
        alone = rom.retire_many(slots, 80)
        engines.append((*engine(), alone))
    for _ in range(8):
        for rom, _, _ in engines:
            rom.advance(50)
    for rom, slots, alone in engines:
        for x, y in zip(rom.retire_many(slots, 80), alone):
            np.testing.assert_array_equal(x, y)
            assert np.isfinite(x).all()
