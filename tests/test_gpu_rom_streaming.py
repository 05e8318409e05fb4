"""Engines whose operators stay on the CU against the kernels that stream them
every step: BF16 against operators padded with zero modes to unequal sizes of more
than 256 modes with more slots than can be shared (k_rom_steps_bf, _bfm), FP64 in
workgroups of four columns, unshared and for launches of many steps, against
workgroups of sixteen. Zero modes change no value and every sum runs in the same
order, so all must agree bit for bit. Each engine's layout is asked for first."""
import numpy as np
import pytest

import shaw_amd

pytestmark = pytest.mark.gpu


def operators(kv, ks, m, steps, skew):
    rng = np.random.default_rng(1000 * kv + ks + m)
    arv = rng.standard_normal((kv, ks)) * (0.5 / np.sqrt(max(kv, ks)))
    ars = -arv.T.copy() if skew else rng.standard_normal((ks, kv)) * (0.5 / np.sqrt(max(kv, ks)))
    return arv, ars, rng.standard_normal((19, kv)), rng.standard_normal((kv, m)), rng.standard_normal((steps, m))


def padded(arv, ars, rows, b, kv, ks):
    pad = lambda a, r, c: np.pad(a, ((0, r - a.shape[0]), (0, c - a.shape[1])))
    return pad(arv, kv, ks), pad(ars, ks, kv), pad(rows, rows.shape[0], kv), pad(b, kv, b.shape[1])


def run(arv, ars, rows, b, f, horizons, precision, macro, slots, launches, filler=0):
    rom = shaw_amd.Rom(arv, ars, 0.2, precision, rows, max_cols=slots, max_samples=f.shape[0] // 5)
    if macro:
        rom.set_macro_steps(macro)
    ids = rom.admit(b, f, horizons, every=5)
    if filler:
        rom.admit(np.ones((b.shape[0], filler)), np.zeros((f.shape[0], filler)), [f.shape[0]] * filler, every=5)
    for n in launches:
        rom.advance(n)
    states = [rom.state(s) for s in ids[:3] + ids[-3:]]
    return rom.retire_many(ids, f.shape[0] // 5), states


def equal(one, two, kv, ks):
    for x, y in zip(one[0], two[0]):
        np.testing.assert_array_equal(x, y)
    for (qv, qs, n), (pv, ps, k) in zip(one[1], two[1]):
        assert n == k
        np.testing.assert_array_equal(qv, pv[:kv])
        np.testing.assert_array_equal(qs, ps[:ks])
    assert max(np.abs(x).max() for x in one[0]) > 0


# kv, ks, columns, slots: each padded size up to 256, dofs of 256 modes with
# groups that are all padding, and one workgroup a tile above 256 modes
BF16 = [(64, 50, 5, 16), (128, 100, 33, 48), (190, 192, 20, 32), (256, 256, 18, 32), (256, 60, 17, 32),
        (70, 256, 16, 16), (250, 130, 20, 32), (384, 380, 20, 1296), (300, 384, 16, 1296)]


@pytest.mark.parametrize("macro", [0, 5])
@pytest.mark.parametrize("precision", [shaw_amd.ROM_BF16X3, shaw_amd.ROM_BF16X4])
@pytest.mark.parametrize("kv,ks,m,slots", BF16)
def test_bf16_equals_streaming(kv, ks, m, slots, precision, macro):
    print(f"[gpu] ROM against streaming kv={kv} ks={ks} M={m} precision={precision} macro={macro}", flush=True)
    kp, sp = (300, 256) if max(kv, ks) <= 256 else (400, 384)
    assert shaw_amd.debug_rom_shape(precision, kv, ks, slots)[:2] == (384 if max(kv, ks) > 256 else (max(kv, ks) + 63) // 64 * 64, 1)
    assert shaw_amd.debug_rom_shape(precision, kp, sp, 2048)[0] == 0
    arv, ars, rows, b, f = operators(kv, ks, m, 300, macro > 0)
    f[100:] = 0.0
    horizons = [300 - 5 * (j % 7) for j in range(m)]
    launches = (1, 2, 7, 90, 200)
    one = run(arv, ars, rows, b, f, horizons, precision, macro, slots, launches)
    two = run(*padded(arv, ars, rows, b, kp, sp), f, horizons, precision, macro, 2048, launches)
    equal(one, two, kv, ks)


# columns, slots just beyond those shared; slots and active columns of the
# sixteen-column engine
FP64 = [(128, 128, 20, 48, 7300, 7250), (193, 256, 9, 272, 2400, 2100), (256, 256, 272, 272, 2400, 2100), (384, 384, 30, 336, 2064, 0),
        (330, 384, 336, 336, 2064, 0), (512, 512, 20, 272, 1040, 0), (449, 512, 272, 272, 1040, 0)]


@pytest.mark.parametrize("kv,ks,m,slots,many,filler", FP64)
def test_fp64_four_columns_long_launches(kv, ks, m, slots, many, filler):
    print(f"[gpu] FP64 ROM long launches kv={kv} ks={ks} M={m}", flush=True)
    square = {128: 128, 256: 256, 384: 384, 512: 512}[ks]
    assert shaw_amd.debug_rom_shape(shaw_amd.ROM_FP64, kv, ks, slots)[:2] == (square, 1)
    assert shaw_amd.debug_rom_shape(shaw_amd.ROM_FP64, square, square, many)[:2] == (square if filler else 0, 1)
    arv, ars, rows, b, f = operators(kv, ks, m, 120, False)
    horizons = [120 - 5 * (j % 7) for j in range(m)]
    one = run(arv, ars, rows, b, f, horizons, shaw_amd.ROM_FP64, 0, slots, (5, 66, 49))
    two = run(*padded(arv, ars, rows, b, square, square), f, horizons, shaw_amd.ROM_FP64, 0, many, (5, 66, 49), filler)
    equal(one, two, kv, ks)
