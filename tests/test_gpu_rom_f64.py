"""FP64 reduced-order engines: workgroups of four columns (k_rom_f64; from 193
modes on shared among workgroups in launches of ten, above 256 of four steps) against
workgroups of sixteen (k_rom_steps). The kernels add a product's terms in the
same order with one rounding each, so every value must agree bit for bit. The
sixteen-column kernel runs the same problem when more than 128 tiles of columns
are active (filler columns) on operators of more than 128 modes (zero padding
changes no value), and above 256 modes when the engine has many slots."""
import numpy as np
import pytest

import shaw_amd

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (63, 20, 3), (64, 64, 5), (65, 128, 17), (128, 127, 16), (129, 129, 20), (192, 150, 33),
         (193, 256, 18), (256, 256, 7), (257, 200, 5), (384, 384, 18), (385, 512, 6)]


def run(arv, ars, rows, b, f, horizons, slots, filler):
    rom = shaw_amd.Rom(arv, ars, 0.2, shaw_amd.ROM_FP64, rows, max_cols=slots, max_samples=f.shape[0] // 5)
    ids = rom.admit(b, f, horizons, every=5)
    if filler:
        n = filler
        rom.admit(np.ones((b.shape[0], n)), np.zeros((f.shape[0], n)), [f.shape[0]] * n, every=5)
    for n in (1, 2, 3, 50, 100):
        rom.advance(n)
    states = [rom.state(s) for s in ids[:3] + ids[-2:]]
    return rom.retire_many(ids, f.shape[0] // 5), states


@pytest.mark.parametrize("kv,ks,m", SIZES)
def test_four_columns_equal_sixteen(kv, ks, m):
    print(f"[gpu] FP64 ROM kv={kv} ks={ks} M={m}", flush=True)
    rng = np.random.default_rng(1000 * kv + ks)
    arv = rng.standard_normal((kv, ks)) * (0.5 / np.sqrt(max(kv, ks)))
    ars = rng.standard_normal((ks, kv)) * (0.5 / np.sqrt(max(kv, ks)))
    rows = rng.standard_normal((21, kv))
    b = rng.standard_normal((kv, m))
    f = rng.standard_normal((150, m))
    horizons = [150 - 5 * (j % 7) for j in range(m)]
    one = run(arv, ars, rows, b, f, horizons, m, 0)
    k = max(kv, ks)
    if k <= 256:
        k = max(k, 129)
        slots, filler = 2400, 2100
    else:
        slots, filler = 2064, 0
    pad = lambda a, r, c: np.pad(a, ((0, r - a.shape[0]), (0, c - a.shape[1])))
    two = run(pad(arv, k, k), pad(ars, k, k), pad(rows, 21, k), pad(b, k, m), f, horizons, slots, filler)
    for x, y in zip(one[0], two[0]):
        np.testing.assert_array_equal(x, y)
    for (qv, qs, n), (pv, ps, c) in zip(one[1], two[1]):
        assert n == c
        np.testing.assert_array_equal(qv, pv[:kv])
        np.testing.assert_array_equal(qs, ps[:ks])
    assert max(np.abs(x).max() for x in one[0]) > 0
