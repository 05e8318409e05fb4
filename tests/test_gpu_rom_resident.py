"""BF16 reduced-order engines of up to 256 modes keep their operators on the
CU; larger ones share them among workgroups where columns are few. Zero modes
change no value of the others, so an engine whose operators are padded with zeros
past 256 modes runs the same problem as a shared one of 384 (in launches below
four steps as one workgroup): both must agree bit for bit (with the kernels that
stream their operators, test_gpu_rom_streaming.py compares), at the edges of the
padded sizes (64, 128, 192, 256), with kv != ks, with uneven horizons, split
runs, partly filled tiles and macro steps."""
import numpy as np
import pytest

import shaw_amd

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (63, 17, 5), (64, 64, 16), (65, 64, 17), (128, 100, 33), (129, 128, 16), (192, 192, 20),
         (50, 193, 16), (256, 256, 18), (250, 131, 40)]


def run(arv, ars, rows, b, f, horizons, precision, macro):
    rom = shaw_amd.Rom(arv, ars, 0.2, precision, rows, max_cols=b.shape[1], max_samples=f.shape[0] // 5)
    if macro:
        rom.set_macro_steps(macro)
    slots = rom.admit(b, f, horizons, every=5)
    for n in (1, 2, 7, 90, 200):
        rom.advance(n)
    states = [rom.state(s) for s in slots[:3] + slots[-3:]]
    return rom.retire_many(slots, f.shape[0] // 5), states


@pytest.mark.parametrize("macro", [0, 5])
@pytest.mark.parametrize("precision", [shaw_amd.ROM_BF16X3, shaw_amd.ROM_BF16X4])
@pytest.mark.parametrize("kv,ks,m", SIZES)
def test_resident_equals_streaming(kv, ks, m, precision, macro):
    print(f"[gpu] resident ROM kv={kv} ks={ks} M={m} precision={precision} macro={macro}", flush=True)
    rng = np.random.default_rng(1000 * kv + ks)
    arv = rng.standard_normal((kv, ks)) * (0.5 / np.sqrt(max(kv, ks)))
    ars = rng.standard_normal((ks, kv)) * (0.5 / np.sqrt(max(kv, ks))) if macro == 0 else -arv.T.copy()
    rows = rng.standard_normal((7, kv))
    b = rng.standard_normal((kv, m))
    f = rng.standard_normal((300, m))
    f[100:] = 0.0
    horizons = [300 - 5 * (j % 7) for j in range(m)]
    big = 260
    pad = lambda a, r, c: np.pad(a, ((0, r - a.shape[0]), (0, c - a.shape[1])))
    one = run(arv, ars, rows, b, f, horizons, precision, macro)
    two = run(pad(arv, big, big), pad(ars, big, big), pad(rows, 7, big), pad(b, big, m), f, horizons, precision, macro)
    for x, y in zip(one[0], two[0]):
        np.testing.assert_array_equal(x, y)
    for (qv, qs, n), (pv, ps, k) in zip(one[1], two[1]):
        assert n == k
        np.testing.assert_array_equal(qv, pv[:kv])
        np.testing.assert_array_equal(qs, ps[:ks])
    assert max(np.abs(x).max() for x in one[0]) > 0
