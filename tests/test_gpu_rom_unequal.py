"""FP64 engines of unequal dofs on both sides of each line of their layout:
padded to a square or at their own sizes, shared, in workgroups of four columns or
of sixteen, they give the same values bit for bit."""
import numpy as np
import pytest

import shaw_amd

pytestmark = pytest.mark.gpu

CASES = [(100, 60, (2048, 2064)), (60, 100, (16, 2064)), (190, 60, (1024, 1040)), (150, 120, (2048, 2064)),
         (250, 64, (256, 272)), (190, 256, (256, 1024, 1040)), (300, 200, (320, 1024, 1040)), (64, 384, (320, 336)),
         (384, 320, (160, 1024, 1040)), (512, 50, (256, 272)), (430, 512, (128, 1024, 1040))]


@pytest.mark.parametrize("kv,ks,slots", CASES)
def test_layouts_agree(kv, ks, slots):
    print(f"[gpu] FP64 ROM kv={kv} ks={ks} slots={slots}", flush=True)
    layouts = [shaw_amd.debug_rom_shape(shaw_amd.ROM_FP64, kv, ks, n) for n in slots]
    assert len(set(layouts)) == len(slots) and layouts[-1][0] == 0
    rng = np.random.default_rng(kv * ks)
    m = 13
    arv = rng.standard_normal((kv, ks)) * (0.5 / np.sqrt(max(kv, ks)))
    ars = rng.standard_normal((ks, kv)) * (0.5 / np.sqrt(max(kv, ks)))
    rows, b, f = rng.standard_normal((5, kv)), rng.standard_normal((kv, m)), rng.standard_normal((120, m))
    horizons = [120 - 5 * (j % 4) for j in range(m)]
    out = []
    for n in slots:
        rom = shaw_amd.Rom(arv, ars, 0.2, shaw_amd.ROM_FP64, rows, max_cols=n, max_samples=24)
        ids = rom.admit(b, f, horizons, every=5)
        for steps in (3, 30, 87):
            rom.advance(steps)
        states = [rom.state(s) for s in (ids[0], ids[-1])]
        out.append((rom.retire_many(ids, 24), states))
    for other in out[1:]:
        for x, y in zip(out[0][0], other[0]):
            np.testing.assert_array_equal(x, y)
        for x, y in zip(out[0][1], other[1]):
            assert x[2] == y[2]
            np.testing.assert_array_equal(x[0], y[0])
            np.testing.assert_array_equal(x[1], y[1])
    assert max(np.abs(x).max() for x in out[0][0]) > 0
