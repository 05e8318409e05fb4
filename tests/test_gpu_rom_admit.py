"""Admission transposes the forcing columns and tables on the device: engines
fed the same columns one by one and all at once hold the same states bit for
bit, at the edges of the transpose's 32 x 32 tiles and with several slots of
uneven horizons retired together."""
import numpy as np
import pytest

import shaw_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv,n,steps", [(1, 1, 1), (17, 31, 33), (64, 32, 32), (70, 33, 65), (40, 65, 130)])
def test_admit_together_equals_one_by_one(kv, n, steps):
    print(f"[gpu] admission kv={kv} n={n} steps={steps}", flush=True)
    rng = np.random.default_rng(kv + n)
    arv = rng.standard_normal((kv, kv)) * 0.1
    rows = rng.standard_normal((3, kv))
    b = rng.standard_normal((kv, n))
    f = rng.standard_normal((steps, n))
    horizons = [max(1, steps - j % 5) for j in range(n)]
    out = []
    for split in (False, True):
        rom = shaw_amd.Rom(arv, -arv.T.copy(), 0.2, shaw_amd.ROM_FP64, rows, max_cols=n, max_samples=steps)
        if split:
            slots = sum((rom.admit(b[:, [j]], f[:, [j]], [horizons[j]], every=1) for j in range(n)), [])
        else:
            slots = rom.admit(b, f, horizons, every=1)
        rom.advance(steps)
        states = [rom.state(s) for s in (slots[0], slots[-1])]
        out.append((rom.retire_many(slots, steps), states))
    for j, (x, y) in enumerate(zip(out[0][0], out[1][0])):
        assert x.shape == (horizons[j], 3)
        np.testing.assert_array_equal(x, y)
    for (av, asx, s), (bv, bs, t) in zip(out[0][1], out[1][1]):
        assert s == t
        np.testing.assert_array_equal(av, bv)
        np.testing.assert_array_equal(asx, bs)
    # the first step's sample is C (f dt) b, exactly as the engine rounds it for one mode
    if kv == 1:
        np.testing.assert_allclose(out[0][0][0][0], rows[:, 0] * (f[0, 0] * 0.2 * b[0, 0]), rtol=1e-15)
