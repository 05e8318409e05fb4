"""Host forcing tables that are small are transposed on the host, others on the
device: engines admitted on both sides of the line (65,536 values of columns and
series) hold the same states and seismograms, with and without macro steps."""
import numpy as np
import pytest

import shaw_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("macro", [0, 10])
@pytest.mark.parametrize("kv,n,steps", [(64, 16, 4032), (64, 16, 4033), (40, 1, 300), (256, 33, 1700)])
def test_small_and_large_tables(kv, n, steps, macro):
    print(f"[gpu] admission kv={kv} n={n} steps={steps} macro={macro}", flush=True)
    rng = np.random.default_rng(kv + n)
    arv = rng.standard_normal((kv, kv)) * (0.5 / np.sqrt(kv))
    rows, b, f = rng.standard_normal((3, kv)), rng.standard_normal((kv, n)), rng.standard_normal((steps, n))
    f[100:] = 0.0
    precision = shaw_amd.ROM_BF16X3 if macro else shaw_amd.ROM_FP64
    out = []
    for longer in (0, 65536 // n + 1):  # a table with more (unused) steps goes the other way
        rom = shaw_amd.Rom(arv, -arv.T.copy(), 0.2, precision, rows, max_cols=n, max_samples=steps // 10)
        if macro:
            rom.set_macro_steps(macro)
        slots = rom.admit(b, np.concatenate([f, np.zeros((longer, n))]), [steps] * n, every=10)
        rom.advance(150)
        out.append(([rom.state(s) for s in (slots[0], slots[-1])], rom.retire_many(slots, steps // 10)))
    for x, y in zip(*[o[0] for o in out]):
        for u, v in zip(x, y):
            np.testing.assert_array_equal(u, v)
    for x, y in zip(out[0][1], out[1][1]):
        assert x.shape == (15, 3)
        np.testing.assert_array_equal(x, y)
