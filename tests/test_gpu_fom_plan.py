"""What the plan of a default handle's launches leaves to the options, the
autotuner and the byte counts."""
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
