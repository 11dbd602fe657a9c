"""Attempts that the morphodynamic checks refuse, with the wide kernels (148
tiles of 16 x 16 cells): the first operator's last stage then follows the
morphodynamic stages and updates only the maxima.  State, step counts and
maxima against the oracle, bit for bit (only +, -, x, / and square roots are
evaluated), alone and in a batch, with the maxima tracked and not."""
import numpy as np
import pytest

from kestrel_amd import workloads
from kestrel_amd.runtime import SLOT_DONE, Batch
from tests.helpers import FIELDS, active_mask, oracle_for, stepper_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("track", [1, 0])
def test_refused_attempts(gpu, batch, track):
    wl = workloads.morpho_cap(256, steps=0, tile=16, radius=392.0, height=1.0, dx=4.0, erosion="simple",
                              deposition="simple", transition="step", damping="rat3")
    wl.cfg.max_dt = 10.0
    wl.cfg.track_maxima = track
    o, g = oracle_for(wl), stepper_for(wl)
    so = o.step_n(6)
    if batch:
        b = Batch(1)
        s = b.attach(g)
        b.start(s, nsteps=6)
        assert b.run()[s] == SLOT_DONE
        sg = b.stats(s)
    else:
        sg = g.step_n(6)
    assert so["rejected"] > 6
    assert (sg["steps"], sg["rejected"]) == (so["steps"], so["rejected"])
    a, c = g.state(), o.state()
    assert a["t"] == c["t"] and np.array_equal(a["tile_state"], c["tile_state"])
    m = active_mask(wl.cfg, c["tile_state"])
    assert int((c["tile_state"] == 1).sum()) >= 128
    for f in FIELDS:
        assert np.array_equal(a[f][m], c[f][m]), f
    if track:
        for k, (x, y) in enumerate(zip(g.maxima(), o.maxima())):
            assert np.array_equal(x[m], y[m]), f"maxima array {k}"
    if batch:
        b.close()
    g.close()
