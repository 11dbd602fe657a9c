"""Batches of more slots than a wavefront has lanes: the slot of a work item
is found over several levels (64 slots are one level, 65 and 130 two), with
empty slots between the used ones; each result is its result alone."""
import numpy as np
import pytest

from kestrel_amd import config as C
from kestrel_amd import scenario as S
from kestrel_amd.runtime import SLOT_DONE, Batch, Stepper
from tests.helpers import FIELDS

pytestmark = pytest.mark.gpu

NSTEPS = 12


def make(k):
    """A small cap release; k changes its size, place and slope."""
    n = 3 + k % 3
    cfg = C.default_config(n, n, 8, 8, dx=1.0, dy=1.0)
    C.hydraulic_only(cfg)
    cfg.bc = C.BC_SPONGE
    cfg.precision = C.PREC_MIXED
    C.derive(cfg)
    b0v = S.topo_xslope(cfg, 0.02 * (1 + k % 7))
    init = S.initial_state(cfg, b0v, [S.Cap(0.3 * (k % 4), 0.0, 2.0 + 0.25 * (k % 11), 1.0, psi=0.1 * (k % 2))])
    g = Stepper(cfg)
    g.set_topography(b0v)
    g.set_state(init)
    return g


@pytest.mark.parametrize("nslot,skip", [(64, 1), (65, 1), (130, 3)])
def test_slots_beyond_a_wavefront(gpu, nslot, skip):
    used = list(range(0, nslot, skip))
    alone = {}
    for k in used:
        g = make(k)
        st = g.step_n(NSTEPS)
        alone[k] = (st, g.state())
        g.close()
    b = Batch(nslot)
    gs = {}
    for k in range(nslot):          # slots are given out in order
        gs[k] = make(k)
        assert b.attach(gs[k]) == k
    for k in range(nslot):
        if k not in alone:
            b.detach(k)
            gs.pop(k).close()
    for k in used:
        b.start(k, nsteps=NSTEPS)
    status = b.run()
    for k in used:
        assert status[k] == SLOT_DONE
        st, ref = alone[k]
        bs = b.stats(k)
        got = gs[k].state()
        assert (bs["steps"], bs["rejected"], got["t"]) == (st["steps"], st["rejected"], ref["t"]), k
        assert np.array_equal(got["tile_state"], ref["tile_state"]), k
        for f in FIELDS:
            assert np.array_equal(got[f], ref[f]), f"slot {k}: {f}"
    b.close()
