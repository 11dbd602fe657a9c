"""A periodic 1D grid of several tiles of which some start as ghosts, among
them the first and the last, against the oracle, bit for bit: their edge
slopes (a 1D tile has sides W and E only) and their activation."""
import numpy as np
import pytest

from kestrel_amd import config as C
from kestrel_amd import scenario as S
from kestrel_amd.runtime import Stepper
from oracle.oracle import Oracle
from tests.helpers import FIELDS, active_mask

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [4, 50, 130])
@pytest.mark.parametrize("first", [0, 1, 4])
def test_ghosts_of_a_periodic_1d_grid(gpu, tile, first):
    cfg = C.default_config(6, 1, tile, 1, dx=1.0)
    C.hydraulic_only(cfg)
    cfg.bc = C.BC_PERIODIC
    C.derive(cfg)
    rng = np.random.default_rng(tile)
    b0v = 0.05 * rng.standard_normal((2, cfg.NX + 1))
    b0v[0, -1] = b0v[0, 0]
    active = np.zeros(6, np.uint8)
    active[first] = 1
    depth = np.where(active[np.arange(cfg.NX) // tile], rng.uniform(0.5, 1.5, cfg.NX), 0.0)[None, :]
    zero = np.zeros((1, cfg.NX))
    b0c = S.cell_topography(cfg, b0v)[0]
    init = S.InitialState(b0c + depth, zero, zero, zero, S._ghost_ring(cfg, active), zero)
    g, o = Stepper(cfg), Oracle(cfg)
    for s in (g, o):
        s.set_topography(b0v)
        s.set_state(init)
        s.step_n(25)
    a, b = g.state(), o.state()
    g.close()
    assert a["t"] == b["t"] and np.array_equal(a["tile_state"], b["tile_state"])
    assert (b["tile_state"] == C.TILE_ACTIVE).sum() > 1, "a ghost must have become active"
    m = active_mask(cfg, b["tile_state"])
    for f in FIELDS:
        assert np.array_equal(a[f][m], b[f][m]), f
