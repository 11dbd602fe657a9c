"""Periodic boundaries over a bed of bt = 0 (whose arrays the stage kernels do
not read), against the oracle, bit for bit: beds whose vertices agree across
the seam and beds whose do not, where the tiles either side each see their own
bed at the joined faces; both sub-block shapes and a 1D grid; a bed exchanged
under a state."""
import numpy as np
import pytest

from kestrel_amd import config as C
from kestrel_amd import scenario as S
from kestrel_amd.runtime import Stepper
from tests.helpers import FIELDS

pytestmark = pytest.mark.gpu

GRIDS = {"small": (3, 2, 16, 16), "wide": (6, 6, 32, 32), "wide_ragged": (8, 7, 50, 21), "oned": (5, 1, 12, 1)}


def _case(grid, joined):
    cfg = C.default_config(*GRIDS[grid], dx=1.0, dy=1.25)
    C.hydraulic_only(cfg)
    cfg.bc = C.BC_PERIODIC
    C.derive(cfg)
    rng = np.random.default_rng(7)
    b0v = 0.2 * rng.standard_normal((cfg.NY + 1, cfg.NX + 1))
    if joined:
        b0v[:, -1] = b0v[:, 0]
        b0v[-1, :] = b0v[0, :]
    # thin flow with dry gaps everywhere: many faces take the bed's slope
    shape = (cfg.NY, cfg.NX)
    depth = np.abs(rng.standard_normal(shape)) * (rng.uniform(size=shape) < 0.7) * 0.2
    b0c = S.cell_topography(cfg, b0v)[0]
    init = S.InitialState(b0c + depth, *(np.zeros(shape) for _ in range(3)),
                          np.full(cfg.ntiles, C.TILE_ACTIVE, np.uint8), np.zeros(shape))
    return cfg, b0v, init


def _run(make, cfg, b0v, init, n=6):
    g = make(cfg)
    g.set_topography(b0v)
    g.set_state(init)
    g.step_n(n)
    return g.state()


@pytest.mark.parametrize("joined", [True, False], ids=["joined", "unequal"])
@pytest.mark.parametrize("grid", GRIDS)
def test_periodic_flat_bed_equals_oracle(gpu, grid, joined):
    from oracle.oracle import Oracle
    cfg, b0v, init = _case(grid, joined)
    a, b = _run(Stepper, cfg, b0v, init), _run(Oracle, cfg, b0v, init)
    assert a["t"] == b["t"]
    for f in FIELDS:
        assert np.array_equal(a[f], b[f]), f"{grid}: {f}"


def test_bed_exchanged_under_a_state(gpu):
    from oracle.oracle import Oracle
    cfg, b0v, init = _case("wide", False)
    want = _run(Oracle, cfg, b0v, init)
    joined = b0v.copy()
    joined[:, -1] = b0v[:, 0]
    joined[-1, :] = joined[0, :]
    g = Stepper(cfg)
    g.set_topography(joined)
    g.set_state(init)
    g.set_topography(b0v)
    g.step_n(6)
    got = g.state()
    for f in FIELDS:
        assert np.array_equal(got[f], want[f]), f
