"""The wide stage kernels (active sets of at least 128 sub-blocks of 16 x 16) against
the oracle, bit for bit (only +, -, x, / and square roots are evaluated):
tiles that the sub-blocks divide and tiles that leave remainders, clear water
and solids in part of the domain (the face pass leaves Hnpsi out where a
sub-block's region carries none), a bed of bt = 0 (its arrays are not read)
and one that differs from 0, and non-active neighbours on every side."""
import numpy as np
import pytest

from kestrel_amd import config as C
from kestrel_amd import scenario as S
from kestrel_amd.runtime import Stepper
from tests.helpers import FIELDS, active_mask

pytestmark = pytest.mark.gpu

CASES = {
    "tile32_water": dict(tile=32, n=12, psi=0.0),
    "tile32_solids": dict(tile=32, n=12, psi=0.3),
    "tile32_bed": dict(tile=32, n=12, psi=0.3, bed=True),
    "tile50_water": dict(tile=50, n=8, psi=0.0),
    "tile50_solids_eddy": dict(tile=50, n=8, psi=0.3, eddy=1e-2),
    "tile21_bed": dict(tile=21, n=12, psi=0.0, bed=True),
    "tile9x37": dict(tile=9, tile_y=37, n=26, ny=7, psi=0.2),
}


@pytest.mark.parametrize("name", CASES)
def test_wide_stage_kernels_equal_oracle(gpu, name):
    from oracle.oracle import Oracle
    k = CASES[name]
    cfg = C.default_config(k["n"], k.get("ny", k["n"]), k["tile"], k.get("tile_y", k["tile"]), dx=1.0, dy=1.25)
    C.hydraulic_only(cfg)
    cfg.bc = C.BC_SPONGE    # a flow that reaches the domain's edge tiles does not halt
    cfg.eddy_viscosity = k.get("eddy", 0.0)
    C.derive(cfg)
    rng = np.random.default_rng(11)
    b0v = S.topo_xslope(cfg, 0.15) + 0.2 * rng.standard_normal((cfg.NY + 1, cfg.NX + 1))
    r = 0.24 * min(cfg.x_size, cfg.y_size)
    # two caps: one carries the solids, the other (and the rest) is clear water
    caps = [S.Cap(-0.4 * r, 0.0, r, 1.0, psi=k["psi"]), S.Cap(0.8 * r, 0.3 * r, 0.5 * r, 0.7)]
    init = S.initial_state(cfg, b0v, caps)
    btv = None
    if k.get("bed"):
        btv = 0.05 * rng.standard_normal((cfg.NY + 1, cfg.NX + 1))
        init.w = init.w + S.cell_topography(cfg, b0v, btv)[1]   # the flow lies on the changed bed
    g = Stepper(cfg)
    g.set_topography(b0v)
    g.set_state(init, btv=btv)
    o = Oracle(cfg)
    o.set_topography(b0v)
    o.set_state(init, btv=btv)
    active = int((init.tile_state == 1).sum())
    assert active * (-(-cfg.nx_per_tile // 16)) * (-(-cfg.ny_per_tile // 16)) >= 128, "the wide kernels must run"
    so, sg = o.step_n(8), g.step_n(8)
    assert (sg["steps"], sg["rejected"]) == (so["steps"], so["rejected"])
    a, b = g.state(), o.state()
    assert a["t"] == b["t"] and np.array_equal(a["tile_state"], b["tile_state"])
    m = active_mask(cfg, b["tile_state"])
    for f in FIELDS:
        assert np.array_equal(a[f][m], b[f][m]), f"{name}: {f}"
    g.close()
