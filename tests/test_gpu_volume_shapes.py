"""kst_volume at the tile shapes and set sizes where its loops and its
reduction end: fewer cells than a wavefront, cells that four loads a thread do
not divide, one active tile, and more active tiles than partial sums.  The bar
is the one of the other volume tests: one ulp of the exact sum of the device's
own per-cell terms."""
import math

import numpy as np
import pytest

from kestrel_amd import config as C
from kestrel_amd import scenario as S
from kestrel_amd.runtime import Stepper
from tests.test_gpu_output import device_terms, ulps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,tile,tile_y,radius,bed", [
    (6, 4, 4, 0.0, False),        # 16 cells a tile, the smallest
    (5, 7, 37, 0.0, True),        # 259 cells
    (3, 32, 33, 0.0, False),      # 1056 cells: a second turn of 32 cells
    (5, 46, 46, 3.0, True),       # one active tile
    (50, 5, 5, 0.0, True),        # 2304 active tiles, 2048 partial sums
])
def test_volume_shapes(gpu, n, tile, tile_y, radius, bed):
    cfg = C.default_config(n, n, tile, tile_y, dx=1.0, dy=1.0)
    C.hydraulic_only(cfg)
    cfg.bc = C.BC_SPONGE
    C.derive(cfg)
    rng = np.random.default_rng(5)
    b0v = S.topo_xslope(cfg, 0.1) + 0.1 * rng.standard_normal((cfg.NY + 1, cfg.NX + 1))
    btv = 0.05 * rng.standard_normal(b0v.shape) if bed else None
    r = radius or float(np.hypot(cfg.x_size, cfg.y_size))
    init = S.initial_state(cfg, b0v, [S.Cap(0.0, 0.0, r, 1.0, psi=0.3)])
    if bed:
        init.w = init.w + S.cell_topography(cfg, b0v, btv)[1]
    g = Stepper(cfg)
    g.set_topography(b0v)
    g.set_state(init, btv=btv)
    st = g.state()
    assert int((st["tile_state"] == 1).sum()) == (1 if radius else (n - 2) ** 2)   # none on the domain edge
    t = device_terms(g, cfg, st)
    v = g.volume()
    for col, q, scale in ((0, 0, 1.0), (2, 1, 1.0), (4, 3, cfg.rhos)):
        exact = math.fsum(t[q])
        assert ulps(v[col] / scale, exact, exact) <= 1, (col, v[col], exact)
    assert abs(v[1] - math.fsum(t[2])) <= 2 * math.ulp(float(np.abs(t[2]).sum()))
    g.close()
