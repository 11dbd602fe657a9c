"""kst_set_state and kst_get_state move the row-major arrays through the
device's rearranging kernels: what goes in comes out, at sizes read back in
one copy (up to 1 MB) and array by array, in tiles that no block of threads
divides, with a bed."""
import numpy as np
import pytest

from kestrel_amd import config as C
from kestrel_amd import scenario as S
from kestrel_amd.runtime import Stepper

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles,tile", [((3, 3), (5, 7)), ((4, 5), (32, 32)), ((9, 7), (50, 33)), ((11, 1), (13, 1))])
def test_state_round_trip(gpu, tiles, tile):
    cfg = C.default_config(tiles[0], tiles[1], tile[0], tile[1], dx=2.0)
    C.hydraulic_only(cfg)
    cfg.bc = C.BC_SPONGE
    C.derive(cfg)
    rng = np.random.default_rng(5)
    shape, verts = (cfg.NY, cfg.NX), (cfg.NY + 1, cfg.NX + 1)
    b0v = rng.standard_normal(verts)
    btv = 0.1 * rng.standard_normal(verts)
    active = np.zeros((tiles[1], tiles[0]), np.uint8)
    active[tiles[1] // 2, tiles[0] // 2] = 1
    f = [rng.standard_normal(shape) for _ in range(4)]
    init = S.InitialState(*f, S._ghost_ring(cfg, active.reshape(-1)), np.abs(rng.standard_normal(shape)))
    g = Stepper(cfg)
    g.set_topography(b0v)
    g.set_state(init, t=3.5, btv=btv)
    st, mx, topo = g.state(), g.maxima(), g.cell_topography()
    g.close()
    tiles_of = S._tile_of_cells(cfg)
    state = init.tile_state[tiles_of]
    on, ghost = state == C.TILE_ACTIVE, state == C.TILE_GHOST
    assert st["t"] == 3.5 and np.array_equal(st["tile_state"], init.tile_state)
    for name, a in zip(("w", "rhoHnu", "rhoHnv", "Hnpsi"), f):
        assert np.array_equal(st[name][on], a[on]), name
        assert np.array_equal(st[name][ghost], topo["b0c"][ghost] if name == "w" else np.zeros(ghost.sum())), name
        assert not st[name][~on & ~ghost].any(), name
    gam = S.gamma(cfg, topo["dbdx"], topo["dbdy"])
    hn = (-topo["btc"] + (f[0] - topo["b0c"])) * gam
    assert np.array_equal(st["Hn"], np.where(on, np.maximum(hn, 0.0), 0.0))
    assert np.array_equal(mx[0], init.hnmax0) and (mx[10] == -1.0).all()
    b0c, btc, bx, by = S.cell_topography(cfg, b0v, btv)
    assert np.array_equal(topo["b0c"], b0c) and np.array_equal(topo["btc"][on], btc[on])
    assert np.array_equal(topo["dbdx"][on], bx[on])
    tj, ti = np.argwhere(active)[0]
    own = (slice(tj * tile[1], (tj + 1) * tile[1]), slice(ti * tile[0], (ti + 1) * tile[0]))
    assert np.array_equal(st["btv"][own], btv[own])
