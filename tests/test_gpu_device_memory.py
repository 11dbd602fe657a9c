"""Device memory: the staging of the boundary's arrays is one bounded buffer for
all handles of the device, given back with the last of them; what a scenario
holds lies within what the server's admission counts for it."""
import numpy as np
import pytest

from kestrel_amd import config as C
from kestrel_amd import serving, workloads
from tests.helpers import stepper_for

pytestmark = pytest.mark.gpu

MB = 1 << 20
STAGE = 64 * MB


def _used():
    import torch
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


def _warm():
    """Code objects, queues and scratch the first launches bring."""
    g = stepper_for(workloads.plain_cap(128, 0, tile=32, cap_x=0.0, cap_radius=10.0))
    g.step_n(2)
    g.state()
    g.close()


def test_staging_is_shared_and_given_back(gpu):
    from kestrel_amd.runtime import Stepper
    _warm()
    wl = workloads.plain_cap(2048, 0, tile=32, cap_x=0.0, cap_radius=100.0)
    start = _used()
    handles, grown = [], []
    for _ in range(2):
        g = Stepper(wl.cfg)
        created = _used()
        g.set_topography(wl.b0v)
        g.set_state(wl.init)
        g.state()
        g.maxima()
        g.cell_topography()
        handles.append(g)
        grown.append(_used() - created)
    assert grown[0] <= STAGE + 2 * MB and grown[1] <= 2 * MB, grown
    for g in handles:
        g.close()
    assert _used() - start <= 2 * MB


@pytest.mark.parametrize("tiles", [(61, 53, 31, 29), (85000, 1, 100, 1)], ids=["2d", "1d"])
def test_arrays_larger_than_the_staging(gpu, tiles):
    """Round trip in chunks: a state, its topography and maxima whose arrays
    do not fit the staging at once (1d: not even one of them)."""
    from kestrel_amd import scenario as S
    from kestrel_amd.runtime import Stepper
    cfg = C.default_config(*tiles, dx=2.0)
    C.hydraulic_only(cfg)
    cfg.bc = C.BC_SPONGE
    C.derive(cfg)
    rng = np.random.default_rng(3)
    shape, verts = (cfg.NY, cfg.NX), (cfg.NY + 1, cfg.NX + 1)
    b0v = rng.standard_normal(verts)
    btv = rng.standard_normal(verts)
    on = np.zeros((tiles[1], tiles[0]), np.uint8)
    on[(1 if tiles[1] > 1 else 0):(tiles[1] - 1 if tiles[1] > 1 else 1), 1:-1] = 1
    f = [rng.standard_normal(shape) for _ in range(4)]
    init = S.InitialState(*f, on.reshape(-1), np.abs(rng.standard_normal(shape)))
    g = Stepper(cfg)
    g.set_topography(b0v)
    g.set_state(init, t=1.5, btv=btv)
    active = init.tile_state[S._tile_of_cells(cfg)] == 1
    b0c, btc, bx, by = S.cell_topography(cfg, b0v, btv)
    st = g.state()
    assert st["t"] == 1.5
    for name, a in zip(("w", "rhoHnu", "rhoHnv", "Hnpsi"), f):
        assert np.array_equal(st[name][active], a[active]), name
    own = np.zeros(verts, bool)   # vertices read from an active tile's copy
    own[:-1, :-1] |= active
    own[-1, :-1] |= active[-1]
    assert np.array_equal(st["btv"][own], btv[own])
    topo = g.cell_topography()
    assert np.array_equal(topo["b0c"], b0c)
    assert np.array_equal(topo["btc"][active], btc[active])
    mx = g.maxima()
    assert np.array_equal(mx[0], init.hnmax0) and (mx[10] == -1.0).all()
    mx[3] = rng.standard_normal(shape)
    g.set_maxima(mx)
    assert np.array_equal(g.maxima()[3], mx[3])
    cells = rng.uniform(size=shape) < 0.5
    new = [rng.standard_normal(shape) for _ in range(3)]
    g.set_cell_topography(*new, cells)
    topo2 = g.cell_topography()
    for name, a in zip(("btc", "dbdx", "dbdy"), new):
        assert np.array_equal(topo2[name], np.where(cells, a, topo[name])), name
    g.close()


@pytest.mark.parametrize("kind,n,tile", [("fp64", 192, 16), ("fp64", 512, 32), ("fp64", 2048, 32), ("mixed", 256, 16),
                                         ("mixed", 512, 50), ("morpho", 256, 32), ("morpho", 1024, 32)])
def test_admission_counts_what_a_scenario_holds(gpu, kind, n, tile):
    _warm()
    keep = stepper_for(workloads.plain_cap(2048, 0, tile=32, cap_x=0.0, cap_radius=100.0))   # the staging at its largest
    if kind == "morpho":
        wl = workloads.morpho_cap(n, 0, tile=tile)
    else:
        wl = workloads.plain_cap(n // tile * tile, 0, tile=tile, cap_x=0.0, cap_radius=0.1 * n)
        wl.cfg.precision = C.PREC_MIXED if kind == "mixed" else C.PREC_FP64
    count = 4 if n <= 512 else 1
    before = _used()
    handles = [stepper_for(wl) for _ in range(count)]
    handles[0].state()
    held = (_used() - before) / count
    for g in handles + [keep]:
        g.close()
    counted = serving.device_bytes(wl.cfg)
    assert held <= counted <= 1.3 * held + 4 * MB, (held, counted)


def test_staging_shared_by_threads(gpu):
    """Two threads with a handle each, one of whose arrays make the shared
    staging grow: each reads back what it set, whatever the other does."""
    import threading

    from kestrel_amd import scenario as S
    from kestrel_amd.runtime import Stepper
    failed = []

    def work(tiles, tile, seed):
        cfg = C.default_config(tiles, tiles, tile, tile)
        C.hydraulic_only(cfg)
        cfg.bc = C.BC_PERIODIC
        C.derive(cfg)
        rng = np.random.default_rng(seed)
        shape = (cfg.NY, cfg.NX)
        g = Stepper(cfg)
        for k in range(12):
            b0v = rng.standard_normal((cfg.NY + 1, cfg.NX + 1))
            f = [rng.standard_normal(shape) for _ in range(5)]
            g.set_topography(b0v)
            g.set_state(S.InitialState(*f[:4], np.ones(cfg.ntiles, np.uint8), f[4]))
            st = g.state()
            ok = all(np.array_equal(st[n], a) for n, a in zip(("w", "rhoHnu", "rhoHnv", "Hnpsi"), f))
            if not (ok and np.array_equal(g.maxima()[0], f[4])):
                failed.append((tiles, k))
        g.close()

    threads = [threading.Thread(target=work, args=a) for a in ((5, 31, 1), (40, 37, 2))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
