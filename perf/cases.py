"""The work that users of the time step have it do, as measurable cases.

A case is one call sequence of a user's program through kestrel_amd.runtime:

  run       a simulation from its initial conditions to an output time on a
            handle that holds the grid: set_state, step_n, state (and the
            running maxima, the hazard map, where "maxima" is set)
  interval  one output interval of a long simulation that stays resident:
            step_n, then the solution file's columns and the Volume.txt sums;
            periodic boundaries, so that it may go on without end
  ensemble  scenarios of different sizes taken up by one batch, advanced
            together and read back
  volume    the Volume.txt sums of a resident state alone

listed() names the measured ones, draw(rng) gives others of the same ranges.
exact() restates the hydraulic step in plain torch, in 64 bits.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from kestrel_amd import config as C
from kestrel_amd import scenario as S
from kestrel_amd.runtime import Batch, Stepper


def listed() -> list:
    return [
        # The smallest call: a few steps on one 40 x 40 tile of a periodic
        # lake (the grid of the lake-at-rest deck), read back each time, as a
        # host program does that couples to another model step by step.
        _case("interval", name="lake_40_8_steps", tiles_x=1, tiles_y=1, tile_x=40, tile_y=40, steps=8),
        # A one-dimensional cap release, 100-cell tiles of one row (the 1D
        # decks' layout), Voellmy drag.
        _case("run", name="cap_1d_3000", tiles_x=30, tiles_y=1, tile_x=100, tile_y=1, dx=1.0, steps=400,
              radius=60.0, drag="voellmy", slope=5.0),
        # The plain cap release at 256 x 256 cells, 1000 steps, with the
        # hazard map: the ordinary small run.
        _case("run", name="cap_256_1000_steps", tiles_x=8, tiles_y=8, tile_x=32, tile_y=32, dx=1.0, steps=1000,
              radius=20.0, slope=10.0, max_dt=0.05, maxima=True),
        # A flux source on the 2D decks' 50 x 50 tiles (not a multiple of any
        # block of threads), concentrated flow, variable drag, eddy viscosity.
        _case("run", name="flux_tiles_of_50", tiles_x=12, tiles_y=12, tile_x=50, tile_y=50, dx=1.0, steps=400,
              flux=20.0, psi=0.3, drag="variable", eddy=1e-2, slope=12.0),
        # A dilute cap over many 50 x 50 tiles: the large ragged run.
        _case("run", name="cap_wide_tiles_of_50", tiles_x=30, tiles_y=30, tile_x=50, tile_y=50, dx=1.0, steps=300,
              radius=450.0, slope=10.0),
        # The plain path at 2048 x 2048, about 1.6 M active cells: a full chip.
        _case("run", name="cap_2048", tiles_x=64, tiles_y=64, tile_x=32, tile_y=32, dx=1.0, steps=600,
              radius=700.0, slope=10.0, max_dt=0.05),
        # The same physics in mixed precision at 1024 x 1024.
        _case("run", name="cap_1024_mixed", tiles_x=32, tiles_y=32, tile_x=32, tile_y=32, dx=1.0, steps=300,
              radius=300.0, slope=10.0, precision="mixed"),
        # A small morphodynamic release (erosion, deposition, redistribution)
        # on 50 x 50 tiles.
        _case("run", name="morpho_cap_tiles_of_50", tiles_x=8, tiles_y=8, tile_x=50, tile_y=50, dx=1.0, steps=200,
              radius=12.0, psi=0.1, drag="variable", slope=11.0, morpho=True),
        # The morphodynamic flow from a source over Gaussian hills, 1024 x
        # 1024 cells of 5 m, eddy viscosity: a few active tiles, many steps.
        _case("run", name="morpho_hills_1024", tiles_x=32, tiles_y=32, tile_x=32, tile_y=32, dx=5.0, steps=600,
              flux=100.0, psi=0.3, drag="pouliquen", eddy=1e-2, hills=32, slope=5.0, morpho=True),
        # A wide morphodynamic release over hills: hundreds of active tiles
        # and thousands of redistribution candidates.
        _case("run", name="morpho_wide_1024", tiles_x=32, tiles_y=32, tile_x=32, tile_y=32, dx=5.0, steps=40,
              radius=1200.0, psi=0.2, drag="variable", hills=32, slope=5.0, morpho=True),
        # An ensemble of sixteen scenarios with their own grids, caps and drag
        # in one batch, mixed precision (the ensemble's own).
        _case("ensemble", name="ensemble_16_mixed", scenarios=16, side_lo=128, side_hi=640, steps=100,
              precision="mixed"),
        # One Volume.txt line of the 2048 x 2048 run.
        _case("volume", name="volume_2048", tiles_x=64, tiles_y=64, tile_x=32, tile_y=32, radius=700.0, slope=10.0),
    ]


_DEFAULTS = dict(tiles_x=8, tiles_y=8, tile_x=32, tile_y=32, dx=1.0, steps=1, radius=0.0, flux=0.0, psi=0.0,
                 slope=0.0, hills=0, drag="chezy", eddy=0.0, limiter="minmod2", precision="fp64", morpho=False,
                 maxima=False, scenarios=0, side_lo=0, side_hi=0, bc="halt", max_dt=10.0)


def _case(kind: str, name: str | None = None, **kw) -> dict:
    c = dict(_DEFAULTS, kind=kind, **kw)
    if name is not None:
        c["name"] = name
    return c


def _log(rng, lo: float, hi: float) -> float:
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng) -> dict:
    """One more case: the kinds as often as listed, sizes over their ranges
    (with sponge boundaries, where a flow that reaches the edge does not halt)."""
    return dict(_drawn(rng), bc="sponge")


def _drawn(rng) -> dict:
    kind = rng.choice(["interval", "line", "cap", "cap", "flux", "mixed", "morpho", "hills", "wide", "ensemble",
                       "volume"])
    tile = rng.choice([16, 20, 25, 32, 32, 40, 50, 50])
    if kind == "interval":
        n = max(1, int(_log(rng, 1, 400) / tile))
        return _case("interval", tiles_x=n, tiles_y=rng.randint(1, max(1, n)), tile_x=tile, tile_y=tile,
                     steps=int(_log(rng, 1, 60)), limiter=rng.choice(["minmod2", "minmod1", "vanalbada"]))
    if kind == "line":
        tile = rng.choice([50, 100, 101, 128])
        n = max(6, int(_log(rng, 600, 20000) / tile))
        return _case("run", tiles_x=n, tiles_y=1, tile_x=tile, tile_y=1, steps=int(_log(rng, 50, 500)),
                     radius=n * tile * rng.uniform(0.01, 0.15), drag=rng.choice(["voellmy", "chezy", "manning"]),
                     slope=rng.uniform(2, 12))
    if kind in ("cap", "mixed"):
        n = max(6, int(_log(rng, 150, 1800) / tile))
        size = n * tile
        return _case("run", tiles_x=n, tiles_y=max(6, int(n * rng.uniform(0.7, 1.0))), tile_x=tile,
                     tile_y=rng.choice([tile, tile, max(8, tile - 3)]), dx=rng.choice([1.0, 1.0, 2.5]),
                     steps=int(_log(rng, 60, 500 if size < 900 else 250)),
                     radius=-rng.uniform(0.05, min(0.28, 0.4 - 2.0 / n)),
                     psi=rng.choice([0.0, 0.0, 0.25]), drag=rng.choice(["chezy", "voellmy", "variable", "manning"]),
                     slope=rng.uniform(4, 14), limiter=rng.choice(["minmod2", "minmod2", "minmod1"]),
                     maxima=size < 500 and rng.random() < 0.5, precision="mixed" if kind == "mixed" else "fp64")
    if kind == "flux":
        n = max(7, int(_log(rng, 150, 800) / tile))
        return _case("run", tiles_x=n, tiles_y=n, tile_x=tile, tile_y=tile, steps=int(_log(rng, 100, 600)),
                     flux=rng.uniform(4, 30), psi=rng.choice([0.0, 0.3]), slope=rng.uniform(5, 14),
                     drag=rng.choice(["chezy", "variable", "pouliquen"]), eddy=rng.choice([0.0, 1e-2]))
    if kind == "morpho":
        n = max(7, int(_log(rng, 150, 500) / tile))
        return _case("run", tiles_x=n, tiles_y=n, tile_x=tile, tile_y=tile, steps=int(_log(rng, 40, 250)),
                     radius=-rng.uniform(0.03, 0.08), psi=rng.uniform(0.05, 0.35), slope=rng.uniform(6, 13),
                     drag=rng.choice(["chezy", "variable", "pouliquen"]), morpho=True,
                     eddy=rng.choice([0.0, 1e-2]))
    if kind == "hills":
        n = int(_log(rng, 400, 1024) / tile)
        return _case("run", tiles_x=n, tiles_y=n, tile_x=tile, tile_y=tile, dx=5.0, steps=int(_log(rng, 150, 600)),
                     flux=rng.uniform(50, 150), psi=0.3, drag="pouliquen", eddy=1e-2, hills=32, slope=5.0, morpho=True)
    if kind == "wide":
        n = int(_log(rng, 350, 1000) / tile)
        return _case("run", tiles_x=n, tiles_y=n, tile_x=tile, tile_y=tile, dx=5.0, steps=rng.randint(10, 40),
                     radius=-rng.uniform(0.1, 0.22), psi=rng.uniform(0.1, 0.3), drag="variable", hills=32, slope=5.0,
                     morpho=True)
    if kind == "ensemble":
        return _case("ensemble", scenarios=rng.randint(4, 20), side_lo=128, side_hi=rng.choice([256, 384, 640]),
                     steps=int(_log(rng, 20, 100)), precision=rng.choice(["mixed", "fp64"]))
    n = max(4, int(_log(rng, 200, 2048) / tile))
    return _case("volume", tiles_x=n, tiles_y=n, tile_x=tile, tile_y=tile, radius=-rng.uniform(0.1, 0.34),
                 slope=rng.uniform(4, 14), psi=rng.choice([0.0, 0.2]))


# ---------------------------------------------------------------------------
# inputs: the bed at the vertices and the painted initial state
# ---------------------------------------------------------------------------

def _sum4(a, b, c, d):
    """Compensated sum of four arrays, as the step sums a cell's vertices (so
    that a dry cell's free surface is its bed to the last bit)."""
    s, k = a, np.zeros_like(a)
    for x in (b, c, d):
        y = x - k
        t = s + y
        k = (t - s) - y
        s = t
    return s


def _members(case: dict) -> list:
    """An ensemble's scenarios as cases of their own; else the case itself.
    The sizes are the case's, not the seed's: the work of every seed is alike."""
    if case["kind"] != "ensemble":
        return [case]
    out = []
    k = case["scenarios"]
    for q in range(k):
        side = int(round(case["side_lo"] * (case["side_hi"] / case["side_lo"]) ** (q / max(1, k - 1)) / 32)) * 32
        out.append(dict(case, kind="run", tiles_x=side // 16, tiles_y=side // 16, tile_x=16, tile_y=16, dx=5.0,
                        radius=-0.06, slope=2.0, hills=16, drag="chezy", member=q))
    return out


def _inputs(case: dict, seed: int) -> dict:
    """Bed, painted fields and active tiles of a case, in plain numpy."""
    rng = np.random.default_rng([int(seed), int(case.get("member", 0)), 7])
    nx, ny, dx = case["tiles_x"] * case["tile_x"], case["tiles_y"] * case["tile_y"], case["dx"]
    lx, ly = nx * dx, ny * dx
    oned = ny == 1
    xv = -0.5 * lx + dx * np.arange(nx + 1)
    yv = -0.5 * ly + dx * np.arange(ny + 1)
    x, y = xv[:-1] + 0.5 * dx, yv[:-1] + 0.5 * dx
    if case["kind"] == "interval":
        # a bed of whole waves, so that it is the same on both sides of the domain
        kx, ky = rng.integers(1, 4, 2)
        px, py = rng.uniform(0, 2 * math.pi, 2)
        bv = 0.15 * (np.sin(2 * math.pi * kx * xv / lx + px)[None, :] + np.sin(2 * math.pi * ky * yv / ly + py)[:, None])
        bv[:, -1] = bv[:, 0]
        bv[-1, :] = bv[0, :]
    else:
        bv = np.broadcast_to(math.tan(math.radians(case["slope"])) * xv[None, :], (ny + 1, nx + 1)).copy()
        width = (0.01 * lx, 0.06 * lx)
        for _ in range(case["hills"]):
            amp, s = rng.uniform(0.02, 0.2) * width[1], rng.uniform(*width)
            cx, cy = rng.uniform(-0.5 * lx, 0.5 * lx), rng.uniform(-0.5 * ly, 0.5 * ly)
            bv += amp * np.exp(-((xv - cx) ** 2) / (2 * s * s))[None, :] * np.exp(-((yv - cy) ** 2) / (2 * s * s))[:, None]
    if oned:
        b = 0.5 * (bv[:1, :-1] + bv[:1, 1:])
        gam = np.sqrt(1.0 + ((bv[:1, 1:] - bv[:1, :-1]) / dx) ** 2)
    else:
        v00, v10, v01, v11 = bv[:-1, :-1], bv[:-1, 1:], bv[1:, :-1], bv[1:, 1:]
        b = 0.25 * _sum4(v00, v10, v01, v11)
        gx, gy = 0.5 * (v10 - v00 + v11 - v01) / dx, 0.5 * (v01 - v00 + v11 - v10) / dx
        gam = np.sqrt(1.0 + gx * gx + gy * gy)
    out = dict(bv=bv, w=b.copy(), hpsi=np.zeros_like(b), ru=np.zeros_like(b), rv=np.zeros_like(b), hn=np.zeros_like(b))
    wet = None
    if case["kind"] == "interval":
        # a lake over the bed with waves on it
        amp = rng.uniform(0.05, 0.15)
        mx, my = rng.integers(1, 4, 2)
        level = 1.0 + amp * np.cos(2 * math.pi * mx * x / lx + rng.uniform(0, 6))[None, :] \
            * np.cos(2 * math.pi * my * y / ly + rng.uniform(0, 6))[:, None]
        out["w"], out["hn"] = level, (level - b) * gam
        active = np.ones((case["tiles_y"], case["tiles_x"]), bool)
    else:
        # a paraboloid cap clear of the domain's edge, or a flux source
        cx, cy = rng.uniform(0.03, 0.08) * lx, 0.0 if oned else rng.uniform(-0.03, 0.03) * ly
        r = case["radius"] if case["radius"] >= 0 else -case["radius"] * min(lx, lx if oned else ly)
        if case["flux"] > 0:
            cx = cx + 0.12 * lx
            cx, cy = float(x[np.argmin(abs(x - cx))]), float(y[np.argmin(abs(y - cy))])
            r = 0.4 * dx
            out["source"] = (cx, cy, r, case["flux"] * rng.uniform(0.9, 1.1), case["psi"])
        r2 = (x[None, :] - cx) ** 2 + (0.0 if oned else (y[:, None] - cy) ** 2)
        wet = r2 <= r * r
        if case["flux"] == 0:
            h = np.where(wet, max(1.0, 0.004 * r) * rng.uniform(0.8, 1.2) * (1.0 - r2 / (r * r)), 0.0)
            out["hn"], out["hpsi"] = h, case["psi"] * h
            out["w"] = np.where(wet, b + h / gam, b)
        active = wet.reshape(case["tiles_y"], case["tile_y"], case["tiles_x"], case["tile_x"]).any(axis=(1, 3))
    out["cells"] = int(wet.sum()) if wet is not None else nx * ny
    out["active"] = active
    if case["kind"] == "run" and case["hills"] and case["scenarios"]:
        out["chezy"] = float(rng.uniform(0.005, 0.05))
    return out


def _config(case: dict, inp: dict):
    cfg = C.default_config(case["tiles_x"], case["tiles_y"], case["tile_x"], case["tile_y"], dx=case["dx"])
    if not case["morpho"]:
        C.hydraulic_only(cfg)
    cfg.bc = C.BCS["periodic" if case["kind"] == "interval" else case["bc"]]
    cfg.max_dt = case["max_dt"]
    cfg.limiter = C.LIMITERS[case["limiter"]]
    cfg.drag = C.DRAGS[case["drag"]]
    cfg.chezy_co = inp.get("chezy", 0.01)
    cfg.eddy_viscosity = case["eddy"]
    cfg.precision = C.PREC_MIXED if case["precision"] == "mixed" else C.PREC_FP64
    C.derive(cfg)
    if "source" in inp:
        x, y, r, q, psi = inp["source"]
        src = C.FluxSource(x, y, r, [0.0, 1.0e9], [q, q], [psi, psi])
        src.num_cells = 1
        C.set_sources(cfg, [src])
    return cfg


def _stepper(case: dict, seed: int):
    inp = _inputs(case, seed)
    cfg = _config(case, inp)
    tiles = np.where(inp["active"].reshape(-1), C.TILE_ACTIVE, C.TILE_OFF).astype(np.uint8)
    init = S.InitialState(inp["w"], inp["ru"], inp["rv"], inp["hpsi"], tiles, inp["hn"])
    g = Stepper(cfg)
    g.set_topography(inp["bv"])
    g.set_state(init)
    return g, init


def prepare(case: dict, seed: int) -> dict:
    """The handles with their grids and topography, and the initial states."""
    members = [_stepper(m, seed) for m in _members(case)]
    st = dict(case=case, members=members)
    if case["kind"] == "ensemble":
        st["batch"] = Batch(len(members))
    return st


_FIELDS = ("w", "rhoHnu", "rhoHnv", "Hnpsi", "Hn", "btv", "tile_state", "t")


def run(state: dict):
    case, members = state["case"], state["members"]
    g, init = members[0]
    if case["kind"] == "volume":
        return g.volume()
    if case["kind"] == "interval":
        g.step_n(case["steps"])
        tiles, fields = g.output_fields()
        return {"tiles": tiles, "fields": fields, "volume": g.volume()}
    if case["kind"] == "ensemble":
        batch = state["batch"]
        slots = []
        for m, m0 in members:
            m.set_state(m0)
            slots.append(batch.attach(m))
            batch.start(slots[-1], nsteps=case["steps"])
        batch.run()
        out = []
        for s, (m, _) in zip(slots, members):
            batch.detach(s)
            st = m.state()
            out.append([st["w"], st["rhoHnu"], st["rhoHnv"]])
        return out
    g.set_state(init)
    g.step_n(case["steps"])
    out = g.state()
    if case["maxima"]:
        out["maxima"] = g.maxima()
    return out


def work(case: dict) -> dict:
    """Bytes and operations of the stage-pass model: per active cell and step
    42 words of 8 bytes over the four Runge-Kutta passes (134 for the Strang
    step) and about 600 operations a pass (8 + 3 of them in a Strang step);
    the initial state in (4 fields) and the result out (5 fields, or the
    file's 14 columns) once; half the words in mixed precision's stages."""
    if case["kind"] == "volume":
        n = _active_cells(case)
        return {"bytes": 40.0 * n, "flops": 60.0 * n}
    total_b = total_f = 0.0
    for m in _members(case):
        n = _active_cells(m)
        grid = m["tiles_x"] * m["tile_x"] * m["tiles_y"] * m["tile_y"]
        words = 134.0 if m["morpho"] else (26.0 if m["precision"] == "mixed" else 42.0)
        total_b += m["steps"] * n * words * 8.0
        total_f += m["steps"] * n * (11 if m["morpho"] else 4) * 600.0
        total_b += grid * 8.0 * (15 if m["kind"] == "interval" else (22 if m["maxima"] else 9))
    return {"bytes": total_b, "flops": total_f}


def _active_cells(case: dict) -> float:
    """Cells of the tiles that the initial condition touches."""
    return float(_inputs(case, 1)["active"].sum()) * case["tile_x"] * case["tile_y"]


# ---------------------------------------------------------------------------
# the hydraulic step in plain torch, 64 bits
# ---------------------------------------------------------------------------

class _Plain:
    """The adaptive SSP-RK3 step over the whole grid at once.  Arrays are
    (NY, NX); a face array holds each cell's west (x) or south (y) face."""

    def __init__(self, case, inp):
        cfg = {"g": 9.81, "rhow": 1000.0, "rhos": 2000.0, "chezy": inp.get("chezy", 0.01), "coulomb": 0.1,
               "manning": 0.03, "pmin": 0.1, "pmax": 0.4, "pbeta": 0.136, "rate": 3.0, "value": 0.2,
               "max_pack": 0.65, "diam": 1e-3, "cfl": 0.25, "thr": 1e-6}
        self.c, self.case, self.inp = cfg, case, inp
        self.nx, self.ny = case["tiles_x"] * case["tile_x"], case["tiles_y"] * case["tile_y"]
        self.oned = self.ny == 1
        dev = "cuda" if torch.cuda.is_available() and self.nx * self.ny > 20000 else "cpu"
        T = self.T = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=dev)
        self.dx, self.nu = case["dx"], case["eddy"]
        self.w, self.ru, self.rv, self.h = (T(inp[k]) for k in ("w", "ru", "rv", "hpsi"))
        self.active = torch.as_tensor(inp["active"], device=dev)
        v = T(inp["bv"])[: self.ny, : self.nx]     # south-west vertices; the rest by wrapping
        e, n, ne = self.at(v, 1, 1), self.at(v, 1, 0), self.at(self.at(v, 1, 1), 1, 0)
        dx = self.dx
        if self.oned:
            self.b, self.bx = 0.5 * (v + e), (e - v) / dx
            self.by = torch.zeros_like(v)
            self.faces = {1: (v, torch.zeros_like(v), 0.5 * (e - self.at(v, -1, 1)) / dx)}
        else:
            self.b = 0.25 * (v + e + n + ne)
            self.bx, self.by = 0.5 * (e - v + ne - n) / dx, 0.5 * (n - v + ne - e) / dx
            west, nwest = self.at(v, -1, 1), self.at(n, -1, 1)
            south, seast = self.at(v, -1, 0), self.at(e, -1, 0)
            # per axis: face bed, slope along the face, slope across it
            self.faces = {1: (0.5 * (v + n), (n - v) / dx, 0.25 * (e + ne - west - nwest) / dx),
                          0: (0.5 * (v + e), (e - v) / dx, 0.25 * (n + ne - south - seast) / dx)}
        self.gam = torch.sqrt(1.0 + self.bx ** 2 + self.by ** 2)
        self.source = None
        if "source" in inp:
            x, y, r, q, psi = inp["source"]
            X = (torch.arange(self.nx, device=dev) + 0.5) * dx - 0.5 * self.nx * dx
            Y = (torch.arange(self.ny, device=dev) + 0.5) * dx - 0.5 * self.ny * dx
            inside = ((X[None, :] - x) ** 2 + (Y[:, None] - y) ** 2 < r * r).double()
            self.source = (inside * q / dx / dx, inside * psi * q / dx / dx)
        self.flags = self.near(self.depth(self.w))

    @staticmethod
    def at(a, k, axis):
        """The value k cells along the axis."""
        return torch.roll(a, -k, axis)

    def depth(self, w):
        return torch.clamp((w - self.b) * self.gam, min=0.0)

    def cells(self, tiles):
        return tiles.repeat_interleave(self.case["tile_y"], 0).repeat_interleave(self.case["tile_x"], 1)

    def near(self, hn):
        """Tiles beside an active tile whose edge cells toward them are wet."""
        ty, tx, sy, sx = self.case["tiles_y"], self.case["tiles_x"], self.case["tile_y"], self.case["tile_x"]
        wet = ((hn > self.c["thr"]) & self.cells(self.active)).reshape(ty, sy, tx, sx)
        new = torch.zeros_like(self.active)
        for edge, k, axis in ((wet[:, :, :, -1].any(1), 1, 1), (wet[:, :, :, 0].any(1), -1, 1),
                              (wet[:, -1].any(2), 1, 0), (wet[:, 0].any(2), -1, 0)):
            if not (self.oned and axis == 0):
                new |= torch.roll(edge, k, axis)
        return new

    def limit(self, a, b):
        kind = self.case["limiter"]
        if kind == "vanalbada":
            den = a * a + b * b
            return torch.where(den == 0, 0.0, (a * a * b + a * b * b) / torch.where(den == 0, 1.0, den))
        m = torch.minimum(a.abs(), b.abs())
        if kind == "minmod2":
            m = torch.minimum(1.3 * m, 0.5 * (a + b).abs())
        return torch.where(a * b <= 0, 0.0, torch.copysign(m, a))

    def slope(self, q, axis, mask=True):
        s = self.limit(self.at(q, 1, axis) - q, q - self.at(q, -1, axis)) / self.dx
        return torch.where(self.act, s, 0.0) if mask else s

    def drag(self, hn, u, v, psi, speed2):
        c, kind = self.c, self.case["drag"]
        g = c["g"] / self.gam
        chezy = c["chezy"] * speed2
        if kind == "chezy":
            return chezy
        if kind == "voellmy":
            return chezy + c["coulomb"] * g * hn
        safe = torch.where(hn > c["thr"], hn, 1.0)
        if kind == "manning":
            return g * c["manning"] ** 2 / safe ** (1.0 / 3.0)
        number = torch.sqrt(speed2) / torch.sqrt(g * safe) * c["diam"] / safe
        pouliquen = (c["pmin"] + (c["pmax"] - c["pmin"]) * number / (c["pbeta"] + number)) * g * hn
        if kind == "pouliquen":
            return torch.where(speed2 > 0, pouliquen, 0.0)
        f = 0.5 * (1.0 + torch.tanh(c["rate"] * (psi - c["value"])))
        return chezy * (1.0 - f) + torch.where(speed2 > 0, pouliquen, 0.0) * f

    def rhs(self, w, ru, rv, h):
        """Rates of w, rho Hn u, rho Hn v, Hn psi, the drag factor, the CFL
        minimum, and the velocities and depth."""
        c, dx, act = self.c, self.dx, self.act
        hn = torch.where(act, self.depth(w), 0.0)
        den = hn * hn + torch.clamp(hn * hn, min=c["thr"] ** 2)
        psi = torch.clamp(2.0 * hn * torch.clamp(h, min=0.0) / den, max=c["max_pack"])
        rho = c["rhow"] + (c["rhos"] - c["rhow"]) * psi
        u = 2.0 * hn * ru / den / rho
        v = torch.zeros_like(u) if self.oned else 2.0 * hn * rv / den / rho
        ew, eu, ev, eh = (torch.zeros_like(w) for _ in range(4))
        cfl = torch.full((), math.inf, device=w.device, dtype=torch.float64)
        for axis, (fb, along, across) in self.faces.items():
            fg = torch.sqrt(1.0 + along ** 2 + across ** 2)
            at = lambda a: self.at(a, -1, axis)          # noqa: E731  the cell on the face's low side
            east = self.at(fb, 1, axis)
            sw = self.slope(w, axis, False)
            hi, lo = w + 0.5 * dx * sw, w - 0.5 * dx * sw
            below = (hi < east) | (lo < fb)
            wl = at(torch.where(below, w + 0.5 * (east - fb), hi))
            wr = torch.where(below, w + 0.5 * (fb - east), lo)
            sh = 0.5 * dx * self.slope(h, axis)
            below = (h + sh < 0) | (h - sh < 0)
            hl, hr = at(torch.where(below, h, h + sh)), torch.where(below, h, h - sh)
            su, sv, sr = self.slope(u, axis), self.slope(v, axis), self.slope(rho, axis)
            ul, ur = at(u + 0.5 * dx * su), u - 0.5 * dx * su
            vl, vr = at(v + 0.5 * dx * sv), v - 0.5 * dx * sv
            rl, rr = at(rho + 0.5 * dx * sr), rho - 0.5 * dx * sr
            Hl, Hr = (wl - fb) * fg, (wr - fb) * fg
            ql, qr = rl * Hl * ul, rr * Hr * ur
            if self.oned:                                # the line keeps the conserved rho Hn v
                s = 0.5 * dx * self.slope(rv, axis)
                pl, pr = at(rv + s), rv - s
            else:
                pl, pr = rl * Hl * vl, rr * Hr * vr
            nl, nr = (ul, ur) if axis == 1 else (vl, vr)
            k = c["g"] * (1.0 + along ** 2) / fg ** 3
            cl, cr = torch.sqrt(k * torch.clamp(Hl, min=0.0)), torch.sqrt(k * torch.clamp(Hr, min=0.0))
            ap = torch.clamp(torch.maximum(nr + cr, nl + cl), min=0.0)
            an = torch.clamp(torch.minimum(nr - cr, nl - cl), max=0.0)
            mine = act | at(act)
            for a, gam in ((ap, at(self.gam)), (-an, self.gam)):
                t = torch.clamp(gam / fg, max=1.0) ** 2 * dx / a
                cfl = torch.minimum(cfl, torch.where(mine & (a > 2.220446049250313e-16), t, math.inf).min())
            dif = ap - an
            some = dif >= 1e-10
            inv = torch.where(some, 1.0 / torch.where(some, dif, 1.0), 0.0)
            flux = lambda l, r, fl, fr: ((r - l) * ap * an + ap * fl - an * fr) * inv   # noqa: E731
            hyl, hyr = 0.5 * c["g"] * rl * (wl - fb) ** 2, 0.5 * c["g"] * rr * (wr - fb) ** 2
            out = lambda f: f - self.at(f, 1, axis)      # noqa: E731  in minus out
            ew = ew + out(flux(Hl * fg, Hr * fg, Hl * nl * fg, Hr * nr * fg)) / dx / self.gam ** 2
            eh = eh + out(flux(hl * fg, hr * fg, hl * nl * fg, hr * nr * fg)) / dx / self.gam
            hyd = out((ap * hyl - an * hyr) * inv)
            du, dv = out(flux(ql, qr, ql * nl, qr * nr)), out(flux(pl, pr, pl * nl, pr * nr))
            if self.nu:
                dl, dr = self.nu * rl * torch.clamp(Hl, min=0.0), self.nu * rr * torch.clamp(Hr, min=0.0)
                du = du - out(torch.where(some, 0.5 * (dl * at(su) + dr * su), 0.0))
                dv = dv - out(torch.where(some, 0.5 * (dl * at(sv) + dr * sv), 0.0))
            if self.oned:
                fu = fv = 1.0 / self.gam
            else:
                cross = -self.bx * self.by / self.gam
                fu = (1.0 + self.by ** 2) / self.gam if axis == 1 else cross
                fv = cross if axis == 1 else (1.0 + self.bx ** 2) / self.gam
            eu, ev = eu + (du + hyd * fu) / dx, ev + (dv + hyd * fv) / dx
        if self.source is not None:
            ew, eh = ew + self.source[0] / self.gam ** 2, eh + self.source[1] / self.gam
        push = c["g"] * rho * (w - self.b) / self.gam
        eu, ev = eu - push * self.bx, ev - push * self.by
        speed2 = u * u * (1.0 + self.bx ** 2) + v * v * (1.0 + self.by ** 2) + 2.0 * self.bx * self.by * u * v
        speed = torch.sqrt(speed2)
        on = (hn > c["thr"]) & (speed > 1e-8)
        fric = self.drag(hn, u, v, psi, speed2)
        im = torch.where(on, -fric / torch.where(on, hn * speed, 1.0), 0.0)
        return ew, eu, ev, eh, im, cfl, (u, v, hn, psi, rho, speed)

    def advice(self, m):
        c = self.c
        top = self.case["max_dt"]
        if not bool(self.active.all()):
            m = min(m, top)
        return min(c["cfl"] * m, self.dx ** 2 / self.nu if self.nu else top, top)

    def step(self):
        edge = torch.zeros_like(self.active)
        if self.case["kind"] != "interval":
            edge[:, [0, -1]] = True
            if not self.oned:
                edge[[0, -1], :] = True
        self.active = self.active | (self.flags & ~edge)
        act = self.act = self.cells(self.active)
        u0 = (self.w, self.ru, self.rv, self.h)
        e = self.rhs(*u0)
        dt = 0.9 * self.advice(e[5].item())
        while True:
            d = 1.0 - dt * e[4]
            u1 = (u0[0] + dt * e[0], (u0[1] + dt * e[1]) / d, (u0[2] + dt * e[2]) / d, u0[3] + dt * e[3])
            u1 = tuple(torch.where(act, a, b) for a, b in zip(u1, u0))
            f = self.rhs(*u1)
            if self.advice(f[5].item()) < dt:
                dt = 0.9 * self.advice(f[5].item())
                continue
            d = 1.0 - dt * f[4]
            u2 = (0.75 * u0[0] + 0.25 * (u1[0] + dt * f[0]), 0.75 * u0[1] + 0.25 * (u1[1] + dt * f[1]) / d,
                  0.75 * u0[2] + 0.25 * (u1[2] + dt * f[2]) / d, 0.75 * u0[3] + 0.25 * (u1[3] + dt * f[3]))
            u2 = tuple(torch.where(act, a, b) for a, b in zip(u2, u0))
            f = self.rhs(*u2)
            if self.advice(f[5].item()) < dt:
                dt = 0.9 * self.advice(f[5].item())
                continue
            break
        d, p, q = 1.0 - dt * f[4], 1.0 / 3.0, 2.0 / 3.0
        u3 = (p * u0[0] + q * (u2[0] + dt * f[0]), p * u0[1] + q * (u2[1] + dt * f[1]) / d,
              p * u0[2] + q * (u2[2] + dt * f[2]) / d, p * u0[3] + q * (u2[3] + dt * f[3]))
        u3 = tuple(torch.where(act, a, b) for a, b in zip(u3, u0))
        f = self.rhs(*u3)
        d = 1.0 + dt * dt * f[4] ** 2
        self.w, self.h = u3[0], u3[3]
        self.ru = torch.where(act, (u3[1] - dt * dt * f[1] * f[4]) / d, u0[1])
        self.rv = torch.where(act, (u3[2] - dt * dt * f[2] * f[4]) / d, u0[2])
        self.last = f[6]
        self.flags = self.near(f[6][2])
        return dt

    def fields(self):
        """state()'s arrays: zero outside the active tiles and their ghosts."""
        a = self.active.double()[None, None]
        if self.oned:
            near = torch.nn.functional.max_pool2d(a, (1, 3), 1, (0, 1))[0, 0] > 0
        else:
            near = torch.nn.functional.max_pool2d(a, 3, 1, 1)[0, 0] > 0
        held, act = self.cells(near), self.cells(self.active)
        out = {k: torch.where(held, x, 0.0) for k, x in
               (("w", self.w), ("rhoHnu", self.ru), ("rhoHnv", self.rv), ("Hnpsi", self.h))}
        out["Hn"] = torch.where(act, self.depth(self.w), 0.0)
        return {k: x.cpu().numpy() for k, x in out.items()}

    def columns(self):
        """The solution file's columns, tile by tile (every tile active)."""
        u, v, hn, psi, rho, speed = self.last
        hn = self.depth(self.w)
        cols = (hn, speed, u, v, rho, psi, self.ru, self.rv, self.h, self.w, self.b, torch.zeros_like(u), self.bx,
                self.by)
        k = self.case
        a = torch.stack(cols).reshape(14, k["tiles_y"], k["tile_y"], k["tiles_x"], k["tile_x"])
        return a.permute(1, 3, 0, 2, 4).reshape(-1, 14, k["tile_y"], k["tile_x"]).cpu().numpy()

    def sums(self):
        """The Volume.txt columns over a bed that has not changed."""
        c, act = self.c, self.cells(self.active).double()
        area = self.dx ** 2
        vol = (self.gam * (self.w - self.b) * self.gam * act).sum().item() * area
        solids = (self.gam * self.h * act).sum().item() * area
        mass = c["rhow"] * vol + (c["rhos"] - c["rhow"]) * solids
        return np.array([vol, 0.0, mass, 0.0, solids * c["rhos"], 0.0])


def exact(case: dict, seed: int):
    """What run() returns, by plain torch in 64 bits.  None for morphodynamic
    runs: their redistribution corrects one cell after another in sorted
    order, which takes minutes in plain Python."""
    if case["morpho"]:
        return None
    sims = [_Plain(m, _inputs(m, seed)) for m in _members(case)]
    t = 0.0
    for s in sims:
        for _ in range(0 if case["kind"] == "volume" else case["steps"]):
            t += s.step()
    if case["kind"] == "volume":
        return sims[0].sums()
    if case["kind"] == "interval":
        return {"tiles": None, "fields": sims[0].columns(), "volume": sims[0].sums()}
    if case["kind"] == "ensemble":
        return [[f["w"], f["rhoHnu"], f["rhoHnv"]] for f in (s.fields() for s in sims)]
    out = dict(sims[0].fields(), btv=None, tile_state=None, t=t)
    if case["maxima"]:
        out["maxima"] = None
    return out
