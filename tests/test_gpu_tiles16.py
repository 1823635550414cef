"""The tiles of 16 of the work queue (swift_amd/csrc/sph_tile.h): their
windows, hit lists and in-wave smoothing-length iteration against the chunk
grid with its separate ghost rounds, bit for bit, and against the oracle.

Boxes where the tiling can go wrong: cells that are no multiple of 16, cells
with few particles, radii that give a lane more hits than its list
holds and a tile more candidates than a window, partly active and inhibited
particles, and starts that need many rounds.
"""
from __future__ import annotations

import numpy as np
import pytest

from parity import assert_parity

pytestmark = pytest.mark.gpu


def _box(name):
    from swift_amd import HydroProps, ics
    if name == "ragged":
        return HydroProps(ncell=(3, 4, 3)), ics.modulated_box(13, seed=2, amp=0.3)
    if name == "lists":  # 500 neighbours at the start, all cells in reach
        st = ics.modulated_box(15, seed=3, amp=0.2)
        st["h"] = np.full_like(st["h"], 0.33 / 1.936492)
        return HydroProps(ncell=(3, 3, 3)), st
    if name == "windows":  # 3000 particles in a cell, half of it in reach
        st = ics.clustered_box(9000, seed=4, n_spheres=3, a_min=0.02,
                               a_max=0.05)
        st["h"] = np.minimum(st["h"] * np.float32(1.9),
                             np.float32(0.24 / 1.936492))
        return HydroProps(ncell=(4, 4, 4)), st
    if name == "few":  # 8 particles in a cell
        st = ics.lattice_box(6, seed=5, jitter=0.3)
        st["h"] = np.full_like(st["h"], 0.09)
        return HydroProps(ncell=(3, 3, 3), eta=0.85), st
    st = ics.modulated_box(14, seed=6, amp=0.4)
    st["h"] *= np.float32(0.6)
    if name == "half":
        ics.set_active_fraction(st, 0.5, seed=7)
        # the state that inactive neighbours bring along
        st["rho"] = np.ones_like(st["rho"])
        st["pressure"] = (st["u"] * np.float32(2 / 3)).astype(np.float32)
        st["soundspeed"] = np.sqrt(st["pressure"] * np.float32(5 / 3))
    else:
        rng = np.random.default_rng(8)
        st["time_bin"][rng.uniform(size=st["h"].size) < 0.2] = \
            ics.TIME_BIN_INHIBITED
    return HydroProps(ncell=(3, 3, 4)), st


def _run(props, st, mode, shape, graph=False, waves=0):
    from swift_amd import Engine
    with Engine(props) as eng:
        eng.set_regrid(False)
        eng.set_schedule(mode, waves)
        for loop in ("density", "gradient", "force"):
            eng.set_tile_shape(loop, *shape)
        eng.set_particles(st)
        eng.save_state()
        for _ in range(3 if graph else 1):
            eng.restore_state()
            s = eng.pass_graph() if graph else eng.pass_batched()
        return s, eng.results()


@pytest.mark.parametrize("box", ["ragged", "lists", "windows", "few", "half",
                                 "inhibited"])
def test_tiles16_match_grid(orc, box):
    props, st = _box(box)
    s0, r0 = _run(props, st, 0, (16, 16))
    act = st["time_bin"] <= props.max_active_bin
    chk = {k: np.array(v, copy=True) for k, v in st.items()}
    chk["h"] = r0["h"]
    assert_parity(r0, orc.pass_fp64(props, chk), act)
    for kw in (dict(mode=1, shape=(16, 16)), dict(mode=1, shape=(16, 8)),
               dict(mode=1, shape=(16, 32)),
               dict(mode=2, shape=(16, 16), waves=5),
               dict(mode=1, shape=(16, 16), graph=True)):
        s1, r1 = _run(props, st, **kw)
        for k in r0:
            assert np.array_equal(r0[k][act], r1[k][act], equal_nan=True), (kw, k)
        for k in ("ghost_rounds", "n_density_all", "n_density", "n_force"):
            assert s0[k] == s1[k], (kw, k)
    if box == "windows":
        assert s0["ghost_rounds"] >= 4


def test_tiles16_unconverged_is_an_error():
    """More rounds needed than allowed: status 3 from both forms."""
    import dataclasses
    from swift_amd import SwsphError
    props, st = _box("ragged")
    props = dataclasses.replace(props, max_iter=2)
    for kw in (dict(mode=0, shape=(16, 16)), dict(mode=1, shape=(16, 16)),
               dict(mode=1, shape=(16, 16), graph=True)):
        with pytest.raises(SwsphError, match="status 3"):
            _run(props, st, **kw)


@pytest.mark.parametrize("n_side,ncell", [(9, 3), (16, 4), (17, 4), (20, 5),
                                          (32, 8), (33, 8)])
def test_tile_order_over_the_xcds(n_side, ncell):
    """Gradient and force tiles are dealt to the XCDs in runs whose length
    grows with the number of tiles (256 tiles and a few more, 500, 2048 and
    more, and fewer than 8 runs): eager, and captured with a grid for more
    tiles than there are, every tile once -- the grid schedule's sums."""
    from swift_amd import Engine, HydroProps, ics
    st = ics.modulated_box(n_side, seed=n_side)
    out = []
    for mode in ("grid", "queue", "graph"):
        with Engine(HydroProps(ncell=(ncell,) * 3)) as eng:
            eng.set_schedule(0 if mode == "grid" else 1)
            eng.set_particles(st)
            if mode == "graph":
                eng.save_state()
                for _ in range(2):
                    eng.restore_state()
                    eng.pass_graph()
            else:
                eng.pass_batched()
            out.append(eng.results())
    for r in out[1:]:
        for k, v in out[0].items():
            assert np.array_equal(v, r[k]), k


@pytest.mark.parametrize("mode,shapes,want", [
    # counters, three for the tile table, density, chunk bounds, gradient,
    # force
    (1, ((16, 16),) * 3, 8),
    # the loops that reuse the table clear its queue heads
    (2, ((16, 16),) * 3, 10),
    # a tile table per loop, a second chunk table, and the sweeps of the
    # extra ghost and the force records
    (1, ((16, 16), (32, 32), (16, 16)), 17)])
def test_launches_are_counted_as_issued(mode, shapes, want):
    from swift_amd import Engine
    props, st = _box("ragged")
    with Engine(props) as eng:
        eng.set_regrid(False)
        eng.set_schedule(mode)
        for loop, s in zip(("density", "gradient", "force"), shapes):
            eng.set_tile_shape(loop, *s)
        eng.set_particles(st)
        eng.pass_batched()
        assert eng.pass_batched()["launches"] == want


def test_tiles16_few_of_many():
    """Far more tiles possible than there are (64^3 particles, 3 % active): the
    eager loops read the count back and reuse it with the table, the captured
    ones run a grid for the count at the capture and a small one for tiles
    beyond it.  The grid schedule's results bit for bit."""
    from swift_amd import HydroProps, ics
    st = ics.modulated_box(64, seed=12, amp=0.3)
    ics.set_active_fraction(st, 0.03, seed=13)
    st["rho"] = np.ones_like(st["rho"])
    st["pressure"] = (st["u"] * np.float32(2 / 3)).astype(np.float32)
    st["soundspeed"] = np.sqrt(st["pressure"] * np.float32(5 / 3))
    props = HydroProps(ncell=(14, 14, 14))
    act = st["time_bin"] <= props.max_active_bin
    tiles = st["h"].size // 16 + 14 ** 3 + 1
    assert tiles - int(act.sum()) > 4096 and act.sum() > 4096
    s0, r0 = _run(props, st, 0, (16, 16))
    for kw in (dict(mode=1, shape=(16, 16)),
               dict(mode=1, shape=(16, 16), graph=True),
               dict(mode=2, shape=(16, 16))):
        s1, r1 = _run(props, st, **kw)
        for k in r0:
            assert np.array_equal(r0[k], r1[k], equal_nan=True), (kw, k)
        for k in ("ghost_rounds", "n_density_all", "n_density", "n_force"):
            assert s0[k] == s1[k], (kw, k)


@pytest.mark.parametrize("box", ["lists", "windows", "images"])
@pytest.mark.parametrize("how", ["tasks", "graph of tasks"])
def test_tiles16_tasks_over_several_windows(orc, box, how):
    """Self and pair tasks and the ghosts behind them -- per cell and as
    bundles -- on cells whose candidates fill more than one window or whose
    hits overfill a lane's list: the oracle's results at the same h."""
    from swift_amd import Engine, ics
    if box == "images":  # 2700 particles in a cell: one image is two windows
        props, _ = _box("windows")
        st = ics.clustered_box(14000, seed=4, n_spheres=3, a_min=0.02,
                               a_max=0.05)
        st["h"] = np.minimum(st["h"] * np.float32(1.9),
                             np.float32(0.24 / 1.936492))
    else:
        props, st = _box(box)
    with Engine(props) as eng:
        eng.set_regrid(False)
        eng.set_particles(st)
        s = eng.pass_plain() if how == "tasks" else eng.sched_pass()[1]
        res = eng.results()
        counts = [eng.cell_count(c) for c in range(eng.num_cells())]
    if box == "images":
        assert max(counts) > 2048
    if box != "lists":
        assert s["ghost_rounds"] >= 4
    act = st["time_bin"] <= props.max_active_bin
    chk = {k: np.array(v, copy=True) for k, v in st.items()}
    chk["h"] = res["h"]
    assert_parity(res, orc.pass_fp64(props, chk), act)
    with Engine(props) as eng:
        eng.set_regrid(False)
        eng.set_particles(st)
        eng.pass_batched()
        ref = eng.results(["h"])
    # (sums in another order can end the iteration a step apart)
    assert np.allclose(ref["h"], res["h"], rtol=2 * props.h_tolerance)


@pytest.mark.parametrize("nc,big", [
    (3, {}), (3, {0: 1024}), (3, {5: 1025, 26: 1087}), (4, {15: 16385}),
    (4, {16: 3000, 17: 2900, 18: 2800, 31: 5000}), (4, {0: 1500, 63: 40000}),
    (3, {c: 1100 + 37 * c for c in range(27)}),
    (5, {c: 1030 + c for c in range(0, 125, 2)})])
@pytest.mark.parametrize("mixed", [False, True])
def test_tile_builder_takes_every_particle(nc, big, mixed):
    """The builder's list holds the active particles of the selected cells,
    where a wave takes a cell, where a cell is shared by the waves of its
    block (more than 1024 slots and a fifth of the block's), and where every
    cell has a block: seen through init_cells, which clears their density."""
    from swift_amd import Engine, HydroProps
    from swift_amd.ics import TIME_BIN_INHIBITED
    rng = np.random.default_rng(nc + len(big))
    ncells = nc ** 3
    counts = rng.integers(0, 40, ncells)
    for c, k in big.items():
        counts[c] = k
    cell = rng.permutation(np.repeat(np.arange(ncells), counts))
    corner = np.stack([cell // (nc * nc), cell // nc % nc, cell % nc], 1)
    n = cell.size
    st = {k: np.ones(n, np.float32) for k in (
        "m", "u", "rho", "pressure", "soundspeed", "f", "balsara",
        "alpha_visc", "alpha_diff", "div_v_prev")}
    st["x"] = (corner + rng.uniform(0.01, 0.99, (n, 3))) / nc
    st["v"] = np.zeros((n, 3), np.float32)
    st["h"] = np.full(n, 0.01, np.float32)
    st["time_bin"] = (rng.choice([1, 2, 3, 5, TIME_BIN_INHIBITED], n) if mixed
                      else np.full(n, 2)).astype(np.int8)
    with Engine(HydroProps(ncell=(nc,) * 3, max_active_bin=2)) as eng:
        eng.set_particles(st)
        act = st["time_bin"] <= 2
        left = np.ones(n, bool)
        for sel in (np.arange(0, ncells, 3), np.arange(ncells - 1, -1, -1)):
            eng.init_cells(sel)
            left &= ~(act & np.isin(cell, sel))
            assert np.array_equal(eng.get("rho"), left.astype(np.float32))


@pytest.mark.parametrize("n_side,ncell,frac", [(31, 3, 1.0), (31, 3, 0.1)])
def test_tiles16_of_large_cells(n_side, ncell, frac):
    """Every cell has a block of the builder (1100 particles in each of 27):
    the grid schedule's results, eager and captured."""
    from swift_amd import HydroProps, ics
    st = ics.modulated_box(n_side, seed=n_side, amp=0.3)
    if frac < 1:
        ics.set_active_fraction(st, frac, seed=1)
        st["rho"] = np.ones_like(st["rho"])
        st["pressure"] = (st["u"] * np.float32(2 / 3)).astype(np.float32)
        st["soundspeed"] = np.sqrt(st["pressure"] * np.float32(5 / 3))
    props = HydroProps(ncell=(ncell,) * 3)
    s0, r0 = _run(props, st, 0, (16, 16))
    for kw in (dict(mode=1, shape=(16, 16)), dict(mode=1, shape=(16, 16),
                                                  graph=True)):
        s1, r1 = _run(props, st, **kw)
        for k in r0:
            assert np.array_equal(r0[k], r1[k], equal_nan=True), (kw, k)
        assert s0["n_density_all"] == s1["n_density_all"], kw
