"""Large bundles of loop tasks (swsph_run_tasks) run as tiles of the work
queue with a mask of stencil images per cell; small ones merge on the host.
Both must give the sums of the same tasks bit for bit where the bundles meet
the same images, and refuse the same tasks.

Boxes: 10^3 cells at 2 and 12 % active (14000 tasks in a loop, cells with no
active particle), and 5^3 cells (1750 tasks) where every cell has more
particles than a tile.  The large bundle of one box is cut into parts that
leave the cells with partial masks; its sums are added in another order, so
they are compared at FP32 summation order.
"""
from __future__ import annotations

import numpy as np
import pytest

from parity import DENSITY_FIELDS, FORCE_FIELDS

pytestmark = pytest.mark.gpu

SELF, PAIR = 0, 1
FIELDS = ["h", "rho", "wcount", "div_v", "rot_v", "v_sig", "laplace_u",
          "alpha_visc_max_ngb", "a_hydro", "u_dt", "h_dt", "n_density",
          "n_gradient", "n_force", "min_ngb_time_bin"]


def _tasks(eng):
    out = []
    for c in range(eng.num_cells()):
        cx, cy, cz = eng.cell_coords(c)
        out.append((SELF, c, c))
        for o in range(14, 27):
            out.append((PAIR, c, eng.cell_id(cx + o // 9 - 1,
                                             cy + (o // 3) % 3 - 1,
                                             cz + o % 3 - 1)))
    return out


def _pass(eng, loops):
    n = eng.num_cells()
    for c in range(n):
        eng.hydro_init_cell(c)
    for name, end in (("density", "runner_do_ghost"),
                      ("gradient", "runner_do_extra_ghost"),
                      ("force", "runner_do_end_hydro_force")):
        for b in loops:
            eng.run_tasks(name, b)
        for c in range(n):
            getattr(eng, end)(c)
    return eng.results(FIELDS)


def _box(n_side, ncell, frac, seed):
    from swift_amd import Engine, HydroProps, ics
    st = ics.modulated_box(n_side, seed=seed)
    props = HydroProps(ncell=(ncell,) * 3)
    with Engine(props) as eng:
        eng.set_particles(st)
        eng.pass_batched()
        base = eng.results()
    for k in ("h", "rho", "pressure", "soundspeed", "f", "balsara",
              "alpha_visc", "alpha_diff"):
        st[k] = base[k].astype(st[k].dtype)
    if frac < 1:
        ics.set_active_fraction(st, frac, seed=seed)
    return st, HydroProps(ncell=(ncell,) * 3)


def _run(st, props, cut):
    from swift_amd import Engine
    with Engine(props) as eng:
        eng.set_particles(st)
        return _pass(eng, cut(_tasks(eng)))


def _by_cell(tasks):
    """Bundles of one cell's tasks, merged on the host."""
    return [tasks[k:k + 14] for k in range(0, len(tasks), 14)]


def _close(a, b, act):
    """The same sums in another order: the oracle comparison's tolerances,
    of the largest value of the field."""
    for k in FIELDS:
        x, y = a[k][act].astype(np.float64), b[k][act].astype(np.float64)
        if a[k].dtype.kind in "iu":
            assert np.array_equal(x, y), k
            continue
        tol = {**DENSITY_FIELDS, **FORCE_FIELDS}.get(k, (1e-5, 0))[0]
        assert np.abs(x - y).max() <= tol * np.abs(y).max(), k


@pytest.mark.parametrize("n_side,ncell,frac", [(40, 10, 0.02), (40, 10, 0.12),
                                               (20, 5, 1.0)])
def test_large_bundle(n_side, ncell, frac):
    st, props = _box(n_side, ncell, frac, seed=n_side)
    act = st["time_bin"] <= props.max_active_bin
    whole = _run(st, props, lambda t: [t])
    # the whole stencil in one bundle: the batched pass's order of sums
    from swift_amd import Engine
    with Engine(props) as eng:
        eng.set_schedule(0)
        eng.set_particles(st)
        eng.pass_batched()
        ref = eng.results(FIELDS)
    for k in ("h", "rho", "wcount", "n_density", "n_gradient", "n_force"):
        assert np.array_equal(whole[k][act], ref[k][act]), k
    _close(whole, ref, act)
    _close(_run(st, props, _by_cell), ref, act)
    # partial masks above the threshold
    _close(_run(st, props, lambda t: [t[:1100], t[1100:]]), ref, act)


def test_large_bundle_errors():
    from swift_amd import Engine
    from swift_amd._lib import SwsphError
    st, props = _box(20, 5, 1.0, seed=3)
    with Engine(props) as eng:
        eng.set_particles(st)
        t = _tasks(eng)
        far = eng.cell_id(2, 2, 2)
        n = eng.num_cells()
        for bad, what in (((PAIR, t[1][2], t[1][1]), "twice"),
                          ((SELF, 0, 0), "twice"),
                          ((PAIR, 0, far), "not neighbours"),
                          ((PAIR, 0, 0), "not neighbours"),
                          ((7, 0, 0), "unknown type"),
                          ((SELF, n, n), "out of range"),
                          ((PAIR, 0, -1), "out of range")):
            with pytest.raises(SwsphError, match=what):
                eng.run_tasks("density", t + [bad])
        # the refused bundles did nothing
        got = _pass(eng, [t])
    ref = _run(st, props, lambda t: [t])
    for k in FIELDS:
        assert np.array_equal(got[k], ref[k]), k
