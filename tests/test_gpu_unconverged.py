"""What a pass whose smoothing lengths do not converge (status 3) leaves
behind: the same in every form of the pass, with nothing behind the ghost
begun, so that it can be repeated with more iterations.
"""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# fields that only the stages behind the ghost write
LATER = ("v_sig", "laplace_u", "alpha_visc_max_ngb", "alpha_visc",
         "alpha_diff", "div_v_dt", "div_v_prev", "a_hydro", "u_dt", "h_dt",
         "n_gradient", "n_force", "min_ngb_time_bin")
# (schedule, shapes of the three loops, method of the pass)
GRID = (0, ((16, 16),) * 3, "pass_batched")
FORMS = [
    (1, ((16, 16),) * 3, "pass_batched"),
    (1, ((16, 16),) * 3, "pass_graph"),
    (2, ((16, 16),) * 3, "pass_batched"),
    (1, ((16, 16),) * 3, "pass_batched_noalloc"),
    (1, ((16, 8), (32, 16), (8, 8)), "pass_batched"),
    (1, ((16, 16), (4, 8), (16, 16)), "pass_graph"),
    (1, ((16, 16), (16, 16), (4, 8)), "pass_batched"),
    (2, ((16, 16), (32, 32), (4, 8)), "pass_batched"),
]


def _start():
    """Half of the particles near their converged h, the others far off, in
    the middle of a run (dissipation coefficients set)."""
    from swift_amd import HydroProps, ics
    st = ics.modulated_box(13, seed=2, amp=0.3)
    rng = np.random.default_rng(5)
    n = st["h"].size
    st["h"][rng.uniform(size=n) < 0.5] *= np.float32(0.75)
    st["alpha_visc"] = rng.uniform(0.1, 1.5, n).astype(np.float32)
    st["alpha_diff"] = rng.uniform(0.0, 0.5, n).astype(np.float32)
    st["div_v_prev"] = rng.normal(size=n).astype(np.float32)
    return HydroProps(ncell=(3, 4, 3)), st


def _engine(props, form):
    from swift_amd import Engine
    mode, shapes, _ = form
    eng = Engine(props)
    eng.set_regrid(False)
    eng.set_schedule(mode)
    for loop, s in zip(("density", "gradient", "force"), shapes):
        eng.set_tile_shape(loop, *s)
    return eng


def _fail(eng, form):
    """One pass that ends with status 3; the number of particles it names."""
    from swift_amd import SwsphError
    with pytest.raises(SwsphError, match="status 3") as err:
        getattr(eng, form[2])()
    return int(str(err.value).split(" particles")[0].split()[-1])


@pytest.mark.parametrize("form", [GRID] + FORMS)
def test_unconverged_pass_ends_at_the_ghost(form):
    """Gradient, extra ghost and force leave the particles as they were."""
    props, st = _start()
    with _engine(dataclasses.replace(props, max_iter=3), form) as eng:
        eng.set_particles(st)
        before = eng.results(LATER)
        count = _fail(eng, form)
        after = eng.results(LATER)
    assert 0 < count < st["h"].size
    for k in LATER:
        assert np.array_equal(before[k], after[k]), k


DENSITY = ("h", "rho", "rho_dh", "wcount", "wcount_dh", "div_v", "rot_v",
           "pressure", "soundspeed", "f", "balsara", "n_density")


def _fail_and_repeat(form):
    """All fields after status 3, and after the pass repeated from there with
    enough iterations."""
    props, st = _start()
    with _engine(dataclasses.replace(props, max_iter=3), form) as eng:
        eng.set_particles(st)
        _fail(eng, form)
        failed = eng.results()
        eng.set_props(props)
        getattr(eng, form[2])()
        return failed, eng.results()


@pytest.mark.parametrize("form", FORMS)
def test_unconverged_pass_can_be_repeated(form):
    """A particle that did not converge is left with the raw density sums at
    its last h, a converged one finished, bit for bit as the grid schedule's
    separate ghost rounds leave them; the repeated pass agrees as well (its
    gradient and force sums where the tiles add in the grid's order)."""
    ref = _fail_and_repeat(GRID)
    got = _fail_and_repeat(form)
    same = [s[0] == 16 for s in form[1]]
    for k in ref[0]:
        assert np.array_equal(ref[0][k], got[0][k]), k
        if k in DENSITY or all(same):
            assert np.array_equal(ref[1][k], got[1][k]), k


def _ghost_tasks(eng, how):
    """The ghosts of all cells; how many of the calls ended with status 3."""
    from swift_amd import SwsphError
    nc = eng.num_cells()
    if how == "bundle":
        calls = [lambda: eng.runner_do_ghost_cells(range(nc))]
    else:
        calls = [lambda c=c, o=o: eng.runner_do_ghost(c, o, how)
                 for c in range(nc) for o in range(how)]
    failed = 0
    for call in calls:
        try:
            call()
        except SwsphError as err:
            assert "status 3" in str(err)
            failed += 1
    return failed


@pytest.mark.parametrize("how", [1, 2, "bundle"])
def test_ghost_goes_on_where_it_ended(how):
    """A ghost task that ran out of iterations, called again, goes on with
    the bracket and the sums at the h it had reached: the same results as one
    that had enough iterations."""
    props, st = _start()
    out = []
    for first in (props.max_iter, 3):
        with _engine(dataclasses.replace(props, max_iter=first),
                     FORMS[0]) as eng:
            eng.set_particles(st)
            nc = eng.num_cells()
            eng.init_cells(range(nc))
            nz, ny, nx = props.ncell[2], props.ncell[1], props.ncell[0]
            pairs = set()
            for c in range(nc):
                x, y, z = c // (ny * nz), (c // nz) % ny, c % nz
                for d in np.ndindex(3, 3, 3):
                    o = (((x + d[0] - 1) % nx) * ny + (y + d[1] - 1) % ny) \
                        * nz + (z + d[2] - 1) % nz
                    if o != c:
                        pairs.add((min(c, o), max(c, o)))
            eng.run_tasks("density", [(0, c, c) for c in range(nc)]
                          + [(1, a, b) for a, b in sorted(pairs)])
            failed = _ghost_tasks(eng, how)
            if first == 3:
                assert failed > 0
                eng.set_props(props)
                _ghost_tasks(eng, how)
            else:
                assert failed == 0
            out.append(eng.results(DENSITY))
    for k in DENSITY:
        assert np.array_equal(out[0][k], out[1][k]), k


@pytest.mark.parametrize("shape", [(16, 16), (8, 8)])
def test_ghost_leaves_inactive_particles(shape):
    """Particles flagged by a pass that failed, inactive in the next one, are
    not the business of the ghosts of that step."""
    props, st = _start()
    late = np.random.default_rng(6).uniform(size=st["h"].size) < 0.5
    low = int(st["time_bin"].max())
    st["time_bin"][late] = low + 4
    with _engine(dataclasses.replace(props, max_iter=3), FORMS[0]) as eng:
        eng.set_particles(st)
        _fail(eng, FORMS[0])
        eng.set_props(dataclasses.replace(props, max_active_bin=low))
        eng.pass_batched()
        before = eng.results(DENSITY)
        eng.set_tile_shape("density", *shape)
        nc = eng.num_cells()
        eng.init_cells(range(nc))
        for c in range(nc):
            eng.runner_doself1_branch_density(c)
        eng.set_props(dataclasses.replace(props, max_active_bin=low,
                                          h_tolerance=1.0))
        assert _ghost_tasks(eng, 1) == 0
        after = eng.results(DENSITY)
    assert late.any()
    for k in DENSITY:
        assert np.array_equal(before[k][late], after[k][late]), k
