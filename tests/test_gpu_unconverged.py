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
# (schedule, shapes of the three loops, replayed)
GRID = (0, ((16, 16),) * 3, False)
FORMS = [
    (1, ((16, 16),) * 3, False),
    (1, ((16, 16),) * 3, True),
    (2, ((16, 16),) * 3, False),
    (1, ((16, 8), (32, 16), (8, 8)), False),
    (1, ((16, 16), (4, 8), (16, 16)), True),
    (1, ((16, 16), (16, 16), (4, 8)), False),
    (2, ((16, 16), (32, 32), (4, 8)), False),
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
        eng.pass_graph() if form[2] else eng.pass_batched()
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
