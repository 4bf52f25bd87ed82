"""The time loops carry the CFL minimum of a step's new state over to the next
step: states set between calls, members that join or are stepped by themselves
between launches, and launches cut differently all give the steps that a fresh
reduction gives."""
import numpy as np
import pytest

import zisafvm_amd as z
from zisafvm_amd import workloads as W

pytestmark = pytest.mark.gpu


def _alone(wl, u, steps, t=0.0):
    s = z.Solver(wl.mesh, wl.params)
    s.set_state(u)
    if wl.steady is not None:
        s.set_steady_state(wl.steady)
    for _ in range(steps):
        dt = s.cfl_dt(wl.cfl)
        s.step(t, dt)
        t += dt
    return s.get_state(), t


def _solver(wl):
    s = z.Solver(wl.mesh, wl.params)
    s.set_state(wl.u0)
    if wl.steady is not None:
        s.set_steady_state(wl.steady)
    return s


WLS = {"vortex": lambda: W.vortex_2d(n=13), "isothermal": lambda: W.isothermal_2d(n=11, amplitude=1e-3, order=3),
       "polytrope": lambda: W.polytrope_3d(n=8, amplitude=1e-3)}


@pytest.mark.parametrize("name", sorted(WLS))
@pytest.mark.parametrize("noalloc", [False, True])
def test_advance_after_new_states(gpu, name, noalloc):
    wl = WLS[name]()
    hot = wl.u0 * np.array([1.0, 1.1, 1.1, 1.1, 1.21])  # faster, so smaller steps
    s = _solver(wl)
    run = s.advance_noalloc if noalloc else s.advance
    for u, k in ((wl.u0, 3), (hot, 2), (wl.u0, 1), (hot, 4)):
        s.set_state(u)
        t, steps = run(wl.cfl, 0.0, 1.0, max_steps=k, check_every=2)
        ref, t_ref = _alone(wl, u, k)
        assert steps == k and abs(t - t_ref) <= 1e-15
        np.testing.assert_array_equal(s.get_state(), ref)


@pytest.mark.parametrize("cuts", [(5,), (1, 1, 1, 1, 1), (2, 0, 3)])
def test_batch_launches_cut_differently(gpu, cuts):
    wls = [WLS["vortex"](), WLS["isothermal"]()]
    solvers = [_solver(w) for w in wls]
    b = z.Batch(wls[0].params, sum(w.mesh.n_cells for w in wls), 4000, 2)
    for w, s in zip(wls, solvers):
        b.add(s, w.cfl, 0.0, 1.0, 5)
    for c in cuts:
        b.run(c)
    for w, s in zip(wls, solvers):
        np.testing.assert_array_equal(s.get_state(), _alone(w, w.u0, 5)[0])


def test_batch_member_set_and_joined_between_launches(gpu):
    a, c = WLS["vortex"](), WLS["isothermal"]()
    hot = a.u0 * np.array([1.0, 1.1, 1.1, 1.1, 1.21])
    sa, sc = _solver(a), _solver(c)
    b = z.Batch(a.params, a.mesh.n_cells + c.mesh.n_cells, 4000, 2)
    slot = b.add(sa, a.cfl, 0.0, 1.0)
    b.launch(2)
    sa.set_state(hot)  # waits for the steps in flight
    b.run(2)
    ref, _ = _alone(a, hot, 2)
    np.testing.assert_array_equal(sa.get_state(), ref)
    sa.step(0.0, 1e-4)  # a step of its own, outside the batch
    after = sa.get_state()
    b.add(sc, c.cfl, 0.0, 1.0, 3)
    b.run(4)
    np.testing.assert_array_equal(sa.get_state(), _alone(a, after, 4)[0])
    np.testing.assert_array_equal(sc.get_state(), _alone(c, c.u0, 3)[0])
    assert b.query(slot)["active"] and b.query(slot)["steps"] == 8
