"""Host arrays of the calls that return states and tendencies, on both sides of
the size (32 pages) from which their pages are mapped ahead: a new tendency
equals one added to zeros, one added to values equals their sum, and batches
whose members change between launches give what single runs give."""
import numpy as np
import pytest

import zisafvm_amd as z
from zisafvm_amd import workloads as W


@pytest.mark.gpu
@pytest.mark.parametrize("n", [16, 40, 41, 64])  # 512, 3200, 3362, 8192 cells; 32 pages hold 3276
def test_states_and_tendencies(gpu, n):
    wl = W.vortex_2d(n=n)
    s = z.Solver(wl.mesh, wl.params)
    s.set_state(wl.u0)
    np.testing.assert_array_equal(s.get_state(), wl.u0)
    new = s.rate(wl.u0)
    assert new.shape == wl.u0.shape and not np.signbit(new[new == 0.0]).any()
    np.testing.assert_array_equal(new, s.rate(wl.u0, dudt=np.zeros_like(wl.u0)))
    base = np.random.default_rng(n).normal(size=wl.u0.shape)
    np.testing.assert_array_equal(s.rate(wl.u0, dudt=base.copy()), base + new)


@pytest.mark.gpu
def test_members_that_change_between_launches(gpu):
    cfl, wls = 0.4, [W.vortex_2d(n=k) for k in (12, 16, 20)]

    def alone(wl, steps):
        s = z.Solver(wl.mesh, wl.params)
        s.set_state(wl.u0)
        b = z.Batch(wl.params, wl.mesh.n_cells, 2 * wl.mesh.n_cells, 1)
        b.add(s, cfl, 0.0, 1.0)
        b.run(steps)
        return s.get_state()

    solvers = [z.Solver(wl.mesh, wl.params) for wl in wls]
    for s, wl in zip(solvers, wls):
        s.set_state(wl.u0)
    b = z.Batch(wls[0].params, sum(w.mesh.n_cells for w in wls[1:]), 4 * wls[2].mesh.n_cells, 2)
    first = b.add(solvers[0], cfl, 0.0, 1.0)
    second = b.add(solvers[1], cfl, 0.0, 1.0)
    with pytest.raises(z.ZfvError):
        b.add(solvers[2], cfl, 0.0, 1.0)  # full: refused when it is added
    b.run(3)
    b.remove(first)  # leaves, and another takes its slot before the next launch
    assert b.add(solvers[2], cfl, 0.0, 1.0) == first
    assert b.query(second)["steps"] == 3 and b.query(first)["steps"] == 0
    b.launch(2)
    b.remove(second)  # waits for the steps in flight
    b.run(2)
    for k, steps in enumerate((3, 5, 4)):
        np.testing.assert_array_equal(solvers[k].get_state(), alone(wls[k], steps))
