"""From 96 steps asked for on, in one run or several, runs replay graphs of eight
steps, then single ones: counts around those sizes, repeated with other work on
the device between the replays, equal to steps launched one by one."""
import numpy as np
import pytest

import zisafvm_amd as z
from zisafvm_amd import workloads as W

COUNTS = [7, 8, 47, 48, 95, 96, 101]


@pytest.mark.gpu
@pytest.mark.parametrize("n", COUNTS)
def test_steps(gpu, n):
    wl = W.isothermal_2d(n=12, order=3, amplitude=1e-3)
    s = z.Solver(wl.mesh, wl.params)
    s.set_steady_state(wl.steady)
    s.set_state(wl.u0)
    dt = s.cfl_dt(0.3)
    for k in range(n):
        s.step(k * dt, dt)
    ref = s.get_state()
    for _ in range(4):
        s.rate(wl.u0)  # other work on the same buffers
        s.set_state(wl.u0)
        s.steps(n, 0.0, dt)
        np.testing.assert_array_equal(s.get_state(), ref)
    s.set_state(wl.u0)  # another dt in between: captured again
    s.steps(n, 0.0, 0.5 * dt)
    s.set_state(wl.u0)
    s.steps(n, 0.0, dt)
    np.testing.assert_array_equal(s.get_state(), ref)


@pytest.mark.gpu
@pytest.mark.parametrize("reject", [0.0, 0.01])
@pytest.mark.parametrize("n", COUNTS)
def test_advance(gpu, n, reject):
    wl = W.vortex_2d(n=12)
    s = z.Solver(wl.mesh, wl.params)
    got = []
    for every in (1, n, n, n):
        s.set_state(wl.u0)
        t, steps = s.advance(0.4, 0.0, 10.0, max_steps=n, check_every=every, drho_crit_rel=reject, max_exponent=4)
        got.append((s.get_state(), t, steps, s.rejected_steps))
        s.rate(wl.u0)
    for u, t, steps, rejected in got[1:]:
        np.testing.assert_array_equal(u, got[0][0])
        assert (t, steps, rejected) == got[0][1:]


@pytest.mark.gpu
@pytest.mark.parametrize("n", COUNTS)
def test_batch(gpu, n):
    wls = [W.vortex_2d(n=k) for k in (10, 14)]
    got = []
    for per_run in (1, n, n):
        solvers = [z.Solver(wl.mesh, wl.params) for wl in wls]
        b = z.Batch(wls[0].params, sum(w.mesh.n_cells for w in wls), 1000, 2)
        for s, wl in zip(solvers, wls):
            s.set_state(wl.u0)
            b.add(s, 0.4, 0.0, 10.0)
        for _ in range(n // per_run):
            b.run(per_run)
        if per_run == n:  # again, in the graphs that the first run left
            for s, wl in zip(solvers, wls):
                s.set_state(wl.u0)
            for slot in (0, 1):
                b.remove(slot)
            for s in solvers:
                b.add(s, 0.4, 0.0, 10.0)
            b.run(n)
        got.append([s.get_state() for s in solvers])
    for g in got[1:]:
        for a, r in zip(g, got[0]):
            np.testing.assert_array_equal(a, r)
