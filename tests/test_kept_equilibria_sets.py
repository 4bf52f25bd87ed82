"""Kept equilibria (steps_per_recompute > 1) mean the same in every physics
set: an isothermal member steps with the light set by itself and with the full
set beside an isentropic member, so its cells' equilibria are kept by one set
and read by another whenever such a member joins or leaves."""
import numpy as np
import pytest

import zisafvm_amd as z
from zisafvm_amd import workloads as W
from emu_binding import Emu, EmuBatch
from conftest import wb_err, with_recompute

STEPS = 2
KEPT = 7  # calls between recomputes: the second run of two steps starts on kept equilibria


def _run(sets, order):
    """Two runs of an isothermal member, each alone ("light") or beside an
    isentropic one ("full"); its change over the second."""
    a = W.isothermal_2d(n=10, order=order, amplitude=1e-3)
    b = W.isentropic_2d(n=8, order=order, ghost_layers=2)
    a.params = with_recompute(a.params, KEPT, 1e-2)
    ea = Emu(a.mesh, a.params)
    for s in sets:
        wls = [a] if s == "light" else [a, b]
        batch = EmuBatch([ea] + [Emu(w.mesh, w.params) for w in wls[1:]], wls, [0.45] * len(wls), [1.0] * len(wls),
                         [STEPS] * len(wls))
        batch.run(STEPS)
        u, t, steps, _ = batch.member(0)
        assert steps == STEPS
    return a, (u - a.u0) / t


@pytest.mark.parametrize("order", [2, 3])
@pytest.mark.parametrize("sets", [("light", "full"), ("full", "light")])
def test_kept_equilibria_are_read_as_they_were_kept(sets, order):
    a, got = _run(sets, order)
    _, ref = _run(("light", "light"), order)
    # the sets' averages differ by rounding only (1e-11: the tolerance of runs
    # of several steps against the oracle)
    errs = wb_err(got, ref, a.mesh, a.u0, a.params.gamma)
    assert max(errs) <= 1e-11, errs


@pytest.mark.gpu
@pytest.mark.parametrize("sets", [("light", "full"), ("full", "light")])
def test_kept_equilibria_on_the_device(gpu, sets):
    def run(sets):
        a = W.isothermal_2d(n=10, order=3, amplitude=1e-3)
        b = W.isentropic_2d(n=8, order=3, ghost_layers=2)
        a.params = with_recompute(a.params, KEPT, 1e-2)
        sa, sb = z.Solver(a.mesh, a.params), z.Solver(b.mesh, b.params)
        sa.set_steady_state(a.steady)
        sb.set_steady_state(b.steady)
        batch = z.Batch(a.params, a.mesh.n_cells + b.mesh.n_cells, 4000, 2)
        for s in sets:
            sa.set_state(a.u0)
            slots = [batch.add(sa, 0.45, 0.0, 1.0, STEPS)]
            if s == "full":
                sb.set_state(b.u0)
                slots.append(batch.add(sb, 0.45, 0.0, 1.0, STEPS))
            batch.run(STEPS)
            t = batch.query(slots[0])["t"]
            for k in slots:
                batch.remove(k)
        return a, (sa.get_state() - a.u0) / t

    a, got = run(sets)
    errs = wb_err(got, run(("light", "light"))[1], a.mesh, a.u0, a.params.gamma)
    assert max(errs) <= 1e-11, errs
