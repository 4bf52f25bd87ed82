"""The linear isentropic equilibrium starts its iteration from the closed-form
root where the two roots are well apart (4 v / r^2 <= 0.02, v the variance of
the cell's potential and r its specific enthalpy) and from the usual guess
elsewhere: stars whose cells lie on both sides, against the oracle, which always
starts from the guess."""
import numpy as np
import pytest

import zisafvm_amd as z
from zisafvm_amd import workloads as W
from oracle.zfv_ref import Oracle
from emu_binding import Emu
from conftest import wb_err

TOL = 1e-12  # the parity tolerance of a rate of change


def _check(make, n):
    wl = W.polytrope_3d(n=n, amplitude=1e-3)
    m, u = wl.mesh, wl.u0
    # phi = -2 K rho along the unperturbed star, nearly linear in a cell
    rho = W.polytrope_n1(np.asarray(m.corners).reshape(-1, 3))[:, 0].reshape(m.n_cells, -1)
    phi = -2.0 * rho
    v = ((phi - phi.mean(1, keepdims=True)) ** 2).sum(1) / 20.0
    r = 2.0 * (u[:, 4] - 0.5 * (u[:, 1:4] ** 2).sum(1) / u[:, 0]) / u[:, 0]
    from_root = (4.0 * v <= 0.02 * r * r)[m.ghost == 0]
    assert 0.1 < from_root.mean() < 0.99
    errs = wb_err(make(m, wl.params).rate(u), Oracle(m, wl.params).rate(u), m, u, 2.0)
    print("n", n, "from the root", from_root.mean(), "wb err", errs, flush=True)
    assert max(errs) <= TOL, errs


@pytest.mark.parametrize("n", [10, 16])
def test_both_starts_emulated(n):
    _check(Emu, n)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [10, 16])
def test_both_starts(gpu, n):
    _check(z.Solver, n)
