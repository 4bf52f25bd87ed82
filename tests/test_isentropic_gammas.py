"""The general isentropic equilibrium over gases: 1/(gamma-1) a half of a whole
number (products and a square root on the device) and not (pow), with every
flux BC's mesh edges, against the oracle; the emulation uses pow throughout."""
import pytest

import zisafvm_amd as z
from zisafvm_amd import workloads as W
from oracle.zfv_ref import Oracle
from emu_binding import Emu
from conftest import wb_err

TOL = 1e-12  # the parity tolerance of a rate of change
GAMMAS = [7.0 / 5.0, 5.0 / 3.0, 4.0 / 3.0, 1.5, 1.2, 1.3, 1.9]


def _check(make, gamma, order):
    wl = W.isentropic_2d(n=11, order=order, amplitude=1e-3, gamma=gamma, flux_bc=2)
    ref = Oracle(wl.mesh, wl.params).rate(wl.u0)
    errs = wb_err(make(wl.mesh, wl.params).rate(wl.u0), ref, wl.mesh, wl.u0, gamma)
    print("gamma", gamma, "order", order, "wb err", errs, flush=True)
    assert max(errs) <= TOL, errs


@pytest.mark.parametrize("gamma", GAMMAS)
def test_gases_emulated(gamma):
    _check(Emu, gamma, 3)


@pytest.mark.gpu
@pytest.mark.parametrize("order", [2, 3, 4])
@pytest.mark.parametrize("gamma", GAMMAS)
def test_gases(gpu, gamma, order):
    _check(z.Solver, gamma, order)
