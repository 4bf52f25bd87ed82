"""The pseudo-inverses are stored in tiles of one wavefront's cells (16 in 2D,
12 in 3D): meshes whose last tile is partly filled, for every kernel shape
with whole and partial row chunks, against the oracle."""
import numpy as np
import pytest

import zisafvm_amd as z
from zisafvm_amd import workloads as W
from oracle.zfv_ref import Oracle
from emu_binding import Emu
from conftest import rel_err, wb_err

TOL = 1e-12  # the parity tolerance of a rate of change

# (cells modulo the tile size: 162 % 16 = 2, 242 % 16 = 2, 338 % 16 = 2; the
# atmosphere's 9 x (9 + 6) x 2 = 270 % 16 = 14; 3135 % 12 = 3)
CASES = {
    "order2_162": lambda: (W.vortex_2d(n=9), dict(order=2, edge_deg=2)),
    "order3_242": lambda: (W.vortex_2d(n=11), dict(order=3)),
    "order4_338": lambda: (W.vortex_2d(n=13), dict(order=4)),
    "isothermal_order4_270": lambda: (W.isothermal_2d(n=9, amplitude=1e-3), None),
    "polytrope3d_3135": lambda: (W.polytrope_3d(n=10, amplitude=1e-3), None),
}


def _case(name):
    wl, kw = CASES[name]()
    p = wl.params if kw is None else z.make_params(n_dims=2, **kw)
    assert wl.mesh.n_cells % (16 if p.n_dims == 2 else 12) != 0
    return wl, p


def _check(got, wl, p):
    ref = Oracle(wl.mesh, p).rate(wl.u0)
    errs = rel_err(got, ref) if p.gravity == 0 else wb_err(got, ref, wl.mesh, wl.u0, p.gamma)
    assert max(errs) <= TOL, errs


@pytest.mark.parametrize("name", sorted(CASES))
def test_partly_filled_last_tile_emulated(name):
    wl, p = _case(name)
    _check(Emu(wl.mesh, p).rate(wl.u0), wl, p)


@pytest.mark.gpu
@pytest.mark.parametrize("threads", [64, 128, 256])
@pytest.mark.parametrize("name", sorted(CASES))
def test_partly_filled_last_tile(gpu, name, threads):
    wl, p = _case(name)
    s = z.Solver(wl.mesh, p)
    s.tune(threads)
    got = s.rate(wl.u0)
    _check(got, wl, p)
    # a plain run uses correctly rounded operations only: equal to the emulation
    if p.gravity == 0:
        np.testing.assert_array_equal(got, Emu(wl.mesh, p).rate(wl.u0))
