"""The update's tiles of faces (32 triangles, 20 tetrahedra a wavefront): meshes
of less than one tile, of partly filled last tiles, tiles of more than 64 faces
(cells in an order without locality), boundary faces with each flux BC; steps
against the oracle, conservation over the whole mesh."""
import numpy as np
import pytest

import zisafvm_amd as z
from zisafvm_amd import workloads as W
from oracle.zfv_ref import Oracle
from conftest import rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-12  # the parity tolerance of a rate of change


def _scattered_2d(n):
    """n disjoint pairs of triangles."""
    a = np.array([[0.0, 0.0, 0.0], [1.0, 0.0, 0.0], [0.0, 1.0, 0.0], [1.0, 1.0, 0.0]])
    corners, ids = [], []
    for k in range(n):
        v = 0.1 * a * (1.0 + 0.3 * np.sin(k)) + np.array([0.3 * (k % 7), 0.3 * (k // 7), 0.0])
        for t in ((0, 1, 2), (1, 3, 2)):
            corners.append(v[list(t)])
            ids.append([4 * k + j for j in t])
    c = np.array(corners)
    return z.Mesh(2, np.array(ids, dtype=np.int32), c, np.zeros(2 * n, dtype=np.uint8))


def _state(mesh):
    return W.cell_average(mesh, lambda x: W.conserved(1.0 + 0.2 * np.sin(3 * x[:, 0]), 0.3 + 0.1 * x[:, 1], -0.2 + 0 * x[:, 0],
                                                      0.1 * x[:, 2], 1.0 + 0.1 * (x ** 2).sum(axis=1), 1.4))


@pytest.mark.parametrize("flux_bc", [0, 1])
@pytest.mark.parametrize("flux", [z.ZFV_FLUX_HLLC, z.ZFV_FLUX_RUSANOV])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 40])
def test_tiles_of_many_faces(gpu, n, flux, flux_bc):
    # all pairs but the first are ghosts (first order, no flux between them):
    # the first tile then holds its pair's face and 64 boundary faces
    mesh = _scattered_2d(n)
    mesh.ghost[2:] = 1
    u = _state(mesh)
    p = z.make_params(n_dims=2, order=2, n_biased=3, flux=flux, flux_bc=flux_bc)
    ref = Oracle(mesh, p).rate(u)
    errs = rel_err(z.Solver(mesh, p).rate(u), ref)
    assert max(errs) <= TOL, errs


@pytest.mark.parametrize("flux_bc", [0, 1])
@pytest.mark.parametrize("flux", [z.ZFV_FLUX_HLLC, z.ZFV_FLUX_RUSANOV])
@pytest.mark.parametrize("dims,n", [(2, 8), (2, 12), (2, 13), (3, 7), (3, 8)])
def test_bounded_meshes(gpu, dims, n, flux, flux_bc):
    mesh = (z.lattice_mesh_2d(n, jitter=0.2, seed=9, periodic=(False, False), ghost_layers=2) if dims == 2
            else z.ball_mesh_3d(n, radius=1.0, ghost_radius=0.6, jitter=0.1, seed=5))
    u = _state(mesh)
    p = z.make_params(n_dims=dims, order=3, flux=flux, flux_bc=flux_bc)
    errs = rel_err(z.Solver(mesh, p).rate(u), Oracle(mesh, p).rate(u))  # ghosts included
    assert max(errs) <= TOL, errs


@pytest.mark.parametrize("n", [8, 9, 33])
def test_fluxes_cancel_over_a_periodic_mesh(gpu, n):
    # every face's flux leaves one cell and enters the other, whichever
    # wavefronts evaluate it: the sum over the mesh is rounding of the cells' sums
    wl = W.vortex_2d(n=n)
    L = z.Solver(wl.mesh, wl.params).rate(wl.u0)
    vol = wl.mesh.volumes()
    for v in (0, 1, 2, 4):
        assert abs((vol * L[:, v]).sum()) <= 1e-14 * np.abs(vol * L[:, v]).sum() * np.sqrt(wl.mesh.n_cells)
