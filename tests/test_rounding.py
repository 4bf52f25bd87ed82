"""Rounding errors of the kernels' math against 80-bit arithmetic: the rate of
change evaluated in double precision on the library's own tables, and single
formulas whose faster forms must lose no more than the plain ones."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import zisafvm_amd as z
from zisafvm_amd import workloads as W
from emu_binding import Emu
from conftest import pressure_scale

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "zisafvm_amd", "csrc")


def _ptr(a):
    return ctypes.c_void_p(a.ctypes.data)


def _library(folder, name, *more):
    out = str(folder / (name + ".so"))
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-fopenmp", "-ffp-contract=off", "-w", "-shared", "-o", out,
                    os.path.join(HERE, "cpp", name + ".cpp")] + [os.path.join(CSRC, m) for m in more], check=True)
    return ctypes.CDLL(out)


@pytest.fixture(scope="module")
def extended(tmp_path_factory):
    return _library(tmp_path_factory.mktemp("extended"), "extended", "setup.cpp", "mesh.cpp")


@pytest.fixture(scope="module")
def units(tmp_path_factory):
    return _library(tmp_path_factory.mktemp("rounding"), "rounding")


def _weno_rusanov(w):
    w.params.reconstruction, w.params.flux = z.ZFV_WENO_AO, z.ZFV_FLUX_RUSANOV
    return w


# the root mean square error over the cells and variables, relative to each
# variable's largest rate, that the plain formulas reach: a division per
# quotient, the basis functions one by one, the source's face terms in full
# (weights, point values, HLLC's star state and the face terms have other forms)
CASES = {
    "vortex_o3": (lambda s: W.vortex_2d(n=16, order=3, beta=3.0 + s, seed=s), 2.26e-15),
    "vortex_o4": (lambda s: W.vortex_2d(n=16, order=4, beta=3.0 + s, seed=s), 2.28e-15),
    "vortex_o3_weno_rusanov": (lambda s: _weno_rusanov(W.vortex_2d(n=16, order=3, beta=3.0 + s, seed=s)), 2.32e-15),
    "isothermal_o3": (lambda s: W.isothermal_2d(n=14, order=3, amplitude=1e-4, seed=s), 2.47e-11),
    "isothermal_o4": (lambda s: W.isothermal_2d(n=14, order=4, amplitude=1e-4, seed=s), 4.89e-11),
    "isentropic_o3": (lambda s: W.isentropic_2d(n=14, order=3, amplitude=1e-4, seed=s), 3.61e-11),
}


def _check(extended, make, name):
    case, bound = CASES[name]
    errs = []
    for seed in (1, 2, 3, 4):
        w = case(seed)
        u = np.ascontiguousarray(w.u0)
        ref = np.zeros(u.shape, dtype=np.longdouble)
        mesh = w.mesh.c_struct()
        assert extended.ext_rate(ctypes.byref(mesh), ctypes.byref(w.params), _ptr(u), _ptr(ref), 0, None) == 0
        got = make(w.mesh, w.params).rate(u)
        keep = np.ix_(w.mesh.ghost == 0, [0, 1, 2, 4])
        errs.append(float((((got - ref)[keep] / np.abs(ref[keep]).max(axis=0)) ** 2).mean()))
    err = np.sqrt(np.mean(errs))
    print(name, "rms", err, "bound", bound, flush=True)
    assert err <= bound


@pytest.mark.parametrize("name", sorted(CASES))
def test_rate_rounds_no_worse_than_the_plain_formulas(extended, name):
    _check(extended, Emu, name)


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(CASES))
def test_rate_on_the_device_rounds_no_worse_than_the_plain_formulas(gpu, extended, name):
    _check(extended, z.Solver, name)


@pytest.mark.parametrize("order,RT", [(3, 4.0), (3, 0.74), (3, 0.72), (3, 0.5), (4, 4.0), (4, 0.74)])
def test_series_averages_leave_out_less_than_rounding(extended, order, RT):
    # inside the range, at its edge, across it and outside, in 80-bit arithmetic:
    # the terms left out of the averages (1e-17) and of the exponentials near
    # them (3e-18) times the largest pressures, against the pressures that cancel
    mesh = z.lattice_mesh_2d(10, jitter=0.2, seed=4, periodic=(True, False), ghost_layers=3)
    p = z.make_params(n_dims=2, order=order, equilibrium=z.ZFV_EQ_ISOTHERMAL, gravity=z.ZFV_GRAVITY_AXIAL, gravity_g=1.0)
    if order == 4:
        p.edge_deg = 4

    def f(x):
        rho = np.exp(-x[:, 1] / RT)
        return W.conserved(rho, 0.1 * rho, 0.0 * rho, 0.0 * rho,
                           RT * rho * (1.0 + 1e-2 * np.sin(6.28 * x[:, 0])), 1.4)

    u = np.ascontiguousarray(W.cell_average(mesh, f))
    cm, both, part = mesh.c_struct(), [], np.zeros(2)
    for series in (0, 1):
        out = np.zeros(u.shape, dtype=np.longdouble)
        assert extended.ext_rate(ctypes.byref(cm), ctypes.byref(p), _ptr(u), _ptr(out), series, _ptr(part)) == 0
        both.append(out)
    diff = np.abs(both[1] - both[0])[mesh.ghost == 0].max() / pressure_scale(mesh, u, 1.4)
    print("order", order, "RT", RT, "part of the range", part, "difference", float(diff), flush=True)
    assert diff <= 1e-16
    assert (diff > 0.0) == (part[0] <= 1.0)  # the series ran where a cell is in range


def test_hllc_of_a_state_at_rest_is_its_pressure(units):
    # no mass or energy crosses the face, exactly; the pressure to a few places
    rng = np.random.default_rng(3)
    n, gamma = 20000, 1.4
    p = np.exp(rng.uniform(-3.0, 3.0, n))
    u = np.stack([np.exp(rng.uniform(-3.0, 3.0, n)), np.zeros(n), np.zeros(n), p / (gamma - 1.0)], axis=1)
    a = rng.uniform(0.0, 2.0 * np.pi, n)
    nn = np.stack([np.cos(a), np.sin(a)], axis=1)
    f = np.empty((n, 4))
    units.unit_hllc(ctypes.c_double(gamma), n, _ptr(u), _ptr(u), _ptr(nn), _ptr(f))
    assert not f[:, 0].any() and not f[:, 3].any()
    assert (np.abs(f[:, 1:3] - p[:, None] * nn) <= 4 * np.finfo(float).eps * p[:, None]).all()


@pytest.mark.parametrize("dims,degree", [(2, 1), (2, 2), (2, 3), (3, 1), (3, 2)])
def test_nested_polynomial_is_the_sum_over_the_basis(units, dims, degree):
    from oracle import zfv_ref as R

    units.unit_poly.restype = ctypes.c_double
    dof = [1, 3, 6, 10][degree] if dims == 2 else [1, 4, 10][degree]
    rng = np.random.default_rng(11)
    for _ in range(50):
        a, c, X = rng.normal(size=dof), rng.normal(size=dof), np.append(rng.uniform(-2.0, 2.0, dims), [0.0] * (3 - dims))
        c[:dims + 1] = 0.0
        ref = R.poly_eval(dims, degree, a[:, None], c, X)[0]
        # each of the terms and sums of both forms rounds once
        size = np.abs(a) @ (np.maximum(1.0, np.abs(X).max()) ** degree + np.abs(c))
        assert abs(units.unit_poly(dims, degree, dof, _ptr(a), _ptr(c), _ptr(X)) - ref) <= 4 * dof * 2.3e-16 * size


@pytest.mark.parametrize("gamma", [7.0 / 5.0, 5.0 / 3.0, 4.0 / 3.0, 1.5, 2.0, 1.2, 9.0 / 7.0, 11.0 / 9.0, 1.1, 3.0, 1.3])
def test_equilibrium_power_to_half_a_place(units, gamma):
    # as accurate as pow: half a unit in the last place, and 1 % of one beyond
    # (the powers of 1.4e1 .. 4.5 orders of magnitude, both sides of one)
    x = np.exp(np.random.default_rng(5).uniform(-5.0, 5.0, 100000))
    y = np.empty_like(x)
    units.unit_eq_pow(ctypes.c_double(gamma), len(x), _ptr(x), _ptr(y))
    ref = x.astype(np.longdouble) ** np.longdouble(1.0 / (gamma - 1.0))
    ulp = np.spacing(ref.astype(float))
    assert (np.abs(y - ref) <= 0.51 * ulp).all(), float((np.abs(y - ref) / ulp).max())
