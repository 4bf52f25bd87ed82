"""Up to the line from which the linear isentropic solve no longer starts at its
closed-form root (kRootsApart), the iteration from the reference's guess reaches
that very root: random states and potentials, the iteration and its limits as
the kernels have them, here in numpy."""
import os
import re

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "zisafvm_amd", "csrc")
N = 200000


def _solve(R0, E0, v, off, x0, x1):
    """Newton's iteration of R = u / (2 K), E = R (u + v / u) / 2 with u = h +
    off for (h, K) from (x0, x1): converged, h, K."""
    at0, at1 = 1e-13 * 2.0 * E0 / R0, 1e-13 * E0 / R0 ** 2
    dx0 = np.full(N, np.inf)
    dx1, ok = dx0.copy(), np.ones(N, dtype=bool)
    last = []  # the steps before
    for it in range(20):
        run = ok & ~((abs(dx0) <= at0) & (abs(dx1) <= at1))
        a, u = 0.5 / x1, x0 + off
        R, E = a * u, x1 * a * a * (u * u + v)
        f0, f1, inv = R0 - R, E0 - E, 1.0 / (R * R - a * E)
        dx0 = np.where(run, (E * f0 - R * f1) * inv, dx0)
        dx1 = np.where(run, x1 * (R * f0 - a * f1) * inv, dx1)
        x0, x1 = np.where(run, x0 - dx0, x0), np.where(run, x1 - dx1, x1)
        if it >= 4:  # the rates of convergence that end the iteration
            rates = [np.log(abs(d) / abs(p)) / np.log(abs(p) / abs(q)) for d, p, q in zip((dx0, dx1), *last)]
            ok &= ~(run & ~((dx0 <= at0) & (dx1 <= at1)) & ~((rates[0] >= 0) & (rates[1] >= 0)))
        last = [(dx0, dx1)] + last[:1]
    return ok & (abs(dx0) <= 1e3 * at0) & (abs(dx1) <= 1e3 * at1), x0, x1


@pytest.mark.parametrize("deviations", [0.0, 1.0, 6.0])
def test_guess_and_root_lead_to_the_same_equilibrium(deviations):
    line = float(re.search(r"kRootsApart = ([0-9.]+);", open(os.path.join(CSRC, "stage_math.hpp")).read()).group(1))
    rng = np.random.default_rng(1)
    R0, E0 = 10 ** rng.uniform(-6, 6, N), 10 ** rng.uniform(-6, 6, N)
    r = 2.0 * E0 / R0
    part = np.where(np.arange(N) % 2, rng.uniform(0.0, line, N), 10 ** rng.uniform(-14.0, np.log10(line), N))
    v = 0.25 * part * r * r
    off = deviations * rng.uniform(-1.0, 1.0, N) * np.sqrt(v)  # the reference potential off the mean
    with np.errstate(all="ignore"):
        found, h, K = _solve(R0, E0, v, off, r.copy(), E0 / R0 ** 2)
    u = 0.5 * (r + np.sqrt(r * r - 4.0 * v))
    assert found.all()
    assert (abs(h - (u - off)) <= 1e-11 * r).all() and (abs(K - 0.5 * u / R0) <= 1e-11 * K).all()
