"""The update that the kernels run (update.hpp), on the host under
AddressSanitizer: over the tiles the setup builds, per-cell states and the
device's order of bookkeeping, the lanes of a wavefront and the tiles of a
launch in any order.  Rates, steps under the frozen BC, the time loop with and
without step rejection, and batches equal loops over faces and cells bit for
bit; every table entry is checked against the mesh's faces."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "zisafvm_amd", "csrc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("update") / "update_check")
    subprocess.run(["g++", "-std=c++17", "-g", "-O1", "-fopenmp", "-ffp-contract=off", "-fsanitize=address",
                    "-fno-omit-frame-pointer", "-w", os.path.join(HERE, "cpp", "update_check.cpp"),
                    os.path.join(CSRC, "setup.cpp"), os.path.join(CSRC, "mesh.cpp"), "-o", out], check=True)
    return out


# dims, cells per side (pairs: pairs), mesh, flux BC, edge degree: less than one
# tile, partly filled last tiles, tiles of more than 64 faces, each kernel shape
CASES = [(2, 4, "bounded", 1, 1), (2, 6, "periodic", 0, 3), (2, 9, "bounded", 1, 5), (2, 8, "ghosts", 1, 3),
         (2, 11, "ghosts", 0, 5), (2, 1, "pairs", 1, 1), (2, 16, "pairs", 1, 1), (2, 17, "pairs", 0, 3),
         (2, 40, "pairs", 1, 5), (3, 5, "bounded", 1, 2), (3, 7, "ghosts", 0, 3), (3, 8, "ghosts", 1, 2)]


@pytest.mark.parametrize("flux", [0, 1])
@pytest.mark.parametrize("dims,n,mesh,flux_bc,edge_deg", CASES)
def test_update_on_the_host(check, dims, n, mesh, flux_bc, edge_deg, flux):
    r = subprocess.run([check, str(dims), str(n), mesh, str(flux), str(flux_bc), str(edge_deg), str(7 * n + flux)],
                       capture_output=True, text=True, timeout=300)
    print(r.stdout[-2000:], r.stderr[-4000:])
    assert r.returncode == 0 and "update_check: OK" in r.stdout
