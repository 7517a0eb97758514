"""libqbh.so on the CPU: loads, exports the header's API, host-side logic matches the oracle."""
import ctypes
import os
import re

import numpy as np
import pytest

from oracle.basis import Basis, UnitCell, density_grid, factorizable

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def header_functions():
    src = open(os.path.join(ROOT, "include", "qbh.h")).read()
    return sorted(set(re.findall(r"^\s*(?:int|const char\*)\s+(qbh_\w+)\s*\(", src, re.M)))


def test_library_exports_every_declared_function():
    from qball_amd import capi
    L = capi.lib()
    names = header_functions()
    assert len(names) >= 20
    for n in names:
        assert hasattr(L, n), n
        assert n in capi.SIGNATURES, n


def test_context_without_gpu_fails_cleanly():
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    from qball_amd import capi
    h = ctypes.c_void_p()
    rc = capi.lib().qbh_ctx_create(0, None, ctypes.byref(h))
    assert rc != 0 and not h.value


@pytest.mark.parametrize("a,ecut,real", [
    (np.diag([20.52] * 3), 12.5, True),
    (np.diag([10.26] * 3), 12.5, False),
    (np.array([[7.1, 0.3, -0.2], [0.9, 6.4, 0.5], [-0.4, 1.1, 8.3]]), 9.0, True),
    (np.array([[7.1, 0.3, -0.2], [0.9, 6.4, 0.5], [-0.4, 1.1, 8.3]]), 9.0, False),
    (np.array([[0.0, 3.825, 3.825], [3.825, 0.0, 3.825], [3.825, 3.825, 0.0]]), 15.0, True),
])
def test_rods_build_matches_oracle(a, ecut, real):
    from qball_amd import capi
    r = capi.rods_build(a, ecut, real=real)
    ob = Basis(UnitCell(a), ecut, force_complex=not real)
    for k in ("rod_h", "rod_k", "rod_lmin", "rod_size"):
        assert np.array_equal(r[k], getattr(ob, k)), k
    assert r["np"] == ob.np


def test_factorizable_matches_oracle():
    from qball_amd import capi
    for n in range(1, 3000):
        assert capi.factorizable(n) == factorizable(n)


def test_workload_density_grid_matches_oracle():
    from qball_amd.workload import density_grid_np
    a = np.diag([20.52] * 3)
    assert density_grid_np(a, 12.5) == density_grid(UnitCell(a), 12.5)[1]


def test_enl_of_a_failed_call_is_an_error(tmp_path):
    """nl_read_enl on a Hamiltonian whose stream cannot be synchronised (no device here) reports
    it instead of returning what an earlier call left in the pinned slot."""
    import shutil
    import subprocess
    import torch
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    from qball_amd import lib
    lib()
    src = tmp_path / "enl.hip"
    src.write_text("""
#include "qbh_ham.h"
#include <cstdio>
int main() {
  double pin[qbh::PIN_SIZE] = {}, red = 0.0, enl = -1.0;
  pin[qbh::PIN_ENL] = 42.0;  // an earlier call's energy
  qbh::Ctx c;
  c.pin = pin;
  qbh::Ham h;
  h.ctx = &c;
  h.P = 1;
  h.red = &red;
  const int r = qbh::nl_read_enl(&h, nullptr, &enl);
  c.pin = nullptr;
  std::printf("%d %g %zu\\n", r, enl, c.last_error.size());
}
""")
    pkg = os.path.join(ROOT, "qball_amd")
    obj, exe = str(tmp_path / "enl.o"), str(tmp_path / "enl")
    subprocess.run([hipcc, "-std=c++17", "--cuda-host-only", "-I" + os.path.join(pkg, "csrc"), "-c",
                    str(src), "-o", obj], check=True)
    subprocess.run([hipcc, obj, "-o", exe, "-L" + pkg, "-lqbh", "-Wl,-rpath," + pkg], check=True)
    rc, enl, msg = subprocess.run([exe], check=True, capture_output=True,
                                  text=True).stdout.split()
    assert int(rc) != 0 and float(enl) != 42.0 and int(msg) > 0


@pytest.mark.parametrize("which,R,C,Q,tile,slices", [
    # measured slower on 64-wide tiles: FP32 slices of 5500 to 9088 (F and the product after it),
    # FP64 with few workgroups a CU (4 slices 3.13 ms, large tile with 24 2.86)
    (1, 1600, 300, 290810, 128, 53), (1, 1600, 390, 290810, 128, 40),
    (1, 1600, 520, 290810, 128, 32), (0, 1320, 900, 57052, None, 8), (0, 2048, 300, 145406, None, 16),
    # faster on small tiles
    (0, 32, 16, 2302, 32, 29), (0, 256, 128, 18278, 32, 16), (1, 256, 128, 18278, 32, 35),
    (1, 1560, 390, 145406, 64, 40), (0, 1320, 200, 57052, 64, 24), (2, 16, 2302, 32, 32, 1),
    # as fast on the large tile
    (0, 2048, 1024, 145838, 128, 16), (2, 1024, 145838, 2048, 128, 1), (4, 1024, 1024, 145838, 128, 14)])
def test_product_tiles(which, R, C, Q, tile, slices):
    """Tile and slice rule of the matrix-core products at measured shapes (None: either tile,
    with at least that many slices)."""
    from helpers import product_tile
    got = product_tile(which, R, C, Q)
    if tile is None:
        assert got[1] >= slices
    else:
        assert got == (tile, slices)
