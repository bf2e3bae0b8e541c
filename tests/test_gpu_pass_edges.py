"""The CG's chained passes at the edges of their blocks and tiles (64 cells a wavefront, 256 a tile,
1,024 blocks of one tile), for every pressure path of the backend, against a banded direct solve."""
import ctypes

import numpy as np
import pytest
import scipy.linalg as sl

from dopamine_amd._lib import lib
from test_gpu_pressure_abi import _call

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("selector,ksp", [("jacobi", "cg"), ("jacobi", "pipecg"), ("mixed", "cg"), ("boomeramg", "cg"),
                                          ("mixed-multigrid", "cg")])
@pytest.mark.parametrize("n", [2, 63, 65, 255, 257, 2047, 2049, 16385, 262145])
def test_chain_solve(n, selector, ksp):
    """A chain with couplings 1 and a diagonal raised by 0.5 (well conditioned, so the solution's
    relative error is at most 10 times the residual's 1e-10)."""
    L = lib()
    own, nb = np.arange(n - 1), np.arange(1, n)
    coeff, skip = np.ones(n - 1), np.zeros(n - 1, dtype=int)
    diag = np.full(n, 2.5)
    diag[[0, -1]] = 1.5
    b = np.random.default_rng(n).standard_normal(n)
    band = np.zeros((3, n))
    band[0, 1:], band[1], band[2, :-1] = -1.0, diag, -1.0
    want = sl.solve_banded((1, 1), band, b)
    L.fvm_petsc_insert_option.argtypes = [ctypes.c_char_p]
    L.fvm_petsc_set_pressure_solver.argtypes = [ctypes.c_char_p]
    L.fvm_petsc_insert_option(f"-ksp_type {ksp}".encode())
    L.fvm_petsc_backend_finalize()
    L.fvm_petsc_set_pressure_solver(selector.encode())
    try:
        print(f"[gpu] chain of {n} cells, {selector} {ksp}", flush=True)
        rc, x, its, res = _call(n, own, nb, skip, diag, b, coeff, np.zeros(n), 1e-10, 1e-300, 1)
    finally:
        L.fvm_petsc_insert_option(b"-ksp_type cg")
        L.fvm_petsc_backend_finalize()
    assert rc == 0
    assert np.linalg.norm(x - want) <= 1e-9 * np.linalg.norm(want)
