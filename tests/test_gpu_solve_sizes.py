"""The batched LU and triangular solves (camp_eval_lu_solve) at the sizes
where their program changes shape: tails shorter than a wavefront's 64
unknowns, exactly 64, one more (a head of one pivot), the last size solved in
the right-hand side itself (128) and the first in a scratch vector (129).

The matrices I - gamma J are strictly diagonally dominant by rows (condition
number below 1e3), so an elimination without pivoting is backward stable and
the solution agrees with LAPACK's to 1e3 * nv * eps < 1e-10."""
import numpy as np
import pytest

from camp_amd.core import CampSolver
from camp_amd.mechanisms import synthetic_mechanism

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nv", [5, 8, 9, 31, 63, 64, 65, 72, 100, 127, 128, 129, 160])
def test_lu_solve_sizes(nv):
    mech = synthetic_mechanism(nv, nv + 4 if nv < 100 else nv // 2, seed=nv)
    n_cells = 5
    sol = CampSolver(mech, n_cells)
    pat = sol.pattern()
    rows = pat["rowval"]
    cols = np.repeat(np.arange(sol.nv), np.diff(pat["colptr"]))
    rng = np.random.default_rng(nv)
    jac = rng.uniform(-1.0, 1.0, size=(n_cells, sol.nnz)) * 10.0 ** rng.uniform(-4, 1, sol.nnz)
    gamma = 0.8
    m = np.zeros((n_cells, sol.nv, sol.nv))
    m[:, rows, cols] = -gamma * jac
    diag = rows == cols
    off = np.abs(m).sum(2) - np.abs(m[:, range(sol.nv), range(sol.nv)])
    jac[:, diag] = -(1.0 + off[:, rows[diag]]) / gamma
    m[:, rows, cols] = -gamma * jac
    m += np.eye(sol.nv)
    b = rng.standard_normal((n_cells, sol.nv))
    rc, x = sol.eval_lu_solve(jac, gamma, b)
    assert rc == 0
    want = np.linalg.solve(m, b[:, :, None])[:, :, 0]
    assert np.max(np.abs(x - want)) <= 1e-10 * np.max(np.abs(want))
