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
from camp_amd.mechanisms import Mechanism, Reaction, synthetic_mechanism

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


def _chains(nv, n_cells):
    """Two unbranched chains of nv / 2 species, each turning into the next: the
    factors have no fill and no products, so an infinite entry reaches the
    unknowns after it in its chain and no others."""
    half = nv // 2
    rx = [Reaction("ARRHENIUS", [i], [(i + 1, 1.0)], {"A": 1.0e-3})
          for i in range(nv - 1) if i + 1 != half]
    sol = CampSolver(Mechanism(["S%d" % i for i in range(nv)], [1] * nv, [1.0e-8] * nv, rx), n_cells)
    pat = sol.pattern()
    rows = pat["rowval"]
    cols = np.repeat(np.arange(sol.nv), np.diff(pat["colptr"]))
    jac = np.where(rows == cols, -1.0, 1.0) * np.ones((n_cells, sol.nnz))
    return sol, rows, cols, jac


@pytest.mark.parametrize("nv", [20, 100, 160])
def test_infinite_values_stay_where_the_pattern_has_them(nv):
    """An infinite Jacobian entry or right-hand side in one chain: the
    factorisation (whose pivots are all finite) succeeds, and past 128 solver
    variables every unknown that the entry does not reach is the one of the same
    cell without it, bit for bit.  Up to 128 the solution is NaN as a whole."""
    half, at = nv // 2, nv - 7
    sol, rows, cols, jac = _chains(nv, 3)
    b = np.random.default_rng(nv).uniform(1.0, 2.0, (3, nv))
    jac[1, (rows == at) & (cols == at - 1)] = np.inf
    b[2, at] = np.inf
    rc, x = sol.eval_lu_solve(jac, 0.5, b)
    assert rc == 0
    clean = sol.eval_lu_solve(np.where(np.isinf(jac), 1.0, jac), 0.5, np.where(np.isinf(b), 1.0, b))[1]
    assert np.array_equal(x[0], clean[0])
    for c in (1, 2):
        if nv > 128:
            assert np.array_equal(x[c, :at], clean[c, :at])
            assert np.isposinf(x[c, at:]).all()
        else:
            assert np.isnan(x[c]).all()


@pytest.mark.parametrize("scale", [2.0 ** -1000, 2.0 ** -1060, 2.0 ** 1015])
def test_quotients_at_the_ends_of_the_range(scale):
    """x = D^-1 b of 160 decoupled unknowns is a division each, correctly rounded
    also where the right-hand side or the quotient is subnormal or nearly
    overflows."""
    nv = 160
    sol, rows, cols, jac = _chains(nv, 2)
    rng = np.random.default_rng(5)
    diag = rng.uniform(1.0, 100.0, (2, nv)) * 2.0 ** rng.integers(-3, 3, (2, nv))
    jac[:, rows != cols] = 0.0
    jac[:, rows == cols] = -diag[:, rows[rows == cols]]
    b = rng.uniform(1.0, 2.0, (2, nv)) * scale
    rc, x = sol.eval_lu_solve(jac, 1.0, b)
    assert rc == 0 and np.array_equal(x, b / (1.0 + diag))
