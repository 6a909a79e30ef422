"""Programs at the edges of what the kernels' tables can describe."""
import dataclasses

import numpy as np
import pytest

from camp_amd.core import CampSolver
from camp_amd.mechanisms import box_mechanism, synthetic_cells

pytestmark = pytest.mark.gpu


def test_no_solver_variables(oracle_lib):
    """Every species constant: nothing to integrate, and the empty f, LU and
    solve programs must not be read past their ends.  As in the oracle, the
    step fails (its error norm is 0 / 0) and leaves the state alone; the layer
    entry points have nothing to return."""
    box = box_mechanism(1)
    mech = dataclasses.replace(box, var_type=[2] * box.n_state)
    n = 3
    cells = synthetic_cells(box, n, seed=2)
    gpu, ref = CampSolver(mech, n), oracle_lib.Oracle(mech, n)
    assert gpu.nv == 0
    for s in (gpu, ref):
        s.set_rates(cells.rates)
    assert gpu.eval_deriv(cells.state, cells.env, 1.0, True)[0] == 0
    assert gpu.eval_jac(cells.state, cells.env, 1.0)[0] == 0
    a, b = cells.state.copy(), cells.state.copy()
    assert gpu.solve(a, cells.env, 0.0, 60.0) == ref.run(b, cells.env, 0.0, 60.0, mode=1)
    assert np.array_equal(a, b)
