"""Programs at the edges of what the kernels' tables can describe."""
import ctypes
import dataclasses

import numpy as np
import pytest
import torch

from camp_amd.core import CampSolver
from camp_amd.mechanisms import (Mechanism, Reaction, box_mechanism, cb05_scale_mechanism,
                                 synthetic_cells)
from camp_amd.multiphase import multiphase_cells, multiphase_mechanism

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


def ring_mechanism(n):
    """n species, each turning into the next at 1e-3 / s: a sparse Jacobian
    whose factors fill little, so that vectors, not factors, take the LDS."""
    rx = [Reaction("ARRHENIUS", [i], [((i + 1) % n, 1.0)], {"A": 1.0e-3}) for i in range(n)]
    return Mechanism(["S%d" % i for i in range(n)], [1] * n, [1.0e-10] * n, rx, rel_tol=1.0e-6)


def ring_solution(y0, t):
    """The ring's exact solution: its modes are Fourier modes."""
    n = y0.shape[1]
    w = np.exp(-2j * np.pi * np.arange(n) / n) - 1.0
    return np.fft.ifft(np.fft.fft(y0, axis=1) * np.exp(1.0e-3 * t * w), axis=1).real


ENV = np.array([298.0, 101325.0])


@pytest.mark.parametrize("n", [720, 1300])
def test_layers_of_a_wide_mechanism(n):
    """Four cells of 720 species, or two of 1300, are more than a CU's LDS: f
    and J run with fewer wavefronts a block (the rates are 1e-3 y to rounding),
    also after a small solver has launched the same kernels, and the step does
    not see an error that the layers' set-up left behind.  The step is not
    stiff: an error per step of 1e-6 of the solution over at most some hundred
    steps stays under 1e-3."""
    n_cells = 3
    gpu = CampSolver(ring_mechanism(n), n_cells)
    env = np.tile(ENV, (n_cells, 1))
    y0 = np.random.default_rng(3).uniform(1.0, 2.0, (n_cells, n))
    small = CampSolver(ring_mechanism(100), n_cells)
    assert small.eval_deriv(y0[:, :100], env)[0] == 0
    want = 1.0e-3 * (np.roll(y0, 1, axis=1) - y0)
    for est in (False, True):
        rc, f = gpu.eval_deriv(y0, env, 1.0, est)
        assert rc == 0 and np.allclose(f, want, rtol=1e-12, atol=1e-15)
        rc, jac = gpu.eval_jac(y0, env, 1.0)
        assert rc == 0 and np.allclose(np.abs(jac), 1.0e-3, rtol=1e-12, atol=0.0)
    y = y0.copy()
    assert gpu.solve(y, env, 0.0, 60.0) == 0
    assert np.allclose(y, ring_solution(y0, 60.0), rtol=1e-3, atol=0.0)


def test_layers_where_the_estimate_has_no_scratch():
    """400 species in a ring of 6300 reactions: f's own LDS fits a CU, its
    vector y - y_hist does not and is formed entry by entry."""
    n, n_rxn, n_cells = 400, 6300, 2
    rx = [Reaction("ARRHENIUS", [r % n], [((r + 1) % n, 1.0)], {"A": 2.0 ** -14})
          for r in range(n_rxn)]
    mech = Mechanism(["S%d" % i for i in range(n)], [1] * n, [1.0e-10] * n, rx, rel_tol=1.0e-6)
    gpu = CampSolver(mech, n_cells)
    env = np.tile(ENV, (n_cells, 1))
    y0 = np.random.default_rng(4).uniform(1.0, 2.0, (n_cells, n))
    rate = y0 * np.bincount(np.arange(n_rxn) % n) * 2.0 ** -14
    want = np.roll(rate, 1, axis=1) - rate
    assert gpu.eval_jac(y0, env, 1.0)[0] == 0
    rc, f = gpu.eval_deriv(y0, env, 1.0, True)
    assert rc == 0 and np.allclose(f, want, rtol=1e-12, atol=1e-15)


def test_large_launch_of_a_wide_mechanism():
    """1300 species: the default placement fits a CU's LDS, the placement with
    the factors in global memory (and all vectors in LDS) does not.  A launch
    of many cells runs all the same (tolerance as above)."""
    n, n_cells = 1300, 4100
    gpu = CampSolver(ring_mechanism(n), n_cells)
    y0 = np.tile(np.random.default_rng(3).uniform(1.0, 2.0, (4, n)), (n_cells // 4, 1))
    y = y0.copy()
    assert gpu.solve(y, np.tile(ENV, (n_cells, 1)), 0.0, 60.0) == 0
    assert np.allclose(y, ring_solution(y0, 60.0), rtol=1e-3, atol=0.0)


@pytest.mark.parametrize("n, cells_per_block", [(300, 4), (1300, 1), (1500, 1)])
def test_placements_that_do_not_fit(n, cells_per_block):
    """Four cells of 300 species a workgroup fit with placement 1 only, one of
    1300 with placement 1 only, one of 1500 with none: the others run with
    their vectors in global memory, and the result is the same bit for bit, also
    with every wavefront's memory filled with NaNs before each cell."""
    n_cells = 5
    y0 = np.random.default_rng(5).uniform(1.0, 2.0, (n_cells, n))
    got = []
    for place in (1, 0, 2):
        gpu = CampSolver(ring_mechanism(n), n_cells)
        assert gpu.set_placement(place) == place
        assert gpu.set_cells_per_block(cells_per_block) == cells_per_block
        gpu.set_poison(place == 2)
        y = y0.copy()
        assert gpu.solve(y, np.tile(ENV, (n_cells, 1)), 0.0, 60.0) == 0
        got.append(y)
    assert np.allclose(got[0], ring_solution(y0, 60.0), rtol=1e-3, atol=0.0)
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])


def test_many_aerosol_species_and_few_reactions(oracle_lib):
    """80 bins of 11 solutes, two of them partitioning: the phases' and ion
    pairs' quotients do not fit the scratch at once and go in chunks, and the
    species' partial derivatives not at all.  No more LDS is taken for them:
    two cells a workgroup fit.  f and J as in the oracle (1e-12 relative: both
    accumulate in extended precision, and the chunks keep the order), the step
    as the oracle's at the 1e-4 / 1e-8 bar of the other multi-phase tests."""
    mp = multiphase_mechanism(1, n_bins=80, n_simpol=2, n_aqeq=1)
    n = 2
    cells = multiphase_cells(mp, n, seed=2)
    kw = dict(rel_tol=1e-8, abs_tol=np.full(mp.n_state, 1e-12), max_steps=100000)
    gpu, ref = CampSolver(mp, n, **kw), oracle_lib.Oracle(mp, n, **kw)
    for s in (gpu, ref):
        s.set_rates(cells.rates)
    st, env = cells.state, cells.env
    ref.update_env(env)
    rc, jac = gpu.eval_jac(st, env, 10.0)
    want = np.stack([ref.eval_jac(c, st[c], 10.0)[1] for c in range(n)])
    assert rc == 0 and (np.abs(jac - want) <= 1e-12 * np.abs(want) + 1e-280).all()
    rc, f = gpu.eval_deriv(st, env, 10.0, False)
    want = np.stack([ref.eval_f(c, st[c], 10.0, False)[1] for c in range(n)])
    assert rc == 0 and (np.abs(f - want) <= 1e-12 * np.abs(want) + 1e-280).all()
    assert gpu.set_cells_per_block(2) == 2
    a, b = st.copy(), st.copy()
    assert gpu.solve(a, env, 0.0, 1.0) == 0
    assert ref.run(b, env, 0.0, 1.0, mode=1) == 0
    assert (np.abs(a - b) <= 1e-4 * np.abs(b) + 1e-8).all()


def test_layer_calls_of_a_large_grid_return_their_memory():
    """f, then one factorisation and solve of 30000 cells (680 MB of device
    arrays): what the second call took is free again, and the calls give the
    same results as before, whichever came before them."""
    n = 30000
    mech = cb05_scale_mechanism(1)
    gpu = CampSolver(mech, n)
    cells = synthetic_cells(mech, 1, seed=2)
    state, env = np.tile(cells.state, (n, 1)), np.tile(cells.env, (n, 1))
    gpu.set_rates({k: np.repeat(v, n) for k, v in cells.rates.items()})
    f0 = gpu.eval_deriv(state, env)[1]
    free = torch.cuda.mem_get_info()[0]
    rows = gpu.pattern()["rowval"]
    cols = np.repeat(np.arange(gpu.nv), np.diff(gpu.pattern()["colptr"]))
    jac = np.tile(np.where(rows == cols, -1.0, 1e-3), (n, 1))
    b = np.ones((n, gpu.nv))
    x0 = gpu.eval_lu_solve(jac, 0.5, b)[1]
    assert torch.cuda.mem_get_info()[0] > free - (64 << 20)
    assert np.array_equal(gpu.eval_deriv(state, env)[1], f0)
    assert np.array_equal(gpu.eval_lu_solve(jac, 0.5, b)[1], x0)


@pytest.mark.parametrize("n, per_species", [(50, 18), (100, 3), (200, 2)])
@pytest.mark.parametrize("place", [0, 1, 2])
def test_more_reactions_than_a_lane_holds_and_than_factors(n, per_species, place):
    """Rings with several reactions a species: more than 256 terms, whose rate
    constants the lanes no longer hold all of, more rate constants than LU
    factors (J stages them in the factors' place), and more than 128 solver
    variables (solved in a scratch vector), one step with every placement and
    every wavefront's memory filled with NaNs (tolerance as above)."""
    n_cells = 5
    rx = [Reaction("ARRHENIUS", [i], [((i + 1) % n, 1.0)], {"A": 1.0e-3 / per_species})
          for _ in range(per_species) for i in range(n)]
    mech = Mechanism(["S%d" % i for i in range(n)], [1] * n, [1.0e-10] * n, rx, rel_tol=1.0e-6)
    gpu = CampSolver(mech, n_cells)
    assert len(rx) > 256 and (n > 128 or len(rx) > gpu.lu_nnz)
    gpu.set_placement(place)
    gpu.set_poison(True)
    y0 = np.random.default_rng(6).uniform(1.0, 2.0, (n_cells, n))
    y = y0.copy()
    assert gpu.solve(y, np.tile(ENV, (n_cells, 1)), 0.0, 60.0) == 0
    assert np.allclose(y, ring_solution(y0, 60.0), rtol=1e-3, atol=0.0)


def test_layers_ignore_an_error_left_by_the_caller():
    """A HIP call of the caller's that failed (a device that is not there) leaves
    its error for the next one to ask: f and J do not take it for theirs."""
    mech = box_mechanism(1)
    cells = synthetic_cells(mech, 2, seed=2)
    gpu = CampSolver(mech, 2)
    gpu.set_rates(cells.rates)
    assert gpu.eval_deriv(cells.state, cells.env)[0] == 0
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64.so" in line)
    hip = ctypes.CDLL(path)
    for call in (gpu.eval_deriv, gpu.eval_jac):
        assert hip.hipSetDevice(99) != 0
        assert call(cells.state, cells.env)[0] == 0
    hip.hipGetLastError()
