"""Block-Jacobi PCG with one launch per iteration, at the edges of its shapes.

A work-group takes 1, 2, 4 or 8 vertex rows (up to 256, 512, 1024 and 2048
vertices); larger systems take two launches per iteration. The reference is
the plain block-Jacobi PCG of its own kernels on the same system, which the
deflated solve is without coarse columns.

Bars: iteration counts to a relative residual of 1e-6 agree to one (the two
sum in different orders, so a residual may end up on either side of the
tolerance); with the coarse space the costs of the accepted states agree to
1e-8 relative with plain block-Jacobi PCG solving to 1e-11 in every step (the
solves stop at 1e-10 of the right-hand side, and an accepted step's cost
depends on the remaining error to second order; a rejected candidate's does to
first order, times the condition of the system, and is left out).
"""
import numpy as np
import pytest

from maplab_amd import abi, learned, problem
from maplab_amd.solver import DeviceProblem

pytestmark = pytest.mark.gpu


def opts(**kw):
    o = abi.default_options()
    for k, v in kw.items():
        setattr(o, k, v)
    return o


def walk(n, per=12):
    return problem.workload_map(2, seed=4, num_keyframes=n, num_landmarks=per * n)


@pytest.mark.parametrize("n", [2, 5, 33, 256, 257, 258, 512, 514, 1025, 1026, 2048, 2049, 2050])
def test_iterations_match_the_plain_pcg(n):
    with DeviceProblem(walk(n)) as dev:
        o = opts(pcg_coarse_nodes=-1)
        got = learned.rcs_pcg_iterations(dev, o, 1e2, abi.PRECOND_DEFLATED, 1e-6, 20000)
        want = learned.rcs_pcg_iterations(dev, o, 1e2, abi.PRECOND_BLOCK_JACOBI, 1e-6, 20000)
        capped = learned.rcs_pcg_iterations(dev, o, 1e2, abi.PRECOND_DEFLATED, 1e-30, 3)
    print(f"{n} keyframes: {got} iterations, plain {want}", flush=True)
    assert want > 0 and abs(got - want) <= max(1, want // 50)
    assert capped == -1


@pytest.mark.parametrize("n", [40, 300, 1026])
def test_tight_tolerances_are_reached(n):
    # The coarse space takes fewer iterations than the plain PCG, also where
    # the residual has fallen to 1e-12 of the right-hand side.
    with DeviceProblem(walk(n)) as dev:
        got, want = (learned.rcs_pcg_iterations(dev, opts(), 1e4, pc, 1e-12, 20000)
                     for pc in (abi.PRECOND_DEFLATED, abi.PRECOND_BLOCK_JACOBI))
    print(f"{n} keyframes: {got} iterations, plain {want}", flush=True)
    assert 0 < got < want


@pytest.mark.parametrize("n", [40, 257, 520, 1026])
def test_deflated_log_matches_the_plain_pcg(n):
    m = walk(n)
    logs = []
    for kw in (dict(pcg_relative_tolerance=1e-10),
               dict(pcg_relative_tolerance=1e-11, pcg_preconditioner=abi.PRECOND_BLOCK_JACOBI)):
        with DeviceProblem(m) as dev:
            sm, rows = dev.solve(opts(max_num_iterations=3, pcg_max_iterations=50000, **kw))
            logs.append((np.array([r.cost for r in rows]), dev.download_state(),
                         [r.step_is_successful for r in rows]))
        with DeviceProblem(m) as dev:
            _, again = dev.solve(opts(max_num_iterations=3, pcg_max_iterations=50000, **kw))
            np.testing.assert_array_equal([r.cost for r in again], logs[-1][0])
            np.testing.assert_array_equal(dev.download_state()[0], logs[-1][1][0])
    assert logs[0][2] == logs[1][2]
    ok = np.array(logs[0][2], bool)
    ok[0] = True  # the start
    assert ok[1:].any()
    np.testing.assert_allclose(logs[0][0][ok], logs[1][0][ok], rtol=1e-8)


def test_partial_sums_of_large_maps_give_the_same_solve():
    # Above 2048 vertices an iteration is two launches: both sums of its
    # partials, in every work-group or once, give the same bits.
    m = walk(2100)
    logs = []
    for partials in (0, 1, 2):
        with DeviceProblem(m) as dev:
            dev.set_schedule(4, 4, 1, partials)
            _, rows = dev.solve(opts(max_num_iterations=2, pcg_relative_tolerance=1e-4, pcg_max_iterations=200))
            logs.append(([(r.cost, r.linear_solver_iterations) for r in rows], dev.download_state()[0]))
    for log, state in logs[1:]:
        assert log == logs[0][0]
        np.testing.assert_array_equal(state, logs[0][1])
