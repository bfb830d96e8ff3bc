"""The PCG of small systems without a coarse space (one launch a solve, up to
31 vertices) behind the calls that measure it, and one-launch iterations of
systems as small that have a coarse space."""
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


def ring(n):
    return problem.workload_map(1, seed=7, num_keyframes=n, num_landmarks=60 * n)


@pytest.mark.parametrize("n", [2, 10, 31, 32])
def test_time_kernels_times_the_solver_that_runs(n):
    # Up to 32 keyframes (one of them constant) a solve is one launch: there is
    # no time of an iteration's launch, and the count is that of the solve.
    with DeviceProblem(ring(n)) as dev:
        o = opts(max_num_iterations=1)
        kt = dev.time_kernels(o, repeats=3)
        plain = learned.rcs_pcg_iterations(dev, o, o.initial_trust_region_radius, abi.PRECOND_BLOCK_JACOBI,
                                           o.pcg_relative_tolerance, 20000)
        sm, rows = dev.solve(o)
    assert abs(kt.pcg_iterations - plain) <= max(1, plain // 50)
    assert kt.num_variable_vertices < 32 and kt.pcg_coarse_columns == 0
    assert kt.pcg_spmv_ms == 0 and kt.pcg_update_ms == 0 and kt.pcg_solve_ms > 0
    assert kt.pcg_iterations == rows[1].linear_solver_iterations > 0


def test_time_kernels_of_a_larger_map():
    with DeviceProblem(ring(40)) as dev:
        kt = dev.time_kernels(opts(), repeats=3)
    assert kt.pcg_spmv_ms > 0 and kt.pcg_update_ms == 0 and kt.pcg_coarse_columns > 0


@pytest.mark.parametrize("n", [2, 10, 32])
@pytest.mark.parametrize("nodes", [-1, 1, 2])
def test_one_launch_iterations_of_small_systems(n, nodes):
    # The plain PCG is the reference; a coarse space takes no more iterations
    # (but for the rounding of the last).
    with DeviceProblem(ring(n)) as dev:
        o = opts(pcg_coarse_nodes=nodes)
        got, plain = (learned.rcs_pcg_iterations(dev, o, 1e2, pc, 1e-8, 20000)
                      for pc in (abi.PRECOND_DEFLATED, abi.PRECOND_BLOCK_JACOBI))
    print(n, nodes, got, plain, flush=True)
    assert plain > 0 and got > 0
    if nodes < 0:
        assert abs(got - plain) <= max(1, plain // 50)
    else:
        assert got <= plain + 2


def test_an_iteration_cap_too_large_for_one_launch():
    # Above 16384 iterations a solve is one launch an iteration again: the same
    # system, sums in another order.
    out = []
    for cap in (16384, 16385, 20000):
        with DeviceProblem(ring(12)) as dev:
            o = opts(max_num_iterations=4, pcg_max_iterations=cap)
            one = dev.time_kernels(o, repeats=1).pcg_spmv_ms == 0
            assert one == (cap == 16384)
            sm, rows = dev.solve(o)
            out.append(([r.cost for r in rows], [r.linear_solver_iterations for r in rows], dev.download_state()[0]))
    for costs, its, v in out[1:]:
        np.testing.assert_allclose(costs, out[0][0], rtol=1e-9)
        assert np.abs(np.array(its) - out[0][1]).max() <= 1
        np.testing.assert_allclose(v, out[0][2], atol=1e-7)
    assert out[1][0] == out[2][0]
