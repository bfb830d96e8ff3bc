"""Which systems the deflated PCG iterates in one launch: those of up to 512
vertices, and larger ones whose S is sparse enough that a work-group of 4 or 8
rows is not the longer way. On both sides of each line the solve takes the
steps of plain block-Jacobi PCG, in no more iterations.

Bar: both solve to 1e-12 of the right-hand side. An accepted step's cost depends
on the rest to second order, times the condition of the system; on the
2049-keyframe walk, the worst here, the first step's cost is 1e-7 from the
converged one at 1e-10, with either solver, 2e-10 at 1e-12 and 6e-11 at 1e-13."""
import numpy as np
import pytest

from maplab_amd import abi, problem
from maplab_amd.solver import DeviceProblem

pytestmark = pytest.mark.gpu

# workload (1: a ring that every keyframe sees whole), seed, keyframes, landmarks, one launch
MAPS = [(1, 1, 300, 1000, True), (1, 1, 513, 800, True), (1, 1, 540, 800, False), (1, 1, 1000, 500, False),
        (1, 1, 1100, 400, False), (2, 1, 600, 12000, False), (2, 1, 1000, 20000, True), (2, 1, 1025, 20500, True),
        (2, 1, 1026, 20520, False), (2, 1, 2000, 24000, False), (2, 3, 2000, 24000, True), (2, 3, 2049, 24000, True),
        (2, 3, 2060, 24000, False)]


@pytest.mark.parametrize("workload, seed, n, landmarks, one", MAPS)
def test_dispatch_by_vertices_and_density(workload, seed, n, landmarks, one):
    m = problem.workload_map(workload, seed=seed, num_keyframes=n, num_landmarks=landmarks)
    runs = []
    for pc in (abi.PRECOND_DEFLATED, abi.PRECOND_BLOCK_JACOBI):
        o = abi.default_options()
        o.max_num_iterations = 2
        o.pcg_max_iterations = 20000
        o.pcg_preconditioner = pc
        o.pcg_relative_tolerance = 1e-12
        with DeviceProblem(m) as dev:
            if pc == abi.PRECOND_DEFLATED:
                k = abi.default_options()
                k.pcg_max_iterations = 20
                kt = dev.time_kernels(k, repeats=1)
            _, rows = dev.solve(o)
        runs.append(([r.cost for r in rows], [r.step_is_successful for r in rows],
                     np.array([r.linear_solver_iterations for r in rows])))
    V, B = kt.num_variable_vertices, kt.schur_blocks / kt.num_variable_vertices
    times = 0 if V <= 512 else 5 if V <= 1024 else 12
    want = V <= 2048 and V >= times * B
    print(f"{V} vertices, {B:.1f} blocks a row: one launch {want}", runs[0][2], runs[1][2], flush=True)
    assert (kt.pcg_update_ms == 0) == want
    assert want == one
    good = np.array(runs[0][1], bool)
    good[0] = True
    assert runs[0][1] == runs[1][1]
    np.testing.assert_allclose(np.array(runs[0][0])[good], np.array(runs[1][0])[good], rtol=1e-8)
    assert (runs[0][2][1:] <= runs[1][2][1:]).all()
