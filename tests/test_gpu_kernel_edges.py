"""Kernels at the sizes where their shapes change, against the oracle or the
general path."""
import numpy as np
import pytest

from maplab_amd import abi, learned, problem
from maplab_amd.solver import DeviceProblem
from oracle import gnn_oracle as go
from test_gpu_learned import _dataset, opts, walk
from test_gpu_quality import many_observer_map
from test_oracle_quality import quality_options

pytestmark = pytest.mark.gpu


# A system without a coarse space (up to 31 vertices) is solved by one
# work-group in one launch: 3 x 64 rows of 16 waves x 12 columns.
@pytest.mark.parametrize("n", [2, 3, 4, 11, 12, 13, 21, 22, 23, 31, 32, 33])
def test_one_launch_pcg_matches_the_plain_pcg(n):
    m = problem.workload_map(2, seed=6, num_keyframes=n, num_landmarks=30 * n)
    logs = []
    for pc in (abi.PRECOND_DEFLATED, abi.PRECOND_BLOCK_JACOBI):
        with DeviceProblem(m) as dev:
            _, rows = dev.solve(opts(max_num_iterations=4, pcg_preconditioner=pc, pcg_relative_tolerance=1e-12,
                                     pcg_max_iterations=5000))
            logs.append([(r.cost, r.step_is_successful, r.linear_solver_iterations) for r in rows])
    print(f"{n} keyframes: {logs}", flush=True)
    # Accepted states: solves to 1e-12 differ to second order in the cost.
    a, b = ([c for k, (c, ok, _) in enumerate(log) if ok or k == 0] for log in logs)
    np.testing.assert_allclose(a, b, rtol=1e-9)
    if n <= 31:  # the same method, summed in another order
        # (a residual near the tolerance may fall on either side of it)
        for (_, _, i), (_, _, j) in zip(*logs):
            assert abs(i - j) <= max(2, j // 10)


# Four landmarks share a wave (16 lanes each), rays beyond those kept in LDS
# are read again.
@pytest.mark.parametrize("n", [2, 15, 16, 17, 63, 64, 65, 255, 256, 257])
def test_landmark_quality_observer_counts(oracle, n):
    m = many_observer_map(n_obs=max(n, 5), seed=n)
    keep = np.concatenate([np.flatnonzero(m.obs_landmark == 0)[:n], np.flatnonzero(m.obs_landmark == 1)])
    for k in ("obs_vertex", "obs_landmark", "obs_camera", "obs_keypoint", "obs_sigma"):
        setattr(m, k, np.ascontiguousarray(getattr(m, k)[keep]))
    for angle in (5.0, 40.0):
        o = quality_options(min_observation_angle_deg=angle, min_observers=3)
        with DeviceProblem(m) as dev:
            assert dev.landmark_quality(o).tolist() == oracle.landmark_quality(m, o).tolist()


@pytest.mark.parametrize("tangent", [False, True])
@pytest.mark.parametrize("blocks", [(), (0,), (8,), (1, 4, 7), tuple(range(9))])
def test_evaluate_writes_the_blocks_asked_for(tangent, blocks):
    m = problem.workload_map(2, seed=8, num_keyframes=20, num_landmarks=333)
    with DeviceProblem(m) as dev:
        res, jac, cost = dev.evaluate(tangent=tangent)
        res_b, jac_b, cost_b = dev.evaluate(tangent=tangent, blocks=blocks)
    np.testing.assert_array_equal(res, res_b)
    assert cost == cost_b and set(jac_b) == set(blocks)
    for b in blocks:
        np.testing.assert_array_equal(jac[b], jac_b[b])


# Rows not a multiple of 4 or 128, and a row without edges (one vertex).
# Tolerances: the BF16 activations' (test_gpu_learned.py).
@pytest.mark.parametrize("sizes", [(4, 2), (3, 2), (6, 2, 5), (127,), (129,), (90, 2, 41)])
def test_network_sizes(sizes):
    data, _, _ = _dataset([walk(n, 20 * n, n) for n in sizes])
    rng = np.random.default_rng(1)
    params = learned.init_params(2) + (rng.normal(size=learned.num_params()) * 0.02).astype(np.float32)
    theta, loss, grad = learned.evaluate(data, params)
    theta2, loss2, _ = learned.evaluate(data, params, want_grad=False)
    np.testing.assert_array_equal(theta, theta2)
    assert loss == loss2
    g = go.Graph(data.row_ptr, data.col, data.rev, data.node_feat, data.edge_feat)
    ref_loss, ref_grad, ref_theta = go.loss_and_grad(params.astype(np.float64), g, data.qc.astype(np.float64))
    print(f"{sizes}: {data.nodes} rows, {data.slots} slots", flush=True)
    assert np.abs(theta - ref_theta).max() <= 2e-2 * np.abs(ref_theta).max()
    assert abs(loss - ref_loss) <= 1e-3 * abs(ref_loss) + 1e-6
    if np.linalg.norm(ref_grad) > 0:
        assert np.linalg.norm(grad - ref_grad) < 3e-2 * np.linalg.norm(ref_grad)


@pytest.mark.parametrize("field, value", [("col", -1), ("col", 1 << 20), ("rev", -1), ("rev", 1 << 24)])
def test_network_refuses_indices_out_of_range(field, value):
    data, _, _ = _dataset([walk(5, 100, 1)])
    idx = getattr(data, field)
    idx[len(idx) // 2] = value
    with pytest.raises(Exception):
        learned.evaluate(data, learned.init_params(0))
