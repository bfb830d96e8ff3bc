"""Constant landmarks whose anchor vertex is variable: nothing is eliminated,
but their observations couple the observer with the anchor. The tile kernel
takes them as a factor 1e20 I of the anchor and 1e-20 of the observations', so
that the products of the two are theirs and the observations' own vanish
(k_landmark_prep). S and the right-hand side against the oracle entry by entry
(bars as in test_gpu_schur.py), and solves against the oracle's."""
import numpy as np
import pytest

from cases import tiny_map
from maplab_amd import abi, learned, problem
from maplab_amd.solver import DeviceProblem

pytestmark = pytest.mark.gpu

MAPS = {
    "one_camera": lambda: tiny_map(np.random.default_rng(11), dist_type=1, n_vertices=7, n_landmarks=60),
    "two_cameras_two_missions": lambda: tiny_map(np.random.default_rng(12), dist_type=2, n_vertices=12,
                                                 n_landmarks=150, global_missions=True, n_cameras=2),
    "several_tiles_a_landmark": lambda: tiny_map(np.random.default_rng(13), dist_type=1, n_vertices=300,
                                                 n_landmarks=4),
    "walk": lambda: problem.workload_map(2, seed=5, num_keyframes=50, num_landmarks=3000),
}


def R(q):
    """Rotation of a JPL quaternion (x y z w), frame to frame of the quaternion."""
    x, y, z, w = q
    return np.array([[1 - 2 * (y * y + z * z), 2 * (x * y + z * w), 2 * (x * z - y * w)],
                     [2 * (x * y - z * w), 1 - 2 * (x * x + z * z), 2 * (y * z + x * w)],
                     [2 * (x * z + y * w), 2 * (y * z - x * w), 1 - 2 * (x * x + y * y)]])


def constant(case, every):
    """Every n-th landmark constant, anchored in a vertex of its own choice."""
    m = MAPS[case]().normalized()
    for l in range(m.num_landmarks if m.num_landmarks < 1000 else 0):
        a, b = m.landmark_store_vertex[l], 1 + l % (m.num_vertices - 1)
        A, B = m.vertices[a], m.vertices[b]
        p = R(A[:4]).T @ m.landmarks[l] + A[4:]
        if m.vertex_mission[a] != m.vertex_mission[b]:
            F, G = m.baseframes[m.vertex_mission[a]], m.baseframes[m.vertex_mission[b]]
            p = R(G[:4]).T @ (R(F[:4]) @ p + F[4:] - G[4:])
        m.landmarks[l] = R(B[:4]) @ (p - B[4:])
        m.landmark_store_vertex[l] = b
    m.landmark_constant = (np.arange(m.num_landmarks) % every == 0).astype(np.uint8)
    variable = m.vertex_constant[m.landmark_store_vertex] == 0
    assert (variable & (m.landmark_constant == 1)).any()  # the case this file is about
    return m.normalized()


@pytest.mark.parametrize("case", list(MAPS))
@pytest.mark.parametrize("every", [1, 2, 3])
@pytest.mark.parametrize("radius", [1e4, 3.0])
def test_system_matches_oracle(oracle, case, every, radius):
    m = constant(case, every)
    o = abi.default_options()
    print(f"{case}: every {every}, radius {radius}", flush=True)
    with DeviceProblem(m) as dev:
        S, b = learned.rcs_system(dev, o, radius)
    ref_S, ref_b, _ = oracle.reduced_camera_system(m, o, radius)
    assert S.shape == ref_S.shape
    n = S.shape[0] // 6
    nz = lambda A: np.abs(A.reshape(n, 6, n, 6)).max(axis=(1, 3)) > 0
    assert nz(S)[nz(ref_S)].all()
    err = np.abs(S - ref_S).max()
    print(f"  max |S| {np.abs(ref_S).max():.3e}, max |dS| {err:.3e}, max |db| {np.abs(b - ref_b).max():.3e}")
    assert err <= 1e-12 * np.abs(ref_S).max()
    np.testing.assert_allclose(b, ref_b, rtol=0, atol=1e-12 * np.abs(ref_b).max())


@pytest.mark.parametrize("case", ["one_camera", "two_cameras_two_missions"])
@pytest.mark.parametrize("every", [1, 2])
def test_solve_matches_oracle(oracle, case, every):
    m = constant(case, every)
    o = abi.default_options()
    o.max_num_iterations = 5
    o.pcg_relative_tolerance = 1e-13
    with DeviceProblem(m) as dev:
        sm, rows = dev.solve(o)
        v, l = dev.download_state()
    ref_sm, _, ref_v, ref_l, _ = oracle.solve(m, o, linear_solver=oracle.SCHUR_DIRECT, threads=1)
    assert abs(sm.final_cost - ref_sm.final_cost) <= 1e-8 * ref_sm.final_cost
    np.testing.assert_allclose(v, ref_v, atol=1e-6)
    np.testing.assert_array_equal(l[m.landmark_constant == 1], m.landmarks[m.landmark_constant == 1])
