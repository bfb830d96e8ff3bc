"""Where one-launch PCG iterations stop when a single step takes r'r down by
more than 64 bits hold.

Nearly block-diagonal systems: every landmark is stored in the constant first
vertex; most are constant (their observations couple no two vertices), the rest
have a weight of 1/s^2 of theirs. Block-Jacobi leaves a relative residual of
about 1/s^2 after one iteration and 1/s^4 after two, so a relative tolerance of
1e-12 needs exactly two for s between 1e4 and 4e4 (about 1e-9 .. 1e-10, then its
square), where r'r falls by 1e18 and more in the first. The reference is plain
block-Jacobi PCG in numpy on the same S and rhs, and the device's own two-kernel
one.
"""
import numpy as np
import pytest

from maplab_amd import abi, learned, problem
from maplab_amd.solver import DeviceProblem

pytestmark = pytest.mark.gpu

TOL = 1e-12
RADIUS = 1e4


def rotation(q):
    x, y, z, w = q[:, 0], q[:, 1], q[:, 2], q[:, 3]
    return np.stack([1 - 2 * (y * y + z * z), 2 * (x * y + z * w), 2 * (x * z - y * w),
                     2 * (x * y - z * w), 1 - 2 * (x * x + z * z), 2 * (y * z + x * w),
                     2 * (x * z + y * w), 2 * (y * z - x * w), 1 - 2 * (x * x + y * y)], -1).reshape(-1, 3, 3)


def weakly_coupled(n, s, seed):
    m = problem.workload_map(2, seed=seed, num_keyframes=n, num_landmarks=40 * n).normalized()
    R, p = rotation(m.vertices[:, :4]), m.vertices[:, 4:]
    a = m.landmark_store_vertex
    pM = np.einsum("lji,lj->li", R[a], m.landmarks) + p[a]
    m.landmarks = (pM - p[0]) @ R[0].T
    m.landmark_store_vertex = np.zeros(m.num_landmarks, np.int32)
    m.vertex_constant = np.zeros(n, np.uint8)
    m.vertex_constant[0] = 1
    weak = np.arange(m.num_landmarks) % 8 == 0
    m.landmark_constant = (~weak).astype(np.uint8)
    m.obs_sigma = np.where(weak[m.obs_landmark], s, 1.0) * m.obs_sigma
    return m.normalized()


def plain_pcg_residuals(S, b, iterations):
    n = len(b) // 6
    Minv = [np.linalg.inv(S[6 * i:6 * i + 6, 6 * i:6 * i + 6]) for i in range(n)]
    prec = lambda r: np.concatenate([Minv[i] @ r[6 * i:6 * i + 6] for i in range(n)])
    x, r = np.zeros_like(b), b.copy()
    z = prec(r)
    p, rz = z.copy(), r @ z
    out = []
    for _ in range(iterations):
        q = S @ p
        alpha = rz / (p @ q)
        x, r = x + alpha * p, r - alpha * q
        z = prec(r)
        rz, old = r @ z, rz
        p = z + rz / old * p
        out.append(np.linalg.norm(r) / np.linalg.norm(b))
    return out


@pytest.mark.parametrize("n", [40, 300])
def test_stops_at_the_tolerance_and_not_before(n):
    got, plain = [], []
    scales = np.logspace(4.0, 4.6, 12)
    for k, s in enumerate(scales):
        with DeviceProblem(weakly_coupled(n, s, 1 + k)) as dev:
            o = abi.default_options()
            o.loss_type = abi.LOSS_TRIVIAL
            o.pcg_coarse_nodes = -1
            if n == 40:
                res = plain_pcg_residuals(*learned.rcs_system(dev, o, RADIUS), 2)
                assert res[0] > 10 * TOL and res[1] < 0.1 * TOL, res
            print(f"{n} keyframes, s {s:.3g}", flush=True)
            got.append(learned.rcs_pcg_iterations(dev, o, RADIUS, abi.PRECOND_DEFLATED, TOL, 100))
            plain.append(learned.rcs_pcg_iterations(dev, o, RADIUS, abi.PRECOND_BLOCK_JACOBI, TOL, 100))
    print(got, plain)
    assert plain == [2] * len(scales)
    assert got == plain


def test_stops_at_once_on_a_block_diagonal_system():
    # No landmark is variable: one iteration leaves rounding errors only.
    m = weakly_coupled(40, 1.0, 3)
    m.landmark_constant[:] = 1
    with DeviceProblem(m.normalized()) as dev:
        o = abi.default_options()
        o.loss_type = abi.LOSS_TRIVIAL
        o.pcg_coarse_nodes = -1
        for tol in (1e-6, 1e-12):
            assert learned.rcs_pcg_iterations(dev, o, RADIUS, abi.PRECOND_DEFLATED, tol, 100) == 1
        # A step is valid and the state finite, whatever the scalars cancel to.
        o.max_num_iterations = 3
        o.pcg_relative_tolerance = 1e-14
        sm, rows = dev.solve(o)
        v, l = dev.download_state()
        assert np.isfinite(v).all() and np.isfinite(l).all()
        assert rows[1].step_is_successful and sm.final_cost < sm.initial_cost
