"""The network workspace of a solver's handle (maplab_amd/csrc/ba_gnn.hip):
cleared in the order of the stream that uses it."""
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "maplab_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"


def test_cleared_on_the_callers_stream(tmp_path):
    if not os.path.exists(HIPCC) or shutil.which("g++") is None:
        pytest.skip("hipcc or g++ is not available")
    obj, exe = str(tmp_path / "ba_gnn.o"), str(tmp_path / "gnn_workspace_clear")
    subprocess.run([HIPCC, "--offload-host-only", "-O1", "-fPIC", "-std=c++17", "-I", CSRC, "-c", "-o", obj,
                    os.path.join(CSRC, "ba_gnn.hip")], check=True)
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I", CSRC,
                    # The object's device code is not built.
                    "-Wl,--unresolved-symbols=ignore-in-object-files", "-o", exe, os.path.join(HERE, "native", "gnn_workspace_clear.cc"), obj], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout + out.stderr


@pytest.mark.gpu
def test_first_solve_of_a_new_structure_repeats():
    """Every change of the active landmarks makes a new workspace; the first
    solve in it gives what the second gives, bit for bit."""
    from maplab_amd import abi, learned, problem
    from maplab_amd.solver import DeviceProblem
    m = problem.workload_map(2, seed=5, num_keyframes=150, num_landmarks=30000).normalized()
    o = abi.default_options()
    o.max_num_iterations = 2
    o.pcg_preconditioner = abi.PRECOND_LEARNED_DEFLATED
    rng = np.random.default_rng(1)
    with DeviceProblem(m) as dev:
        learned.Model.load().install(dev)
        for k in range(4):
            # Few landmarks, so that blocks of S come and go with the mask.
            mask = (rng.random(m.num_landmarks) < (0.02 + 0.01 * k)).astype(np.uint8)
            dev.set_landmark_active(mask)
            out = []
            for _ in range(2):
                print(f"mask {k}: {int(mask.sum())} landmarks", flush=True)
                dev.upload_state(m.vertices, m.landmarks)
                sm, rows = dev.solve(o)
                out.append((*dev.download_state(), np.array([r.cost for r in rows]),
                            np.array([r.linear_solver_iterations for r in rows])))
            for a, b in zip(*out):
                np.testing.assert_array_equal(a, b)
