"""The sums of a frame that a launch of several frames stores are those of one launch per
frame, bit for bit: a run's results do not depend on the pieces it is advanced in.  More
trajectories than a group of many frames would need slots for, lattice and matrix hopping."""
import numpy as np
import pytest

from helpers import c2_spec, system
from pincosimulator_amd import Engine, System
from test_gpu_sparse import sparse_matrix, spec_of

pytestmark = pytest.mark.gpu

RUNS = {"4x4": (16, 1500), "1x64": (64, 700), "9x11": (99, 600), "matrix": (72, 400)}


@pytest.mark.parametrize("name", list(RUNS))
@pytest.mark.parametrize("precision", [32, 64])
def test_sums_by_pieces(name, precision):
    n, n_traj = RUNS[name]
    print(f"{name}, FP{precision}, {n_traj} trajectories", flush=True)
    if name == "matrix":
        spec = spec_of(sparse_matrix(n, 3, 5), frame_steps=3, t_end=0.005 * 90.25,
                       omega={"base": 0.5, "noise": ("gaussian", 0.2)})
    else:
        nx, ny = map(int, name.split("x"))
        spec = c2_spec(nx=nx, ny=ny, dt=0.01, frame_steps=3, t_end=0.01 * 90.25)
    eng = Engine(System(**spec) if name == "matrix" else system(spec), precision=precision, kernel="generic")
    res = []
    for piece in (1, 7, 10 ** 6):
        info = eng.begin(np.arange(n_traj, dtype=np.uint64))
        while info["segments_done"] < info["n_segments"]:
            eng.advance(piece)
            info = eng.info()
        res.append(eng.read())
    eng.close()
    assert res[0].n_frames == 31
    for r in res[1:]:
        for k in ("sum_n", "sum_n2", "sum_nk", "sum_beta", "traj_m2", "traj_m4"):
            np.testing.assert_array_equal(getattr(r, k), getattr(res[0], k))
