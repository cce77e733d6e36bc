"""Matrix hopping above the ahead kernel's sizes and batches stores several frames per
launch too: advanced segment by segment, in uneven pieces and at once, with and without
the states, with a frame after every step and steps after the last one, with several
trajectories per wave and a last wave partly filled, drawn and fixed parameters, and one
launch per frame with a drive F(t): the same states, means and sums bit for bit, and the
frames against the FP64 oracle."""
import numpy as np
import pytest

from helpers import FP32_BAR, rel_err
from pincosimulator_amd import Engine, System
from test_gpu_sparse import reference, sparse_matrix, spec_of

pytestmark = pytest.mark.gpu

RUNS = {"300": (300, 6, 21, dict(frame_steps=3, t_end=0.005 * 31.25), {}),
        "single steps": (450, 4, 5, dict(frame_steps=1, t_end=0.005 * 70.25), {}),
        "no first frame": (512, 3, 530, dict(frame_steps=9, t_end=0.005 * 40.25), dict(store_initial=False)),
        "packed": (20, 3, 2101, dict(frame_steps=4, t_end=0.005 * 24.25), {}),
        "drive": (300, 6, 21, dict(frame_steps=3, t_end=0.005 * 31.25), {})}


@pytest.mark.parametrize("name", list(RUNS))
@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("traj", [False, True])
def test_frames_in_groups(name, precision, traj):
    n, most, n_traj, kw, opt = RUNS[name]
    spec = spec_of(sparse_matrix(n, most, n), **kw)
    spec["omega"] = {"base": spec["omega"], "noise": ("gaussian", 0.2)}
    if name == "drive":
        rng = np.random.default_rng(n)
        spec["F_t"] = (np.array([0.02, 0.06, 0.11]), rng.normal(size=(3, n)) + 1j * rng.normal(size=(3, n)))
        spec["F"] = 0.0
    print(f"{name}, FP{precision}, states {traj}", flush=True)
    eng = Engine(System(**spec), precision=precision, kernel="generic")
    ids = np.arange(n_traj, dtype=np.uint64) * 9
    res = []
    for piece in (1, 3, 10 ** 6):
        info = eng.begin(ids, traj=traj, final=True, **opt)
        while info["segments_done"] < info["n_segments"]:
            eng.advance(piece)
            info = eng.info()
        res.append(eng.read())
    eng.close()
    assert res[0].n_frames > 1
    for r in res[1:]:
        for k in ("beta_final", "traj_m2", "traj_m4", "sum_n", "sum_n2", "sum_beta") + (("traj",) if traj else ()):
            np.testing.assert_array_equal(getattr(r, k), getattr(res[0], k))
        assert not np.any(r.sum_nk)
    if traj and "store_initial" not in opt:
        ref = reference(spec, ids[[0, -1]])
        assert rel_err(res[2].traj[[0, -1]], ref) < (FP32_BAR if precision == 32 else 1e-9)
