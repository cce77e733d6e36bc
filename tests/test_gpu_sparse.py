"""Matrix hopping with few nonzeros per column, on the sparse step kernel
(kernel="generic", FP64, or FP32 with parameters drawn per trajectory): per
trajectory against the FP64 oracle over its forms -- periodic and open Lieb
chains, asymmetric random couplings of one to six nonzeros per column (C_ij !=
C_ji pins the product's direction), odd and single sites, one to 32 trajectories
per wave with a last wave partly filled, two to eight sites per lane, drawn
parameters, F(t), resumed steps -- and at its limit of 512 sites.  FP64 bar 1e-9
as for the other FP64 paths, FP32 bar FP32_BAR."""
import numpy as np
import pytest

import oracle
from helpers import FP32_BAR, rel_err
from pincosimulator_amd import Engine, System

pytestmark = pytest.mark.gpu


def sparse_matrix(n, most, seed):
    """Random couplings, at most `most` nonzeros in a column, some columns empty."""
    rng = np.random.default_rng(seed)
    C = np.zeros((n, n))
    for j in range(n):
        k = int(rng.integers(0, most + 1)) if j else min(most, n)
        C[rng.choice(n, min(k, n), replace=False), j] = rng.uniform(-1.0, 1.0, min(k, n))
    return C


def spec_of(C, **kw):
    n = C.shape[0]
    rng = np.random.default_rng(n)
    s = dict(nx=1, ny=n, dt=0.005, gamma=1.0, J=0.0, U=0.1 + 0.02j, F=1.2 * np.exp(1j * rng.uniform(0, 6, n)),
             omega=0.3 * rng.standard_normal(n), beta_init=0.0, beta_sigma=0.5, frame_steps=20, seed=77, t_start=0.0,
             t_end=0.3, lattice="matrix", coupling=C, detuning=0.2, onsite="detuning-E")
    s.update(kw)
    return s


def reference(spec, ids):
    p = dict(spec, lattice=oracle.LAT_DENSE, E=spec["omega"])
    return np.array([oracle.run_trajectory(p, int(t))[0] for t in ids])


def check(spec, ids, precision, tol):
    eng = Engine(System(**spec), precision=precision, kernel="generic")
    res = eng.run(ids, traj=True)
    eng.close()
    pick = sorted({0, 1, len(ids) // 2, len(ids) - 2, len(ids) - 1} & set(range(len(ids))))
    ref = reference(spec, ids[pick])
    assert res.traj[pick].shape == ref.shape
    err = rel_err(res.traj[pick], ref)
    print(f"  {err:.2e}")
    assert err < tol
    z = res.traj
    for k, v in (("sum_n", np.abs(z) ** 2), ("sum_beta", z)):
        assert rel_err(getattr(res, k), v.sum(axis=0)) < 1e-12
    assert np.all(res.sum_nk == 0)


CASES = [("lieb24 periodic", oracle.lieb_coupling(24, 4.0, 4.0, True), 33), ("lieb24", oracle.lieb_coupling(24, 1.0, 1.0, False), 7),
         ("one site", np.zeros((1, 1)), 130), ("two sites", sparse_matrix(2, 1, 3), 67), ("odd", sparse_matrix(37, 3, 5), 11),
         ("six a column", sparse_matrix(45, 6, 6), 10), ("128 sites", sparse_matrix(128, 3, 8), 5),
         ("129 sites, four lanes' worth", sparse_matrix(129, 4, 9), 3), ("257 sites", sparse_matrix(257, 2, 10), 3),
         ("512 sites", sparse_matrix(512, 6, 11), 2)]


@pytest.mark.parametrize("name,C,n_traj", CASES, ids=[c[0].replace(" ", "-") for c in CASES])
@pytest.mark.parametrize("form", ["fp64", "fp64-drawn", "fp32-drawn", "fp64-drive"])
def test_sparse_matches_oracle(name, C, n_traj, form):
    n = C.shape[0]
    spec = spec_of(C)
    rng = np.random.default_rng(n + 1)
    if form.endswith("drawn"):
        spec["omega"] = {"base": spec["omega"], "noise": ("gaussian", 0.2)}
        spec["F"] = {"base": spec["F"], "noise": ("uniform", 0.3)}
    if form == "fp64-drive":
        spec["F_t"] = (np.array([0.02, 0.11, 0.2]), rng.normal(size=(3, n)) + 1j * rng.normal(size=(3, n)))
        spec["F"] = 0.0
    print(f"sparse {name} {form}", flush=True)
    check(spec, np.arange(n_traj, dtype=np.uint64) * 5 + 2, 32 if form == "fp32-drawn" else 64,
          FP32_BAR if form == "fp32-drawn" else 1e-9)


@pytest.mark.parametrize("n,n_traj", [(24, 60000), (72, 20000), (200, 6000)])
@pytest.mark.parametrize("precision", [32, 64])
def test_many_trajectories(n, n_traj, precision):
    """Enough trajectories for four and eight sites per lane and several rounds of the grid."""
    spec = spec_of(sparse_matrix(n, 3, n), t_end=0.05, frame_steps=5,
                   omega={"base": 0.5, "noise": ("gaussian", 0.2)})
    print(f"sparse FP{precision} {n} sites, {n_traj} trajectories", flush=True)
    check(spec, np.arange(n_traj, dtype=np.uint64) + 9, precision, 1e-9 if precision == 64 else FP32_BAR)


def test_uncoupled_site_that_overflows_stays_alone():
    """A site without bonds that runs away must not reach its neighbours in the index."""
    C = np.zeros((10, 10))
    C[:5, :5] = sparse_matrix(5, 2, 1)
    spec = spec_of(C, t_end=0.2)
    F = np.array(spec["F"])
    F[[5, 9]] = 1e200
    spec["F"] = F
    print("sparse with a site that overflows", flush=True)
    eng = Engine(System(**spec), precision=64, kernel="generic")
    res = eng.run(np.arange(3), traj=True)
    eng.close()
    ref = reference(spec, range(3))
    keep = [0, 1, 2, 3, 4, 6, 7, 8]
    assert not np.all(np.isfinite(res.traj[..., [5, 9]]))
    assert rel_err(res.traj[..., keep], ref[..., keep]) < 1e-9


def test_resume_continues_the_noise():
    spec = spec_of(oracle.lieb_coupling(24, 1.0, 1.0, True), t_end=0.4)
    ids = np.arange(6, dtype=np.uint64)
    print("sparse resume", flush=True)
    whole = Engine(System(**spec), precision=64).run(ids, final=True).beta_final
    half = Engine(System(**dict(spec, t_end=0.2)), precision=64).run(ids, final=True)
    rest = Engine(System(**dict(spec, t_start=0.2, t_end=0.4)), precision=64)
    out = rest.run(ids, init="previous", beta_prev=half.beta_final, step0=half.n_steps, final=True).beta_final
    np.testing.assert_array_equal(out, whole)
