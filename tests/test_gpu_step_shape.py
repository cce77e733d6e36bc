"""twmc_query reports the launch that steps the batch: workgroups, threads and LDS by step
kernel, so that the batches on either side of a rule are seen to run on different ones
(the other tests compare their results)."""
import numpy as np
import pytest
import torch

from helpers import c2_spec, system
from pincosimulator_amd import Engine, System
from test_gpu_band import band_matrix, matrix_spec
from test_gpu_sparse import sparse_matrix, spec_of

pytestmark = pytest.mark.gpu

TAB = 768 * 8  # FP64 Box-Muller tables


def shape(spec, n_traj, precision, kernel="generic"):
    eng = Engine(System(**spec) if "coupling" in spec else system(spec), precision=precision, kernel=kernel)
    eng.run(np.arange(n_traj, dtype=np.uint64))
    st = eng.stats()
    eng.close()
    return st["grid"], st["block"], st["lds_bytes"]


def lattice(nx, ny, **kw):
    return c2_spec(**dict(dict(nx=nx, ny=ny, dt=0.005, t_end=0.005 * 3.25, frame_steps=3), **kw))


def drawn(**kw):
    return dict(F={"base": 0.9 - 0.4j, "noise": ("uniform", 0.3)}, **kw)


@pytest.mark.parametrize("precision,nx,ny,per_cu", [(64, 4, 4, 8), (64, 5, 13, 4), (64, 16, 16, 2), (32, 1, 64, 16),
                                                    (32, 9, 21, 2)])
def test_ahead_line(precision, nx, ny, per_cu):
    line = per_cu * torch.cuda.get_device_properties(0).multi_processor_count
    print(f"{nx}x{ny}, FP{precision}", flush=True)
    few, many = (shape(lattice(nx, ny), b, precision) for b in (line, line + 1))
    n = nx * ny
    assert few[:2] == (line, 256 if n <= 128 else 512)
    assert many[1] == (64 if n <= 128 else 128)


@pytest.mark.parametrize("nx,ny,kw,line,block,other", [(16, 16, drawn(), 12, 128, 128), (1, 512, {}, 4, 256, 256),
                                                       (64, 64, {}, 2, 1024, 1024)])
def test_nn_line_fp64(nx, ny, kw, line, block, other):
    """Even rows: the LDS kernel's own launch below; one trajectory fewer per CU in its registers."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    line = line * cus + (nx == 64)
    print(f"{nx}x{ny}", flush=True)
    few, many = (shape(lattice(nx, ny, **kw), b, 64) for b in (line - 1, line))
    pairs = (nx * ny + 2 * block - 1) // (2 * block) * block
    assert many[1:] == (block, TAB + 16 + pairs * 2 * 16 * (2 if kw else 1))
    assert few[1] == other and few[2] != many[2]


@pytest.mark.parametrize("nx,ny,kw,block", [(5, 13, {}, 64), (27, 41, {}, 576), (63, 63, {}, 1024), (16, 16, drawn(), 128),
                                            (64, 64, drawn(), 1024)])
def test_nn_fp32(nx, ny, kw, block):
    print(f"{nx}x{ny}", flush=True)
    slots = 1024 if 512 < nx * ny / 2 <= 1024 else block * (2 if nx * ny > 2048 else 1)
    got = shape(lattice(nx, ny, **kw), 4500, 32, kernel="auto")
    assert got[1:] == (block, 16 + slots * 2 * 8 * (2 if kw else 1))


def test_matrix_and_stacked():
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    spec = spec_of(sparse_matrix(72, 3, 5), frame_steps=3, t_end=0.005 * 3.25)
    assert shape(spec, 8 * cus, 64)[:2] == (8 * cus, 256)
    sparse = shape(spec, 8 * cus + 1, 64)
    assert sparse[0] <= (8 * cus + 4) // 4 and sparse[1] == 256
    dense = spec_of(np.eye(72) + 0.1, frame_steps=3, t_end=0.005 * 3.25)
    assert shape(dense, 300, 64)[:2] == (300, 256)
    assert shape(matrix_spec(band_matrix(72, 2, False, 3), frame_steps=3, t_end=0.005 * 3.25), 300, 32, "band")[1] == 64
    stack = shape(lattice(36, 50), 5000, 32, kernel="auto")
    assert stack[1:] == (1024, 64 + 2 * 4096 * 8) and stack[0] <= 2 * cus
    assert shape(lattice(64, 64), 64, 32, kernel="auto")[:2] == (64, 1024)
