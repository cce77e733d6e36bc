"""Inference on either side of the number of rows from which the layer-by-layer products
take it (8192, 4096 with up to three layers of up to 64), against the FP64 numpy oracle
with the bar of test_gpu_mlp.py (1e-5 of the largest output), and training steps of a
small batch between them: both paths use the same buffers."""
import numpy as np
import pytest

from oracle import mlp_oracle as mo
from pincosimulator_amd.mlp import MLP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in,hidden,depth,n_out,limit", [(5, 16, 2, 7, 4096), (5, 40, 3, 34, 8192), (3, 96, 1, 9, 8192)])
def test_forward_by_rows(n_in, hidden, depth, n_out, limit):
    ws = mo.widths(n_in, hidden, depth, n_out)
    m = MLP(n_in, n_out, n_hidden=hidden, n_hidden_layers=depth, seed=5)
    rng = np.random.default_rng(limit)
    x = rng.normal(size=(limit + 1, n_in)).astype(np.float32)
    t = rng.normal(size=(limit + 1, n_out)).astype(np.float32)
    for rows in (limit + 1, limit, limit + 1, 3):
        print(f"mlp {n_in}-{depth}x{hidden}-{n_out} rows {rows}", flush=True)
        yo, _ = mo.forward(m.params.astype(np.float64), ws, x[:rows].astype(np.float64))
        y = m.forward(x[:rows])
        assert np.max(np.abs(y - yo)) < 1e-5 * np.max(np.abs(yo))
        m.train(x[:130], t[:130], epochs=1, batch=65)
    m.close()
