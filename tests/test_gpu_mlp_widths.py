"""The network's fused kernels (widths up to 256) and the layer-by-layer ones
above, at the edges of their tiles: rows around the four-sample workgroups and
the 64-row gradient chunks, widths that are no multiple of four (4-byte weight
loads), of 16 (gradient tiles) and the widest fused one, one and many layers.
Against the FP64 numpy oracle with the bars of test_gpu_mlp.py (outputs 1e-5,
loss 1e-5, gradients 1e-4 of a layer's largest entry, an Adam step 1e-6)."""
import numpy as np
import pytest

from oracle import mlp_oracle as mo
from pincosimulator_amd.mlp import MLP

pytestmark = pytest.mark.gpu

# n_in, n_out, hidden width, hidden layers, rows
CASES = [(5, 34, 256, 3, 64), (1, 1, 1, 1, 1), (5, 34, 255, 2, 5), (3, 7, 65, 2, 3), (256, 256, 256, 1, 67),
         (17, 16, 16, 4, 130), (4, 34, 8, 15, 9), (6, 2, 5, 0, 66), (255, 33, 30, 2, 129), (5, 34, 260, 2, 66)]


def layers(ws):
    o = 0
    for a, b in zip(ws[:-1], ws[1:]):
        yield slice(o, o + a * b)
        yield slice(o + a * b, o + a * b + b)
        o += a * b + b


@pytest.mark.parametrize("n_in,n_out,hidden,depth,rows", CASES)
def test_widths_match_oracle(n_in, n_out, hidden, depth, rows):
    print(f"mlp {n_in}-{depth}x{hidden}-{n_out} rows {rows}", flush=True)
    ws = mo.widths(n_in, hidden, depth, n_out)
    m = MLP(n_in, n_out, n_hidden=hidden, n_hidden_layers=depth, seed=8)
    rng = np.random.default_rng(rows)
    p = m.params
    p += (0.1 * rng.normal(size=p.size)).astype(np.float32)  # biases too
    m.params = p
    x = rng.normal(size=(rows, n_in)).astype(np.float32)
    t = rng.normal(size=(rows, n_out)).astype(np.float32)
    w = (rng.uniform(size=(rows, n_out)) * 2.0).astype(np.float32)
    p64, x64, t64, w64 = (v.astype(np.float64) for v in (p, x, t, w))
    yo, _ = mo.forward(p64, ws, x64)
    y = m.forward(x)
    assert np.max(np.abs(y - yo)) < 1e-5 * np.max(np.abs(yo))
    lo, go = mo.loss_grad(p64, ws, x64, t64, w64)
    loss, g = m.loss_grad(x, t, w)
    assert abs(loss - lo) < 1e-5 * lo
    for s in layers(ws):
        assert np.max(np.abs(g[s] - go[s])) <= 1e-4 * np.max(np.abs(go[s]))
    # one Adam step over all rows, then the gradient at the new parameters (W^T kept by the update)
    lr, b1, b2, eps = 1e-3, 0.9, 0.999, 0.1
    m.train(x, t, w, epochs=1, batch=rows, lr=lr, beta1=b1, beta2=b2, eps=eps)
    p1 = p64 - lr * go / (np.abs(go) + eps)
    assert np.max(np.abs(m.params - p1)) < 1e-6
    _, g1 = m.loss_grad(x, t, w)
    _, go1 = mo.loss_grad(m.params.astype(np.float64), ws, x64, t64, w64)
    for s in layers(ws):
        assert np.max(np.abs(g1[s] - go1[s])) <= 1e-4 * np.max(np.abs(go1[s]))
    # three epochs of small batches are the same twice, with the losses kept per epoch
    if rows >= 8:
        m.params = p
        h1 = m.train(x, t, w, epochs=3, batch=7)
        q1 = m.params
        m.params = p
        h2 = m.train(x, t, w, epochs=3, batch=7)
        np.testing.assert_array_equal(q1, m.params)
        np.testing.assert_array_equal(h1, h2)
        assert np.all(np.isfinite(h1)) and h1.size == 3
    m.close()
