"""The fused MLP layers at the shapes they take and the edges of their tiles (64 rows a block, 32 rows a block
of the weight gradients' operands), against the FP64 oracle with bf16 rounding at the same points.  Sums are
32-bit, so what differs is an activation or gradient that rounds the other way now and then: one bf16 ulp
(2^-8 of the value) in the few whose sum lies within 1e-6 of a rounding boundary, well below 1e-3 of the norm."""
import numpy as np
import pytest

from oracle import mlp as M
from zombie_amd import learned_cv as LC

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


@pytest.mark.parametrize("dim,freq,hidden,layers", [(3, 32, 128, 4), (2, 16, 128, 1), (3, 16, 128, 2), (2, 32, 128, 3),
                                                    (3, 32, 64, 4), (2, 16, 64, 1), (3, 16, 64, 3), (2, 32, 64, 2)])
@pytest.mark.parametrize("rows", [1, 33, 64, 65, 2500])
def test_fused_shapes_match_oracle(gpu, dim, freq, hidden, layers, rows):
    torch = gpu
    net = LC.MLP(LC.MLPConfig(in_dim=dim, n_frequencies=freq, hidden=hidden, n_hidden_layers=layers, frequency_sigma=2.0,
                              seed=rows), max_batch=rows)
    rng = np.random.default_rng(rows + freq + hidden)
    x = rng.uniform(-1, 1, (rows, dim)).astype(np.float32)
    y = np.sin(2 * x).prod(1).astype(np.float32) + np.float32(0.5)
    xt, yt = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
    theta, B = net.get_parameters(), net.frequencies()
    v, gx = net.evaluate(xt)
    only, _ = net.evaluate(xt, gradient=False)
    cb, gb = M.input_gradient(theta, B, x, hidden, layers, bf16=True)
    assert torch.equal(v, only)
    assert _rel(v.cpu().numpy(), cb) < 2e-3 and _rel(gx.cpu().numpy(), gb) < 5e-3
    loss, g = net.gradients(xt, yt)
    lb, pb = M.gradients(theta, B, x, y, hidden, layers, bf16=True)
    assert abs(loss - lb) < 1e-3 * abs(lb) and _rel(g, pb) < 5e-3
    loss2, g2 = net.gradients(xt, yt)
    assert loss2 == loss and np.array_equal(g, g2)      # sums in a fixed order
    net.train_step(xt, yt, 1e-3)                        # the first Adam step: lr g / (|g| + eps)
    step = -1e-3 * g / (np.abs(g) + 1e-8)
    assert np.abs(net.get_parameters() - theta - step).max() < 2e-6
    # the bf16 copies follow the parameters
    cb, _ = M.input_gradient(net.get_parameters(), B, x, hidden, layers, bf16=True)
    assert _rel(net.evaluate(xt, gradient=False)[0].cpu().numpy(), cb) < 2e-3
