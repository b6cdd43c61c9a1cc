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


def _near_rounding_boundaries(f, n):
    """n arguments in [-6, 6] whose f lies within one 32-bit ulp of the middle between two bf16 values."""
    rng = np.random.default_rng(0)
    out = np.empty(0, np.float32)
    while len(out) < n:
        z = rng.uniform(-6, 6, 1 << 20).astype(np.float32)
        v = f(z.astype(np.float64))
        ulp = np.spacing(np.abs(v).astype(np.float32)).astype(np.float64)
        out = np.concatenate([out, z[np.abs(v / ulp % 65536 - 32768) < 1]])
    return out[:n]


def test_activations_equal_those_of_the_gemm_path(gpu):
    """The activation and its derivative as the GEMM path computes them (16 and 8 frequencies; an IEEE division
    each), at pre-activations where half a 32-bit ulp decides the bf16 rounding.  Zero weights make the
    pre-activations the biases; output weights of +1 and -1 on pairs of equal units make the value exactly 0, so
    that one row's gradients are the rounded activations (output weights) and derivatives (biases) themselves."""
    torch = gpu
    sig = lambda z: 1 / (1 + np.exp(-z))
    z = np.concatenate([_near_rounding_boundaries(lambda z: z * sig(z), 256),
                        _near_rounding_boundaries(lambda z: sig(z) * (1 + z * (1 - sig(z))), 256),
                        # where exp(-z) nears the end of its range and beyond, and where sigmoid is 1
                        np.linspace(-100, -80, 48), [-1e3, -1e30, -3e38, 0, 1e-30, -1e-30, 16, 17, 18, 80, 100, 1e3, 1e10,
                                                     1e18, -1e10, -1e18]]).astype(np.float32)
    x, y = torch.zeros((1, 2), device="cuda"), torch.full((1,), -1.0, device="cuda")
    got = []
    for freq in (16, 8):
        net = LC.MLP(LC.MLPConfig(in_dim=2, n_frequencies=freq, hidden=128, n_hidden_layers=1), max_batch=64)
        rows = []
        for zs in z.reshape(-1, 64):
            theta = np.zeros_like(net.get_parameters())
            at = 2 * freq * 128
            theta[at:at + 128] = np.repeat(zs, 2)
            theta[at + 128:at + 256:2], theta[at + 129:at + 256:2] = 1, -1
            net.set_parameters(theta)
            _, g = net.gradients(x, y)
            rows.append(np.concatenate([g[at:at + 128], g[at + 128:at + 256]]))
        got.append(np.concatenate(rows))
    assert np.isfinite(got[0]).all() and (got[0][:8 * 256] != 0).all()
    # below 2^-126 the reciprocal is 0: activations under 100 * 2^-126 may be too
    assert ((got[0] == got[1]) | (np.abs(got[0] - got[1]) < 100 * 2.0 ** -126)).all()
    assert np.array_equal(got[0][:8 * 256], got[1][:8 * 256])
