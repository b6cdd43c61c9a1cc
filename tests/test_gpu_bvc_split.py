"""The splat's split over sample chunks and its tiles of 256 sorted samples: sizes around the wave, tile and
chunk edges, a mixed cache against one cache per category, and a captured call (which runs in one chunk)."""
import numpy as np
import pytest

from zombie_amd import _abi as A
from zombie_amd import engine as E

pytestmark = pytest.mark.gpu


def _inputs(torch, dim, n, m, seed):
    rng = np.random.default_rng(seed)
    t = lambda a, d=np.float32: torch.from_numpy(np.ascontiguousarray(a, d)).cuda()
    nr = rng.normal(size=(n, dim))
    ty = rng.choice([A.ZG_SAMPLE_ON_ABSORBING_BOUNDARY, A.ZG_SAMPLE_ON_REFLECTING_BOUNDARY, A.ZG_SAMPLE_IN_DOMAIN], n)
    S = dict(pt=rng.normal(size=(n, dim)) * 0.6, normal=nr / np.linalg.norm(nr, axis=1, keepdims=True),
             type=ty.astype(np.uint8), normal_aligned=(rng.random(n) < 0.3).astype(np.uint8), pdf=rng.uniform(0.5, 2.0, n),
             solution=rng.normal(size=n), normal_derivative=rng.normal(size=n), contribution=rng.normal(size=n),
             robin_coeff=np.where(ty == A.ZG_SAMPLE_ON_REFLECTING_BOUNDARY, rng.choice([0.0, 0.3, 3.0], n), 0.0))
    X = dict(pt=rng.normal(size=(m, dim)) * 0.5, type=rng.choice([0, A.ZG_SAMPLE_ON_ABSORBING_BOUNDARY], m).astype(np.uint8),
             dist_abs=rng.uniform(0, 1, m), dist_refl=rng.uniform(0, 1, m))
    u8 = ("type", "normal_aligned")
    samples = E.BvcSamples(**{k: t(v, np.uint8 if k in u8 else np.float32) for k, v in S.items()})
    evals = E.BvcEvalPoints(pt=t(X["pt"]), dist_to_absorbing=t(X["dist_abs"]), dist_to_reflecting=t(X["dist_refl"]),
                            type=t(X["type"], np.uint8))
    return S, X, samples, evals


@pytest.mark.parametrize("n,m", [(1, 1), (255, 64), (256, 65), (257, 63), (1000, 1), (20001, 130)])
@pytest.mark.parametrize("dim,mu2", [(2, 0.0), (3, 0.0), (3, 2.0)])
def test_edges_match_oracle(gpu, oracle_lib, dim, mu2, n, m):
    torch = gpu
    S, X, samples, evals = _inputs(torch, dim, n, m, 7 * n + m + dim)
    ost = oracle_lib.BvcStats(m, dim)
    oracle_lib.bvc_splat(dim, S, X, ost, radius_clamp=1e-2, robin_cutoff=1.0, cutoff_abs=0.02, absorption=mu2)
    st = E.BvcStats.zeros(m, dim)
    E.bvc_splat(dim, samples, evals, st, radius_clamp=1e-2, robin_coeff_cutoff=1.0, cutoff_dist_to_absorbing=0.02,
                absorption=mu2)
    assert np.array_equal(st.n.cpu().numpy(), ost.n)
    # a pair's estimate carries about ten float roundings (6e-8 each) of its terms, of which the largest is
    # that of the squared distance seen through 1 / r^3 (x 3): 4e-6 of the terms, whose size the root mean
    # square of the estimates gives (largest over the points: single points can cancel)
    k = np.maximum(ost.n, 1)
    rms = np.sqrt((ost.m2 / k + ost.mean ** 2).max()) + 1e-30
    grms = np.sqrt((ost.grad_m2 / k[..., None] + ost.grad_mean ** 2).max()) + 1e-30
    assert np.abs(st.mean.cpu().numpy() - ost.mean).max() <= 4e-6 * rms
    assert np.abs(st.grad_mean.cpu().numpy() - ost.grad_mean).max() <= 4e-6 * grms


def test_captured_call(gpu):
    torch = gpu
    _, _, samples, evals = _inputs(torch, 3, 5000, 200, 3)
    want, got = E.BvcStats.zeros(200, 3), E.BvcStats.zeros(200, 3)
    E.bvc_splat(3, samples, evals, E.BvcStats.zeros(200, 3))
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        E.bvc_splat(3, samples, evals, got)
    for _ in range(3):
        E.bvc_splat(3, samples, evals, want)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(want.n, got.n)
        # the chunks' FP64 sums are added in another order
        assert (want.mean - got.mean).abs().max() <= 1e-12 * want.mean.abs().max()
        assert (want.grad_m2 - got.grad_m2).abs().max() <= 1e-10 * want.grad_m2.abs().max()


@pytest.mark.parametrize("n", [200, 200000])
@pytest.mark.parametrize("dim,mu2", [(2, 0.0), (3, 0.0), (3, 2.25)])
def test_sums_have_no_common_error(gpu, dim, mu2, n):
    """A pair's estimate e is off by up to ten float roundings, 1e-7 root mean square.  Over many pairs they
    average out, to 1e-7 sqrt(sum e^2) / |sum e|, which at n = 200,000 is far less than an error that all pairs share,
    such as that of 1 / (4 pi) rounded to 32 bits (4e-8).  Five standard deviations, and 1e-8 for what is shared."""
    torch = gpu
    rng = np.random.default_rng(dim)
    y = rng.normal(size=(n, dim))
    y /= np.linalg.norm(y, axis=1, keepdims=True)
    normal = y.astype(np.float32)
    y = (y * rng.uniform(0.1, 0.7, (n, 1))).astype(np.float32)
    f = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda()
    one, zero = np.ones(n), np.zeros(n)
    x = np.zeros((1, dim), np.float32)
    x[0, 0] = 0.01
    got, want, tol = [], [], []
    xy = (x.astype(np.float64) - y)
    r = np.linalg.norm(xy, axis=1)
    nx = (xy * normal).sum(1)
    mr = np.sqrt(mu2) * r
    G = -np.log(r) / (2 * np.pi) if dim == 2 else np.exp(-mr) / (4 * np.pi * r)
    K = 1 / (2 * np.pi * r ** 2) if dim == 2 else np.exp(-mr) * (mr + 1) / (4 * np.pi * r ** 3)
    for src, u in ((True, zero), (False, -one)):   # G alone, P alone (and their squares)
        s = E.BvcSamples(pt=f(y), normal=f(normal), pdf=f(one), solution=f(u), normal_derivative=f(zero), contribution=f(one),
                         type=torch.full((n,), A.ZG_SAMPLE_IN_DOMAIN if src else A.ZG_SAMPLE_ON_ABSORBING_BOUNDARY,
                                         dtype=torch.uint8, device="cuda"))
        st = E.BvcStats.zeros(1, dim)
        E.bvc_splat(dim, s, E.BvcEvalPoints(pt=f(x), dist_to_absorbing=f([1.0])), st, absorption=mu2)
        c = 4 if src else 0
        e = G if src else nx * K
        mean, m2 = float(st.mean[0, c]), float(st.m2[0, c])
        got += [mean, m2 / n + mean ** 2]
        want += [e.mean(), (e ** 2).mean()]
        tol += [1e-8 + 5e-7 * np.sqrt((e ** 2).sum()) / abs(e.sum()), 1e-8 + 1e-6 * np.sqrt((e ** 4).sum()) / (e ** 2).sum()]
    err = np.abs(np.array(got) / want - 1)
    assert (err <= tol).all(), (err, tol)
