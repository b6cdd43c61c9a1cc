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
