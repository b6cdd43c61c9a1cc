"""Claims are cut smaller than walks_per_lane where lanes would idle: same counts, and estimates that differ
by the order of FP64 additions only, on both sides of the rule (16 claims per lane of the grid)."""
import numpy as np
import pytest

from zombie_amd import _abi as A
from zombie_amd import engine as E
from zombie_amd import problems as PB

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,walks,waves_per_cu", [(1, 1, 0), (1, 65, 0), (300, 33, 0), (3000, 64, 4), (3000, 257, 4)])
def test_claim_size_does_not_change_estimates(gpu, n, walks, waves_per_cu):
    torch = gpu
    p = PB.star2d(n_segments=128, grid_res=8)
    rng = np.random.default_rng(n + walks)
    pt = torch.from_numpy((rng.uniform(-0.4, 0.4, (n, 2))).astype(np.float32)).cuda()
    sc = E.Scene(p.positions, p.indices, None, p.domain_min, p.domain_max)
    d = sc.closest_point(pt, want_point=False)[0]
    nw = torch.from_numpy(rng.integers(max(1, walks - 3), walks + 1, n).astype(np.int32)).cuda()
    out = []
    for wpl in (1, 8, 64):
        st = E.DeviceStats.zeros(n)
        E.wos_solve(sc, p.pde, p.settings, E.DevicePoints(pt=pt, dist_to_absorbing=d, n_walks=nw, n_walks_max=walks), st,
                    E.SolveOptions(seed=5, walks_per_lane=wpl, waves_per_cu=waves_per_cu))
        out.append(st)
    for st in out[1:]:
        assert torch.equal(st.n, out[0].n) and torch.equal(st.n, nw.long())
        assert torch.equal(st.walk_length, out[0].walk_length)
        assert (st.mean - out[0].mean).abs().max() <= 1e-13 * walks


@pytest.mark.parametrize("kind,n,walks", [("wos", 3000, 1000), ("wos", 2500, 257), ("wost", 2500, 257), ("gradient", 24000, 64),
                                          ("batch", 3000, 257)])
def test_claims_of_several_walks(gpu, kind, n, walks):
    """Sizes at which the rule leaves claims of several walks, with a last claim that is not full, on a grid of one
    wave per SIMD and CU: the same estimates as with claims of one walk."""
    torch = gpu
    probs = [PB.star2d(n_segments=128, grid_res=8)] if kind != "batch" else \
        [PB.screened_instance(t, 1.0, np.array([1.0, 0.5, -0.2]), 3) for t in (300, 900)]
    p = probs[0]
    rng = np.random.default_rng(n + walks)
    pt = torch.from_numpy((rng.uniform(-0.4, 0.4, (n, 3 if kind == "batch" else 2))).astype(np.float32)).cuda()
    scenes = [E.Scene(q.positions, q.indices, None, q.domain_min, q.domain_max) for q in probs]
    sc = scenes[0]
    d = torch.cat([q.closest_point(t.contiguous(), want_point=False)[0] for q, t in zip(scenes, pt.chunk(len(scenes)))])
    dp = E.DevicePoints(pt=pt, dist_to_absorbing=d, n_walks=torch.full((n,), walks, dtype=torch.int32, device="cuda"),
                        n_walks_max=walks)
    if kind == "gradient":
        dp.estimation_quantity = torch.full((n,), A.ZG_ESTIMATE_SOLUTION_AND_GRADIENT, dtype=torch.uint8, device="cuda")
    # lanes of the grid: multiprocessors * waves_per_cu / 4 blocks of 256; a gradient solve's last stage has half the walks
    lanes = torch.cuda.get_device_properties(0).multi_processor_count // 4 * 256
    per_lane = n * (walks // 2 if kind == "gradient" else walks) // (16 * lanes)
    assert per_lane >= 2
    out = []
    for wpl in (1, 8, 64):
        claim = min(wpl, per_lane)
        assert (claim > 1) == (wpl > 1)
        st = E.DeviceStats.zeros(n, dim=2 if kind == "gradient" else 0)
        opts = E.SolveOptions(seed=5, walks_per_lane=wpl, waves_per_cu=1)
        if kind == "batch":
            inst = torch.arange(n, device="cuda", dtype=torch.int32) // (n // 2)
            E.batch_wos_solve(E.Batch(scenes, [q.pde for q in probs]), p.settings, dp, inst, st, opts)
        else:
            (E.wost_solve if kind == "wost" else E.wos_solve)(sc, p.pde, p.settings, dp, st, opts)
        out.append(st)
    for st in out[1:]:
        assert torch.equal(st.n, out[0].n) and torch.equal(st.walk_length, out[0].walk_length)
        assert (st.mean - out[0].mean).abs().max() <= 1e-13 * walks
        if kind == "gradient":
            assert torch.equal(st.n_grad, out[0].n_grad)
            scale = 1.0 + out[0].grad_mean.abs().max()
            assert (st.grad_mean - out[0].grad_mean).abs().max() <= 1e-9 * scale
