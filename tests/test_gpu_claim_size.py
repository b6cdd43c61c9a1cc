"""Claims are cut smaller than walks_per_lane where lanes would idle: same counts, and estimates that differ
by the order of FP64 additions only, on both sides of the rule (16 claims per lane of the grid)."""
import numpy as np
import pytest

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
