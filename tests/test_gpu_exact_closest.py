"""Closest-point queries over the oriented boxes against the axis-aligned ones and a brute-force scan in float64,
and walk on stars over them against the axis-aligned boxes (a distance tolerance of 1e-7) on the same random streams."""
import numpy as np
import pytest

from zombie_amd import engine as E
from zombie_amd import problems as PB

pytestmark = pytest.mark.gpu


def _brute(V, I, x):
    """Distances of x [n, d] to all segments / triangles, float64."""
    T = V.astype(np.float64)[I]
    x = x.astype(np.float64)[:, None]

    def seg(a, b):
        e = b - a
        t = np.clip(((x - a) * e).sum(-1) / np.maximum((e * e).sum(-1), 1e-300), 0, 1)
        return ((x - a - t[..., None] * e) ** 2).sum(-1)
    if V.shape[1] == 2:
        return np.sqrt(seg(T[:, 0], T[:, 1]).min(1))
    a, b, c = T[:, 0], T[:, 1], T[:, 2]
    d2 = np.minimum(np.minimum(seg(a, b), seg(b, c)), seg(c, a))
    n = np.cross(b - a, c - a)
    nn = np.maximum((n * n).sum(-1), 1e-300)
    v = (np.cross(x - a, c - a) * n).sum(-1) / nn
    w = (np.cross(b - a, x - a) * n).sum(-1) / nn
    inside = (v >= 0) & (w >= 0) & (v + w <= 1) & (nn > 1e-300)
    return np.sqrt(np.where(inside, ((x - a) * n).sum(-1) ** 2 / nn, d2).min(1))


@pytest.mark.parametrize("width,leaf", [(4, 2), (8, 4)])
@pytest.mark.parametrize("kind", ["star", "sphere", "slivers", "one", "far"])
def test_distances_match_brute_force(gpu, kind, width, leaf):
    torch = gpu
    rng = np.random.default_rng(1)
    if kind == "star":
        V, I = PB.star_curve(151)
    elif kind == "one":
        V, I = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0]], float), np.array([[0, 1, 2]])
    else:
        V, I = PB.icosphere(2)
        if kind == "slivers":
            V = V * [1.0, 0.02, 3.0]
        if kind == "far":
            V = V + [300.0, -40.0, 7.0]
    V, I = V.astype(np.float32), I.astype(np.int32)
    sc = E.Scene(V, I, None, V.min(0) - 1, V.max(0) + 1, bvh_width=width, leaf_size=leaf)
    lo, hi = V.min(0), V.max(0)
    x = rng.uniform(lo - 0.5 * (hi - lo) - 0.1, hi + 0.5 * (hi - lo) + 0.1, (1003, V.shape[1])).astype(np.float32)
    x[:20] = V[I[rng.integers(0, len(I), 20)]].mean(1)      # on the surface
    d = sc.closest_point(torch.from_numpy(x).cuda(), want_point=False)[0].cpu().numpy()
    # the same mesh as a reflecting boundary has no oriented boxes: the same distances, bit for bit
    sr = E.Scene(V, I, np.ones(len(I), np.uint8), V.min(0) - 1, V.max(0) + 1, bvh_width=width, leaf_size=leaf)
    dr = sr.closest_point(torch.from_numpy(x).cuda(), boundary=1, want_point=False)[0].cpu().numpy()
    assert np.array_equal(d, dr)
    if kind == "slivers":
        return   # a sliver's closest point is ill-conditioned in float in either query
    # float distances: a few ulps of the coordinates (the closest point's rounding) and of the distance
    tol = 8 * 2.0 ** -24 * (np.abs(V).max() + np.abs(x).max())
    assert np.abs(d - _brute(V, I, x)).max() <= tol


@pytest.mark.parametrize("width,leaf", [(4, 1), (8, 2)])
def test_boxes_of_a_large_mesh(gpu, width, leaf):
    """More child slots than the waves that build the boxes take at once (32,768)."""
    torch = gpu
    V, I = PB.icosphere(6)
    V = PB.sh_displace(V, 3).astype(np.float32)
    I = I.astype(np.int32)
    x = np.random.default_rng(4).uniform(-1.5, 1.5, (5000, 3)).astype(np.float32)
    d = []
    for boundary in (0, 1):
        sc = E.Scene(V, I, np.full(len(I), boundary, np.uint8), V.min(0) - 1, V.max(0) + 1, bvh_width=width, leaf_size=leaf)
        nodes = sc.info.n_absorbing_nodes + sc.info.n_reflecting_nodes
        assert nodes * width > 32768
        d.append(sc.closest_point(torch.from_numpy(x).cuda(), boundary=boundary, want_point=False)[0])
    assert torch.equal(*d)


@pytest.mark.parametrize("segments,slits", [(64, 1), (700, 6)])
def test_walk_on_stars_same_walks(gpu, segments, slits):
    torch = gpu
    p = PB.mixed2d(n_segments=segments, n_slits=slits, max_len=64)
    sc = E.Scene(p.positions, p.indices, p.is_reflecting, p.domain_min, p.domain_max, solve_double_sided=True)
    rng = np.random.default_rng(2)
    pt = torch.from_numpy(rng.uniform(-0.4, 0.4, (500, 2)).astype(np.float32)).cuda()
    d = sc.closest_point(pt, want_point=False)[0]
    reps = []
    for tol in (0.0, 1e-7):
        dp = E.DevicePoints(pt=pt, dist_to_absorbing=d, n_walks=torch.full((500,), 32, dtype=torch.int32, device="cuda"),
                            n_walks_max=32)
        st = E.DeviceStats.zeros(500)
        reps.append((E.wost_solve(sc, p.pde, p.settings, dp, st, E.SolveOptions(seed=4, distance_tolerance=tol)), st))
    (ra, sa), (rb, sb) = reps
    # a radius off by 1e-7 decorrelates a walk only after many reflections: most of 64 steps agree
    assert ra.total_walks == rb.total_walks
    assert abs(ra.total_steps - rb.total_steps) <= 0.01 * rb.total_steps
    se = (sa.variance() / 32).sqrt()
    assert ((sa.mean - sb.mean).abs() <= 6 * se + 1e-6).all()
