"""Points with NaN or infinite coordinates, and rays of unbounded length: queries and walks end, find nothing
where nothing is (distance FLT_MAX, no hit), and leave the other points of their wave alone.  Every combination of
the coordinates below takes part, since what a box test makes of such a point depends on which coordinates are
not finite, and whether it enters the empty slots of a node."""
import itertools

import numpy as np
import pytest

from zombie_amd import _abi as A
from zombie_amd import engine as E
from zombie_amd import problems as PB

pytestmark = pytest.mark.gpu

FLT_MAX = float(np.finfo(np.float32).max)
COORDS = (0.25, np.nan, np.inf, -np.inf, 3e38, 1e30, -1e30)


def _mesh(dim):
    V, I = PB.star_curve(151) if dim == 2 else PB.icosphere(2)
    return V.astype(np.float32), I.astype(np.int32)


def _points(dim):
    """Ordinary points with every combination of COORDS between them, and which rows are ordinary."""
    odd = np.array(list(itertools.product(COORDS, repeat=dim)), np.float32)
    rng = np.random.default_rng(3)
    x = rng.uniform(-0.4, 0.4, (2 * len(odd), dim)).astype(np.float32)
    x[1::2] = odd
    return x, (np.abs(x) < 1e20).all(1)


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("width,leaf", [(4, 2), (8, 4)])
@pytest.mark.parametrize("boundary", [0, 1])
def test_closest_point_ends_and_finds_nothing(gpu, dim, width, leaf, boundary):
    torch = gpu
    V, I = _mesh(dim)
    sc = E.Scene(V, I, np.full(len(I), boundary, np.uint8), V.min(0) - 1, V.max(0) + 1, bvh_width=width, leaf_size=leaf)
    x, ordinary = _points(dim)
    out = sc.closest_point(torch.from_numpy(x).cuda(), boundary=boundary, want_normal=True, want_prim=True)
    d, cp, nr, pr = (t.cpu().numpy() for t in out)
    assert (d[~ordinary] == FLT_MAX).all() and (pr[~ordinary] == -1).all()
    assert (cp[~ordinary] == 0).all() and (nr[~ordinary] == 0).all()
    alone = sc.closest_point(torch.from_numpy(x[ordinary]).cuda(), boundary=boundary, want_normal=True, want_prim=True)
    for a, b in zip(alone, (d, cp, nr, pr)):
        assert np.array_equal(a.cpu().numpy(), b[ordinary])
    assert (d[ordinary] < 2).all()


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("tolerance", [0.0, 0.2])
def test_walks_from_such_points_end(gpu, dim, tolerance):
    torch = gpu
    V, I = _mesh(dim)
    sc = E.Scene(V, I, None, V.min(0) - 0.1, V.max(0) + 0.1)
    x, ordinary = _points(dim)
    pde = E.make_pde(dirichlet=E.function(A.ZG_FN_EXP_COS, A.ZG_EVAL_VALUE, (1.0, 1.0)), is_source_constant=True)
    ws = E.walk_settings_host(1e-3, 1e-3, 32, False)

    def solve(rows, dist=None):
        pt = torch.from_numpy(np.ascontiguousarray(x[rows])).cuda()
        d = sc.closest_point(pt, want_point=False)[0] if dist is None else torch.full((len(pt),), dist, device="cuda")
        n = len(pt)
        st = E.DeviceStats.zeros(n)
        dp = E.DevicePoints(pt=pt, dist_to_absorbing=d, n_walks=torch.full((n,), 8, dtype=torch.int32, device="cuda"),
                            n_walks_max=8)
        E.wos_solve(sc, pde, ws, dp, st, E.SolveOptions(seed=5, distance_tolerance=tolerance))
        return st

    everywhere = np.ones(len(x), bool)
    st = solve(everywhere)
    assert (st.n.cpu().numpy()[ordinary] == 8).all()
    assert torch.isfinite(st.mean[torch.from_numpy(ordinary).cuda()]).all()
    solve(everywhere, dist=0.0)   # at once on the boundary: the walk's only query is the projection


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("width", [4, 8])
def test_unbounded_rays_end(gpu, dim, width):
    """Along a diagonal every axis of an empty slot's box (all corners at 1e30) is crossed at the same parameter."""
    torch = gpu
    V, I = _mesh(dim)
    sc = E.Scene(V, I, None, V.min(0) - 1, V.max(0) + 1, bvh_width=width, leaf_size=1)
    dirs = np.array(list(itertools.product((-1, 0, 1), repeat=dim)), np.float32)
    dirs = dirs[(dirs != 0).any(1)]
    odd = np.array(list(itertools.product((0.25, np.nan, np.inf), repeat=dim)), np.float32)
    inner = np.full_like(dirs, 0.013) * np.arange(1, dim + 1, dtype=np.float32)   # off the mesh's symmetry planes
    o = np.concatenate([inner, 3 * dirs, np.repeat(odd, len(dirs), 0)])
    d = np.concatenate([dirs, dirs, np.tile(dirs, (len(odd), 1))])
    out = []
    for t_max in (10.0, FLT_MAX):
        t = torch.full((len(o),), t_max, device="cuda")
        hit, th, _, _ = sc.intersect_ray(torch.from_numpy(o).cuda(), torch.from_numpy(d).cuda(), t)
        out.append((hit.cpu().numpy(), th.cpu().numpy()))
    (h0, t0), (h1, t1) = out
    assert np.array_equal(h0, h1) and np.array_equal(t0[h0 == 1], t1[h0 == 1])
    assert (h1[:len(dirs)] == 1).all()
    assert (h1[len(dirs):2 * len(dirs)] == 0).all()    # outside, away from the mesh
    assert (h1[~np.isfinite(o).all(1)] == 0).all()


@pytest.mark.parametrize("dim,interleave", [(2, False), (2, True), (3, False), (3, True)])
def test_walks_on_stars_from_such_points_end(gpu, dim, interleave):
    torch = gpu
    p = PB.mixed2d(n_segments=64, n_slits=2, max_len=16) if dim == 2 else PB.lprism3d(n_sub=2, n_z=2)
    sc = E.Scene(p.positions, p.indices, p.is_reflecting, p.domain_min, p.domain_max,
                 solve_double_sided=p.solve_double_sided)
    x, ordinary = _points(dim)
    pt = torch.from_numpy(x).cuda()
    n = len(x)
    ws = E.walk_settings_host(1e-3, 1e-3, 16, p.solve_double_sided)
    dp = E.DevicePoints(pt=pt, dist_to_absorbing=sc.closest_point(pt, want_point=False)[0],
                        n_walks=torch.full((n,), 4, dtype=torch.int32, device="cuda"), n_walks_max=4)
    st = E.DeviceStats.zeros(n)
    E.wost_solve(sc, p.pde, ws, dp, st, E.SolveOptions(seed=5, wost_interleave_queries=interleave))
    assert torch.isfinite(st.mean[torch.from_numpy(ordinary).cuda()]).all()


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("width", [4, 8])
def test_copied_tree_has_zeros_in_empty_slots(gpu, dim, width):
    V, I = _mesh(dim)
    sc = E.Scene(V, I, None, V.min(0) - 1, V.max(0) + 1, bvh_width=width, leaf_size=1)
    nodes, _ = sc.copy_bvh(0)
    nodes = nodes.reshape(sc.info.n_absorbing_nodes, -1)
    child = nodes.view(np.int32)[:, 2 * dim * width:(2 * dim + 1) * width]
    empty = nodes[:, :width] == np.float32(1e30)
    assert empty.any() and np.array_equal(child == 0, empty)
