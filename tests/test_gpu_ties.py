"""Equally near primitives: the two segments (or the triangles) that share the closest vertex or edge.  Exact
queries over the oriented boxes meet them in another order than the traversal of the axis-aligned boxes, and must
name the same one wherever a caller can tell."""
import numpy as np
import pytest

from zombie_amd import _abi as A
from zombie_amd import engine as E
from zombie_amd import problems as PB

pytestmark = pytest.mark.gpu


def _gear(teeth=12):
    """Closed polygon between radii 0.5 and 1: seen from inside, the vertices at 0.5 are convex and closest for whole
    wedges of points."""
    t = np.arange(2 * teeth) * np.pi / teeth
    r = np.where(np.arange(2 * teeth) % 2 == 0, 1.0, 0.5)
    V = np.stack([r * np.cos(t), r * np.sin(t)], 1).astype(np.float32)
    i = np.arange(2 * teeth, dtype=np.int32)
    return V, np.stack([i, (i + 1) % (2 * teeth)], 1).astype(np.int32)


@pytest.mark.parametrize("kind,double_sided", [("wos", True), ("wost", False), ("wost", True)])
@pytest.mark.parametrize("eval_", [A.ZG_EVAL_NORMAL_DERIVATIVE, A.ZG_EVAL_ROBIN])
def test_boundary_data_that_read_the_normal(gpu, kind, double_sided, eval_):
    """Counting solves traverse the axis-aligned boxes on the same walks: the same estimates, up to the order of
    64-bit sums of 64 values of order one."""
    torch = gpu
    V, I = _gear()
    n, walks = 2000, 64
    pt = torch.from_numpy(np.random.default_rng(0).uniform(-0.3, 0.3, (n, 2)).astype(np.float32)).cuda()
    sc = E.Scene(V, I, None, V.min(0) - 1e-3, V.max(0) + 1e-3, solve_double_sided=double_sided)
    d = sc.closest_point(pt, want_point=False)[0]
    pde = E.make_pde(dirichlet=E.function(A.ZG_FN_EXP_COS, eval_, (1.0, 1.0, 0.0, 0.0, 0.0, 0.5)), is_source_constant=True)
    ws = E.walk_settings_host(1e-3, 1e-3, 1024, double_sided)
    out = []
    for count in (0, 1):
        dp = E.DevicePoints(pt=pt, dist_to_absorbing=d, n_walks=torch.full((n,), walks, dtype=torch.int32, device="cuda"),
                            n_walks_max=walks)
        st = E.DeviceStats.zeros(n)
        (E.wos_solve if kind == "wos" else E.wost_solve)(sc, pde, ws, dp, st, E.SolveOptions(seed=3, count_visits=count))
        out.append(st)
    assert torch.equal(out[0].walk_length, out[1].walk_length)
    assert (out[0].mean - out[1].mean).abs().max() <= walks * 2.0 ** -52


def _mesh(dim):
    """Nonconvex shapes whose vertices (and edges) are closest for whole regions of points, inside and outside."""
    if dim == 2:
        return _gear()
    V, I = PB.icosphere(2)
    V = V * (1.0 + 0.3 * np.sin(5 * V[:, :1]) * np.cos(7 * V[:, 1:2]))
    return V.astype(np.float32), I.astype(np.int32)


@pytest.mark.parametrize("dim,width,leaf", [(2, 4, 2), (2, 8, 4), (3, 4, 1), (3, 4, 2), (3, 8, 4)])
def test_closest_point_names_the_same_primitive(gpu, dim, width, leaf):
    """Point, normal and primitive of every query equal those of the axis-aligned traversal (the same mesh as a
    reflecting boundary), bit for bit: in the regions of vertices and edges, on them, and anywhere."""
    torch = gpu
    V, I = _mesh(dim)
    rng = np.random.default_rng(5)
    T = V[I].astype(np.float64)
    edges = np.concatenate([T[:, [a, (a + 1) % dim]] for a in range(dim)])
    mid = edges[rng.integers(0, len(edges), 4000)]
    w = rng.random((4000, 1))
    on_edge = mid[:, 0] * w + mid[:, 1] * (1 - w)
    x = np.concatenate([V, V * 1.3, V * 0.8, on_edge, on_edge * 1.2, on_edge * 0.9,
                        rng.uniform(-1.6, 1.6, (8000, dim))]).astype(np.float32)
    out = []
    for boundary in (0, 1):
        sc = E.Scene(V, I, np.full(len(I), boundary, np.uint8), V.min(0) - 1, V.max(0) + 1, bvh_width=width, leaf_size=leaf)
        r = sc.closest_point(torch.from_numpy(x).cuda(), boundary=boundary, want_normal=True, want_prim=True)
        out.append([a.cpu().numpy() for a in r])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    # ties take part: the brute-force minimum is shared by several primitives for many of these points
    d, _, _, prim = out[0]
    a, e = T[:, 0], T[:, 1] - T[:, 0]
    if dim == 2:
        t = np.clip(((x[:, None] - a) * e).sum(-1) / (e * e).sum(-1), 0, 1)
        all_d = np.linalg.norm(x[:, None] - a - t[..., None] * e, axis=-1)
        assert ((all_d <= all_d.min(1, keepdims=True) + 1e-7).sum(1) > 1).mean() > 0.2
