"""Signed distance at octree vertices (right-hand side of the fit), GPU
against the oracle (replaces igl::signed_distance, ThinShells.cpp:481-509)."""
import numpy as np
import pytest

import oracle as O
from helpers import case, exact_winding_number, fitted
from its_amd import meshes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,R", [("icosphere", 64), ("bunny", 32), ("torus", 32)])
def test_sdf_at_vertices(ctx, name, R):
    from its_amd import _capi
    F = fitted(name, R)
    c = F.case
    g = _capi.Octree(ctx, c.tris, c.origin, c.width, R)
    b = g.sdf_at_vertices(c.V, c.F)
    np.testing.assert_array_equal(np.sign(b), np.sign(F.b))
    assert np.abs(b - F.b).max() <= 1e-12


def test_sdf_sphere_closed_form(ctx):
    from its_amd import meshes
    V, Fc = meshes.icosphere(4)
    rng = np.random.default_rng(2)
    P = rng.uniform(-1.5, 1.5, size=(3000, 3))
    d = ctx.signed_distance(V, Fc, P)
    r = np.linalg.norm(P, axis=1)
    # inscribed polyhedron: within the chord sagitta of the unit sphere
    assert np.all(np.abs(d - (r - 1)) < 5e-3)
    far = np.abs(r - 1) > 0.01
    assert np.all(np.sign(d[far]) == np.sign(r[far] - 1))


def test_sdf_culling_keeps_exact_results(ctx):
    """Points on vertices and edge midpoints (ties between triangles), just off
    the surface and far away: the bounding-sphere culling must leave the
    binary64 distance identical to the full search of the oracle."""
    from its_amd import _capi
    c = case("bunny", 32)
    rng = np.random.default_rng(7)
    V, F = c.V, c.F
    mids = 0.5 * (V[F[:, 0]] + V[F[:, 1]])
    near = V[rng.choice(len(V), 500)] + 1e-4 * rng.standard_normal((500, 3))
    far = rng.uniform(-3, 4, size=(500, 3))
    P = np.concatenate([V[:500], mids[:500], near, far])
    d = ctx.signed_distance(V, F, P)
    ref = O.signed_distance(V, F, P)
    # the culling decides which triangles get the binary64 distance: exact
    assert np.abs(np.abs(d) - np.abs(ref)).max() <= 1e-12
    # the sign comes from the binary32 winding number, unchanged by the
    # culling; on the surface and where the open mesh leaves w near 1/2 it is
    # a tie, so compare it only where the binary64 winding number is clear
    w = np.array([O.winding_number(V, F, p) for p in P])
    clear = (np.abs(ref) > 1e-6) & (np.abs(w - 0.5) > 0.05)
    assert clear.sum() > 900
    np.testing.assert_array_equal(np.sign(d[clear]), np.sign(ref[clear]))


def _tree_cases():
    from its_amd import meshes
    V, F = meshes.icosphere(3)
    F = F.astype(np.int32)
    out = {}
    # unwelded triangle soup: every edge is open, no boundary fan is kept
    out["soup"] = (V[F].reshape(-1, 3), np.arange(3 * len(F), dtype=np.int32).reshape(-1, 3))
    # half the faces reversed: winding numbers between 0 and 1
    Ff = F.copy()
    Ff[::2] = Ff[::2, ::-1]
    out["flipped"] = (V, Ff)
    # a closed sphere with every face twice (winding 2 inside), plus
    # degenerate triangles (a repeated vertex, three collinear points)
    Fd = np.concatenate([F, F, [[0, 0, 1], [2, 2, 2]]]).astype(np.int32)
    out["doubled_degenerate"] = (V, Fd)
    # non-manifold: a second sphere sharing one edge, plus a fin of three
    # triangles on that edge
    V2 = V + np.array([2.0, 0, 0])
    a, b = F[0, 0], F[0, 1]
    Vn = np.concatenate([V, V2, [[0.5, 3.0, 0.0], [0.5, -3.0, 0.0], [0.5, 0.0, 3.0]]])
    F2 = F + len(V)
    F2[F2 == len(V) + a] = a
    F2[F2 == len(V) + b] = b
    m = 2 * len(V)
    out["nonmanifold"] = (Vn, np.concatenate([F, F2, [[a, b, m], [b, a, m + 1], [a, b, m + 2]]]).astype(np.int32))
    out["single"] = (np.array([[0.0, 0, 0], [1.0, 0, 0], [0, 1.0, 0]]), np.array([[0, 1, 2]], dtype=np.int32))
    return out


@pytest.mark.parametrize("name", ["soup", "flipped", "doubled_degenerate", "nonmanifold", "single"])
def test_sdf_tree_mesh_kinds(ctx, name):
    """The triangle tree's pruned nearest search and boundary-fan winding
    number against the brute-force oracle on meshes that are open, doubly
    covered, non-manifold, inconsistently oriented or degenerate."""
    V, F = _tree_cases()[name]
    print(f"[sdf tree] {name} V={len(V)} F={len(F)}", flush=True)
    rng = np.random.default_rng(11)
    lo, hi = V.min(0), V.max(0)
    P = np.concatenate([rng.uniform(lo - 0.3 * (hi - lo), hi + 0.3 * (hi - lo), size=(1500, 3)),
                        V[rng.choice(len(V), 300)] + 1e-3 * rng.standard_normal((300, 3)), V[:50]])
    d = ctx.signed_distance(V, F, P)
    ref = O.signed_distance(V, F, P)
    assert np.abs(np.abs(d) - np.abs(ref)).max() <= 1e-12
    w = np.array([O.winding_number(V, F, p) for p in P])
    clear = (np.abs(ref) > 1e-6) & (np.abs(w - 0.5) > 0.05)
    assert clear.sum() > 1000
    np.testing.assert_array_equal(np.sign(d[clear]), np.sign(ref[clear]))


def test_sdf_tree_large_mesh(ctx):
    """200k-triangle knot tube: deep tree, long fans."""
    from its_amd import meshes
    V, F = meshes.torus_knot_tube()
    F = F.astype(np.int32)
    print(f"[sdf tree] knot V={len(V)} F={len(F)}", flush=True)
    rng = np.random.default_rng(5)
    lo, hi = V.min(0), V.max(0)
    P = np.concatenate([rng.uniform(lo - 0.1, hi + 0.1, size=(400, 3)),
                        V[rng.choice(len(V), 200)] + 0.02 * rng.standard_normal((200, 3))])
    d = ctx.signed_distance(V, F, P)
    ref = O.signed_distance(V, F, P)
    assert np.abs(np.abs(d) - np.abs(ref)).max() <= 1e-12
    far = np.abs(ref) > 1e-6
    np.testing.assert_array_equal(np.sign(d[far]), np.sign(ref[far]))


@pytest.mark.parametrize("name", ["icosphere", "torus", "knot", "flipped_sphere"])
def test_sdf_ray_signs(ctx, name):
    """Closed meshes: signs settled by the +z ray crossings (exact
    orientation tests, ITS_TUNE_SDF_RAY = 1) against the winding-number fan
    sum (ITS_TUNE_SDF_RAY = 0).  Away from the surface (|d| > 1e-9) the
    signed distances are identical bit for bit.  Within 1e-9 of it (here
    edge midpoints, rounded off their edges by about 1e-17) the binary32 fan
    sum can miss the side; wherever the two differ the ray's sign is checked
    against the exact winding number (rational arithmetic along an axis ray,
    tests/helpers.py), negative where it is at least 1."""
    from its_amd import _capi, meshes
    if name == "icosphere":
        V, F = meshes.noisy_icosphere(seed=3, level=4)
    elif name == "torus":
        V, F = meshes.torus(48, 96)
    elif name == "knot":
        V, F = meshes.torus_knot_tube(n_seg=400, n_ring=24)
        V = meshes.jitter(V, 1e-3, seed=7)
    else:   # inward orientation: winding number -1 inside, so no point is negative
        V, F = meshes.icosphere(3)
        F = F[:, ::-1].copy()
    V = _capi.model_to_unit_cube(V)
    rng = np.random.default_rng(11)
    g = np.linspace(-0.05, 1.05, 45)
    grid = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    P = np.concatenate([grid, rng.uniform(-0.2, 1.2, size=(20000, 3)), V,
                        0.5 * (V[F[:, 0]] + V[F[:, 1]]), V + rng.normal(scale=1e-6, size=V.shape)])
    old = _capi.tune_get(_capi.TUNE_SDF_RAY)
    try:
        _capi.tune_set(_capi.TUNE_SDF_RAY, 0)
        d_fan = ctx.signed_distance(V, F, P)
        _capi.tune_set(_capi.TUNE_SDF_RAY, 1)
        d_ray = ctx.signed_distance(V, F, P)
    finally:
        _capi.tune_set(_capi.TUNE_SDF_RAY, old)
    assert np.array_equal(np.abs(d_ray), np.abs(d_fan))
    # the two paths may differ only within 1e-9 of the surface, and there the
    # ray's side is the oracle's
    diff = np.nonzero(d_ray.view(np.uint64) != d_fan.view(np.uint64))[0]
    assert np.all(np.abs(d_fan[diff]) <= 1e-9)
    sel = diff if len(diff) <= 300 else rng.choice(diff, 300, replace=False)
    w = []
    for i in sel:
        wi = None
        for axis, sign in ((0, 1), (1, 1), (2, 1), (0, -1), (1, -1), (2, -1)):
            wi = exact_winding_number(V, F, P[i], axis, sign)
            if wi is not None:
                break
        w.append(wi)
    print(f"[sdf ray] {name}: {len(F)} triangles, {len(P)} points, {int((d_ray < 0).sum())} inside; "
          f"the fan sum's sign differs at {len(diff)}, all within 1e-9 of the surface", flush=True)
    assert all(wi is not None for wi in w)
    assert np.array_equal(np.signbit(d_ray[sel]), np.array(w) >= 1)
    if name == "flipped_sphere":
        # (within rounding of an edge line the ray leaves a point to the fan
        # sum, whose binary32 side is unreliable that close)
        assert not np.signbit(d_ray[np.abs(d_ray) > 1e-9]).any()
    else:
        assert (d_ray < 0).sum() > 1000


@pytest.mark.parametrize("N", [32768, 49151, 49152, 49153, 65021])
@pytest.mark.parametrize("name", ["icosphere", "open", "single", "nine", "collapsed"])
def test_sdf_packets(ctx, name, N):
    """Point sets walked in packets of 16 (from 49,152 points) against the
    same points in calls small enough to be walked one by one: identical bit
    for bit, since both take the exact minimum and exact crossings; and a
    sample of them against the brute-force oracle.  Dense points on the
    surface, a few far ones and coordinates that are huge, infinite or NaN;
    meshes of one bucket, two buckets and many levels, and one with faces of no
    area on chords of the sphere, with points around their centres."""
    from its_amd import meshes
    V, F = meshes.noisy_icosphere(seed=3, level=3)
    V = np.ascontiguousarray(V)
    if name == "open":
        F = F[40:]
    elif name == "single":
        F = F[:1]
    elif name == "nine":
        F = F[:9]
    chords = []
    if name == "collapsed":
        far = [(0, int(np.argmin(V @ V[0]))), (7, int(np.argmin(V @ V[7]))), (9, int(np.argmin(V @ V[9])))]
        V = np.concatenate([V, [0.5 * (V[far[2][0]] + V[far[2][1]])]])
        chords = [[far[0][0], far[0][0], far[0][1]], [far[1][0], far[1][1], far[1][1]],
                  [far[2][0], len(V) - 1, far[2][1]]]
        F = np.concatenate([F, chords])
    F = np.ascontiguousarray(F, np.int32)
    rng = np.random.default_rng(N)
    P = V[rng.integers(0, len(V), N)] + 0.03 * rng.standard_normal((N, 3))
    for q, f in enumerate(chords):
        P[30 + q::20] = V[f].mean(0) + 0.02 * rng.standard_normal(P[30 + q::20].shape)
    P[::97] = rng.uniform(-8, 8, size=(len(P[::97]), 3))
    P[5], P[777], P[-1] = [1e30, 0, 0], [np.inf, 0, 0], [np.nan, 0.1, 0.2]
    P[20:25] = V[F[0, 0]]   # ties between the triangles of a vertex
    d = ctx.signed_distance(V, F, P)
    one = np.concatenate([ctx.signed_distance(V, F, p) for p in np.array_split(P, 4)])
    print(f"[sdf packets] {name} N={N}: {int(np.signbit(d).sum())} negative", flush=True)
    clear = np.abs(d) > 1e-9   # nearer, a point that rays leave undecided takes the binary32 fan sum
    np.testing.assert_array_equal(np.abs(d), np.abs(one))
    np.testing.assert_array_equal(np.signbit(d[clear]), np.signbit(one[clear]))
    k = rng.choice(np.nonzero(np.isfinite(P).all(1) & (np.abs(P) < 1e3).all(1))[0], 2000, replace=False)
    assert np.isfinite(d[k]).all()
    assert np.abs(np.abs(d[k]) - np.abs(O.signed_distance(V, F, P[k]))).max() <= 1e-12


@pytest.mark.parametrize("T", [1, 7, 8, 9, 63, 64, 65, 511, 513, 4097, 81920])
def test_sdf_one_by_one(ctx, T):
    """The walk of one point a wavefront against the brute-force oracle: meshes
    that end inside a bucket or a leaf of 64, below and above 512 leaves.  At the
    sphere's centre every leaf is needed, so that with 1,280 of them the frontier
    stays above the leaves; far away rays and distances start outside."""
    V, F = meshes.icosphere(6) if T > 20000 else meshes.noisy_icosphere(seed=3, level=4)
    F = np.ascontiguousarray(F[:T], np.int32)
    assert len(F) == T
    rng = np.random.default_rng(T)
    P = np.concatenate([np.zeros((1, 3)), 1e-3 * rng.standard_normal((20, 3)), 5 * rng.standard_normal((20, 3)),
                        V[F[rng.integers(0, T, 60), 0]] + 0.02 * rng.standard_normal((60, 3)), [[40.0, 0, 0]]])
    print(f"[sdf one by one] T={T}", flush=True)
    d = ctx.signed_distance(V, F, P)
    ref = O.signed_distance(V, F, P)
    assert np.abs(np.abs(d) - np.abs(ref)).max() <= 1e-12
    w = np.array([O.winding_number(V, F, p) for p in P])
    clear = (np.abs(ref) > 1e-6) & (np.abs(w - 0.5) > 1e-3)
    assert clear.sum() > 90
    np.testing.assert_array_equal(np.signbit(d[clear]), np.signbit(ref[clear]))


def _collapsed_mesh(order):
    """Closed sphere and one face on the chord between two far vertices i and
    j, of no area: a repeated corner (the distance to it is 0 / 0 for half of
    space in one of the orders) or three collinear ones."""
    V, F = meshes.icosphere(3)
    i, j = 0, int(np.argmin(V @ V[0]))
    V = np.concatenate([V, [0.3 * V[i] + 0.7 * V[j]]])
    face = {"iij": [i, i, j], "ijj": [i, j, j], "iji": [i, j, i], "line": [i, len(V) - 1, j]}[order]
    return np.ascontiguousarray(V), np.concatenate([F, [face]]).astype(np.int32), i, j


@pytest.mark.parametrize("N", [2000, 50021])
@pytest.mark.parametrize("order", ["iij", "ijj", "iji", "line"])
def test_sdf_collapsed_face(ctx, order, N):
    """Points around a face of no area far from all others, one by one and in
    packets, against the brute-force oracle: the face bounds no distance that
    it does not have."""
    V, F, i, j = _collapsed_mesh(order)
    rng = np.random.default_rng(N)
    P = V[i] + rng.uniform(-0.05, 1.05, (N, 1)) * (V[j] - V[i]) + 0.02 * rng.standard_normal((N, 3))
    P[: N // 2] = V[F[-1]].mean(0) + 0.02 * rng.standard_normal((N // 2, 3))   # around its centre
    print(f"[sdf collapsed] {order} N={N}", flush=True)
    d = ctx.signed_distance(V, F, P)
    ref = O.signed_distance(V, F, P)
    assert np.isfinite(d).all()
    assert np.abs(np.abs(d) - np.abs(ref)).max() <= 1e-12


@pytest.mark.parametrize("order", ["iij", "line"])
def test_sdf_collapsed_face_at_vertices(ctx, order):
    """The same at the octree's vertices, some of which lie along the face."""
    from its_amd import _capi
    V, F, _, _ = _collapsed_mesh(order)
    V = O.normalize(V)
    o, _, w = O.uniform_bbox(V)
    g = _capi.Octree(ctx, meshes.triangles(V, F), o, w, 32)
    print(f"[sdf collapsed] {order} n={g.num_verts}", flush=True)
    b = g.sdf_at_vertices(V, F)
    assert np.isfinite(b).all()
    assert np.abs(np.abs(b) - np.abs(O.signed_distance(V, F, g.verts()[0]))).max() <= 1e-12


def _rim_mesh(kind):
    rng = np.random.default_rng(21)
    if kind in ("limit", "over", "long", "too_long"):
        # two rings of n quads: 4n triangles, 2n boundary half edges; the ray and
        # the rim take one per two triangles, and 4,096, at most
        n = {"limit": 300, "over": 300, "long": 2048, "too_long": 2049}[kind]
        a = 2 * np.pi * np.arange(n) / n
        V = np.concatenate([np.stack([np.cos(a), np.sin(a), z + 0 * a], 1) for z in (-0.7, 0.1, 0.8)])
        V = V + rng.uniform(-1e-3, 1e-3, V.shape)
        i, j = np.arange(n), (np.arange(n) + 1) % n
        F = np.concatenate([np.stack(t, 1) for o in (0, n) for t in ((i + o, j + o, j + o + n), (i + o, j + o + n, i + o + n))])
        return V, np.ascontiguousarray(F[1 if kind == "over" else 0:], np.int32)
    V, F = meshes.noisy_icosphere(seed=2, level=3)
    if kind == "patch":
        F = F[np.linalg.norm(V[F].mean(1) - V[5], axis=1) > 0.2]
    elif kind == "holes":
        F = F[rng.random(len(F)) > 0.05]
    elif kind == "flipped":
        flip = rng.random(len(F)) < 0.03
        F = np.where(flip[:, None], F[:, ::-1], F)
    elif kind == "doubled":   # 60 triangles twice, three degenerate ones
        F = np.concatenate([F[100:], F[300:360], [[5, 5, 9], [7, 8, 8], [4, 4, 4]]])
    return V, np.ascontiguousarray(F, np.int32)


@pytest.mark.parametrize("N", [1, 63, 2000, 50021])
@pytest.mark.parametrize("kind", ["patch", "holes", "flipped", "doubled", "limit", "over", "long", "too_long"])
def test_sdf_rim_signs(ctx, kind, N):
    """Meshes with a boundary: distances are the brute-force oracle's (on a
    sample), signs those of the winding number summed over all triangles in
    binary64, wherever that is farther than 1e-4 from 1/2 (binary32 sums of 1,000
    angles)."""
    import torch
    V, F = _rim_mesh(kind)
    rng = np.random.default_rng(N)
    lo, hi = V.min(0), V.max(0)
    P = rng.uniform(lo - 0.1 * (hi - lo), hi + 0.1 * (hi - lo), (N, 3))
    near = rng.random(N) < 0.5
    P[near] = V[rng.integers(len(V), size=near.sum())] + rng.normal(0, 0.01, (near.sum(), 3))
    print(f"[rim] {kind} T={len(F)} N={N}", flush=True)
    d = ctx.signed_distance(V, F, P)
    T, Q = torch.from_numpy(V[F]).cuda(), torch.from_numpy(P).cuda()
    w = torch.zeros(N, dtype=torch.float64, device="cuda")
    for s in range(0, N, 4000):
        a, b, c = (T[None, :, k] - Q[s:s + 4000, None] for k in range(3))
        la, lb, lc = a.norm(dim=2), b.norm(dim=2), c.norm(dim=2)
        det = (a * torch.linalg.cross(b, c)).sum(2)
        den = la * lb * lc + (a * b).sum(2) * lc + (b * c).sum(2) * la + (c * a).sum(2) * lb
        w[s:s + 4000] = torch.atan2(det, den).sum(1) / (2 * np.pi)
    w = w.cpu().numpy()
    assert np.isfinite(d).all()
    k = rng.choice(N, min(N, 1000), replace=False)
    assert np.abs(np.abs(d[k]) - np.abs(O.signed_distance(V, F, P[k]))).max() <= 1e-12
    sure = (np.abs(w - 0.5) > 1e-4) & (np.abs(d) > 1e-9)
    assert sure.mean() > 0.9
    assert np.array_equal(np.signbit(d)[sure], (w > 0.5)[sure])


def test_sdf_rim_many_points(ctx):
    """More points than the rim kernel's resident blocks take at once: the
    same points in calls that need one round, bit for bit."""
    V, F = _rim_mesh("patch")
    rng = np.random.default_rng(8)
    N = 300_007
    P = rng.uniform(V.min(0) - 0.1, V.max(0) + 0.1, (N, 3))
    print(f"[rim] patch T={len(F)} N={N}", flush=True)
    d = ctx.signed_distance(V, F, P)
    one = np.concatenate([ctx.signed_distance(V, F, p) for p in np.array_split(P, 10)])
    clear = np.abs(d) > 1e-9
    np.testing.assert_array_equal(np.abs(d), np.abs(one))
    np.testing.assert_array_equal(np.signbit(d[clear]), np.signbit(one[clear]))


def test_sdf_points_beyond_a_launch(ctx):
    """2^29 + 3 points (13 GB) around a mesh with a boundary: more work items
    than one launch dimension holds, for the rim kernel.  The points are one
    set of 2^20 over and over, so the results are that set's."""
    import psutil
    if psutil.virtual_memory().available < 40 << 30:
        pytest.skip("needs 40 GiB of host memory")
    V, F = _rim_mesh("patch")
    rng = np.random.default_rng(4)
    B, N = 1 << 20, (1 << 29) + 3
    T = rng.uniform(V.min(0) - 0.2, V.max(0) + 0.2, (B, 3))
    base = ctx.signed_distance(V, F, T)
    P = np.empty((N, 3))
    for s in range(0, N, B):
        P[s:s + B] = T[:min(B, N - s)]
    print(f"[sdf] N={N}", flush=True)
    d = ctx.signed_distance(V, F, P)
    clear = np.abs(base) > 1e-9
    for s in range(0, N, B):
        n = min(B, N - s)
        assert np.array_equal(np.abs(d[s:s + n]), np.abs(base[:n]))
        assert np.array_equal(d[s:s + n][clear[:n]], base[:n][clear[:n]])


@pytest.mark.parametrize("hole", [False, True])
def test_sdf_many_half_edges(ctx, hole):
    """Above 2^23 half edges they are sorted, not hashed, to find the boundary:
    the ray's signs are the fan walk's."""
    from its_amd import _capi
    V, F = meshes.torus(1700, 850)
    assert 3 * len(F) > 1 << 23
    if hole:
        F = np.ascontiguousarray(F[np.linalg.norm(V[F].mean(1) - V[1000], axis=1) > 0.01])
    rng = np.random.default_rng(5)
    P = V[rng.integers(len(V), size=3000)] + rng.normal(0, 0.02, (3000, 3))
    print(f"[many half edges] T={len(F)}", flush=True)
    d = ctx.signed_distance(V, F, P)
    old = _capi.tune_get(_capi.TUNE_SDF_RAY)
    _capi.tune_set(_capi.TUNE_SDF_RAY, 0)
    fan = ctx.signed_distance(V, F, P)
    _capi.tune_set(_capi.TUNE_SDF_RAY, old)
    assert np.array_equal(d, fan)
    assert 0.3 < np.signbit(d).mean() < 0.7
