"""GPU construction of the input CDT (gcdt_build_cdt_device) against the host
builder and, where its library is built (oracle/_ref, compiled from the
reference's own source), the reference's Triangle ("pzQnc", mesh.cpp:397): the
same triangles and the same segments where no four points are cocircular, a
valid constrained Delaunay triangulation everywhere (exact checker), identical
output run to run, segments split where they pass through input points,
segments that cross hundreds of triangles, and the result refined by the GPU
path."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _canon(T):
    T = np.asarray(T).reshape(-1, 3)
    r = np.argmin(T, axis=1)
    i = np.arange(len(T))
    return set(map(tuple, np.stack([T[i, r], T[i, (r + 1) % 3], T[i, (r + 2) % 3]], 1).tolist()))


def _segset(S):
    return set(tuple(sorted(x)) for x in np.asarray(S).reshape(-1, 2).tolist())


def _valid(oracle, P, T, N, S):
    tot, viol, mina, ex = oracle.check_mesh(P, T, N, S, P, S, 1e-6)
    assert tot == 0, viol


FAMILIES = [(2000, 100, 0, 1), (20000, 1000, 1, 2), (60000, 3000, 0, 3), (20000, 1000, 3, 4),
            (20000, 1000, 4, 5), (20000, 1000, 5, 6), (20000, 1000, 6, 7)]


def _family(gpu, n, ns, dist, seed):
    L = 1000.0 * (n / 10000) ** 0.5
    return gpu.generate_pslg(n, ns, L=L, maxlen=0.05 * L, dist=dist, min_angle=5.0, seed=seed)


@pytest.mark.parametrize("n,ns,dist,seed", FAMILIES)
def test_gpu_cdt_equals_host_builder(gpu, oracle, n, ns, dist, seed):
    print(f"gpu cdt n={n} dist={dist}", flush=True)
    P, S0 = _family(gpu, n, ns, dist, seed)
    T, N, S = gpu.build_cdt(P, S0, device=True)
    _valid(oracle, P, T, N, S)
    T2, N2, S2 = gpu.build_cdt(P, S0, device=True)
    assert np.array_equal(T, T2) and np.array_equal(N, N2) and np.array_equal(S, S2)
    Th, Nh, Sh = gpu.build_cdt(P, S0)
    assert _canon(T) == _canon(Th) and _segset(S) == _segset(Sh)


@pytest.mark.parametrize("n,ns,dist,seed", FAMILIES)
def test_gpu_cdt_equals_triangle(gpu, oracle, n, ns, dist, seed):
    if not os.path.exists(oracle.TRIREF_SO):
        pytest.skip("reference Triangle not built")
    P, S0 = _family(gpu, n, ns, dist, seed)
    T, N, S = gpu.build_cdt(P, S0, device=True)
    Pt, Tt, Nt, St = oracle.triangle_cdt(P, S0)
    assert _canon(T) == _canon(Tt)
    assert _segset(S) == _segset(St)


def test_gpu_cdt_precision_family(gpu, oracle):
    """Jittered lattice, exactly cocircular groups, segments along lattice
    lines: where four points are cocircular any Delaunay choice is valid, so
    the mesh is held to the exact checker and to the segments and triangle
    count of Triangle (of the host builder where Triangle is not built)."""
    P, S0 = gpu.generate_pslg(20000, 400, L=1000.0 * 0.02 ** 0.5, maxlen=20.0, dist=2,
                              min_angle=5.0, seed=2)
    T, N, S = gpu.build_cdt(P, S0, device=True)
    Pt, Tt, Nt, St = oracle.triangle_cdt(P, S0)
    assert len(T) == len(Tt)
    assert _segset(S) == _segset(St)
    _valid(oracle, P, T, N, S)


def test_gpu_cdt_segment_through_points(gpu, oracle):
    """A segment through three input points is split into four pieces; a
    grid of points (every quadrilateral cocircular) with segments along its
    lines and diagonals; compared with Triangle, or the host builder where
    Triangle is not built."""
    g = 12
    xs, ys = np.meshgrid(np.arange(g, dtype=np.float64), np.arange(g, dtype=np.float64))
    P = np.stack([xs.ravel(), ys.ravel()], 1)
    idx = lambda x, y: y * g + x
    S0 = np.array([[idx(0, 2), idx(8, 2)], [idx(1, 1), idx(7, 7)], [idx(10, 0), idx(10, 9)],
                   [idx(3, 9), idx(9, 3)]], np.int32)
    T, N, S = gpu.build_cdt(P, S0, device=True)
    Pt, Tt, Nt, St = oracle.triangle_cdt(P, S0)
    assert _segset(S) == _segset(St)
    assert len(T) == len(Tt)
    _valid(oracle, P, T, N, S)
    # the first input segment comes out as its 8 unit pieces, in order
    assert [tuple(x) for x in S[:8].tolist()] == [(idx(k, 2), idx(k + 1, 2)) for k in range(8)]


def test_gpu_cdt_feeds_the_refinement(gpu, oracle):
    P, S0 = gpu.generate_pslg(30000, 1500, L=1000.0 * 3 ** 0.5, maxlen=80.0, dist=1,
                              min_angle=5.0, seed=9)
    T, N, S = gpu.build_cdt(P, S0, device=True)
    r = gpu.refine(P, T, N, S, theta=25.0, claim_iters=3, shared_ring=1)
    assert r.stats["status"] == 0
    c = gpu.check_mesh(r.points, r.triangles, r.neighbors, r.segments, points_in=P,
                       segments_in=S, theta=25.0)
    assert gpu.violations(c) == 0, c


@pytest.mark.parametrize("n,dist,seed", [(3, 0, 21), (7, 0, 22), (3000, 0, 23), (5001, 3, 24)])
def test_gpu_cdt_without_segments(gpu, oracle, n, dist, seed):
    """A bare point set, right after a build with segments whose freed device
    memory it may be given: only the hull edges come out as segments."""
    print(f"gpu cdt without segments n={n}", flush=True)
    Q, S0 = gpu.generate_pslg(3000, 300, L=500.0, maxlen=50.0, dist=0, min_angle=5.0, seed=20)
    gpu.build_cdt(Q, S0, device=True)
    P = gpu.generate_pslg(max(n, 40), 1, L=1000.0, maxlen=500.0, dist=dist, min_angle=5.0,
                          seed=seed)[0][:n]
    none = np.zeros((0, 2), np.int32)
    T, N, S = gpu.build_cdt(P, none, device=True)
    Th, Nh, Sh = gpu.build_cdt(P, none)
    assert _canon(T) == _canon(Th) and _segset(S) == _segset(Sh)
    assert len(S) == int((N == -1).sum())
    _valid(oracle, P, T, N, S)


def _crossed(P, T, a, b):
    """Triangles of the triangulation T that segment (a, b) crosses (no other
    point lies on it)."""
    E = np.unique(np.sort(np.concatenate([T[:, [0, 1]], T[:, [1, 2]], T[:, [2, 0]]]), axis=1),
                  axis=0)
    E = E[~np.isin(E, [a, b]).any(1)]
    side = lambda X, Y, Z: ((Y[..., 0] - X[..., 0]) * (Z[..., 1] - X[..., 1]) -
                            (Y[..., 1] - X[..., 1]) * (Z[..., 0] - X[..., 0]))
    A, B, U, V = P[a], P[b], P[E[:, 0]], P[E[:, 1]]
    return int(((side(A, B, U) * side(A, B, V) < 0) & (side(U, V, A) * side(U, V, B) < 0)).sum()) + 1


@pytest.mark.parametrize("n,seed,sizes", [(20000, 31, (280, 153, 308, 304, 11)),
                                          (90000, 32, (618, 299, 606, 582, 29))])
def test_gpu_cdt_long_segments(gpu, oracle, n, seed, sizes):
    """Segments that cross more triangles than a region kept in LDS (128) and
    than the first region capacity (512, grown when a pass is stuck)."""
    print(f"gpu cdt long segments n={n}", flush=True)
    P = np.random.default_rng(seed).uniform(0, 1000, (n, 2))
    near = lambda x, y: int(np.argmin((P[:, 0] - x) ** 2 + (P[:, 1] - y) ** 2))
    S0 = np.array([(near(20, y), near(x, y + 3)) for y, x in
                   ((100, 980), (300, 500), (500, 980), (700, 980), (900, 60))], np.int32)
    T0 = gpu.build_cdt(P, np.zeros((0, 2), np.int32))[0]
    assert tuple(_crossed(P, T0, a, b) for a, b in S0) == sizes
    T, N, S = gpu.build_cdt(P, S0, device=True)
    Th, Nh, Sh = gpu.build_cdt(P, S0)
    assert _canon(T) == _canon(Th) and _segset(S) == _segset(Sh)
    assert np.array_equal(S[:len(S0)], S0)
    _valid(oracle, P, T, N, S)


def test_gpu_cdt_long_segments_cocircular(gpu, oracle):
    """Long regions of an integer grid, where every quadrilateral is
    cocircular and the exact kernel retriangulates."""
    g = 72
    xs, ys = np.meshgrid(np.arange(g, dtype=np.float64), np.arange(g, dtype=np.float64))
    P = np.stack([xs.ravel(), ys.ravel()], 1)
    S0 = np.array([[0, 70 * g + 71], [10 * g, 69 * g + 50]], np.int32)  # slopes 70/71, 59/50
    T, N, S = gpu.build_cdt(P, S0, device=True)
    Th, Nh, Sh = gpu.build_cdt(P, S0)
    assert _segset(S) == _segset(Sh) and len(T) == len(Th)
    assert np.array_equal(S[:2], S0)
    _valid(oracle, P, T, N, S)
