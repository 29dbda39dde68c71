"""Runs of small passes in one launch (k_small_rounds) against the separate
kernels, and the separate kernels' own variants against each other.  The
training logs need the separate kernels, so the same options with log_training
= 1 never take the one-launch path: mesh and statistics have to be equal bit
for bit.  The inputs cross the limits of the path: passes of
more and fewer candidates than it takes, cavities beyond its LDS and undecided
signs (left to the exact kernel inside a pass), capacity doubling and mesh
growth, the selection by priority, a round limit, and lists reallocated while
they grow (vmm = 0)."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CHOSEN = dict(pred_mode=1, claim_iters=3, seg_claim_iters=2, mix_below=4, shared_ring=1,
              cand_factor=3, learned_shift=1)
CASES = [
    (9, 0, {}),
    (40, 1, {}),
    (300, 0, {}),
    (300, 0, dict(CHOSEN, priority=1)),
    (301, 1, dict(CHOSEN, priority=2)),
    (2000, 0, dict(CHOSEN, priority=2)),
    (2000, 1, dict(CHOSEN, priority=1, vmm=0)),
    (1203, 3, dict(CHOSEN, priority=2, theta=30.0)),
    (1200, 2, dict(CHOSEN, priority=1)),
    (700, 0, dict(max_rounds=7)),
    (700, 0, dict(CHOSEN, priority=2, max_rounds=11)),
    (900, 0, dict(cand_min=40, cand_factor=2)),
    (900, 1, dict(cand_min=40, cand_factor=2, priority=0)),
    (800, 1, dict(cav_cap0=4)),
    (800, 0, dict(CHOSEN, priority=1, cav_cap0=4, cav_cap_max=8)),
    (800, 0, dict(CHOSEN, priority=2, cav_lds_cap=6)),
    (600, 0, dict(cand_budget=16 * 208, cav_cap_max=64)),
    (700, 1, dict(CHOSEN, priority=2, mode=0)),
    (1500, 0, dict(mode=0, deletion=0)),
    (1500, 1, dict(mode=0, deletion=1, vmm=0)),
    (500, 0, dict(mode=1, deletion=2, claim_iters=2, mix_below=300)),
]
SAME = ["rounds", "seg_passes", "bad_passes", "status", "seg_splits", "inserted", "lost",
        "rej_encroach", "rej_blocked", "rej_overflow", "giveups", "cand_evals", "deleted", "flips",
        "n_points", "n_triangles", "n_subsegs", "final_cav_cap", "pred_fp32", "pred_fp64",
        "pred_exact", "pred_dd", "tri_examined_seg", "tri_examined_bad", "ws_ints_seg",
        "ws_ints_bad", "big_cavities"]


def _run(gpu, mesh, opt, log):
    o = dict(opt)
    s = gpu.Session(*mesh, theta=o.pop("theta", 25.0), mode=o.pop("mode", 1), log_training=log,
                    cav_lds_cap=o.pop("cav_lds_cap", 32), **o)
    try:
        if opt.get("priority") == 2:
            s.set_priority_model(np.load(os.path.join(os.path.dirname(gpu.__file__),
                                                      "priority_mlp.npy")))
        s.run()
        st = s.run()  # the second run starts from a used session
        return s.download(), st
    finally:
        s.close()


@pytest.mark.parametrize("n,dist,opt", CASES)
def test_small_rounds_equal_separate_kernels(gpu, n, dist, opt):
    print(f"small rounds n={n} dist={dist} {opt}", flush=True)
    P, S0 = gpu.generate_pslg(n, max(1, n // 20), L=64.0 * n ** 0.5, maxlen=1280.0, dist=dist,
                              min_angle=5.0, seed=100 + n)
    mesh = (P,) + tuple(gpu.build_cdt(P, S0))
    a, sa = _run(gpu, mesh, opt, 0)
    b, sb = _run(gpu, mesh, opt, 1)
    assert {k: sa[k] for k in SAME} == {k: sb[k] for k in SAME}
    assert np.array_equal(a.points.view(np.uint64), b.points.view(np.uint64))
    for f in ("triangles", "neighbors", "segments", "pstatus", "tstatus"):
        assert np.array_equal(getattr(a, f), getattr(b, f)), f


@pytest.mark.parametrize("dist,opt", [(0, dict(CHOSEN, priority=1, mix_below=0)),
                                      (1, dict(claim_iters=2)), (0, dict(mode=0))])
def test_located_candidates_equal_inline(gpu, dist, opt):
    """A first bad pass of more than 16,384 candidates is located by a lane per
    candidate in the host loop; the graph loop's cavities locate their own."""
    print(f"located dist={dist} {opt}", flush=True)
    n = 14000
    P, S0 = gpu.generate_pslg(n, n // 20, L=64.0 * n ** 0.5, maxlen=1280.0, dist=dist,
                              min_angle=5.0, seed=77)
    mesh = (P,) + tuple(gpu.build_cdt(P, S0))
    a, sa = _run(gpu, mesh, dict(opt, graph=0, cand_min=1 << 20), 0)
    b, sb = _run(gpu, mesh, dict(opt, graph=1, cand_min=1 << 20), 0)
    for k in ("rounds", "inserted", "seg_splits", "giveups", "flips", "cand_evals"):
        assert sa[k] == sb[k], k
    assert np.array_equal(a.points.view(np.uint64), b.points.view(np.uint64))
    assert np.array_equal(a.triangles, b.triangles) and np.array_equal(a.neighbors, b.neighbors)
    # one round holds one bad pass: the first is large enough to be located
    first = _run(gpu, mesh, dict(opt, graph=0, cand_min=1 << 20, max_rounds=1), 0)[1]
    assert first["bad_passes"] == 1 and first["cand_evals"] > 16384


def _encroached(P, T, S):
    """Subsegments with the apex of an adjacent triangle strictly inside their
    diametral circle."""
    key = lambda a, b: np.minimum(a, b).astype(np.int64) * len(P) + np.maximum(a, b)
    want = key(S[:, 0], S[:, 1])
    hit = []
    for j in range(3):
        c, a, b = T[:, j], T[:, (j + 1) % 3], T[:, (j + 2) % 3]
        inside = ((P[a] - P[c]) * (P[b] - P[c])).sum(1) < 0
        hit.append(key(a[inside], b[inside]))
    return int(np.isin(want, np.concatenate(hit)).sum())


@pytest.mark.parametrize("opt", [dict(CHOSEN, priority=1, mix_below=0), dict(mode=0)])
def test_located_subsegments_equal_inline(gpu, opt):
    """A first segment pass of more than 16,384 subsegments, the same way."""
    print(f"located subsegments {opt}", flush=True)
    n = 60000
    P, S0 = gpu.generate_pslg(n, 40000, L=64.0 * n ** 0.5, maxlen=400.0, dist=0, min_angle=5.0,
                              seed=78)
    mesh = (P,) + tuple(gpu.build_cdt(P, S0))
    assert _encroached(P, mesh[1], mesh[3]) > 16384
    o = dict(opt, theta=20.7)
    a, sa = _run(gpu, mesh, dict(o, graph=0), 0)
    b, sb = _run(gpu, mesh, dict(o, graph=1), 0)
    for k in ("rounds", "seg_passes", "inserted", "seg_splits", "giveups", "flips", "cand_evals"):
        assert sa[k] == sb[k], k
    assert np.array_equal(a.points.view(np.uint64), b.points.view(np.uint64))
    assert np.array_equal(a.triangles, b.triangles) and np.array_equal(a.segments, b.segments)


@pytest.mark.parametrize("n,seed,rounds,cap", [(20, 1, 1, 4), (40, 1, 3, 8), (60, 2, 1, 8),
                                               (100, 1, 1, 4)])
def test_cavity_capacity_at_the_round_limit(gpu, n, seed, rounds, cap):
    """A pass that overflows a cavity and is also the last round: the capacity
    a run ends with does not depend on the path its last pass took."""
    print(f"capacity at round limit n={n} rounds={rounds}", flush=True)
    P, S0 = gpu.generate_pslg(n, max(1, n // 20), L=64.0 * n ** 0.5, maxlen=1280.0, dist=0,
                              min_angle=5.0, seed=seed)
    mesh = (P,) + tuple(gpu.build_cdt(P, S0))
    opt = dict(cav_cap0=cap, max_rounds=rounds)
    a, sa = _run(gpu, mesh, opt, 0)
    b, sb = _run(gpu, mesh, opt, 1)
    assert sa["rounds"] == rounds and sa["rej_overflow"] > 0
    assert {k: sa[k] for k in SAME} == {k: sb[k] for k in SAME}
    assert np.array_equal(a.triangles, b.triangles)


def test_evaluations_off_the_fast_path(gpu):
    """big_cavities: the evaluations left to the exact kernel.  The number
    does not depend on the path, grows as the fast path's capacity shrinks,
    and counts undecided signs alone when every cavity fits."""
    P, S0 = gpu.generate_pslg(800, 40, L=64.0 * 800 ** 0.5, maxlen=1280.0, dist=0, min_angle=5.0,
                              seed=900)
    mesh = (P,) + tuple(gpu.build_cdt(P, S0))
    big = {}
    for cap in (4, 8, 32):
        opt = dict(CHOSEN, priority=1, mix_below=0, cav_lds_cap=cap, cav_cap0=32)
        st = [_run(gpu, mesh, opt, log)[1] for log in (0, 1)]
        st.append(_run(gpu, mesh, dict(opt, graph=1), 0)[1])
        assert st[0]["big_cavities"] == st[1]["big_cavities"] == st[2]["big_cavities"], cap
        big[cap] = st[0]["big_cavities"]
    assert big[4] > big[8] > big[32]


@pytest.mark.parametrize("k,cap", [(40, 36), (40, 64), (60, 48), (60, 64), (68, 69), (72, 69),
                                   (72, 70), (72, 128), (72, 256)])
def test_fast_path_capacity_above_the_default(gpu, oracle, k, cap):
    """cav_lds_cap beyond 32 holds in small passes too: only cavities beyond
    the caller's capacity, or beyond the 69 triangles the one-launch rounds have
    room for, leave the fast path."""
    from test_gpu_parity import circle_pslg
    print(f"fast path capacity k={k} cap={cap}", flush=True)
    mesh = circle_pslg(oracle, k=k, n_out=30)
    opt = dict(CHOSEN, priority=1, cav_lds_cap=cap, cav_cap0=256)
    a, sa = _run(gpu, mesh, opt, 0)
    b, sb = _run(gpu, mesh, opt, 1)
    # deferred candidates are examined again: two counts follow the capacity
    same = [q for q in SAME if cap <= 69 or q not in ("big_cavities", "tri_examined_bad")]
    assert {q: sa[q] for q in same} == {q: sb[q] for q in same}
    assert np.array_equal(a.points.view(np.uint64), b.points.view(np.uint64))
    assert np.array_equal(a.triangles, b.triangles)
    if cap >= k and k < 69:  # the ring's fan of k - 2 triangles is one cavity: it fits now
        narrow = _run(gpu, mesh, dict(opt, cav_lds_cap=32), 0)[1]
        assert narrow["big_cavities"] > sa["big_cavities"]


def test_profile_rows_hold_every_pass(gpu):
    """profile = 1: the cavity rows time every pass that the statistics count,
    the small ones too, and profiling does not change the mesh."""
    P, S0 = gpu.generate_pslg(2000, 100, L=64.0 * 2000 ** 0.5, maxlen=1280.0, dist=0,
                              min_angle=5.0, seed=400)
    mesh = (P,) + tuple(gpu.build_cdt(P, S0))
    res = []
    for profile in (0, 1):
        s = gpu.Session(*mesh, theta=25.0, mode=1, profile=profile, priority=1, **CHOSEN)
        try:
            st = s.run()
            res.append((st, s.download(), s.kernel_times()))
        finally:
            s.close()
    (sa, a, _), (sb, b, kt) = res
    assert {k: sa[k] for k in SAME} == {k: sb[k] for k in SAME}
    assert np.array_equal(a.points.view(np.uint64), b.points.view(np.uint64))
    assert kt["bad_cavity"]["launches"] == sb["bad_passes"]
    assert kt["bad_cavity"]["items"] == sb["cand_evals"]
    assert kt["seg_cavity"]["launches"] == sb["seg_passes"]
    assert kt["apply"]["items"] == sb["inserted"] + sb["seg_splits"]


# what does not depend on how many lanes test a triangle at the same time
LANE_SAME = [k for k in SAME if not k.startswith(("pred_", "tri_examined"))]


@pytest.mark.parametrize("case", ["uniform", "overflow", "deferred", "chew", "ring"])
@pytest.mark.parametrize("lanes", [8, 32, 64])
def test_lane_groups_equal_the_default(gpu, oracle, case, lanes):
    """The filtered cavity kernel with 8, 32 and 64 lanes per candidate against
    16: cavities that overflow the capacity, that leave the fast path, and
    stars longer than a lane group.  (The training logs keep every pass out of
    the one-launch rounds, whose group size is fixed.)"""
    print(f"lane groups {case} {lanes}", flush=True)
    opt = {"uniform": dict(CHOSEN, priority=1), "overflow": dict(cav_cap0=4),
           "deferred": dict(CHOSEN, priority=1, cav_lds_cap=6), "chew": dict(mode=0, claim_iters=2),
           "ring": dict(CHOSEN, priority=1, cav_cap0=128, cav_lds_cap=128)}[case]
    if case == "ring":
        from test_gpu_parity import circle_pslg
        mesh = circle_pslg(oracle)
    else:
        P, S0 = gpu.generate_pslg(2500, 125, L=64.0 * 50, maxlen=1280.0, dist=1, min_angle=5.0,
                                  seed=500)
        mesh = (P,) + tuple(gpu.build_cdt(P, S0))
    a, sa = _run(gpu, mesh, opt, 1)
    b, sb = _run(gpu, mesh, dict(opt, cavity_lanes=lanes), 1)
    assert {k: sa[k] for k in LANE_SAME} == {k: sb[k] for k in LANE_SAME}
    if case == "overflow":
        assert sa["rej_overflow"] > 0
    if case == "deferred":
        assert sa["big_cavities"] > 1000
    assert np.array_equal(a.points.view(np.uint64), b.points.view(np.uint64))
    for f in ("triangles", "neighbors", "segments", "pstatus", "tstatus"):
        assert np.array_equal(getattr(a, f), getattr(b, f)), f
