"""Performance cases: the work a user of this framework has it do.

Every case is one pass through public entry points of gpu_cdt_refine_amd.
The kinds, and what each stands for in real use:

  dropin   the C++ drop-in GPU_Refine_Quality, host triangulateio in and out:
           the call a program of the reference makes.  Latency-bound at a few
           hundred points (a mesher called in a loop), throughput-bound at
           10^6 points (the headline workload of bench.py).
  session  a CDT resident in device memory, refined again and again and
           downloaded (parameter studies): the library's default options (the
           plain path), and the graph-driven loop.
  refine   the one-shot C ABI gcdt_refine_host, every buffer allocated by the
           call, here on the precision-stress family (exactly cocircular and
           jittered lattice points: the exact predicate stages).
  batch    many small PSLGs with their own angle and mode refined together,
           with the split into per-instance results.
  cdt      construction of the constrained Delaunay triangulation on the GPU
           from points and segments in host memory: the step before every
           refinement.
  check    the exact invariant checker on a refined mesh in device memory, the
           non-allocating entry point of serving loops (meshes of up to about
           350,000 triangles), auditing against an angle of the caller's.
  mlp      one full-batch step of the claim-priority network's training:
           forward (inference) and gradient, from host arrays.

Meshes and counts are compared exactly: every sign is exact and every choice
(candidate order, claims, numbering) is deterministic, so a refined mesh is
the same bit for bit whatever kernels made it.

A case names its PSLG ("base", the generator's seed); the seed of prepare()
is the unit of length it is given in, a power of two.  Every coordinate, and
so every input and output point, differs from seed to seed, while the sizes
of the outputs stay those of the case.  A CDT's points are also renumbered by
the seed, and a check's angle depends on it.
"""
import os

import numpy as np
import torch

import gpu_cdt_refine_amd as g

SPACING = 64.0  # mean distance of neighbouring input points in the base unit
MODEL = os.path.join(os.path.dirname(g.__file__), "priority_mlp.npy")


def listed():
    return [
        # a mesher called on one small part at a time: launches and round trips
        dict(name="dropin-300", kind="dropin", n=300, dist=0, base=1, theta=25.0, offcenter=1,
             ruppert=1),
        # a small part in Chew mode (vertex deletion) at a demanding angle
        dict(name="dropin-3k-chew30", kind="dropin", n=2999, dist=0, base=2, theta=30.0,
             offcenter=1, ruppert=0),
        # Gaussian-clustered points, the family and angle of the learned-priority benchmark
        dict(name="dropin-41k-clustered28", kind="dropin", n=41003, dist=1, base=3, theta=28.0,
             offcenter=1, ruppert=1),
        # the headline workload: 10^6 uniform points, 50,000 segments, 25 degrees
        dict(name="dropin-1M", kind="dropin", n=1_000_000, dist=0, base=4, theta=25.0, offcenter=1,
             ruppert=1),
        # library defaults (no model, FP64 filter), circumcenters, Chew mode, resident input
        dict(name="session-plain-150k", kind="session", form="plain", n=150_001, dist=0, base=5,
             theta=25.0, offcenter=0, ruppert=0),
        # the device-driven loop (hipGraph), disk-shaped domain
        dict(name="session-graph-20k", kind="session", form="graph", n=20_011, dist=3, base=6,
             theta=25.0, offcenter=1, ruppert=1),
        # one-shot call on the precision-stress family
        dict(name="refine-precision-12k", kind="refine", n=12_007, dist=2, base=7, theta=25.0,
             offcenter=1, ruppert=1),
        # 16 instances of 200 to 20,000 points, angles 20.7 to 30 degrees, both modes
        dict(name="batch-16", kind="batch", k=16, nmax=20_000, base=8),
        # CDT construction, small and large
        dict(name="cdt-4k", kind="cdt", n=4001, dist=1, base=9),
        dict(name="cdt-500k", kind="cdt", n=500_009, dist=0, base=10),
        # invariant check of a mesh of about 3 * 10^5 triangles
        dict(name="check-30k", kind="check", n=30_003, dist=0, base=11, theta=25.0,
             offcenter=1, ruppert=1),
        # a training step of the priority network on 200,000 logged candidates
        dict(name="mlp-200k", kind="mlp", n=200_003),
    ]


def _log_int(rng, lo, hi):
    return int(round(np.exp(rng.uniform(np.log(lo), np.log(hi)))))


def draw(rng):
    kind = rng.choice(["dropin", "dropin", "dropin", "dropin", "session", "session", "refine",
                       "batch", "cdt", "cdt", "check", "mlp"])
    if kind == "mlp":
        return dict(kind="mlp", n=_log_int(rng, 3000, 400_000))
    base = rng.randint(100, 1_000_000)
    if kind == "batch":
        return dict(kind="batch", k=rng.randint(2, 16), nmax=_log_int(rng, 500, 30_000), base=base)
    if kind == "cdt":
        return dict(kind="cdt", n=_log_int(rng, 300, 500_000), dist=rng.choice([0, 1, 3]),
                    base=base)
    c = dict(kind=kind, dist=rng.choice([0, 0, 1, 3, 4, 5]), base=base,
             theta=round(rng.uniform(20.0, 30.0), 2), offcenter=rng.choice([0, 1, 1]),
             ruppert=rng.choice([0, 1, 1]))
    if kind == "dropin":
        c["n"] = _log_int(rng, 200, 300_000)
    elif kind == "session":
        c["form"] = rng.choice(["plain", "graph", "chosen"])
        c["n"] = _log_int(rng, 500, 150_000 if c["form"] != "graph" else 60_000)
    elif kind == "refine":
        c["n"] = _log_int(rng, 300, 30_000)
        c["dist"] = rng.choice([0, 1, 2])
    else:
        c["n"] = _log_int(rng, 500, 12_000)
    return c


def _unit(seed):
    """2^-6 .. 2^6: single-precision products of six lengths stay in range."""
    return 2.0 ** (int(seed) % 13 - 6)


def _pslg(n, dist, base, seed):
    """Points and about n / 20 segments (n / 50 along lattice lines for the
    precision-stress family) of at most 20 point spacings."""
    nseg = max(1, n // (50 if dist == 2 else 20))
    P, S = g.generate_pslg(n, nseg, L=SPACING * n ** 0.5, maxlen=20.0 * SPACING, dist=dist,
                           min_angle=5.0, seed=base)
    return P * _unit(seed), S


def _cdt(n, dist, base, seed):
    P, S = _pslg(n, dist, base, seed)
    T, N, SS = g.build_cdt(P, S)
    return P, T, N, SS


def _batch_sizes(case):
    k = case["k"]
    return np.exp(np.log(200) + (np.arange(k) + 0.5) / k * np.log(case["nmax"] / 200)).astype(int)


def _chosen(**over):
    o = dict(g.CHOSEN_FORM)
    o.update(over)
    return o


def _form(name):
    if name == "plain":  # the library's defaults
        return {}
    if name == "graph":  # the device-driven loop; the hand-over below needs the host loop
        return _chosen(graph=1, mix_below=0, graph_rounds=1, graph_seg_passes=3)
    return _chosen()


def _session(case, mesh, form):
    s = g.Session(*mesh, theta=case["theta"], insert=case["offcenter"], mode=case["ruppert"],
                  **_form(form))
    if form != "plain":
        s.set_priority_model(np.load(MODEL))
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        # features in the ranges the cavity kernel writes them, targets
        # log2(1 + conflict degree)
        rng = np.random.default_rng(int(seed) + 1)
        n = case["n"]
        X = np.zeros((n, g.MLP_IN), np.float32)
        X[:, 0] = rng.uniform(0.0, 0.5, n)
        X[:, 1] = rng.gamma(2.0, 0.15, n)
        X[:, 2] = rng.poisson(4.0, n) / 16.0
        X[:, 3] = X[:, 2] + 2 / 16.0
        X[:, 4] = np.minimum(rng.exponential(0.5, n), 1.0)
        X[:, 5] = rng.integers(0, 80, n) / 256.0
        X[:, 7] = 1.0
        t = np.log2(1.0 + rng.poisson(3.0 + 20.0 * X[:, 2])).astype(np.float32)
        return dict(kind=kind, X=X, t=t, params=g.mlp_init(int(seed) + 1))
    base = case["base"]
    if kind == "cdt":
        P, S = _pslg(case["n"], case["dist"], base, seed)
        order = np.random.default_rng(int(seed) + 1).permutation(len(P)).astype(np.int32)
        Q = np.empty_like(P)
        Q[order] = P  # point i is called order[i]
        return dict(kind=kind, P=Q, S=order[S])
    if kind == "batch":
        k = case["k"]
        rng = np.random.default_rng(base)
        ins = [_cdt(int(n), i % 2, base + 17 * i, seed) for i, n in enumerate(_batch_sizes(case))]
        b = g.Batch(ins, theta=20.7 + 9.3 * rng.permutation(k) / k, insert=1,
                    mode=rng.integers(0, 2, k), **_chosen())
        b.set_priority_model(np.load(MODEL))
        return dict(kind=kind, batch=b)
    mesh = _cdt(case["n"], case["dist"], base, seed)
    kw = dict(theta=case["theta"], insert=case["offcenter"], mode=case["ruppert"])
    if kind == "session":
        return dict(kind=kind, session=_session(case, mesh, case["form"]))
    if kind == "check":
        r, _ = g.dropin_refine(*mesh, **kw)
        arrays = [r.points, r.triangles, r.neighbors, r.segments, mesh[0], mesh[3]]
        return dict(kind=kind, mesh=[torch.from_numpy(a).cuda() for a in arrays],
                    theta=case["theta"] + 0.5 + 0.1 * (int(seed) % 13),
                    out=torch.zeros(13, dtype=torch.int64, device="cuda"))
    return dict(kind=kind, mesh=mesh, kw=kw)


def _mesh(r, status=True):
    out = [r.points, r.triangles, r.neighbors, r.segments]
    return out + [r.pstatus, r.tstatus] if status else out


def run(state):
    kind = state["kind"]
    if kind == "dropin":
        r, _ = g.dropin_refine(*state["mesh"], **state["kw"])
        return _mesh(r, status=False)
    if kind == "session":
        state["session"].run()
        return _mesh(state["session"].download())
    if kind == "refine":
        return _mesh(g.refine(*state["mesh"], **state["kw"], **_chosen(priority=1)))
    if kind == "batch":
        state["batch"].run()
        return [a for r in state["batch"].results() for a in _mesh(r, status=False)]
    if kind == "cdt":
        return list(g.build_cdt(state["P"], state["S"], device=True))
    if kind == "check":
        P, T, N, S, P0, S0 = state["mesh"]
        g.check_mesh_device_noalloc(P.data_ptr(), len(P), T.data_ptr(), N.data_ptr(), len(T),
                                    S.data_ptr(), len(S), P0.data_ptr(), len(P0), S0.data_ptr(),
                                    len(S0), state["theta"], state["out"].data_ptr(),
                                    torch.cuda.current_stream().cuda_stream)
        return state["out"]
    y = g.mlp_forward(state["X"], state["params"])
    grad, loss = g.mlp_grad(state["X"], state["t"], state["params"])
    return [y, grad, loss]


def _triangles_out(n, theta):
    """Output triangles of a refinement, roughly (about 10 per input point at
    25 degrees, 19 at 30, 6 at 20)."""
    return n * 10.3 * np.exp(0.122 * (theta - 25.0))


def _mesh_in_bytes(n):
    return 16 * n + 24 * 2 * n + 8 * (n // 20)


def work(case):
    """Inputs read once and outputs written once: points 16 B, triangles and
    neighbours 24 B, segments 8 B, status bytes.  Predicates and
    constructions are counted as no work: a refinement is not bound by
    arithmetic."""
    kind = case["kind"]
    if kind == "mlp":
        n, p = case["n"], 16 * 64 + 64 + 64 * 64 + 64 + 64 + 1
        fwd = 2 * n * (16 * 64 + 64 * 64 + 64)
        return {"bytes": 4 * (16 * n + n + n + 2 * p), "flops": fwd + 3 * fwd}
    if kind == "cdt":
        n = case["n"]
        return {"bytes": 16 * n + 2 * 8 * (n // 20) + 24 * 2 * n, "flops": 0}
    if kind == "batch":
        n = int(_batch_sizes(case).sum())
        t = float(_triangles_out(n, 25.5))
        return {"bytes": int(_mesh_in_bytes(n) + 24 * t + 16 * t / 2 + 8 * (n // 10)), "flops": 0}
    n = case["n"]
    t = float(_triangles_out(n, case["theta"]))
    if kind == "check":
        return {"bytes": int(24 * t + 16 * t / 2 + 16 * n), "flops": 0}
    status = t + t / 2 if kind in ("session", "refine") else 0
    return {"bytes": int(_mesh_in_bytes(n) + 24 * t + 16 * t / 2 + 8 * (n // 10) + status),
            "flops": 0}


def tolerance(case):
    if case["kind"] != "mlp":
        return "exact"
    # BF16 inputs of every product, FP32 sums in whatever order the blocks
    # and atomics take: the order alone moves a gradient by about 1e-6 of its
    # norm; a hidden activation rounded the other way by about 1e-3.
    return {"rel": 2e-3, "max": 2e-2}


def exact(case, seed):
    """The network in float64 (no BF16 rounding); nothing to compute for
    meshes, whose outputs are indices and correctly placed copies."""
    if case["kind"] != "mlp":
        return None
    s = prepare(case, seed)
    X, t, p = (s[k].astype(np.float64) for k in ("X", "t", "params"))
    n, i, h = len(X), g.MLP_IN, g.MLP_H
    cut = np.cumsum([i * h, h, h * h, h, h])
    W1, b1, W2, b2, W3, b3 = np.split(p, cut)
    W1, W2 = W1.reshape(i, h), W2.reshape(h, h)
    h1 = np.maximum(X @ W1 + b1, 0.0)
    h2 = np.maximum(h1 @ W2 + b2, 0.0)
    y = h2 @ W3 + b3
    e = y - t
    dy = 2.0 * e / n
    d2 = np.outer(dy, W3) * (h2 > 0.0)
    d1 = (d2 @ W2.T) * (h1 > 0.0)
    grad = np.concatenate([(X.T @ d1).ravel(), d1.sum(0), (h1.T @ d2).ravel(), d2.sum(0),
                           h2.T @ dy, [dy.sum()]])
    return [y, grad, float((e * e).mean())]
