"""The checker's coverage walk over both of its edge lists against the CPU
checker: the compact one, kept in the edge hash's memory, and the index lists
it falls back to when there are too many subsegments for that memory (here
each of them is listed many times)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("times", [1, 2, 60])
def test_coverage_lists(gpu, oracle, times):
    print(f"coverage lists times={times}", flush=True)
    P, S0 = gpu.generate_pslg(40, 4, L=400.0, maxlen=200.0, dist=0, min_angle=5.0, seed=5)
    T, N, S = gpu.build_cdt(P, S0)
    r = gpu.refine(P, T, N, S, theta=20.0)
    So = np.ascontiguousarray(np.tile(r.segments, (times, 1)))
    # 64 bytes per subsegment against 12 per slot of a hash of 6 slots a triangle
    slots = 1 << max(10, int(np.ceil(np.log2(6 * len(r.triangles) + 16))))
    assert (64 * len(So) > 12 * slots) == (times == 60)
    g = gpu.check_mesh(r.points, r.triangles, r.neighbors, So, points_in=P, segments_in=S,
                       theta=20.0)
    tot, cpu, mina, nex = oracle.check_mesh(r.points, r.triangles, r.neighbors, So, P, S, 20.0)
    assert g["coverage"] == cpu["segment_not_covered"]
    assert g["quality"] == cpu["quality"] and g["exempt"] == nex
    assert abs(g["min_angle"] - mina) < 1e-6
