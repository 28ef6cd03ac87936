"""GEMM tasks at the lines between the 32 x 32 tiles with a split inner
dimension and the 64 x 64 tiles: a side of 32 or less, leaves of up to 256, inner
dimensions around the 16 and 64 steps of a wavefront's share, empty inner
dimension and sizes below their capacity.  |C - ref| <= (p + 4) u (|A| |B| +
|C0|), the bound of a sum of p products in any order."""
import numpy as np
import pytest

pytest.importorskip("hmat_amd")
import task_records as tr  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("many", [False, True])   # the same products in a launch of 64 x 64 tiles
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_gemm_thin(fp32, ta, tb, many):
    rng = np.random.default_rng(17)
    dt = np.float32 if fp32 else np.float64
    tasks, keep = [], []
    #   capacities m, n, p; actual m, n, p
    for cap, act in [((1, 1, 1), None), ((15, 16, 15), None), ((16, 17, 16), None), ((32, 33, 17), None),
                     ((33, 32, 63), None), ((300, 8, 64), None), ((9, 300, 65), None), ((2049, 8, 256), None),
                     ((64, 65, 128), None), ((98, 97, 129), None), ((256, 256, 256), None),
                     ((257, 256, 40), None), ((256, 40, 257), None), ((31, 31, 1000), None),
                     ((40, 12, 300), (33, 7, 300)), ((60, 60, 30), (17, 33, 0)), ((98, 33, 60), (98, 33, 41)),
                     ((32, 98, 50), (0, 98, 50))]:
        m, n, p = act or cap
        cm, cn, cp = cap
        A = rng.standard_normal((cp, cm) if ta else (cm, cp)).astype(dt).astype(np.float64)
        B = rng.standard_normal((cn, cp) if tb else (cp, cn)).astype(dt).astype(np.float64)
        C0 = rng.standard_normal((cm, cn)).astype(dt).astype(np.float64)
        acc = len(tasks) % 2
        h = [tr.dev(A, fp32), tr.dev(B, fp32), tr.dev(C0, fp32), tr.ints([m]), tr.ints([n]), tr.ints([p])]
        t = tr.FTask()
        t.type, t.mode, t.ta, t.tb, t.alpha = tr.T_GEMM, acc, ta, tb, -0.5
        t.m.s, t.n.s, t.p.s = cap
        if act:
            t.m.d, t.n.d, t.p.d = (x.data_ptr() for x in h[3:])
        t.A, t.B, t.C = (x.data_ptr() for x in h[:3])
        t.lda, t.ldb, t.ldc = A.shape[0], B.shape[0], cm
        tasks.append(t)
        keep.append((A.T if ta else A, B.T if tb else B, C0, acc, h, (m, n, p)))
    if many:
        # C (2112 x 2048) = y (2112 x 1) y[:2048]^T: 33 x 32 tiles of 64 x 64
        x, y = tr.dev(np.zeros((2112, 2048)), fp32), tr.dev(np.zeros((2112, 1)), fp32)
        t = tr.FTask()
        t.type, t.alpha, t.tb, t.m.s, t.n.s, t.p.s = tr.T_GEMM, 1.0, 1, 2112, 2048, 1
        t.A, t.B, t.C, t.lda, t.ldb, t.ldc = y.data_ptr(), y.data_ptr(), x.data_ptr(), 2112, 2112, 2112
        tasks.append(t)
    print(f"gemm thin fp32={fp32} ta={ta} tb={tb}", flush=True)
    assert tr.run(tasks, tr.T_GEMM, fp32) == [0, 0]
    u = 2.0 ** -24 if fp32 else 2.0 ** -53
    for A, B, C0, acc, h, (m, n, p) in keep:
        got = tr.host(h[2])
        want = C0.copy()
        want[:m, :n] = acc * C0[:m, :n] - 0.5 * A[:m, :p] @ B[:p, :n]
        bound = np.zeros_like(C0)
        bound[:m, :n] = (p + 4) * u * (np.abs(A[:m, :p]) @ np.abs(B[:p, :n]) + np.abs(C0[:m, :n]))
        assert (np.abs(got - want) <= bound).all(), (A.shape, B.shape, (m, n, p))
