"""Core SVD of the recompressions on one wavefront (FADD and RKRK) at the edges
of its register forms (16, 24 and 32 columns) and above, with cores that
are rectangular, rank deficient, zero or of one column, against numpy's
truncated SVD.  The singular values fall by 0.6 a step, so the cut at eps has a
relative gap of 0.4 and the truncated matrix moves by a few K u / 0.4 of its
norm (K <= 40, u = 2^-53: below 1e-12; 1e-11 asked).  In FP32 the operands are
rounded first and the result carries the rounding of its panels and the 3e-7
that the Gram form leaves out: 1e-5, as in the other tests of these kernels."""
import numpy as np
import pytest

pytest.importorskip("hmat_amd")
import task_records as tr  # noqa: E402

pytestmark = pytest.mark.gpu
EPS = 1e-4


def _rk(rng, m, n, k, fp32):
    a = np.linalg.qr(rng.standard_normal((m, k)))[0] * 0.6 ** np.arange(k)
    b = np.linalg.qr(rng.standard_normal((n, k)))[0]
    dt = np.float32 if fp32 else np.float64
    return a.astype(dt).astype(np.float64), b.astype(dt).astype(np.float64)


def _check(got, S, fp32, what):
    u, s, vt = np.linalg.svd(S, full_matrices=False)
    k = got[0].shape[1]
    if s[0] == 0.0:
        assert k == 0, what
        return
    kw = tr.find_k(s, EPS)
    want = (u[:, :kw] * s[:kw]) @ vt[:kw]
    R = got[0] @ got[1].T
    if not fp32:
        assert k == kw and np.linalg.norm(R - want) <= 1e-11 * s[0], what
    else:
        assert abs(k - kw) <= 1, what
        assert np.linalg.norm(S - R) <= 2 * np.linalg.norm(S - want) + 1e-5 * s[0], what


@pytest.mark.parametrize("fp32", [False, True])
def test_fadd_core_sizes(fp32):
    rng = np.random.default_rng(11)
    tasks, keep = [], []
    #   m, n, rank of the target, of the part, kind
    for m, n, kt, kp, kind in [(70, 90, 1, 1, "full"), (70, 90, 2, 1, "full"), (70, 90, 7, 8, "full"),
                               (99, 65, 8, 8, "full"), (99, 65, 8, 9, "full"), (99, 65, 12, 12, "full"),
                               (99, 65, 12, 13, "full"), (99, 65, 16, 15, "full"), (130, 140, 16, 16, "full"),
                               (130, 140, 16, 17, "full"), (130, 140, 20, 20, "full"), (700, 900, 9, 8, "full"),
                               (700, 900, 16, 16, "full"), (900, 800, 18, 21, "full"), (130, 140, 20, 21, "full"), (70, 90, 6, 6, "same"), (700, 900, 14, 14, "same"),
                               (70, 90, 5, 5, "zero")]:
        ta, tb = _rk(rng, m, n, kt, fp32)
        pa, pb = _rk(rng, m, n, kp, fp32)
        if kind == "same":     # every column twice: half the core's rank
            pa, pb = ta.copy(), tb.copy()
        if kind == "zero":
            ta[:], pa[:] = 0.0, 0.0
        cap = min(m, n, kt + kp)
        TA, TB = np.zeros((m, cap)), np.zeros((n, cap))
        TA[:, :kt], TB[:, :kt] = ta, tb
        h = [tr.dev(TA, fp32), tr.dev(TB, fp32), tr.ints([kt]), tr.dev(pa, fp32), tr.dev(pb, fp32), tr.ints([kp])]
        t = tr.FTask()
        t.type, t.eps, t.nparts = tr.T_FADD, EPS, 1
        t.tgt = tr.rkref(h[0], h[1], m, n, cap, h[2])
        t.parts[0].rk = tr.rkref(h[3], h[4], m, n, kp, h[5])
        t.parts[0].alpha = 0.5
        tasks.append(t)
        keep.append((ta @ tb.T + 0.5 * pa @ pb.T, h, (m, n, kt, kp, kind)))
    print(f"core SVD fadd fp32={fp32}", flush=True)
    assert tr.run(tasks, tr.T_FADD, fp32) == [0, 0]
    for S, h, what in keep:
        k = int(h[2].cpu().numpy()[0])
        _check((tr.host(h[0])[:, :k], tr.host(h[1])[:, :k]), S, fp32, what)


@pytest.mark.parametrize("fp32", [False, True])
def test_rkrk_core_sizes(fp32):
    rng = np.random.default_rng(12)
    tasks, keep = [], []
    m, p, n = 60, 45, 50
    for k1, k2 in [(1, 1), (1, 32), (32, 1), (2, 3), (5, 30), (30, 5), (16, 16), (16, 17), (17, 16), (24, 24),
                   (25, 24), (31, 32), (32, 32), (33, 32), (32, 33), (40, 40)]:
        a1, b1 = _rk(rng, m, p, k1, fp32)
        b2, a2 = _rk(rng, n, p, k2, fp32)
        # the left factor's decay sits in a1, the right one's in b2: both panels of the core
        # are orthonormal, so weigh the core itself
        b1 = (b1 * 0.6 ** np.arange(k1)).astype(np.float32 if fp32 else np.float64).astype(np.float64)
        cap = min(k1, k2)
        h = [tr.dev(a1, fp32), tr.dev(b1, fp32), tr.dev(a2, fp32), tr.dev(b2, fp32),
             tr.dev(np.zeros((m, cap)), fp32), tr.dev(np.zeros((n, cap)), fp32),
             tr.ints([k1]), tr.ints([k2]), tr.ints([0])]
        t = tr.FTask()
        t.type, t.eps = tr.T_RKRK, EPS
        t.parts[0].rk = tr.rkref(h[0], h[1], m, p, k1, h[6])
        t.parts[1].rk = tr.rkref(h[2], h[3], p, n, k2, h[7])
        t.tgt = tr.rkref(h[4], h[5], m, n, cap, h[8])
        tasks.append(t)
        u, s, vt = np.linalg.svd(b1.T @ a2)
        kw = tr.find_k(s, EPS)
        keep.append((a1 @ (u[:, :kw] * s[:kw]) @ vt[:kw] @ b2.T, kw, s, h, (k1, k2)))
    print(f"core SVD rkrk fp32={fp32}", flush=True)
    assert tr.run(tasks, tr.T_RKRK, fp32) == [0, 0]
    for want, kw, s, h, what in keep:
        k = int(h[8].cpu().numpy()[0])
        got = tr.host(h[4])[:, :k] @ tr.host(h[5])[:, :k].T
        assert abs(k - kw) <= (1 if fp32 else 0), (what, k, kw)
        # the outer panels have norm 1: a change of the core's cut moves the result by as much;
        # one rank more or less at the cut is eps s[0]
        tol = (1e-5 if k == kw else EPS) if fp32 else 1e-11
        assert np.linalg.norm(got - want) <= tol * s[0], what


@pytest.mark.parametrize("eps", [1e-6, 1e-7])
def test_fadd_fp32_tight_eps(eps):
    """FP32 sums of more than 32 columns at cuts near the panels' rounding.  The
    recompression works in FP64, so the distance to the exact sum is that of the
    cut, at most sqrt(K) eps s[0], and the rounding of the new panels A, B
    (2^-24 each of entries whose products sum to |A| |B^T|, whose norm is at
    most the sum of the singular values)."""
    rng = np.random.default_rng(13)
    tasks, keep = [], []
    for m, n, kt, kp in [(130, 140, 16, 17), (130, 140, 18, 18), (70, 90, 20, 20), (700, 900, 20, 20),
                         (130, 140, 20, 21)]:
        K = kt + kp

        def panels(k):
            a = np.linalg.qr(rng.standard_normal((m, k)))[0] * 10.0 ** (-8.0 * np.arange(k) / k)
            b = np.linalg.qr(rng.standard_normal((n, k)))[0]
            return a.astype(np.float32).astype(np.float64), b.astype(np.float32).astype(np.float64)
        (ta, tb), (pa, pb) = panels(kt), panels(kp)
        TA, TB = np.zeros((m, K)), np.zeros((n, K))
        TA[:, :kt], TB[:, :kt] = ta, tb
        h = [tr.dev(TA, True), tr.dev(TB, True), tr.ints([kt]), tr.dev(pa, True), tr.dev(pb, True), tr.ints([kp])]
        t = tr.FTask()
        t.type, t.eps, t.nparts = tr.T_FADD, eps, 1
        t.tgt = tr.rkref(h[0], h[1], m, n, K, h[2])
        t.parts[0].rk = tr.rkref(h[3], h[4], m, n, kp, h[5])
        t.parts[0].alpha = 0.5
        tasks.append(t)
        keep.append((ta @ tb.T + 0.5 * pa @ pb.T, h, (m, n, kt, kp)))
    assert tr.run(tasks, tr.T_FADD, True) == [0, 0]
    for S, h, what in keep:
        k = int(h[2].cpu().numpy()[0])
        R = tr.host(h[0])[:, :k] @ tr.host(h[1])[:, :k].T
        s = np.linalg.svd(S, compute_uv=False)
        kw = tr.find_k(s, eps)
        err, cut = np.linalg.norm(S - R), np.linalg.norm(s[kw:])
        print(f"fp32 eps={eps} {what}: rank {k} of {kw}, error {err / s[0]:.2e}, cut {cut / s[0]:.2e}", flush=True)
        assert abs(k - kw) <= 1, (what, k, kw)
        assert err <= 1.01 * max(cut, eps * s[0]) + 2 * 2.0 ** -24 * s.sum(), what
