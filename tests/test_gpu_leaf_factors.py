"""POTRF and GETRF leaves at the edges of their 16-column panels and of the two
rows per lane, up to the 128 rows of the LDS form and beyond, in both
precisions: backward error |A - L L^T| <= c n u |L| |L^T| (c = 8: 16-term
panels and FP64 sums in another order; + the rounding of 32-bit storage), the
pivots of LAPACK's getrf exactly, equal magnitudes included (the first row
wins), and failing pivots reported."""
import numpy as np
import pytest
import scipy.linalg as sl

pytest.importorskip("hmat_amd")
import task_records as tr  # noqa: E402

pytestmark = pytest.mark.gpu
SIZES = (1, 2, 15, 16, 17, 31, 33, 63, 64, 65, 79, 97, 112, 113, 125, 127, 128, 129)


def _run(typ, mats, fp32, piv=None):
    dev = [tr.dev(a, fp32) for a in mats]
    tasks = []
    for q, (a, d) in enumerate(zip(mats, dev)):
        t = tr.FTask()
        t.type, t.m.s, t.A, t.lda = typ, len(a), d.data_ptr(), len(a)
        if piv is not None:
            t.B = piv[q].data_ptr()
        tasks.append(t)
    return dev, tr.run(tasks, typ, fp32)


@pytest.mark.parametrize("fp32", [False, True])
def test_potrf_sizes(fp32):
    rng = np.random.default_rng(5)
    dt = np.float32 if fp32 else np.float64
    mats = []
    for n in SIZES:
        g = rng.standard_normal((n, n))
        mats.append((g @ g.T / n + 0.1 * np.eye(n)).astype(dt).astype(np.float64))
    mats = [np.tril(a) + np.tril(a, -1).T for a in mats]
    dev, flags = _run(tr.T_POTRF, mats, fp32)
    assert flags == [0, 0]
    print(f"potrf sizes fp32={fp32}", flush=True)
    for a, d in zip(mats, dev):
        n, L = len(a), tr.host(d)
        assert np.array_equal(np.triu(L, 1), np.zeros((n, n)))
        u = 8 * n * (2.0 ** -24 if fp32 else 2.0 ** -53)
        assert (np.abs(L @ L.T - a) <= u * (np.abs(L) @ np.abs(L.T))).all(), n
    bad = mats[12].copy()
    bad[97, 97] = -1.0
    assert _run(tr.T_POTRF, [mats[3], bad], fp32)[1][1] != 0


@pytest.mark.parametrize("fp32", [False, True])
def test_getrf_sizes(fp32):
    rng = np.random.default_rng(6)
    dt = np.float32 if fp32 else np.float64
    mats = [rng.standard_normal((n, n)).astype(dt).astype(np.float64) for n in SIZES]
    # equal magnitudes in every column: entries +-1 on a dominant permutation
    for n in (16, 40, 100):
        mats.append(np.where(rng.random((n, n)) < 0.5, -1.0, 1.0) + 0.0)
    keep = [m for m in mats if abs(np.linalg.det(m / np.abs(m).max())) > 0 and np.linalg.cond(m) < 1e5]
    piv = [tr.ints(np.full(len(a), -1)) for a in keep]
    dev, flags = _run(tr.T_GETRF, keep, fp32, piv)
    assert flags == [0, 0]
    print(f"getrf sizes fp32={fp32}: {len(keep)}", flush=True)
    for a, d, p in zip(keep, dev, piv):
        n, F = len(a), tr.host(d)
        L, U = np.tril(F, -1) + np.eye(n), np.triu(F)
        pv = p.cpu().numpy()
        if set(np.unique(np.abs(a))) != {1.0}:
            assert np.array_equal(pv, sl.lapack.dgetrf(a)[1])
        else:
            assert pv[0] == 0  # all of the first column is equal: the first row
        B = a.copy()
        for i, q in enumerate(pv):
            B[[i, q]] = B[[q, i]]
        u = 8 * n * (2.0 ** -24 if fp32 else 2.0 ** -53)
        assert (np.abs(L @ U - B) <= u * (np.abs(L) @ np.abs(U))).all(), n
    sing = keep[9].copy()
    sing[:, 20] = 0.0
    assert _run(tr.T_GETRF, [keep[3], sing], fp32, [tr.ints(np.zeros(128)), tr.ints(np.zeros(128))])[1][1] != 0


def test_pivots_below_the_reciprocals_range():
    """Pivots whose reciprocal overflows (FP64): zeros below them stay zeros, and
    the quotients of entries of their size are those of the same leaf scaled up.
    The other columns do not see them (their rows of L or U are zero or of
    1e-310), so the bounds are those of the sizes test."""
    rng = np.random.default_rng(8)
    tiny = 3.0 * 2.0 ** -1030
    for n in (17, 40, 100):
        g = rng.standard_normal((n, n))
        spd = g @ g.T / n + 0.1 * np.eye(n)
        j = n // 2
        spd[j, :], spd[:, j] = 0.0, 0.0
        spd[j, j] = tiny
        dev, flags = _run(tr.T_POTRF, [spd], False)
        L = tr.host(dev[0])
        assert flags == [0, 0] and np.isfinite(L).all() and abs(L[j, j] - tiny ** 0.5) <= 1e-15 * tiny ** 0.5
        assert (np.abs(L @ L.T - spd) <= 8 * n * 2.0 ** -53 * (np.abs(L) @ np.abs(L.T)) + 2.0 ** -1074).all(), n
        lu = rng.standard_normal((n, n))
        lu[:, j] = 0.0
        lu[j, :] = 0.0
        lu[j, j] = tiny
        piv = [tr.ints(np.full(n, -1))]
        dev, flags = _run(tr.T_GETRF, [lu], False, piv)
        F = tr.host(dev[0])
        want, pv, info = sl.lapack.dgetrf(lu)
        assert flags == [0, 0] and info == 0 and np.isfinite(F).all()
        assert np.array_equal(piv[0].cpu().numpy(), pv)
        L, U = np.tril(F, -1) + np.eye(n), np.triu(F)
        B = lu.copy()
        for i, q in enumerate(pv):
            B[[i, q]] = B[[q, i]]
        assert (np.abs(L @ U - B) <= 8 * n * 2.0 ** -53 * (np.abs(L) @ np.abs(U)) + 2.0 ** -1074).all(), n
    # a leaf that is tiny throughout: powers of two (no entry is rounded on the
    # way), LU of the scaled leaf
    n = 24
    a = np.tril(2.0 ** rng.integers(-3, 0, (n, n)), -1) * np.where(rng.random((n, n)) < 0.5, -1.0, 1.0)
    a = np.where(rng.random((n, n)) < 0.8, 0.0, a) + np.eye(n)
    piv = [tr.ints(np.full(n, -1))]
    dev, flags = _run(tr.T_GETRF, [a * 2.0 ** -1040], False, piv)
    want = sl.lapack.dgetrf(a)[0]
    assert flags == [0, 0] and np.array_equal(np.tril(tr.host(dev[0]), -1), np.tril(want, -1))
