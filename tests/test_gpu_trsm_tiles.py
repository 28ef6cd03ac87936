"""TRSM tasks at the edges of their tiles and blocks: widths around the 64
columns of a workgroup and the 16 of a wavefront, orders around the 16-row
blocks and the 128 rows solved in registers at a time, row interchanges, and
identity / sum / copy tasks longer than one run of entries.

Backward error: with u the unit roundoff of the arithmetic (FP64) and s that of
the storage, |L X - B| <= (n u c + s) |L| |X| per entry; the blocked form
multiplies by inverted 16 x 16 diagonal blocks, whose condition numbers here
are below 30, so c = 64 covers it."""
import numpy as np
import pytest

pytest.importorskip("hmat_amd")
import task_records as tr  # noqa: E402

pytestmark = pytest.mark.gpu


def _lower(n, rng):
    L = np.tril(rng.standard_normal((n, n)) / np.sqrt(n))
    L[np.arange(n), np.arange(n)] = 1.0 + rng.random(n)
    return L


@pytest.mark.parametrize("fp32", [False, True])
def test_trsm_tiles_and_blocks(fp32):
    rng = np.random.default_rng(17)
    modes = (0, 1, 2, 0 | tr.TRSM_TRANS_A, 2 | tr.TRSM_UNIT, 1 | tr.TRSM_PIV | tr.TRSM_UNIT)
    sizes = ((1, 1), (15, 16), (16, 17), (17, 65), (127, 64), (128, 129), (129, 1), (144, 40), (257, 70), (300, 16))
    dt = np.float32 if fp32 else np.float64
    tasks, keep = [], []
    for mode in modes:
        for n, other in sizes:
            L = _lower(n, rng).astype(dt).astype(np.float64)
            stored = L.T.copy() if mode & tr.TRSM_TRANS_A else L
            X = rng.standard_normal((other, n) if (mode & 3) == 0 else (n, other)).astype(dt).astype(np.float64)
            piv = np.array([rng.integers(i, n) for i in range(n)])
            a_, x_, p_ = tr.dev(stored, fp32), tr.dev(X, fp32), tr.ints(piv)
            t = tr.FTask()
            t.type, t.mode, t.n.s, t.m.s = tr.T_TRSM, mode, n, other
            t.A, t.lda, t.B, t.C, t.ldc = a_.data_ptr(), n, p_.data_ptr(), x_.data_ptr(), X.shape[0]
            tasks.append(t)
            keep.append((mode, L, X, piv, a_, x_, p_))
    print(f"trsm tiles fp32={fp32}: {len(tasks)} tasks", flush=True)
    assert tr.run(tasks, tr.T_TRSM, fp32) == [0, 0]
    for mode, L, B, piv, a_, x_, p_ in keep:
        n = len(L)
        if mode & tr.TRSM_UNIT:
            L = L - np.diag(np.diag(L)) + np.eye(n)
        if mode & tr.TRSM_PIV:
            B = B.copy()
            for i, p in enumerate(piv):
                B[[i, p]] = B[[p, i]]
        X = tr.host(x_)
        if (mode & 3) == 0:
            X, B = X.T, B.T
        M = L.T if (mode & 3) == 2 else L
        bound = (64 * n * 2.0 ** -53 + (2.0 ** -23 if fp32 else 0.0)) * (np.abs(M) @ np.abs(X) + np.abs(B))
        assert (np.abs(M @ X - B) <= bound).all(), (mode, L.shape, X.shape)


def test_elementwise_runs():
    """An identity, a sum of slices and a transposing copy of more entries than
    one workgroup's run: every entry is written once, exactly."""
    import torch
    n = 150
    eye = torch.full((n, n), 7.0, dtype=torch.float64, device="cuda")
    z = tr.FTask()
    z.type, z.mode, z.m.s, z.n.s, z.C, z.ldc = tr.T_ZERO, 1, n, n, eye.data_ptr(), n
    assert tr.run([z], tr.T_ZERO) == [0, 0]
    assert torch.equal(eye.cpu(), torch.eye(n, dtype=torch.float64))
    m, c, s = 311, 33, 9
    w = torch.arange(m * c * s, dtype=torch.float64, device="cuda").reshape(s, c, m)
    out = torch.ones(c, m, dtype=torch.float64, device="cuda")
    k = tr.FTask()
    k.type, k.mode, k.m.s, k.n.s, k.p.s = tr.T_SUMK, 1, m, c, s
    k.A, k.lda, k.ldb, k.C, k.ldc = w.data_ptr(), m, m * c, out.data_ptr(), m
    assert tr.run([k], tr.T_SUMK) == [0, 0]
    assert torch.equal(out, w.sum(dim=0) + 1.0)
    src = torch.randn(m, n, dtype=torch.float64, device="cuda")   # column-major n x m
    dst = torch.zeros(n, m, dtype=torch.float64, device="cuda")   # column-major m x n
    a = tr.FTask()
    a.type, a.mode, a.ta, a.alpha, a.m.s, a.n.s = tr.T_AXPY, 1, 1, 1.0, m, n
    a.A, a.lda, a.C, a.ldc = src.data_ptr(), n, dst.data_ptr(), m
    assert tr.run([a], tr.T_AXPY) == [0, 0]
    assert torch.equal(dst, src.T)
