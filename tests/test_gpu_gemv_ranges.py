"""The H-gemv at the edges of its plan: destination ranges of 1 to 512 rows (the
kernels take 128 at a time), column runs of 32, right-hand sides around the
16 and 32 of a matrix-core tile, panels of several 1,024-row chunks, both
storages, FP32 and complex matrices, alpha and beta.

Reference: the product with the stored leaves (to_dense) in FP64.  Both sides
round each of at most N products and sums: 4 N u relative to |A| |x| (FP32:
the stored entries are the same, the result is rounded to 32 bits)."""
import numpy as np
import pytest

hmat_amd = pytest.importorskip("hmat_amd")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,leaf,sym,vt,height", [
    (5, 8, True, hmat_amd.HMAT_DOUBLE_PRECISION, 1.0), (700, 33, True, hmat_amd.HMAT_DOUBLE_PRECISION, 0.5),
    (1290, 129, True, hmat_amd.HMAT_DOUBLE_PRECISION, 4.0), (2001, 260, True, hmat_amd.HMAT_DOUBLE_PRECISION, 8.0),
    (1777, 500, False, hmat_amd.HMAT_DOUBLE_PRECISION, 6.0), (1500, 65, False, hmat_amd.HMAT_SIMPLE_PRECISION, 3.0),
    (901, 150, True, hmat_amd.HMAT_SIMPLE_PRECISION, 3.0), (600, 90, False, hmat_amd.HMAT_DOUBLE_COMPLEX, 2.0),
    (5200, 128, True, hmat_amd.HMAT_DOUBLE_PRECISION, 30.0)])
def test_gemv_ranges(n, leaf, sym, vt, height):
    import torch
    rng = np.random.default_rng(n)
    th = 2 * np.pi * rng.random(n)
    pts = np.column_stack([np.cos(th), np.sin(th), height * rng.random(n)])
    h = hmat_amd.HMatrix(hmat_amd.ClusterTree(pts, leaf), lower_symmetric=sym, value_type=vt)
    if vt == hmat_amd.HMAT_DOUBLE_COMPLEX:
        h.assemble(kind=hmat_amd.KERNEL_HELMHOLTZ, wavenumber=2.0, reg=0.05, nugget=1.0)
        A = h.to_dense(embedded=True)
        wide = 2
    else:
        h.assemble(kind=hmat_amd.KERNEL_EXPONENTIAL if sym else hmat_amd.KERNEL_SHIFTED_EXPONENTIAL, shift=0.1)
        A = h.to_dense(precision=1 if vt == hmat_amd.HMAT_SIMPLE_PRECISION else 0)
        wide = 1
    f32 = vt == hmat_amd.HMAT_SIMPLE_PRECISION
    dt = torch.float32 if f32 else torch.float64
    N = n * wide
    for nrhs in (1, 2, 16, 17, 33):
        x = torch.tensor(rng.standard_normal((nrhs, N)), dtype=dt, device="cuda")
        y0 = torch.tensor(rng.standard_normal((nrhs, N)), dtype=dt, device="cuda")
        y = y0.clone()
        torch.cuda.synchronize()
        h.gemv_device(x.data_ptr(), y.data_ptr(), nrhs, alpha=0.75, beta=-0.5, precision=1 if f32 else 0)
        torch.cuda.synchronize()
        X, Y0 = x.double().cpu().numpy().T, y0.double().cpu().numpy().T
        want = 0.75 * (A @ X) - 0.5 * Y0
        bound = 4 * N * 2.0 ** -53 * (np.abs(A) @ np.abs(X) + np.abs(Y0)) + (2.0 ** -23 * np.abs(want) if f32 else 0.0)
        assert (np.abs(y.double().cpu().numpy().T - want) <= bound).all(), nrhs
    print(f"gemv ranges n={n} leaf={leaf}", flush=True)
    h.close()


@pytest.mark.parametrize("rows,cols", [(1500, 200), (200, 1500), (130, 129), (700, 110)])
def test_gemv_two_trees(rows, cols):
    """Different row and column trees: x ends at the last column, whatever the
    rows (a row's position is no position of x)."""
    import ctypes as C
    import torch
    rng = np.random.default_rng(rows)
    P, Q = rng.random((rows, 3)) * [1, 1, 6], rng.random((cols, 3)) * [1, 1, 6]
    tr, tc = hmat_amd.ClusterTree(P, 100), hmat_amd.ClusterTree(Q, 100)

    @hmat_amd.PREPARE_FUNC
    def prepare(r0, rc, c0, cc, rows_h2c, rows_c2h, cols_h2c, cols_c2h, ctx, info):
        blocks[len(blocks) + 1] = (np.array(rows_h2c[r0:r0 + rc]), np.array(cols_h2c[c0:c0 + cc]))
        info[0].user_data = len(blocks)

    @hmat_amd.COMPUTE_FUNC
    def compute(data, r0, rc, c0, cc, out):
        ri, ci = blocks[data]
        d = P[ri[r0:r0 + rc]][:, None] - Q[ci[c0:c0 + cc]][None]
        np.ctypeslib.as_array(C.cast(out, C.POINTER(C.c_double)), shape=(cc, rc))[:] = \
            np.exp(-np.sqrt((d * d).sum(axis=2))).T

    blocks = {}
    h = hmat_amd.HMatrix(tr, lower_symmetric=False)
    h.close()
    lib = hmat_amd.load()
    adm = lib.hmat_create_admissibility_standard(2.0)
    h.handle = h.iface.create_empty_hmatrix_admissibility(tr.handle, tc.handle, 0, adm)
    lib.hmat_delete_admissibility(adm)
    h.iface.set_low_rank_epsilon(h.handle, 1e-4)
    h.assemble_functions(block=compute, prepare=prepare)
    A = np.zeros((rows, cols))
    for m, n, r0, c0, kind, rank, a, b in h.leaves():
        A[r0:r0 + m, c0:c0 + n] = a if kind == 0 else a @ b.T
    print(f"gemv two trees {rows} x {cols}", flush=True)
    for nrhs in (1, 2):
        X, Y = rng.standard_normal((cols, nrhs)), rng.standard_normal((rows, nrhs))
        want = 0.75 * (A @ X) - 0.5 * Y
        bound = 4 * (rows + cols) * 2.0 ** -53 * (np.abs(A) @ np.abs(X) + np.abs(Y))
        x, y = torch.tensor(X.T.copy(), device="cuda"), torch.tensor(Y.T.copy(), device="cuda")
        torch.cuda.synchronize()
        h.gemv_device(x.data_ptr(), y.data_ptr(), nrhs, alpha=0.75, beta=-0.5)
        assert (np.abs(y.cpu().numpy().T - want) <= bound).all()
        x, y = np.asfortranarray(X[np.argsort(tc.indices)]), np.asfortranarray(Y[np.argsort(tr.indices)])
        al, be = C.c_double(0.75), C.c_double(-0.5)
        assert h.iface.gemv(b"N", C.cast(C.byref(al), C.c_void_p), h.handle, x.ctypes.data,
                            C.cast(C.byref(be), C.c_void_p), y.ctypes.data, nrhs) == 0
        assert (np.abs(y[tr.indices] - want) <= bound).all()
    h.close()


def test_gemv_more_right_hand_sides_than_a_grid_has_rows():
    import torch
    n, nrhs = 60, 70001
    h = hmat_amd.HMatrix(hmat_amd.ClusterTree(np.random.default_rng(1).random((n, 3)), 16))
    h.assemble()
    A = h.to_dense()
    x = torch.randn(nrhs, n, dtype=torch.float64, device="cuda")
    y0 = torch.randn(nrhs, n, dtype=torch.float64, device="cuda")
    y = y0.clone()
    torch.cuda.synchronize()
    h.gemv_device(x.data_ptr(), y.data_ptr(), nrhs, alpha=2.0, beta=1.0)
    X, Y = x.cpu().numpy(), y0.cpu().numpy()
    bound = 4 * n * 2.0 ** -53 * (np.abs(X) @ (2.0 * np.abs(A)) + np.abs(Y))
    assert (np.abs(y.cpu().numpy() - (2.0 * (X @ A) + Y)) <= bound).all()
    h.close()
