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
