"""The truncated SVD of admissible leaves below 100 rows and columns against
LAPACK's, at the sizes around which the kernel changes its form (52 rows, 99
rows, rectangular blocks either way) and at loose and tight cuts, blocks of
zeros included.

Bound: the kernel's factors are those of a matrix within c u ||G|| of G
(c = 1,000 for the reductions of 100-row columns); a cut between sigma_k and
sigma_{k+1} turns that into c u ||G|| (1 + sigma_k / (sigma_k - sigma_{k+1}))."""
import numpy as np
import pytest

hmat_amd = pytest.importorskip("hmat_amd")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,leaf,eps,kind,length", [
    (4 * 99, 99, 1e-4, hmat_amd.KERNEL_EXPONENTIAL, 0.5), (4 * 53 - 1, 53, 1e-4, hmat_amd.KERNEL_EXPONENTIAL, 0.5),
    (4 * 52, 52, 1e-10, hmat_amd.KERNEL_GAUSSIAN, 1.0), (4 * 98 - 3, 98, 1e-10, hmat_amd.KERNEL_GAUSSIAN, 2.0),
    (8 * 17, 17, 1e-4, hmat_amd.KERNEL_EXPONENTIAL, 0.5), (8 * 3, 3, 1e-2, hmat_amd.KERNEL_EXPONENTIAL, 0.5),
    (4 * 70, 70, 1e-4, hmat_amd.KERNEL_GAUSSIAN, 0.01)])
def test_svd_leaves(n, leaf, eps, kind, length):
    rng = np.random.default_rng(n)
    pts = np.column_stack([rng.random(n), rng.random(n), 12.0 * rng.random(n)])
    tree = hmat_amd.ClusterTree(pts, leaf)
    P = pts[tree.indices]
    h = hmat_amd.HMatrix(tree, lower_symmetric=False, lowrank_eps=eps)
    h.assemble(kind=kind, length=length, nugget=0.0, eps=eps)
    seen = 0
    for m, k, r0, c0, kd, rank, a, b in h.leaves():
        if kd == 0 or max(m, k) >= 100:
            continue
        seen += 1
        d = np.linalg.norm(P[r0:r0 + m, None, :] - P[None, c0:c0 + k, :], axis=2)
        G = np.exp(-d / length) if kind == hmat_amd.KERNEL_EXPONENTIAL else np.exp(-d * d / length ** 2)
        U, s, Vt = np.linalg.svd(G)
        want = int((s > eps * s[0]).sum()) if s[0] > 0 else 0
        assert rank == want
        nxt = s[want] if want < len(s) else 0.0
        gap = 1.0 + (s[want - 1] / (s[want - 1] - nxt) if want else 0.0)
        T = (U[:, :want] * s[:want]) @ Vt[:want]
        assert np.linalg.norm(a @ b.T - T) <= 1e3 * 2.0 ** -53 * s[0] * gap
    print(f"svd leaves n={n}: {seen} blocks", flush=True)
    assert seen > 0
    h.close()


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_svd_leaves_non_finite(bad):
    """One entry of one block is infinite or NaN (host functions): its column (its row
    in a block with more columns than rows) is left out, the rest of the block and
    every other block stay."""
    import ctypes as C
    n, eps = 197, 1e-6
    rng = np.random.default_rng(3)
    pts = np.column_stack([rng.random(n), rng.random(n), 12.0 * rng.random(n)])
    tree = hmat_amd.ClusterTree(pts, 50)
    P = pts[tree.indices]
    K = np.exp(-np.linalg.norm(P[:, None] - P[None], axis=2) / 2.0)
    h = hmat_amd.HMatrix(tree, lower_symmetric=False, lowrank_eps=eps)
    where = [(r0 + 5, c0 + 7) for m, k, r0, c0, kd in h.leaf_shapes() if kd == 1][:2]
    for at in where:
        K[at] = bad
    pos = np.argsort(tree.indices)

    @hmat_amd.INTERACTION_FUNC
    def entry(ctx, i, j, out):
        C.cast(out, C.POINTER(C.c_double))[0] = K[pos[i], pos[j]]
    h.assemble_functions(simple=entry, eps=eps)
    hit = 0
    for m, k, r0, c0, kd, rank, a, b in h.leaves():
        if kd == 0:
            continue
        G = K[r0:r0 + m, c0:c0 + k].copy()
        if not np.isfinite(G).all():
            hit += 1
            if m >= k:
                G[:, ~np.isfinite(G).all(axis=0)] = 0.0
            else:
                G[~np.isfinite(G).all(axis=1), :] = 0.0
        U, s, Vt = np.linalg.svd(G)
        want = int((s > eps * s[0]).sum())
        T = (U[:, :want] * s[:want]) @ Vt[:want]
        gap = 1.0 + s[want - 1] / (s[want - 1] - s[want])
        assert rank == want
        assert np.linalg.norm(a @ b.T - T) <= 1e3 * 2.0 ** -53 * s[0] * gap
    assert hit == 2
    h.close()
