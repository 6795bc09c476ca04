"""shk_solve_csr's one-launch Jacobi CG (csrc/resident.hip) at the edges of its launch shape: one
row, a started second workgroup (512 rows), two and three rows per thread, rows of eight
and of nine entries (the latter take the two-kernel solve), and rows that no longer fit.

Both solves stop with max|b - A x| <= tol max|b| in FP64, so max|A (x1 - x2)| <= 2 tol max|b|
up to the rounding of the recurrence; ProfileKernels=1 runs the two-kernel solve."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(n, band, seed):
    """SPD: unit chain plus `band` random long couplings, strictly diagonally dominant."""
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    A = sp.diags([-rng.random(max(n - 1, 0))], [1], shape=(n, n)).tolil() if n > 1 else sp.lil_matrix((n, n))
    A = A.tocsr()
    for k in range(band):
        off = int(rng.integers(2, max(3, n // 2))) + k
        if off < n:
            A = A + sp.diags([-rng.random(n - off)], [off], shape=(n, n))
    A = A + A.T
    A = sp.csr_matrix(A)
    d = np.asarray(abs(A).sum(axis=1)).ravel() + 0.02 + 0.05 * rng.random(n)
    A = sp.csr_matrix(A + sp.diags([d], [0]))
    A.sort_indices()
    return A, rng.standard_normal(n)


@pytest.mark.parametrize("n,band", [(1, 0), (2, 0), (511, 1), (513, 2), (5000, 3), (140000, 2), (263000, 2),
                                    (5000, 4), (400000, 1)])
def test_csr_resident(n, band):
    import torch
    import shiokaze_amd as shk
    A, b = _system(n, band, n + band)
    dev = [torch.from_numpy(a).cuda() for a in (A.indptr.astype(np.int64), A.indices.astype(np.int64), A.data, b)]
    tol = 1e-8
    s = shk.PCGSolver(config={"Preconditioner": "jacobi", "Residual": tol})
    xs, its = [], []
    for profile in (0, 1):
        s.configure("ProfileKernels", profile)
        x, r = s.solve(*dev)
        assert r["status"] == 0
        x = x.cpu().numpy()
        assert np.abs(b - A @ x).max() <= tol * np.abs(b).max() * (1 + 1e-4)
        xs.append(x)
        its.append(r["count"])
    assert abs(its[0] - its[1]) <= 2
    s.configure("ProfileKernels", 0)
    assert np.array_equal(s.solve(*dev)[0].cpu().numpy(), xs[0])   # one order of summation
    s.configure("MaxIterations", 3)
    assert s.solve(*dev)[1]["count"] == min(3, its[0])
    z, r = s.solve(*dev[:3], torch.zeros_like(dev[3]))
    assert r["status"] == 0 and r["count"] == 0 and not z.any()
    s.close()


@pytest.mark.parametrize("rowptr", [(-8, -4, -1), (-3, -2, -1), (5, 3, -1)])
def test_rowptr_below_zero_is_refused(rowptr):
    """Rows of few entries whose rowptr ends below 0: refused before a kernel follows it."""
    import torch
    import shiokaze_amd as shk
    s = shk.PCGSolver(config={"Preconditioner": "jacobi"})
    dev = (torch.tensor(rowptr, device="cuda"), torch.zeros(8, dtype=torch.int64, device="cuda"),
           torch.ones(8, dtype=torch.float64, device="cuda"), torch.ones(2, dtype=torch.float64, device="cuda"))
    with pytest.raises(shk.ShkError, match="rowptr"):
        s.solve(*dev)
    s.close()
