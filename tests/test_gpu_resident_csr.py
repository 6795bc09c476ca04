"""shk_solve_csr's one-launch Jacobi CG (csrc/resident.hip) at the edges of its launch shape: one
row, a started second workgroup (512 rows), two and three rows per thread (from 131,073 and
262,145 rows on 256 compute units), rows of eight and of nine entries, and the last system
that fits (393,216 rows).  Rows of nine entries and systems beyond that take the two-kernel
solve; shk_kernel_stats' counters say which ran.

Both solves stop with max|b - A x| <= tol max|b| in FP64, so max|A (x1 - x2)| <= 2 tol max|b|
up to the rounding of the recurrence; ProfileKernels=1 runs the two-kernel solve."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(n, band, seed, extra=0):
    """SPD: unit chain plus `band` random long couplings, strictly diagonally dominant; `extra`
    disjoint pairs of rows get one more coupling."""
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    A = sp.diags([-rng.random(max(n - 1, 0))], [1], shape=(n, n)).tolil() if n > 1 else sp.lil_matrix((n, n))
    A = A.tocsr()
    for k in range(band):
        off = int(rng.integers(2, max(3, n // 2))) + k
        if off < n:
            A = A + sp.diags([-rng.random(n - off)], [off], shape=(n, n))
    if extra:
        free = rng.permutation(np.arange(n // 4, n // 2))[:extra], rng.permutation(np.arange(n // 2, 3 * n // 4))[:extra]
        A = A + sp.csr_matrix((-rng.random(extra), free), shape=(n, n))
    A = A + A.T
    A = sp.csr_matrix(A)
    d = np.asarray(abs(A).sum(axis=1)).ravel() + 0.02 + 0.05 * rng.random(n)
    A = sp.csr_matrix(A + sp.diags([d], [0]))
    A.sort_indices()
    return A, rng.standard_normal(n)


def _counts(s):
    """One-launch solves of the handle that ran and that gave up."""
    import ctypes
    out = []
    for name in (b"one_launch", b"one_launch_gave_up"):
        n, ms = ctypes.c_int64(), ctypes.c_double()
        assert s.lib.shk_kernel_stats(s.ctx, name, ctypes.byref(n), ctypes.byref(ms)) == 0
        out.append(n.value)
    return tuple(out)


@pytest.mark.parametrize("n,band,extra,longest", [
    (1, 0, 0, 1), (2, 0, 0, 2), (511, 1, 0, 5), (513, 2, 0, 7), (5000, 2, 40, 8), (5000, 3, 0, 9), (131072, 1, 9, 6),
    (131073, 1, 0, 5), (140000, 2, 0, 7), (262145, 2, 50, 8), (263000, 2, 0, 7), (5000, 4, 0, 11), (393216, 1, 0, 5),
    (393217, 1, 0, 5), (400000, 1, 0, 5)])
def test_csr_resident(n, band, extra, longest):
    import torch
    import shiokaze_amd as shk
    A, b = _system(n, band, n + band, extra)
    assert np.diff(A.indptr).max() == longest
    fits = longest <= 8 and n <= 393216
    dev = [torch.from_numpy(a).cuda() for a in (A.indptr.astype(np.int64), A.indices.astype(np.int64), A.data, b)]
    tol = 1e-8
    s = shk.PCGSolver(config={"Preconditioner": "jacobi", "Residual": tol})
    xs, its = [], []
    for profile in (0, 1):
        s.configure("ProfileKernels", profile)
        x, r = s.solve(*dev)
        assert r["status"] == 0
        assert _counts(s) == (1 if fits and not profile else 0, 0)
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
