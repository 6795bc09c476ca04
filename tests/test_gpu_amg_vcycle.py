"""One V-cycle of the CSR multigrid (csrc/amg.hip) against the numpy restatement at the sizes
where its launches change: a matrix that is its own coarsest level (k_amg_coarse; up to 1024 rows
where nothing pairs up), the coarsest level alone in k_amg_tail (up to 128 rows, and a stalled one
of several hundred), several levels in it, the first level of at most 256 rows, which is in it,
and one of more, which is not, and levels of one launch each.

After one iteration of CG from zero x = (b.z / z.Az) z with z = M b, so the first iterate shows
the V-cycle and the r.z partials.  All sums are FP64 and differ in order only: 1e-16 a term times a
coarsest matrix of condition below 1e4 times a few levels, far below the 1e-10 asked for."""
import numpy as np
import pytest
import scipy.sparse as sp

from oracle import amg_oracle as G

pytestmark = pytest.mark.gpu


def _chain(n, alone, seed):
    """A chain of n rows with random couplings and `alone` rows coupled to none, shuffled in."""
    rng = np.random.default_rng(seed)
    w = 0.5 + rng.random(max(n - 1, 0))
    A = sp.diags([-w, -w], [-1, 1], shape=(n, n)).tocsr() if n else sp.csr_matrix((0, 0))
    A = sp.block_diag([m for m in (A, sp.csr_matrix((alone, alone))) if m.shape[0]]).tocsr()
    A = sp.csr_matrix(A + sp.diags([np.asarray(abs(A).sum(axis=1)).ravel() + 0.02 + 0.1 * rng.random(n + alone)], [0]))
    if alone:
        p = rng.permutation(n + alone)
        A = A[p][:, p].tocsr()
    A.sort_indices()
    return A, rng.standard_normal(n + alone)


def _grid(nx, ny, nz, seed):
    rng = np.random.default_rng(seed)
    one = lambda n: sp.diags([-np.ones(n - 1), -np.ones(n - 1)], [-1, 1])  # noqa: E731
    W = sp.kron(sp.kron(one(nz), sp.eye(ny)), sp.eye(nx)) + sp.kron(sp.kron(sp.eye(nz), one(ny)), sp.eye(nx)) + sp.kron(
        sp.kron(sp.eye(nz), sp.eye(ny)), one(nx))
    W = sp.csr_matrix(W)
    W.data *= 1.0 + 1e-3 * np.arange(W.nnz) / W.nnz
    W = sp.csr_matrix(0.5 * (W + W.T))
    A = sp.csr_matrix(W + sp.diags([np.asarray(abs(W).sum(axis=1)).ravel() + 0.01], [0]))
    A.sort_indices()
    return A, rng.standard_normal(nx * ny * nz)


# (system, rows of the levels as the restatement builds them)
CASES = [(lambda: _chain(1, 0, 0), [1]), (lambda: _chain(128, 0, 1), [128]), (lambda: _chain(0, 1000, 2), [1000]),
         (lambda: _chain(129, 0, 3), [129, 33]), (lambda: _chain(600, 600, 4), None), (lambda: _chain(250, 150, 5), None),
         (lambda: _chain(480, 100, 5), None),
         (lambda: _chain(1024, 0, 6), None), (lambda: _chain(1300, 0, 7), None), (lambda: _grid(17, 15, 13, 8), None),
         (lambda: _grid(45, 40, 33, 9), None)]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_first_iterate(case):
    import torch
    import shiokaze_amd as shk
    make, rows = CASES[case]
    A, b = make()
    levels = G.hierarchy(A)
    sizes = [lv[0].shape[0] for lv in levels]
    print(f"[gpu] amg levels {sizes}")
    assert rows is None or sizes == rows
    z = G.vcycle(levels, b)
    want = (b @ z) / (z @ (A @ z)) * z
    dev = [torch.from_numpy(a).cuda() for a in (A.indptr.astype(np.int64), A.indices.astype(np.int64), A.data, b)]
    s = shk.PCGSolver(config={"Preconditioner": "mg", "Residual": 1e-30, "MaxIterations": 1})
    for _ in range(2):   # the second with the hierarchy kept
        x, r = s.solve(*dev)
        assert r["count"] == 1
        assert np.linalg.norm(x.cpu().numpy() - want) <= 1e-10 * np.linalg.norm(want)
    s.close()


def test_cases_reach_the_edges():
    """The level sizes that the cases are there for."""
    sizes = [[lv[0].shape[0] for lv in G.hierarchy(make()[0])] for make, _ in CASES]
    assert any(len(s) == 1 and s[0] > 256 for s in sizes)                       # one stalled level
    assert any(len(s) == 2 and s[-1] <= 128 for s in sizes)                     # the coarsest alone in the tail
    assert any(len(s) > 1 and 256 < s[-1] <= 1024 for s in sizes)               # a stalled coarsest in the tail
    assert any(len([n for n in s[1:] if n <= 256]) >= 3 for s in sizes)         # several levels in the tail
    assert any(250 <= n <= 256 for s in sizes for n in s[1:]) and any(256 < n <= 330 for s in sizes for n in s[1:])
    assert any(len([n for n in s[1:] if n > 256]) >= 2 for s in sizes)          # levels of one launch each
