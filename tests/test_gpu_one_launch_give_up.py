"""A one-launch solve (csrc/resident.hip) whose workgroups stop waiting for each other: the call
then runs the two-kernel iteration and returns its result, and the context does not try again
for a number of solves.  OneLaunchWait forces the condition from the host: below one tick
of the 100 MHz clock every workgroup gives up at its first wait; a few microseconds stop some
in later exchanges, with the vectors part way.  Every kernel ends normally either way.

The two-kernel iteration is ProfileKernels=1's, deterministic, so the results agree bit for bit.
"""
import numpy as np
import pytest

from test_gpu_resident import _fields, _project, _solver
from test_gpu_resident_csr import _counts, _system

pytestmark = pytest.mark.gpu

NOW, SOON = "1e-9", "2e-6"


@pytest.mark.parametrize("wait", [NOW, SOON])
@pytest.mark.parametrize("precision,precond", [("fp64", "none"), ("fp64", "jacobi"), ("mixed", "none"),
                                               ("mixed", "jacobi")])
@pytest.mark.parametrize("shape", [(40, 33, 35), (150, 140, 130), (129, 264)], ids=str)
def test_project_gives_up(shape, precision, precond, wait):
    import torch
    d, dx = _fields(shape, 3, 2)
    with _solver(shape, dx, Precision=precision, Preconditioner=precond, Residual=1e-6) as ps:
        ps.configure("ProfileKernels", 1)
        want, vel = _project(ps, d)
        x = ps.export_system()["x"].clone()
        ps.configure("ProfileKernels", 0)
        ps.configure("OneLaunchWait", wait)
        got, vel2 = _project(ps, d)
        ran, gave_up = _counts(ps)
        if wait == SOON and ran:   # the waits may all have been that short
            return
        # the first inner solve gives up, the others of the call do not try
        assert (ran, gave_up) == (0, 1)
        for k in ("status", "count", "outer", "reresid", "true_relres_inf"):
            assert got[k] == want[k]
        assert torch.equal(ps.export_system()["x"], x)
        assert all(torch.equal(a, b) for a, b in zip(vel, vel2))


@pytest.mark.parametrize("noalloc", [False, True])
def test_csr_gives_up(noalloc):
    import torch
    import shiokaze_amd as shk
    A, b = _system(5000, 2, 7)
    dev = [torch.from_numpy(a).cuda() for a in (A.indptr.astype(np.int64), A.indices.astype(np.int64), A.data, b)]
    s = shk.PCGSolver(config={"Preconditioner": "jacobi", "Residual": 1e-8, "ProfileKernels": 1})
    x, r = s.solve(*dev)
    s.configure("ProfileKernels", 0)
    for wait in (NOW, SOON):
        s.configure("ProfileKernels", 0)   # counts from 0
        s.configure("OneLaunchWait", wait)
        x2, r2 = s.solve(*dev, noalloc=noalloc)
        if _counts(s)[1]:
            assert r2["count"] == r["count"] and torch.equal(x, x2)
        else:
            assert wait == SOON
    s.close()


def test_rest_after_giving_up():
    """32 solves without another try, then 64; a solve that runs through ends it, 0 switches
    the form off."""
    shape = (24, 24, 24)
    d, dx = _fields(shape, 1, 0)
    with _solver(shape, dx, Precision="fp64", Preconditioner="jacobi", Residual=1e-4) as ps:
        ps.configure("OneLaunchWait", NOW)
        tries = []
        for _ in range(1 + 32 + 1 + 64 + 1):
            _project(ps, d)
            tries.append(_counts(ps)[1])
        assert tries == [1] * 33 + [2] * 65 + [3] and _counts(ps)[0] == 0
        ps.configure("OneLaunchWait", 0.67)   # setting the key ends the rest
        for _ in range(3):
            _project(ps, d)
        assert _counts(ps) == (3, 3)
        ps.configure("OneLaunchWait", 0)
        _project(ps, d)
        assert _counts(ps) == (3, 3)
        import shiokaze_amd as shk
        for bad in ("-1", "31", "x", "nan"):
            with pytest.raises(shk.ShkError):
                ps.configure("OneLaunchWait", bad)
