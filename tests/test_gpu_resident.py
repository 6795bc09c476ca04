"""The one-launch CG solve (csrc/resident.hip) against the two-kernel iteration.

ProfileKernels=1 runs the two-kernel iteration, so both solve the same system on one
context.  Each stops with max|b - A x| <= tol max|b|, hence max|A (x1 - x2)| <= 2 tol
max|b| whatever the summation orders.  The sizes are the edges of the launch shape: one
brick, a started second workgroup (8 waves of 1 brick each), and on 256 compute units both
sides of the 2048, 4096, 6144, 8192 and 12,288 bricks at which a wave takes 2, 3, 4 and 6
FP32 bricks (2 FP64 ones up to 4096) and the two-kernel iteration takes over, in 2D one size
of each.  The active bricks are asserted, so that no row drifts to another kernel, and
shk_kernel_stats' counters say which solve ran.
"""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _fields(shape, kind, seed):
    import torch
    from shiokaze_amd import scene
    sc = scene.generate(kind, shape, seed) if len(shape) == 3 else scene.generate2d(kind, shape, seed)
    keys = ("fluid", "solid", "u", "v", "us", "vs") + (("w", "ws") if len(shape) == 3 else ())
    return {k: torch.from_numpy(np.ascontiguousarray(sc[k])).cuda() for k in keys}, sc["dx"]


def _solver(shape, dx, **cfg):
    import shiokaze_amd as shk
    cls = shk.MacPressureSolver3 if len(shape) == 3 else shk.MacPressureSolver2
    return cls(shape, dx, config=cfg)


def _project(ps, d):
    axes = "uvw" if "w" in d else "uv"
    vel = [d[a].clone() for a in axes]
    return ps.project(1.0, vel, d["solid"], [d[a + "s"] for a in axes], d["fluid"]), vel


def _apply(sy, x):
    """A x of an exported system (dense cells, low-face couplings)."""
    y = sy["diag"] * x
    axes = {"cx": x.dim() - 1, "cy": x.dim() - 2, "cz": x.dim() - 3 if x.dim() == 3 else 0}
    if x.dim() == 2:
        axes = {"cx": 1, "cz": 0}
    for k, a in axes.items():
        n = x.shape[a]
        if n < 2:
            continue
        c = sy[k].narrow(a, 1, n - 1)
        y.narrow(a, 1, n - 1).sub_(c * x.narrow(a, 0, n - 1))
        y.narrow(a, 0, n - 1).sub_(c * x.narrow(a, 1, n - 1))
    return y


# shape, the bricks it lies between (more than, at most), bricks per wave in FP32 and FP64 (0: two
# kernels)
SHAPES = [((8, 8, 8), 0, 1, 1, 1), ((19, 24, 13), 0, 2048, 1, 1), ((33, 30, 41), 0, 2048, 1, 1),
          ((16, 120, 100), 0, 2048, 1, 1), ((115, 126, 135), 1950, 2048, 1, 1), ((122, 130, 127), 1950, 2048, 1, 1),
          ((129, 117, 127), 2048, 2200, 2, 2), ((145, 156, 165), 3900, 4096, 2, 2), ((162, 150, 160), 4096, 4200, 3, 0),
          ((176, 170, 182), 4096, 6144, 3, 0), ((175, 186, 195), 5950, 6144, 3, 0), ((187, 187, 187), 6144, 6300, 4, 0),
          ((196, 207, 216), 8000, 8192, 4, 0), ((210, 198, 208), 8192, 8400, 6, 0),
          ((223, 234, 243), 12000, 12288, 6, 0), ((241, 241, 241), 12288, 12500, 0, 0),
          ((70, 37), 0, 2048, 1, 1), ((129, 264), 0, 2048, 1, 1), ((1500, 1200), 0, 2048, 1, 1),
          ((2000, 1800), 2048, 4096, 2, 2), ((2600, 2600), 4096, 6144, 3, 0), ((3000, 2700), 6144, 8192, 4, 0),
          ((3300, 3200), 8192, 12288, 6, 0)]


# where two kernels run anyway the Jacobi row shows it
ROWS = [(*row[:3], row[4] if precision == "fp64" else row[3], precision, precond) for row in SHAPES
        for precision in ("fp64", "mixed") for precond in ("none", "jacobi")
        if precond == "jacobi" or (row[4] if precision == "fp64" else row[3])]


@pytest.mark.parametrize("shape,above,most,per_wave,precision,precond", ROWS,
                         ids=["{0}-{4}-{5}".format(*row) for row in ROWS])
def test_resident_matches_two_kernels(shape, above, most, per_wave, precision, precond):
    d, dx = _fields(shape, 3 if min(shape) > 12 else 1, 4)
    # plain CG of the large 2D grids does not get to 1e-6 in the 30,000 iterations of the default cap
    tol = 1e-3 if precond == "none" and len(shape) == 2 and most > 4096 else 1e-6
    with _solver(shape, dx, Precision=precision, Preconditioner=precond, Residual=tol) as ps:
        xs, its = [], []
        for profile in (0, 1):
            ps.configure("ProfileKernels", profile)
            r, _ = _project(ps, d)
            # the recurrence residual of an FP64 solve differs from the true one by rounding
            assert r["status"] == 0 and r["true_relres_inf"] <= tol * (1 + 1e-4)
            its.append(r["count"])
            assert above < r["active_bricks"] <= most
            ran = ps.kernel_stats("one_launch")[0], ps.kernel_stats("one_launch_gave_up")[0]
            assert ran == (r["outer"] if per_wave and not profile else 0, 0)
            assert (ps.kernel_stats("axpy_norm")[0] > 0) == (profile == 1)
            sy = ps.export_system()
            xs.append(sy["x"].clone())
        bmax = float(sy["rhs"].abs().max())
        assert float(_apply(sy, xs[0] - xs[1]).abs().max()) <= 2 * tol * bmax * (1 + 1e-3)
        print(f"[gpu] {shape} {precision} {precond}: {r['active_bricks']} bricks, {per_wave} a wave, its {its}")
        # FP64 plain CG: 20 random renumberings of the unknowns alone spread the counts of the small
        # shapes over 246..270, 558..593 and 1322..1397 (the oracle's CPU solve).  The others do
        # not see the order of the FP64 sums
        assert abs(its[0] - its[1]) <= (max(3, 0.1 * its[1]) if (precision, precond) == ("fp64", "none") else 2)


def test_resident_outcomes():
    """Cap, zero right-hand side and NaN end as the two-kernel iteration ends them."""
    import torch
    d, dx = _fields((40, 33, 35), 3, 1)
    with _solver((40, 33, 35), dx, Precision="fp64", Preconditioner="jacobi", Residual=1e-8) as ps:
        got = []
        for profile in (0, 1):
            ps.configure("ProfileKernels", profile)
            row = []
            ps.configure("MaxIterations", 7)
            row.append(_project(ps, d)[0])
            ps.configure("MaxIterations", 3000)
            still = dict(d, u=torch.zeros_like(d["u"]), v=torch.zeros_like(d["v"]), w=torch.zeros_like(d["w"]))
            row.append(_project(ps, still)[0])
            bad = dict(d, u=torch.full_like(d["u"], float("nan")))
            row.append(_project(ps, bad)[0])
            got.append([(r["status"], r["count"]) for r in row])
        assert got[0] == got[1]
        assert got[0][0] == (1, 7)


def test_resident_threads():
    """Contexts of several threads solve at once: the launches share the compute units."""
    shapes = [(120, 110, 100), (64, 64, 64), (90, 130, 80), (40, 50, 45)]
    jobs = []
    for k, shape in enumerate(shapes):
        d, dx = _fields(shape, 3, k)
        ps = _solver(shape, dx, Precision="mixed", Preconditioner="jacobi", Residual=1e-6)
        r, vel = _project(ps, d)
        jobs.append((ps, d, r, vel))
    out = [None] * len(jobs)

    def work(k):
        ps, d, _, _ = jobs[k]
        out[k] = [_project(ps, d) for _ in range(3)]

    ts = [threading.Thread(target=work, args=(k,)) for k in range(len(jobs))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for k, (ps, d, r, vel) in enumerate(jobs):
        for r2, vel2 in out[k]:
            assert r2["status"] == r["status"] == 0 and r2["count"] == r["count"]
            assert all(bool((a == b).all()) for a, b in zip(vel, vel2))
        ps.close()
