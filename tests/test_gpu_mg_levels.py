"""Multigrid on both sides of the edges of its level-0 launches (csrc/mg.hip): up to 2048 active
bricks a wave takes two z-planes of a brick, above it the whole brick; up to 8192 the r.z
partials go to the Krylov kernels as the blocks write them (2048 of them at most), above it
k_mg_fold sums them first.  One V-cycle against the numpy restatement (FP32 passes of at most 16
terms a cell, a few roundings of 6e-8 per level, against FP64), and a projection, whose CG
takes its beta from those partials: with a wrong one it would not get there in a few times ten
iterations.  The active bricks are asserted, so that no row drifts to another kernel."""
import numpy as np
import pytest

from gpu_helpers import log, to_device
from test_gpu_mg_tail import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,above,most", [((115, 126, 135), 1950, 2048), ((129, 117, 127), 2048, 2200),
                                          ((196, 207, 216), 8000, 8192), ((210, 198, 208), 8192, 8400)], ids=str)
def test_levels_3d(scenes, n, above, most):
    import shiokaze_amd
    sc = scenes(3, n, 4)
    d = to_device(sc)
    with shiokaze_amd.MacPressureSolver3(sc["shape"], sc["dx"],
                                         config={"Preconditioner": "mg", "Residual": 1e-6}) as ps:
        r = ps.project(1.0, (d["u"], d["v"], d["w"]), d["solid"], (d["us"], d["vs"], d["ws"]), d["fluid"])
        log(f"[gpu] mg {n}: {r['active_bricks']} bricks, {r['count']} its")
        assert above < r["active_bricks"] <= most
        assert r["status"] == 0 and r["true_relres_inf"] <= 1e-6 and r["count"] <= 60
        s = {k: v.cpu().numpy().astype(np.float64) for k, v in ps.export_scaled().items()}
        _check(s["mask"], s["hx"], s["hy"], s["hz"], lambda v: ps.mg_apply(v.cuda()), 1)


@pytest.mark.parametrize("n,above,most", [((1500, 1200), 1500, 2048), ((2000, 1800), 2048, 8192),
                                          ((3300, 3200), 8192, 10000)], ids=str)
def test_levels_2d(n, above, most):
    from shiokaze_amd import MacPressureSolver2
    from test_gpu_2d import _dev, _scaled_2d, _scene
    sc = _scene(3, n, 4)
    ny, nx = sc["fluid"].shape
    d = _dev(sc)
    with MacPressureSolver2((nx, ny), sc["dx"], config={"Preconditioner": "mg", "Residual": 1e-6}) as ps:
        r = ps.project(1.0, (d["u"], d["v"]), d["solid"], (d["us"], d["vs"]), d["fluid"])
        log(f"[gpu] 2D mg {n}: {r['active_bricks']} bricks, {r['count']} its")
        assert above < r["active_bricks"] <= most
        assert r["status"] == 0 and r["true_relres_inf"] <= 1e-6 and r["count"] <= 90
        mask, hx, hz = _scaled_2d({k: v.cpu().numpy() for k, v in ps.export_system().items()})
        emb = lambda a: a.reshape(ny, 1, nx)  # noqa: E731
        _check(emb(mask), emb(hx), np.zeros((ny, 1, nx)), emb(hz),
               lambda v: ps.mg_apply(v.reshape(ny, nx).contiguous().cuda()), 3)
