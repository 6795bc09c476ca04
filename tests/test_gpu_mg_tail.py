"""One V-cycle against the numpy restatement at the sizes where the one-workgroup coarse end
(k_mg_tail, csrc/mg.hip) changes shape: the coarsest level alone, odd and even extents, the
first level that fits as a dense grid (16^3, 64^2) and one that no longer does (17^3, 65 x 64),
and uneven grids.  FP32 passes of at most 16 terms a cell against FP64: a few roundings (6e-8)
per level, two passes each way, far below the 1e-5 asked for."""
import numpy as np
import pytest

from gpu_helpers import to_device
from oracle import mg_oracle as MG

pytestmark = pytest.mark.gpu


def _check(mask, hx, hy, hz, apply, seed):
    import torch
    rng = np.random.default_rng(seed)
    r = (rng.standard_normal(mask.shape) * mask).astype(np.float32)
    z = apply(torch.from_numpy(r)).cpu().numpy().astype(np.float64).reshape(mask.shape)
    ref = MG.vcycle(MG.hierarchy(MG.scaled_level0(mask, hx, hy, hz)), r.astype(np.float64))
    assert np.linalg.norm(z - ref) <= 1e-5 * np.linalg.norm(ref)
    assert np.all(z[mask == 0] == 0)


@pytest.mark.parametrize("n", [(8, 8, 8), (9, 9, 9), (16, 17, 15), (32, 32, 32), (34, 34, 34), (33, 36, 29),
                               (40, 20, 9), (70, 61, 52)], ids=str)
def test_tail_3d(scenes, n):
    import shiokaze_amd
    sc = scenes(3, n, 1)
    d = to_device(sc)
    with shiokaze_amd.MacPressureSolver3(sc["shape"], sc["dx"], config={"Preconditioner": "mg"}) as ps:
        ps.project(1.0, (d["u"], d["v"], d["w"]), d["solid"], (d["us"], d["vs"], d["ws"]), d["fluid"])
        s = {k: v.cpu().numpy().astype(np.float64) for k, v in ps.export_scaled().items()}
        _check(s["mask"], s["hx"], s["hy"], s["hz"], lambda r: ps.mg_apply(r.cuda()), 1)


@pytest.mark.parametrize("n", [(8, 8), (128, 128), (130, 128), (96, 80)], ids=str)
def test_tail_2d(n):
    from shiokaze_amd import MacPressureSolver2
    from test_gpu_2d import _dev, _scaled_2d, _scene
    sc = _scene(3, n, 3)
    ny, nx = sc["fluid"].shape
    d = _dev(sc)
    with MacPressureSolver2((nx, ny), sc["dx"], config={"Preconditioner": "mg"}) as ps:
        ps.project(1.0, (d["u"], d["v"]), d["solid"], (d["us"], d["vs"]), d["fluid"])
        mask, hx, hz = _scaled_2d({k: v.cpu().numpy() for k, v in ps.export_system().items()})
        emb = lambda a: a.reshape(ny, 1, nx)  # noqa: E731
        _check(emb(mask), emb(hx), np.zeros((ny, 1, nx)), emb(hz),
               lambda r: ps.mg_apply(r.reshape(ny, nx).contiguous().cuda()), 3)
