"""The narrow-band passes over cell lists and groups of four cells, at the sizes where they
can go wrong: rows that are and are not multiples of four, grids whose last group of 4, 16
or 4096 cells is started only, arrays that are only byte- or float-aligned, and masks
whose active value is not 1.  All against the oracle bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(21, 13, 9), (20, 14, 11), (17, 16, 16), (35, 33, 31), (2, 3, 5)]


def _inputs(shape, seed):
    nx, ny, nz = shape
    dx = 1.0 / max(shape)
    rng = np.random.default_rng(seed)
    z, y, x = np.meshgrid(*[(np.arange(n) + 0.5) * dx for n in (nz, ny, nx)], indexing="ij")
    phi = (y - 0.4 * ny * dx + 0.15 * np.sin(9 * x) * np.cos(7 * z)) * (1.0 + 0.4 * np.sin(5 * x))
    phi = (phi + 0.2 * dx * rng.standard_normal(phi.shape)).astype(np.float32)
    band = (np.abs(phi) < 3 * dx).astype(np.uint8)
    return dx, np.clip(phi, -3 * dx, 3 * dx).astype(np.float32), band


def _dev(a, offset):
    """a on the GPU, `offset` elements past an allocation's start."""
    import torch
    t = torch.zeros(a.size + offset, dtype=torch.float32 if a.dtype == np.float32 else torch.uint8, device="cuda")
    t[offset:] = torch.from_numpy(np.ascontiguousarray(a).reshape(-1)).cuda()
    return t[offset:].view(a.shape)


@pytest.fixture(scope="module")
def oracle():
    from oracle import oracle as O
    return O


def _liquid(shape, dx):
    import shiokaze_amd as shk
    ps = shk.MacPressureSolver3(shape, dx)
    return ps, shk.MacLiquidVelocity(ps)


@pytest.mark.parametrize("offset,active", [(0, 1), (1, 1), (3, 255)])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_redistance(oracle, shape, offset, active):
    dx, phi, band = _inputs(shape, 1)
    ps, lv = _liquid(shape, dx)
    with ps:
        for width in (1, 3):
            dphi, dband = _dev(phi, offset), _dev(band * np.uint8(active), offset)
            cnt = lv.redistance(dphi, dband, width)
            ophi, oband, ocnt = oracle.redistance(dx, phi, band, width)
            assert cnt == ocnt
            np.testing.assert_array_equal(dband.cpu().numpy(), oband)
            np.testing.assert_array_equal(dphi.cpu().numpy(), ophi)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("maccormack", [1, 0])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_advect_levelset(oracle, shape, maccormack, offset):
    dx, phi, band = _inputs(shape, 2)
    nx, ny, nz = shape
    rng = np.random.default_rng(5)
    faces = [(nz, ny, nx + 1), (nz, ny + 1, nx), (nz + 1, ny, nx)]
    vel = [rng.uniform(-2, 2, s).astype(np.float32) for s in faces]
    masks = [(rng.random(s) < 0.9).astype(np.uint8) for s in faces]
    want = oracle.advect_levelset(dx, 0.7 * dx, phi, band, vel, masks, 3 * dx, maccormack=bool(maccormack))
    ps, lv = _liquid(shape, dx)
    with ps:
        ps.configure("MacCormack", maccormack)
        dphi = _dev(phi, offset)
        lv.advect_levelset(0.7 * dx, dphi, _dev(band, offset), [_dev(v, 0) for v in vel], [_dev(m, 0) for m in masks],
                           3 * dx)
        np.testing.assert_array_equal(dphi.cpu().numpy(), want)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_extrapolate_levelset(oracle, shape, offset):
    dx, phi, band = _inputs(shape, 3)
    nx, ny, nz = shape
    z, y, x = np.meshgrid(*[np.arange(n + 1) * dx for n in (nz, ny, nx)], indexing="ij")
    bg = np.float32(3 * dx)
    for solid in ((y - 0.3 * ny * dx + 0.2 * x).astype(np.float32), (y + dx).astype(np.float32)):
        sband = (np.abs(solid) < 3 * dx).astype(np.uint8)
        sol = np.clip(solid, -bg, bg)
        ophi, oband, ocnt = oracle.extrapolate_levelset(dx, sol, phi, band, bg, solid_band=sband)
        ps, lv = _liquid(shape, dx)
        with ps:
            dphi, dband = _dev(phi, offset), _dev(band, offset)
            cnt = lv.extrapolate_levelset(_dev(sol, offset), dphi, dband, float(bg), solid_band=_dev(sband, offset))
            assert cnt == ocnt
            np.testing.assert_array_equal(dband.cpu().numpy(), oband)
            np.testing.assert_array_equal(dphi.cpu().numpy(), ophi)


@pytest.mark.parametrize("offset,weno", [(0, 0), (1, 0), (0, 1)])
@pytest.mark.parametrize("maccormack,shape", [(1, (103, 84, 67)), (0, (151, 130, 109))])
@pytest.mark.parametrize("kind", ["thin", "third", "all"])
def test_advect_levelset_thin_and_wide_bands(oracle, kind, maccormack, shape, offset, weno):
    """Grids large enough for a list (more than 524,288 cells, 2,097,152 for the one
    semi-Lagrangian pass): a band of a few percent goes by its list, one of a third and one
    of all cells by the mask (bands.h).  A second call uses the other counter."""
    nx, ny, nz = shape
    dx = 1.0 / nx
    z, y, x = np.meshgrid(*[(np.arange(n) + 0.5) * dx for n in (nz, ny, nx)], indexing="ij")
    phi = (y - 0.4 * ny * dx + 0.05 * np.sin(9 * x) * np.cos(7 * z)).astype(np.float32)
    band = (np.abs(phi) < {"thin": 2 * dx, "third": 0.12, "all": 9.0}[kind]).astype(np.uint8)
    low, high = {"thin": (0, 0.05), "third": (0.25, 0.5), "all": (0.99, 1)}[kind]
    assert low < band.mean() <= high
    rng = np.random.default_rng(5)
    faces = [(nz, ny, nx + 1), (nz, ny + 1, nx), (nz + 1, ny, nx)]
    vel = [rng.uniform(-2, 2, s).astype(np.float32) for s in faces]
    masks = [(rng.random(s) < 0.9).astype(np.uint8) for s in faces]
    ps, lv = _liquid(shape, dx)
    with ps:
        ps.configure("MacCormack", maccormack)
        ps.configure("WENO", weno)
        dphi, dband = _dev(phi, offset), _dev(band, offset)
        dvel, dmasks = [_dev(v, 0) for v in vel], [_dev(m, 0) for m in masks]
        for _ in range(2):
            phi = oracle.advect_levelset(dx, 0.7 * dx, phi, band, vel, masks, 3 * dx, maccormack=bool(maccormack),
                                         weno=bool(weno))
            lv.advect_levelset(0.7 * dx, dphi, dband, dvel, dmasks, 3 * dx)
            np.testing.assert_array_equal(dphi.cpu().numpy(), phi)
