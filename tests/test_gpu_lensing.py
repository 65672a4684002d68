"""GPU lens planes (2-D paint, density plane, Gaussian smoothing) and their
adjoints against the oracle."""
import numpy as np
import pytest
import torch

from oracle import lensing as ol
from oracle import painting as op
from oracle import utils as ou

pytestmark = pytest.mark.gpu


def dev(x):
    return torch.as_tensor(np.asarray(x, np.float32), device="cuda")


def rel_err(got, ref):
    return np.abs(np.asarray(got, np.float64) - ref).max() / max(np.abs(ref).max(), 1e-30)


@pytest.mark.parametrize("shape,weighted", [((64, 64), True), ((37, 50), False), ((512, 512), True)])
def test_cic_paint_2d_matches_oracle(gpu, shape, weighted):
    from jaxpm_amd import painting
    print(f"cic_paint_2d {shape} weighted={weighted}", flush=True)
    r = np.random.default_rng(10)
    n = 20000
    pos = (r.uniform(-1.2, 2.2, size=(n, 2)) * np.array(shape)).astype(np.float32)
    w = r.uniform(0.2, 2.0, n).astype(np.float32) if weighted else None
    base = r.normal(size=shape).astype(np.float32)
    got = painting.cic_paint_2d(dev(base), dev(pos), None if w is None else dev(w)).cpu().numpy()
    ref = op.cic_paint_2d(base, pos, w)
    assert rel_err(got, ref) < 2e-6
    with pytest.raises(ValueError):
        painting.cic_paint_2d(dev(base), dev(pos), dev(np.ones(n - 1)))


def test_cic_paint_2d_gradients(gpu):
    """Mesh, weight and position cotangents: the weight cotangent is the
    periodic bilinear read of the plane cotangent; the position cotangent
    matches float64 central differences of the oracle along random
    directions."""
    from scipy import ndimage

    from jaxpm_amd import painting
    r = np.random.default_rng(11)
    shape, n = (24, 20), 300
    pos = (r.uniform(-0.5, 1.5, size=(n, 2)) * np.array(shape)).astype(np.float32)
    w = r.uniform(0.5, 1.5, n).astype(np.float32)
    g = r.normal(size=shape)
    mt, pt, wt = dev(np.zeros(shape)).requires_grad_(True), dev(pos).requires_grad_(True), dev(w).requires_grad_(True)
    (painting.cic_paint_2d(mt, pt, wt) * dev(g)).sum().backward()
    assert np.allclose(mt.grad.cpu().numpy(), g.astype(np.float32))
    read = ndimage.map_coordinates(g, pos.astype(np.float64).T, order=1, mode="grid-wrap")
    assert rel_err(wt.grad.cpu().numpy(), read) < 1e-5
    gp = pt.grad.cpu().numpy().astype(np.float64)
    for k in range(4):
        u = r.normal(size=pos.shape) * 1e-4
        f = lambda x: np.sum(op.cic_paint_2d(np.zeros(shape), x, w.astype(np.float64)) * g)  # noqa: E731
        fd = (f(pos + u) - f(pos - u)) / 2
        assert abs(np.sum(gp * u) - fd) < 2e-3 * np.abs(gp * u).sum()


@pytest.mark.parametrize("res,sigma", [(64, None), (128, 1.5), (100, 2.0)])
def test_density_plane_matches_oracle(gpu, res, sigma):
    from jaxpm_amd import lensing
    print(f"density_plane res={res} sigma={sigma}", flush=True)
    r = np.random.default_rng(12)
    nx = 64
    pos = r.uniform(-0.3, 1.3, size=(60000, 3)).astype(np.float32) * nx
    got = lensing.density_plane(dev(pos), (nx, nx, nx), 30.0, 10.0, res, smoothing_sigma=sigma).cpu().numpy()
    ref = ol.density_plane(pos, (nx, nx, nx), 30.0, 10.0, res, smoothing_sigma=sigma, dtype=np.float32)
    assert got.shape == (res, res)
    assert rel_err(got, ref.astype(np.float64)) < 3e-6


@pytest.mark.parametrize("n", [64, 100, 512])
def test_gaussian_smoothing_matches_oracle(gpu, n):
    from jaxpm_amd import utils
    im = np.random.default_rng(13).normal(size=(n, n)).astype(np.float32)
    got = utils.gaussian_smoothing(dev(im), 1.3).cpu().numpy()
    assert rel_err(got, ou.gaussian_smoothing(im, 1.3)) < 3e-6
    with pytest.raises(ValueError):
        utils.gaussian_smoothing(dev(np.zeros((8, 16))), 1.0)


def test_density_plane_gradient(gpu):
    """Position cotangent of the smoothed density plane against float64
    central differences of the oracle along random directions (particles
    kept away from the slab faces, where the selection jumps)."""
    from jaxpm_amd import lensing
    r = np.random.default_rng(14)
    nx, res, center, width = 32, 32, 16.0, 8.0
    pos = r.uniform(0, nx, size=(3000, 3)).astype(np.float32)
    pos[:, 2] = np.where(r.uniform(size=3000) < 0.5, r.uniform(12.5, 19.5, 3000), r.uniform(21, 30, 3000))
    g = r.normal(size=(res, res))
    pt = dev(pos).requires_grad_(True)
    (lensing.density_plane(pt, (nx, nx, nx), center, width, res, smoothing_sigma=1.0) * dev(g)).sum().backward()
    gp = pt.grad.cpu().numpy().astype(np.float64)
    assert np.all(gp[:, 2] == 0)
    f = lambda x: np.sum(ol.density_plane(x, (nx, nx, nx), center, width, res, smoothing_sigma=1.0) * g)  # noqa: E731
    for k in range(4):
        u = r.normal(size=pos.shape) * 1e-4
        fd = (f(pos + u) - f(pos - u)) / 2
        assert abs(np.sum(gp * u) - fd) < 2e-3 * np.abs(gp * u).sum()


@pytest.mark.parametrize("res,n,frac", [(1, 786432, 1.0), (63, 786433, 0.3), (64, 800000, 1.0), (65, 786432, 0.02),
                                        (200, 790001, 0.5), (1024, 900000, 0.25), (4096, 786432, 1.0)])
def test_sorted_density_plane(gpu, res, n, frac):
    """The plane of many particles (sorted by 64-pixel tiles, several windows
    a tile at the small resolutions) against float64 sums of the float32
    coordinates' deposits: float32 weights (1.2e-7) and results (1.2e-7)
    leave less than 1e-6 of the largest pixel."""
    from jaxpm_amd import lensing
    from oracle import painting as op
    print(f"sorted density_plane res={res} n={n} frac={frac}", flush=True)
    r = np.random.default_rng(15)
    nx = 50
    pos = (r.uniform(-0.3, 1.3, size=(n, 3)) * nx).astype(np.float32)
    pos[:, 2] = np.where(r.uniform(size=n) < frac, r.uniform(21, 29, n), r.uniform(31, 49, n)).astype(np.float32)
    got = lensing.density_plane(dev(pos), (nx, nx, nx), 25.0, 10.0, res).cpu().numpy()
    xy = np.mod(pos[:, :2], np.float32(nx)) / np.float32(nx) * np.float32(res)
    w = ((pos[:, 2] > 20) & (pos[:, 2] <= 30)).astype(np.float64)
    ref = op.cic_paint_2d(np.zeros((res, res)), xy.astype(np.float64), w) / ((nx / res) ** 2 * 10.0)
    assert rel_err(got, ref) < 1e-6


def test_sorted_density_plane_nonfinite(gpu):
    """NaN and infinite coordinates reach the same pixels as with one atomic
    per corner, and particles of a NaN z none."""
    from jaxpm_amd import _lib, lensing
    print("sorted density_plane non-finite", flush=True)
    r = np.random.default_rng(16)
    pos = (r.uniform(0, 1, size=(786432, 3)) * 64).astype(np.float32)
    pos[5], pos[70000], pos[9], pos[11, 2] = (np.nan, 40.5, 30), (20.25, np.inf, 30), (np.nan, -np.inf, 30), np.nan
    p = dev(pos)
    got = lensing.density_plane(p, (64, 64, 64), 30.0, 10.0, 100)
    ref = torch.empty_like(got)
    _lib.call("jpm_density_plane_f32", _lib.stream(), _lib.ptr(p), p.shape[0], 64, 64, 30.0, 10.0, 100, _lib.ptr(ref))
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and bool(torch.isnan(ref).any())
    ok = ~torch.isnan(ref)
    assert rel_err(got[ok].cpu().numpy(), ref[ok].double().cpu().numpy()) < 3e-6


def test_density_plane_of_more_particles_than_one_sort(gpu):
    """2^27 particles and a few more are sorted in two turns.  The plane is
    linear in the particles: against the sum of the planes of its two turns,
    each rounded to float32 as windows, as a pixel and by the normalisation."""
    from jaxpm_amd import _ops
    n, res = 2 ** 27 + 900001, 200
    print(f"density plane n={n}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(21)
    pos = torch.rand((n, 3), generator=gen, device="cuda") * 64
    args = ((64, 64, 64), 32.0, 16.0, res)
    whole = _ops.density_plane(pos, *args)
    first, rest = _ops.density_plane(pos[:2 ** 27], *args), _ops.density_plane(pos[2 ** 27:], *args)
    ref = first.double() + rest.double()
    assert float(whole.double().sum()) > 0
    assert float(((whole.double() - ref).abs() / ref).max()) < 6 * 2.0 ** -24
