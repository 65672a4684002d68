"""Float64 paths under the x64 switch (the reference's equivalence tests run
with jax_enable_x64, tests/test_distributed_pm.py:30): cic_paint, cic_read,
cic_paint_dx, cic_read_dx and pm_forces in float64 against the float64
oracle at double-precision tolerances, and the float32 default for float64
input when the switch is off (as in JAX)."""
import warnings

import numpy as np
import pytest
import torch

from oracle import painting as op
from oracle import pm as opm

pytestmark = pytest.mark.gpu


@pytest.fixture
def x64():
    from jaxpm_amd import config
    config.update("jax_enable_x64", True)
    yield
    config.update("jax_enable_x64", False)


def lattice(shape):
    return np.stack(np.meshgrid(*[np.arange(s) for s in shape], indexing="ij"), -1)


def rel(got, ref):
    return np.abs(np.asarray(got) - ref).max() / np.abs(ref).max()


@pytest.mark.parametrize("shape", [(16, 16, 16), (12, 20, 9)])
def test_paint_read_f64(gpu, x64, shape):
    from jaxpm_amd import painting
    r = np.random.default_rng(1)
    n = 5000
    pos = r.uniform(-4, max(shape) + 4, (n, 3))
    w = r.normal(size=n)
    mesh0 = r.normal(size=shape)
    got = painting.cic_paint(torch.as_tensor(mesh0, device=gpu), torch.as_tensor(pos, device=gpu),
                             torch.as_tensor(w, device=gpu))
    assert got.dtype == torch.float64
    assert rel(got.cpu().numpy(), op.cic_paint(mesh0, pos, w)) < 1e-13
    m = r.normal(size=shape)
    rd = painting.cic_read(torch.as_tensor(m, device=gpu), torch.as_tensor(pos, device=gpu))
    assert rd.dtype == torch.float64
    assert rel(rd.cpu().numpy(), op.cic_read(m, pos)) < 1e-14


def test_relative_f64(gpu, x64):
    from jaxpm_amd import painting
    shape = (16, 8, 12)
    r = np.random.default_rng(2)
    disp = r.normal(scale=1.3, size=(*shape, 3))
    w = r.uniform(0.5, 1.5, shape)
    got = painting.cic_paint_dx(torch.as_tensor(disp, device=gpu), weight=torch.as_tensor(w, device=gpu))
    assert got.dtype == torch.float64
    assert rel(got.cpu().numpy(), op.cic_paint_dx(disp, w)) < 1e-13
    m = r.normal(size=shape)
    rd = painting.cic_read_dx(torch.as_tensor(m, device=gpu), torch.as_tensor(disp, device=gpu))
    assert rel(rd.cpu().numpy(), op.cic_read_dx(m, disp)) < 1e-14


@pytest.mark.parametrize("shape,absolute", [((16, 16, 16), True), ((12, 16, 20), True), ((16, 16, 16), False)])
def test_pm_forces_f64(gpu, x64, shape, absolute):
    from jaxpm_amd import pm
    r = np.random.default_rng(3)
    d = r.normal(scale=0.7, size=(*shape, 3))
    pos = lattice(shape) + d if absolute else d
    got = pm.pm_forces(torch.as_tensor(pos, device=gpu), mesh_shape=shape, paint_absolute_pos=absolute)
    assert got.dtype == torch.float64
    ref = opm.pm_forces(pos, mesh_shape=shape, paint_absolute_pos=absolute)
    assert rel(got.cpu().numpy(), ref) < 1e-12


def test_pm_forces_f64_options(gpu, x64):
    """Order-0 gradient, long-range split and a given real density."""
    from jaxpm_amd import pm
    shape = (16, 16, 16)
    r = np.random.default_rng(4)
    pos = lattice(shape) + r.normal(scale=0.7, size=(*shape, 3))
    got = pm.pm_forces(torch.as_tensor(pos, device=gpu), mesh_shape=shape, r_split=1.5, grad_order=0)
    pots = opm.force_potentials(np.fft.fftn(op.cic_paint(np.zeros(shape), pos)), 1.5, order=0)
    ref = np.stack([op.cic_read(p, pos) for p in pots], -1)
    assert rel(got.cpu().numpy(), ref) < 1e-12
    rho = r.normal(size=shape)
    got = pm.pm_forces(torch.as_tensor(pos, device=gpu), delta=torch.as_tensor(rho, device=gpu))
    ref = opm.pm_forces(pos, delta=rho)
    assert rel(got.cpu().numpy(), ref) < 1e-12


def test_f64_is_forward_only(gpu, x64):
    from jaxpm_amd import painting
    pos = torch.zeros((10, 3), dtype=torch.float64, device=gpu, requires_grad=True)
    with pytest.raises(NotImplementedError):
        painting.cic_paint(torch.zeros((8, 8, 8), dtype=torch.float64, device=gpu), pos)


def test_float64_input_without_x64_runs_float32(gpu):
    """With the switch off, float64 input is computed in float32 (JAX's
    default), with a warning the first time."""
    from jaxpm_amd import _convert, config, painting
    assert not config.x64_enabled()
    _convert._warned_f64 = False
    pos = np.random.default_rng(5).uniform(0, 8, (100, 3))
    with warnings.catch_warnings(record=True) as wl:
        warnings.simplefilter("always")
        out = painting.cic_paint(torch.zeros((8, 8, 8), device=gpu), pos)
    assert out.dtype == torch.float32
    assert any("jax_enable_x64" in str(w.message) for w in wl)


@pytest.mark.parametrize("shape,n", [((16, 16, 16), 131072), ((33, 17, 70), 140000), ((1, 50, 33), 131073),
                                     ((2, 2, 2), 150000), ((48, 40, 31), 262144)])
def test_sorted_paint_f64(gpu, x64, shape, n):
    """The paint of many particles (tile sort and LDS windows, several chunks
    a tile): ragged tiles, axes of one tile and of one cell, positions past
    both ends.  Sums of n deposits of |w| <= 1 in double: below 1e-13 of the
    largest cell, as the atomic form's tests allow."""
    from jaxpm_amd import painting
    print(f"sorted paint f64 {shape} n={n}", flush=True)
    r = np.random.default_rng(6)
    pos = r.uniform(-1.2, 2.1, (n, 3)) * shape
    w = r.uniform(0.5, 1.0, n)
    mesh0 = r.normal(size=shape)
    got = painting.cic_paint(torch.as_tensor(mesh0, device=gpu), torch.as_tensor(pos, device=gpu),
                             torch.as_tensor(w, device=gpu))
    assert rel(got.cpu().numpy(), op.cic_paint(mesh0, pos, w)) < 1e-13


@pytest.mark.parametrize("shape", [(64, 64, 32), (66, 51, 40)])
def test_sorted_relative_paint_and_forces_f64(gpu, x64, shape):
    """Displacements that put corners on, just below and past the mesh ends
    (dropped corners among them), and the forces that paint in their own
    workspace, with one and with three particles per cell."""
    from jaxpm_amd import painting, pm
    print(f"sorted relative f64 {shape}", flush=True)
    r = np.random.default_rng(7)
    disp = r.normal(scale=1.3, size=(*shape, 3))
    disp[0, :, :, 0] = -1e-17
    disp[1, :, :, 1] = np.round(disp[1, :, :, 1])
    disp[2, :, :, 2] = -2.5 * shape[2]
    got = painting.cic_paint_dx(torch.as_tensor(disp, device=gpu))
    assert rel(got.cpu().numpy(), op.cic_paint_dx(disp)) < 1e-13
    got = pm.pm_forces(torch.as_tensor(disp, device=gpu), mesh_shape=shape, paint_absolute_pos=False)
    assert rel(got.cpu().numpy(), opm.pm_forces(disp, mesh_shape=shape, paint_absolute_pos=False)) < 1e-12
    pos = np.concatenate([(lattice(shape) + r.normal(scale=0.7, size=(*shape, 3))).reshape(-1, 3) for _ in range(3)])
    got = pm.pm_forces(torch.as_tensor(pos, device=gpu), mesh_shape=shape)
    assert rel(got.cpu().numpy(), opm.pm_forces(pos, mesh_shape=shape)) < 1e-12


def test_sorted_paint_f64_nonfinite(gpu, x64):
    """Non-finite positions and weights reach the cells that one atomic per
    corner puts them in."""
    from jaxpm_amd import _lib, painting
    print("sorted paint f64 non-finite", flush=True)
    shape, n = (32, 16, 20), 140000
    r = np.random.default_rng(8)
    pos, w = r.uniform(0, 16, (n, 3)), r.uniform(0.5, 1.0, n)
    pos[3, 0], pos[500, 2], pos[7000, 1], w[20000] = np.nan, np.inf, -1e300, np.inf
    p, wt = torch.as_tensor(pos, device=gpu), torch.as_tensor(w, device=gpu)
    got = painting.cic_paint(torch.zeros(shape, dtype=torch.float64, device=gpu), p, wt)
    ref = torch.zeros(shape, dtype=torch.float64, device=gpu)
    _lib.call("jpm_cic_paint_f64", _lib.stream(), *shape, _lib.ptr(p), n, _lib.ptr(wt), 1.0, _lib.ptr(ref), 0)
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(torch.isinf(got), torch.isinf(ref))
    ok = torch.isfinite(ref)
    assert not bool(ok.all()) and rel(got[ok].cpu().numpy(), ref[ok].cpu().numpy()) < 1e-13


def _concentrated(kind, shape, n, r):
    """Positions of which most share few tiles, in many chunks each."""
    pos = r.uniform(0, 1, (n, 3)) * shape
    part = slice(None) if kind == "one tile" else slice(None, None, 2)
    pos[part] = np.minimum(17.0, np.array(shape) / 2) + r.uniform(-3, 9, pos[part].shape)
    return pos


@pytest.mark.parametrize("kind", ["one tile", "half"])
@pytest.mark.parametrize("shape,n", [((40, 33, 64), 131072), ((64, 64, 64), 300001)])
def test_clustered_paint_and_forces_f64(gpu, x64, kind, shape, n):
    """Most particles in the 2^3 tiles that a cluster of 12^3 cells touches, in
    chunks of 1024 and 2048: sums of some 10^3 deposits of at most 1 a cell,
    below 1e-13 of the largest."""
    from jaxpm_amd import painting, pm
    print(f"clustered f64: {kind} {shape} n={n}", flush=True)
    r = np.random.default_rng(11)
    pos = _concentrated(kind, shape, n, r)
    w = r.uniform(0.5, 1.0, n)
    pt = torch.as_tensor(pos, device=gpu)
    got = painting.cic_paint(torch.zeros(shape, dtype=torch.float64, device=gpu), pt, torch.as_tensor(w, device=gpu))
    assert rel(got.cpu().numpy(), op.cic_paint(np.zeros(shape), pos, w)) < 1e-13
    got = pm.pm_forces(pt, mesh_shape=shape)
    assert rel(got.cpu().numpy(), opm.pm_forces(pos, mesh_shape=shape)) < 1e-12


def test_clustered_relative_f64(gpu, x64):
    """Displacements that bring every second particle to one tile."""
    from jaxpm_amd import painting, pm
    shape = (66, 51, 40)
    print(f"clustered relative f64 {shape}", flush=True)
    r = np.random.default_rng(12)
    disp = r.normal(scale=1.3, size=(*shape, 3))
    disp[::2] = r.uniform(18, 30, disp[::2].shape) - lattice(shape)[::2]
    got = painting.cic_paint_dx(torch.as_tensor(disp, device=gpu))
    assert rel(got.cpu().numpy(), op.cic_paint_dx(disp)) < 1e-13
    got = pm.pm_forces(torch.as_tensor(disp, device=gpu), mesh_shape=shape, paint_absolute_pos=False)
    assert rel(got.cpu().numpy(), opm.pm_forces(disp, mesh_shape=shape, paint_absolute_pos=False)) < 1e-12


@pytest.mark.parametrize("shape,n", [((32, 32, 32), 2 ** 17 - 1), ((32, 32, 32), 2 ** 17), ((48, 33, 32), 2 ** 19 - 1),
                                     ((48, 33, 32), 2 ** 19), ((128, 128, 128), 2 ** 18), ((128, 128, 129), 2 ** 18),
                                     ((256, 256, 256), 2 ** 18 - 1), ((256, 256, 256), 2 ** 18), ((1, 512, 700), 2 ** 17),
                                     ((2048, 2048, 1), 2 ** 18), ((2064, 2048, 1), 2 ** 18), ((17, 16, 16), 2 ** 20)])
def test_f64_paint_on_each_side_of_its_rules(gpu, x64, shape, n):
    """Counts, particles per cell and tiles on each side of the sort's rules and
    of its passes', against the atomic form: the same deposits in another
    order, up to some 10^4 a cell."""
    from jaxpm_amd import _lib, _ops
    print(f"f64 paint rules {shape} n={n}", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(9)
    pos = (torch.rand((n, 3), generator=gen, device=gpu, dtype=torch.float64) * 1.5 - 0.2) * \
        torch.tensor(shape, dtype=torch.float64, device=gpu)
    base = torch.randn(shape, generator=gen, device=gpu, dtype=torch.float64)
    got = _ops.paint_f64(base.clone(), pos)
    ref = base.clone()
    _lib.call("jpm_cic_paint_f64", _lib.stream(), *shape, _lib.ptr(pos), n, None, 1.0, _lib.ptr(ref), 0)
    assert float((got - ref).abs().max()) <= 1e-13 * float(ref.abs().max())
