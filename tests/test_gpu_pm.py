"""GPU parity of FFTs, k-space passes, pm_forces, lpt and linear_field
against the oracle (float64 NumPy restatement of the reference)."""
import numpy as np
import pytest
import torch

from oracle import cosmology as oc
from oracle import pm as opm
from tests.conftest import LPT_SCALE_FACTORS, SIM_CONFIGS

pytestmark = pytest.mark.gpu


def dev(x, dtype=torch.float32):
    return torch.as_tensor(np.asarray(x), device="cuda").to(dtype)


def host(t):
    return t.detach().cpu().numpy()


def rel_err(got, ref):
    return np.abs(np.asarray(got, np.complex128) - ref).max() / max(np.abs(ref).max(), 1e-30)


def lattice(shape):
    return np.stack(np.meshgrid(*[np.arange(s) for s in shape], indexing="ij"), -1).astype(np.float32)


@pytest.mark.parametrize("shape", [(16, 16, 16), (32, 32, 64), (12, 10, 9)])
def test_fft_transforms(gpu, shape):
    from jaxpm_amd import _ops, distributed
    r = np.random.default_rng(20)
    x = r.normal(size=shape).astype(np.float32)
    hk = host(_ops.r2c(dev(x)))
    assert rel_err(hk, np.fft.rfftn(x)) < 2e-6
    back = host(_ops.c2r(dev(hk, torch.complex64), shape)) / x.size
    assert rel_err(back, x) < 2e-6
    full = host(distributed.fft3d(dev(x)))
    assert rel_err(full, np.fft.fftn(x)) < 2e-6
    z = (r.normal(size=shape) + 1j * r.normal(size=shape)).astype(np.complex64)
    assert rel_err(host(distributed.fft3d(dev(z, torch.complex64))), np.fft.fftn(z)) < 2e-6
    # ifft3d of a non-Hermitian spectrum is Re(ifftn), as pifft3d(x).real
    assert rel_err(host(distributed.ifft3d(dev(z, torch.complex64))), np.fft.ifftn(z).real) < 2e-6


@pytest.mark.parametrize("shape,batch", [((2, 2, 4), 1), ((2, 4, 2048), 1), ((1024, 2, 8), 1), ((4, 1024, 4), 1),
                                         ((64, 32, 128), 1), ((8, 16, 32), 3), ((96, 48, 24), 1), ((6, 12, 12), 2),
                                         ((768, 6, 12), 1), ((12, 768, 1536), 1), ((24, 384, 192), 1),
                                         ((96, 96, 96), 2), ((1, 96, 192), 1)])
def test_native_fft_shapes(gpu, shape, batch):
    """Meshes whose axes are powers of two (2 to 1024, 2048 along z) or
    3 * 2^k (6 to 768, 1536 along z) take the library's own transforms,
    radix-3 stages included: batched, against numpy in float64, and the
    inverse of an arbitrary half spectrum against numpy's irfftn."""
    from jaxpm_amd import _ops
    print(f"fft {shape} batch={batch}", flush=True)
    r = np.random.default_rng(27)
    x = r.normal(size=(batch, *shape)).astype(np.float32)
    hk = host(_ops.r2c(dev(x)))
    ref = np.fft.rfftn(x.astype(np.float64), axes=(1, 2, 3))
    assert rel_err(hk, ref) < 3e-6
    z = (r.normal(size=ref.shape) + 1j * r.normal(size=ref.shape)).astype(np.complex64)
    got = host(_ops.c2r(dev(z, torch.complex64), shape))
    want = np.fft.irfftn(z.astype(np.complex128), s=shape, axes=(1, 2, 3)) * np.prod(shape)
    assert rel_err(got, want) < 3e-6


@pytest.mark.parametrize("n", [16, 24, 32, 48, 64, 96, 128])
@pytest.mark.parametrize("nx,batch", [(2, 1), (12, 3), (64, 1)])
def test_plane_transforms(gpu, n, nx, batch):
    """Meshes whose (y, z) planes fit LDS take the z and y passes together:
    against numpy in float64 on both sides of every rule on the plane count,
    and a mesh of a batch has the bits of the mesh alone (planes of 128 take
    one route in the batch of 108 planes and the other alone)."""
    from jaxpm_amd import _ops
    shape = (nx, n, n)
    print(f"plane fft {shape} batch={batch}", flush=True)
    r = np.random.default_rng(31)
    x = r.normal(size=(batch, *shape)).astype(np.float32)
    got = _ops.r2c(dev(x))
    ref = np.fft.rfftn(x.astype(np.float64), axes=(1, 2, 3))
    assert rel_err(host(got), ref) < 3e-6
    z = (r.normal(size=ref.shape) + 1j * r.normal(size=ref.shape)).astype(np.complex64)
    back = _ops.c2r(dev(z, torch.complex64), shape)
    want = np.fft.irfftn(z.astype(np.complex128), s=shape, axes=(1, 2, 3)) * np.prod(shape)
    assert rel_err(host(back), want) < 3e-6
    if nx == 12:
        many = np.concatenate([x, x, x])
        assert torch.equal(_ops.r2c(dev(many))[:batch], got)
        assert torch.equal(_ops.c2r(dev(np.concatenate([z, z, z]), torch.complex64), shape)[:batch], back)
    if batch > 1:
        assert torch.equal(_ops.r2c(dev(x[1])), got[1])
        assert torch.equal(_ops.c2r(dev(z[1], torch.complex64), shape), back[1])


@pytest.mark.parametrize("order,fd,r_split,deconv", [(1, False, 0.0, False), (0, False, 0.0, False),
                                                     (1, True, 0.0, False), (1, False, 1.5, False),
                                                     (1, False, 0.0, True)])
def test_kspace_force_pass(gpu, order, fd, r_split, deconv):
    from jaxpm_amd import _ops
    from oracle import kernels as ok
    shape = (16, 16, 32)
    r = np.random.default_rng(21)
    rho = r.normal(size=shape).astype(np.float32)
    spec = _ops.kspace_force(_ops.r2c(dev(rho)), shape, r_split, 1.0 / rho.size, _ops.kflags(order, fd, deconv))
    phi = host(_ops.c2r(spec, shape, clobber=True))
    kv = ok.fftk(shape)
    pot = np.fft.fftn(rho) * ok.invlaplace_kernel(kv, fd) * ok.longrange_kernel(kv, r_split)
    if deconv:
        pot = pot * ok.cic_compensation(kv)
    for d in range(3):
        ref = np.fft.ifftn(-ok.gradient_kernel(kv, d, order) * pot).real
        assert rel_err(phi[d], ref) < 5e-6, d


@pytest.mark.parametrize("config", SIM_CONFIGS)
@pytest.mark.parametrize("absolute", [True, False])
def test_pm_forces(gpu, config, absolute):
    from jaxpm_amd import pm
    shape, _ = config
    print(f"pm_forces {shape} absolute={absolute}", flush=True)
    r = np.random.default_rng(22)
    disp = r.normal(scale=1.5, size=(*shape, 3)).astype(np.float32)
    pos = lattice(shape) + disp if absolute else disp
    got = host(pm.pm_forces(dev(pos), mesh_shape=shape, paint_absolute_pos=absolute))
    ref = opm.pm_forces(pos, mesh_shape=shape, paint_absolute_pos=absolute)
    assert got.shape == ref.shape
    assert rel_err(got, ref) < 2e-5
    # deterministic paint inside the pipeline agrees and repeats bitwise
    a = pm.pm_forces(dev(pos), mesh_shape=shape, paint_absolute_pos=absolute, deterministic=True)
    b = pm.pm_forces(dev(pos), mesh_shape=shape, paint_absolute_pos=absolute, deterministic=True)
    assert torch.equal(a, b)
    assert rel_err(host(a), ref) < 2e-5


def test_pm_forces_given_delta(gpu):
    from jaxpm_amd import distributed, pm
    shape = (16, 16, 16)
    r = np.random.default_rng(23)
    delta = r.normal(size=shape).astype(np.float32)
    pos = lattice(shape) + r.normal(scale=0.7, size=(*shape, 3)).astype(np.float32)
    ref = opm.pm_forces(pos, delta=delta)
    assert rel_err(host(pm.pm_forces(dev(pos), delta=dev(delta))), ref) < 2e-5
    dk = distributed.fft3d(dev(delta))
    assert rel_err(host(pm.pm_forces(dev(pos), delta=dk)), ref) < 2e-5


def _pair_cosmo(**kw):
    from jaxpm_amd import cosmology as pc
    return pc.Planck18(**kw), oc.Cosmology(**{**dict(Omega_c=0.2607, Omega_b=0.0490, h=0.6766, n_s=0.9665,
                                                      sigma8=0.8102), **kw})


@pytest.mark.parametrize("config", SIM_CONFIGS)
@pytest.mark.parametrize("a", LPT_SCALE_FACTORS)
@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("absolute", [True, False])
def test_lpt(gpu, config, a, order, absolute):
    from jaxpm_amd import pm
    shape, box = config
    print(f"lpt {shape} a={a} order={order} absolute={absolute}", flush=True)
    pcos, ocos = _pair_cosmo()
    r = np.random.default_rng(24)
    ic = r.normal(scale=2.0, size=shape).astype(np.float32)
    particles = lattice(shape) if absolute else None
    got = pm.lpt(pcos, dev(ic), None if particles is None else dev(particles), a=a, order=order)
    ref = opm.lpt(ocos, ic, particles, a=a, order=order)
    for g, rr in zip(got, ref):
        assert rel_err(host(g), rr) < 3e-5


@pytest.mark.parametrize("shape", [(2, 2, 4), (16, 24, 20), (48, 6, 96), (64, 32, 8), (33, 17, 34), (5, 7, 9), (1, 8, 10),
                                   (9, 16, 64)])
@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("absolute", [True, False])
def test_lpt_passes_give_the_bits_of_the_separate_steps(gpu, shape, order, absolute):
    """lpt's fused passes (one forward transform, the shear fields' shared x
    pass, the source formed in the inverse z pass, force and growth products in
    one pass) against the entry points they stand for, one by one: the same
    float operations, so the same bits.  Mesh axes of the library's own
    transforms and of others, an axis of one cell, marches and waves that end
    early."""
    from jaxpm_amd import _ops, pm
    print(f"lpt passes {shape} order={order} absolute={absolute}", flush=True)
    pcos, _ = _pair_cosmo()
    r = np.random.default_rng(28)
    ic = dev(r.normal(size=shape))
    parts = dev(lattice(shape) + r.normal(scale=0.4, size=(*shape, 3))) if absolute else None
    got = pm.lpt(pcos, ic, parts, a=0.1, order=order)
    m = ic.numel()
    pos = parts.reshape(-1, 3) if absolute else torch.zeros((m, 3), device="cuda")

    def force(field):
        phi = _ops.c2r(_ops.kspace_potential(_ops.r2c(field), shape, 0.0, 1.0 / m), shape)
        return _ops.read(_ops.fd4_gradient(phi), pos, relative=not absolute).reshape(*shape, 3)

    c = [float(v) for v in pm.lpt_coefficients(pcos, 0.1, order)]
    f1 = force(ic)
    dx = c[0] * f1
    p, f = c[1] * dx, c[2] * f1
    if order == 2:
        phi6 = _ops.c2r(_ops.kspace_shear6(_ops.r2c(ic), shape, 1.0 / m), shape)
        f2 = force(_ops.lpt2_source(phi6))
        dx2 = c[3] * f2
        dx, p, f = dx + dx2, p + c[4] * dx2, f + c[5] * f2
    for g, ref in zip(got, (dx, p, f)):
        assert g.shape == ref.shape and torch.equal(g, ref)


@pytest.mark.parametrize("shape", [(2, 2, 4), (16, 24, 96), (128, 6, 8), (33, 17, 34), (1, 8, 10)])
@pytest.mark.parametrize("ntab", [2, 37])
def test_linear_field_passes_give_the_bits_of_the_separate_steps(gpu, shape, ntab):
    from jaxpm_amd import _ops
    print(f"linear field passes {shape} ntab={ntab}", flush=True)
    r = np.random.default_rng(29)
    noise, box = dev(r.normal(size=shape)), [3.0 * s for s in shape]
    k = np.linspace(0.05, 1.2, ntab)
    ktab, pktab = dev(k), dev(np.exp(-k))
    got = _ops.linear_field(noise, box, ktab, pktab)
    fk = _ops.kspace_linear_field(_ops.r2c(noise), shape, box, ktab, pktab, 1.0 / noise.numel())
    assert torch.equal(got, _ops.c2r(fk, shape))


def test_linear_field_tabulated(gpu):
    from jaxpm_amd import cosmology as pc
    from jaxpm_amd import pm
    shape, box = (32, 32, 64), (256., 256., 512.)
    k, pk = pc.pk_table(pc.Planck18())
    noise = np.random.default_rng(25).normal(size=shape).astype(np.float32)
    got = host(pm.linear_field(shape, box, pm.TabulatedPk(k, pk), dev(noise)))
    ref = opm.linear_field(shape, box, lambda x: np.interp(x, k, pk), noise)
    assert rel_err(got, ref) < 2e-5
    # a generic callable takes the same path's numbers
    got2 = host(pm.linear_field(shape, box, lambda x: np.interp(x, k, pk), dev(noise)))
    assert rel_err(got2, ref) < 2e-5


def test_make_ode_fn(gpu):
    from jaxpm_amd import ode
    from oracle import ode as oo
    pcos, ocos = _pair_cosmo()
    shape = (16, 16, 16)
    r = np.random.default_rng(26)
    pos = lattice(shape) + r.normal(scale=0.5, size=(*shape, 3)).astype(np.float32)
    vel = r.normal(scale=0.1, size=(*shape, 3)).astype(np.float32)
    dp, dv = ode.make_ode_fn(shape)((dev(pos), dev(vel)), 0.5, pcos)
    rp, rv = oo.make_ode_fn(shape)((pos, vel), 0.5, ocos)
    assert rel_err(host(dp), rp) < 1e-6
    assert rel_err(host(dv), rv) < 2e-5


def test_pm_forces_gradient_matches_finite_differences(gpu):
    """d/dx of <u, pm_forces(x)> through the hand-written adjoints vs float64
    central differences of the oracle along random directions."""
    from jaxpm_amd import pm
    shape = (8, 8, 8)
    r = np.random.default_rng(27)
    pos = (lattice(shape) + r.normal(scale=0.8, size=(*shape, 3))).astype(np.float32)
    u = r.normal(size=(*shape, 3))
    pt = dev(pos).requires_grad_(True)
    (pm.pm_forces(pt, mesh_shape=shape) * dev(u)).sum().backward()
    grad = host(pt.grad).astype(np.float64)
    eps = 1e-5
    for j in range(6):
        d = r.normal(size=pos.shape)
        lp = np.sum(opm.pm_forces(pos + eps * d, mesh_shape=shape) * u)
        lm = np.sum(opm.pm_forces(pos - eps * d, mesh_shape=shape) * u)
        fd = (lp - lm) / (2 * eps)
        an = np.sum(grad * d)
        assert abs(an - fd) < 1e-3 * (abs(fd) + 1e-3), (j, an, fd)


@pytest.mark.parametrize("shape", [(16, 16, 32), (8, 6, 5), (1, 2, 4)])
def test_fd4_stencil_equals_kspace_gradient(gpu, shape):
    """-D_d IFFT[P] == IFFT[-g_d P] (gradient_kernel order 1), and the
    divergence kernel is the stencil's transpose."""
    from jaxpm_amd import _ops
    from oracle import kernels as ok
    r = np.random.default_rng(28)
    phi = r.normal(size=shape).astype(np.float32)
    got = host(_ops.fd4_gradient(dev(phi)))
    kv = ok.fftk(shape)
    for d in range(3):
        ref = np.fft.ifftn(-ok.gradient_kernel(kv, d) * np.fft.fftn(phi)).real
        assert np.abs(got[d] - ref).max() < 2e-5 * max(np.abs(phi).max(), 1.0)
    g3 = r.normal(size=(3, *shape)).astype(np.float32)
    lhs = float(np.sum(got.astype(np.float64) * g3))
    rhs = float(np.sum(phi.astype(np.float64) * host(_ops.fd4_divergence(dev(g3)))))
    assert abs(lhs - rhs) < 1e-4 * (abs(lhs) + 1.0)


def test_kspace_potential(gpu):
    from jaxpm_amd import _ops
    from oracle import kernels as ok
    shape = (16, 12, 20)
    r = np.random.default_rng(29)
    rho = r.normal(size=shape).astype(np.float32)
    pot = host(_ops.c2r(_ops.kspace_potential(_ops.r2c(dev(rho)), shape, 1.2, 1.0 / rho.size), shape))
    kv = ok.fftk(shape)
    ref = np.fft.ifftn(np.fft.fftn(rho) * ok.invlaplace_kernel(kv) * ok.longrange_kernel(kv, 1.2)).real
    assert rel_err(pot, ref) < 5e-6


@pytest.mark.parametrize("absolute", [False, True])
def test_lpt2_of_a_field_at_an_odd_offset(gpu, absolute):
    """Initial conditions that start 4 bytes past an 8-byte boundary give the
    bits of an aligned copy, in the workspace of the shape."""
    from jaxpm_amd import cosmology as pc
    from jaxpm_amd import pm
    shape = (32, 16, 48)
    print(f"lpt2 odd offset {shape} absolute={absolute}", flush=True)
    r = np.random.default_rng(52)
    ic = dev(r.normal(size=shape))
    odd = torch.empty(ic.numel() + 1, device="cuda")[1:].reshape(shape)
    odd.copy_(ic)
    assert odd.data_ptr() % 8 == 4
    parts = dev(r.uniform(0, 16, size=(700, 3))) if absolute else None
    got = pm.lpt(pc.Cosmology(), odd, parts, a=0.1, order=2)
    ref = pm.lpt(pc.Cosmology(), ic, parts, a=0.1, order=2)
    assert all(torch.equal(g, w) for g, w in zip(got, ref))
