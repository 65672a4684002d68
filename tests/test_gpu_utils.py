"""GPU binned power spectra against the oracle (utils.py:76-151)."""
import numpy as np
import pytest
import torch

from oracle import utils as ou

pytestmark = pytest.mark.gpu


def dev(x):
    return torch.as_tensor(np.asarray(x, np.float32), device="cuda")


CASES = [((32, 32, 32), None, None), ((16, 24, 20), (64., 96., 80.), None), ((12, 12, 12), (12.,) * 3, None),
         ((15, 9, 11), (30., 18., 22.), 0.25), ((32, 32, 64), (100., 100., 200.), 7), ((8, 8, 8), None,
                                                                                      [0.5, 1.0, 1.7, 2.5])]


@pytest.mark.parametrize("shape,box,kedges", CASES)
def test_power_spectrum_auto(gpu, shape, box, kedges):
    """P(k) within 1e-5 relative of the float64 oracle (the float32 FFT is the
    only difference); |k| bins and mode counts identical."""
    from jaxpm_amd import utils
    print(f"pk auto {shape} box={box} kedges={kedges}", flush=True)
    m = np.random.default_rng(40).normal(size=shape).astype(np.float32)
    k, p = utils.power_spectrum(dev(m), box_shape=box, kedges=kedges)
    rk, rp = ou.power_spectrum(m, box_shape=box, kedges=kedges)
    assert k.shape == rk.shape and p.shape == rp.shape
    assert np.array_equal(np.isnan(k), np.isnan(rk))
    ok = ~np.isnan(rk)
    np.testing.assert_allclose(k[ok], rk[ok], rtol=1e-12)
    np.testing.assert_allclose(p.cpu().numpy()[ok], rp[ok], rtol=1e-5)


@pytest.mark.parametrize("shape,box", [((16, 16, 16), (64.,) * 3), ((12, 10, 14), (36., 30., 42.))])
def test_power_spectrum_cross_multipoles(gpu, shape, box):
    from jaxpm_amd import utils
    r = np.random.default_rng(41)
    a = r.normal(size=shape).astype(np.float32)
    b = (0.6 * a + r.normal(size=shape)).astype(np.float32)
    los = (0.3, -1.0, 2.0)
    for mesh2 in (None, b):
        for poles in ([0, 1, 2, 4], 2, [0]):
            print(f"pk {shape} cross={mesh2 is not None} poles={poles}", flush=True)
            k, p = utils.power_spectrum(dev(a), None if mesh2 is None else dev(mesh2), box_shape=box,
                                        multipoles=poles, los=los)
            rk, rp = ou.power_spectrum(a, mesh2, box_shape=box, multipoles=poles, los=los)
            assert p.shape == rp.shape
            np.testing.assert_allclose(k, rk, rtol=1e-12)
            got = p.cpu().numpy()
            np.testing.assert_allclose(got, rp, rtol=1e-5, atol=1e-5 * np.abs(rp).max())


@pytest.mark.parametrize("shape,bins,poles", [((6, 5, 126), 9, [0, 2, 4]), ((5, 3, 127), 400, [0, 1, 2, 3, 4]),
                                              ((4, 6, 128), 700, [0, 2, 4, 6]), ((3, 2, 1), 3, [0, 3]),
                                              ((2, 4, 2), 5, [0, 2]), ((7, 9, 33), 1300, [0, 2])])
def test_power_spectrum_wave_and_slot_edges(gpu, shape, bins, poles):
    """Rows of 63, 64, 65, 1, 2 and 17 modes against waves of 64, mode counts
    that end inside a wave, and slot counts that give a workgroup 4, 2 and 1
    waves.  Within 1e-5 of the largest value, as the float32 transforms are
    the only difference; a bin of few modes has no smaller error."""
    from jaxpm_amd import utils
    r = np.random.default_rng(44)
    a = r.normal(size=shape).astype(np.float32)
    b = (0.6 * a + r.normal(size=shape)).astype(np.float32)
    edges = np.linspace(0.01, 1.02 * np.pi * np.sqrt(3.0), bins)
    los = (0.3, -1.0, 2.0)
    for mesh2 in (None, b):
        print(f"pk edges {shape} bins={bins} poles={poles} cross={mesh2 is not None}", flush=True)
        k, p = utils.power_spectrum(dev(a), None if mesh2 is None else dev(mesh2), kedges=edges, multipoles=poles,
                                    los=los)
        rk, rp = ou.power_spectrum(a, mesh2, kedges=edges, multipoles=poles, los=los)
        got = p.cpu().numpy()
        assert np.array_equal(np.isnan(k), np.isnan(rk)) and np.array_equal(np.isnan(got), np.isnan(rp))
        ok = ~np.isnan(rk)
        np.testing.assert_allclose(k[ok], rk[ok], rtol=1e-12)
        np.testing.assert_allclose(got[:, ok], rp[:, ok], rtol=1e-5, atol=1e-5 * np.abs(rp[:, ok]).max())


def test_transfer_coherence(gpu):
    from jaxpm_amd import utils
    r = np.random.default_rng(42)
    a = r.normal(size=(16, 16, 16)).astype(np.float32)
    b = (a + 0.5 * r.normal(size=a.shape)).astype(np.float32)
    box = (50.,) * 3
    for fn in ("transfer", "coherence"):
        k, t = getattr(utils, fn)(dev(a), dev(b), box)
        rk, rt = getattr(ou, fn)(a, b, box)
        np.testing.assert_allclose(t.cpu().numpy(), rt, rtol=1e-5)
    out = utils.pktranscoh(dev(a), dev(b), box)
    np.testing.assert_allclose(out[3].cpu().numpy(), ou.transfer(a, b, box)[1], rtol=1e-5)
    np.testing.assert_allclose(out[4].cpu().numpy(), ou.coherence(a, b, box)[1], rtol=1e-5)


def test_power_spectrum_256_plane_wave_and_repeatability(gpu):
    """At the benchmark's 256^3 mesh: a single plane wave lands in exactly one
    bin with the analytic power, and repeated calls agree bitwise."""
    from jaxpm_amd import utils
    n, L, m = 256, 1024., 10
    x = torch.arange(n, device="cuda", dtype=torch.float32)
    amp = 3.0
    mesh = (amp * torch.cos(2 * np.pi * m * x / n))[None, None, :].expand(n, n, n).contiguous()
    k, p = utils.power_spectrum(mesh, box_shape=(L,) * 3)
    p = p.cpu().numpy()
    nz = np.nonzero(np.abs(p) > 1e-6 * np.abs(p).max())[0]
    assert len(nz) == 1
    b = nz[0]
    kw = 2 * np.pi * m / L
    # two modes, |X_ortho|^2 = (amp M / 2)^2 / M each, over the bin's mode count
    dig_count = _bin_count(n, L, k, b)
    expect = 2 * (amp * n ** 3 / 2) ** 2 / n ** 3 / dig_count * (L / n) ** 3
    assert abs(k[b] - kw) < 2 * np.pi / L
    np.testing.assert_allclose(p[b], expect, rtol=1e-5)
    r = np.random.default_rng(43)
    g = torch.as_tensor(r.normal(size=(n, n, n)).astype(np.float32), device="cuda")
    _, p1 = utils.power_spectrum(g, box_shape=(L,) * 3)
    _, p2 = utils.power_spectrum(g, box_shape=(L,) * 3)
    assert torch.equal(p1, p2)


def _bin_count(n, L, k, b):
    """Modes in bin b of the default edges, counted on the host in float64
    with the float32 |k| of the reference."""
    f = 2 * np.pi * n / L * np.fft.fftfreq(n)
    ksq = f[:, None, None] ** 2 + f[None, :, None] ** 2 + f[None, None, :] ** 2
    kk = np.sqrt(ksq.astype(np.float32))
    dk = 4 * np.pi / L
    edges = np.arange(dk, np.pi * n / L, dk) + dk / 2
    return int(np.sum(np.digitize(kk.reshape(-1), edges) == b + 1))


@pytest.mark.parametrize("poles", [[0], [0, 0], [0, 1, 2]])
def test_cross_spectrum_of_modes_that_are_not_finite(gpu, poles):
    """A mode of infinite product and its mirror, the conjugate, sum to an
    infinite real and an undefined imaginary part, in the monopole of an
    isotropic call as among other poles; the other bins stay finite."""
    from jaxpm_amd import _ops
    print(f"cross spectrum not finite {poles}", flush=True)
    shape = (16, 12, 20)
    gen = torch.Generator(device="cuda").manual_seed(31)
    s1 = torch.randn((16, 12, 11), generator=gen, device="cuda", dtype=torch.complex64)
    s2 = torch.randn((16, 12, 11), generator=gen, device="cuda", dtype=torch.complex64)
    s1[1, 2, 3] = complex(float("inf"), 1.0)
    s2[1, 2, 3] = complex(1.0, 1.0)
    edges = np.linspace(0.3, 3.0, 10)
    fac = [2 * np.pi] * 3
    out = _ops.power_spectrum_sums(s1, s2, shape, fac, edges, poles, (0.0, 0.0, 1.0)).cpu().numpy()
    k = 2 * np.pi * np.sqrt((1 / 16) ** 2 + (2 / 12) ** 2 + (3 / 20) ** 2)
    hit = int(np.digitize(np.float32(k), edges))
    rest = np.arange(out.shape[1]) != hit
    assert np.isfinite(out[:, rest]).all()
    assert np.isposinf(out[2, hit]) and np.isnan(out[2 + len(poles), hit])
