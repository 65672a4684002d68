"""GPU parity of CIC paint / read and their adjoints against the oracle."""
import numpy as np
import pytest
import torch

from oracle import painting as op

pytestmark = pytest.mark.gpu


def dev(x):
    return torch.as_tensor(np.asarray(x), dtype=torch.float32, device="cuda")


def host(t):
    return t.detach().cpu().numpy().astype(np.float64)


def lattice(shape):
    return np.stack(np.meshgrid(*[np.arange(s) for s in shape], indexing="ij"), -1).astype(np.float32)


def close(got, ref, rel=2e-6):
    """FP32 sums of O(10) deposits: error relative to the largest value."""
    scale = max(np.abs(ref).max(), 1.0)
    err = np.abs(got - ref).max() / scale
    assert err < rel, f"max error {err:.3e} (x{scale:.3g})"


@pytest.mark.parametrize("shape", [(8, 8, 8), (16, 12, 10), (32, 32, 64)])
def test_paint_absolute(gpu, shape):
    from jaxpm_amd import painting
    print(f"paint absolute {shape}", flush=True)
    r = np.random.default_rng(10)
    n = int(np.prod(shape))
    L = np.array(shape)
    pos = r.uniform(-0.5, 1.5, size=(n, 3)).astype(np.float32) * L  # wrap on both sides
    w = r.normal(size=n).astype(np.float32)
    base = r.normal(size=shape).astype(np.float32)
    got = host(painting.cic_paint(dev(base), dev(pos)))
    close(got, op.cic_paint(base, pos))
    got = host(painting.cic_paint(dev(np.zeros(shape)), dev(pos), weight=dev(w)))
    close(got, op.cic_paint(np.zeros(shape), pos, w))


@pytest.mark.parametrize("shape", [(8, 8, 8), (16, 12, 10), (32, 32, 64)])
def test_paint_relative(gpu, shape):
    from jaxpm_amd import painting
    print(f"paint relative {shape}", flush=True)
    r = np.random.default_rng(11)
    disp = r.normal(scale=3.0, size=(*shape, 3)).astype(np.float32)
    disp[0, 0, 0] = (-1e-9, 0.0, 0.0)   # rounds onto index L in float32: dropped
    got = host(painting.cic_paint_dx(dev(disp)))
    ref = op.cic_paint_dx(disp, dtype=np.float32).astype(np.float64)
    close(got, ref)
    w = r.uniform(0.5, 2.0, size=shape).astype(np.float32)
    close(host(painting.cic_paint_dx(dev(disp), weight=dev(w))), op.cic_paint_dx(disp, w, dtype=np.float32))


def test_paint_weight_shape_error(gpu):
    from jaxpm_amd import painting
    with pytest.raises(ValueError, match="Weight shape must match particle shape"):
        painting.cic_paint_dx(dev(np.zeros((4, 4, 4, 3))), weight=dev(np.ones(5)))


def test_deterministic_paint_is_bitwise_reproducible(gpu):
    from jaxpm_amd import painting
    shape = (32, 32, 32)
    r = np.random.default_rng(12)
    # clustered: every particle in a few cells -> heavy atomic contention
    pos = (16 + r.normal(scale=1.5, size=(32768, 3))).astype(np.float32)
    a = painting.cic_paint(dev(np.zeros(shape)), dev(pos), deterministic=True)
    b = painting.cic_paint(dev(np.zeros(shape)), dev(pos), deterministic=True)
    assert torch.equal(a, b)
    plain = painting.cic_paint(dev(np.zeros(shape)), dev(pos))
    close(host(a), host(plain), rel=1e-5)  # float32 atomics lose ~1e-7 per deposit
    close(host(a), op.cic_paint(np.zeros(shape), pos), rel=5e-7)


def test_paint_large_mass_conservation(gpu):
    """256^3 particles on a 256^3 mesh: sum(mesh) == N, uniform and clustered."""
    from jaxpm_amd import painting
    shape = (256, 256, 256)
    n = 256 ** 3
    g = torch.Generator(device="cuda").manual_seed(1)
    pos = torch.rand((n, 3), generator=g, device="cuda") * 256
    for p in (pos, 128 + 4 * torch.randn((n, 3), generator=g, device="cuda")):
        m = painting.cic_paint(torch.zeros(shape, device="cuda"), p)
        total = m.double().sum().item()
        assert abs(total - n) < 1e-5 * n, total
        md = painting.cic_paint(torch.zeros(shape, device="cuda"), p, deterministic=True)
        assert abs(md.double().sum().item() - n) < 1e-6 * n
        assert (m - md).abs().max().item() < 1e-3 * max(1.0, md.abs().max().item())


def test_paint_128_vs_oracle(gpu):
    from jaxpm_amd import painting
    shape = (128, 128, 128)
    r = np.random.default_rng(13)
    pos = (lattice(shape).reshape(-1, 3) + r.normal(scale=2.0, size=(128 ** 3, 3))).astype(np.float32)
    close(host(painting.cic_paint(dev(np.zeros(shape)), dev(pos))), op.cic_paint(np.zeros(shape), pos))


@pytest.mark.parametrize("shape", [(8, 8, 8), (16, 12, 10), (32, 32, 64)])
def test_read_absolute_and_relative(gpu, shape):
    from jaxpm_amd import painting
    print(f"read {shape}", flush=True)
    r = np.random.default_rng(14)
    mesh = r.normal(size=shape).astype(np.float32)
    n = int(np.prod(shape))
    pos = (r.uniform(-0.5, 1.5, size=(n, 3)) * np.array(shape)).astype(np.float32)
    close(host(painting.cic_read(dev(mesh), dev(pos))), op.cic_read(mesh, pos))
    disp = r.normal(scale=3.0, size=(*shape, 3)).astype(np.float32)
    close(host(painting.cic_read_dx(dev(mesh), dev(disp))), op.cic_read_dx(mesh, disp, dtype=np.float32))
    # lattice read returns node values exactly
    np.testing.assert_array_equal(host(painting.cic_read(dev(mesh), dev(lattice(shape)))), mesh)
    # three meshes in one call
    m3 = r.normal(size=(3, *shape)).astype(np.float32)
    got = host(painting.cic_read(dev(m3), dev(pos)))
    for c in range(3):
        close(got[:, c], op.cic_read(m3[c], pos))


def test_read_paint_transpose_and_position_gradients(gpu):
    from jaxpm_amd import painting
    shape = (16, 16, 16)
    r = np.random.default_rng(15)
    n = 4096
    pos = r.uniform(0, 16, size=(n, 3))
    # keep away from cell faces so that central differences stay on one piece
    frac = pos - np.floor(pos)
    pos = np.floor(pos) + np.clip(frac, 0.01, 0.99)
    pos = pos.astype(np.float32)
    g = r.normal(size=shape).astype(np.float32)
    w = r.normal(size=n).astype(np.float32)
    lhs = (painting.cic_paint(dev(np.zeros(shape)), dev(pos), weight=dev(w)).double() * dev(g).double()).sum()
    rhs = (dev(w).double() * painting.cic_read(dev(g), dev(pos)).double()).sum()
    assert abs(lhs.item() - rhs.item()) < 1e-5 * abs(lhs.item())

    # d/dpos of sum(u * read(g, pos)) against float64 central differences
    u = r.normal(size=n)
    pt = dev(pos).requires_grad_(True)
    (painting.cic_read(dev(g), pt) * dev(u)).sum().backward()
    eps = 1e-4
    dread = np.zeros((n, 3))
    for d in range(3):
        e = np.zeros(3)
        e[d] = eps
        dread[:, d] = (op.cic_read(g, pos + e) - op.cic_read(g, pos - e)) / (2 * eps)
    close(host(pt.grad), dread * u[:, None], rel=1e-4)

    # d/dpos of <paint(pos, w), g>: same derivative with u = w
    pt = dev(pos).requires_grad_(True)
    (painting.cic_paint(dev(np.zeros(shape)), pt, weight=dev(w)) * dev(g)).sum().backward()
    close(host(pt.grad), dread * w[:, None], rel=1e-4)

    # mesh cotangent of read is the paint of the cotangent
    mt = dev(g).requires_grad_(True)
    (painting.cic_read(mt, dev(pos)) * dev(u)).sum().backward()
    close(host(mt.grad), op.cic_paint(np.zeros(shape), pos, u))


def test_compensate_cic(gpu):
    from jaxpm_amd import painting
    r = np.random.default_rng(16)
    f = r.normal(size=(16, 16, 32)).astype(np.float32)
    close(host(painting.compensate_cic(dev(f))), op.compensate_cic(f), rel=5e-6)


# ----------------------------------------------------------- binned paint

BINNED_SHAPES = [(8, 8, 8), (12, 10, 9), (17, 33, 20), (48, 48, 48), (32, 32, 64)]


@pytest.mark.parametrize("shape", BINNED_SHAPES)
@pytest.mark.parametrize("deterministic", [False, True])
def test_binned_paint_absolute(gpu, shape, deterministic):
    from jaxpm_amd import _ops
    print(f"binned abs {shape} det={deterministic}", flush=True)
    r = np.random.default_rng(40)
    n = int(np.prod(shape))
    pos = (r.uniform(-0.5, 1.5, size=(n, 3)) * np.array(shape)).astype(np.float32)
    w = r.normal(size=n).astype(np.float32)
    base = r.normal(size=shape).astype(np.float32)
    m = dev(base)
    _ops.paint(m, dev(pos), deterministic=deterministic)                       # accumulate
    close(host(m), op.cic_paint(base, pos))
    m = dev(np.zeros(shape))
    _ops.paint(m, dev(pos), weight=dev(w), deterministic=deterministic, zero=True)
    close(host(m), op.cic_paint(np.zeros(shape), pos, w))
    # weights not 16-byte aligned (the weight bound's vector loads start
    # after a scalar head)
    wpad = dev(np.concatenate([[0.0], w]).astype(np.float32))
    m = dev(np.zeros(shape))
    _ops.paint(m, dev(pos), weight=wpad[1:], deterministic=deterministic, zero=True)
    close(host(m), op.cic_paint(np.zeros(shape), pos, w))


@pytest.mark.parametrize("shape", BINNED_SHAPES)
def test_binned_paint_relative(gpu, shape):
    from jaxpm_amd import _ops
    r = np.random.default_rng(41)
    disp = r.normal(scale=3.0, size=(*shape, 3)).astype(np.float32)
    disp[0, 0, 0] = (-1e-9, 0.0, 0.0)
    m = dev(np.zeros(shape))
    _ops.paint(m, dev(disp), relative=True, zero=True)
    close(host(m), op.cic_paint_dx(disp, dtype=np.float32))
    m2 = dev(np.zeros(shape))
    _ops.paint(m2, dev(disp), relative=True, zero=True, deterministic=True)
    close(host(m2), op.cic_paint_dx(disp, dtype=np.float32))


@pytest.mark.parametrize("deterministic", [False, True])
def test_binned_paint_three_channels(gpu, deterministic):
    from jaxpm_amd import _ops
    shape = (24, 40, 32)
    r = np.random.default_rng(42)
    n = 30000
    pos = (r.uniform(0, 1, size=(n, 3)) * np.array(shape)).astype(np.float32)
    w3 = r.normal(size=(n, 3)).astype(np.float32)
    got = host(_ops.paint_multi(shape, dev(pos), dev(w3), deterministic=deterministic))
    for c in range(3):
        close(got[c], op.cic_paint(np.zeros(shape), pos, w3[:, c]))
    atomic = host(_ops.paint_multi(shape, dev(pos), dev(w3), method="atomic"))
    close(got, atomic, rel=1e-5)


def test_binned_paint_heavy_tile_and_empty(gpu):
    """One tile holding 50k particles (13 chunks), most tiles empty, and the
    bitwise reproducibility of the fixed-point mode."""
    from jaxpm_amd import _ops
    shape = (64, 64, 64)
    r = np.random.default_rng(43)
    pos = (20 + r.uniform(0, 8, size=(50000, 3))).astype(np.float32)
    pos[:10] = r.uniform(0, 64, size=(10, 3))
    m = dev(np.zeros(shape))
    _ops.paint(m, dev(pos), zero=True)
    close(host(m), op.cic_paint(np.zeros(shape), pos), rel=2e-6)
    a = dev(np.zeros(shape))
    b = dev(np.zeros(shape))
    _ops.paint(a, dev(pos), zero=True, deterministic=True)
    _ops.paint(b, dev(pos), zero=True, deterministic=True)
    assert torch.equal(a, b)
    close(host(a), op.cic_paint(np.zeros(shape), pos), rel=5e-7)
    # no particles: zero mesh / untouched mesh
    z = dev(np.ones(shape))
    _ops.paint(z, dev(np.zeros((0, 3))), zero=True)
    assert float(z.abs().max()) == 0.0


def test_binned_matches_atomic_at_256(gpu):
    from jaxpm_amd import _ops
    shape = (256, 256, 256)
    n = 256 ** 3
    g = torch.Generator(device="cuda").manual_seed(3)
    for p in (torch.rand((n, 3), generator=g, device="cuda") * 256,
              128 + 6 * torch.randn((n, 3), generator=g, device="cuda")):
        a = torch.zeros(shape, device="cuda")
        b = torch.zeros(shape, device="cuda")
        _ops.paint(a, p, method="binned")
        _ops.paint(b, p, method="atomic")
        scale = max(1.0, float(b.abs().max()))
        assert float((a - b).abs().max()) < 2e-5 * scale
        assert abs(a.double().sum().item() - n) < 1e-5 * n


# Over 32768 tiles the tile sort counts and scatters with wavefront-run
# global atomics instead of LDS histograms; a thin mesh reaches that regime
# with few cells (257 x 128 x 1 tiles).
MANY_TILES = (4112, 2048, 1)


@pytest.mark.parametrize("deterministic", [False, True])
def test_binned_paint_over_32768_tiles(gpu, deterministic):
    from jaxpm_amd import _ops
    print(f"binned many tiles det={deterministic}", flush=True)
    shape = MANY_TILES
    r = np.random.default_rng(44)
    n = 400000
    pos = (r.uniform(-0.2, 1.2, size=(n, 3)) * np.array(shape)).astype(np.float32)
    pos[:50000] = (r.normal(size=(50000, 3)) * 3 + np.array([100.0, 300.0, 0.5])).astype(np.float32)
    m = dev(np.zeros(shape))
    _ops.paint(m, dev(pos), zero=True, deterministic=deterministic)
    close(host(m), op.cic_paint(np.zeros(shape), pos), rel=2e-6)
    w3 = r.normal(size=(n, 3)).astype(np.float32)
    got = host(_ops.paint_multi(shape, dev(pos), dev(w3), deterministic=deterministic))
    for c in range(3):
        close(got[c], op.cic_paint(np.zeros(shape), pos, w3[:, c]), rel=2e-6)


@pytest.mark.parametrize("shape", [(16, 16, 16), (17, 33, 20), (64, 32, 48)])
@pytest.mark.parametrize("nc", [1, 3])
def test_sorted_read_matches_direct(gpu, shape, nc):
    """The tile-sorted read gives the direct read's values bit for bit
    (positions wrapping on both sides, a heavy tile split over chunks), and
    matches the oracle."""
    from jaxpm_amd import _ops, painting
    r = np.random.default_rng(60)
    n = 3 * int(np.prod(shape))
    pos = (r.uniform(-0.5, 1.5, size=(n, 3)) * np.array(shape)).astype(np.float32)
    heavy = min(20000, n // 2)
    pos[:heavy] = 3.3 + r.normal(scale=0.4, size=(heavy, 3))
    meshes = r.normal(size=(nc, *shape)).astype(np.float32)
    m = dev(meshes if nc > 1 else meshes[0])
    direct = host(_ops.read(m, dev(pos)))
    srt = host(_ops.read(m, dev(pos), method="sorted"))
    np.testing.assert_array_equal(srt, direct)
    ref = np.stack([op.cic_read(meshes[c], pos) for c in range(nc)], -1)
    close(srt.reshape(n, nc), ref)
    api = host(painting.cic_read(dev(meshes[0]), dev(pos), method="sorted"))
    np.testing.assert_array_equal(api, host(_ops.read(dev(meshes[0]), dev(pos))))


@pytest.mark.parametrize("n", [1, 255, 256, 1025, 131071, 131072, 524287, 524289, 4194303, 4194305])
def test_default_slices_give_the_same_bits(gpu, n):
    """The sort's slice follows the particle count; the fixed-point paint is
    the same bits whatever the slice (against slices of 16384), at the counts
    where the default changes and in slices that end inside a wave."""
    from jaxpm_amd import _lib
    print(f"default slice n={n}", flush=True)
    shape = (48, 33, 20)
    r = np.random.default_rng(60)
    pos = torch.as_tensor((r.uniform(-0.2, 1.2, (n, 3)) * shape).astype(np.float32), device="cuda")
    w = torch.as_tensor(r.normal(size=n).astype(np.float32), device="cuda")
    out = []
    for flags in (_lib.ZERO_MESH, _lib.ZERO_MESH | _lib.tune_flags(slice_code=3)):
        mesh = torch.empty(shape, device="cuda")
        wsb = _lib.size("jpm_cic_paint_binned_workspace_size", *shape, n, 1, flags)
        ws = torch.empty(wsb, dtype=torch.uint8, device="cuda")
        _lib.call("jpm_cic_paint_binned_f32", _lib.stream(), *shape, _lib.ptr(pos), n, _lib.ptr(w), 1.0, 1,
                  _lib.ptr(mesh), flags, _lib.ptr(ws), wsb)
        out.append(mesh)
    assert torch.equal(out[0], out[1])
    m = float(w.double().sum())
    assert abs(float(out[0].double().sum()) - m) < 1e-5 * float(w.double().abs().sum())


@pytest.mark.parametrize("shape", [(3, 4, 1), (4, 3, 2), (2, 2, 3), (5, 1, 7), (1, 1, 64), (6, 5, 65)])
def test_reads_at_the_ends_of_rows(gpu, shape):
    """The reads and position cotangents that load both z corners at once:
    rows of one to three cells, particles in the last cell of a row, on its
    edge and wrapped past it, dropped relative corners.  Against the oracle's
    float32 corners (reads) and float64 gradient, at the other reads'
    tolerance."""
    from jaxpm_amd import _ops
    from oracle import adjoint as oa
    print(f"row ends {shape}", flush=True)
    r = np.random.default_rng(61)
    meshes = r.normal(size=(3, *shape)).astype(np.float32)
    pos = (r.uniform(-0.6, 1.7, (200, 3)) * shape).astype(np.float32)
    pos[:60, 2] = shape[2] - 1 + r.uniform(0, 1, 60).astype(np.float32)
    got = host(_ops.read(dev(meshes), dev(pos)))
    close(got, np.stack([op.cic_read(x, pos, dtype=np.float32) for x in meshes], -1).astype(np.float64))
    grad = host(_ops.grad_pos(dev(meshes[0]), dev(pos)))
    close(grad, oa.cic_read_grad(meshes[0].astype(np.float64), pos.astype(np.float64)))
    m = shape[0] * shape[1] * shape[2]
    disp = r.uniform(-1.5, 1.5, (m, 3)).astype(np.float32)
    disp[::5, 2] = np.float32(-1e-9)
    disp[1::5] = 0
    got = host(_ops.read(dev(meshes), dev(disp), relative=True))
    close(got, np.stack([op.cic_read_dx(x, disp.reshape(*shape, 3), dtype=np.float32).reshape(-1) for x in meshes],
                        -1).astype(np.float64))


@pytest.mark.parametrize("shape", [(16, 16, 16), (20, 33, 17), (5, 40, 64), (48, 16, 9), (1, 1, 4194352)])
def test_paint_cells_in_and_out_of_the_box(gpu, shape):
    """The window index of a floor cell, by its three rules: inside the tile,
    one period away, farther away, on full and partial tiles and on an axis
    whose cells a float cannot number exactly; with lanes that share a cell,
    whose corners go in another order per lane.  Coordinates are multiples of
    1/8 (1/2 on the long axis) and weights small integers, so every sum is
    exact in float32 and the mesh has to equal the float64 sum."""
    from jaxpm_amd import _ops
    print(f"paint cells {shape}", flush=True)
    r = np.random.default_rng(41)
    n = 6000
    L = np.array(shape, dtype=np.float64)
    step = np.where(L > 1e6, 2, 8)
    pos = r.integers(0, (L * step).astype(np.int64), size=(n, 3)) / step
    pos[: n // 3] = pos[0] + r.integers(-8, 9, size=(n // 3, 3)) / step     # many lanes in a few cells
    periods = r.choice([0, 0, 0, 1, -1, 2, -3], size=(n, 3)) * np.where(L > 1e6, 0, 1)
    pos = pos + periods * L
    w = r.integers(-4, 5, size=n).astype(np.float32)
    assert np.array_equal(pos.astype(np.float32), pos)
    ref = np.zeros(shape)
    f = np.floor(pos)
    for o in range(8):
        b = np.array([o & 1, (o >> 1) & 1, (o >> 2) & 1])
        cell = (f + b).astype(np.int64) % np.array(shape)
        wt = np.prod(1.0 - np.abs(pos - (f + b)), axis=1) * w
        np.add.at(ref, tuple(cell.T), wt)
    got = _ops.paint(torch.zeros(shape, device="cuda"), dev(pos), weight=dev(w))
    assert np.array_equal(host(got), ref)
    bad = dev(pos).clone()
    bad[7, 1] = float("nan")
    bad[11, 2] = float("inf")
    assert torch.isnan(_ops.paint(torch.zeros(shape, device="cuda"), bad, weight=dev(w))).any()


@pytest.mark.parametrize("shape", [(16, 16, 16), (32, 32, 48), (40, 24, 20), (48, 17, 33)])
def test_relative_paint_writes_cells_directly(gpu, shape):
    """Relative paints on full and partial tiles: added to a mesh and into a
    fresh one, on tiles of one chunk, of several and of none, with corners that
    float rounding puts one cell outside their window (node + displacement one
    ulp below 16, where adding 1 rounds up to 17); and three weighted channels
    against the atomic kernel.  Tolerances are those of the paints above."""
    from jaxpm_amd import _ops
    print(f"relative paint {shape}", flush=True)
    r = np.random.default_rng(45)
    disp = r.normal(scale=2.0, size=(*shape, 3)).astype(np.float32)
    node = lattice(shape)
    edge = np.nextafter(np.float32(16.0), np.float32(0.0))
    if shape[0] > 16:
        disp[5, :, :, 0] = edge - np.float32(5.0)
        assert np.float32(np.float32(5.0) + disp[5, 0, 0, 0]) == edge
    if shape[0] == 32:   # most particles in one tile, which takes several chunks
        disp[8:] = (np.float32(4.0) + r.uniform(0, 8, size=disp[8:].shape).astype(np.float32)) - node[8:]
    base = r.normal(size=shape).astype(np.float32)
    w = r.normal(size=shape).astype(np.float32)
    ref = op.cic_paint_dx(disp, weight=w, dtype=np.float32)
    close(host(_ops.paint(dev(np.full(shape, 7.0)), dev(disp), weight=dev(w), relative=True, zero=True)), ref)
    close(host(_ops.paint(dev(base), dev(disp), weight=dev(w), relative=True)), base + ref)
    w3 = dev(r.normal(size=(int(np.prod(shape)), 3)))
    close(host(_ops.paint_multi(shape, dev(disp), w3, relative=True)),
          host(_ops.paint_multi(shape, dev(disp), w3, relative=True, method="atomic")), rel=1e-5)


@pytest.mark.parametrize("nc", [1, 3])
@pytest.mark.parametrize("shape,n", [((16, 16, 16), 5000), ((20, 33, 17), 11220), ((32, 32, 48), 40000),
                                     ((64, 48, 40), 61441), ((48, 48, 48), 13000), ((9, 40, 64), 1)])
def test_read_cotangents_from_one_sort(gpu, shape, n, nc):
    """The cotangents of a read from one tile sort: both equal those of the
    paint and of the direct kernel bit for bit, on full and partial tiles, at
    counts on both sides of the rules on particles per cell and per tile, with
    positions out of the box and one that is not finite."""
    from jaxpm_amd import _ops
    print(f"read vjp {shape} n={n} nc={nc}", flush=True)
    r = np.random.default_rng(47)
    pos = (r.uniform(-0.6, 1.7, size=(n, 3)) * np.array(shape)).astype(np.float32)
    pos[: n // 4] = np.floor(pos[: n // 4])
    meshes, cot = dev(r.normal(size=(nc, *shape))), dev(r.normal(size=(n, nc)))
    p = dev(pos)
    gm, gp = _ops.read_vjp(meshes, p, cot)
    assert torch.equal(gm, _ops.paint_multi(shape, p, cot))
    assert torch.equal(gp, _ops.grad_pos(meshes, p, cot=cot))
    p[n // 2, 1] = float("nan")
    gm, gp = _ops.read_vjp(meshes, p, cot)
    direct = _ops.grad_pos(meshes, p, cot=cot)
    assert torch.equal(gp.isnan(), direct.isnan()) and torch.equal(gp.nan_to_num(), direct.nan_to_num())
    assert torch.equal(gm.isnan(), _ops.paint_multi(shape, p, cot).isnan())


@pytest.mark.parametrize("n", [(1 << 22) - 1, (1 << 22) + 4097])
def test_paint_of_many_particles_is_exact(gpu, n):
    """Both sides of the count from which each XCD's slices fill their own part
    of a tile: coordinates are multiples of 1/8 and weights small integers, so
    the mesh has to equal the float64 sum."""
    from jaxpm_amd import _ops
    shape = (40, 33, 50)
    print(f"many particles {n}", flush=True)
    r = np.random.default_rng(48)
    pos = r.integers(0, np.array(shape) * 8, size=(n, 3), dtype=np.int32)
    w = r.integers(-4, 5, size=n).astype(np.float32)
    f, u = pos >> 3, (pos & 7) / 8.0
    ref = np.zeros(int(np.prod(shape)))
    for o in range(8):
        b = np.array([o & 1, (o >> 1) & 1, (o >> 2) & 1])
        c = (f + b) % np.array(shape)
        wt = np.prod(np.where(b, u, 1.0 - u), axis=1) * w
        ref += np.bincount((c[:, 0] * shape[1] + c[:, 1]) * shape[2] + c[:, 2], wt, ref.size)
    p = dev(pos / 8.0)
    got = _ops.paint(torch.empty(shape, device="cuda"), p, weight=dev(w), zero=True)
    assert np.array_equal(host(got).reshape(-1), ref)
    vals = dev(r.normal(size=shape))
    assert torch.equal(_ops.read(vals, p, method="sorted"), _ops.read(vals, p))


@pytest.mark.parametrize("shape,n", [((16, 16, 16), 4096), ((20, 33, 17), 3000), ((64, 48, 40), 60000),
                                     ((32, 32, 32), 0)])
@pytest.mark.parametrize("relative", [False, True])
def test_paint_onto_a_mesh(gpu, shape, n, relative):
    """mesh + paint in one pass has the bits of painting a copy, and leaves the
    mesh; tiles of no, one and several chunks, full and partial."""
    from jaxpm_amd import _ops
    if relative and n != int(np.prod(shape)):
        n = int(np.prod(shape))
    print(f"paint onto {shape} n={n} relative={relative}", flush=True)
    r = np.random.default_rng(49)
    pos = (r.uniform(0, 1, size=(n, 3)) * np.array(shape)).astype(np.float32)
    if shape[0] == 64 and not relative:
        pos[:40000] = 20 + r.uniform(0, 8, size=(40000, 3))
    base, p, w = dev(r.normal(size=shape)), dev(pos), dev(r.normal(size=n))
    keep = base.clone()
    got = _ops.paint_onto(base, p, weight=w, relative=relative)
    assert torch.equal(base, keep)
    assert torch.equal(got, _ops.paint(keep, p, weight=w, relative=relative))


@pytest.mark.parametrize("nc,n", [(1, 6000), (1, 900), (3, 6000)])
def test_read_cotangents_where_floor_plus_one_skips_a_cell(gpu, nc, n):
    """From 2^24 on a coordinate's floor + 1 rounds to itself or two cells up;
    both kernels of the position cotangent take the cell it rounds to."""
    from jaxpm_amd import _ops
    shape = (20, 18, 17)
    print(f"read vjp past 2^24 nc={nc} n={n}", flush=True)
    r = np.random.default_rng(48)
    pos = (r.uniform(0, 1, size=(n, 3)) * np.array(shape)).astype(np.float32)
    far = np.float32([16777216, 16777218, -16777218, -16777216, 16777214.0, 33554430, -33554430, 33554434, 2147483520,
                      -2147483648, 3e9, np.inf, -np.inf])
    for a in range(3):
        at = slice(a * len(far), (a + 1) * len(far))
        pos[at, a] = far
    pos[100:200] = r.choice(far[:6], (100, 3))
    meshes, cot = dev(r.normal(size=(nc, *shape))), dev(r.normal(size=(n, nc)))
    p = dev(pos)
    gp, direct = _ops.read_vjp(meshes, p, cot)[1], _ops.grad_pos(meshes, p, cot=cot)
    assert torch.equal(gp.isnan(), direct.isnan()) and torch.equal(gp.nan_to_num(), direct.nan_to_num())


def _one_ulp_below(shape, edge):
    """Displacements of a lattice at rest but for the plane x = 5, one float
    below ``edge`` (2^-20 below 16, 2^-19 below 32), where adding 1 rounds up:
    its high corner is the cell edge + 1, outside its tile's window, with the
    weight -2^-20; and the mesh that this paints, exactly."""
    disp = np.zeros((*shape, 3), np.float32)
    x = np.nextafter(np.float32(edge), np.float32(0))
    disp[5, :, :, 0] = x - np.float32(5)
    assert np.float32(5) + disp[5, 0, 0, 0] == x and x + np.float32(1) == edge + 1
    mesh = np.ones(shape, np.float32)
    mesh[5] -= 1
    mesh[edge - 1] += np.float32(edge) - x
    mesh[edge + 1] -= np.float32(edge) - x
    return disp, mesh


def test_relative_batch_paints_corners_outside_their_windows(gpu):
    """Corners outside their windows in the second and third simulations of a
    batch: the marks of their tiles and their cells lie past the first's."""
    from jaxpm_amd import integrate
    shapes, edges = [(32, 32, 32), (32, 32, 32), (48, 17, 40), (48, 17, 40)], [None, 16, 32, 16]
    print("relative batch, corners outside windows", flush=True)
    want = [(np.zeros((*s, 3), np.float32), np.ones(s, np.float32)) if e is None else _one_ulp_below(s, e)
            for s, e in zip(shapes, edges)]
    st = integrate.BatchStepper(shapes, [int(np.prod(s)) for s in shapes], relative=True)
    got = host(st.paint(dev(np.concatenate([d.reshape(-1, 3) for d, _ in want])))).reshape(-1)
    assert np.array_equal(got, np.concatenate([m.reshape(-1) for _, m in want]))


def test_relative_paint_of_many_tiles_marks_corners_outside_their_windows(gpu):
    """More tiles than their marks fit in the last chunk's windows: they lie
    behind the overflow mesh."""
    from jaxpm_amd import _ops
    shape = (352, 352, 352)
    print(f"relative paint {shape}, corners outside windows", flush=True)
    disp, mesh = _one_ulp_below(shape, 16)
    d, m = dev(disp), dev(mesh)
    assert torch.equal(_ops.paint(torch.full(shape, 7.0, device="cuda"), d, relative=True, zero=True), m)
    assert torch.equal(_ops.paint(torch.full(shape, 2.0, device="cuda"), d, relative=True), m + 2.0)
    assert torch.equal(_ops.paint(torch.zeros(shape, device="cuda"), d, relative=True, method="atomic"), m)


@pytest.mark.parametrize("nc", [1, 3])
@pytest.mark.parametrize("shape", [(40, 33, 1), (1, 1, 1), (1, 30, 1), (2, 1, 1)])
def test_reads_of_one_z_plane(gpu, shape, nc):
    """Meshes of one cell along z, whose two z corners are that cell: the read
    and its position cotangent against the mesh repeated along z (nz 2), where
    the general corners hold the same values."""
    from jaxpm_amd import _ops
    print(f"one z plane {shape} nc={nc}", flush=True)
    r = np.random.default_rng(53)
    n = 3000
    pos = (r.uniform(-1.2, 2.3, size=(n, 3)) * np.array(shape)).astype(np.float32)
    pos[:500] = np.floor(pos[:500])
    flat = dev(r.normal(size=(nc, *shape)))
    two = flat.expand(nc, *shape[:2], 2).contiguous()
    p, cot = dev(pos), dev(r.normal(size=(n, nc)))
    assert torch.equal(_ops.read(flat, p), _ops.read(two, p))
    assert torch.equal(_ops.grad_pos(flat, p, cot=cot), _ops.grad_pos(two, p, cot=cot))
    f64, p64 = flat.double(), p.double()
    assert torch.equal(_ops.read_f64(f64, p64), _ops.read_f64(two.double(), p64))
