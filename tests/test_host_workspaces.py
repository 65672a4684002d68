"""Workspace sizes against what a call is about: the forms that trade memory
for time give way where the memory is out of proportion.  Sizes are computed
on the host; no GPU."""
import os

import pytest


@pytest.fixture
def size():
    from jaxpm_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("libjaxpm_hip.so not built")
    _lib.load()
    return _lib.size


@pytest.mark.parametrize("side,n", [(400, 2 ** 17), (400, 2 ** 18), (400, 10 ** 6 - 1), (320, 2 ** 18),
                                    (256, 2 ** 18 - 1), (257, 2 ** 18)])
def test_sparse_f64_paint_takes_none(size, side, n):
    """Few particles per tile: their atomics beat a window a tile."""
    assert size("jpm_cic_paint_f64_workspace_size", side, side, side, n) == 0


@pytest.mark.parametrize("shape", [(64, 64, 64), (100, 100, 100), (65, 65, 65), (17, 17, 17), (128, 128, 128),
                                   (256, 256, 256), (400, 400, 400), (1, 512, 512), (2048, 2048, 1)])
@pytest.mark.parametrize("n", [2 ** 17, 2 ** 18 + 1, 10 ** 6, 2 ** 20, 2 ** 21 + 1, 2 ** 24])
def test_f64_paint_workspace_follows_the_particles(size, shape, n):
    assert size("jpm_cic_paint_f64_workspace_size", *shape, n) <= 48 * n


@pytest.mark.parametrize("n", [2 ** 27, 2 ** 27 + 1, 2 ** 28, 2 ** 30, 2 ** 32 - 1])
@pytest.mark.parametrize("res", [64, 1000, 1024, 4096])
def test_density_plane_workspace_is_bounded(size, n, res):
    """The records of 2^27 particles and the windows and sums of the plane,
    however many particles there are."""
    tiles = ((res + 63) // 64) ** 2
    windows = (2 ** 27 // 8192 + tiles) * (65 * 65 * 4 + 16)
    assert size("jpm_density_plane_workspace_size", n, res) <= 16 * 2 ** 27 + windows + 8 * res * res + 32 * tiles + 4096


@pytest.mark.parametrize("shape,native", [((256, 256, 256), True), ((64, 96, 48), True), ((512, 512, 512), True),
                                          ((100, 125, 90), False), ((64, 64, 63), False)])
def test_lpt_workspace_holds_what_the_shape_needs(size, shape, native):
    """First order: a half spectrum, three force meshes, a potential.  Second:
    seven more spectra and a second potential, and the six shear meshes only on
    shapes that the library's own FFT does not take."""
    nx, ny, nz = shape
    m, h = nx * ny * nz, nx * ny * (nz // 2 + 1)
    slack = 8 * 256
    assert size("jpm_lpt_workspace_size", *shape, 1) <= 8 * h + 4 * 3 * m + 4 * m + slack
    assert size("jpm_lpt_workspace_size", *shape, 2) <= 8 * 8 * h + 2 * 4 * m + (0 if native else 4 * 6 * m) + slack


def test_counts_below_which_no_workspace_is_asked_for(size):
    """The Python layer's constants are the library's."""
    from jaxpm_amd import _ops
    n = _ops.PAINT_F64_WS_MIN
    assert size("jpm_cic_paint_f64_workspace_size", 50, 50, 50, n) > 0
    n = _ops.DENSITY_PLANE_WS_MIN
    assert size("jpm_density_plane_workspace_size", n, 100) > 0
    for shape in ((1, 1, 1), (16, 16, 16), (50, 50, 50), (256, 256, 256)):
        for less in (1, 1000, 10 ** 5):
            assert size("jpm_cic_paint_f64_workspace_size", *shape, _ops.PAINT_F64_WS_MIN - less) == 0
    for res in (1, 64, 1000, 4096, 20000):
        for less in (1, 1000, 10 ** 5):
            assert size("jpm_density_plane_workspace_size", _ops.DENSITY_PLANE_WS_MIN - less, res) == 0
