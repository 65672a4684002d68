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


@pytest.mark.parametrize("shape", [(64, 64, 64), (100, 100, 100), (65, 65, 65), (17, 17, 17), (128, 128, 128),
                                   (256, 256, 256), (400, 400, 400), (1, 512, 512), (2048, 2048, 1)])
@pytest.mark.parametrize("n", [2 ** 17, 2 ** 18 + 1, 10 ** 6, 2 ** 20, 2 ** 21 + 1, 2 ** 24])
def test_f64_paint_workspace_follows_the_particles(size, shape, n):
    assert size("jpm_cic_paint_f64_workspace_size", *shape, n) <= 64 * n
