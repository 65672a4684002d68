"""The shortcuts of the relative corners (jmod and fold_period of
jaxpm_amd/csrc/tiles.hpp) as the compiler sees them: the header compiled for
the host, in float32 and float64, against the general expressions they stand
for, bit for bit."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

SOURCE = """
#include "tiles.hpp"
namespace jpm { int fail(int code, const char *, ...) { return code; } }
#define EXPORT(T, S)                                                                                       \\
  extern "C" void jmod_##S(long n, const T *x, T L, T *out) {                                              \\
    for (long i = 0; i < n; ++i) out[i] = jpm::jmod(x[i], L);                                              \\
  }                                                                                                        \\
  extern "C" void fold_##S(long n, const T *x, T L, T *out) {                                              \\
    for (long i = 0; i < n; ++i) out[i] = jpm::fold_period(x[i], L);                                       \\
  }
EXPORT(float, float32)
EXPORT(double, float64)
"""


@pytest.fixture(scope="module")
def compiled(tmp_path_factory):
    from jaxpm_amd import build
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        pytest.skip("hipcc not found")
    d = tmp_path_factory.mktemp("fold")
    (d / "fold.hip").write_text(SOURCE)
    subprocess.run([exe, "-x", "hip", "--offload-host-only", "-O3", "-std=c++17", "-fPIC", "-shared",
                    "-ffp-contract=off", f"-I{build.INCLUDE}", f"-I{build.CSRC}", "-o", str(d / "fold.so"),
                    str(d / "fold.hip")], check=True, capture_output=True)
    return ctypes.CDLL(str(d / "fold.so"))


def call(lib, name, x, L):
    t = {np.float32: ctypes.c_float, np.float64: ctypes.c_double}[x.dtype.type]
    f = getattr(lib, f"{name}_{x.dtype.name}")
    f.argtypes = [ctypes.c_long, ctypes.c_void_p, t, ctypes.c_void_p]
    f.restype = None
    out = np.empty_like(x)
    f(x.size, x.ctypes.data, t(L), out.ctypes.data)
    return out


def jmod_general(x, L):
    with np.errstate(invalid="ignore"):
        m = np.fmod(x, L)
    return np.where((m != 0) & (m < 0), m + L, m)


def fold_general(nd, L):
    with np.errstate(invalid="ignore"):
        return nd - np.rint(nd / L) * L


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 9, 16, 17, 100, 192, 1024, 4097, 2 ** 24 + 2, 2 ** 31 - 1])
def test_compiled_shortcuts_are_exact(compiled, dtype, n):
    F = dtype
    L = F(n)
    r = np.random.default_rng(n % 1000)
    x = [(r.uniform(-3, 4, 100000).astype(F) * L).astype(F), r.uniform(-2, 2, 20000).astype(F),
         (r.uniform(-1e-6, 1e-6, 20000).astype(F) + r.integers(-2, 4, 20000).astype(F) * L).astype(F),
         np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1e30, -1e30, np.finfo(F).tiny, -np.finfo(F).tiny], F)]
    for k in (-2, -1.25, -1, -0.75, -0.5, -0.25, 0.25, 0.5, 0.75, 1, 1.25, 1.5, 2):
        up = down = F(k) * L
        for _ in range(6):
            x.append(np.array([up, down], F))
            up, down = np.nextafter(up, F(np.inf)), np.nextafter(down, F(-np.inf))
    x = np.concatenate(x)
    assert x.dtype == F
    for name, general in (("jmod", jmod_general), ("fold", fold_general)):
        want = general(x, L)
        assert want.dtype == F
        assert np.array_equal(call(compiled, name, x, L), want, equal_nan=True), name


def test_a_wrong_threshold_is_caught(compiled):
    """The comparison sees a fold whose shortcut reached past half a period."""
    x = np.linspace(-2, 2, 4001).astype(np.float32) * np.float32(9)
    wrong = np.where(np.abs(x) <= np.float32(0.6) * 9, x, fold_general(x, np.float32(9)))
    assert not np.array_equal(call(compiled, "fold", x, 9.0), wrong)
