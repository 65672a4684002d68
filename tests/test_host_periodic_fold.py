"""The shortcuts of the relative corners (jmod and fold_period in
jaxpm_amd/csrc/tiles.hpp) against the general expressions they stand for, bit
for bit, in float32 NumPy: jnp.remainder as fmod with +L when negative, and
nd - rint(nd / L) L."""
import numpy as np
import pytest

F = np.float32


def jmod_general(x, L):
    with np.errstate(invalid="ignore"):
        m = np.fmod(x, L).astype(F)
    return np.where((m != 0) & (m < 0), (m + L).astype(F), m)


def jmod_short(x, L):
    out = jmod_general(x, L)
    out = np.where((x >= L) & (x < F(2) * L), (x - L).astype(F), out)
    out = np.where((x < 0) & (x > -L), (x + L).astype(F), out)
    return np.where((x >= 0) & (x < L), x, out)


def fold_general(nd, L):
    with np.errstate(invalid="ignore"):
        return (nd - (np.rint((nd / L).astype(F)) * L).astype(F)).astype(F)


def fold_short(nd, L):
    a = np.abs(nd)
    out = fold_general(nd, L)
    out = np.where((a >= F(0.75) * L) & (a <= F(1.25) * L), (nd - np.copysign(L, nd)).astype(F), out)
    return np.where(a <= F(0.25) * L, nd, out)


def near(v, steps=6):
    out = [F(v)]
    for d in (-np.inf, np.inf):
        u = F(v)
        for _ in range(steps):
            u = np.nextafter(u, F(d))
            out.append(u)
    return out


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 9, 16, 17, 100, 192, 255, 1024, 4097, 2 ** 24 + 2, 2 ** 31 - 1])
def test_shortcuts_are_exact(n):
    L = F(n)
    r = np.random.default_rng(n % 1000)
    x = [r.uniform(-3, 4, 200000).astype(F) * L, r.uniform(-2, 2, 50000).astype(F),
         (r.uniform(-1e-6, 1e-6, 50000).astype(F) + r.integers(-2, 4, 50000).astype(F) * L).astype(F),
         F([0, np.inf, -np.inf, np.nan, 1e30, -1e30, 1e-45, -1e-45])]
    for k in (-2, -1.25, -1, -0.75, -0.5, -0.25, 0.25, 0.5, 0.75, 1, 1.25, 1.5, 2):
        x.append(np.array(near(F(k) * L), F))
    x = np.concatenate(x)
    assert np.array_equal(jmod_short(x, L), jmod_general(x, L), equal_nan=True)
    assert np.array_equal(fold_short(x, L), fold_general(x, L), equal_nan=True)
