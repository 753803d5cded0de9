"""The block-Jacobi eigensolver at the edges of its blocks: sizes around the
32-wide blocks and 64-wide pairs, odd and even block counts, and matrices
whose rotations are large, tiny, absent or degenerate."""
import ctypes

import numpy as np
import pytest

from mopac_gpu_amd import lib as L

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps
SIZES = (1, 2, 31, 32, 33, 63, 64, 65, 96, 127, 128, 129, 192, 200, 321)


def _matrix(kind, n):
    rng = np.random.Generator(np.random.PCG64(n))
    a = rng.standard_normal((n, n))
    a = 0.5 * (a + a.T)
    if kind == "near_diagonal":
        return np.diag(np.linspace(-30.0, 10.0, n)) + 1.0e-7 * a
    if kind == "degenerate":
        q = np.linalg.qr(a)[0]
        return (q * np.repeat([-2.0, 3.0], [n // 2, n - n // 2])) @ q.T
    if kind == "graded":
        s = 10.0 ** np.linspace(3.0, -9.0, n)
        return a * np.sqrt(s[:, None] * s[None, :])
    if kind == "tiny_coupling":
        return np.diag(np.full(n, 2.5)) + 1.0e-40 * a
    return a


@pytest.mark.parametrize("kind", ("dense", "near_diagonal", "degenerate", "graded", "tiny_coupling"))
@pytest.mark.parametrize("n", SIZES)
def test_eigenpairs(n, kind):
    a = _matrix(kind, n)
    a = 0.5 * (a + a.T)
    v = np.array(a, order="F")
    w = np.zeros(n)
    info = ctypes.c_int(-9)
    L.load().mhip_dsyevd(n, L.ptr(v), n, L.ptr(w), ctypes.byref(info))
    assert info.value == 0
    scale = max(1.0, np.abs(a).max())
    # the sweeps stop with every off-diagonal element below 1e-12 of the
    # largest diagonal one (at most n of them add up in a column), and about
    # a dozen sweeps of n rotations each round by a few eps
    rot = 12 * 4 * n * EPS
    assert np.abs(v.T @ v - np.eye(n)).max() <= rot
    top = max(1.0, np.abs(np.linalg.eigvalsh(a)).max())
    assert np.abs(a @ v - v * w).max() <= (1.0e-12 * np.sqrt(n) + rot) * top
    assert np.abs(w - np.linalg.eigvalsh(a)).max() <= (1.0e-12 * np.sqrt(n) + rot) * max(top, scale)
    assert np.all(np.diff(w) >= 0.0)


@pytest.mark.parametrize("n", (33, 64, 130))
def test_nan_has_a_place_in_the_order(n):
    """A NaN spreads over the levels and vectors; each keeps a place of its own
    (their order is an index), and the next matrix is not touched by it."""
    a = _matrix("dense", n)
    a[0, n - 1] = a[n - 1, 0] = np.nan
    v = np.array(a, order="F")
    w = np.zeros(n)
    info = ctypes.c_int(-9)
    L.load().mhip_dsyevd(n, L.ptr(v), n, L.ptr(w), ctypes.byref(info))
    assert info.value != 0 or np.isnan(v).any()
    test_eigenpairs(n, "dense")


@pytest.mark.parametrize("scale", (1e5, 1e18, 1e20, 1e40, 1e150))
@pytest.mark.parametrize("n", (33, 64, 128, 130, 192))
def test_eigenpairs_of_huge_matrices(n, scale):
    """The rotations' angles start in FP32, whose squares end at 3e38, and the
    padding's entries are about 1e4.  Same bounds as above."""
    a = _matrix("dense", n)
    v = np.array(scale * a, order="F")
    w = np.zeros(n)
    info = ctypes.c_int(-9)
    L.load().mhip_dsyevd(n, L.ptr(v), n, L.ptr(w), ctypes.byref(info))
    assert info.value == 0
    rot = 12 * 4 * n * EPS
    top = np.abs(np.linalg.eigvalsh(a)).max()
    assert np.abs(v.T @ v - np.eye(n)).max() <= rot
    assert np.abs(a @ v - v * (w / scale)).max() <= (1.0e-12 * np.sqrt(n) + rot) * top
    assert np.abs(w / scale - np.linalg.eigvalsh(a)).max() <= (1.0e-12 * np.sqrt(n) + rot) * top
