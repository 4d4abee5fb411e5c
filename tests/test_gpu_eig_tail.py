"""Bisection, vectors and back-transformation of the device eigensolver where they can go wrong: row counts at
the edges of the blocks of 64 that a lane holds, principal minors that vanish at a bisection point, split
tridiagonals, and norms far from one.  All steps are backward stable: eigenvalues to 1e-12 of the norm,
residuals of unit vectors to 1e-11 of it, orthonormality to 1e-11."""
import numpy as np
import pytest

from q3_amd.planewave import DeviceArray, hegv_device

pytestmark = pytest.mark.gpu


def _check(ctx, h, nvec):
    n = len(h)
    dH = DeviceArray.from_host(ctx, np.asfortranarray(h.astype(np.complex128)))
    dS = DeviceArray.from_host(ctx, np.asfortranarray(np.eye(n, dtype=np.complex128)))
    dX = DeviceArray(ctx, 16 * n * nvec)
    w = hegv_device(ctx, n, dH, n, dS, n, nvec, dX, n)
    x = dX.download((n, nvec))
    ref = np.linalg.eigvalsh(h)
    norm = np.abs(ref).max()
    assert np.abs(w - ref[:nvec]).max() <= 1e-12 * norm
    assert np.abs(h @ x - x * w).max() <= 1e-11 * norm
    assert np.abs(x.conj().T @ x - np.eye(nvec)).max() <= 1e-11


def _random(n):
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    return a + a.conj().T


@pytest.mark.parametrize("n", [2, 9, 10, 63, 66, 130, 194, 255, 258, 320, 322, 400, 447, 449, 577, 640, 705, 769, 833])
def test_row_blocks(gpu_context, n):
    _check(gpu_context, _random(n), max(1, min(n, 40)))


@pytest.mark.parametrize("n", [8, 9, 64, 65, 201])
@pytest.mark.parametrize("kind", ["zero_diagonal", "wilkinson", "split", "weak"])
def test_vanishing_minors(gpu_context, n, kind):
    d, e = np.zeros(n), np.ones(n - 1)
    if kind == "wilkinson":  # pairs that agree to rounding
        d = np.abs(np.arange(n) - n // 2).astype(float)
    elif kind == "split":
        e[::3] = 0.0
    elif kind == "weak":
        e[::2] = 1e-30
    _check(gpu_context, np.diag(d) + np.diag(e, 1) + np.diag(e, -1), n)


@pytest.mark.parametrize("scale", [2.0**-300, 2.0**300])
@pytest.mark.parametrize("n", [20, 140])
def test_scaled(gpu_context, n, scale):
    _check(gpu_context, _random(n) * scale, n)
