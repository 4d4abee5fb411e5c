"""Device eigensolver at the edges of its tridiagonalisations: sizes at, below and above the columns and
rows that a wavefront or a workgroup holds and where one kernel takes over from another, and matrices
whose reflectors are partly the identity (diagonal, tridiagonal, block diagonal, rank one).
Householder reduction and the steps after it are backward stable: eigenvalues to 1e-12 of the norm,
residuals and orthonormality to 1e-11."""
import numpy as np
import pytest

from q3_amd.planewave import DeviceArray, hegv_device

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 4, 15, 16, 17, 31, 33, 63, 64, 65, 96, 97, 127, 128, 129, 145, 191, 193, 256, 257, 321, 384, 385,
         511, 512, 513]


def _check(ctx, h):
    n = len(h)
    dH = DeviceArray.from_host(ctx, np.asfortranarray(h))
    dS = DeviceArray.from_host(ctx, np.asfortranarray(np.eye(n, dtype=np.complex128)))
    dX = DeviceArray(ctx, 16 * n * n)
    w = hegv_device(ctx, n, dH, n, dS, n, n, dX, n)
    x = dX.download((n, n))
    norm = np.linalg.norm(h, 2)
    assert np.abs(w - np.linalg.eigvalsh(h)).max() <= 1e-12 * norm
    assert np.abs(h @ x - x * w).max() <= 1e-11 * norm
    assert np.abs(x.conj().T @ x - np.eye(n)).max() <= 1e-11


def _random(n):
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    return a + a.conj().T


@pytest.mark.parametrize("n", SIZES)
def test_sizes(gpu_context, n):
    _check(gpu_context, _random(n))


@pytest.mark.parametrize("n", [5, 32, 70, 100, 130, 300])
@pytest.mark.parametrize("kind", ["diagonal", "tridiagonal", "blocks", "rank_one"])
def test_identity_reflectors(gpu_context, n, kind):
    h = _random(n)
    i = np.arange(n)
    if kind == "diagonal":
        h = np.diag(np.diag(h))
    elif kind == "tridiagonal":
        h = np.where(np.abs(i[:, None] - i) <= 1, h, 0.0)
    elif kind == "blocks":
        h = np.where(i[:, None] // 7 == i // 7, h, 0.0)
    else:
        v = h[:, :1]
        h = v @ v.conj().T / n + np.diag(i.astype(float))
    _check(gpu_context, h)
