"""FP32 complex GEMM: every workgroup tile at the remainders of its rows, columns and K stages, split and
unsplit, the built-in choice, and operands that are only 8-byte aligned, against numpy.
Rounding the operands and FP32 sums of up to 300 terms err by about eps sqrt(k) times the terms' rms
each, with eps = 6e-8: <= 1e-6 sqrt(k) times the product of the largest elements."""
import ctypes

import numpy as np
import pytest

from q3_amd import FP64, MIXED
from q3_amd import workloads as W
from q3_amd._lib import check, lib
from q3_amd.planewave import DeviceArray, zgemm
from tests.helpers import kcase, rel_err
from tests.test_gpu_hamiltonian import _applicator

pytestmark = pytest.mark.gpu

TILES = ["4x5", "4x4", "4x2", "2x5", "2x4", "2x2", "2x1", "1x2"]
SHAPES = [(1, 1, 1), (127, 31, 15), (128, 32, 16), (129, 33, 17), (63, 79, 31), (64, 80, 32), (65, 81, 33), (33, 47, 100),
          (257, 65, 40), (16, 17, 255)]


def _rand(shape, seed):
    rng = np.random.default_rng(seed)
    return np.asfortranarray(rng.standard_normal(shape) + 1j * rng.standard_normal(shape))


def _check(got, want, A, B, C, k):
    scale = np.abs(A).max() * np.abs(B).max() * np.sqrt(k)
    assert np.abs(got - want).max() <= 1e-6 * scale + 1e-14 * np.abs(C).max()


@pytest.mark.parametrize("transa", ["N", "C"])
@pytest.mark.parametrize("tile", ["", *(f"{t}/1" for t in TILES), *(f"{t}/3" for t in TILES), *(f"{t}/8" for t in TILES)])
def test_tiles_at_their_remainders(gpu_context, monkeypatch, transa, tile):
    if tile:
        monkeypatch.setenv("Q3X_GEMM_TILE", tile)
    for m, n, k in SHAPES:
        A = _rand((m, k) if transa == "N" else (k, m), m + 3 * k)
        B, C = _rand((k + 2, n), n + 7), _rand((m + 1, n), 11)
        want = 0.5 * ((A if transa == "N" else A.conj().T) @ B[:k]) - 2.0 * C[:m]
        dA, dB, dC = (DeviceArray.from_host(gpu_context, x) for x in (A, B, C))
        zgemm(gpu_context, transa, m, n, k, 0.5, dA, A.shape[0], dB, k + 2, -2.0, dC, m + 1, MIXED)
        got = dC.download((m + 1, n))
        _check(got[:m], want, A, B, C, k)
        np.testing.assert_array_equal(got[m:], C[m:])  # rows past m stay


@pytest.mark.parametrize("transa", ["N", "C"])
@pytest.mark.parametrize("which", [0, 1, 2])
def test_operands_aligned_to_eight_bytes(gpu_context, transa, which):
    m, n, k = 70, 41, 300
    A = _rand((m, k) if transa == "N" else (k, m), 1)
    B, C = _rand((k, n), 2), _rand((m, n), 3)
    want = (A if transa == "N" else A.conj().T) @ B + C
    ptrs, keep = [], []
    for i, x in enumerate((A, B, C)):
        shift = 1 if i == which else 0  # doubles before the matrix
        raw = np.zeros(2 * x.size + 2)
        raw[shift:shift + 2 * x.size] = x.ravel(order="F").view(np.float64)
        d = DeviceArray.from_host(gpu_context, raw)
        keep.append((d, shift, raw))
        ptrs.append(ctypes.c_void_p(d.ptr + 8 * shift))
    check(lib().q3x_zgemm(gpu_context.h, transa.encode(), m, n, k, 1.0, ptrs[0], A.shape[0], ptrs[1], k, 1.0, ptrs[2],
                          m, MIXED))
    d, shift, raw = keep[2]
    got = d.download(raw.shape, np.float64)[shift:shift + 2 * C.size].view(np.complex128).reshape((m, n), order="F")
    _check(got, want, A, B, C, k)


@pytest.mark.parametrize("tile", ["", *(f"{t}/1" for t in TILES), *(f"{t}/0" for t in TILES)])
def test_projector_products(gpu_context, monkeypatch, tile):
    """The complex64 projectors' two products, with columns of odd length."""
    case = kcase(W.small_test_cell(11.0), 0)  # 169 plane waves
    h = _applicator(gpu_context, case)
    for nb in (1, 17, 35):
        psi = W.random_psi(case.kp.kinetic_energy_squared, nb, seed=nb)
        ref = h.apply_batch(psi, FP64)
        if tile:
            monkeypatch.setenv("Q3X_GEMM_TILE", tile)
        assert rel_err(h.apply_batch(psi, MIXED), ref) <= 2e-6
        monkeypatch.delenv("Q3X_GEMM_TILE", raising=False)
