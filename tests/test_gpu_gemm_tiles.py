"""FP64 complex GEMM: every workgroup tile at the remainders of its rows, columns and K stages, split
and unsplit, the built-in choice, and operands that are only 8-byte aligned, against numpy.
FP64 products err by at most a few eps sqrt(k) of the largest terms: <= 1e-13 of their scale."""
import ctypes

import numpy as np
import pytest

from q3_amd import FP64
from q3_amd._lib import check, lib
from q3_amd.planewave import DeviceArray, zgemm

pytestmark = pytest.mark.gpu

TILES = ["4x4", "4x2", "2x5", "2x4", "2x3", "2x2", "2x1", "1x2"]
# rows / columns one short of, at and past one and two tiles; k around the stages of 8 and 16
SHAPES = [(1, 1, 1), (127, 31, 7), (128, 32, 8), (129, 33, 9), (63, 79, 15), (64, 80, 16), (65, 81, 17), (33, 47, 33),
          (257, 65, 40), (16, 17, 255)]


def _rand(shape, seed):
    rng = np.random.default_rng(seed)
    return np.asfortranarray(rng.standard_normal(shape) + 1j * rng.standard_normal(shape))


def _check(got, want, A, B, C, k):
    scale = np.abs(A).max() * np.abs(B).max() * np.sqrt(k) + np.abs(C).max()
    assert np.abs(got - want).max() <= 1e-13 * scale


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
        zgemm(gpu_context, transa, m, n, k, 0.5, dA, A.shape[0], dB, k + 2, -2.0, dC, m + 1, FP64)
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
                          m, FP64))
    d, shift, raw = keep[2]
    got = d.download(raw.shape, np.float64)[shift:shift + 2 * C.size].view(np.complex128).reshape((m, n), order="F")
    _check(got, want, A, B, C, k)
