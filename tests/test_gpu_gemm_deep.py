"""FP64 products of few rows and columns and a long k: A B splits k over the chip as A^H B does.  Values against
numpy (<= 1e-13 of the terms' scale, as FP64 sums err by a few eps sqrt(k) of it), and the time of A B within
three times that of the A^H B of the same sizes, which reads the same bytes (on one workgroup it takes a
hundred times as long)."""
import time

import numpy as np
import pytest

from q3_amd import FP64
from q3_amd.planewave import DeviceArray, zgemm

pytestmark = pytest.mark.gpu


def _rand(shape, seed):
    rng = np.random.default_rng(seed)
    return np.asfortranarray(rng.standard_normal(shape) + 1j * rng.standard_normal(shape))


@pytest.mark.parametrize("m,n,k", [(1, 1, 5003), (7, 18, 32361), (33, 31, 4099), (130, 17, 12289), (160, 160, 8191)])
def test_values(gpu_context, m, n, k):
    A, B, C = _rand((m, k), 1), _rand((k, n), 2), _rand((m + 1, n), 3)
    want = 0.5 * (A @ B) - 2.0 * C[:m]
    dA, dB, dC = (DeviceArray.from_host(gpu_context, x) for x in (A, B, C))
    zgemm(gpu_context, "N", m, n, k, 0.5, dA, m, dB, k, -2.0, dC, m + 1, FP64)
    got = dC.download((m + 1, n))
    scale = np.abs(A).max() * np.abs(B).max() * np.sqrt(k) + np.abs(C).max()
    assert np.abs(got[:m] - want).max() <= 1e-13 * scale
    np.testing.assert_array_equal(got[m:], C[m:])  # rows past m stay


def _microseconds(ctx, transa, m, n, k, A, B, C):
    lda = m if transa == "N" else k
    best = np.inf
    for _ in range(6):  # the first round is the warm-up
        ctx.synchronize()
        t = time.perf_counter()
        for _ in range(10):
            zgemm(ctx, transa, m, n, k, 1.0, A, lda, B, k, 0.0, C, m, FP64)
        ctx.synchronize()
        best = min(best, (time.perf_counter() - t) / 10)
    return 1e6 * best


@pytest.mark.parametrize("m,n,k", [(7, 18, 32361), (32, 32, 51627), (160, 160, 51627)])
def test_time_of_a_long_k(gpu_context, m, n, k):
    A, B = DeviceArray.from_host(gpu_context, _rand((m, k), 1)), DeviceArray.from_host(gpu_context, _rand((k, n), 2))
    C = DeviceArray(gpu_context, 16 * m * n)
    t = {op: _microseconds(gpu_context, op, m, n, k, A, B, C) for op in "NC"}
    print(f"{m} x {n} x {k}: A B {t['N']:.1f} us, A^H B {t['C']:.1f} us", flush=True)
    assert t["N"] <= 3 * t["C"]
