"""FP64 products of matrices that are only 8-byte aligned: each workgroup tile on either side of the line where it
takes over and at remainders of its rows and columns, against numpy (<= 1e-13 of the terms' scale, as FP64 sums
err by a few eps sqrt(k) of it), and the time of a tall A^H B against that of the aligned product."""
import ctypes
import time

import numpy as np
import pytest

from q3_amd import FP64
from q3_amd._lib import check, lib
from q3_amd.planewave import DeviceArray

pytestmark = pytest.mark.gpu


def _on_device(ctx, shape, seed, shift):
    raw = np.random.default_rng(seed).standard_normal(2 * shape[0] * shape[1] + 2)
    host = raw[shift:shift + 2 * shape[0] * shape[1]].view(np.complex128).reshape(shape, order="F")
    d = DeviceArray.from_host(ctx, raw)
    return host, d, ctypes.c_void_p(d.ptr + 8 * shift)


def _product(ctx, transa, m, n, k, beta, a, b, c):
    check(lib().q3x_zgemm(ctx.h, transa.encode(), m, n, k, 1.0, a, m if transa == "N" else k, b, k, beta, c, m, FP64))


# A B: rounds of 64 x 32 tiles against 1.75 of 128 x 32: 3/3.5, 4/5.25, 4/3.5, 5/5.25, 8/7, 8/7, 9/8.75; A^H B: 64 x 80
# tiles from 3e8 multiply-adds
@pytest.mark.parametrize("transa,m,n,k", [
    ("N", 12287, 128, 9), ("N", 12417, 129, 7), ("N", 16384, 127, 8), ("N", 16385, 128, 5), ("N", 32640, 127, 3),
    ("N", 32641, 128, 17), ("N", 33333, 97, 1),
    ("C", 64, 80, 60000), ("C", 65, 80, 57691), ("C", 65, 80, 57693), ("C", 129, 160, 14537), ("C", 130, 81, 30001),
])
def test_values(gpu_context, transa, m, n, k):
    A, da, pa = _on_device(gpu_context, (m, k) if transa == "N" else (k, m), 1, 1)
    B, db, pb = _on_device(gpu_context, (k, n), 2, 1)
    C, dc, pc = _on_device(gpu_context, (m, n), 3, 1)
    want = (A if transa == "N" else A.conj().T) @ B + C
    _product(gpu_context, transa, m, n, k, 1.0, pa, pb, pc)
    got = dc.download((2 * m * n + 2,), np.float64)[1:-1].view(np.complex128).reshape((m, n), order="F")
    scale = np.abs(A).max() * np.abs(B).max() * np.sqrt(k) + np.abs(C).max()
    assert np.abs(got - want).max() <= 1e-13 * scale


def test_time_of_a_tall_overlap(gpu_context):
    """320 x 80 x 51,627: 1.3 times the aligned product's time on 64 x 80 tiles, 1.9 times on 64 x 32."""
    m, n, k = 320, 80, 51627
    best = []
    for shift in (0, 1):
        _, da, pa = _on_device(gpu_context, (k, m), 1, shift)
        _, db, pb = _on_device(gpu_context, (k, n), 2, shift)
        _, dc, pc = _on_device(gpu_context, (m, n), 3, shift)
        t = []
        for _ in range(8):  # the first rounds are the warm-up
            gpu_context.synchronize()
            t0 = time.perf_counter()
            for _ in range(20):
                _product(gpu_context, "C", m, n, k, 0.0, pa, pb, pc)
            gpu_context.synchronize()
            t.append((time.perf_counter() - t0) / 20)
        best.append(min(t))
    print(f"aligned {1e6 * best[0]:.1f} us, 8-byte aligned {1e6 * best[1]:.1f} us", flush=True)
    assert best[1] <= 1.6 * best[0]
