"""Several contexts solving subspace problems with n > 128 at once, as the workers of a batch do: each of the
multi-workgroup tridiagonalisations exchanges its words with its own workgroups only, so every solve gives the
values of the solve alone, whether it ran to its end or was redone on one workgroup (forced here for every row
count that the redo is built for)."""
import threading

import numpy as np
import pytest

from q3_amd import Context
from q3_amd._lib import lib
from q3_amd.planewave import DeviceArray, hegv_device

pytestmark = pytest.mark.gpu


def _random(n):
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    return a + a.conj().T


def _solve(ctx, h, times=1):
    n = len(h)
    dH = DeviceArray.from_host(ctx, np.asfortranarray(h))
    dS = DeviceArray.from_host(ctx, np.asfortranarray(np.eye(n, dtype=np.complex128)))
    dX = DeviceArray(ctx, 16 * n * n)
    return [(hegv_device(ctx, n, dH, n, dS, n, n, dX, n), dX.download((n, n))) for _ in range(times)]


def _check(h, w, x):
    # Householder reduction and the steps after it are backward stable
    norm = np.linalg.norm(h, 2)
    assert np.abs(w - np.linalg.eigvalsh(h)).max() <= 1e-12 * norm
    assert np.abs(h @ x - x * w).max() <= 1e-11 * norm
    assert np.abs(x.conj().T @ x - np.eye(len(h))).max() <= 1e-11


def test_several_contexts_at_once():
    sizes = [129, 160, 200, 256, 320, 400]
    contexts = [Context(0) for _ in sizes]
    results, errors = [None] * len(sizes), []

    def work(i):
        try:
            results[i] = _solve(contexts[i], _random(sizes[i]), 5)
        except Exception as e:  # reported by the main thread
            errors.append((sizes[i], e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for n, r in zip(sizes, results):
        for w, x in r:
            _check(_random(n), w, x)
    for c in contexts:
        c.close()


@pytest.mark.parametrize("n", [129, 256, 257, 384, 450, 513, 700, 769])
def test_redo_at_every_row_count(gpu_context, n):
    before = lib().q3x_eig_barrier_redos_total()
    lib().q3x_debug_force_barrier_giveups(1)
    try:
        (w, x), = _solve(gpu_context, _random(n))
    finally:
        lib().q3x_debug_force_barrier_giveups(0)
    assert lib().q3x_eig_barrier_redos_total() == before + 1
    _check(_random(n), w, x)
