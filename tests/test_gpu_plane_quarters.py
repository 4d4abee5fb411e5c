"""The plane kernels' pruned form (occupied sticks and columns in the outer quarters of the plane) and the
general one, on either side of the line: cells whose sphere reaches into the inner blocks of the box
(k outside the first zone shifts it there) and cells whose sphere does not.  The form that runs is the one that
the sphere asks for; H psi and the density of both against numpy, and against the generic kernels where those
hold the plane, FP64 to rounding and mixed to 2e-6."""
import numpy as np
import pytest

from q3_amd import FP64, MIXED, PlanewaveHamiltonianApplicator
from q3_amd import workloads as W
from q3_amd._lib import Q3XError, lib
from q3_amd.planewave import Crystal, PlanewaveBasis
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu


def _cubic(n):
    e = (n - 1) // 2
    alat = 10.0
    ecut = ((e + 0.5) * 2.0 * np.pi / alat) ** 2 / 4.0
    c = Crystal(np.eye(3), alat, np.array([[0.1, 0.2, 0.3]]), np.zeros(1, np.int32))
    b = PlanewaveBasis(c, ecut, 0.0, True, (1, 1, 1))
    assert b.wave_dims == (n, n, n)
    return c, b


def _inner(n, i):
    """Whether index i lies outside the first and last quarter blocks of the kernel's split n = a b."""
    a, b = {24: (6, 4), 30: (6, 5), 32: (8, 4), 48: (8, 6), 60: (10, 6), 72: (9, 8), 75: (15, 5), 96: (12, 8),
            108: (12, 9)}[n]
    q = (a + 3) // 4
    return np.any((i // b >= q) & (i // b < a - q))


@pytest.mark.parametrize("n", [24, 30, 32, 48, 60, 72, 75, 96, 108])
@pytest.mark.parametrize("k", [(0.1, -0.2, 0.3), (0.5, 0.5, 0.0), (1.7, 0.0, 0.4), (-0.3, 2.6, 0.0)])
def test_both_sides_of_the_line(gpu_context, monkeypatch, n, k):
    c, b = _cubic(n)
    kp = b.compute_gk(k)
    i1, i2 = kp.fft_map // (n * n), kp.fft_map // n % n
    inside = not (_inner(n, i1) or _inner(n, i2))
    print(f"n={n} k={k}: {'pruned' if inside else 'general'}", flush=True)
    psi = W.random_psi(kp.kinetic_energy_squared, 3, seed=n)
    v = W.local_potential(c, b, [W.synthetic_species(0)])
    # plane waves outside the box get the kinetic term only
    held = np.flatnonzero(kp.fft_map >= 0)
    w = np.array([0.5, 1.0, 2.0])
    ref = kp.kinetic_energy_squared[:, None] * psi
    rho = np.zeros(n ** 3)
    for s in range(3):
        box = np.zeros(n ** 3, np.complex128)
        box[kp.fft_map[held]] = psi[held, s]
        f = np.fft.ifftn(box.reshape(n, n, n), norm="forward")
        rho += w[s] * np.abs(f.ravel()) ** 2
        ref[held, s] += np.fft.fftn(f * np.reshape(v, (n, n, n)), norm="forward").ravel()[kp.fft_map[held]]

    h = PlanewaveHamiltonianApplicator(gpu_context, b)
    h.update_potential(v)
    h.prepare_kpoint(kp)
    assert lib().q3x_debug_plane_form(h.h, FP64) == (2 if inside else 1)
    assert lib().q3x_debug_plane_form(h.h, MIXED) == (2 if inside else 1)
    got = h.apply_batch(psi, FP64)
    assert rel_err(got, ref) <= 1e-13
    assert rel_err(h.apply_batch(psi, MIXED), ref) <= 2e-6
    if len(held) == kp.npw:
        assert rel_err(h.density(psi, w).ravel(), rho) <= 1e-13
    else:
        with pytest.raises(Q3XError):
            h.density(psi, w)

    monkeypatch.setenv("Q3X_FFT_KERNELS", "generic")
    g = PlanewaveHamiltonianApplicator(gpu_context, b)
    g.update_potential(v)
    try:
        g.prepare_kpoint(kp)
    except Q3XError as e:
        assert "does not fit in LDS" in str(e) and n >= 96
        return
    assert lib().q3x_debug_plane_form(g.h, FP64) == 0
    assert rel_err(got, g.apply_batch(psi, FP64)) <= 1e-13


def test_sizes_fall_on_both_sides(gpu_context):
    _, b = _cubic(48)
    sides = set()
    for k in [(0.1, -0.2, 0.3), (1.7, 0.0, 0.4)]:
        m = b.compute_gk(k).fft_map
        sides.add(bool(_inner(48, m // (48 * 48)) or _inner(48, m // 48 % 48)))
    assert sides == {False, True}
