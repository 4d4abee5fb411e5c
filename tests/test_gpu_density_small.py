"""Density of small boxes on either side of the lines (points of the box, points times columns) between adding
to rho directly and reducing partial planes, against numpy to 1e-13 (rounding of transforms and of sums of up to 13 columns)."""
import numpy as np
import pytest

from q3_amd import PlanewaveHamiltonianApplicator
from q3_amd import workloads as W
from tests.helpers import rel_err
from tests.test_gpu_plane_quarters import _cubic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,columns", [(24, 1), (24, 12), (24, 13), (36, 3), (36, 4), (40, 1)])
def test_small_boxes(gpu_context, n, columns):
    c, b = _cubic(n)
    kp = b.compute_gk((0.1, -0.2, 0.3))
    psi = W.random_psi(kp.kinetic_energy_squared, columns, seed=n)
    w = np.linspace(0.5, 2.0, columns)
    ref = np.zeros(n ** 3)
    for s in range(columns):
        box = np.zeros(n ** 3, np.complex128)
        box[kp.fft_map] = psi[:, s]
        ref += w[s] * np.abs(np.fft.ifftn(box.reshape(n, n, n), norm="forward").ravel()) ** 2
    h = PlanewaveHamiltonianApplicator(gpu_context, b)
    h.update_potential(W.local_potential(c, b, [W.synthetic_species(0)]))
    h.prepare_kpoint(kp)
    assert rel_err(h.density(psi, w).ravel(), ref) <= 1e-13
