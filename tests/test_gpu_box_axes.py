"""Boxes with two equal axes in every order: the transforms put the equal axes into the plane.
Against the oracle: FP64 to 1e-10, mixed to 2e-6, projectors and the Gamma trick included; against
the generic kernels to rounding.  The density of boxes with n1 != n2 is refused as ever."""
import numpy as np
import pytest

from q3_amd import FP64, MIXED, PlanewaveHamiltonianApplicator
from q3_amd import workloads as W
from q3_amd._lib import Q3XError
from q3_amd.planewave import Crystal, PlanewaveBasis
from tests.helpers import kcase, rel_err
from tests.test_gpu_hamiltonian import _applicator, _oracle

pytestmark = pytest.mark.gpu

AXES = [(2.0, 1.0, 1.0), (1.0, 2.0, 1.0), (1.0, 1.0, 2.0), (1.0, 1.5, 1.5), (1.5, 1.0, 1.5)]


def _case(axes, alat=7.0, ecut=22.0):
    c = Crystal(np.diag(axes), alat, np.array([[0.1, 0.2, 0.3], [0.6, 0.45, 0.7]]), np.zeros(2, np.int32))
    return kcase(W.Workload(f"axes{axes}{alat}", c, ecut, (1, 1, 1), np.array([[0.15, -0.1, 0.05]]), 5, 3,
                            [W.synthetic_species(0)]), 0)


@pytest.mark.parametrize("axes", AXES)
def test_equal_axes_in_every_order(gpu_context, axes, monkeypatch):
    case = _case(axes)
    d = case.basis.wave_dims
    assert len(set(d)) == 2
    psi = W.random_psi(case.kp.kinetic_energy_squared, 5, seed=3)
    ref = _oracle(case, psi)
    h = _applicator(gpu_context, case)
    assert rel_err(h.apply_batch(psi, FP64), ref) <= 1e-10
    assert rel_err(h.apply_batch(psi, MIXED), ref) <= 2e-6
    monkeypatch.setenv("Q3X_FFT_KERNELS", "generic")
    g = _applicator(gpu_context, case)
    assert rel_err(g.apply_batch(psi, FP64), h.apply_batch(psi, FP64)) <= 1e-13
    if d[0] != d[1]:
        with pytest.raises(Q3XError):
            h.density(psi, np.ones(5))


@pytest.mark.parametrize("axes", AXES[:3])
def test_gamma_trick_on_equal_axes(gpu_context, axes):
    case = _case(axes)
    c = case.w.crystal
    gb = PlanewaveBasis(c, case.w.ecutwfc_ry, 0.0, True, (1, 1, 1), gamma_only=True)
    fb = case.basis
    gk, fk = gb.compute_gk([0, 0, 0]), fb.compute_gk([0, 0, 0])
    psi = gk.random_psi(3, 5)
    full = np.zeros((fk.npw, 3), np.complex128, order="F")
    where = {int(m): i for i, m in enumerate(fk.fft_map)}
    plus = np.array([where[int(m)] for m in gk.fft_map])
    minus = np.array([where[int(m)] for m in gk.minus_fft_map])
    full[minus], full[plus] = psi.conj(), psi
    out = []
    for b, k, x in ((gb, gk, psi), (fb, fk, full)):
        h = PlanewaveHamiltonianApplicator(gpu_context, b)
        h.update_potential(W.local_potential(c, b, case.w.species))
        h.prepare_kpoint(k)
        out.append(h.apply_batch(x, FP64))
    assert rel_err(out[0], out[1][plus]) <= 1e-12
