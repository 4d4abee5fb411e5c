"""Boxes whose two equal axes are the transforms' planes and whose sticks have a length without a two-level
kernel: the generic z-stick kernels over few and many sticks a workgroup against the oracle (FP64 to 1e-10,
mixed to 2e-6), the same values for a band alone and in a block, and the time of one band within 1.8 times
that of a box of nearly the same size whose stick length has a two-level kernel."""
import time

import numpy as np
import pytest

from q3_amd import FP64, MIXED
from q3_amd import workloads as W
from q3_amd.planewave import DeviceArray
from tests.helpers import rel_err
from tests.test_gpu_box_axes import _case
from tests.test_gpu_hamiltonian import _applicator, _oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("axes,alat,ecut,box", [((1.75, 1, 1), 7.0, 40.0, (50, 30, 30)), ((0.7, 1, 1), 7.0, 40.0, (20, 30, 30)),
                                                ((1.25, 1, 1), 7.0, 25.0, (27, 24, 24)), ((1, 0.5, 1), 15.0, 30.0, (54, 27, 54))])
def test_bands_alone_and_in_blocks(gpu_context, axes, alat, ecut, box):
    case = _case(axes, alat, ecut)
    assert case.basis.wave_dims == box
    h = _applicator(gpu_context, case)
    psi = W.random_psi(case.kp.kinetic_energy_squared, 23, seed=1)
    block = {p: h.apply_batch(psi, p) for p in (FP64, MIXED)}
    assert rel_err(block[FP64], _oracle(case, psi)) <= 1e-10
    assert rel_err(block[MIXED], block[FP64]) <= 2e-6
    for n in (1, 2, 9):  # (the projector GEMMs may split their sums otherwise)
        assert rel_err(h.apply_batch(psi[:, :n], FP64), block[FP64][:, :n]) <= 1e-13
        assert rel_err(h.apply_batch(psi[:, :n], MIXED), block[FP64][:, :n]) <= 2e-6


def test_time_of_one_band(gpu_context):
    """50 x 30 x 30 (generic sticks) against 54 x 30 x 30 (two-level ones); 2.3 times with 3 workgroups of sticks."""
    best = []
    for axis, box in ((1.75, (50, 30, 30)), (1.9, (54, 30, 30))):
        case = _case((axis, 1, 1), 7.0, 40.0)
        assert case.basis.wave_dims == box
        h = _applicator(gpu_context, case)
        psi = DeviceArray.from_host(gpu_context, W.random_psi(case.kp.kinetic_energy_squared, 1, seed=1))
        out = DeviceArray(gpu_context, 16 * case.kp.npw)
        h.set_projectors(np.zeros((case.kp.npw, 0), np.complex128), np.zeros(0, np.int32), np.zeros(0))
        t = []
        for _ in range(8):  # the first rounds are the warm-up
            gpu_context.synchronize()
            t0 = time.perf_counter()
            for _ in range(200):
                h.apply_device(psi.ptr, out.ptr, 1, FP64)
            gpu_context.synchronize()
            t.append((time.perf_counter() - t0) / 200)
        best.append(min(t))
    print(f"50 x 30 x 30 {1e6 * best[0]:.1f} us, 54 x 30 x 30 {1e6 * best[1]:.1f} us", flush=True)
    assert best[0] <= 1.8 * best[1]
