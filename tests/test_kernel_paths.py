"""Kernels and dispatch branches at the sizes where they can go wrong, against the FP64 oracle or the path that they
replace."""
import numpy as np
import pytest

from lbm_amd import LBMForce
import oracle_lib
from parity import Setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", [1, 77, 20240607])
def test_fp64_normals_match_the_oracle(seed):
    """One step from rest writes nothing but noise: w_q times a sum of 15 normals.  Each normal is within 1e-15 of the
    exact one on either side (radius 7e-16, cosine 7e-16 of at most 6.7), so the populations agree to 1e-14 of the
    largest."""
    s = Setup((9, 5, 64), tau=0.7)

    def conf(f):
        f.setTemperature(300.0)
        f.setFluidFluctuations(True)
        f.setRandomNumberSeed(seed)
    s.configure.append(conf)
    ref, gpu = s.build(oracle_lib.load_oracle()), s.build(None, storage=LBMForce.FP64)
    ref.step(1)
    gpu.step(1)
    a, b = gpu.getFluidState(), ref.getFluidState()
    assert np.abs(b).max() > 0
    assert np.abs(a - b).max() <= 1e-14*np.abs(b).max()
