"""The times that lbm_profile_fused and lbm_batch_profile_fused record are those of the lattice pass alone."""
import ctypes

import numpy as np
import pytest

from lbm_amd import LBMForce, _lib
from lbm_amd.batch import Batch
from lbm_amd.harness import DeviceParticles
from parity import Setup
from test_batch import make_replica, uneven_replicas

pytestmark = pytest.mark.gpu


def timed_pass(ctx, dp, steps):
    """The median of the recorded passes (ms) of `steps` steps in one call, and their number."""
    lib = ctx.lib
    _lib.check(lib, lib.lbm_profile_fused(ctx.handle, 1, None, None))
    dp.step(steps)
    launches, count = (ctypes.c_float*steps)(), ctypes.c_int()
    _lib.check(lib, lib.lbm_profile_fused_launches(ctx.handle, launches, steps, ctypes.byref(count)))
    _lib.check(lib, lib.lbm_profile_fused(ctx.handle, 0, None, None))
    return sorted(launches)[steps//2], count.value


def test_the_recorded_pass_holds_no_particle_work():
    """A 16^3 lattice, whose pass takes some 5 us, in a System of one million particles that the fluid does not see, whose
    update moves 150 MB: the recorded pass is that of a System of one particle, within a factor of three."""
    passes = []
    for particles in (1, 1000000):
        s = Setup((16, 16, 16), tau=0.7)
        s.add_particles(np.zeros((particles, 3)), coupled=False)
        ctx = s.build()
        dp = DeviceParticles(ctx)
        dp.step(12)
        median, count = timed_pass(ctx, dp, 12)
        assert count == 12
        passes.append(median)
    assert 0 < passes[1] <= 3*passes[0]


def test_the_recorded_pass_of_a_batch_holds_no_particle_work():
    """The same with one million beads at rest in a replica of 16^3, which leave the fluid at rest too."""
    passes = []
    for beads in (1, 1000000):
        replica = make_replica((16, 16, 16), 0.7, 1, 0.0, 7, stencil=LBMForce.NearestNode, fluct=False)
        replica.velocities = np.zeros((beads, 3))
        if beads > 1:
            replica.positions = np.random.default_rng(1).uniform(0, 16, size=(beads, 3))
            replica.masses = np.full(beads, 100.0)
            for i in range(1, beads):
                replica.force.addParticle(i)
        batch = Batch([replica])
        batch.step(10)
        batch.profileFused(True)
        batch.step(10)
        total, count = batch.profileFused(False)
        assert count == 10
        passes.append(total/count)
    assert 0 < passes[1] <= 3*passes[0]


def test_profiled_steps_are_the_others_bits():
    """A batch stepped with recording on and off, and a lattice, against runs that never recorded."""
    runs = []
    for profile in (False, True):
        batch = Batch(uneven_replicas())
        batch.step(3)
        if profile:
            batch.profileFused(True)
        batch.step(8)
        if profile:
            batch.profileFused(False)
        batch.step(13)
        rng = np.random.default_rng(1)
        s = Setup((20, 9, 12), tau=0.7)
        s.add_particles(rng.uniform(0, [20, 9, 12], size=(300, 3)), velocities=rng.normal(size=(300, 3)))

        def conf(f):
            f.setFriction(10.0)
            f.setTemperature(300.0)
            f.setFluidFluctuations(True)
            f.setRandomNumberSeed(9)
            f.setInterpolationStencil(LBMForce.Trilinear)
        s.configure.append(conf)
        ctx = s.build()
        dp = DeviceParticles(ctx)
        dp.step(3)
        if profile:
            timed_pass(ctx, dp, 8)
        else:
            dp.step(8)
        dp.step(5)
        fields = [a for r in range(4) for a in batch.getFluidFields(r)]
        runs.append([*fields, *(a for pair in batch.getParticles() for a in pair), *dp.pull(), ctx.getFluidState()])
    for a, b in zip(*runs):
        assert np.array_equal(a, b)
