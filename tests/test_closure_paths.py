"""Every path of the closure's step (nodes pulled or read from a velocity field, a tile of 16 beads shared by a work-group or
one per wave, the fallback beside them) with a network whose corrections are not zero, force by force."""
import numpy as np
import pytest

from lbm_amd import LBMForce
from lbm_amd.closure import MLPClosure, pairs, stats
from lbm_amd.harness import DeviceParticles
from parity import Setup
from test_closure import mo, network_with
from test_closure_oracle import random_state

pytestmark = pytest.mark.gpu

FRICTION, MASS, DX, DT = 10.0, 100.0, 1.0, 0.01


def walled_setup(n, beads, stencil, temperature=0.0):
    """A random fluid between two solid planes, beads everywhere between them (half-way ones, whose frames tie, first)."""
    rng = np.random.default_rng(beads)
    pos = rng.uniform([0, 0, 0.6], [n, n, n - 1.6], size=(beads, 3))
    pos[:beads//20] = np.floor(pos[:beads//20]) + 0.5
    s = Setup((n, n, n), tau=0.7)
    s.state = random_state(n, rng)
    s.state.reshape(19, n, n*n)[:, [0, n - 1]] = 0.0       # no fluid in the walls
    s.add_particles(pos, mass=MASS, velocities=rng.normal(scale=0.2, size=(beads, 3)))

    def conf(f):
        f.setSolidNodes([i for k in (0, n - 1) for i in range(k*n*n, (k + 1)*n*n)])
        f.setWallScheme(LBMForce.BounceBack)
        f.setFriction(FRICTION)
        f.setTemperature(temperature)
        f.setRandomNumberSeed(11)
        f.setInterpolationStencil(stencil)
    s.configure.append(conf)
    return s, pos


def bounded_network(context):
    """A network with random weights, its bound on the beads' velocities such that a quarter of the beads exceed it; the
    network, the beads' inputs and whether each exceeds the bound."""
    feats, _ = pairs(context)
    net, norm = network_with(np.random.default_rng(3), scale=0.1)
    largest = np.abs(feats[:, 84:87]*np.float32(norm["v_scale"])).max(axis=1)
    bound = float(np.quantile(largest, 0.75)) if len(feats) > 1 else 1e3
    net.setNormalization(**dict(norm, v_bound=bound))
    return net, feats, largest > np.float32(bound)


@pytest.mark.parametrize("n,beads,storage", [(24, 1, LBMForce.FP32), (24, 15, LBMForce.FP32), (24, 17, LBMForce.FP32),
                                             (24, 511, LBMForce.FP32), (24, 511, LBMForce.FP16), (24, 511, LBMForce.BF16),
                                             (24, 511, LBMForce.FP64), (24, 513, LBMForce.FP32), (32, 32768, LBMForce.FP32),
                                             (32, 32769, LBMForce.FP32), (32, 40007, LBMForce.FP16)],
                         ids=["1", "15", "17", "511-pulled", "511-pulled-fp16", "511-pulled-bf16", "511-pulled-fp64",
                              "513-field", "32768-field", "32769-field-per-wave", "40007-field-per-wave"])
def test_forces_of_every_path(n, beads, storage):
    """In distribution the nearest node's force and friction m dx/dt Du, with Du the network's output for the bead's inputs
    (lbm_closure_pairs) turned back from its frame: 5e-3 of the largest correction, the tolerance of the network against
    its emulation, as an input's rounding to FP16 may differ by one place.  Out of it (the bound on the velocity, or a wall
    node among the 27) the Keys force, bit for bit."""
    s, pos = walled_setup(n, beads, LBMForce.Keys)
    keys = s.build(None, storage=storage)
    near = walled_setup(n, beads, LBMForce.NearestNode)[0].build(None, storage=storage)
    net, feats, fast = bounded_network(keys)
    z = np.floor(pos[:, 2] + 0.5).astype(int) % n
    ood = fast | (z <= 1) | (z >= n - 2)
    p, sg = mo.frame_of(pos, DX, (n, n, n))
    du = mo.from_frame(net.forward(feats).astype(np.float64), p, sg)
    for c in (keys, near):
        c.setStepCount(1)
    f_keys, f_near = keys.getForces(), near.getForces()
    net.attach(keys)
    f = keys.getForces()
    assert stats(keys) == (beads - ood.sum(), ood.sum())
    correction = FRICTION*MASS*DX/DT*du
    assert np.array_equal(f[ood], f_keys[ood])
    if (~ood).any():
        largest = np.abs(correction[~ood]).max()
        assert largest > 0.01*np.abs(f_near).max()
        assert np.abs(f - f_near - correction)[~ood].max() <= 5e-3*largest
    if beads > 100:
        assert 0 < ood.sum() < beads


@pytest.mark.parametrize("n,beads", [(24, 300), (24, 900), (32, 33000)], ids=["pulled", "field", "field-per-wave"])
def test_device_steps_with_network_and_fallback_are_those_of_the_host(n, beads):
    """Eight device-resident steps, the network's and the fallback's forces added to the caller's array on the device, against
    the host's steps, which add them themselves (the rounding of positions and velocities over eight steps: 1e-12)."""
    results = []
    for device in (False, True):
        c = walled_setup(n, beads, LBMForce.Keys, temperature=300.0)[0].build(None, storage=LBMForce.FP64)
        net, _, _ = bounded_network(c)
        net.attach(c)
        if device:
            dp = DeviceParticles(c)
            dp.step(8)
            dp.pull()
        else:
            c.step(8)
        network, fallback = stats(c)
        assert network > beads and fallback > beads and network + fallback == 8*beads
        results.append((c.positions, c.velocities, c.getFluidState()))
    (x0, v0, s0), (x1, v1, s1) = results
    assert np.abs(x1 - x0).max() <= 1e-12*n
    assert np.abs(v1 - v0).max() <= 1e-12*np.abs(v0).max()
    assert np.abs(s1 - s0).max() <= 1e-12*np.abs(s0).max()
