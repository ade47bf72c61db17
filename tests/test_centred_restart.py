"""Restarts of the centred drag with dense particles on lattices where the solve forms its matrix by rows: the particles are
processed in a node order that each Context sorts for itself, and the results must not depend on it."""
import numpy as np
import pytest

from lbm_amd import LBMForce
from parity import Setup

pytestmark = pytest.mark.gpu


def run_restarted(setup, storage, steps, split, query):
    """The uninterrupted run and one restarted from a checkpoint at step `split`, with the host's positions, velocities and
    step count; query: a force evaluation between steps in the second one only."""
    def result(c):
        return c.positions.copy(), c.velocities.copy(), c.getFluidState(), np.asarray(c.getWallForce())
    first = setup.build(None, storage=storage)
    first.step(split)
    data, host = first.createCheckpoint(), (first.positions.copy(), first.velocities.copy(), first.getStepCount())
    first.step(steps - split)
    second = setup.build(None, storage=storage)
    second.setPositions(host[0])
    second.setVelocities(host[1])
    second.setStepCount(host[2])
    second.loadCheckpoint(data)
    for _ in range(steps - split):
        if query:
            second.getForces()
        second.step(1)
    return result(first), result(second)


@pytest.mark.parametrize("stencil", [LBMForce.Trilinear, LBMForce.Keys], ids=["trilinear", "keys"])
@pytest.mark.parametrize("grid,beads", [((12, 12, 12), 130), ((17, 16, 14), 700)])
def test_restart_with_rows_is_bit_identical(grid, beads, stencil):
    """Beads that change their nodes within the run, so that a Context restarted at step 30 processes them in another order
    than the one that sorted them at its first step: the same bits, with force evaluations between the steps too."""
    rng = np.random.default_rng(beads)
    s = Setup(grid, tau=0.8)
    s.add_particles(rng.uniform(0, grid, size=(beads, 3)), velocities=rng.normal(scale=2.0, size=(beads, 3)))

    def conf(f):
        f.setFriction(5.0)
        f.setTemperature(300.0)
        f.setFluidFluctuations(True)
        f.setRandomNumberSeed(5)
        f.setDragScheme(LBMForce.Centered)
        f.setInterpolationStencil(stencil)
    s.configure.append(conf)
    for query in (False, True):
        first, second = run_restarted(s, LBMForce.FP64, 60, 30, query)
        assert np.abs(first[2]).max() > 0
        for a, b in zip(first, second):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("query", [False, True], ids=["steps", "queries"])
def test_restart_after_a_crowd_dispersed_is_bit_identical(query):
    """A crowd of 90 particles that start their stencils in one cell of 4^3 nodes (of 64 entries), so that the solves begin by
    the spread, and then fly on into the next cells, so that they go by the rows: a Context that never saw the crowd takes
    the same solves as one that did."""
    grid, crowd = (24, 16, 16), 90
    rng = np.random.default_rng(1)
    s = Setup(grid, tau=0.8)
    s.add_particles(rng.uniform(0, grid, size=(60, 3)), velocities=rng.normal(scale=0.2, size=(60, 3)))
    s.add_particles(rng.uniform([5.05, 5.05, 5.05], [8.95, 8.95, 8.95], size=(crowd, 3)),
                    velocities=np.tile([8.0, 0.0, 0.0], (crowd, 1)))

    def conf(f):
        f.setFriction(0.5)
        f.setTemperature(300.0)
        f.setRandomNumberSeed(5)
        f.setDragScheme(LBMForce.Centered)
        f.setInterpolationStencil(LBMForce.Keys)
    s.configure.append(conf)
    first, second = run_restarted(s, LBMForce.FP64, 60, 36, query)
    assert np.abs(first[2]).max() > 0
    for a, b in zip(first, second):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("stencil", [LBMForce.Trilinear, LBMForce.ThreePoint, LBMForce.Keys],
                         ids=["trilinear", "threepoint", "keys"])
@pytest.mark.parametrize("grid,beads", [((12, 12, 12), 130), ((13, 7, 9), 301)], ids=["rows", "spread"])
def test_restart_keeps_the_wall_force(grid, beads, stencil):
    """Between walls: the wall force of a restarted run, with the reactions of the beads whose stencils reach the walls, is
    bit-identical too, with the solve by rows and, on axes of fewer than 12 nodes, by the spread."""
    rng = np.random.default_rng(beads)
    nx, ny, nz = grid
    s = Setup(grid, tau=0.8)
    s.add_particles(rng.uniform(0, grid, size=(beads, 3)), velocities=rng.normal(scale=2.0, size=(beads, 3)))

    def conf(f):
        f.setSolidNodes([i for k in (0, nz - 1) for i in range(k*nx*ny, (k + 1)*nx*ny)])
        f.setWallScheme(LBMForce.BounceBack)
        f.setFriction(5.0)
        f.setTemperature(300.0)
        f.setFluidFluctuations(True)
        f.setRandomNumberSeed(5)
        f.setDragScheme(LBMForce.Centered)
        f.setInterpolationStencil(stencil)
    s.configure.append(conf)
    first, second = run_restarted(s, LBMForce.FP64, 60, 30, False)
    assert np.abs(first[3]).max() > 0
    for a, b in zip(first, second):
        assert np.array_equal(a, b)
