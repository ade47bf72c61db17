"""The rows of the population layout: the memory that a lattice takes, and every chunk that the lattice pass may take of its
rows, padded and unpadded, with each storage type."""
import gc

import numpy as np
import pytest
import torch

from lbm_amd import LBMForce
from lbm_amd.batch import Batch
from parity import Setup, equilibrium_state, lockstep
from test_batch import make_replica

pytestmark = pytest.mark.gpu

STORAGE = {"fp16": LBMForce.FP16, "bf16": LBMForce.BF16, "fp32": LBMForce.FP32, "fp64": LBMForce.FP64}
BYTES = {"fp16": 2, "bf16": 2, "fp32": 4, "fp64": 8}
# Rows that end in every way: one chunk and less, exact ones, those that grow by a quarter and by just more, those that idle
# lanes, several chunks.
ROWS = [1, 2, 3, 5, 8, 9, 12, 13, 16, 17, 24, 25, 26, 33, 40, 48, 50, 65, 100]


def free_memory():
    gc.collect()                                # what earlier tests left
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


@pytest.mark.parametrize("storage", list(STORAGE))
@pytest.mark.parametrize("nx", ROWS)
def test_a_lattice_takes_at_most_a_quarter_more_than_its_populations(nx, storage):
    """The device memory of a fluid of about 2 M nodes: two arrays of 19 populations per node, a quarter of it at most for
    rows padded to whole chunks, and 16 MB for the rest (the reductions, allocation granules)."""
    edge = int(round((2e6/nx)**0.5))
    s = Setup((nx, edge, edge), tau=0.7)
    s.build(None, storage=STORAGE[storage]).step(1)     # what the first run of a kernel loads
    before = free_memory()
    context = s.build(None, storage=STORAGE[storage])
    taken = before - free_memory()
    populations = 2*19*nx*edge*edge*BYTES[storage]
    assert 0.9*populations <= taken <= 1.25*populations + 16e6
    del context


def test_a_batch_takes_at_most_a_quarter_more_than_its_populations():
    """As above for replicas of 17 and of 3 nodes along x, which whole chunks would double and grow fivefold."""
    sizes = [(17, 200, 200), (3, 400, 400)]
    replicas = [make_replica(size, 0.7, 0, 1.5, 7, rng_seed=1) for size in sizes]
    Batch(replicas).step(1)
    before = free_memory()
    batch = Batch(replicas)
    taken = before - free_memory()
    nodes = sum(a*b*c for a, b, c in sizes)
    assert taken <= 1.25*2*19*4*nodes + 24*nodes + 32e6
    del batch


@pytest.mark.parametrize("nx", [n for n in ROWS if n > 1])
def test_rows_match_the_oracle(nx):
    """An irregular solid block and reactions on nodes of every touched-mask word, against the FP64 oracle (the tolerance of
    the parity tests)."""
    rng = np.random.default_rng(nx)
    ny, nz = 5, 6
    s = Setup((nx, ny, nz), tau=0.7)
    s.add_particles(rng.uniform(0, [nx, ny, nz], size=(40, 3)), velocities=rng.normal(scale=0.5, size=(40, 3)))

    def conf(f):
        if nx > 2:
            f.setSolidNodes([i + nx*(2 + ny*3) for i in range(nx//2)] + [nx - 1])
            f.setWallScheme(LBMForce.BounceBack)
        f.setBodyAcceleration((0.1, 0.05, -0.02))
        f.setFriction(10.0)
        f.setTemperature(0.0)
        f.setInterpolationStencil(LBMForce.Trilinear)
    s.configure.append(conf)
    worst, _, _ = lockstep(s, 12, check_every=4, storage=LBMForce.FP32)
    assert max(worst.values()) <= 1e-5, worst


def forced_fluid(nx, repeats, storage):
    """Density and velocity after 6 steps of a fluid whose nodes are the same in each of `repeats` periods along x, with a
    body force of 1e-3 lattice units, in lattice units, and its largest population."""
    ny, nz = 5, 3
    rng = np.random.default_rng(nx)
    rho, u = rng.uniform(0.97, 1.03, size=(nz*ny, nx)), rng.uniform(-0.02, 0.02, size=(nz*ny, nx, 3))
    rho, u = np.tile(rho, (1, repeats)), np.tile(u, (1, repeats, 1))
    s = Setup((nx*repeats, ny, nz), tau=0.7)
    s.state = equilibrium_state(rho.size, rho.reshape(-1), u.reshape(-1, 3))

    def conf(f):
        f.setTemperature(0.0)
        f.setBodyAcceleration((10.0, 5.0, -2.0))
    s.configure.append(conf)
    c = s.build(None, storage=storage)
    c.step(6)
    density, velocity = c.getFluidFields()
    shape = (nz*ny, repeats, nx)
    return (density/s.density).reshape(shape), (velocity*0.01).reshape(*shape, 3), np.abs(c.getFluidState()).max()


@pytest.mark.parametrize("storage", ["fp32", "fp64"])
@pytest.mark.parametrize("nx", ROWS)
def test_rows_are_those_of_a_lattice_of_whole_chunks(nx, storage):
    """A periodic fluid against itself repeated along x 32 times, where the rows hold whole chunks: the same bits in every
    period."""
    rho, u, _ = forced_fluid(nx, 1, STORAGE[storage])
    rhos, us, _ = forced_fluid(nx, 32, STORAGE[storage])
    assert np.abs(u).max() > 0.004
    assert np.array_equal(np.broadcast_to(rho, rhos.shape), rhos)
    assert np.array_equal(np.broadcast_to(u, us.shape), us)


@pytest.mark.parametrize("nx", ROWS)
def test_rows_in_half_precision_follow_fp32(nx):
    """The stochastic rounding differs from node to node, so the fluid is compared with FP32's: each step rounds a population
    by at most 2^-10 of the largest one, and ten of them carry a component of the momentum, 19 the density.  A node left out
    of one step would lack the body force's 1e-3.  (BF16 takes the same chunks as FP16.)"""
    rho, u, _ = forced_fluid(nx, 1, LBMForce.FP32)
    rho16, u16, largest = forced_fluid(nx, 1, LBMForce.FP16)
    bound = 6*10*largest*2.0**-10
    assert bound < 1e-3
    assert np.abs(u16 - u).max() <= bound
    assert np.abs(rho16 - rho).max() <= 1.9*bound


@pytest.mark.parametrize("storage", list(STORAGE))
@pytest.mark.parametrize("nx", ROWS)
def test_rows_grouped_in_blocks_give_the_same_bits(nx, storage, monkeypatch):
    """The layout changes no result: rows padded or not by default against rows in blocks of two and four, which are never
    padded, in a fluctuating fluid with beads (FP16 and BF16 round each node by a hash of its index)."""
    rng = np.random.default_rng(nx)
    s = Setup((nx, 8, 6), tau=0.7)
    s.add_particles(rng.uniform(0, [nx, 8, 6], size=(30, 3)), velocities=rng.normal(scale=0.5, size=(30, 3)))

    def conf(f):
        f.setFriction(10.0)
        f.setTemperature(300.0)
        f.setFluidFluctuations(True)
        f.setRandomNumberSeed(3)
        f.setInterpolationStencil(LBMForce.Trilinear)
    s.configure.append(conf)
    results = []
    for block in ("1", "2", "4"):
        monkeypatch.setenv("LBM_AMD_ROW_BLOCK", block)
        c = s.build(None, storage=STORAGE[storage])
        c.step(6)
        results.append((c.getFluidState(), c.positions, c.velocities, *c.getFluidFields()))
    for other in results[1:]:
        for a, b in zip(results[0], other):
            assert np.array_equal(a, b)


def test_many_rows_of_one_node():
    """134 M rows of one node (20 GB of populations): every node gains the body force in a step, so that the momentum is
    their number times 1e-3 lattice units to FP32 storage's resolution, and the mass is theirs.  With 32 threads to a row
    the threads would not be counted in 32 bits."""
    s = Setup((1, 16384, 8200), tau=0.7)

    def conf(f):
        f.setTemperature(0.0)
        f.setBodyAcceleration((0.0, 10.0, 0.0))
    s.configure.append(conf)
    c = s.build(None, storage=LBMForce.FP32)
    c.step(1)
    mass, momentum = c.getFluidTotals()
    n = 16384*8200
    assert abs(mass - n) <= 1e-6*n
    assert abs(momentum[1] - 1e-3*n) <= 2e-6*1e-3*n
    assert np.abs(momentum[[0, 2]]).max() <= 1e-6*1e-3*n
