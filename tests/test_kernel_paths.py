"""Kernels and dispatch branches at the sizes where they can go wrong, against the FP64 oracle or the path that they
replace."""
import os
import sys

import numpy as np
import pytest

from lbm_amd import LBMForce
from lbm_amd.batch import Batch
from lbm_amd.closure import MLPClosure, NUM_INPUTS, stats
from lbm_amd.harness import DeviceParticles
import oracle_lib
from parity import Setup, lockstep
from test_batch import make_replica, run_single

sys.path.insert(0, os.path.join(oracle_lib.ROOT, "oracle"))
import mlp_oracle as mo  # noqa: E402

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


@pytest.mark.parametrize("beads,walls,bonds", [(1, True, False), (256, True, True), (257, True, True), (300, False, True)])
def test_merged_launch_between_steps_is_bit_identical(beads, walls, bonds):
    """Twelve steps in one call (update, reflection and other forces of the steps between in one launch) against twelve
    calls of one step (a launch each); beads beside the walls, so that some are reflected."""
    rng = np.random.default_rng(beads)
    s = Setup((16, 12, 20), tau=0.7)
    s.add_particles(rng.uniform([0, 0, 0.2], [16, 12, 18.8], size=(beads, 3)), velocities=rng.normal(scale=3.0, size=(beads, 3)))

    def conf(f):
        if walls:
            f.setSolidNodes([i for k in (0, 19) for i in range(k*192, (k + 1)*192)])
            f.setWallScheme(LBMForce.BounceBack)
        f.setFriction(10.0)
        f.setTemperature(300.0)
        f.setFluidFluctuations(True)
        f.setRandomNumberSeed(9)
        f.setInterpolationStencil(LBMForce.Trilinear)
    s.configure.append(conf)
    results = []
    for calls, steps in ((1, 12), (12, 1)):
        ctx = s.build()
        dp = DeviceParticles(ctx)
        if bonds:
            dp.setBonds(np.stack([np.arange(beads - 1), np.arange(1, beads)], axis=1), 100.0, 0.5)
        for _ in range(calls):
            dp.step(steps)
        pos, vel = dp.pull()
        results.append((pos, vel, ctx.getFluidState(), ctx.getWallForce()))
    for a, b in zip(*results):
        assert np.array_equal(a, b)
    if walls and beads > 1:
        assert np.abs(results[0][3]).max() > 0


@pytest.mark.parametrize("storage,tolerance", [(LBMForce.FP32, 1e-5), (LBMForce.FP64, 1e-11)], ids=["fp32", "fp64"])
@pytest.mark.parametrize("nx", [1, 15, 16, 17, 31, 32, 33, 48, 65])
def test_row_chunks_match_the_oracle(nx, storage, tolerance):
    """Rows that end at, before and past the chunks of 16 and 32 nodes that the lattice pass takes, with an irregular
    solid block and reactions on nodes of every touched-mask word (tolerances of the parity tests)."""
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
    worst, _, _ = lockstep(s, 12, check_every=4, storage=storage)
    assert max(worst.values()) <= tolerance, worst


@pytest.mark.parametrize("rows", [1, 16, 17, 255, 256, 257, 8192, 8193])
def test_gradients_at_chunk_edges_match_the_oracle(rows):
    """Minibatches at the edges of the tiles of 16 rows, the chunks of 256 and the 32 chunks up to which one launch sums and
    updates (the tolerance of the gradients' parity test: FP16 operands, 2e-2 of a block's norm)."""
    rng = np.random.default_rng(rows)
    net = MLPClosure(seed=7)
    net.setNormalization(u_scale=50.0, v_scale=20.0, out_scale=40.0, u_bound=1e3, v_bound=1e3)
    raw = rng.normal(scale=0.02, size=(rows, NUM_INPUTS)).astype(np.float32)
    target = rng.normal(scale=0.02, size=(rows, 3)).astype(np.float32)
    g, loss = net.gradients(raw, target)
    params = net.getParameters().astype(np.float64)
    x = mo.normalize(raw.astype(np.float64), 50.0, 20.0)
    ref = mo.backward(params, x, target.astype(np.float64)*40.0, emulate16=True)
    assert abs(loss - mo.loss(params, x, target.astype(np.float64)*40.0, emulate16=True)) <= 1e-3*loss
    assert np.linalg.norm(g - ref) <= 2e-2*np.linalg.norm(ref)


@pytest.mark.parametrize("n,beads", [(24, 1), (24, 15), (24, 17), (24, 511), (24, 513), (32, 40000)],
                         ids=["1", "15", "17", "511-pulled", "513-field", "40000-field-per-wave"])
def test_closure_step_with_a_zero_network_is_the_nearest_coupling(n, beads):
    """Every path of the closure's step (nodes pulled, from a velocity field, tiles shared by a work-group or one per wave)
    at the edges of its tiles of 16 beads: with all parameters zero the correction is zero and the run is the nearest-node
    coupling's, bit for bit, between walls and with bounds that no bead exceeds; beads near the walls fall back."""
    rng = np.random.default_rng(beads)
    pos = rng.uniform([0, 0, 4], [n, n, n - 5], size=(beads, 3))
    vel = rng.normal(scale=0.2, size=(beads, 3))
    results = []
    for stencil in (LBMForce.Keys, LBMForce.NearestNode):
        s = Setup((n, n, n), tau=0.7)
        s.add_particles(pos, velocities=vel)

        def conf(f, stencil=stencil):
            f.setSolidNodes([i for k in (0, n - 1) for i in range(k*n*n, (k + 1)*n*n)])
            f.setWallScheme(LBMForce.BounceBack)
            f.setFriction(10.0)
            f.setTemperature(300.0)
            f.setFluidFluctuations(True)
            f.setRandomNumberSeed(11)
            f.setInterpolationStencil(stencil)
        s.configure.append(conf)
        ctx = s.build()
        if stencil == LBMForce.Keys:
            net = MLPClosure(seed=1)
            net.setParameters(np.zeros(11408))
            net.attach(ctx)
        dp = DeviceParticles(ctx)
        dp.step(5)
        out = dp.pull()
        results.append((out[0], out[1], ctx.getFluidState()))
        if stencil == LBMForce.Keys:
            assert stats(ctx) == (5*beads, 0)
    for a, b in zip(*results):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("stencil", [LBMForce.NearestNode, LBMForce.Trilinear, LBMForce.ThreePoint, LBMForce.Keys],
                         ids=["nearest", "trilinear", "threepoint", "keys"])
@pytest.mark.parametrize("grid,open_faces,beads", [((3, 2, 17), False, 37), ((6, 5, 7), True, 37), ((50, 48, 46), False, 4300)],
                         ids=["narrower-than-the-stencil", "open-faces", "in-node-order"])
def test_slots_of_a_group_are_those_formed_per_particle(grid, open_faces, beads, stencil, monkeypatch):
    """The stencil slots that a group's lanes form for each other against those formed once per particle beforehand, bit for
    bit: slots merged on narrow lattices and past open faces, and wrapped at periodic ones, with every other particle
    coupled and a group left over in the last wavefront; enough particles for the node order in one case."""
    rng = np.random.default_rng(beads + stencil)
    s = Setup(grid, tau=0.8)
    for i in range(beads):
        s.add_particles(rng.uniform(0, grid), velocities=rng.normal(scale=0.5, size=(1, 3)), coupled=i % 2 == 0)

    def conf(f):
        if open_faces:
            for face in range(6):
                f.setFaceBoundary(face, LBMForce.Velocity)
            f.setFaceVelocity(LBMForce.ZMax, (0.2, 0.1, 0))
        f.setFriction(10.0)
        f.setTemperature(300.0)
        f.setRandomNumberSeed(5)
        f.setInterpolationStencil(stencil)
    s.configure.append(conf)
    runs = []
    for setup in ("0", "1"):
        monkeypatch.setenv("LBM_AMD_STENCIL_SETUP", setup)
        c = s.build(None, storage=LBMForce.FP32)
        c.step(5)
        runs.append((c.getFluidState(), c.positions.copy(), c.velocities.copy(), c.getForces()))
    assert np.abs(runs[0][0]).max() > 0
    for a, b in zip(*runs):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("stencil", [LBMForce.Trilinear, LBMForce.ThreePoint, LBMForce.Keys],
                         ids=["trilinear", "threepoint", "keys"])
@pytest.mark.parametrize("grid,beads,crowd", [((12, 12, 12), 1, 0), ((12, 13, 15), 70, 0), ((31, 16, 23), 900, 0),
                                              ((24, 20, 14), 40, 60), ((24, 20, 14), 40, 140)],
                         ids=["one", "three-cells", "long-rows", "nearly-full", "overflowing"])
def test_centred_matrix_rows_match_the_spread(grid, beads, crowd, stencil, monkeypatch):
    """The centred drag's solve with the matrix formed by rows against the solve that spreads over the nodes: the smallest
    lattice and those whose last cells take a remainder, particles alone and with some hundred neighbours, a cell of up to 60
    (of 64 entries) and one of 140, after which the solve is repeated by the spread with its bits.  Both stop at a residual
    of 1e-13 of the right-hand side; the matrix' condition is below 100 here, so the forces agree to 1e-11 of the largest.
    Runs are reproducible, also with a check after each iteration."""
    rng = np.random.default_rng(beads + crowd)
    pos = rng.uniform(0, grid, size=(beads, 3))
    pos = np.concatenate([pos, [4.5, 8.5, 4.5] + rng.uniform(-0.4, 0.4, size=(crowd, 3))])
    vel = rng.normal(scale=0.5, size=pos.shape)
    masses = rng.uniform(50, 200, size=len(pos))
    s = Setup(grid, tau=0.8)
    for x, v, m in zip(pos, vel, masses):
        s.add_particles([x], mass=m, velocities=[v])

    def conf(f):
        f.setSolidNodes(list(range(grid[0]*grid[1])))
        f.setWallScheme(LBMForce.BounceBack)
        f.setFriction(10.0)
        f.setTemperature(300.0)
        f.setRandomNumberSeed(5)
        f.setDragScheme(LBMForce.Centered)
        f.setInterpolationStencil(stencil)
    s.configure.append(conf)

    def forces(rows, planned="1"):
        monkeypatch.setenv("LBM_AMD_CG_ROWS", rows)
        monkeypatch.setenv("LBM_AMD_CG_PLANNED", planned)
        c = s.build(None, storage=LBMForce.FP64)
        c.step(3)
        return c.getForces(), c.getFluidState()
    spread, rows = forces("0"), forces("1")
    assert np.abs(spread[0]).max() > 0
    assert np.abs(rows[0] - spread[0]).max() <= 1e-11*np.abs(spread[0]).max()
    for again in (forces("1"), forces("1", planned="0")):
        for a, b in zip(rows, again):
            assert np.array_equal(a, b)
    if crowd > 100:
        for a, b in zip(rows, spread):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("stencil,centred", [(LBMForce.NearestNode, False), (LBMForce.Trilinear, True),
                                             (LBMForce.ThreePoint, False), (LBMForce.ThreePoint, True), (LBMForce.Keys, False),
                                             (LBMForce.Keys, True)],
                         ids=["nearest", "trilinear-centred", "threepoint", "threepoint-centred", "keys", "keys-centred"])
@pytest.mark.parametrize("grid,beads", [((6, 6, 6), 20), ((32, 8, 7), 300), ((33, 7, 9), 900), ((64, 9, 10), 700),
                                        ((67, 11, 6), 1500)])
def test_tile_spread_on_any_periodic_lattice_is_that_of_the_atomics(grid, beads, stencil, centred, monkeypatch):
    """The one-writer spread on lattices whose tiles are narrower than 32 x 4 x 4, down to 3 nodes: rows that share words of the
    touched mask with other tiles, beads that reach back across the periodic faces, solid nodes and a crowd that overflows its
    bin; the reactions are the atomics', bit for bit, over steps that use both sets of bins."""
    rng = np.random.default_rng(beads)
    pos = np.concatenate([rng.uniform(0, grid, size=(beads, 3)), rng.uniform(2.0, 2.3, size=(150, 3))])
    s = Setup(grid, tau=0.8)
    s.add_particles(pos, velocities=rng.normal(scale=0.3, size=pos.shape))

    def conf(f):
        f.setSolidNodes(list(range(grid[0])))
        f.setWallScheme(LBMForce.BounceBack)
        f.setFriction(10.0)
        f.setTemperature(300.0)
        f.setFluidFluctuations(True)
        f.setRandomNumberSeed(5)
        f.setDragScheme(LBMForce.Centered if centred else LBMForce.Explicit)
        f.setInterpolationStencil(stencil)
    s.configure.append(conf)
    runs = []
    for spread in ("atomic", "tiles"):
        monkeypatch.setenv("LBM_AMD_SPREAD", spread)
        c = s.build(None, storage=LBMForce.FP32)
        c.step(5)
        runs.append((c.getFluidState(), c.positions.copy(), c.velocities.copy(), c.getForces()))
    assert np.abs(runs[0][0]).max() > 0
    for a, b in zip(*runs):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("storage", [LBMForce.FP16, LBMForce.FP32, LBMForce.FP64], ids=["fp16", "fp32", "fp64"])
@pytest.mark.parametrize("beads,coupled,fluct", [(255, True, False), (257, True, True), (512, True, False),
                                                 (513, True, False), (513, False, False)])
def test_particles_in_front_of_the_lattice_pass_are_bit_identical(beads, coupled, fluct, storage):
    """Eight steps in one call (the particles' work between the steps in the first work-groups of the pass) against eight
    calls of one step (launches of its own), at the edges of the work-groups of 256 and 512, and for particles that the
    fluid does not see."""
    rng = np.random.default_rng(beads)
    s = Setup((20, 9, 12), tau=0.7)
    s.add_particles(rng.uniform(0, [20, 9, 12], size=(beads, 3)), velocities=rng.normal(size=(beads, 3)), coupled=coupled)

    def conf(f):
        f.setFriction(10.0)
        f.setTemperature(300.0 if fluct else 0.0)
        f.setFluidFluctuations(fluct)
        f.setBodyAcceleration((0.1, 0.05, -0.02))
        f.setRandomNumberSeed(9)
        f.setInterpolationStencil(LBMForce.Trilinear)
    s.configure.append(conf)
    results = []
    for calls, steps in ((1, 8), (8, 1)):
        ctx = s.build(None, storage=storage)
        dp = DeviceParticles(ctx)
        dp.setBonds(np.stack([np.arange(beads - 1), np.arange(1, beads)], axis=1), 100.0, 0.5)
        for _ in range(calls):
            dp.step(steps)
        pos, vel = dp.pull()
        results.append((pos, vel, ctx.getFluidState()))
    for a, b in zip(*results):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("beads", [(0, 0), (0, 1), (200, 55), (256, 1), (1900, 149)])
def test_batch_particles_in_front_of_the_pass_match_single_replicas(beads):
    """The Verlet update in the first work-groups of the batched pass, without particles, at the edges of a work-group of
    256 and of the 8 that are reserved at a time (2,048 particles and one more): the single-lattice runs' bits over replayed
    and single steps."""
    replicas = [make_replica((13, 9, 8), 0.7, beads[0], 2.5, 11, rng_seed=1), make_replica((8, 8, 33), 0.9, beads[1], 1.5, 7, rng_seed=2)]
    batch = Batch(replicas)
    batch.step(23)
    batch.synchronize()
    particles = batch.getParticles()
    for r, replica in enumerate(replicas):
        for a, b in zip(run_single(replica, 23), (*batch.getFluidFields(r), *particles[r])):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("rows", [1, 5, 1506, 1507, 3013, 20000])
def test_normalization_of_the_pairs_is_that_of_the_host(rows):
    """The scales and bounds that training takes from its pairs, with rows at the edges of the work-groups' stride (131,072
    values, 1,506.6 rows), against NumPy in FP64: the sums of at most 1.6 million squares agree to 1e-13, the largest
    magnitudes exactly."""
    rng = np.random.default_rng(rows)
    x = rng.normal(scale=0.02, size=(rows, NUM_INPUTS)).astype(np.float32)
    t = rng.normal(scale=0.3, size=(rows, 3)).astype(np.float32)
    net = MLPClosure(seed=3)
    net.train(x, t, epochs=1, batch=256, lr=1e-4, decay=0.9, seed=3)
    got = net.getNormalization()
    u, v = x[:, 3:84].astype(np.float64), x[:, 84:].astype(np.float64)
    scales = [1/np.sqrt((a*a).mean()) for a in (u, v, t.astype(np.float64))]
    want = dict(u_scale=scales[0], v_scale=scales[1], out_scale=scales[2], u_bound=np.abs(u).max()*scales[0],
                v_bound=np.abs(v).max()*scales[1])
    for name, value in want.items():
        assert abs(got[name] - value) <= 1e-13*value, name


@pytest.mark.parametrize("stencil,grid", [(LBMForce.NearestNode, (20, 9, 12)), (LBMForce.Keys, (20, 9, 12)), (LBMForce.Keys, (20, 14, 12))],
                         ids=["nearest", "keys-spread", "keys-rows"])
def test_centred_device_steps_are_those_of_the_host(stencil, grid):
    """The centred drag's forces added to the caller's array by the solve (stencils) or after the step (nearest node), with
    every other particle coupled: eight device-resident steps in one call, the particles' work between them in the pass or in
    a launch of its own, against the host's steps, which add the forces themselves (the rounding of the positions and
    velocities over eight steps: 1e-12)."""
    rng = np.random.default_rng(3)
    s = Setup(grid, tau=0.8)
    for i in range(80):
        s.add_particles(rng.uniform(0, grid), velocities=rng.normal(scale=0.3, size=(1, 3)), coupled=i % 2 == 0)

    def conf(f):
        f.setFriction(10.0)
        f.setTemperature(300.0)
        f.setRandomNumberSeed(9)
        f.setDragScheme(LBMForce.Centered)
        f.setInterpolationStencil(stencil)
    s.configure.append(conf)
    host, device = s.build(None, storage=LBMForce.FP64), s.build(None, storage=LBMForce.FP64)
    host.step(8)
    dp = DeviceParticles(device)
    dp.step(8)
    pos, vel = dp.pull()
    assert np.abs(pos - host.positions).max() <= 1e-12*max(grid)
    assert np.abs(vel - host.velocities).max() <= 1e-12*np.abs(host.velocities).max()


@pytest.mark.parametrize("storage", [LBMForce.FP16, LBMForce.FP32, LBMForce.FP64], ids=["fp16", "fp32", "fp64"])
@pytest.mark.parametrize("grid,beads", [((20, 14, 12), 400), ((9, 8, 7), 150)], ids=["rows", "spread"])
def test_centred_moment_field_gives_the_pulled_moments(grid, beads, storage, monkeypatch):
    """The centred drag's setup from the moment field against the populations pulled per stencil slot, bit for bit, between
    walls and with the momentum removal every second step; the rule between them only weighs their times."""
    rng = np.random.default_rng(beads)
    nx, ny, nz = grid
    s = Setup(grid, tau=0.8)
    s.add_particles(rng.uniform(0, grid, size=(beads, 3)), velocities=rng.normal(scale=0.3, size=(beads, 3)))

    def conf(f):
        f.setSolidNodes([i for k in (0, nz - 1) for i in range(k*nx*ny, (k + 1)*nx*ny)])
        f.setWallScheme(LBMForce.BounceBack)
        f.setFriction(10.0)
        f.setTemperature(300.0)
        f.setFluidFluctuations(True)
        f.setFluidMomentumRemovalFrequency(2)
        f.setRandomNumberSeed(5)
        f.setDragScheme(LBMForce.Centered)
        f.setInterpolationStencil(LBMForce.Keys)
    s.configure.append(conf)
    runs = []
    for field in ("0", "1"):
        monkeypatch.setenv("LBM_AMD_FIELD", field)
        c = s.build(None, storage=storage)
        c.step(5)
        runs.append((c.getFluidState(), c.positions.copy(), c.velocities.copy(), c.getWallForce(), c.getForces()))
    assert np.abs(runs[0][0]).max() > 0
    for a, b in zip(*runs):
        assert np.array_equal(a, b)


def test_centred_spread_in_several_launches_matches_the_rows(monkeypatch):
    """1.5 M centred Keys particles, whose spread takes two launches of at most 2^20 work-groups, against the matrix rows (both
    stop at a residual of 1e-13 of the right-hand side: the forces agree to 1e-11 of the largest, as in the rows' test)."""
    n, beads = 240, 1500000
    rng = np.random.default_rng(2)
    s = Setup((n, n, n), tau=0.8)
    s.masses, s.coupled = [100.0]*beads, list(range(beads))
    s.positions, s.velocities = list(rng.uniform(0, n, size=(beads, 3))), list(rng.normal(scale=0.5, size=(beads, 3)))

    def conf(f):
        f.setFriction(10.0)
        f.setTemperature(0.0)
        f.setDragScheme(LBMForce.Centered)
        f.setInterpolationStencil(LBMForce.Keys)
    s.configure.append(conf)
    forces = []
    for rows in ("0", "1"):
        monkeypatch.setenv("LBM_AMD_CG_ROWS", rows)
        c = s.build()
        c.step(1)
        forces.append(c.getForces())
    assert np.abs(forces[0]).min(axis=1).max() > 0
    assert np.abs(forces[0] - forces[1]).max() <= 1e-11*np.abs(forces[0]).max()
