"""The work that users of this framework have it do, as timed cases.

Every case is one call pattern of a program that uses the package: coupled lattice steps with the particles on the
device or on the host, batched replicas, the centred drag, the learned closure, the closure network's training and
evaluation.  A lattice pass advances a kept simulation by `steps` steps and then reads what such a program reads: the
particles and the density and velocity of every node, into page-locked arrays that it keeps.

exact() is the same work in 64 bits with torch alone: the D3Q19 regularized collision with Guo forcing and Philox
noise, half-way bounce-back, the stencil couplings and the network, written here from their equations.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "openmm-lbm_amd"))

from lbm_amd import closure as closure_api  # noqa: E402
from lbm_amd.batch import Batch, Replica  # noqa: E402
from lbm_amd.context import Context, System, VerletIntegrator  # noqa: E402
from lbm_amd.force import LBMForce  # noqa: E402
from lbm_amd.harness import DeviceParticles  # noqa: E402

DX, DT, DENSITY, MASS, FRICTION = 1.0, 0.01, 602.214, 100.0, 10.0     # nm, ps, Da/nm^3, Da, 1/ps
KT300 = 1.380649e-23*6.02214076e23/1000.0*300.0                       # kJ/mol
CELL = DENSITY*DX**3
WIDTH = {"nearest": 1, "trilinear": 2, "threepoint": 3, "keys": 4}
BYTES = {"fp32": 4, "fp16": 2, "bf16": 2, "fp64": 8}
CHAIN, BOND_K, BOND_R0 = 50, 1000.0, 0.38


def _lattice(name, size, **more):
    case = dict(kind="lattice", nx=size[0], ny=size[1], nz=size[2], storage="fp32", stencil="keys", beads=0, chains=False,
                walls=False, fluct=True, centred=False, closure=False, host=False, tau=0.6, steps=100)
    case.update(more)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # The smallest coupled run: a 32^3 shear box with 64 trilinear beads, T = 0 (latency and launches).
        _lattice("beads_32", (32, 32, 32), stencil="trilinear", beads=64, fluct=False, tau=0.8, steps=100),
        # A small system driven from the host, as an OpenMM program does: positions and velocities in host arrays
        # at every step.
        _lattice("beads_30_host", (30, 30, 30), stencil="nearest", beads=110, host=True, tau=0.8, steps=50),
        # The production channel: 256^3 between bounce-back planes, 20,000 Keys beads, fluctuating.
        _lattice("channel_256_fp32", (256, 256, 256), beads=20000, walls=True, steps=100),
        # The same channel without fluctuations in half-precision storage.
        _lattice("channel_256_fp16", (256, 256, 256), beads=20000, walls=True, fluct=False, storage="fp16", steps=100),
        # A fluctuating fluid alone in double precision (a validation run).
        _lattice("fluid_128_fp64", (128, 128, 128), storage="fp64", tau=0.7, steps=100),
        # Odd sizes between walls, half-precision storage with fluctuations, three-point beads.
        _lattice("ragged_fp16", (150, 117, 86), storage="fp16", stencil="threepoint", beads=3001, walls=True, tau=0.7,
                 steps=100),
        # Independent replicas of uneven size stepped together (a seed-averaged study).
        dict(name="replicas_32", kind="batch", replicas=32, largest=96, beads=2000, stencil="trilinear", fluct=True,
             steps=100),
        # Crowded polymer chains with the Keys stencil: 2,000 chains of 50 beads in 128^3.
        _lattice("chains_keys", (128, 128, 128), beads=100000, chains=True, tau=0.7, steps=100),
        # The same chains coupled through the learned closure.
        _lattice("chains_closure", (128, 128, 128), beads=100000, chains=True, closure=True, tau=0.7, steps=100),
        # The centred drag with the Keys stencil on crowded beads (a conjugate-gradient solve at every step).
        _lattice("crowded_centred", (120, 120, 120), beads=56320, centred=True, tau=0.8, steps=20),
        # Training the closure network on 200,000 pairs, two epochs of minibatches.
        dict(name="train_200k", kind="train", rows=200000, batch=2048, epochs=2),
        # Evaluating the network on host arrays.
        dict(name="forward_50k", kind="forward", rows=50001),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _size(rng, low, high):
    """Three edges with about a power-law spread of node counts, one in three of them multiples of 32."""
    edge = _log(rng, low, high)
    edges = [max(16, min(high, int(edge*rng.uniform(0.7, 1.4)))) for _ in range(3)]
    if rng.random() < 0.34:
        edges = [max(32, e//32*32) for e in edges]
    return edges


def draw(rng):
    pick = rng.choice(["channel", "box", "host", "fluid", "chains", "closure", "centred", "batch", "train", "forward"])
    stencil = rng.choice(["trilinear", "threepoint", "keys", "keys"])
    tau = round(rng.uniform(0.55, 1.0), 3)
    if pick == "channel":
        size = _size(rng, 32, 200)
        return _lattice(None, size, stencil=stencil, beads=_log(rng, 50, max(60, size[0]*size[1]*size[2]//800)), walls=True,
                        fluct=rng.random() < 0.5, storage=rng.choice(["fp32", "fp32", "fp16"]), tau=tau,
                        steps=rng.randint(20, 60))
    if pick == "box":
        size = _size(rng, 24, 160)
        return _lattice(None, size, stencil=stencil, beads=_log(rng, 50, 20000), fluct=rng.random() < 0.5, tau=tau,
                        storage=rng.choice(["fp32", "fp32", "fp64"]), steps=rng.randint(20, 60))
    if pick == "host":
        size = _size(rng, 20, 96)
        return _lattice(None, size, stencil=rng.choice(["nearest", "trilinear", "keys"]), beads=_log(rng, 50, 20000),
                        host=True, fluct=rng.random() < 0.5, tau=tau, steps=rng.randint(10, 40))
    if pick == "fluid":
        fluct = rng.random() < 0.7
        return _lattice(None, _size(rng, 32, 192), fluct=fluct, walls=not fluct, tau=tau, steps=rng.randint(20, 60),
                        storage=rng.choice(["fp32", "fp16", "fp64"]))
    if pick in ("chains", "closure"):
        size = [max(32, e) for e in _size(rng, 48, 128)]
        beads = CHAIN*max(1, _log(rng, 2000, 100000)//CHAIN)
        return _lattice(None, size, beads=beads, chains=True, closure=pick == "closure", tau=tau, steps=rng.randint(20, 60))
    if pick == "centred":
        return _lattice(None, _size(rng, 32, 128), stencil=rng.choice(["nearest", "trilinear", "keys"]),
                        beads=_log(rng, 200, 40000), centred=True, tau=tau, steps=rng.randint(5, 20))
    if pick == "batch":
        return dict(kind="batch", replicas=rng.randint(3, 40), largest=rng.choice([48, 64, 96]), beads=_log(rng, 100, 2000),
                    stencil=rng.choice(["nearest", "trilinear", "keys"]), fluct=rng.random() < 0.8,
                    steps=rng.randint(20, 60))
    if pick == "train":
        return dict(kind="train", rows=_log(rng, 3000, 200000), batch=rng.choice([500, 1024, 2048, 4096]),
                    epochs=rng.randint(1, 3))
    return dict(kind="forward", rows=_log(rng, 100, 400000))


# ---------------------------------------------------------------------------------------------------------------------
# Inputs, from the case and the seed alone.
# ---------------------------------------------------------------------------------------------------------------------
def _particles(case, rng):
    """Positions (nm) and velocities (nm/ps)."""
    n, size = case["beads"], np.array([case["nx"], case["ny"], case["nz"]], dtype=float)*DX
    if case["chains"]:
        pos = np.zeros((n//CHAIN, CHAIN, 3))
        pos[:, 0] = rng.uniform(0, 1, size=(n//CHAIN, 3))*size
        hop = rng.normal(size=(n//CHAIN, CHAIN - 1, 3))
        hop *= BOND_R0/np.linalg.norm(hop, axis=2, keepdims=True)
        pos[:, 1:] = pos[:, :1] + np.cumsum(hop, axis=1)
        pos = pos.reshape(-1, 3) % size
    else:
        pos = rng.uniform(0, 1, size=(n, 3))*size
    if case["walls"]:
        pos[:, 2] = rng.uniform(1.5, case["nz"] - 2.5, size=n)*DX
    return pos, rng.normal(size=(n, 3))*math.sqrt(KT300/MASS)


def _inputs(case, seed):
    rng = np.random.default_rng(seed)
    pos, vel = _particles(case, rng)
    u0 = rng.normal(size=3)
    speed = 3e-4 if case["fluct"] else 0.02               # lattice units; the thermal velocity of a node is 6e-4
    return dict(pos=pos, vel=vel, seed=int(rng.integers(1, 2**31 - 1)), u0=speed*u0/np.linalg.norm(u0))


def _drive(case):
    """The body acceleration along x (lattice units): a thermal fluid at rest between no walls has none."""
    return 1e-6 if case["walls"] or not case["fluct"] else 0.0


def _solid_nodes(case):
    plane = case["nx"]*case["ny"]
    last = plane*(case["nz"] - 1)
    return list(range(plane)) + list(range(last, last + plane)) if case["walls"] else []


def _network(rng):
    """Parameters of an 87 -> 64 -> 64 -> 3 network in the library's flat layout (padded to 96 inputs, 16 outputs)."""
    w1, w2, w3 = np.zeros((96, 64)), rng.normal(size=(64, 64))/8.0, np.zeros((64, 16))
    w1[:87] = rng.normal(size=(87, 64))/math.sqrt(87.0)
    w3[:, :3] = rng.normal(size=(64, 3))/8.0
    b3 = np.zeros(16)
    b3[:3] = 0.1*rng.normal(size=3)
    parts = [w1, 0.1*rng.normal(size=64), w2, 0.1*rng.normal(size=64), w3, b3]
    return np.concatenate([p.reshape(-1) for p in parts]).astype(np.float32)


# Scales of a fluid and beads at 300 K; the bounds leave about one bead in 100,000 to the fallback, as in a trained run.
# The corrections of this untrained network are kept small against the thermal velocity, so that it does not heat the run.
NORM = dict(u_scale=1500.0, v_scale=600.0, out_scale=20000.0, u_bound=5.3, v_bound=6.0)


def _pairs(rows, seed):
    """Training pairs with the distribution of a thermal fluid: offsets, node velocities, the bead's velocity; the
    target is a smooth function of them and a part that the inputs do not hold."""
    rng = np.random.default_rng(seed)
    x = np.empty((rows, 87), dtype=np.float32)
    x[:, :3] = -np.sort(-rng.uniform(0, 1, size=(rows, 3)), axis=1)
    x[:, 3:84] = rng.standard_normal((rows, 81), dtype=np.float32)/np.float32(NORM["u_scale"])
    x[:, 84:] = rng.standard_normal((rows, 3), dtype=np.float32)/np.float32(NORM["v_scale"])
    t = 0.3*x[:, :3]*(x[:, 45:48] - x[:, 42:45]) + 0.05*x[:, 3:6] + 1e-5*rng.standard_normal((rows, 3), dtype=np.float32)
    return x, t.astype(np.float32)


def _force(case, inputs):
    f = LBMForce()
    f.setGridSize(case["nx"], case["ny"], case["nz"])
    f.setFluidDensity(DENSITY)
    f.setKinematicViscosity((case["tau"] - 0.5)/3.0*DX*DX/DT)
    f.setFluidMomentumRemovalFrequency(0)
    f.setStorage({"fp32": LBMForce.FP32, "fp16": LBMForce.FP16, "fp64": LBMForce.FP64}[case["storage"]])
    f.setInitialFluidVelocity(tuple(inputs["u0"]*DX/DT))
    f.setBodyAcceleration((_drive(case)*DX/DT**2, 0.0, 0.0))
    f.setFriction(FRICTION)
    f.setTemperature(300.0 if case["fluct"] else 0.0)
    f.setFluidFluctuations(case["fluct"])
    f.setRandomNumberSeed(inputs["seed"])
    f.setInterpolationStencil({"nearest": LBMForce.NearestNode, "trilinear": LBMForce.Trilinear,
                               "threepoint": LBMForce.ThreePoint, "keys": LBMForce.Keys}[case["stencil"]])
    f.setDragScheme(LBMForce.Centered if case["centred"] else LBMForce.Explicit)
    if case["walls"]:
        f.setSolidNodes(_solid_nodes(case))
        f.setWallScheme(LBMForce.BounceBack)
    for i in range(case["beads"]):
        f.addParticle(i)
    return f


def _wall(case):
    return KT300, 0.5*DX, 0.5*DX, (case["nz"] - 1.5)*DX


def _wall_force(case):
    eps, sigma, lo, hi = _wall(case)

    def f(pos):
        out = np.zeros_like(pos)
        d1, d2 = pos[:, 2] - lo, hi - pos[:, 2]
        out[:, 2] = 12*eps*((sigma/d1)**12/d1 - (sigma/d2)**12/d2)
        return out
    return f


def _bonds(case):
    first = np.arange(case["beads"]).reshape(-1, CHAIN)[:, :-1].reshape(-1)
    return np.stack([first, first + 1], axis=1).astype(np.int32)


def _pinned(count):
    t = torch.empty(int(count), dtype=torch.float64, pin_memory=torch.cuda.is_available())
    return t.numpy()


def _p(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def prepare(case, seed):
    if case["kind"] == "lattice":
        inputs = _inputs(case, seed)
        system = System((case["nx"]*DX, case["ny"]*DX, case["nz"]*DX))
        for _ in range(max(1, case["beads"])):
            system.addParticle(MASS)
        extra = [_wall_force(case)] if case["walls"] and case["host"] else []
        ctx = Context(system, VerletIntegrator(DT), _force(case, inputs), extraForces=extra)
        ctx.setPositions(inputs["pos"] if case["beads"] else np.zeros((1, 3)))
        ctx.setVelocities(inputs["vel"] if case["beads"] else np.zeros((1, 3)))
        state = dict(case=case, ctx=ctx, rho=_pinned(ctx.numNodes), u=_pinned(3*ctx.numNodes).reshape(-1, 3))
        if case["closure"]:
            net = closure_api.MLPClosure(seed=1)
            net.setParameters(_network(np.random.default_rng(seed + 1)))
            net.setNormalization(**NORM)
            net.attach(ctx)
        if not case["host"]:
            state["dp"] = dp = DeviceParticles(ctx)
            if case["walls"] and case["beads"]:
                dp.setWallPotential(*_wall(case))
            if case["chains"]:
                dp.setBonds(_bonds(case), BOND_K, BOND_R0)
        return state
    if case["kind"] == "batch":
        plan = _replicas(case, seed)
        replicas = []
        for sub, inputs in plan:
            box = (sub["nx"]*DX, sub["ny"]*DX, sub["nz"]*DX)
            replicas.append(Replica(_force(sub, inputs), box, DT, np.full(sub["beads"], MASS), inputs["pos"], inputs["vel"]))
        batch = Batch(replicas)
        sizes = [sub["nx"]*sub["ny"]*sub["nz"] for sub, _ in plan]
        beads = sum(sub["beads"] for sub, _ in plan)
        return dict(case=case, batch=batch, first=np.concatenate([[0], np.cumsum(sizes)]), rho=_pinned(sum(sizes)),
                    u=_pinned(3*sum(sizes)).reshape(-1, 3), pos=_pinned(3*beads).reshape(-1, 3),
                    vel=_pinned(3*beads).reshape(-1, 3))
    net = closure_api.MLPClosure(seed=1)
    params = _network(np.random.default_rng(seed + 1))
    net.setParameters(params)
    if case["kind"] == "train":
        x, t = _pairs(case["rows"], seed)
        return dict(case=case, net=net, params=params, x=x, t=t)
    net.setNormalization(**NORM)
    return dict(case=case, net=net, x=_pairs(case["rows"], seed)[0])


def run(state):
    case = state["case"]
    if case["kind"] == "lattice":
        ctx = state["ctx"]
        if case["host"]:
            ctx.step(case["steps"])
        else:
            state["dp"].step(case["steps"])
            state["dp"].pull()
        status = ctx.lib.lbm_get_fluid_fields(ctx.handle, _p(state["rho"]), _p(state["u"]), 0)
        if status != 0:
            raise RuntimeError(ctx.lib.lbm_last_error().decode())
        if not case["beads"]:
            return [state["rho"], state["u"]]
        return [state["rho"], state["u"], ctx.positions, ctx.velocities]
    if case["kind"] == "batch":
        batch, first = state["batch"], state["first"]
        batch.step(case["steps"])
        for r in range(case["replicas"]):
            at = slice(int(first[r]), int(first[r + 1]))
            if batch.lib.lbm_batch_get_fluid_fields(batch.handle, r, _p(state["rho"][at]), _p(state["u"][at])) != 0:
                raise RuntimeError(batch.lib.lbm_last_error().decode())
        if batch.lib.lbm_batch_get_particles(batch.handle, _p(state["pos"]), _p(state["vel"])) != 0:
            raise RuntimeError(batch.lib.lbm_last_error().decode())
        return [state["rho"], state["u"], state["pos"], state["vel"]]
    if case["kind"] == "train":
        net = state["net"]
        net.setParameters(state["params"])
        losses = net.train(state["x"], state["t"], epochs=case["epochs"], batch=case["batch"], lr=1e-3, decay=0.9, seed=3)
        return [losses, net.getParameters()]
    return state["net"].forward(state["x"])


def work(case):
    """Bytes: per step, every population read once and written once and the beads' positions, velocities and forces;
    then the fields and particles that are read out.  Floating operations of the collision, the noise and the stencils."""
    if case["kind"] in ("train", "forward"):
        per_row = 2*(87*64 + 64*64 + 64*3)
        if case["kind"] == "forward":
            return {"bytes": case["rows"]*4*(87 + 3), "flops": case["rows"]*per_row}
        return {"bytes": case["epochs"]*case["rows"]*4*(87 + 3), "flops": case["epochs"]*case["rows"]*3*per_row}
    if case["kind"] == "batch":
        parts = [(s["nx"]*s["ny"]*s["nz"], s["beads"]) for s, _ in _replicas(case, 0)]
        nodes, beads, size = sum(p[0] for p in parts), sum(p[1] for p in parts), 4
    else:
        nodes, beads, size = case["nx"]*case["ny"]*case["nz"], case["beads"], BYTES[case["storage"]]
    slots = WIDTH[case["stencil"]]**3
    step_bytes = nodes*2*19*size + beads*8*12
    step_flops = nodes*(260 + (240 if case["fluct"] else 0)) + beads*slots*60
    return {"bytes": case["steps"]*step_bytes + nodes*(19*size + 32) + beads*48, "flops": case["steps"]*step_flops}


def _replicas(case, seed):
    """The replicas of a batch: uneven edges (the sizes from the case, so that its work does not hang on the seed),
    relaxation times, temperatures as the force's 300 K or 0, seeds and bead counts."""
    shape = np.random.default_rng(case["replicas"]*1000 + case["largest"])
    edges = [e for e in (24, 32, 33, 48, 60, 64, 96) if e <= case["largest"]]
    plan = []
    for r in range(case["replicas"]):
        n = int(shape.choice(edges))
        sub = _lattice(None, (n, n, n), stencil=case["stencil"], beads=int(shape.integers(50, case["beads"] + 1)),
                       fluct=case["fluct"], tau=round(float(shape.uniform(0.55, 1.0)), 4), steps=case["steps"])
        plan.append((sub, _inputs(sub, 1000003*(r + 1) + seed)))
    return plan


# ---------------------------------------------------------------------------------------------------------------------
# The same in 64 bits.
# ---------------------------------------------------------------------------------------------------------------------
CX = [0, 1, -1, 0, 0, 0, 0, 1, -1, 1, -1, 0, 0, 0, 0, 1, -1, -1, 1]
CY = [0, 0, 0, 1, -1, 0, 0, 1, -1, -1, 1, 1, -1, 1, -1, 0, 0, 0, 0]
CZ = [0, 0, 0, 0, 0, 1, -1, 0, 0, 0, 0, 1, -1, -1, 1, 1, -1, 1, -1]
OPP = [0, 2, 1, 4, 3, 6, 5, 8, 7, 10, 9, 12, 11, 14, 13, 16, 15, 18, 17]
C = np.array([CX, CY, CZ], dtype=float)
W = np.array([1/3] + [1/18]*6 + [1/36]*12)


def _noise_basis():
    """The 15 noisy modes (six of the stress, nine ghosts) at the 19 velocities, each divided by its norm: [15][19]."""
    x, y, z = C
    x2, y2, z2 = x*x, y*y, z*z
    e = [x2 - 1/3, y2 - 1/3, z2 - 1/3, x*y, x*z, y*z, y*(x2 - 1/3), z*(x2 - 1/3), x*(y2 - 1/3),
         0.5*x*(y2 + 2*z2 - 1), 0.5*y*(x2 + 2*z2 - 1), 0.5*z*(x2 + 2*y2 - 1),
         x2*y2 - x2/3 - y2/3 + z2/6 + 1/18,
         2/7*x2*y2 + x2*z2 - 3/7*x2 + y2/14 - 2/7*z2 + 1/14,
         0.4*x2*y2 + 0.4*x2*z2 + y2*z2 - 0.1*x2 - 0.4*y2 - 0.4*z2 + 0.1]
    return np.array([m/math.sqrt(float((W*m*m).sum())) for m in e])


def _philox(c, key):
    """Philox4x32-10 (Salmon et al., SC'11) of four counter words (int64 tensors or numbers), 32-bit words."""
    mask = 0xFFFFFFFF

    def mul(a, b):
        low = a*(b & 0xFFFF)
        t = a*(b >> 16) + (low >> 16)
        return t >> 16, ((t & 0xFFFF) << 16) | (low & 0xFFFF)
    c, k0, k1 = list(c), key[0], key[1]
    for _ in range(10):
        h0, l0 = mul(0xD2511F53, c[0])
        h1, l1 = mul(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
    return c


def _box_muller(radius, angle):
    r = torch.sqrt(-2.0*torch.log((radius.double() + 1.0)*2.0**-32))
    t = angle.double()*(2.0*math.pi/65536.0)
    return r*torch.cos(t), r*torch.sin(t)


class _Exact:
    """One lattice with its beads in 64 bits; f: pre-collision deviations f_q - w_q, [19][nz][ny][nx]."""

    def __init__(self, case, inputs, network=None):
        self.case, self.network = case, network
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.shape = (case["nz"], case["ny"], case["nx"])
        self.n = case["nx"]*case["ny"]*case["nz"]
        self.size = self.t([case["nx"], case["ny"], case["nz"]])
        self.omega, self.seed = 1.0/case["tau"], inputs["seed"]
        self.g = [_drive(case), 0.0, 0.0]
        self.gamma, self.m = FRICTION*DT, MASS/CELL
        self.kT = KT300*DT**2/(CELL*DX**2) if case["fluct"] else 0.0
        u = inputs["u0"]
        cu = C.T @ u
        eq = W*(3*cu + 4.5*cu*cu - 1.5*float(u @ u))
        self.f = self.t(eq)[:, None].expand(19, self.n).clone()
        self.solid = None
        if case["walls"]:
            self.solid = torch.zeros(self.n, dtype=torch.bool, device=self.dev)
            self.solid[torch.tensor(_solid_nodes(case), device=self.dev)] = True
        self.pos, self.vel = self.t(inputs["pos"]), self.t(inputs["vel"])
        self.basis, self.c = self.t(_noise_basis()), self.t(C)
        self.nodes = torch.arange(self.n, device=self.dev)
        if case["chains"]:
            self.bonds = torch.tensor(_bonds(case), dtype=torch.long, device=self.dev)

    def t(self, a):
        return torch.tensor(np.asarray(a, dtype=float), dtype=torch.float64, device=self.dev)

    def other_forces(self):
        f = torch.zeros_like(self.pos)
        if self.case["walls"]:
            eps, sigma, lo, hi = _wall(self.case)
            d1, d2 = self.pos[:, 2] - lo, hi - self.pos[:, 2]
            f[:, 2] += 12*eps*((sigma/d1)**12/d1 - (sigma/d2)**12/d2)
        if self.case["chains"]:
            i, j = self.bonds.T
            d = self.pos[j] - self.pos[i]
            box = self.size*DX
            d = d - box*torch.round(d/box)
            r = d.norm(dim=1, keepdim=True)
            pull = BOND_K*(r - BOND_R0)/r*d
            f.index_add_(0, i, pull)
            f.index_add_(0, j, -pull)
        return f

    def slots(self, stencil, pos):
        """Nodes and weights of the stencils: [beads][w^3]."""
        s = pos/DX
        s = s - torch.floor(s/self.size)*self.size
        w = WIDTH[stencil]
        if stencil in ("nearest", "threepoint"):
            first = torch.floor(s + 0.5) - (1 if stencil == "threepoint" else 0)
        else:
            first = torch.floor(s) - (1 if stencil == "keys" else 0)
        at = first[:, :, None] + torch.arange(w, device=self.dev)
        r = (s[:, :, None] - at).abs()
        if stencil == "nearest":
            k = torch.ones_like(r)
        elif stencil == "trilinear":
            k = 1 - r
        elif stencil == "threepoint":
            inner = (1 + torch.sqrt((1 - 3*r*r).clamp(min=0)))/3
            outer = (5 - 3*r - torch.sqrt((1 - 3*(1 - r)**2).clamp(min=0)))/6
            k = torch.where(r <= 0.5, inner, torch.where(r < 1.5, outer, torch.zeros_like(r)))
        else:
            k = torch.where(r <= 1, 1 - 2.5*r**2 + 1.5*r**3, 2 - 4*r + 2.5*r**2 - 0.5*r**3)
        idx = torch.remainder(at, self.size[None, :, None]).long()
        nx, ny = self.case["nx"], self.case["ny"]
        node = idx[:, 0, None, None, :] + nx*(idx[:, 1, None, :, None] + ny*idx[:, 2, :, None, None])
        weight = k[:, 0, None, None, :]*k[:, 1, None, :, None]*k[:, 2, :, None, None]
        return node.flatten(1), weight.flatten(1), s

    def random(self, step):
        n = len(self.pos)
        if self.kT == 0:
            return torch.zeros((n, 3), dtype=torch.float64, device=self.dev)
        i = torch.arange(n, device=self.dev)
        key = (self.seed, 0x50415254)
        radii = _philox((i, step, 0, 0), key)
        angles = _philox((i, step, 0, 2), key)[0]
        a = _box_muller(radii[0], angles & 0xFFFF)
        b = _box_muller(radii[1], angles >> 16)
        return math.sqrt(2*self.gamma*self.m*self.kT)*torch.stack([a[0], a[1], b[0]], dim=1)

    def closure_velocity(self, u):
        """u(nearest) + the network's correction, the Keys interpolation where an input is out of bounds."""
        node, _, s = self.slots("nearest", self.pos)
        near = torch.floor(s + 0.5)
        off = s - near
        axis = torch.argsort(-off.abs(), dim=1, stable=True)
        sign = torch.where(off < 0, -1.0, 1.0).to(torch.float64)
        sign = torch.gather(sign, 1, axis)
        grid = torch.stack(torch.meshgrid(*[torch.arange(-1, 2, device=self.dev)]*3, indexing="ij"), -1).reshape(-1, 3)
        grid = grid.flip(1).to(torch.float64)                 # the node at (a, b, c) of the bead's frame, a fastest
        d = torch.zeros((len(off), 27, 3), dtype=torch.float64, device=self.dev)
        d.scatter_(2, axis[:, None, :].expand(-1, 27, -1), sign[:, None, :]*grid[None])
        idx = torch.remainder(near[:, None, :] + d, self.size).long()
        flat = idx[..., 0] + self.case["nx"]*(idx[..., 1] + self.case["ny"]*idx[..., 2])
        un = torch.gather(u[flat], 2, axis[:, None, :].expand(-1, 27, -1))*sign[:, None, :]*NORM["u_scale"]
        v = torch.gather(self.vel*DT/DX, 1, axis)*sign*NORM["v_scale"]
        o = 2*torch.gather(off.abs(), 1, axis)
        out = (un.abs() > NORM["u_bound"]).flatten(1).any(1) | (v.abs() > NORM["v_bound"]).any(1)
        du = _mlp(self.network, torch.cat([o, un.flatten(1), v], dim=1))/NORM["out_scale"]
        back = torch.zeros_like(du).scatter_(1, axis, du*sign)
        return node, u[node[:, 0]] + back, out

    def couple(self, step, rho, j, other):
        """The coupling forces and the reaction on the nodes, lattice units."""
        case, h = self.case, 0.5
        fluid = torch.ones_like(rho) if self.solid is None else (~self.solid).to(rho.dtype)
        noise = self.random(step)
        v = self.vel*DT/DX
        unit = CELL*DX/DT**2
        reaction = torch.zeros((self.n, 3), dtype=torch.float64, device=self.dev)
        u = (j/rho).T*fluid[:, None]
        if case["closure"]:
            node, ub, out = self.closure_velocity(u)
            at, weight, _ = self.slots("keys", self.pos[out])
            ub[out] = (weight[..., None]*u[at]).sum(1)
            force = -self.gamma*self.m*(v - ub) + noise
            reaction.index_add_(0, node[~out, 0], -force[~out])
            reaction.index_add_(0, at.flatten(), -(weight[..., None]*force[out][:, None]).flatten(0, 1))
            return force*unit, reaction
        node, weight, _ = self.slots(case["stencil"], self.pos)
        wf = weight*fluid[node]
        if not case["centred"]:
            force = -self.gamma*self.m*(v - (wf[..., None]*u[node]).sum(1)) + noise
        else:
            g = self.t(self.g)
            a = self.gamma*h
            ub = (wf[..., None]*(u + h*g*fluid[:, None])[node]).sum(1)
            b = (-self.gamma*self.m*(v + h*other/unit/self.m - ub) + noise)/self.m
            inv = wf/rho[node]

            def apply(x):
                s = torch.zeros((self.n, 3), dtype=torch.float64, device=self.dev)
                s.index_add_(0, node.reshape(-1), (weight[..., None]*x[:, None]).reshape(-1, 3))
                return x*((1 + a)/self.m) + a*(inv[..., None]*s[node]).sum(1)
            diag = ((1 + a)/self.m + a*(weight*inv).sum(1))[:, None]
            force = b/diag
            r = b - apply(force)
            z = r/diag
            d, rz = z, (r*z).sum(0)
            for _ in range(400):
                ad = apply(d)
                alpha = rz/(d*ad).sum(0).clamp(min=1e-300)
                force, r = force + alpha*d, r - alpha*ad
                if bool(((r*r).sum(0) <= 1e-28*(b*b).sum(0)).all()):
                    break
                z = r/diag
                new = (r*z).sum(0)
                d, rz = z + new/rz.clamp(min=1e-300)*d, new
        reaction.index_add_(0, node.reshape(-1), -(wf[..., None]*force[:, None]).reshape(-1, 3))
        return force*unit, reaction

    def fluid_noise(self, step, rho):
        block = torch.arange(3, device=self.dev)[:, None]
        w = _philox((self.nodes[None], step, 0, block), (self.seed, 0x464C5549))
        words = [w[k % 4][k // 4] for k in range(12)]
        r = []
        for p in range(8):
            r += _box_muller(words[p], (words[8 + p//2] >> (16*(p & 1))) & 0xFFFF)
        ghost = torch.sqrt(3*self.kT*rho)
        stress = ghost*math.sqrt(self.omega*(2 - self.omega))
        modes = torch.stack(r[:15])
        modes[:6] *= stress
        modes[6:] *= ghost
        return (self.t(W)[:, None]*self.basis.T) @ modes

    def step(self, step):
        f, w = self.f, self.t(W)[:, None]
        dr = f.sum(0)
        rho, j = 1 + dr, self.c @ f
        if self.solid is not None:
            rho = torch.where(self.solid, torch.ones_like(rho), rho)
        force = rho*self.t(self.g)[:, None]
        if self.case["beads"]:
            bead, other = None, self.other_forces()
            bead, reaction = self.couple(step, rho, j, other)
            force = force + reaction.T
            self.vel = self.vel + DT*(other + bead)/MASS
            self.pos = self.pos + DT*self.vel
        u = (j + 0.5*force)/rho
        e = dr*torch.ones_like(f) + 3*(self.c.T @ (j + force))
        for a in range(3):
            for b in range(a, 3):
                cc = (self.c[a]*self.c[b])[:, None]
                pi = (cc*f).sum(0) - j[a]*j[b]/rho - (dr/3 if a == b else 0)
                p = rho*u[a]*u[b] + (1 - self.omega)*pi + 0.5*(u[a]*force[b] + u[b]*force[a])
                e += 4.5*(cc - (1/3 if a == b else 0))*p*(1 if a == b else 2)
        post = w*e
        if self.kT > 0:
            post += self.fluid_noise(step, rho)
        grid = post.reshape(19, *self.shape)
        self.f = torch.stack([torch.roll(grid[q], (CZ[q], CY[q], CX[q]), (0, 1, 2)) for q in range(19)]).reshape(19, -1)
        if self.solid is not None:
            wall = self.solid.reshape(self.shape)
            for q in range(1, 19):
                # A fluid node gets back along -c_q what it sent along c_q into a solid node.
                ahead = torch.roll(wall, (-CZ[q], -CY[q], -CX[q]), (0, 1, 2)).reshape(-1) & ~self.solid
                self.f[OPP[q]] = torch.where(ahead, post[q], self.f[OPP[q]])
            self.f[:, self.solid] = 0

    def outputs(self):
        f = self.f
        rho = 1 + f.sum(0)
        u = (((self.c @ f)/rho + 0.5*self.t(self.g)[:, None])*DX/DT).T.contiguous()
        rho = rho*DENSITY
        if self.solid is not None:
            rho, u = rho.masked_fill(self.solid, 0.0), u.masked_fill(self.solid[:, None], 0.0)
        return [rho.cpu().numpy(), u.cpu().numpy(), self.pos.cpu().numpy(), self.vel.cpu().numpy()]


def _mlp(params, x):
    p = torch.as_tensor(params, dtype=torch.float64, device=x.device)
    w1, b1, w2, b2 = p[:6144].reshape(96, 64)[:87], p[6144:6208], p[6208:10304].reshape(64, 64), p[10304:10368]
    w3, b3 = p[10368:11392].reshape(64, 16)[:, :3], p[11392:11395]
    silu = torch.nn.functional.silu
    return silu(silu(x @ w1 + b1) @ w2 + b2) @ w3 + b3


def exact(case, seed):
    if case["kind"] == "train":
        # The order of the minibatches is drawn inside the library: no value follows from the inputs alone.
        return None
    if case["kind"] == "forward":
        x = torch.tensor(_pairs(case["rows"], seed)[0], dtype=torch.float64)
        x[:, 3:84] *= NORM["u_scale"]
        x[:, 84:] *= NORM["v_scale"]
        return (_mlp(_network(np.random.default_rng(seed + 1)), x)/NORM["out_scale"]).numpy()
    plan = _replicas(case, seed) if case["kind"] == "batch" else [(case, _inputs(case, seed))]
    network = _network(np.random.default_rng(seed + 1)) if case.get("closure") else None
    parts = []
    for sub, inputs in plan:
        e = _Exact(sub, inputs, network)
        for s in range(sub["steps"]):
            e.step(s)
        parts.append(e.outputs())
    out = [np.concatenate([p[k] for p in parts]) for k in range(4)]
    return out if parts[0][2].size else out[:2]
