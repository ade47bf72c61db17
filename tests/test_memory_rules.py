"""The library's rules of device memory (lbm_memory.h) on a device that runs out of it, which a small program plays: its hipMalloc
gives out no more than it is told to hold (CPU; needs a C++ compiler and HIP's headers); and one lattice on a GPU with little
memory left."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

DEVICE = r"""
#include "lbm_memory.h"
#include <cstdio>
#include <map>
static std::map<void*, size_t> held;
static size_t questions = 0, capacity = 0, used = 0, serial = 0, fragment = ~(size_t) 0;
static hipError_t last = hipSuccess;
extern "C" hipError_t hipMalloc(void** p, size_t n) {
    if (used + n > capacity || n > fragment)
        return last = hipErrorOutOfMemory;
    *p = (void*) (0x1000 + 0x1000*++serial);
    held[*p] = n;
    used += n;
    return hipSuccess;
}
extern "C" hipError_t hipFree(void* p) {
    if (!held.count(p))
        return last = hipErrorInvalidValue;
    used -= held[p];
    held.erase(p);
    return hipSuccess;
}
extern "C" hipError_t hipGetLastError() {
    hipError_t e = last;
    last = hipSuccess;
    return e;
}
extern "C" hipError_t hipMemGetInfo(size_t* free, size_t* total) {
    questions++;
    *free = capacity - used;
    *total = capacity;
    return hipSuccess;
}
#define CHECK(what) if (!(what)) { printf("line %d: %s\n", __LINE__, #what); return 1; }
constexpr size_t GB = 1ull << 30;
int main() {
"""


def run(tmp_path, body):
    if shutil.which("g++") is None or not os.path.exists(os.path.join(ROCM, "include", "hip", "hip_runtime_api.h")):
        pytest.skip("no C++ compiler or no HIP headers")
    source, program = tmp_path/"rules.cpp", tmp_path/"rules"
    source.write_text(DEVICE + body + "    return 0;\n}\n")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"), "-I",
                    os.path.join(ROOT, "openmm-lbm_amd", "csrc"), str(source), "-o", str(program)], check=True)
    done = subprocess.run([str(program)], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stdout


def test_kept_field_memory_gives_way_to_a_larger_call(tmp_path):
    """A call that finds too little memory beside what an earlier one left with the owner takes that too; a failure leaves
    no error for the next call, and nothing is held twice or lost."""
    run(tmp_path, r"""
    lbm::FieldStage stage;
    capacity = 3*GB/2;
    void* small = stage.get(GB/4);
    CHECK(small && stage.done(small) == hipSuccess && used == GB/4);
    CHECK(stage.get(GB/8) == small);                       // a smaller call shares it
    void* kept = stage.get(GB);                            // grown, and kept
    CHECK(kept && used == GB && stage.done(kept) == hipSuccess && used == GB);
    void* large = stage.get(5*GB/4);                       // not beside the kept block
    CHECK(large && used == 5*GB/4 && hipGetLastError() == hipSuccess);
    CHECK(stage.done(large) == hipSuccess && used == 0);
    CHECK(stage.get(2*GB) == nullptr && hipGetLastError() == hipSuccess && used == 0);
    kept = stage.get(GB/2);
    CHECK(kept && stage.done(kept) == hipSuccess && used == GB/2);
    capacity = GB;
    CHECK(stage.get(GB) != nullptr && used == GB);         // grown where both would not fit
    capacity = 4*GB;
    large = stage.get(2*GB);                               // beside the kept block where there is room
    CHECK(large && used == 3*GB && stage.done(large) == hipSuccess && used == GB);
    stage.free();
    CHECK(used == 0);
""")


def test_optional_memory_leaves_the_reserve(tmp_path):
    """All the parts of a set or none: with room for them beside the reserve, without, and where a part fails although the
    device's figure had room for it."""
    run(tmp_path, r"""
    void *a = nullptr, *b = nullptr;
    CHECK(lbm::reservedBytes(1000) == 209000);
    capacity = 4*GB;
    CHECK(lbm::spareBytes(3*GB) == GB && lbm::spareBytes(4*GB) == 0 && lbm::spareBytes(5*GB) == 0);
    CHECK(lbm::allocateOptional({{&a, GB/2}, {&b, GB/2}}, 3*GB) && a && b && used == GB);
    CHECK(hipFree(a) == hipSuccess && hipFree(b) == hipSuccess);
    CHECK(!lbm::allocateOptional({{&a, GB/2}, {&b, GB/2 + 1}}, 3*GB) && !a && !b && used == 0);
    capacity = GB;
    fragment = GB/4;                                       // no block larger than this
    CHECK(!lbm::allocateOptional({{&a, GB/8}, {&b, GB/2}}, 0) && !a && !b && used == 0);
    CHECK(hipGetLastError() == hipSuccess);
""")


def test_padded_rows_share_the_room(tmp_path):
    """Two arrays for each lattice, by their shares of the nodes, in what stays free beside the reserve of all; small arrays
    are tried without a question, and the device is asked once."""
    run(tmp_path, r"""
    capacity = 2*GB + 209*1000;
    lbm::PaddingRoom room{1000};
    CHECK(room.holds(lbm::SMALL_BYTES, 1) && questions == 0);
    CHECK(room.holds(GB, 1000) && !room.holds(GB + 1, 1000) && room.holds(GB/4, 250) && !room.holds(GB/4 + 1, 250));
    CHECK(questions == 1);
""")


@pytest.mark.gpu
def test_a_centred_solver_fits_where_it_did_without_rows():
    """One million centred Keys particles in 200^3, which need 3.5 GB, on a device with 4.2 GB free: the 1.7 GB of the matrix
    rows are done without, and the lattice steps and is read out."""
    import numpy as np
    import torch
    from lbm_amd import LBMForce
    from parity import Setup

    n, beads = 200, 1000000
    s = Setup((n, n, n), tau=0.7)
    rng = np.random.default_rng(1)
    s.masses, s.coupled = [100.0]*beads, list(range(beads))
    s.positions, s.velocities = list(rng.uniform(0, n, size=(beads, 3))), list(np.zeros((beads, 3)))

    def conf(f):
        f.setFriction(10.0)
        f.setTemperature(0.0)
        f.setBodyAcceleration((1.0, 0.0, 0.0))
        f.setDragScheme(LBMForce.Centered)
        f.setInterpolationStencil(LBMForce.Keys)
    s.configure.append(conf)
    small = Setup((12, 12, 12))
    small.configure.append(conf)
    small.add_particles(rng.uniform(0, 12, size=(40, 3)))
    small.build().step(1)                                  # what the first run of a kernel loads
    torch.cuda.empty_cache()
    fill = torch.empty(max(0, torch.cuda.mem_get_info()[0] - int(4.2e9)), dtype=torch.uint8, device="cuda")
    try:
        c = s.build()
        c.step(1)
        forces, (rho, u) = c.getForces(), c.getFluidFields()
        assert np.isfinite(forces).all() and np.isfinite(rho).all() and u[:, 0].min() > 0
        del c
    finally:
        del fill
        torch.cuda.empty_cache()
