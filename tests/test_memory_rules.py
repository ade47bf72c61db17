"""The library's rules of device memory (lbm_memory.h) on a device that runs out of it, which a small program plays: its hipMalloc
gives out no more than it is told to hold (CPU; needs a C++ compiler and HIP's headers)."""
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
static size_t capacity = 0, used = 0, serial = 0;
static hipError_t last = hipSuccess;
extern "C" hipError_t hipMalloc(void** p, size_t n) {
    if (used + n > capacity)
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
