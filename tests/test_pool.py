"""The library's device memory: an owner's buffers go back on their own device (on the CPU, with a stand-in for the
HIP runtime), and a destroyed plan's memory is the device's again."""
import os
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "ddfacet_amd", "csrc")
STUB = """#pragma once
#include <cstddef>
typedef int hipError_t;
typedef void* hipStream_t;
constexpr hipError_t hipSuccess = 0;
hipError_t hipGetDevice(int*);
hipError_t hipSetDevice(int);
hipError_t hipDeviceSynchronize();
hipError_t hipStreamSynchronize(hipStream_t);
hipError_t hipFreeAsync(void*, hipStream_t);
"""


def test_buffers_go_back_on_their_own_device():
    with tempfile.TemporaryDirectory() as d:
        os.makedirs(os.path.join(d, "hip"))
        with open(os.path.join(d, "hip", "hip_runtime.h"), "w") as f:
            f.write(STUB)
        exe = os.path.join(d, "pool_check")
        subprocess.run(["g++", "-O1", "-std=c++17", "-I", d, "-I", CSRC, os.path.join(HERE, "pool_check.cpp"), "-o", exe],
                       check=True, capture_output=True, timeout=120)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stdout


@pytest.mark.gpu
def test_a_destroyed_plan_gives_its_memory_back():
    import torch
    from ddfacet_amd.device import trim_memory
    from ddfacet_amd.facets import DeviceFacetSet
    from ddfacet_amd.problems import random_problem
    keep = 4 << 30
    P = random_problem(3, nant=20, ntime=100, nchan=100, nfacet=64, facet_spacing_px=4, npix=32, bda="pervis")
    fs = DeviceFacetSet(P, with_model=True)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    info = fs.plan_batched()
    assert info["device_bytes"] > keep
    fs.destroy_plan()
    assert torch.cuda.mem_get_info()[0] >= before - keep - (64 << 20)
    trim_memory()
    assert torch.cuda.mem_get_info()[0] >= before - (64 << 20)
