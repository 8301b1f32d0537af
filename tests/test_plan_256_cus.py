"""The planner on a GPU of 256 CUs, without one: a preloaded stand-in answers
the few HIP queries the planner makes (device, CU count, occupancy, whether an
address is host memory), in a process of its own per test."""

from __future__ import annotations

import json
import os
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

STAND_IN = r"""
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>
extern "C" {
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 160 << 10;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 3;
  return hipSuccess;
}
// addresses from 2^40 up are pinned host memory
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  a->type = (size_t)p >= (1ull << 40) ? hipMemoryTypeHost : hipMemoryTypeDevice;
  return hipSuccess;
}
}
"""

PRELUDE = """
import ctypes, json, os, random
import torch
from vllm_fastdecoder_amd import _lib, ops
lib = _lib.load_lib()
def done(x):
    print("RESULT " + json.dumps(x))
"""


@pytest.fixture(scope="module")
def planner(tmp_path_factory):
    """Runs a piece of Python against the planner; its done(x) is returned."""
    d = tmp_path_factory.mktemp("stand_in")
    src, so = d / "hip.cpp", d / "hip.so"
    src.write_text(STAND_IN)
    subprocess.run(["g++", "-O1", "-fPIC", "-shared", "-w", "-I/opt/rocm/include", str(src), "-o",
                    str(so)], check=True)

    def run(code: str):
        env = {k: v for k, v in os.environ.items() if not k.startswith("FD_")}
        env["LD_PRELOAD"] = ":".join(x for x in (str(so), env.get("LD_PRELOAD")) if x)
        r = subprocess.run([sys.executable, "-c", PRELUDE + code], cwd=ROOT, env=env,
                           capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr[-3000:]
        return json.loads(r.stdout.split("RESULT ")[1])

    return run


def test_remembered_sizes_follow_every_override(planner):
    """workspace_bytes under another FD_HOST_WGS (or FD_BALANCE) is the
    library's answer for it, not the one remembered."""
    got = planner("""
out = []
for name, values in (("FD_HOST_WGS", "0 32 128 512"), ("FD_BALANCE", "0 64 400")):
    for v in values.split():
        os.environ[name] = v
        size = ctypes.c_size_t()
        _lib.check(lib.fd_paged_decode_workspace_size(33, 32, 8, 128, 16, 226, ctypes.byref(size)))
        out.append([ops.workspace_bytes(33, 32, 8, 128, 16, 226), size.value])
    del os.environ[name]
done(out)
""")
    assert all(a == b for a, b in got) and len({b for _, b in got[:4]}) > 1
