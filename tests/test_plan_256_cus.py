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


SHAPES = """
rng = random.Random(5)
def shape():
    H, KVH, D = rng.choice(((32, 8, 128), (32, 32, 128), (64, 8, 128), (16, 8, 256), (28, 4, 128),
                            (40, 8, 112), (14, 2, 64), (24, 8, 128), (71, 1, 64), (8, 1, 80)))
    return rng.randint(1, 80), H, KVH, D
"""


def test_two_tier_need_covers_the_launch(planner):
    """A workspace of exactly fd_decode_workspace_need's bytes gives a two-tier
    call the plan that an unlimited one gives it, counters or not."""
    got = planner(SHAPES + """
need, bad, workers = ctypes.c_size_t(), [], 0
for _ in range(1500):
    n, H, KVH, D = shape()
    a, b = rng.randint(1, 300), rng.choice((1, 3, 20, 300))
    dt = rng.choice((torch.float16, torch.bfloat16, torch.float32))
    _lib.check(lib.fd_decode_workspace_need(n, H, KVH, D, 16, a + b, ops._DT[dt], 1, 0,
                                            ctypes.byref(need)))
    for counted in (True, False):
        os.environ.pop("FD_HOST_WGS", None)
        free = ops.split_plan_info(n, H, KVH, D, 16, a, b, dt, 1 << 40, counted)
        workers += free["host_workgroups"] > 0
        if ops.split_plan_info(n, H, KVH, D, 16, a, b, dt, need.value, counted) != free:
            bad.append((n, H, KVH, D, a, b, str(dt), counted))
done([len(bad), bad[:3], workers])
""")
    assert got[0] == 0, got
    assert got[2] > 500


def test_a_cache_found_in_host_memory_is_not_refused_its_hbm_workspace(planner):
    """One tier at a pinned address (or one the lookup takes for it) with the
    workspace of the HBM launch: planned again only where that fits. The calls
    here pass every check and end at the launch, for want of a GPU."""
    got = planner(SHAPES + """
need, status = ctypes.c_size_t(), {}
for _ in range(6000):
    n, H, KVH, D = shape()
    n, W = 4 * n, rng.randint(1, 600)
    total = int(rng.random() * n * W * 16)
    _lib.check(lib.fd_decode_workspace_need(n, H, KVH, D, 16, W, 0, 0, total, ctypes.byref(need)))
    p = 1 << 20
    rc = lib.fd_paged_decode_counted(
        p, H * D, D, 1 << 41, 1 << 41, KVH * 16 * D, 16 * D, D, 4, p, W, W, p, None, n, H, KVH, D,
        16, 0.1, 0, p, H * D, D, 0, p, n, p if need.value else None, need.value, None, total, p)
    status[rc] = status.get(rc, 0) + 1
done(status)
""")
    assert set(got) == {"4"}, got  # FD_ERR_HIP


def test_host_workers_go_by_the_tables_widths(planner):
    """On both sides of each line of the rule (plan_host_workers)."""
    got = planner("""
def workers(n, H, KVH, a, b, D=128):
    return ops.split_plan_info(n, H, KVH, D, 16, a, b, torch.bfloat16)["host_workgroups"] > 0
done([
    workers(64, 32, 8, 112, 1), workers(64, 32, 8, 100, 2), workers(64, 32, 8, 112, 112),
    workers(40, 8, 1, 178, 10), workers(12, 16, 8, 88, 5), workers(12, 16, 8, 59, 5),
    workers(2, 32, 8, 46, 11), workers(2, 32, 8, 22, 11), workers(2, 32, 8, 22, 44),
    workers(24, 32, 8, 31, 31), workers(24, 32, 8, 32, 32), workers(24, 32, 8, 16, 32),
    workers(64, 16, 16, 32, 32), workers(33, 32, 32, 63, 63), workers(33, 32, 32, 64, 64),
    workers(65, 32, 8, 112, 1)])
""")
    assert got == [True, True, True,
                   False, True, False,
                   False, False, True,
                   False, True, True,
                   True, False, True,
                   False]


def test_uncounted_launches_are_cut_by_length_where_that_pays_for_the_clearing(planner):
    """A launch that the cut by width leaves whole, counted and not: a table
    of 28, 48 and 49 blocks; one whose rows it splits."""
    got = planner("""
def parts(n, H, KVH, W, counted):
    return ops.split_plan_info(n, H, KVH, 128, 16, W, 0, torch.float16, counted=counted,
                               host_pinned=False)["balanced_parts"] > 0
done([parts(2, 32, 32, w, c) for w in (28, 44, 48, 49, 512) for c in (True, False)])
""")
    assert got == [False, False, True, False, True, False, True, True, True, True]
