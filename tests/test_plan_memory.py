"""The memory of the library's plans, on the CPU (plan_memory.cpp: the set-up functions of
libmbgpu.so over a host stand-in of the runtime's memory calls; nothing is launched).

* A device allocation that fails, at every place where one is made, is an error of that call
  alone: the calls that follow, with the parameters before or the same ones again, find every
  buffer, large enough and with their own plan's contents.
* A set-up with the parameters of the one before makes no allocation and no free, and the key of
  the captured evaluation stays as it is.
* The server's estimate of a cluster's memory counts its neighbour rows as large as they are.
* MBGPU_POISON=1 fills every buffer of floating-point numbers, whatever their element type.
"""
import importlib
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "dlpoly2-mbpol-heat_amd")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is not installed")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan_memory") / "plan_memory")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-I", os.path.join(PKG, "csrc"),
                    os.path.join(HERE, "plan_memory.cpp"), "-x", "none", "-o", exe, "-L", PKG, "-lmbgpu",
                    "-Wl,-rpath," + PKG], check=True, capture_output=True, text=True)
    return exe


def run(program, *args, env=()):
    r = subprocess.run([program, *args], capture_output=True, text=True, timeout=600, env={**os.environ, **dict(env)})
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.stdout + r.stderr)[:4000]


@pytest.mark.parametrize("part", ["elec", "water", "mbpol"])
def test_failed_allocations(program, part):
    run(program, part + "_failures")


def test_repeated_calls_allocate_nothing(program):
    run(program, "elec_repeats")


def test_poison_fills_every_floating_point_buffer(program):
    run(program, "elec_poison", env={"MBGPU_POISON": "1"})


@pytest.mark.parametrize("nw", [16, 112, 704])
def test_server_counts_the_rows_of_a_cluster(program, nw):
    serve = importlib.import_module("dlpoly2-mbpol-heat_amd.serve")
    r = subprocess.run([program, "cluster_rows", str(nw)], capture_output=True, text=True, timeout=60, check=True)
    assert serve.slot_bytes(nw, cluster=True) - serve.slot_bytes(nw) == int(r.stdout.split()[0])
