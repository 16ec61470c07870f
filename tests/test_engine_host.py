"""The engine's host code (stream contexts, output pools, copies to the host)
over a stand-in device: streams are host threads, kernels are replaced by work
that is easy to check (tests/host).  No GPU."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host")


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host") / "engine_host_test")
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    include = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(hipcc))), "include")
    r = subprocess.run(
        ["g++", "-std=c++17", "-O1", "-pthread", "-Wall", "-Wno-subobject-linkage", "-Wno-attributes",
         "-D__HIP_PLATFORM_AMD__", "-isystem", include, "-D__align__(x)=__attribute__((aligned(x)))",
         "-DHIP_SYMBOL(x)=(&(x))", "engine_host_test.cpp", "stub_device.cpp", "-o", exe],
        cwd=HERE, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def run(case, *args, timeout=60):
        p = subprocess.run([exe, case, *map(str, args)], capture_output=True, text=True, timeout=timeout)
        assert p.returncode == 0, p.stdout + p.stderr

    return run


def test_shared_pool_sequence(host):
    """Two contexts on one pool: passes, digests and a copy of the last outputs,
    the context that made the pool closed first."""
    host("shared_pool_sequence", 3)


def test_shared_pool_on_two_threads(host):
    host("shared_pool_threads", 30)


def test_shared_pool_without_graphs(host):
    host("shared_pool_without_graphs")


def test_failed_copy_leaves_nothing_in_flight(host):
    host("failed_copy_leaves_nothing_in_flight")


def test_waiting_for_the_device_is_idle(host):
    host("waiting_for_the_device_is_idle")


def test_arrays_at_chunk_edges(host):
    host("arrays_at_chunk_edges")
