"""Host code of the upload in C++ programs of its own: the regrouping of the upward tables, its result and
its failures, and device memory for several arrays at once (no GPU)."""
import os
import subprocess

from conftest import ROOT


def test_grouped_tables_and_failing_allocations(tmp_path):
    exe = tmp_path / "up_groups_check"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-pthread", "-o", str(exe),
                           os.path.join(ROOT, "tests", "up_groups_check.cpp")])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)


def test_device_memory_for_all_arrays_or_none(tmp_path):
    exe = tmp_path / "device_alloc_check"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__",
                           "-I/opt/rocm/include", "-o", str(exe),
                           os.path.join(ROOT, "tests", "device_alloc_check.cpp")])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)
