"""The regrouping of the upward tables (host code of the upload): its result and its failures."""
import os
import subprocess

from conftest import ROOT


def test_grouped_tables_and_failing_allocations(tmp_path):
    exe = tmp_path / "up_groups_check"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-pthread", "-o", str(exe),
                           os.path.join(ROOT, "tests", "up_groups_check.cpp")])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)
