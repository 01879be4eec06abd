"""The server's copies and launches are waited for before a job ends, on whichever stream they were queued
(tests/server_order.c runs the library against HIP calls of its own that only count; no GPU)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "muscle.jl_amd", "lib")


def test_nothing_queued_after_a_job(tmp_path):
    if not shutil.which("gcc"):
        pytest.skip("needs gcc")
    exe = str(tmp_path / "server_order")
    # -rdynamic: the library's HIP calls find the program's definitions first
    subprocess.run(["gcc", "-O1", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "server_order.c"), "-o", exe,
                    "-L" + LIB, "-lmuscle_hip", "-Wl,-rpath," + LIB, "-Wl,-rpath-link,/opt/rocm/lib",
                    "-Wl,--allow-shlib-undefined", "-lpthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.startswith("ok: 32 jobs"), r.stdout + r.stderr
