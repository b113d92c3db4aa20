"""Rsteps per launch, and what follows from them: a plan's memory, the batches
its searches launch, admission (tests/native/plan_check.cpp: the host logic
against a stand-in of the HIP runtime)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "prestozl_amd", "csrc")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("plan") / "plan_check")
    stub = os.path.join(HERE, "native", "hipstub")
    cmd = ["g++", "-std=c++17", "-O1", "-g", "-pthread", "-I" + stub, "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
           os.path.join(stub, "hipstub.cpp"), os.path.join(HERE, "native", "plan_check.cpp")]
    cmd += [os.path.join(CSRC, f) for f in ("pzl_engine.cpp", "pzl_server.cpp", "pzl_geometry.cpp", "pzl_stats.cpp")]
    r = subprocess.run(cmd + ["-o", out], capture_output=True, text=True, timeout=600)
    if r.returncode != 0:
        pytest.fail("build failed:\n" + r.stderr[-3000:])
    return out


@pytest.mark.parametrize("check", ["exact", "rule", "memory", "server", "overflow", "deadline", "tuner", "pinned",
                                   "row_sets"])
def test_plan(exe, check):
    r = subprocess.run([exe, check], capture_output=True, text=True, timeout=300)
    print(r.stdout[-3000:], r.stderr[-3000:])
    assert r.returncode == 0
