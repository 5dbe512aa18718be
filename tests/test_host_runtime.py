"""The library's host code (handles, device memory, server) over a HIP runtime
of host memory with two devices (tests/hostrt): the device a block belongs to,
calls where device memory runs out, and what a server's budget holds."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
DIR = os.path.join(HERE, "hostrt")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")

CASES = ["pool_device", "pool_bound", "handle_device", "row_plan", "error_flags",
         "label_on_a_full_device", "label_without_lists",
         "server_budget", "state_on_a_full_device", "phases_read_back",
         "trajectory_launches", "waveforms_memory", "failed_growth", "trim", "server_device"]


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    out = tmp_path_factory.mktemp("hostrt")
    flags = ["-std=c++17", "-O1", "-g", "-ffp-contract=off", "-pthread", "-D__HIP_PLATFORM_AMD__",
             "-I" + os.path.join(ROCM, "include"), "-I" + os.path.join(ROOT, "include"),
             "-fsanitize=address"]
    srcs = [os.path.join(ROOT, "dsim_amd", "csrc", s)
            for s in ("host.cpp", "sim.cpp", "phase.cpp", "serve.cpp")]
    srcs += [os.path.join(DIR, s) for s in ("stub_hip.cpp", "driver.cpp")]
    objs, jobs = [], []
    for s in srcs:
        objs.append(str(out / (os.path.basename(s) + ".o")))
        jobs.append(subprocess.Popen(["g++", *flags, "-c", s, "-o", objs[-1]],
                                     stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True))
    for j in jobs:
        log = j.communicate()[0]
        assert j.returncode == 0, log[-4000:]
    exe = str(out / "driver")
    r = subprocess.run(["g++", "-fsanitize=address", "-pthread", "-o", exe, *objs],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    return exe


@pytest.mark.parametrize("case", CASES)
def test_host_runtime(driver, case):
    env = dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0:detect_leaks=0")
    r = subprocess.run([driver, case], capture_output=True, text=True, timeout=120, env=env)
    assert r.returncode == 0 and f"{case}: ok" in r.stdout, r.stdout + r.stderr[-4000:]
