"""The library's host code (threads on one context, staging, captures) on the
CPU: its sources compiled for the host alone and linked with a stand-in of the
HIP calls they make (tests/native/host_hip.cpp)."""
import os
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from sister_amd import build as B

NATIVE = os.path.join(B.ROOT, "tests", "native")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host_calls"))
    srcs = [os.path.join(B.CSRC, s) for s in B.SOURCES] + [
        os.path.join(NATIVE, s) for s in ("host_hip.cpp", "host_calls_check.cpp")]

    def compile_one(src):
        obj = os.path.join(out, os.path.basename(src) + ".o")
        subprocess.run([B.HIPCC, "-x", "hip", f"--offload-arch={B.ARCH}", "--offload-host-only", "-O1", "-std=c++17",
                        "-I", os.path.join(B.ROOT, "include"), "-c", src, "-o", obj], check=True)
        return obj

    with ThreadPoolExecutor(4) as pool:
        objs = list(pool.map(compile_one, srcs))
    # the device code images that a full build would link in
    names = set(re.findall(r"__hip_fatbin_\w+", subprocess.run(["nm", "-u", *objs], capture_output=True, text=True,
                                                               check=True).stdout))
    exe = os.path.join(out, "host_calls_check")
    subprocess.run(["g++", *objs, *[f"-Wl,--defsym={n}=0" for n in sorted(names)], "-no-pie", "-lpthread", "-o", exe],
                   check=True)
    return exe


@pytest.mark.parametrize("name", ["host_form_threads", "host_form_beside_batches", "host_form_refused",
                                  "forms_capture_once", "graph_branches"])
def test_host_calls(check, name, tmp_path):
    r = subprocess.run([check, name, str(tmp_path / "file")], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.returncode, r.stdout + r.stderr)
