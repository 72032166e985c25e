"""The library's host-side copies and batches (vq_amd/csrc/vq_api_host.hip and host_batch.hpp: the copying
threads and their lock-free queues, staged copies, the pipeline of host rows) WITHOUT a GPU, under the
thread sanitizer and under the address and undefined-behaviour sanitizers: a C++ driver
(tests/stub/host_copies_main.cpp) compiled by g++ against a stand-in for the HIP runtime (tests/stub/cpu_hip)
with two devices and streams that are threads."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STUB = os.path.join(ROOT, "tests", "stub")


@pytest.mark.parametrize("sanitize", ["thread", "address,undefined"])
def test_host_copies_under_sanitizers(tmp_path, sanitize):
    exe = str(tmp_path / "host_copies")
    flags = ["-O2", "-g", "-std=c++17", "-fno-omit-frame-pointer", "-fsanitize=" + sanitize, "-Wall",
             "-Wno-unused-function", "-I", os.path.join(STUB, "cpu_hip")]
    subprocess.check_call(["g++", *flags, os.path.join(STUB, "host_copies_main.cpp"), "-o", exe, "-lpthread"])
    # the harness preloads a library of its own; the sanitizer's runtime has to come first
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:abort_on_error=0:verify_asan_link_order=0",
               UBSAN_OPTIONS="halt_on_error=1:print_stacktrace=1", TSAN_OPTIONS="halt_on_error=1:exitcode=66")
    res = subprocess.run([exe], env=env, capture_output=True, text=True, timeout=300)
    if "unexpected memory mapping" in res.stderr:
        pytest.skip("the sanitizer's runtime does not start under this kernel's address layout")
    assert res.returncode == 0, res.stdout[-2000:] + res.stderr[-4000:]
    assert "host copies: ok" in res.stdout
    assert "Sanitizer" not in res.stderr and "runtime error" not in res.stderr
