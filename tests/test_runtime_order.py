"""The host side of poly_hip_order_after without a GPU: the runtime's own code against a HIP
runtime that tests/runtime_order_main.cc acts out.  Events are kept per call in flight and not
per thread, belong to the device of the stream they are recorded on whatever device the
caller is on, and one that a capture has seen is not recorded on another stream."""
import os
import subprocess

import pytest

import hostcheck

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "polygrad_amd", "csrc")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("order") / "runtime_order")
    subprocess.run([hostcheck.CLANG, "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + CSRC, "-I" + os.path.join(CSRC, "..", "..", "include"), os.path.join(HERE, "runtime_order_main.cc"), os.path.join(CSRC, "runtime_hip.cc"),
                    "-o", out, "-L/opt/rocm/lib", "-lamdhip64", "-lhiprtc", "-lpthread", "-Wl,-rpath,/opt/rocm/lib"], check=True)
    return out


@pytest.mark.skipif(not os.path.exists(hostcheck.CLANG), reason="no host clang with AddressSanitizer")
@pytest.mark.parametrize("what", ["threads", "device", "capture"])
def test_order_after(driver, what):
    r = subprocess.run([driver, what], capture_output=True, text=True, timeout=60, env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
