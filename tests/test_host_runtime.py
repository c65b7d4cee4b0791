"""The library's host code on the CPU: every source of libavionic.so compiled for
the host alone, with AddressSanitizer and UndefinedBehaviorSanitizer, over a
stand-in HIP runtime (tests/sanitize/hip_stub.cpp) whose kernels do nothing.
Each scenario of tests/sanitize/engine_host.cpp is one run; a sanitizer report,
an objection of the stand-in (an executable destroyed before its stream was
waited for, a call that a capture forbids, a launch out of range), device memory
left allocated or a failed check fails it."""
import concurrent.futures as cf
import glob
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
CLANG = "/opt/rocm/llvm/bin/clang++"
SAN = "-fsanitize=address,undefined"
ENV = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:detect_stack_use_after_return=1",
           UBSAN_OPTIONS="print_stacktrace=1:halt_on_error=1")

pytestmark = pytest.mark.skipif(not (os.path.exists(HIPCC) and os.path.exists(CLANG)),
                                reason="no ROCm compiler")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = tmp_path_factory.mktemp("host")
    csrc = os.path.join(ROOT, "avionic_amd", "csrc")
    here = os.path.join(ROOT, "tests", "sanitize")

    def host_object(src):
        obj = str(out / (os.path.basename(src) + ".o"))
        r = subprocess.run([HIPCC, "-c", "-x", "hip", "--cuda-host-only", "--offload-arch=gfx950",
                            "-O1", "-g", "-std=c++17", "-w", "-Xarch_host", SAN,
                            "-I" + os.path.join(ROOT, "include"), src, "-o", obj],
                           capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-4000:]
        return obj

    srcs = glob.glob(os.path.join(csrc, "*.cpp")) + glob.glob(os.path.join(csrc, "*.hip"))
    with cf.ThreadPoolExecutor(8) as ex:
        objs = list(ex.map(host_object, sorted(srcs)))
    exe = str(out / "engine_host")
    # the device binaries that the host code would register do not exist here
    r = subprocess.run([CLANG, "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-O1", "-g", SAN,
                        "-I/opt/rocm/include", os.path.join(here, "engine_host.cpp"),
                        os.path.join(here, "hip_stub.cpp"), *objs, "-o", exe, "-lpthread",
                        "-Wl,--unresolved-symbols=ignore-all"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    return exe


@pytest.mark.parametrize("scenario", ["mixed", "variants", "capture_error", "launch_sets",
                                      "budget", "out_of_memory", "host_memory"])
def test_engine_host(exe, scenario):
    r = subprocess.run([exe, scenario], capture_output=True, text=True, timeout=240, env=ENV)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-6000:]
    assert f"{scenario} ok" in r.stdout
