"""Loads the built library over tests/cpp/fake_hip.cc, the host-only stand-in
of the HIP runtime: for a process of its own (the real runtime must not be
loaded in it), started by test_host_runtime.py with the stand-in's path."""
import ctypes as C
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def build(path):
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-w", "-I", os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"),
                    "-Wl,-soname,libamdhip64.so.7", "-o", path,
                    os.path.join(ROOT, "tests", "cpp", "fake_hip.cc")], check=True)


class FakeHip:
    def __init__(self, path):
        self.lib = C.CDLL(path, mode=C.RTLD_GLOBAL)
        self.lib.fake_hip_log.restype = C.c_char_p
        self.lib.fake_hip_cost.argtypes = [C.c_char_p, C.c_float]
        sys.path.insert(0, ROOT)

    def reset(self):
        self.lib.fake_hip_reset()

    def log(self):
        """What was launched, copied and waited for since the reset."""
        return self.lib.fake_hip_log().decode().split()

    def fail(self, kernel):
        self.lib.fake_hip_fail(kernel.encode())

    def cost(self, kernel, ms):
        self.lib.fake_hip_cost(kernel.encode(), ms)


def launches(log, *kernels):
    """Positions of the launches of a kernel whose name holds one of these."""
    return [i for i, l in enumerate(log) if any(k in l for k in kernels)]
