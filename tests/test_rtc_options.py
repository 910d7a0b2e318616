"""Compiler options of the generated kernels: a hipRTC that does not know a named scheduler must
compile with its own default. LLVM's option parser ends the process at a value it rejects, so
the compilations run in a child process."""

import os
import re
import subprocess
import sys

import pytest

import heyoka_amd as hy

CSRC = os.path.join(os.path.dirname(os.path.abspath(hy.__file__)), "csrc")
OPTIONS = re.findall(r'"-mllvm",\s*"([^"]+)"', open(os.path.join(CSRC, "hyx_runtime.cpp")).read())

CHILD = """
import ctypes as ct, os, sys
L = ct.CDLL("libhiprtc.so.7" if not os.path.exists("/opt/rocm/lib/libhiprtc.so") else "/opt/rocm/lib/libhiprtc.so")
prog = ct.c_void_p()
src = b'extern "C" __global__ void k(double *x) { x[threadIdx.x] *= 2.0; }'
assert L.hiprtcCreateProgram(ct.byref(prog), src, b"k.hip", 0, None, None) == 0
opts = [b"--offload-arch=gfx950", b"-O3", b"-mllvm", sys.argv[1].encode()]
assert L.hiprtcCompileProgram(prog, len(opts), (ct.c_char_p * len(opts))(*opts)) == 0
print("compiled")
"""


def test_the_options_are_found():
    assert len(OPTIONS) >= 2


@pytest.mark.parametrize("opt", OPTIONS + [o.split("=")[0] + "=no-such-name" for o in OPTIONS if "=" in o])
def test_known_and_unknown_values_compile(opt):
    r = subprocess.run([sys.executable, "-c", CHILD, opt], capture_output=True, text=True)
    assert r.returncode == 0 and "compiled" in r.stdout, r.stderr
