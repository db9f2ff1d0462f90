"""lds_allow (csrc/lds_allow.cpp): dynamic LDS above 64 KB is asked for once per kernel, size and
device. Compiled here with stand-ins for the runtime's two calls; no GPU."""
import os
import shutil
import subprocess

import pytest

from conftest import PKG

MAIN = r"""
#include "lds_allow.h"
#include <stdio.h>
static int device = 0, asked = 0, fails = 0, last = 0;
extern "C" hipError_t hipGetDevice(int * d) { *d = device; return hipSuccess; }
extern "C" hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int v) {
    asked++;
    last = v;
    return fails ? hipErrorInvalidValue : hipSuccess;
}
namespace sparkmv {
int fail_hip(const char *, hipError_t) { return -1; }
}
using namespace sparkmv;
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main() {
    static LdsAllowed a, b;
    CHECK(lds_allow(a, nullptr, 65536, "") == 0 && asked == 0);
    CHECK(lds_allow(a, nullptr, 65537, "") == 0 && asked == 1 && last == 65537);
    CHECK(lds_allow(a, nullptr, 65537, "") == 0 && asked == 1);
    CHECK(lds_allow(a, nullptr, 90000, "") == 0 && asked == 2);
    CHECK(lds_allow(a, nullptr, 70000, "") == 0 && asked == 2);   /* less than allowed: not taken back */
    device = 1;                                                    /* another device asks for itself */
    CHECK(lds_allow(a, nullptr, 70000, "") == 0 && asked == 3 && last == 70000);
    device = 0;
    CHECK(lds_allow(a, nullptr, 90000, "") == 0 && asked == 3);
    CHECK(lds_allow(b, nullptr, 70000, "") == 0 && asked == 4);   /* another kernel too */
    fails = 1;
    CHECK(lds_allow(a, nullptr, 100000, "") == -1 && asked == 5);
    CHECK(lds_allow(a, nullptr, 100000, "") == -1 && asked == 6);  /* a refusal is not kept */
    device = 64;                                                    /* past the table: asked each time */
    fails = 0;
    CHECK(lds_allow(a, nullptr, 70000, "") == 0 && lds_allow(a, nullptr, 70000, "") == 0 && asked == 8);
    return 0;
}
"""


def test_allowance_per_kernel_and_device(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    include = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(hipcc))), "include")
    if not os.path.exists(os.path.join(include, "hip", "hip_runtime.h")):
        pytest.skip("no HIP headers")
    csrc, main, exe = os.path.join(PKG, "csrc"), tmp_path / "main.cpp", tmp_path / "lds_allow"
    main.write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", include, "-I", csrc, str(main),
                    os.path.join(csrc, "lds_allow.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
