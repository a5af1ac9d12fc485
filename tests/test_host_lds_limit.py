"""The allowance of dynamic LDS on the CPU, with the runtime's calls replaced:
asked for once on each device, not at all for a launch within the default, and
a refusal is reported and asked for again."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cstdio>
#include "lds_limit.h"

static int device = 0, calls[80], most = 0;
static bool refuse = false;
extern "C" {
hipError_t hipGetDevice(int* d) {
    *d = device;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int bytes) {
    calls[device]++;
    most = bytes;
    return refuse ? hipErrorInvalidValue : hipSuccess;
}
}

#define CHECK(x)                                    \
    if (!(x)) {                                     \
        std::printf("line %d: %s\n", __LINE__, #x); \
        return 1;                                   \
    }

int main() {
    life::LdsLimit l;
    l.allow(nullptr, 64 * 1024, 128 * 1024);
    CHECK(calls[0] == 0);
    for (int d : {0, 3, 0, 63, 3}) {
        device = d;
        l.allow(nullptr, 100000, 128 * 1024);
        CHECK(calls[d] == 1 && most == 128 * 1024);
    }
    device = 1;
    refuse = true;
    bool threw = false;
    try {
        l.allow(nullptr, 100000, 128 * 1024);
    } catch (const life::HipError&) {
        threw = true;
    }
    CHECK(threw && calls[1] == 1);
    refuse = false;
    l.allow(nullptr, 100000, 128 * 1024);
    l.allow(nullptr, 100000, 128 * 1024);
    CHECK(calls[1] == 2);
    device = 70;
    l.allow(nullptr, 100000, 128 * 1024);
    CHECK(calls[70] == 1);
}
"""


def test_allowance_per_device(tmp_path):
    src, exe = tmp_path / "lds.cpp", tmp_path / "lds"
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I",
                           os.path.join(ROOT, "life_amd", "csrc"), "-I", "/opt/rocm/include", "-o", str(exe), str(src)])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
