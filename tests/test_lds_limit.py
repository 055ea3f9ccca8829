"""Kernels of more than 64 KiB of dynamic LDS (csrc/zq3d_lds.h), compiled with g++ against a HIP runtime of host
functions: every device is asked once, a refusal is reported and asked again, and no launcher keeps the
answer of one device for all."""
import glob
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "zq_smokesimulation_amd", "csrc")

FAKE = r"""
#pragma once
typedef int hipError_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1 };
enum hipFuncAttribute { hipFuncAttributeMaxDynamicSharedMemorySize = 8 };
inline int fake_device = 0, fake_calls[70] = {}, fake_bytes = 0;
inline bool fake_refuse = false;
inline hipError_t hipGetDevice(int* d) { *d = fake_device; return hipSuccess; }
inline hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int bytes) {
    fake_calls[fake_device]++;
    fake_bytes = bytes;
    return fake_refuse ? hipErrorInvalidValue : hipSuccess;
}
"""
MAIN = r"""
#include "zq3d_lds.h"
#include <cstdio>
#include <initializer_list>
#define CHECK(c) do { if (!(c)) return std::printf("line %d: %s\n", __LINE__, #c), 1; } while (0)
int main() {
    static zq3d::LdsLimit one, other;
    for (int dev : {0, 3, 63, 64, 0, 3, 63, 0}) {
        fake_device = dev;
        CHECK(one.raise(nullptr, 99000) == hipSuccess && fake_bytes == 99000);
    }
    CHECK(fake_calls[0] == 1 && fake_calls[3] == 1 && fake_calls[63] == 1 && fake_calls[64] == 1);
    fake_device = 0;
    fake_refuse = true;
    CHECK(other.raise(nullptr, 70000) == hipErrorInvalidValue && other.raise(nullptr, 70000) == hipErrorInvalidValue);
    fake_refuse = false;
    CHECK(other.raise(nullptr, 70000) == hipSuccess && other.raise(nullptr, 70000) == hipSuccess);
    CHECK(fake_calls[0] == 4);
    std::printf("ok\n");
    return 0;
}
"""


def test_each_device_is_asked(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(FAKE)
    src = tmp_path / "lds.cpp"
    src.write_text(MAIN)
    exe = str(tmp_path / "lds")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", str(tmp_path), "-I", CSRC, str(src), "-o", exe],
                   check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout


def test_launchers_keep_no_answer_per_process():
    for path in glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.cpp")):
        with open(path) as f:
            assert not re.search(r"hipFuncSetAttribute", f.read()), path
