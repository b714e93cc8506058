"""csrc/kernels/device.h: what launches ask of and set on a device, compiled against a fake runtime."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
RUNTIME = """
#pragma once
#include <cstddef>
enum hipError_t { hipSuccess, hipErrorInvalidValue };
enum { hipDeviceAttributeMultiprocessorCount, hipFuncAttributeMaxDynamicSharedMemorySize };
extern int device, calls[100], cus[100], asked, refuse;
extern hipError_t last;
inline hipError_t hipGetDevice(int* d) { *d = device; return hipSuccess; }
inline hipError_t hipDeviceGetAttribute(int* n, int, int d) { ++asked; *n = cus[d]; return hipSuccess; }
inline hipError_t hipFuncSetAttribute(const void*, int, int) {
  ++calls[device];
  return last = refuse ? hipErrorInvalidValue : hipSuccess;
}
inline hipError_t hipGetLastError() { hipError_t e = last; last = hipSuccess; return e; }
"""
PROGRAM = """
#include "device.h"
int device, calls[100], cus[100], asked, refuse;
hipError_t last;
void kernel() {}
#define CHECK(x) if (!(x)) return __LINE__
int main() {
  static kgc::OncePerDevice once, other;
  refuse = 1;                                   // refused: no route, no error left, asked again
  CHECK(!kgc::allow_lds(once, &kernel, 100000) && last == hipSuccess);
  refuse = 0;
  for (device = 0; device < 3; ++device)        // each device by itself, once
    for (int i = 0; i < 3; ++i) CHECK(kgc::allow_lds(once, &kernel, 100000));
  CHECK(calls[0] == 2 && calls[1] == 1 && calls[2] == 1);
  device = 1;                                   // another kernel has its own
  CHECK(kgc::allow_lds(other, &kernel, 100000) && calls[1] == 2);
  device = 99;                                  // beyond the table: every time
  CHECK(kgc::allow_lds(once, &kernel, 1) && kgc::allow_lds(once, &kernel, 1) && calls[99] == 2);
  for (int d = 0; d < 100; ++d) cus[d] = 32 + d;
  for (device = 0; device < 4; ++device)
    for (int i = 0; i < 3; ++i) CHECK(kgc::device_cus() == 32 + device);
  CHECK(asked == 4);
  return 0;
}
"""


def test_devices_are_asked_one_by_one(tmp_path):
    os.mkdir(tmp_path / "hip")
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (tmp_path / "main.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "main")
    subprocess.run(["g++", "-std=c++17", "-I", str(tmp_path), "-I", os.path.join(ROOT, "csrc", "kernels"),
                    str(tmp_path / "main.cpp"), "-o", exe], check=True)
    assert subprocess.run([exe]).returncode == 0
