"""Host rules of the kernels' launchers, compiled against a fake runtime: what they ask of and set on a
device (csrc/kernels/device.h), and which prompt rows go chunkwise (csrc/kernels/chunk_rows.h)."""
import os
import subprocess

import pytest

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

RULE = """
#include <initializer_list>
#include "chunk_rows.h"
using kgc::chunk_rows_pay;
#define CHECK(x) if (!(x)) return __LINE__
int main() {
  for (long alone : {32, 48}) {
    CHECK(!chunk_rows_pay(0, 0, alone) && !chunk_rows_pay(1, 24, alone) && chunk_rows_pay(1, alone, alone));
    for (long P = 1; P <= 1024; ++P) {
      CHECK(!chunk_rows_pay(P, 8 * P, alone) && !chunk_rows_pay(P, P, alone) && chunk_rows_pay(P, 48 * P, alone));
      for (long n = 1, was = 0; n <= 64; ++n) {    // longer rows never go back
        const bool now = chunk_rows_pay(P, n * P, alone);
        CHECK(now >= was);
        was = now;
      }
    }
    CHECK(chunk_rows_pay(128, 128 * 12, alone) && !chunk_rows_pay(32, 32 * 12, alone) && chunk_rows_pay(32, 512, alone));
  }
  return 0;
}
"""


def _run(tmp_path, program):
    os.mkdir(tmp_path / "hip")
    (tmp_path / "hip" / "hip_runtime.h").write_text(RUNTIME)
    (tmp_path / "main.cpp").write_text(program)
    exe = str(tmp_path / "main")
    subprocess.run(["g++", "-std=c++17", "-I", str(tmp_path), "-I", os.path.join(ROOT, "csrc", "kernels"),
                    str(tmp_path / "main.cpp"), "-o", exe], check=True)
    assert subprocess.run([exe]).returncode == 0


def test_devices_are_asked_one_by_one(tmp_path):
    _run(tmp_path, PROGRAM)


def test_short_rows_stay_token_by_token(tmp_path):
    """Hundreds of chunks of one to eight rows used to go chunkwise from 1024 rows on."""
    _run(tmp_path, RULE)


@pytest.mark.parametrize("cost, H, V, alone", [("4.0, 0.0062, 0.0, 0.85, 0.0021, 20.6, 0.0, 16.5, 0.037, 0.0, 8", 16, 128, 48),
                                               ("6.1, 0.0148, 2.0, 0.72, 0.0014, 13.6, 0.0247, 0.0, 0.0, 0.0147, 3", 8, 256, 32)],
                         ids=["delta", "gla"])
def test_costs_only_add_to_steps_below_1024_rows(tmp_path, cost, H, V, alone):
    """The memory profile has the chunks of the rule by rows from 1024 rows on, and of `least` rows each below."""
    _run(tmp_path, """
#include "chunk_rows.h"
using kgc::chunk_rows_pay;
#define CHECK(x) if (!(x)) return __LINE__
int main() {
  constexpr kgc::ChunkCost cost{%s};
  const long H = %d, V = %d, alone = %d;
  CHECK(!chunk_rows_pay(cost, 0, 0, H, V, alone));
  bool more = false;
  for (long P = 1; P <= 1024; ++P)
    for (long Tp = P; Tp <= 64 * P; ++Tp) {
      const bool rows = chunk_rows_pay(P, Tp, alone), both = chunk_rows_pay(cost, P, Tp, H, V, alone);
      CHECK(both || !rows);
      CHECK(both == rows || (Tp < 1024 && Tp >= cost.least * P));
      more = more || both != rows;
    }
  CHECK(more);
  return 0;
}
""" % (cost, H, V, alone))


def test_chunk_offsets_fit_their_types(tmp_path):
    """A row stride of 2^25 elements (a view of a wide buffer) overflowed the offset of the chunk's last
    row, and so many heads the grid: both stay token by token."""
    _run(tmp_path, """
#include <cstdint>
#include "chunk_rows.h"
using kgc::chunk_fits;
#define CHECK(x) if (!(x)) return __LINE__
int main() {
  CHECK(chunk_fits(2 * 65536 + 3 * 131072, 131072, 1024));                     // far beyond any model
  CHECK(!chunk_fits(1L << 25, 2048, 16) && !chunk_fits(1L << 40, 2048, 16));
  CHECK(!chunk_fits(4096, 2048, 65536) && !chunk_fits(4096, 1L << 23, 16));
  for (long x = 1; x < (1L << 40); x += x / 3 + 1) {     // what is taken stays inside its type
    if (chunk_fits(x, 16, 1)) CHECK(63 * x + 256 <= INT32_MAX && x < (1 << 23));
    if (chunk_fits(16, x, 1)) CHECK(255 * x + x <= INT32_MAX && 63 * x <= INT32_MAX && (x + 15) / 16 <= 65535);
  }
  return 0;
}
""")
