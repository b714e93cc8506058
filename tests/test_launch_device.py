"""Host rules of the kernels' launchers, compiled against a fake runtime: what they ask of and set on a
device (csrc/kernels/device.h), which prompt rows go chunkwise (csrc/kernels/chunk_rows.h), and how decode contexts are cut
into slices (csrc/kernels/decode_slices.h, ops.decode_grid_z)."""
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


@pytest.mark.parametrize("op, H, V, alone, least", [("delta", 16, 128, 48, 8), ("gla", 8, 256, 32, 3)])
def test_costs_only_add_to_steps_below_1024_rows(tmp_path, op, H, V, alone, least):
    """The costs take no step back that the rows send chunkwise, and add none from 1024 rows on nor of fewer than `least`
    rows per sequence."""
    _run(tmp_path, """
#include "chunk_rows.h"
using kgc::chunk_rows_pay, kgc::%s_rows_pay;
#define CHECK(x) if (!(x)) return __LINE__
int main() {
  const long H = %d, V = %d, alone = %d, least = %d;
  CHECK(!%s_rows_pay(0, 0, H, V));
  bool more = false;
  for (long P = 1; P <= 1024; ++P)
    for (long Tp = P; Tp <= 64 * P; ++Tp) {
      const bool rows = chunk_rows_pay(P, Tp, alone), both = %s_rows_pay(P, Tp, H, V);
      CHECK(both || !rows);
      CHECK(both == rows || (Tp < 1024 && Tp >= least * P));
      more = more || both != rows;
    }
  CHECK(more);
  return 0;
}
""" % (op, H, V, alone, least, op, op))


def test_memory_profile_has_the_chunks_of_every_small_step(tmp_path):
    """No step of fewer than 1024 rows that goes chunkwise starts more chunks than the ones that the memory profile
    runs and that go chunkwise, too, by the rules of the kernels, for any heads, budget and number of slots: the profile had
    prompts of three and of eight rows, where the costs often say token by token."""
    from types import SimpleNamespace

    from kubernetes_gpu_cluster_amd.engine.model_runner import ModelRunner
    cases = []
    for H, V in ((2, 128), (4, 512), (8, 256), (16, 128), (16, 256), (32, 128), (32, 64), (64, 128)):
        for budget in (100, 512, 1024, 2048, 16384):
            for seqs, longest in ((16, 8192), (100, 8192), (512, 8192), (1024, 8192), (300, 60)):
                steps = ModelRunner._profile_steps(SimpleNamespace(
                    token_budget=budget, max_model_len=longest, max_num_seqs=seqs, state_layout=[((4, 64), (H, 128, V))]))
                assert all(sum(s) <= budget and len(s) <= seqs and max(s) <= longest and min(s) > 0 for s in steps)
                cases.append("{%d, %d, %d, %d, %d, {%s}}" % (H, V, budget, seqs, longest, ", ".join(
                    "{%d, %d}" % (len(s), sum(s)) for s in steps)))
    _run(tmp_path, """
#include <cstdio>
#include <vector>
#include "chunk_rows.h"
struct Case { long H, V, budget, seqs, longest; std::vector<kgc::ChunkStep> steps; };
int main() {
  const std::vector<Case> cases = {%s};
  int missed = 0;
  for (const Case& c : cases)
    for (auto pay : {kgc::delta_rows_pay, kgc::gla_rows_pay}) {
      long have = 0, most = 0;
      for (auto s : c.steps)
        if (pay(s.P, s.Tp, c.H, c.V) && s.Tp / 32 + s.P > have) have = s.Tp / 32 + s.P;
      for (long P = 1; P <= c.seqs; ++P)
        for (long Tp = P; Tp <= c.budget && Tp <= P * c.longest && Tp < 1024; ++Tp)
          if (Tp / 32 + P > most && pay(P, Tp, c.H, c.V)) most = Tp / 32 + P;
      if (have >= most) continue;
      ++missed;
      printf("%%s %%ld x %%ld, budget %%ld, %%ld slots: %%ld chunks profiled, %%ld possible\\n",
             pay == kgc::gla_rows_pay ? "gla" : "delta", c.H, c.V, c.budget, c.seqs, have, most);
    }
  return missed ? 1 : 0;
}
""" % ", ".join(cases))


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


DECODE = """
#define __host__
#define __device__
#define __forceinline__ inline
#include <initializer_list>
#include "decode_slices.h"
using namespace kgc;
#define CHECK(x) if (!(x)) return __LINE__
"""


def test_decode_slices_cover_the_context_and_keep_a_fixed_length(tmp_path):
    """Every chunk is in one of the slices that the merge reads, whatever the pairs, type and grid; a length set from
    outside holds for every context (4 and 16 were taken for the rule's own and changed)."""
    _run(tmp_path, DECODE + """
int main() {
  for (int fixed : {0, 1, 2, 3, 4, 8, 10, 16, 32})
    for (int64_t pairs : {64, 127, 128, 255, 256, 511, 512, 4096})
      for (bool fp8 : {false, true})
        for (int n = 0; n <= 300; ++n) {
          const int least = decode_min_chunks(decode_least(pairs, fp8, fixed), n);
          CHECK(least >= 2 && (fixed == 0 || least == (fixed < 2 ? 2 : fixed)));
          for (int Z : {1, 2, 3, 4, 7, 16, 32, 150}) {
            const int per = decode_slice_chunks(n, Z, least), used = decode_used_slices(n, Z, least);
            CHECK(per >= least && used <= Z && used * per >= n && (used == 0 ? n == 0 : (used - 1) * per < n));
          }
        }
  return 0;
}
""")


def test_decode_slices_of_a_row_much_longer_than_the_others(tmp_path):
    """Such a row is over last, so its slices are no longer than the grid asks for, 4 chunks, or an eighth of the row up
    to 8; from 256 pairs on 10 chunks, and from 512 on 16 where that is the whole row.  (One row of 500 tokens was two
    slices with 192 pairs and one with 384, and the step 17 to 27 % slower than in slices of 2 and 10 chunks.)"""
    _run(tmp_path, DECODE + """
int main() {
  for (int64_t pairs : {64, 127, 128, 192, 255, 256, 384, 511, 512, 768, 4096})
    for (int n = 1; n <= 300; ++n)
      for (int Z : {2, 3, 4, 9, 11, 16, 32, 150}) {
        const int ask = (n + Z - 1) / Z, eighth = (n + 7) / 8;
        const int most = pairs >= 512 && n <= 16 ? 16 : pairs >= 256 ? 10 : eighth < 4 ? 4 : eighth < 8 ? eighth : 8;
        CHECK(decode_slice_chunks(n, Z, decode_min_chunks(decode_least(pairs, false, 0), n)) <= (ask > most ? ask : most));
      }
  return 0;
}
""")


def test_decode_slices_of_middling_contexts(tmp_path):
    """Below 256 pairs contexts of up to 32 chunks are cut in fours (in twos 16 rows x 520 tokens 19.6 -> 21.9 us, in
    threes 24 x 640 25.7 -> 28.6)."""
    _run(tmp_path, DECODE + """
int main() {
  for (int64_t pairs : {64, 128, 192, 255}) {
    for (int n = 1; n <= 32; ++n) CHECK(decode_min_chunks(decode_least(pairs, false, 0), n) == 4);
    CHECK(decode_min_chunks(decode_least(pairs, false, 0), 33) == 5 && decode_min_chunks(decode_least(pairs, false, 0), 300) == 8);
    CHECK(decode_min_chunks(decode_least(pairs, true, 0), 20) == 2);
  }
  return 0;
}
""")


def test_decode_grids_of_33_to_63_pairs(monkeypatch):
    """On the 4-wave kernel at most 16 slices, and none more for up to 256 tokens (56 pairs x 200 8.7 -> 9.2 us)."""
    from kubernetes_gpu_cluster_amd import ops
    monkeypatch.setenv("KGC_DECODE_WAVE", "1")
    monkeypatch.delenv("KGC_DECODE_WAVE_MIN_PAIRS", raising=False)
    for B in (5, 6, 7):
        assert [ops.decode_grid_z(B, 8, c) for c in (200, 256)] == [1, 1]
        assert all(z <= max(16, -(-1024 // (8 * B))) for z in (ops.decode_grid_z(B, 8, c) for c in range(300, 8192, 100)))
    assert ops.decode_grid_z(4, 8, 200) == 4 and ops.decode_grid_z(4, 8, 4000) == 32


@pytest.mark.parametrize("wave,lim", [("1", None), ("0", None), ("1", "512")])
def test_decode_grids_fit_what_is_set_aside_for_them(monkeypatch, wave, lim):
    """Many slices are for steps of few (row, kv head) pairs: larger ones on the 4-wave kernel (K1w off, or from more pairs
    on) keep a slice per 256 tokens as long as that fills the CUs, and every grid fits the partial rows."""
    from kubernetes_gpu_cluster_amd import ops
    monkeypatch.setenv("KGC_DECODE_WAVE", wave)
    monkeypatch.delenv("KGC_DECODE_WAVE_MIN_PAIRS", raising=False)
    if lim:
        monkeypatch.setenv("KGC_DECODE_WAVE_MIN_PAIRS", lim)
    if wave == "0":
        assert [ops.decode_grid_z(256, 8, c) for c in (640, 8192)] == [1, 1] and ops.decode_grid_z(8, 8, 640) == 3
    for nkv in (1, 2, 8, 32):
        for B in (1, 2, 3, 5, 7, 8, 20, 63, 64, 300, 1024):
            for ctx in (32, 96, 160, 192, 544, 1000, 4000, 8192, 131072):
                z, pairs = ops.decode_grid_z(B, nkv, ctx), B * nkv
                assert 1 <= z <= ops.decode_max_z(-(-ctx // 32), 32)
                assert B * z <= ops.decode_partials(B, 1, 64, -(-ctx // 32), 32, "cpu")[0].numel()
                if not ops.decode_uses_wave(B, nkv):
                    assert (z == 1 or pairs * 4 * z <= 2 * 4096) and (pairs < 64 or z <= -(-4096 // (4 * pairs)))


def test_decode_graphs_have_few_empty_slices():
    """A graph's grid is for any context up to its capacity, and an empty slice costs what a short row does not get back:
    no more slices than one per 256 tokens of capacity, or 16, 8, 4 by the number of pairs; a step that knows its
    longest row has as many as help that row."""
    from kubernetes_gpu_cluster_amd import ops
    for pairs in range(1, 64):
        few = 16 if pairs <= 16 else 8 if pairs <= 32 else 4
        for ctx in (32, 160, 192, 300, 544, 1000, 2048, 4096, 8192, 131072):
            z, own = ops.decode_grid_z(pairs, 1, ctx, capacity=True), ops.decode_grid_z(pairs, 1, ctx)
            assert z <= max(few, min(-(-1024 // pairs), -(-ctx // 256))) and z <= own
    assert [ops.decode_grid_z(7, 8, c, capacity=True) for c in (544, 2048, 8192)] == [4, 8, 19]
    assert [ops.decode_grid_z(4, 8, c, capacity=True) for c in (544, 2048, 8192)] == [8, 8, 32]


def test_order_of_the_prompts_items(tmp_path):
    """The paged prompts' walk has every block of every work item and head group once; and where only the first blocks
    of the work items have rows (short prompts), every XCD has its share of them, and so has a workgroup in two rounds."""
    _run(tmp_path, """
#include <algorithm>
#include <cstdlib>
#include <initializer_list>
#include <set>
#include <tuple>
#include <vector>
#define __host__
#define __device__
#include "prefill_items.h"
#define CHECK(x) if (!(x)) return __LINE__
int main() {
  for (int groups : {1, 2, 3, 4, 6, 8, 16})
    for (int works : {1, 7, 100, 256})
      for (int grid : {96, 200, 512}) {
        const int n = works * groups * kgc::WALK_BLOCKS;
        std::set<std::tuple<int, int, int>> seen;
        for (int r = 0; r * grid < n; ++r)
          for (int b = 0; b < grid; ++b) {
            const int i = kgc::walk_index(r, b, grid, groups % 8 == 0);
            if (i >= n) continue;
            int w, block, g;
            kgc::walk_item(i, groups, w, block, g);
            CHECK(w >= 0 && w < works && block >= 0 && block < kgc::WALK_BLOCKS && g >= 0 && g < groups);
            seen.insert(std::make_tuple(w, block, g));
          }
        CHECK((int)seen.size() == n);
      }
  for (int groups : {1, 2, 4, 8})
    for (int blocks : {1, 2, 3}) {
      const int grid = 512, works = 2 * grid / (groups * kgc::WALK_BLOCKS);       // two rounds
      std::vector<int> of_wg(grid), of_xcd(8);
      for (int r = 0; r < 2; ++r)
        for (int b = 0; b < grid; ++b) {
          int w, block, g;
          kgc::walk_item(kgc::walk_index(r, b, grid, groups % 8 == 0), groups, w, block, g);
          const bool rows = block < blocks;
          of_wg[b] += rows, of_xcd[b & 7] += rows;
        }
      for (int x : of_xcd) CHECK(x == works * groups * blocks / 8);
      const auto most = std::max_element(of_wg.begin(), of_wg.end());
      CHECK(*most <= (blocks + 1) / 2);
    }
  return 0;
}
""")


def test_order_of_the_experts_blocks(tmp_path):
    """Column tiles first where that was measured faster.  The down projection of more than 16 experts (33.3 -> 38.4 us) and
    gate_up of few experts in more than one round of workgroups (123 -> 137) went so, too."""
    _run(tmp_path, """
#include <initializer_list>
#include "moe_order.h"
using kgc::moe_columns_first;
#define CHECK(x) if (!(x)) return __LINE__
int main() {
  for (int pairs : {128, 512, 1280})                           // 32 and 64 experts of 2048 x 1408
    for (int E : {17, 32, 64}) CHECK(!moe_columns_first(false, E, 64, E + pairs / 64, 8, pairs));
  for (int pairs : {4, 8, 64, 128}) {                          // 4 experts of 4096 x 14336, of 2048 x 8192
    CHECK(!moe_columns_first(true, 4, 64, 4 + pairs / 64, 112, pairs));
    CHECK(moe_columns_first(true, 4, 64, 4 + pairs / 64, 64, pairs));
    CHECK(moe_columns_first(false, 4, 64, 4 + pairs / 64, 16, pairs));
  }
  CHECK(!moe_columns_first(false, 12, 64, 16, 8, 256) && !moe_columns_first(false, 3, 64, 3, 8, 16));   // 50 -> 54, 20 -> 21 us
  CHECK(!moe_columns_first(true, 3, 64, 3, 112, 16) && moe_columns_first(true, 2, 64, 2, 112, 16));
  CHECK(moe_columns_first(true, 4, 64, 4, 112, 2) && moe_columns_first(false, 64, 64, 64, 8, 12));       // most have no rows
  CHECK(moe_columns_first(false, 8, 64, 9, 16, 16) && !moe_columns_first(false, 8, 64, 8, 16, 12));
  CHECK(moe_columns_first(false, 16, 64, 17, 16, 64) && !moe_columns_first(true, 8, 64, 9, 112, 64));
  CHECK(moe_columns_first(true, 8, 128, 16, 112, 1024) && !moe_columns_first(true, 8, 128, 15, 112, 960));
  CHECK(!moe_columns_first(true, 8, 128, 16, 28, 1024) && !moe_columns_first(false, 8, 128, 16, 16, 1024));
  return 0;
}
""")


@pytest.mark.parametrize("E,N,K,rows,want", [
    (8, 4096, 14336, 1, 8), (8, 4096, 14336, 6, 2),                   # few pairs: near one workgroup per CU, as ever
    (8, 4096, 14336, 8, 4), (8, 4096, 14336, 256, 4), (8, 4096, 14336, 700, 2), (8, 4096, 14336, 2048, 1),
    (16, 4096, 6400, 8, 1), (16, 4096, 6400, 512, 2),
    (8, 4096, 3584, 256, 1), (32, 2048, 1408, 64, 1), (1, 256, 1 << 20, 64, 16),
    (4, 4096, 14336, 300, 4), (4, 4096, 14336, 100, 2), (8, 6144, 16384, 64, 1),      # less than two rounds, and more: as ever
    (8, 4096, 7168, 256, 1), (8, 5120, 14336, 64, 1), (8, 2048, 8192, 1000, 1)])
def test_expert_down_projection_slices(monkeypatch, E, N, K, rows, want):
    """K-slices of the experts' down projection (top 2, column tiles of 256): two full rounds of workgroups
    where every expert has rows and a slice keeps 48 steps."""
    from kubernetes_gpu_cluster_amd import ops
    monkeypatch.delenv("KGC_MOE_SPLITK", raising=False)
    S = ops.moe_dgemm_splitk(2 * rows, E, N, K, ops.moe_k14m_bm(2 * rows, E), 256)
    assert S == want and 1 <= S <= 16 and K // 64 // S >= 8
