// Shared by the chunkwise recurrences (chunk_scan.hip, chunk_delta.hip, chunk_gla.hip): fp32 operands of the bf16
// matrix cores as sums of bf16 parts, wave-wide running sums in double, and the mapping of work
// items to pieces of ragged sequences.
#pragma once
#include "common.h"

namespace kgc {

// x = sum of NP bf16 parts, each the rounding of what the ones before it leave; two at a time, so
// that one instruction rounds and packs a pair (an infinity leaves NaN)
typedef float f32x2 __attribute__((ext_vector_type(2)));
template <int NP>
__device__ __forceinline__ void split2(float x0, float x1, uint32_t (&p)[NP]) {
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    p[j] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x0, x1}), bf16x2_t));
    if (j + 1 < NP) {
      x0 -= __builtin_bit_cast(float, p[j] << 16);
      x1 -= __builtin_bit_cast(float, p[j] & 0xffff0000u);
    }
  }
}
template <int NP>
__device__ __forceinline__ void split8(const float (&x)[8], bf16x8 (&p)[NP]) {
  u32x4 o[NP];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t w[NP];
    split2<NP>(x[2 * i], x[2 * i + 1], w);
#pragma unroll
    for (int j = 0; j < NP; ++j) o[j][i] = w[j];
  }
#pragma unroll
  for (int j = 0; j < NP; ++j) p[j] = __builtin_bit_cast(bf16x8, o[j]);
}

// hi + lo += a b over the products of parts i, j with i + j <= 2.  SEP: the corrections have a sum
// of their own; added to the main sum one by one, each would round it (SSD: 1.2e-7 from float64,
// 0.8e-7 so).  One-part operands have but two corrections, and no registers left.
template <bool SEP, int NA, int NB>
__device__ __forceinline__ void mm(const bf16x8 (&a)[NA], const bf16x8 (&b)[NB], f32x4& hi, f32x4& lo) {
  f32x4& l = SEP ? lo : hi;
#pragma unroll
  for (int s = 2; s >= 1; --s)
#pragma unroll
    for (int i = 0; i <= s; ++i)
      if (i < NA && s - i < NB) l = mfma16x16x32(a[i], b[s - i], l);
  if constexpr (SEP) hi += mfma16x16x32(a[0], b[0], f32x4{0.f, 0.f, 0.f, 0.f});
  else hi = mfma16x16x32(a[0], b[0], hi);
}

// Products of three parts each, N row tiles a times the columns of b: several sums side by side, since an MFMA
// waits for the one whose sum it continues.  The corrections first, the main products on top of them.
template <int N>
__device__ __forceinline__ void mm3(const bf16x8 (&a)[N][3], const bf16x8 (&b)[3], f32x4 (&c)[N]) {
  constexpr int PA[6] = {0, 1, 2, 0, 1, 0}, PB[6] = {2, 1, 0, 1, 0, 0};
#pragma unroll
  for (int k = 0; k < 6; ++k)
#pragma unroll
    for (int i = 0; i < N; ++i) c[i] = mfma16x16x32(a[i][PA[k]], b[PB[k]], k ? c[i] : f32x4{0.f, 0.f, 0.f, 0.f});
}
// hi + lo += a b, the columns in NB parts (one sum for both: the corrections first)
template <int N, int NB>
__device__ __forceinline__ void mm3_add(const bf16x8 (&a)[N][3], const bf16x8 (&b)[NB], f32x4 (&hi)[N], f32x4 (&lo)[N]) {
  constexpr int PA[6] = {0, 1, 2, 0, 1, 0}, PB[6] = {2, 1, 0, 1, 0, 0};
#pragma unroll
  for (int k = 0; k < 6; ++k)
#pragma unroll
    for (int i = 0; i < N; ++i) {
      if (PB[k] >= NB) continue;
      f32x4& c = k == 5 ? hi[i] : lo[i];
      c = mfma16x16x32(a[i][PA[k]], b[PB[k] < NB ? PB[k] : 0], c);
    }
}

// the same for two row tiles times two column tiles
__device__ __forceinline__ void mm3(const bf16x8 (&a)[2][3], const bf16x8 (&b)[2][3], f32x4 (&c)[2][2]) {
  constexpr int PA[6] = {0, 1, 2, 0, 1, 0}, PB[6] = {2, 1, 0, 1, 0, 0};
#pragma unroll
  for (int k = 0; k < 6; ++k)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        c[i][j] = mfma16x16x32(a[i][PA[k]], b[j][PB[k]], k ? c[i][j] : f32x4{0.f, 0.f, 0.f, 0.f});
}
// hi + lo += a b
__device__ __forceinline__ void mm3_add(const bf16x8 (&a)[2][3], const bf16x8 (&b)[2][3], f32x4 (&hi)[2][2], f32x4 (&lo)[2][2]) {
  constexpr int PA[6] = {0, 1, 2, 0, 1, 0}, PB[6] = {2, 1, 0, 1, 0, 0};
#pragma unroll
  for (int k = 0; k < 6; ++k)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        f32x4& c = k == 5 ? hi[i][j] : lo[i][j];
        c = mfma16x16x32(a[i][PA[k]], b[j][PB[k]], c);
      }
}

// a barrier that leaves the newest N memory operations on their way (a fence would wait for all)
template <int N> __device__ __forceinline__ void meet() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt((N & 15) | (N >> 4) << 14 | 0x70);   // vmcnt(N) lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Order of the instructions up to here from the last sched_barrier: N times one MFMA and V vector instructions, which
// run beside it, an LDS read after every R-th and a memory instruction after every M-th (0: where they fall; in a
// burst they would hold up the wave).  An MFMA of 16 x 16 x 32 takes 8 cycles of issue and 16 of the matrix core, a vector
// instruction 4; two waves of a SIMD overlap them by chance only, half of the time.
template <int N, int V, int R = 0, int M = 0> __device__ __forceinline__ void interleave() {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, V, 0);
    if (R > 0 && i % R == R - 1) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    if (M > 0 && i % M == M - 1) __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
  }
}

// e^x for x <= 0 held in double: the reduction to 2^n 2^f is exact to fp32 however large x is, so
// the error is that of the hardware's 2^f, |f| <= 1/2
__device__ __forceinline__ float exp_d(double x) {
  const double y = (x < -1e4 ? -1e4 : x) * 1.4426950408889634074, n = __builtin_rint(y);
  return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f((float)(y - n)), (int)n);
}

// inclusive running sum (MAX: maximum) over the 64 lanes, by row shifts and row broadcasts
template <int CTRL, int ROWS, bool MAX> __device__ __forceinline__ double scan_step(double x) {
  const double none = MAX ? -INFINITY : 0.0;
  const uint64_t o = __builtin_bit_cast(uint64_t, none), b = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = __builtin_amdgcn_update_dpp((uint32_t)o, (uint32_t)b, CTRL, ROWS, 0xf, false);
  const uint32_t hi = __builtin_amdgcn_update_dpp((uint32_t)(o >> 32), (uint32_t)(b >> 32), CTRL, ROWS,
                                                  0xf, false);
  const double y = __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
  return MAX ? fmax(x, y) : x + y;
}
template <bool MAX> __device__ __forceinline__ double wave_scan(double x) {
  x = scan_step<0x111, 0xf, MAX>(x);         // row_shr 1, 2, 4, 8
  x = scan_step<0x112, 0xf, MAX>(x);
  x = scan_step<0x114, 0xf, MAX>(x);
  x = scan_step<0x118, 0xf, MAX>(x);
  x = scan_step<0x142, 0xa, MAX>(x);         // row_bcast 15 into rows 1 and 3
  return scan_step<0x143, 0xc, MAX>(x);      // row_bcast 31 into rows 2 and 3
}
__device__ __forceinline__ double lane63(double x) {
  const uint64_t b = __builtin_bit_cast(uint64_t, x);
  const uint64_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, 63);
  const uint64_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), 63);
  return __builtin_bit_cast(double, hi << 32 | lo);
}

// what is not finite if a value is not, or the values' sum
template <int N, typename V> __device__ __forceinline__ float nonfinite_sum(const V (&v)[N]) {
  float z = 0.f;
  if constexpr (sizeof(V) == 2) {            // products with zeros, two at a time
    typedef V V2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < N; i += 2) {
      if constexpr (__is_same(V, f16)) z = __builtin_amdgcn_fdot2(V2{v[i], v[i + 1]}, V2{0, 0}, z, false);
      else z = __builtin_amdgcn_fdot2_f32_bf16(V2{v[i], v[i + 1]}, V2{0, 0}, z, false);
    }
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) z += (float)v[i];
  }
  return z;
}
// The products over a chunk multiply a token's value by the masked zeros of the rows before it, which a
// value that is not finite would reach.  v[i]: token tok(i) of the lane's column (one of the four lanes
// that share lane & 15; PAIR: of the two that share lane & 31).  Such values become zero; returned is the column's first such token, from
// which on its outputs and its state have to be made NaN (`none`: every value is finite).  A sum that
// overflows only costs the closer look.
template <bool PAIR = false, int N, typename V, typename F>
__device__ __forceinline__ int take_nonfinite(V (&v)[N], int none, F tok) {
  const float z = nonfinite_sum(v);
  int first = none;
  if (__any(!(fabsf(z) < INFINITY))) {
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (!(fabsf((float)v[i]) < INFINITY)) {
        first = min(first, tok(i));
        v[i] = (V)0.f;
      }
    if (PAIR) {
      const auto p = __builtin_amdgcn_permlane32_swap(first, first, false, false);
      first = min((int)p[0], (int)p[1]);
    } else {
      first = min(first, __shfl_xor(first, 16, 64));
      first = min(first, __shfl_xor(first, 32, 64));
    }
  }
  return first;
}

// Sequence and segment of work item `item` (every lane of every wave gets the same answer)
struct SegItem { int seq, idx, count, first; };
__device__ __forceinline__ SegItem seg_item(int item, const int* qsl, int P, int seg) {
  SegItem r{-1, 0, 0, 0};
  const int lane = threadIdx.x & 63;
  int base = 0;
  for (int p0 = 0; p0 < P; p0 += 64) {
    const int p = p0 + lane;
    const int n = p < P ? max(1, (qsl[p + 1] - qsl[p] + seg - 1) / seg) : 0;
    int inc = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(inc, o, 64);
      if (lane >= o) inc += y;
    }
    const int total = __shfl(inc, 63, 64);
    if (item < base + total) {
      const unsigned long long hit = __ballot(base + inc > item);
      const int l = __ffsll((unsigned long long)hit) - 1;
      r.seq = p0 + l;
      r.count = __shfl(n, l, 64);
      r.first = base + __shfl(inc, l, 64) - r.count;
      r.idx = item - r.first;
      return r;
    }
    base += total;
  }
  return r;
}

// pieces of `rows` tokens (a sequence has one at least) of the sequences before `seq`: segments, or chunks
__device__ __forceinline__ int pieces_before(int seq, const int* qsl, int rows) {
  const int lane = threadIdx.x & 63;
  int n = 0;
  for (int p = lane; p < seq; p += 64) n += max(1, (qsl[p + 1] - qsl[p] + rows - 1) / rows);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
  return n;
}
template <int L> __device__ __forceinline__ int chunks_before(int seq, const int* qsl) { return pieces_before(seq, qsl, L); }

// column c of a k index that MFMAs read permuted, so that accumulators are operands as they lie:
// the 4-column pieces of every 32 go in the order 0 4 1 5 2 6 3 7
__device__ __forceinline__ int mfma_perm(int c) {
  const int p = (c >> 2) & 7;
  return (c & ~31) | ((((p & 3) << 1) | (p >> 2)) << 2) | (c & 3);
}

}  // namespace kgc
