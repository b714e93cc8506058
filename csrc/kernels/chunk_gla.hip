// Chunkwise gated linear attention (Yang et al., 2023) of prompt rows on the matrix cores.  Per
// (sequence, head), with a decay alpha_t per key channel,
//     S_t = diag(alpha_t) S_(t-1) + k_t v_t^T,   o_t = S_t^T q_t .
// Over a chunk of L = 32 tokens, p_t the product of the chunk's decays up to t, r_s of those after s and
// S_0 the state before it (products channel by channel):
//     O   = (Q p) S_0 + A V,     A_ts = sum_c q_tc k_sc alpha_(s+1)c .. alpha_tc  (s <= t)
//     S_L = diag(p_L) S_0 + (K r)^T V
// Q p, K r, p_L and A depend on no state: a first launch computes them for all chunks at once, A from products
// of decays alone (no quotient of products, so no decay is too small).  The walk
// then has no serial step finer than a chunk: a workgroup of 8 waves owns 128 value columns of a head,
// a wave 16 of them with their S in accumulators.
//
// Precision: fp32 operands enter the bf16 MFMAs as three bf16 parts each, six products of parts (16-bit values
// in as many parts as they have: three products in bf16, five in f16), the corrections of the outputs summed apart;
// products p and r are kept in double.
//
// Few long sequences are cut into segments: one walk makes every segment's contribution from a zero state, a
// small launch puts the states together in which the segments start, and the second walk has them all.
//
// Measured (8 heads, 256 value columns, rank 16): 32 x 512 tokens 181 us, 65 of them the first launch and 125 (in a
// trace) the walk.  The first launch was 110 to 119 with A by vector instructions from running products and the decays by
// expf and log1pf: it is bound by issue (1650 instructions a wave, of them 480 for the decays, 200 for products in
// double) and by 148 MB written.  The walk was 158 with values in three parts, a barrier on either side of the operands'
// writing that waited for memory, p_L from memory: it is bound by issue, per wave and chunk 420 vector
// instructions (40 % of them split S), 78 MFMAs, 80 others; from the same addresses and without writing outputs it
// takes 15 us less.  2 x 8192 283 (411; one walk per sequence: 1562), 1 x 4000 96 (127; 659), 4 x 60 20 (31); token by
// token 1340 and 8140.  From float64, relative norm, 4 x 700 tokens: outputs 2.1e-7, states 2.3e-7 (9.1e-7 and
// 1.3e-6 with expf, whose argument's rounding is the same for all of a sequence's decays).
#include <type_traits>
#include "chunk.h"
#include "chunk_rows.h"
#include "device.h"
#include "launch.h"

namespace kgc {

namespace {

constexpr int L = 32, D = 128;               // tokens per chunk, key channels
constexpr int NT = 512;
constexpr int DT = D / 16, LT = L / 16, KD = D / 32;
constexpr int DP = D + 8, LP = L + 8;        // padded LDS rows
constexpr int MAT = 3 * L * L;               // bf16 of one matrix of a chunk: three parts
constexpr int RMAX = 128;                    // rank of the decay projection

struct GlaArgs {
  float* out;                                // [T, H dv]
  const void *proj, *low;                    // q | k | v rows; decay bottleneck rows
  int64_t ps, ls;
  const float *a2, *a2b;                     // [H D, R], [H D]
  float* S;
  const int *qsl, *seq_lens, *slots;
  int P, H, dv, R, num_slots;
  float inv_tau;
  // workspace, per chunk and head; rows past a sequence's end are zero
  float *qp, *kr;                            // [L][D]
  float* pl;                                 // [D]
  bf16* am;                                  // [3][L][L], columns permuted
  int seg, items;                            // tokens per segment, a multiple of the chunk (0: not cut)
  float* seg_state;                          // [items][H][D][dv]: contribution, then state a segment starts from
};

// sum over the sixteen lanes of a row, without the LDS
__device__ __forceinline__ float sum16(float x) {
  auto other = [](float y, auto ctrl) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, y), decltype(ctrl)::value, 0xf, 0xf, true));
  };
  x += other(x, std::integral_constant<int, 0x128>());    // rotated by 8, 4, 2, 1
  x += other(x, std::integral_constant<int, 0x124>());
  x += other(x, std::integral_constant<int, 0x122>());
  return x + other(x, std::integral_constant<int, 0x121>());
}

// sigmoid(x)^(1 / tau) = e^g, g = (min(x, 0) - log(1 + y)) / tau, y = e^-|x|.  The logarithm is 2 atanh(s), s =
// y / (2 + y) <= 1/3, by its series to s^17 (what is left is 2^-29 of it), s with the division's remainder.
// e^g = 2^n e^f, |f| <= log(2) / 2, by its series to f^7 (left: 2^-27): rounded once where n is 0, as a sequence's
// errors add up with its decays'.
__device__ __forceinline__ float decay(float x, float inv_tau) {
  const float y = __builtin_amdgcn_exp2f(-1.44269504f * fabsf(x)), rc = __builtin_amdgcn_rcpf(2.f + y);
  float s = y * rc;
  s = __builtin_fmaf(__builtin_fmaf(-s, y, __builtin_fmaf(-2.f, s, y)), rc, s);
  const float z = s * s;
  float t = 2.f / 17.f;
  t = __builtin_fmaf(t, z, 2.f / 15.f);
  t = __builtin_fmaf(t, z, 2.f / 13.f);
  t = __builtin_fmaf(t, z, 2.f / 11.f);
  t = __builtin_fmaf(t, z, 2.f / 9.f);
  t = __builtin_fmaf(t, z, 2.f / 7.f);
  t = __builtin_fmaf(t, z, 2.f / 5.f);
  t = __builtin_fmaf(t, z, 2.f / 3.f);
  t = __builtin_fmaf(t * z, s, 2.f * s);
  float g = (fminf(x, 0.f) - t) * inv_tau;
  g = g < -150.f ? -150.f : g;               // (0 in 32 bits; NaN stays)
  const float n = __builtin_rintf(1.44269504f * g);
  const float f = __builtin_fmaf(n, 1.90465432e-9f, __builtin_fmaf(n, -0.693147182f, g));
  float e = 1.f / 5040.f;
  e = __builtin_fmaf(e, f, 1.f / 720.f);
  e = __builtin_fmaf(e, f, 1.f / 120.f);
  e = __builtin_fmaf(e, f, 1.f / 24.f);
  e = __builtin_fmaf(e, f, 1.f / 6.f);
  e = __builtin_fmaf(e, f, 0.5f);
  e = __builtin_fmaf(e * f, f, f);
  return __builtin_amdgcn_ldexpf(1.f + e, (int)n);
}

// q p, k r, p_L and A of every chunk: one workgroup per (chunk, head), a wave has 32 channels and each of its lanes
// two of them for eight tokens, 8 lg on; no wave waits for another before the end.  The
// decays come out of the matrix cores in that form.  A by halves: for a block of 2 n tokens, those t of its second half with
// those s of its first are (q_t decays from the middle to t) . (k_s decays after s to the middle), so a tile of 16 x 16
// has all blocks of one size, in fp32 MFMAs, with what lies between two blocks left out (n = 16, 8, 4, 2); the
// rest, s = t and t - 1 in pairs, is summed over lanes.  VEC: rows of pairs, and fours of the decays' rank.
template <typename T, bool VEC>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? 3 : 4) void gla_prep_kernel(const GlaArgs a) {
  __shared__ __align__(16) float Z[4][L][36];          // a wave's rows of q and of k, then its part of A
  const SegItem it = seg_item(blockIdx.x, a.qsl, a.P, L);
  if (it.seq < 0) return;
  const int h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c0 = it.idx * L, len = a.qsl[it.seq + 1] - a.qsl[it.seq], nl = min(L, len - c0);
  const int slot = a.slots[it.seq];
  if (nl <= 0 || slot < 0 || slot >= a.num_slots || a.seq_lens[it.seq] < len) return;
  const int64_t t0 = a.qsl[it.seq] + c0, at = (int64_t)blockIdx.x * a.H + h;
  const int ch = wave * 32 + 2 * lr;
  const T* proj = reinterpret_cast<const T*>(a.proj) + t0 * a.ps + h * D;
  const T* low = reinterpret_cast<const T*>(a.low) + t0 * a.ls;
  typedef T T2 __attribute__((ext_vector_type(2)));
  typedef T T4 __attribute__((ext_vector_type(4)));
  // the decays' arguments: token rows 8 (m >> 2) + (m & 3) (+ 4), columns this lane's channels
  f32x4 x[2][2];
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i >> 1][i & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int tm = 8 * (lr >> 2) + (lr & 3);
  T2 qv[8], kv[8];
  const T* qr = proj + min(8 * lg, nl - 1) * a.ps + ch;
#pragma unroll
  for (int i = 0; i < 8; ++i) {              // (rows past the end: the last one again)
    if (i > 0) qr += 8 * lg + i < nl ? a.ps : 0;
    const T* kr = qr + (int64_t)a.H * D;
    if constexpr (VEC) {
      qv[i] = *reinterpret_cast<const T2*>(qr);
      kv[i] = *reinterpret_cast<const T2*>(kr);
    } else {
      qv[i] = T2{qr[0], qr[1]};
      kv[i] = T2{kr[0], kr[1]};
    }
  }
  for (int j0 = 0; j0 < a.R; j0 += 16) {
    f32x4 lv[2], wv[2];
    const int j = j0 + 4 * lg;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const T* lp = low + min(tm + 4 * n, nl - 1) * a.ls;
      const float* wp = a.a2 + (int64_t)h * D * a.R + (ch + n) * a.R;
      if constexpr (VEC) {
        const int jj = min(j, a.R - 4);
        const T4 u = *reinterpret_cast<const T4*>(lp + jj);
        wv[n] = *reinterpret_cast<const f32x4*>(wp + jj);
#pragma unroll
        for (int i = 0; i < 4; ++i) lv[n][i] = to_f(u[i]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          lv[n][i] = to_f(lp[min(j + i, a.R - 1)]);
          wv[n][i] = wp[min(j + i, a.R - 1)];
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        lv[n][i] = j + i < a.R ? lv[n][i] : 0.f;
        wv[n][i] = j + i < a.R ? wv[n][i] : 0.f;
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int m = 0; m < 2; ++m) x[n][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(lv[n][i], wv[m][i], x[n][m], 0, 0, 0);
  }
  const float scale = 1.f / sqrtf((float)D);
  float q[8][2], k[8][2], al[8][2], u[8][2], w[8][2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const float bias = a.a2b[h * D + ch + m];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float f = decay(x[i >> 2][m][i & 3] + bias, a.inv_tau);
      al[i][m] = 8 * lg + i < nl ? f : 1.f;
      q[i][m] = 8 * lg + i < nl ? to_f(qv[i][m]) * scale : 0.f;
      k[i][m] = 8 * lg + i < nl ? to_f(kv[i][m]) : 0.f;
    }
  }
  // products of the decays before and after these tokens, in double; mid: of the eight between them and the chunk's middle
  double p[2], r[2];
  float mid[2], whole[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    double f = al[0][m];
#pragma unroll
    for (int i = 1; i < 8; ++i) f *= al[i][m];
    const double next = __shfl_xor(f, 16, 64), pair = f * next, far = __shfl_xor(pair, 32, 64);
    const double both = next * far;
    p[m] = lg == 0 ? 1.0 : lg == 1 ? next : lg == 2 ? far : both;
    r[m] = lg == 3 ? 1.0 : lg == 2 ? next : lg == 1 ? far : both;
    mid[m] = lg == 0 || lg == 3 ? (float)next : 1.f;
    whole[m] = (float)(pair * far);
  }
  float *qo = a.qp + at * L * D, *ko = a.kr + at * L * D;
  const int to = 8 * lg * D + ch;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    f32x2 o;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      p[m] *= al[i][m];
      o[m] = (float)(q[i][m] * p[m]);
    }
    *reinterpret_cast<f32x2*>(qo + to + i * D) = o;
  }
#pragma unroll
  for (int i = 7; i >= 0; --i) {
    f32x2 o;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      o[m] = (float)(k[i][m] * r[m]);
      r[m] *= al[i][m];
    }
    *reinterpret_cast<f32x2*>(ko + to + i * D) = o;
  }
  if (lg == 0) *reinterpret_cast<f32x2*>(a.pl + at * D + ch) = f32x2{whole[0], whole[1]};
  // q times the decays from 8 lg on, k times those up to 8 lg + 8
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    float f = 1.f, b = 1.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      f *= al[i][m];
      u[i][m] = q[i][m] * f;
      w[7 - i][m] = k[7 - i][m] * b;
      b *= al[7 - i][m];
    }
  }
  float (*z)[36] = Z[wave];
  auto settle = [] {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  auto put = [&](int row, float v0, float v1) { *reinterpret_cast<f32x2*>(&z[row][2 * lr]) = f32x2{v0, v1}; };
  auto tile = [&]() {                        // rows of q in z[0 ..], rows of k in z[16 ..]
    settle();
    f32x4 d = {0.f, 0.f, 0.f, 0.f};
    f32x4 qz[2], kz[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      qz[i] = *reinterpret_cast<const f32x4*>(&z[lr][8 * lg + 4 * i]);
      kz[i] = *reinterpret_cast<const f32x4*>(&z[16 + lr][8 * lg + 4 * i]);
    }
    settle();
#pragma unroll
    for (int i = 0; i < 8; ++i) d = __builtin_amdgcn_mfma_f32_16x16x4f32(qz[i >> 2][i & 3], kz[i >> 2][i & 3], d, 0, 0, 0);
    return d;
  };
  f32x4 d[4];
  {
    const bool second = lg >= 2;
    const int row = (second ? 0 : 16) + 8 * (lg & 1);
#pragma unroll
    for (int i = 0; i < 8; ++i) put(row + i, (second ? u[i][0] : w[i][0]) * mid[0], (second ? u[i][1] : w[i][1]) * mid[1]);
    d[0] = tile();
  }
  {
    const bool second = lg & 1;
    const int row = (second ? 0 : 16) + 8 * (lg >> 1);
#pragma unroll
    for (int i = 0; i < 8; ++i) put(row + i, second ? u[i][0] : w[i][0], second ? u[i][1] : w[i][1]);
    d[1] = tile();
  }
  {
    float f[2] = {1.f, 1.f}, b[2] = {1.f, 1.f};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int m = 0; m < 2; ++m) f[m] *= al[4 + i][m];
      put(4 * lg + i, q[4 + i][0] * f[0], q[4 + i][1] * f[1]);
      put(16 + 4 * lg + 3 - i, k[3 - i][0] * b[0], k[3 - i][1] * b[1]);
#pragma unroll
      for (int m = 0; m < 2; ++m) b[m] *= al[3 - i][m];
    }
    d[2] = tile();
  }
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int i = 4 * e, row = 4 * lg + 2 * e;
    put(row, q[i + 2][0] * al[i + 2][0], q[i + 2][1] * al[i + 2][1]);
    put(row + 1, q[i + 3][0] * (al[i + 2][0] * al[i + 3][0]), q[i + 3][1] * (al[i + 2][1] * al[i + 3][1]));
    put(16 + row, k[i][0] * al[i + 1][0], k[i][1] * al[i + 1][1]);
    put(16 + row + 1, k[i + 1][0], k[i + 1][1]);
  }
  d[3] = tile();
  float same[8], last[4];
#pragma unroll
  for (int i = 0; i < 8; ++i) same[i] = sum16(q[i][0] * k[i][0] + q[i][1] * k[i][1]);
#pragma unroll
  for (int e = 0; e < 4; ++e)
    last[e] = sum16(q[2 * e + 1][0] * (k[2 * e][0] * al[2 * e + 1][0]) + q[2 * e + 1][1] * (k[2 * e][1] * al[2 * e + 1][1]));
#pragma unroll
  for (int i = 0; i < 4; ++i) {              // tile row 4 lg + i, column lr
    const int row = 4 * lg + i;
    z[16 + row][lr] = d[0][i];
    if (row >> 3 == lr >> 3) z[row + (row & 8) + 8][lr + (lr & 8)] = d[1][i];
    if (row >> 2 == lr >> 2) z[2 * row - (row & 3) + 4][2 * lr - (lr & 3)] = d[2][i];
    if (row >> 1 == lr >> 1) z[2 * row - (row & 1) + 2][2 * lr - (lr & 1)] = d[3][i];
  }
  if (lr == 0) {
#pragma unroll
    for (int i = 0; i < 8; ++i) z[8 * lg + i][8 * lg + i] = same[i];
#pragma unroll
    for (int e = 0; e < 4; ++e) z[8 * lg + 2 * e + 1][8 * lg + 2 * e] = last[e];
  }
  __syncthreads();
  {                                          // four (permuted) columns per store
    const int t = tid >> 3, oct = (tid & 7) >> 1, s = (tid & 1) * 16 + oct * 4;
    f32x4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const f32x4*>(&Z[i][t][s]);
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = s + e <= t ? (v[0][e] + v[1][e]) + (v[2][e] + v[3][e]) : 0.f;
    uint32_t y0[3], y1[3];
    split2<3>(y[0], y[1], y0);
    split2<3>(y[2], y[3], y1);
#pragma unroll
    for (int i = 0; i < 3; ++i)
      *reinterpret_cast<u32x2*>(a.am + at * MAT + i * L * L + t * L + (tid & 7) * 4) = u32x2{y0[i], y1[i]};
  }
}

// MODE 0: whole sequences; 1: segments from zero (states only); 2: segments from the states that they start in
template <typename T, int MODE>
__global__ __launch_bounds__(NT) void gla_walk_kernel(const GlaArgs a) {
  // twice: (k r)^T, q p (parts), A, p_L
  constexpr int QS = 3 * D * LP * 2, AS = QS + (MODE == 1 ? 0 : 3 * L * DP * 2), PS = AS + (MODE == 1 ? 0 : NT * 16), HALF = PS + NT * 4;
  __shared__ __align__(16) char sm[2 * HALF];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int nct = (a.dv + 127) / 128;
  int seq = blockIdx.x, seg_idx = 0, seg_count = 1, item = 0;
  if (MODE != 0) {
    const SegItem it = seg_item(blockIdx.x, a.qsl, a.P, a.seg);
    if (it.seq < 0) return;
    seq = __builtin_amdgcn_readfirstlane(it.seq);
    seg_idx = __builtin_amdgcn_readfirstlane(it.idx);
    seg_count = __builtin_amdgcn_readfirstlane(it.count);
    item = __builtin_amdgcn_readfirstlane(it.first) + seg_idx;
    if (MODE == 1 && seg_idx + 1 == seg_count) return;
  }
  const int h = blockIdx.y / nct, ct = blockIdx.y - h * nct;
  const int col = ct * 128 + wave * 16 + lr;
  const bool colok = col < a.dv;
  const int colc = colok ? col : a.dv - 1;                // columns off the edge: read the last
  int start = a.qsl[seq], len = a.qsl[seq + 1] - start;
  const int pos0 = a.seq_lens[seq] - len, slot = a.slots[seq];
  const int64_t os = (int64_t)a.H * a.dv;
  if (MODE != 0) {
    start += seg_idx * a.seg;
    len = min(a.seg, len - seg_idx * a.seg);
  }
  if (len <= 0) return;
  if (slot < 0 || slot >= a.num_slots || pos0 < 0) {      // padding: defined zeros
    if (MODE != 1 && colok)
      for (int t = lg; t < len; t += 4) a.out[(start + t) * os + (int64_t)h * a.dv + col] = 0.f;
    return;
  }
  // parts of a value, products of two row tiles with them
  constexpr int NV = sizeof(T) == 4 ? 3 : __is_same(T, bf16) ? 1 : 2, NM = NV == 1 ? 6 : NV == 2 ? 10 : 12;
  f32x4 S[DT];
  float* Ss = a.S + ((int64_t)slot * a.H + h) * D * a.dv;
  float* mine = a.seg_state + ((int64_t)item * a.H + h) * D * a.dv;
  const bool own = MODE == 2 && seg_count > 1, zero = MODE == 1 || (pos0 == 0 && !own);
  const float* from = own ? mine : Ss;
#pragma unroll
  for (int i = 0; i < DT; ++i) S[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  // (one branch: as a choice per element they became 32, each of which waited for the load before it; 8 x 256, rows that go
  // on from a state: 128 x 16 131 -> 88 us, 256 x 24 389 -> 200)
  if (__builtin_amdgcn_readfirstlane(!zero)) {
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[i][r] = from[(i * 16 + 4 * lg + r) * a.dv + colc];
    __builtin_amdgcn_sched_barrier(0);
  }
  const T* vb = reinterpret_cast<const T*>(a.proj) + 2 * (int64_t)a.H * D + (int64_t)h * a.dv + colc;
  // Staging: a thread takes 8 columns of one row of q p, and 8 tokens of one column of k r, in both
  // cases the pieces 4 i .. and 16 + 4 i .. of 32: adjacent in the permuted order, one store.  A and p_L as they are
  // (threads past the end of A: its last piece again; four copies of p_L).
  f32x4 rq[2], rt[2];
  u32x4 ra;
  float rp;
  const int ut = tid / 16, uc = (tid % 16 / 4) * 32 + (tid % 4) * 4;
  const int ta = tid / D * 4, tc = tid % D;
  const int qat = ut * D + uc, kat = ta * D + tc, aat = min(tid, MAT / 8 - 1) * 8;
  const int chunk0 = __builtin_amdgcn_readfirstlane(chunks_before<L>(seq, a.qsl)) + (MODE != 0 ? seg_idx * (a.seg / L) : 0);
  auto fetch_q = [&](int ci) {
    const int64_t at = (int64_t)ci * a.H + h;
    const float* qp = a.qp + at * L * D;
    if (MODE != 1) {
#pragma unroll
      for (int i = 0; i < 2; ++i) rq[i] = *reinterpret_cast<const f32x4*>(qp + qat + 16 * i);
      ra = *reinterpret_cast<const u32x4*>(a.am + at * MAT + aat);
    }
    rp = (a.pl + at * D)[tc];
  };
  auto fetch_k = [&](int ci) {
    const float *k0 = a.kr + ((int64_t)ci * a.H + h) * L * D, *k1 = k0 + 16 * D;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      rt[0][i] = k0[kat + i * D];
      rt[1][i] = k1[kat + i * D];
    }
  };
  bf16x8 pq[3], pk[3];
  auto split_f = [&](const f32x4 (&x)[2], bf16x8 (&p)[3]) {
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = x[i >> 2][i & 3];
    split8<3>(y, p);
  };
  auto park_q = [&](char* m) {
    if (MODE != 1) {
#pragma unroll
      for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8*>(m + QS + (i * L * DP + ut * DP + (tid % 16) * 8) * 2) = pq[i];
    }
  };
  auto park_k = [&](char* m) {
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8*>(m + ((i * D + tc) * LP + ta * 2) * 2) = pk[i];
    if (MODE != 1) *reinterpret_cast<u32x4*>(m + AS + tid * 16) = ra;
    reinterpret_cast<float*>(m + PS)[tid] = rp;
  };
  bf16x8 sp[2][3];                           // parts of 32 rows of S; the first ones of the next chunk
  auto split_s = [&](int j) {
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = S[2 * j + (i >> 2)][i & 3];
    split8<3>(x, sp[j & 1]);
  };
  fetch_q(chunk0);
  fetch_k(chunk0);
  if (MODE != 1) {
    split_s(0);
    split_f(rq, pq);
  }
  split_f(rt, pk);
  park_q(sm);
  park_k(sm);
  const T* vrow = vb + (int64_t)(start + 4 * lg) * a.ps;
  char* ob = reinterpret_cast<char*>(a.out + start * os);
  const uint32_t oat = colok ? (4 * lg * (int)os + h * a.dv + col) * 4 : 1u << 30;
  bf16x8 fa[2][2][3];                        // two row tiles of an operand, a step ahead
  auto load_q = [&](const char* m, int j) {
#pragma unroll
    for (int ti = 0; ti < LT; ++ti)
#pragma unroll
      for (int i = 0; i < 3; ++i)
        fa[j & 1][ti][i] = *reinterpret_cast<const bf16x8*>(m + QS + (i * L * DP + (ti * 16 + lr) * DP + j * 32 + lg * 8) * 2);
  };
  // MODE 1: a chunk is over before memory answers, so its loads are those of the one after the next
  T v[LT][4];                                // this lane's v, tokens 4 lg + r of each tile
  auto ask_v = [&](int c0) {                 // (rows past the end: the last one again)
    const int nl = min(L, len - c0);
#pragma unroll
    for (int ti = 0; ti < LT; ++ti) {
      const T* row = vb + (int64_t)(start + c0 + min(ti * 16 + lg * 4, nl - 1)) * a.ps;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (r > 0) row += ti * 16 + lg * 4 + r < nl ? a.ps : 0;
        v[ti][r] = *row;
      }
    }
  };
  const int chunk1 = chunk0 + (len - 1) / L; // the last one
  if (MODE == 1) {
    ask_v(0);
    fetch_q(min(chunk0 + 1, chunk1));
    fetch_k(min(chunk0 + 1, chunk1));
  }
  meet<63>();
  if (MODE != 1) load_q(sm, 0);
  // A chunk: the next one is asked for beside the products with S and put into the other half of the LDS beside the
  // state's update.  One barrier a chunk, which waits for no memory, before the update's last step: by then every wave has
  // read what this half holds, and the next chunk's first operands come beside that step.  (The last chunk
  // is a copy without these.)
  auto chunk = [&](auto last, int c0, int ci, int half) {
    constexpr bool LAST = decltype(last)::value;
    const int nl = LAST ? len - c0 : L;
    const char* m = sm + half * HALF;
    char* mn = sm + (HALF - half * HALF);
    if (MODE != 1)
#pragma unroll
    for (int ti = 0; ti < LT; ++ti)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (LAST) v[ti][r] = vb[(int64_t)(start + c0 + min(ti * 16 + lg * 4 + r, nl - 1)) * a.ps];
        else v[ti][r] = vrow[(int64_t)(ti * 16 + r) * a.ps];
      }
    vrow += (int64_t)L * a.ps;
    f32x4 o[LT], ol[LT];
    bf16x8 fp[LT][3], vp[NV];
    T x[8];
    float z;
    auto tok = [&](int i) { return (i >> 2) * 16 + lg * 4 + (i & 3); };
    auto parts = [&]() {
      if constexpr (NV == 1) {
        vp[0] = bf16x8{x[0], x[1], x[2], x[3], x[4], x[5], x[6], x[7]};
      } else {
        float y[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = to_f(x[i]);
        split8<NV>(y, vp);
      }
    };
    auto split_v = [&]() {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = !LAST || tok(i) < nl ? v[i >> 2][i & 3] : (T)0.f;
      z = nonfinite_sum(x);
      parts();
    };
    __builtin_amdgcn_sched_barrier(0);
    if (MODE != 1) {
#pragma unroll
      for (int ti = 0; ti < LT; ++ti) o[ti] = ol[ti] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < KD; ++j) {
        if (j + 1 < KD) {
          load_q(m, j + 1);
          split_s(j + 1);
        } else {
#pragma unroll
          for (int ti = 0; ti < LT; ++ti)
#pragma unroll
            for (int i = 0; i < 3; ++i)
              fp[ti][i] = *reinterpret_cast<const bf16x8*>(m + AS + (i * L * L + (ti * 16 + lr) * L + lg * 8) * 2);
          split_v();
        }
        if (!LAST && j == 0) fetch_q(ci + 1);
        if (!LAST && j == 1) fetch_k(ci + 1);
        mm3_add(fa[j & 1], sp[j & 1], o, ol);
        if (!LAST && j < 2) interleave<12, 4, 2, 1>();
        else if (j + 1 < KD) interleave<12, 4, 2>();
        else interleave<12, NV == 1 ? 2 : 6, 2>();
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      split_v();
    }
    float badf = 0.f;                        // what a column's state adds up from
    if (__builtin_amdgcn_readfirstlane(__any(!(fabsf(z) < INFINITY)))) {
#pragma unroll
      for (int i = 0; i < NV; ++i) asm volatile("" : "+v"(vp[i]));   // a branch, not selects in every chunk
      const int bad = take_nonfinite(x, L, tok);
      parts();
      badf = bad < L ? NAN : 0.f;
      if (MODE != 1)
#pragma unroll
        for (int ti = 0; ti < LT; ++ti)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (ti * 16 + lg * 4 + e >= bad) ol[ti][e] = NAN;
    }
    f32x4 u[2][2], pl[2][2];                 // products of two row tiles, their decays
    auto load_k = [&](int q) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int i = 0; i < 3; ++i)
          fa[q & 1][t][i] = *reinterpret_cast<const bf16x8*>(m + ((i * D + (2 * q + t) * 16 + lr) * LP + lg * 8) * 2);
        pl[q & 1][t] = *reinterpret_cast<const f32x4*>(m + PS + ((2 * q + t) * 16 + 4 * lg) * 4);
      }
    };
    auto add = [&](int q) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[2 * q + t][e] = __builtin_fmaf(S[2 * q + t][e], pl[q & 1][t][e], u[q & 1][t][e]);
    };
    load_k(0);
    if (MODE != 1) {
      mm3_add(fp, vp, o, ol);
      if (!LAST) split_f(rq, pq);
      interleave<NM, 48 / NM, 1>();
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < DT / 2; ++q) {
      if (!LAST && q == 3) {
        meet<63>();
        if (MODE != 1) load_q(mn, 0);
      }
#pragma unroll
      for (int t = 0; t < 2; ++t) u[q & 1][t] = f32x4{badf, badf, badf, badf};
      mm3_add(fa[q & 1], vp, u[q & 1], u[q & 1]);
      if (q > 0) add(q - 1);
      if (q + 1 < DT / 2) load_k(q + 1);
      if (q == 0 && MODE != 1) {
        // through a descriptor that ends with the chunk's last row: writes past it do nothing
        const auto od = __builtin_amdgcn_make_buffer_rsrc(ob + (int64_t)c0 * os * 4, 0, nl * (int)os * 4, 0x00027000);
#pragma unroll
        for (int ti = 0; ti < LT; ++ti)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float y = o[ti][e] + ol[ti][e];
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, y), od, oat + (ti * 16 + e) * (int)os * 4, 0, 0);
          }
      }
      if (!LAST) {
        if (q == 0) split_f(rt, pk);
        if (q == 1) {
          park_q(mn);
          park_k(mn);
        }
        if (q == 2 && MODE == 1) {
          ask_v(c0 + L);
          fetch_q(min(ci + 2, chunk1));
          fetch_k(min(ci + 2, chunk1));
        }
        if (q == 3 && MODE != 1) split_s(0);
      }
      if (q == 0 && MODE != 1) interleave<NM, 72 / NM, 1, 1>();
      else if (q == 3) interleave<NM, 60 / NM, 1>();
      else interleave<NM, 4, 1>();
      __builtin_amdgcn_sched_barrier(0);
    }
    add(DT / 2 - 1);
  };
  int c0 = 0, ci = chunk0, half = 0;
  for (; c0 + L < len; c0 += L, ++ci, half ^= 1) chunk(std::false_type{}, c0, ci, half);
  chunk(std::true_type{}, c0, ci, half);
  float* dst = MODE == 1 ? mine : Ss;
  if (colok && (MODE != 2 || seg_idx + 1 == seg_count))
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) dst[(i * 16 + 4 * lg + r) * a.dv + col] = S[i][r];
}

// ---- the states in which segments start, in place of the contributions: W elements of a row per thread (4 where rows
// are multiples of it).  What bounds it is memory's latency, so four segments' loads go out before the first of
// them is stored, and a row's decays are read by fewer threads.  Calls of 8 heads of 128 x 256, us: 1 x 1000 tokens 53.2 -> 49.0,
// 1 x 2000 70.6 -> 60.5, 4 x 600 71.0 -> 64.2, 1 x 8192 153.5 -> 145.5.
template <int W>
__global__ __launch_bounds__(256) void gla_chain_kernel(const GlaArgs a) {
  typedef float FW __attribute__((ext_vector_type(W)));
  const int seq = blockIdx.z, h = blockIdx.y, lane = threadIdx.x & 63;
  const int len = a.qsl[seq + 1] - a.qsl[seq], pos0 = a.seq_lens[seq] - len, slot = a.slots[seq];
  if (len <= a.seg || slot < 0 || slot >= a.num_slots || pos0 < 0) return;
  const int first = pieces_before(seq, a.qsl, a.seg);
  const int count = (len + a.seg - 1) / a.seg, per = a.seg / L, sh = D * a.dv;
  const int chunk0 = chunks_before<L>(seq, a.qsl);
  const int at = (blockIdx.x * 256 + threadIdx.x) * W;
  if (at >= sh) return;
  const int64_t step = (int64_t)a.H * sh;
  const float* pl = a.pl + ((int64_t)chunk0 * a.H + h) * D + at / a.dv;
  float* p = a.seg_state + ((int64_t)first * a.H + h) * sh + at;
  FW S = {};
  if (pos0 != 0) S = *reinterpret_cast<const FW*>(a.S + ((int64_t)slot * a.H + h) * sh + at);
  constexpr int U = 4;
  for (int j0 = 0; j0 < count - 1; j0 += U) {
    FW c[U];
    double f[U];                             // the segments' decays
    const float* g[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = min(j0 + u, count - 2);
      c[u] = *reinterpret_cast<const FW*>(p + j * step);
      g[u] = pl + (int64_t)j * per * a.H * D;
      f[u] = 1.0;
    }
#pragma unroll 4
    for (int k = 0; k < per; ++k)
#pragma unroll
      for (int u = 0; u < U; ++u) f[u] *= g[u][(int64_t)k * a.H * D];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (j0 + u >= count - 1) break;
      *reinterpret_cast<FW*>(p + (j0 + u) * step) = S;
#pragma unroll
      for (int r = 0; r < W; ++r) S[r] = __builtin_fmaf((float)f[u], S[r], c[u][r]);
    }
  }
  *reinterpret_cast<FW*>(p + (count - 1) * step) = S;
}

template <typename T>
void run(const GlaArgs& a, int chunks, hipStream_t s) {
  auto pairs = [](const void* p, int64_t stride, int n) {
    return stride % n == 0 && reinterpret_cast<uintptr_t>(p) % (n * sizeof(T)) == 0;
  };
  if (a.R % 4 == 0 && pairs(a.proj, a.ps, 2) && pairs(a.low, a.ls, 4) && reinterpret_cast<uintptr_t>(a.a2) % 16 == 0)
    gla_prep_kernel<T, true><<<dim3(chunks, a.H), 256, 0, s>>>(a);
  else
    gla_prep_kernel<T, false><<<dim3(chunks, a.H), 256, 0, s>>>(a);
  const int y = a.H * ((a.dv + 127) / 128);
  if (a.seg <= 0) {
    gla_walk_kernel<T, 0><<<dim3(a.P, y), NT, 0, s>>>(a);
  } else {
    gla_walk_kernel<T, 1><<<dim3(a.items, y), NT, 0, s>>>(a);
    if (a.dv % 4 == 0 && ((reinterpret_cast<uintptr_t>(a.S) | reinterpret_cast<uintptr_t>(a.seg_state)) & 15) == 0)
      gla_chain_kernel<4><<<dim3((D * a.dv / 4 + 255) / 256, a.H, a.P), 256, 0, s>>>(a);
    else
      gla_chain_kernel<1><<<dim3((D * a.dv + 255) / 256, a.H, a.P), 256, 0, s>>>(a);
    gla_walk_kernel<T, 2><<<dim3(a.items, y), NT, 0, s>>>(a);
  }
}

// Tokens per segment (0: not cut) and a bound of their number: few sequences leave CUs idle, one workgroup
// on each, over the whole walk.
int plan(int P, int Tp, int H, int V, int* items) {
  *items = P;
  const int wgs = H * ((V + 127) / 128), want = (device_cus() + wgs - 1) / wgs;
  if (P * 2 > want) return 0;
  const int seg = segment_rows(P, Tp, want, L, 4);    // one round
  if (Tp / P < 2 * seg) return 0;
  *items = Tp / seg + P;
  return seg;
}

}  // namespace

bool gla_chunk_ok(int P, int Tp, int H, int d, int V, int R) {
  return gla_rows_pay(P, Tp, H, V) && d == D && V >= 16 && R <= RMAX &&
         chunk_fits(0, (long)H * V, (long)H * ((V + 127) / 128));   // (row offsets have 64 bits)
}
// floats of workspace
int64_t gla_chunk_ws(int P, int Tp, int H, int V) {
  int items;
  const int64_t states = plan(P, Tp, H, V, &items) > 0 ? (int64_t)items * H * D * V : 0;
  return (int64_t)(Tp / L + P) * H * (2 * L * D + D + MAT / 2) + states;
}
void launch_gla_chunk(int dtype, float* out, const void* proj, int64_t ps, const void* low, int64_t ls,
                      const float* a2, const float* a2b, float* S, const int* qsl, const int* seq_lens,
                      const int* slots, int P, int Tp, int H, int V, int R, float tau, int num_slots,
                      float* ws, hipStream_t s) {
  const int chunks = Tp / L + P;
  GlaArgs a{};
  a.out = out; a.proj = proj; a.low = low; a.ps = ps; a.ls = ls; a.a2 = a2; a.a2b = a2b; a.S = S;
  a.qsl = qsl; a.seq_lens = seq_lens; a.slots = slots;
  a.P = P; a.H = H; a.dv = V; a.R = R; a.num_slots = num_slots; a.inv_tau = 1.f / tau;
  a.qp = ws;
  a.kr = a.qp + (int64_t)chunks * H * L * D;
  a.pl = a.kr + (int64_t)chunks * H * L * D;
  a.am = reinterpret_cast<bf16*>(a.pl + (int64_t)chunks * H * D);
  a.seg = plan(P, Tp, H, V, &a.items);
  a.seg_state = ws + (int64_t)chunks * H * (2 * L * D + D + MAT / 2);
  if (dtype == DT_BF16) run<bf16>(a, chunks, s);
  else if (dtype == DT_F16) run<f16>(a, chunks, s);
  else run<float>(a, chunks, s);
}

}  // namespace kgc
