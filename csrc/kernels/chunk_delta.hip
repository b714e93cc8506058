// Chunkwise gated delta rule (Yang, Kautz and Hatamizadeh, gated delta networks, 2024) of prompt rows on the
// matrix cores.  Per (sequence, head), with unit
// keys k_t, a decay g_t and a write strength beta_t,
//     u_t = beta_t (v_t - g_t S_(t-1)^T k_t),   S_t = g_t S_(t-1) + k_t u_t^T,   o_t = S_t^T q_t .
// Over a chunk of L = 32 tokens, b_t the running sum of ln g, gamma_t = e^(b_t) and S_0 the state
// before it, the u of the chunk solve a unit lower triangular system:
//     (I + A) U = diag(beta) (V - diag(gamma) K S_0),   A_ts = beta_t e^(b_t - b_s) k_t . k_s  (s < t)
//     O   = diag(gamma) Q S_0 + P U,                    P_ts = e^(b_t - b_s) q_t . k_s         (s <= t)
//     S_L = gamma_L S_0 + sum_s e^(b_L - b_s) k_s u_s^T
// W = (I + A)^-1 diag(beta) and P depend on no state: a first launch computes them for all chunks at
// once (the inverses by blocks of 16 rows), as bf16 parts in the order the walk's MFMAs
// read them.  The walk then has no serial step finer than a chunk: a workgroup of 8 waves owns 128
// value columns of a head, a wave 16 of them with their S in accumulators, and everything between
// two stagings of k and q concerns one wave's columns only:
//     R = V - gamma K S_0,  U = W R,  O = gamma Q S_0 + P U,  S = gamma_L S_0 + K^T U.
// Accumulators are B operands as they lie (mfma_perm), so R, U and S never pass through LDS.
//
// Precision: fp32 operands enter the bf16 MFMAs as three bf16 parts each, six products of parts.  The corrections
// of K S_0 and Q S_0 have sums of their own; those of W R, P U and K^T U are summed first and the main products on top
// of them.  Exponents are differences of running sums kept in double.
//
// Few long sequences are cut into segments: a chunk walk is linear in its state, so a first pass
// walks every segment from zero (with its values) and from the identity (without), a second chains
// S <- M_j S + dS_j over the segments, and the third walks all segments from their own states.
#include <algorithm>
#include <type_traits>
#include "chunk.h"
#include "chunk_rows.h"
#include "device.h"
#include "launch.h"

namespace kgc {

namespace {

constexpr int L = 32, D = 128;               // tokens per chunk, key channels
constexpr int NT = 512, NW = NT / 64;
constexpr int DT = D / 16, LT = L / 16, KD = D / 32;
constexpr int DP = D + 8, LP = L + 8;        // padded LDS rows
constexpr int MAT = 3 * L * L;               // bf16 of one matrix of a chunk: three parts

struct DeltaArgs {
  float* out;                                // [T, H dv]
  const float* qkv;                          // [T, 2 G D + H dv]
  int64_t stride;
  const void* ba;                            // [T, 2 H]: write strength | decay, before activation
  int64_t bas;
  int ba_type;
  const float *a_log, *dt_bias;
  float* S;
  const int *qsl, *seq_lens, *slots;
  int P, H, G, dv, num_slots;
  // workspace
  bf16* wp;                                  // [chunks][H][W, P][3][L][L], columns permuted
  // per token of a chunk, zero past the sequence's end:
  float* gam;                                // [chunks][H][L]: gamma_t
  f32x2* kw;                                 // [chunks][H][L]: e^(b_L - b_t) times rk, the rounding and what it leaves (48
                                             // bits; weights below 2^-126 have fewer)
  float *rk, *rq;                            // [chunks][G][L]: what makes k and q unit (q: d^-1/2 too)
  int seg;                                   // tokens per segment (0: sequences are not cut)
  float* seg_state;                          // [items][H][D][dv + D]: dS | M of a segment
  float* seg_in;                             // [items][H][D][dv]: the state a segment starts from
};

__device__ __forceinline__ float ld_ba(const DeltaArgs& a, int64_t at) {
  return a.ba_type == DT_F32 ? reinterpret_cast<const float*>(a.ba)[at]
         : a.ba_type == DT_F16 ? (float)reinterpret_cast<const f16*>(a.ba)[at]
                               : (float)reinterpret_cast<const bf16*>(a.ba)[at];
}

// inclusive running sum within each half of the wave
__device__ __forceinline__ double half_scan(double x) {
  x = scan_step<0x111, 0xf, false>(x);
  x = scan_step<0x112, 0xf, false>(x);
  x = scan_step<0x114, 0xf, false>(x);
  x = scan_step<0x118, 0xf, false>(x);
  return scan_step<0x142, 0xa, false>(x);
}

// between writing and reading LDS within one wave: its LDS operations execute in order
__device__ __forceinline__ void wave_lds() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// place of a 16-byte unit of W or P, so that 16 lanes read 16 different bank groups
__device__ __forceinline__ int wp_unit(int t, int u) { return t * (L / 8) + (u ^ ((t >> 2) & 3)); }

// ---- W, P, the gates and the norms of every chunk: one wave per (chunk, q / k group) -----------
// Dots, P and A stay in the layout of the MFMAs that made them, [s][t] with t the lane's: a lane's elements of a row are
// the units that the walk reads.  (I + A)^-1 by blocks of 16, a lane per column of each diagonal block of two
// heads: T21 = -T22 A21 T11 in fp32 MFMAs.
__global__ __launch_bounds__(64, 2) void delta_prep_kernel(const DeltaArgs a) {
  constexpr int XR = 20, XB = 16 * XR + 16;  // floats of a row of a block, of a block: the four on banks of their own
  __shared__ __align__(16) float X[4 * XB];  // [head][block]: A, then its inverse
  __shared__ __align__(16) double bs[2][L];
  __shared__ __align__(16) float be[2][L];
  const SegItem it = seg_item(blockIdx.x, a.qsl, a.P, L);
  if (it.seq < 0) return;
  const int g = blockIdx.y, lane = threadIdx.x, lr = lane & 15, lg = lane >> 4;
  const int c0 = it.idx * L, len = a.qsl[it.seq + 1] - a.qsl[it.seq];
  const int nl = min(L, len - c0);
  const int slot = a.slots[it.seq];
  if (nl <= 0 || slot < 0 || slot >= a.num_slots || a.seq_lens[it.seq] < len) return;
  const int64_t t0 = a.qsl[it.seq] + c0;
  const float* qb = a.qkv + t0 * a.stride + g * D;
  const float* kb = qb + (int64_t)a.G * D;
  const int rs = (int)a.stride, hpg = a.H / a.G;

  const int hf = lane >> 5, s = lane & 31;   // gates: this lane's token of head h0 + hf
  const int64_t row = (t0 + min(s, nl - 1)) * a.bas;
  auto head = [&](int h0) { return g * hpg + min(h0 + hf, hpg - 1); };
  float gx = ld_ba(a, row + head(0)), gz = ld_ba(a, row + a.H + head(0));   // land during the dots
  float gb = a.dt_bias[head(0)], ga = a.a_log[head(0)];

  // dots: tiles (0, 0), (1, 0), (1, 1) as D[s][t]; the squares of the same elements give the norms
  f32x4 dk[3], dkl[3], dq[3], dql[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) dk[i] = dkl[i] = dq[i] = dql[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  double n2[2][2] = {{0.0, 0.0}, {0.0, 0.0}};             // [k, q][tile]
  const int at[2] = {min(lr, nl - 1) * rs + lg * 8, min(16 + lr, nl - 1) * rs + lg * 8};
  f32x4 in[2][2][2][2];                      // 32 columns of k and q, the next 32
  auto fetch = [&](int j) {
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (int ti = 0; ti < LT; ++ti)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          in[j & 1][w][ti][i] = *reinterpret_cast<const f32x4*>((w ? qb : kb) + at[ti] + j * 32 + i * 4);
  };
  fetch(0);
#pragma unroll
  for (int j = 0; j < KD; ++j) {
    if (j + 1 < KD) fetch(j + 1);
    __builtin_amdgcn_sched_barrier(0);
    bf16x8 f[2][2][3];
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (int ti = 0; ti < LT; ++ti) {
        const f32x4 x0 = in[j & 1][w][ti][0], x1 = in[j & 1][w][ti][1];
        const float x[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
#pragma unroll
        for (int i = 0; i < 8; ++i) n2[w][ti] = __builtin_fma((double)x[i], (double)x[i], n2[w][ti]);
        split8<3>(x, f[w][ti]);
      }
#pragma unroll
    for (int tile = 0; tile < 3; ++tile) {
      const int ti = tile > 0, si = tile > 1;
      mm<true, 3, 3>(f[0][si], f[0][ti], dk[tile], dkl[tile]);
      mm<true, 3, 3>(f[0][si], f[1][ti], dq[tile], dql[tile]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  float rn[2][2];
#pragma unroll
  for (int w = 0; w < 2; ++w)
#pragma unroll
    for (int ti = 0; ti < LT; ++ti) {
      double n = n2[w][ti];
      n += __shfl_xor(n, 16, 64);
      n += __shfl_xor(n, 32, 64);
      rn[w][ti] = (float)(1.0 / sqrt((n + 1e-6) * (w ? D : 1)));
      const int t = ti * 16 + lr;
      if (lg == 0) (w ? a.rq : a.rk)[((int64_t)blockIdx.x * a.G + g) * L + t] = t < nl ? rn[w][ti] : 0.f;
    }
  float kk[3][4], qk[3][4];                  // dots of unit vectors
#pragma unroll
  for (int tile = 0; tile < 3; ++tile) {
    const int ti = tile > 0, si = tile > 1;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float f = __shfl(rn[0][si], lg * 4 + r, 64);
      kk[tile][r] = (dk[tile][r] + dkl[tile][r]) * (f * rn[0][ti]);
      qk[tile][r] = (dq[tile][r] + dql[tile][r]) * (f * rn[1][ti]);
    }
  }
  const float r0 = __shfl(rn[0][0], s & 15, 64), r1 = __shfl(rn[0][1], s & 15, 64), rks = s < 16 ? r0 : r1;

  for (int h0 = 0; h0 < hpg; h0 += 2) {
    const bool ok = s < nl;
    {
      const int h = head(h0);
      const float x = gx;
      const double z = (double)gz + (double)gb;
      double f = -exp((double)ga) * (z > 40.0 ? z : log1p(exp(z)));
      if (h0 + 2 < hpg) {
        gx = ld_ba(a, row + head(h0 + 2));
        gz = ld_ba(a, row + a.H + head(h0 + 2));
        gb = a.dt_bias[head(h0 + 2)];
        ga = a.a_log[head(h0 + 2)];
      }
      // a decay of e^-1e6 is zero; a finite floor keeps the differences of running sums defined
      const double b = half_scan(!ok ? 0.0 : f < -1e6 ? -1e6 : f);
      const uint64_t bb = __builtin_bit_cast(uint64_t, b);
      const uint32_t bl = __shfl((int)(uint32_t)bb, 31 + 32 * hf, 64), bh = __shfl((int)(bb >> 32), 31 + 32 * hf, 64);
      const double bL = __builtin_bit_cast(double, (uint64_t)bh << 32 | bl);
      bs[hf][s] = b;
      be[hf][s] = ok ? 1.f / (1.f + expf(-x)) : 0.f;
      if (h0 + hf < hpg) {
        a.gam[((int64_t)blockIdx.x * a.H + h) * L + s] = ok ? (float)exp(b) : 0.f;
        const double w = ok ? exp(bL - b) * rks : 0.0;    // as a sum of two floats
        const float wh = (float)w;
        a.kw[((int64_t)blockIdx.x * a.H + h) * L + s] = f32x2{wh, (float)(w - wh)};
      }
    }
    wave_lds();
    // rows of a matrix as three parts, eight (permuted) columns to a store: those of tile (ti, 0), then of (ti, 1)
    auto put = [&](int hh, int mat, int ti, const float (&y)[8]) {
      bf16x8 o[3];
      split8<3>(y, o);
      bf16* dst = a.wp + (((int64_t)blockIdx.x * a.H + g * hpg + h0 + hh) * 2 + mat) * MAT + wp_unit(ti * 16 + lr, lg) * 8;
#pragma unroll
      for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8*>(dst + i * L * L) = o[i];
    };
    float a21[2][4];
    int bad[2] = {L, L};                     // the first token whose row of A or write strength is not finite
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const double tb[2] = {bs[hh][lr], bs[hh][16 + lr]};
      const float bt[2] = {be[hh][lr], be[hh][16 + lr]};
      float A[3][4], P[3][4], z = bt[0] + bt[1];
#pragma unroll
      for (int tile = 0; tile < 3; ++tile) {
        const int ti = tile > 0, si = tile > 1;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int d = tile == 1 ? 16 : lr - (4 * lg + r);   // t - s
          float e = exp_d(tb[ti] - bs[hh][si * 16 + 4 * lg + r]);
          asm volatile("" : "+v"(e));        // (no branches)
          P[tile][r] = d >= 0 ? e * qk[tile][r] : 0.f;
          A[tile][r] = d > 0 ? bt[ti] * e * kk[tile][r] : 0.f;
          z += A[tile][r];
        }
      }
      if (h0 + hh < hpg) {
        put(hh, 1, 0, {P[0][0], P[0][1], P[0][2], P[0][3], 0.f, 0.f, 0.f, 0.f});
        put(hh, 1, 1, {P[1][0], P[1][1], P[1][2], P[1][3], P[2][0], P[2][1], P[2][2], P[2][3]});
      }
      // Products of blocks would carry what is not finite to the rows before it: such rows of A are left out,
      // and those of W written as NaN from the first one on.
      if (__any(!(fabsf(z) < INFINITY))) {
        auto odd = [](float x) { return !(fabsf(x) < INFINITY); };
        bool b0 = odd(bt[0]), b1 = odd(bt[1]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          b0 |= odd(A[0][r]);
          b1 |= odd(A[1][r]) || odd(A[2][r]);
        }
        int f = b0 ? lr : b1 ? 16 + lr : L;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) f = min(f, __shfl_xor(f, o, 64));
        bad[hh] = f;
#pragma unroll
        for (int tile = 0; tile < 3; ++tile)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if ((tile > 0) * 16 + lr >= f) A[tile][r] = 0.f;
      }
      *reinterpret_cast<f32x4*>(X + 2 * hh * XB + lr * XR + 4 * lg) = f32x4{A[0][0], A[0][1], A[0][2], A[0][3]};
      *reinterpret_cast<f32x4*>(X + (2 * hh + 1) * XB + lr * XR + 4 * lg) = f32x4{A[2][0], A[2][1], A[2][2], A[2][3]};
#pragma unroll
      for (int r = 0; r < 4; ++r) a21[hh][r] = A[1][r];
    }
    wave_lds();
    {                                        // column lr of the inverse of block lg, from the top
      float* B = X + lg * XB;
      float T[16];
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        float x[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < t; j += 4) {
          const f32x4 r = *reinterpret_cast<const f32x4*>(B + t * XR + j);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (j + i < t) x[i] += r[i] * T[j + i];
        }
        const float y = -((x[0] + x[1]) + (x[2] + x[3]));
        T[t] = t == lr ? 1.f : t < lr ? 0.f : y;
      }
      wave_lds();
#pragma unroll
      for (int t = 0; t < 16; ++t) B[t * XR + lr] = T[t];
    }
    wave_lds();
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const float *B0 = X + 2 * hh * XB, *B1 = B0 + XB;
      const f32x4 t11 = *reinterpret_cast<const f32x4*>(B0 + lr * XR + 4 * lg);
      const f32x4 t22 = *reinterpret_cast<const f32x4*>(B1 + lr * XR + 4 * lg);
      f32x4 m = {0.f, 0.f, 0.f, 0.f}, t21 = m;
#pragma unroll
      for (int r = 0; r < 4; ++r) m = __builtin_amdgcn_mfma_f32_16x16x4f32(a21[hh][r], B0[(4 * lg + r) * XR + lr], m, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) t21 = __builtin_amdgcn_mfma_f32_16x16x4f32(m[r], t22[r], t21, 0, 0, 0);
      const f32x4 c0 = *reinterpret_cast<const f32x4*>(&be[hh][4 * lg]), c1 = *reinterpret_cast<const f32x4*>(&be[hh][16 + 4 * lg]);
      float w0[8], w1[8];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool in = 4 * lg + r <= lr;
        w0[r] = in ? t11[r] * c0[r] : 0.f;
        w0[4 + r] = 0.f;
        w1[r] = -t21[r] * c0[r];
        w1[4 + r] = in ? t22[r] * c1[r] : 0.f;
      }
      if (bad[hh] < L)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool in = 4 * lg + r <= lr;
          if (lr >= bad[hh] && in) w0[r] = NAN;
          if (16 + lr >= bad[hh]) w1[r] = NAN;
          if (16 + lr >= bad[hh] && in) w1[4 + r] = NAN;
        }
      if (h0 + hh < hpg) {
        put(hh, 0, 0, w0);
        put(hh, 0, 1, w1);
      }
    }
    wave_lds();                              // (the next heads write where these were read)
  }
}

// ---- the walk.  MODE 0: whole sequences; 1: segments from zero and from the identity (states
// only); 2: segments from seg_in -----------------------------------------------------------------
template <int MODE>
__global__ __launch_bounds__(NT) void delta_walk_kernel(const DeltaArgs a) {
  __shared__ __align__(16) bf16 Ks[3 * L * DP], Qs[MODE == 1 ? 8 : 3 * L * DP], KT[3 * D * LP];
  __shared__ __align__(16) bf16 Ws[MAT], Ps[MODE == 1 ? 8 : MAT];
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int seq = blockIdx.x, seg_idx = 0, item = 0, seg_count = 1;
  if (MODE != 0) {
    const SegItem it = seg_item(blockIdx.x, a.qsl, a.P, a.seg);
    if (it.seq < 0) return;
    seq = __builtin_amdgcn_readfirstlane(it.seq);
    seg_idx = __builtin_amdgcn_readfirstlane(it.idx);
    seg_count = __builtin_amdgcn_readfirstlane(it.count);
    item = __builtin_amdgcn_readfirstlane(it.first) + seg_idx;
    if (MODE == 1 && seg_idx + 1 == seg_count) return;
  }
  const int nct = (a.dv + 127) / 128 + (MODE == 1);       // MODE 1: the last block is the identity's
  auto uniform = [](int x) { return __builtin_amdgcn_readfirstlane(x); };   // (a division is the vector unit's)
  const int h = uniform(blockIdx.y / nct), ct = blockIdx.y - h * nct, g = uniform(h / (a.H / a.G));
  const bool ident = MODE == 1 && ct + 1 == nct;
  const int col = (ident ? 0 : ct * 128) + wave * 16 + lr;
  const bool colok = ident || col < a.dv;
  const int colc = colok ? col : a.dv - 1;                // columns off the edge: read the last
  int start = uniform(a.qsl[seq]), len = uniform(a.qsl[seq + 1]) - start;
  const int pos0 = uniform(a.seq_lens[seq]) - len, slot = uniform(a.slots[seq]);
  const int64_t os = (int64_t)a.H * a.dv;
  const int chunk0 = __builtin_amdgcn_readfirstlane(chunks_before<L>(seq, a.qsl)) + (MODE != 0 ? seg_idx * (a.seg / L) : 0);
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
  f32x4 S[DT];
  float* Ss = a.S + ((int64_t)slot * a.H + h) * D * a.dv;
  {
    const float* from = MODE == 2 ? a.seg_in + ((int64_t)item * a.H + h) * D * a.dv : Ss;
    const bool zero = MODE == 1 || (MODE == 0 && pos0 == 0);
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = i * 16 + 4 * lg + r;
        S[i][r] = zero ? (ident && row == col ? 1.f : 0.f) : from[row * a.dv + colc];
      }
  }
  const float* qb = a.qkv + g * D;
  const float* kb = qb + (int64_t)a.G * D;
  const float* vb = a.qkv + 2 * (int64_t)a.G * D + (int64_t)h * a.dv;
  const int vo = ident ? 0 : colc;
  int rs = (int)a.stride, ro = (int)os;
  // (a base in vector registers would make every store of an output a loop over its values)
  const uint64_t ob64 = reinterpret_cast<uint64_t>(a.out + start * os + (int64_t)h * a.dv);
  char* const ob = reinterpret_cast<char*>((uint64_t)(uint32_t)uniform((int)(ob64 >> 32)) << 32 | (uint32_t)uniform((int)ob64));

  // Staging: a thread takes 8 columns of one row of q and k, and 8 tokens of one column of k, in
  // both cases the pieces 4 a .. and 16 + 4 a .. of 32: adjacent in the permuted order, one store.
  // Rows past the sequence's end: through descriptors that end with the chunk's last row, zeros.
  f32x4 rqv[2], rkv[2], rt[2];
  f32x2 kw[8];
  float nk = 0.f, nq = 0.f;
  const int ut = tid / 16, uc = (tid % 16 / 4) * 32 + (tid % 4) * 4, up_ = (tid % 16) * 8;
  const int ta = tid / D * 4, tc = tid % D;
  auto rows_of = [&](const float* p, int c0, int w) {
    const float* r = p + (int64_t)(start + c0) * a.stride;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(r), 0, ((min(L, len - c0) - 1) * rs + w) * 4, 0x00027000);
  };
  auto ld16 = [&](__amdgpu_buffer_rsrc_t r, uint32_t at) { return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0)); };
  auto ld4 = [&](__amdgpu_buffer_rsrc_t r, uint32_t at) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, at, 0, 0)); };
  auto fetch_rows = [&](int c0, int ci) {
    const uint32_t at = (__mul24(ut, rs) + uc) * 4;
    const auto kr = rows_of(kb, c0, D);
    rkv[0] = ld16(kr, at);
    rkv[1] = ld16(kr, at + 64);
    nk = a.rk[((int64_t)ci * a.G + g) * L + ut];
    if (MODE != 1) {
      const auto qr = rows_of(qb, c0, D);
      rqv[0] = ld16(qr, at);
      rqv[1] = ld16(qr, at + 64);
      nq = a.rq[((int64_t)ci * a.G + g) * L + ut];
    }
  };
  auto fetch_cols = [&](int c0, int ci) {
    const auto kr = rows_of(kb, c0, D);
    const uint32_t at = (__mul24(ta, rs) + tc) * 4;
#pragma unroll
    for (int i = 0; i < 8; ++i) rt[i >> 2][i & 3] = ld4(kr, at + ((i >> 2) * 16 + (i & 3)) * rs * 4);
    const f32x2* w = a.kw + ((int64_t)ci * a.H + h) * L + ta;
#pragma unroll
    for (int i = 0; i < 8; ++i) kw[i] = w[(i >> 2) * 16 + (i & 3)];
  };
  auto park_rows = [&](int w0, int w1) {
#pragma unroll
    for (int w = w0; w < w1; ++w) {
      const f32x4* v = w ? rqv : rkv;
      const float f = w ? nq : nk;
      float x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = v[i >> 2][i & 3] * f;
      bf16x8 p[3];
      split8<3>(x, p);
      bf16* base = (w ? Qs : Ks) + ut * DP + up_;
#pragma unroll
      for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8*>(base + i * L * DP) = p[i];
    }
  };
  auto park_cols = [&]() {
    // k^T times the weight of its token in the update, tokens permuted: U is the B operand as it lies
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = __builtin_fmaf(rt[i >> 2][i & 3], kw[i][0], rt[i >> 2][i & 3] * kw[i][1]);
    bf16x8 p[3];
    split8<3>(x, p);
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8*>(KT + (i * D + tc) * LP + ta * 2) = p[i];
  };
  auto split_s = [&](bf16x8 (&sp)[3], int j) {
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = S[2 * j + (i >> 2)][i & 3];
    split8<3>(x, sp);
  };
  struct Own { float v[LT][4]; f32x4 gm[LT]; float gL; };
  // this lane's v and gammas (rows 4 lg + r of each tile)
  auto fetch_own = [&](Own& w, int c0, int ci) {
    const int nl = min(L, len - c0);
    const auto vr = rows_of(vb, c0, a.dv);
    const uint32_t at = (__mul24(lg * 4, rs) + vo) * 4;
    const float* gc = a.gam + ((int64_t)ci * a.H + h) * L;
#pragma unroll
    for (int ti = 0; ti < LT; ++ti) {
      w.gm[ti] = *reinterpret_cast<const f32x4*>(gc + ti * 16 + lg * 4);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        w.v[ti][r] = ld4(vr, at + (ti * 16 + r) * rs * 4);
    }
    w.gL = gc[nl - 1];
  };
  // W or P of a chunk, to LDS as they lie
  auto dma = [&](int ci, int mat, bf16* dst) {
    if (wave < MAT * 2 / 1024)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(a.wp + (((int64_t)ci * a.H + h) * 2 + mat) * MAT + wave * 512 + lane * 8),
          (__attribute__((address_space(3))) void*)(dst + wave * 512), 16, 0, 0);
  };
  auto load_wp = [&](const bf16* m, bf16x8 (&f)[LT][3]) {
#pragma unroll
    for (int ti = 0; ti < LT; ++ti)
#pragma unroll
      for (int i = 0; i < 3; ++i)
        f[ti][i] = *reinterpret_cast<const bf16x8*>(m + i * L * L + wp_unit(ti * 16 + lr, lg) * 8);
  };

  // Staged rows are parked while the last chunk's update runs, columns beside the products with S: k^T is not
  // read before the barrier between the two.  (The last chunk, which has none to stage, is a copy of its own: a branch
  // would end the regions in which vector instructions and MFMAs are interleaved, and staging the same again took steps
  // of short prompts 3 to 8 % longer: 100 x 20 95.7 us, so 89.5, 400 x 16 345 and 307.)
  Own next;
  bf16x8 sp[2][3];                           // parts of 32 rows of S; the first ones of the next chunk
  split_s(sp[0], 0);
  dma(chunk0, 0, Ws);
  fetch_rows(0, chunk0);
  fetch_cols(0, chunk0);
  fetch_own(next, 0, chunk0);
  park_rows(0, MODE == 1 ? 1 : 2);
  auto chunk = [&](auto last, int c0, int ci) {
    constexpr bool LAST = decltype(last)::value;
    const int nl = LAST ? len - c0 : L, cn = c0 + L, cin = ci + 1;
    asm volatile("" : "+s"(rs), "+s"(ro));   // row offsets are computed per chunk, not kept
    meet<MODE == 1 ? 0 : 8>();               // (the last chunk's outputs may still be on their way)
    const Own own = next;
    if (MODE != 1) dma(ci, 1, Ps);
    f32x4 r[LT], rl[LT], o[LT], ol[LT];
#pragma unroll
    for (int ti = 0; ti < LT; ++ti) r[ti] = rl[ti] = o[ti] = ol[ti] = f32x4{0.f, 0.f, 0.f, 0.f};
    // products with S in steps of 32 of its rows, k's and q's in turn: the next step's operands are read, and the
    // next parts of S made, beside the MFMAs
    bf16x8 f[2][LT][3];
    auto load_rows = [&](bf16x8 (&x)[LT][3], const bf16* m, int j) {
#pragma unroll
      for (int ti = 0; ti < LT; ++ti)
#pragma unroll
        for (int i = 0; i < 3; ++i)
          x[ti][i] = *reinterpret_cast<const bf16x8*>(m + i * L * DP + (ti * 16 + lr) * DP + j * 32 + lg * 8);
    };
    load_rows(f[0], Ks, 0);
    __builtin_amdgcn_sched_barrier(0);
    bf16x8 rp[3];
    auto make_r = [&]() {                    // (rows past the end: W is zero there)
      float x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int ti = i >> 2, e = i & 3;
        x[i] = __builtin_fmaf(-own.gm[ti][e], r[ti][e] + rl[ti][e], ident ? 0.f : own.v[ti][e]);
      }
      if (LAST)
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = (i >> 2) * 16 + lg * 4 + (i & 3) >= nl ? 0.f : x[i];
      split8<3>(x, rp);
    };
#pragma unroll
    for (int j = 0; j < KD; ++j) {
      const int k = MODE != 1 ? 0 : j & 1;
      if (MODE != 1) load_rows(f[1], Qs, j);
      else if (j + 1 < KD) load_rows(f[k ^ 1], Ks, j + 1);
      if (MODE == 1 && j + 1 < KD) split_s(sp[(j + 1) & 1], j + 1);
      if (!LAST && j == 0) fetch_rows(cn, cin);       // of the next chunk
      if (!LAST && j == 1) fetch_own(next, cn, cin);
      mm3_add<LT>(f[k], sp[j & 1], r, rl);
      if (!LAST && j < 2) interleave<12, 4, 2, 1>();
      else interleave<12, 4, 2>();
      __builtin_amdgcn_sched_barrier(0);
      if (MODE != 1) {
        if (j + 1 < KD) load_rows(f[0], Ks, j + 1);
        else load_wp(Ws, f[0]);
        if (j + 1 < KD) split_s(sp[(j + 1) & 1], j + 1);
        else make_r();
        mm3_add<LT>(f[1], sp[j & 1], o, ol);
        interleave<12, 4, 2>();
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (MODE == 1) {
      load_wp(Ws, f[0]);
      make_r();
    }
    bf16x8 (&fw)[LT][3] = f[0];
    // U = W R
    bf16x8 up[3];
    int bad = L;                             // first token whose value is not finite
    {
      float x[8];
      f32x4 u[LT];
      mm3<LT>(fw, rp, u);
      park_cols();
      interleave<12, 6>();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = u[i >> 2][i & 3];
      // A row of R or W that is not finite reaches all rows of U, or all from its own on: the last one
      // shows it.  Then U once more without such rows of R, and without what is not finite itself,
      // before P carries it to the rows before it.
      if (__any(!(fabsf(x[7]) < INFINITY))) {
        auto tok = [&](int i) { return (i >> 2) * 16 + lg * 4 + (i & 3); };
        float y[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = (float)rp[0][i];
        bad = take_nonfinite(y, L, tok);
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (tok(i) >= bad) rp[0][i] = rp[1][i] = rp[2][i] = (bf16)0.f;
        mm3<LT>(fw, rp, u);
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = u[i >> 2][i & 3];
        bad = min(bad, take_nonfinite(x, L, tok));
      }
      split8<3>(x, up);
#pragma unroll
      for (int i = 0; i < 3; ++i) asm volatile("" : "+v"(up[i]));   // before the barrier
    }
    const bool some_bad = __builtin_amdgcn_readfirstlane(__any(bad < L));
    meet<0>();                               // k, q and W were read, k^T and P are there
    if (!LAST) dma(cin, 0, Ws);
    auto load_cols = [&](bf16x8 (&x)[LT][3], int dt) {
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int i = 0; i < 3; ++i)
          x[k][i] = *reinterpret_cast<const bf16x8*>(KT + (i * D + (dt + k) * 16 + lr) * LP + lg * 8);
    };
    auto update = [&](int dt) {
      const int k = dt >> 1 & 1;
      if (dt + 2 < DT) load_cols(f[k ^ 1], dt + 2);
      f32x4 t[2];
      mm3<2>(f[k], up, t);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[dt + i][e] = __builtin_fmaf(S[dt + i][e], own.gL, t[i][e]);
    };
    if (MODE != 1) load_wp(Ps, f[1]);
    load_cols(f[0], 0);
    __builtin_amdgcn_sched_barrier(0);
    if (MODE != 1) {
      f32x4 pu[LT];
      mm3<LT>(f[1], up, pu);
#pragma unroll
      for (int ti = 0; ti < LT; ++ti)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[ti][e] = __builtin_fmaf(own.gm[ti][e], o[ti][e] + ol[ti][e], pu[ti][e]);
    }
    if (!LAST) {
      fetch_cols(cn, cin);                   // of the next chunk
      park_rows(0, 1);
    }
    update(0);
    update(2);
    interleave<MODE != 1 ? 36 : 24, 3, 3, LAST ? 0 : 2>();
    __builtin_amdgcn_sched_barrier(0);
    if (some_bad) {                          // (before the last rows' update, which they pass through)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          asm volatile("" : "+v"(S[dt][e]));    // a branch, not selects in every chunk
          if (bad < L) S[dt][e] = NAN;
        }
      if (MODE != 1)
#pragma unroll
        for (int ti = 0; ti < LT; ++ti)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            asm volatile("" : "+v"(o[ti][e]));
            if (ti * 16 + lg * 4 + e >= bad) o[ti][e] = NAN;
          }
    }
    if (MODE != 1) {
      // through a descriptor that ends with the chunk's last value: writes past it do nothing
      const auto od = __builtin_amdgcn_make_buffer_rsrc(ob + (int64_t)c0 * os * 4, 0, ((nl - 1) * ro + a.dv) * 4, 0x00027000);
      const uint32_t at = colok ? (uint32_t)(__mul24(lg * 4, ro) + col) * 4 : 1u << 30;
#pragma unroll
      for (int ti = 0; ti < LT; ++ti)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float y = o[ti][e];
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, y), od, at + (ti * 16 + e) * ro * 4, 0, 0);
        }
      if (!LAST) park_rows(1, 2);
    }
    if (!LAST) split_s(sp[0], 0);
    update(4);
    update(6);
    if (MODE == 1 || LAST) interleave<24, 4, 2>();
    else interleave<24, 6, 2, 3>();
    __builtin_amdgcn_sched_barrier(0);
  };
  int c0 = 0, ci = chunk0;
  for (; c0 + L < len; c0 += L, ++ci) chunk(std::false_type(), c0, ci);
  chunk(std::true_type(), c0, ci);

  if (MODE == 1 || MODE == 0 || seg_idx + 1 == seg_count) {
    // MODE 1: dS and M side by side
    const int w = MODE == 1 ? a.dv + D : a.dv;
    float* dst = MODE == 1 ? a.seg_state + ((int64_t)item * a.H + h) * D * w + (ident ? a.dv : 0) : Ss;
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (colok) dst[(i * 16 + 4 * lg + e) * w + col] = S[i][e];
  }
}

// ---- S_in of every segment: S <- M_j S + dS_j.  A workgroup owns 16 columns of one (sequence, head), each of its 8 waves 16
// rows: the parts of S pass through LDS, the next segment's rows of M are on their way meanwhile.  (One wave for the 16
// columns, M read when it is needed, bound by that chain: 24 us a segment; 1 x 2000 tokens of 16 heads 267 -> 107 us, 1 x 8192
// 616 -> 300.)
__global__ __launch_bounds__(NT) void delta_chain_kernel(const DeltaArgs a) {
  static_assert(NW == DT, "a wave per 16 rows");
  typedef float F4 __attribute__((ext_vector_type(4), aligned(4)));
  __shared__ __align__(16) uint32_t sx[2][KD][3][64][4];
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int seq = blockIdx.x, h = blockIdx.y, col = blockIdx.z * 16 + lr;
  const bool colok = col < a.dv;
  const int colc = colok ? col : a.dv - 1;
  const int len = a.qsl[seq + 1] - a.qsl[seq], pos0 = a.seq_lens[seq] - len, slot = a.slots[seq];
  if (len <= 0 || slot < 0 || slot >= a.num_slots || pos0 < 0) return;
  const int first = pieces_before(seq, a.qsl, a.seg);
  const int count = (len + a.seg - 1) / a.seg, w = a.dv + D;
  const float* Ss = a.S + ((int64_t)slot * a.H + h) * D * a.dv;
  f32x4 S;
#pragma unroll
  for (int e = 0; e < 4; ++e) S[e] = pos0 == 0 ? 0.f : Ss[(wave * 16 + 4 * lg + e) * a.dv + colc];
  F4 m[KD][2];                               // row wave * 16 + lr of M, columns in the permuted order
  f32x4 d;
  auto fetch = [&](int j) {
    const float* st = a.seg_state + ((int64_t)(first + j) * a.H + h) * D * w;
    const float* row = st + (wave * 16 + lr) * w + a.dv + lg * 4;
#pragma unroll
    for (int k = 0; k < KD; ++k)
#pragma unroll
      for (int i = 0; i < 2; ++i) m[k][i] = *reinterpret_cast<const F4*>(row + k * 32 + i * 16);
#pragma unroll
    for (int e = 0; e < 4; ++e) d[e] = st[(wave * 16 + 4 * lg + e) * w + colc];
  };
  if (count > 1) fetch(0);
  for (int j = 0;; ++j) {
    float* dst = a.seg_in + ((int64_t)(first + j) * a.H + h) * D * a.dv;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (colok) dst[(wave * 16 + 4 * lg + e) * a.dv + col] = S[e];
    if (j + 1 == count) break;
    uint32_t p0[3], p1[3];
    split2<3>(S[0], S[1], p0);
    split2<3>(S[2], S[3], p1);
#pragma unroll
    for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x2*>(&sx[j & 1][wave >> 1][p][lane][2 * (wave & 1)]) = u32x2{p0[p], p1[p]};
    bf16x8 fa[KD][3];
#pragma unroll
    for (int k = 0; k < KD; ++k) {
      float x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = m[k][i >> 2][i & 3];
      split8<3>(x, fa[k]);
    }
    const f32x4 dc = d;
    if (j + 2 < count) fetch(j + 1);
    meet<63>();                              // (the parts are there; loads and stores stay on their way)
    f32x4 hi = {0.f, 0.f, 0.f, 0.f}, lo = hi;
#pragma unroll
    for (int k = 0; k < KD; ++k) {
      bf16x8 sp[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) sp[p] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(&sx[j & 1][k][p][lane][0]));
      mm<true, 3, 3>(fa[k], sp, hi, lo);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) S[e] = hi[e] + lo[e] + dc[e];
  }
}

}  // namespace

// Chunkwise for 128 key channels where the rows pay (chunk_rows.h; a chunk's workspace is 200 KB for 16
// heads, which few rows per sequence would multiply, too).  16 x 1000 tokens of 16 heads with 128 x 128
// states: 1328 us token by token, 245 us chunkwise, 55 of it W and P, whose bytes (k and q in, W and P out: 210 MB) take
// 42; 2 x 8192: 7.5 ms and 0.68 ms.  Per wave and chunk the walk issues 580 vector instructions and 168 MFMAs in 11000
// cycles: 7300 of two waves' issue (vector instructions in 52 % of the cycles, the matrix core in 47), 6100 of the LDS that 95
// reads of 1 KB per wave keep busy, the rest the barriers and the chain R -> U.
// What the walk's issue was spent on before (281 us, on the same card): outputs stored in loops over the
// values of a descriptor that was not scalar; weights of k^T in double; 64-bit addresses of every staged element; vector work
// behind the products instead of between them.  And the first launch's (72 us): columns of the inverse of 32 rows, dots
// through LDS.  (Products, systems and update each by itself, sums of two MFMAs added afterwards: 1000 vector instructions,
// 293 us in all; W and P read by every wave from memory: 276.)
bool delta_chunk_ok(const float* qkv, int P, int Tp, int H, int G, int d, int V) {
  return delta_rows_pay(P, Tp, H, V) && d == D && V >= 16 && ((int64_t)H * V) % 4 == 0 &&
         (reinterpret_cast<uintptr_t>(qkv) & 15) == 0 &&
         chunk_fits(2L * G * D + (long)H * V, (long)H * V, (long)H * ((V + 127) / 128 + 1));
}

DeltaWork delta_chunk_plan(int P, int Tp, int H, int G, int V) {
  DeltaWork w;
  w.items = P;
  const int chunks = Tp / L + P, wgs = H * ((V + 127) / 128);
  w.wp = (int64_t)chunks * H * 2 * MAT;
  w.floats = (int64_t)chunks * L * (3 * H + 2 * G);
  const int want = (device_cus() + wgs - 1) / wgs;      // items for one workgroup per CU
  if (P * 3 > want) return w;
  // One round of the third pass, whose segments have 8 chunks at least; where that leaves more than a round of the first
  // one (the identity's workgroups beside the values'), shorter ones that fill it.  us, 8 chunks -> so, 16 heads: 1 x 400 tokens
  // 76 (whole) -> 62, 500 90 (whole) -> 66, 700 117 (whole) -> 72, 1000 106 -> 86, 2 x 500 91 (whole) -> 78; 1 x 2000 in 13 segments instead
  // of 8 114 -> 126.
  int seg = segment_rows(P, Tp, want, L, 8);
  const int first = device_cus() / (wgs + H);
  if (first > 0) seg = std::min(seg, segment_rows(P, Tp, first + P, L, 3));
  if (Tp / P < 3 * seg) return w;
  w.seg = seg;
  w.items = Tp / seg + P;
  w.floats += (int64_t)w.items * H * D * (2 * (int64_t)V + D);
  return w;
}

void launch_delta_chunk(int dtype, float* out, const float* qkv, const void* ba, int64_t bas,
                        const float* a_log, const float* dt_bias, float* S, const int* qsl,
                        const int* seq_lens, const int* slots, int P, int Tp, int H, int G, int V,
                        int num_slots, const DeltaWork& work, void* wp, float* ws, hipStream_t s) {
  DeltaArgs a{};
  a.out = out; a.qkv = qkv; a.stride = 2 * (int64_t)G * D + (int64_t)H * V;
  a.ba = ba; a.bas = bas; a.ba_type = dtype;
  a.a_log = a_log; a.dt_bias = dt_bias; a.S = S;
  a.qsl = qsl; a.seq_lens = seq_lens; a.slots = slots;
  a.P = P; a.H = H; a.G = G; a.dv = V; a.num_slots = num_slots;
  a.wp = (bf16*)wp;
  const int64_t rows = (int64_t)(Tp / L + P) * L;
  a.kw = reinterpret_cast<f32x2*>(ws);
  a.gam = ws + 2 * rows * H;
  a.rk = a.gam + rows * H;
  a.rq = a.rk + rows * G;
  a.seg = work.seg;
  a.seg_state = a.rq + rows * G;
  a.seg_in = a.seg_state + (int64_t)work.items * H * D * (V + D);
  delta_prep_kernel<<<dim3(Tp / L + P, G), 64, 0, s>>>(a);
  const int nct = (V + 127) / 128;
  if (work.seg <= 0) {
    delta_walk_kernel<0><<<dim3(P, H * nct), NT, 0, s>>>(a);
  } else {
    delta_walk_kernel<1><<<dim3(work.items, H * (nct + 1)), NT, 0, s>>>(a);
    delta_chain_kernel<<<dim3(P, H, (V + 15) / 16), NT, 0, s>>>(a);
    delta_walk_kernel<2><<<dim3(work.items, H * nct), NT, 0, s>>>(a);
  }
}

}  // namespace kgc
