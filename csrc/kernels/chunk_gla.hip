// Chunkwise gated linear attention (Yang et al., 2023) of prompt rows on the matrix cores.  Per
// (sequence, head), with a decay alpha_t per key channel,
//     S_t = diag(alpha_t) S_(t-1) + k_t v_t^T,   o_t = S_t^T q_t .
// Over a chunk of L = 32 tokens, p_t the product of the chunk's decays up to t, r_s of those after s and
// S_0 the state before it (products channel by channel):
//     O   = (Q p) S_0 + A V,     A_ts = sum_c q_tc k_sc alpha_(s+1)c .. alpha_tc  (s <= t)
//     S_L = diag(p_L) S_0 + (K r)^T V
// Q p, K r, p_L and A depend on no state: a first launch computes them for all chunks at once, A by
// running products from every s upwards (no quotient of products, so no decay is too small).  The walk
// then has no serial step finer than a chunk: a workgroup of 8 waves owns 128 value columns of a head,
// a wave 16 of them with their S in accumulators.
//
// Precision: fp32 operands enter the bf16 MFMAs as three bf16 parts each, six products of parts, the
// corrections summed apart; products p and r are kept in double.
//
// Few long sequences are cut into segments: one walk makes every segment's contribution from a zero state, a
// small launch puts the states together in which the segments start, and the second walk has them all.
//
// Measured (8 heads, 256 value columns, rank 16): 32 x 512 tokens 259 us, 110 of them the first
// launch (its LDS let two workgroups share a CU, and scalar LDS reads and shuffles held those up: 250; 148 MB
// written) and 145 the walk (splitting S beside the MFMAs, operands a step ahead: 190 without, and reading those
// 148 MB); 2 x 8192 410 (one walk per sequence: 1562), 1 x 4000 127 (659); token by token 1340 and 8140.  From
// float64, relative norm: outputs 7.3e-7, states 1.04e-6.
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

// sum over eight neighbouring lanes, without the LDS
__device__ __forceinline__ float sum8(float x) {
  auto other = [](float y, auto ctrl) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, y), decltype(ctrl)::value, 0xf, 0xf, true));
  };
  x += other(x, std::integral_constant<int, 0xb1>());     // lanes 1 0 3 2
  x += other(x, std::integral_constant<int, 0x4e>());     // lanes 2 3 0 1
  return x + other(x, std::integral_constant<int, 0x141>());   // the eight in reverse
}

// q p, k r, p_L and A of every chunk: one workgroup per (chunk, head)
template <typename T>
__global__ __launch_bounds__(256) void gla_prep_kernel(const GlaArgs a) {
  // 49 KB, so that three workgroups share a CU: the bottleneck's rows lie where the decays come, A where k was
  __shared__ __align__(16) float qs[L][D], ks[L][D], al[L][D];
  __shared__ double half[D];
  static_assert(RMAX <= D && L + 4 <= D, "");
  float (&lw)[L][D] = al;
  float (*X)[L + 4] = reinterpret_cast<float (*)[L + 4]>(&ks[0][0]);
  const SegItem it = seg_item(blockIdx.x, a.qsl, a.P, L);
  if (it.seq < 0) return;
  const int h = blockIdx.y, tid = threadIdx.x;
  const int c0 = it.idx * L, len = a.qsl[it.seq + 1] - a.qsl[it.seq], nl = min(L, len - c0);
  const int slot = a.slots[it.seq];
  if (nl <= 0 || slot < 0 || slot >= a.num_slots || a.seq_lens[it.seq] < len) return;
  const int64_t t0 = a.qsl[it.seq] + c0, at = (int64_t)blockIdx.x * a.H + h;
  const T* proj = reinterpret_cast<const T*>(a.proj) + t0 * a.ps;
  const T* low = reinterpret_cast<const T*>(a.low) + t0 * a.ls;
  for (int e = tid; e < nl * a.R; e += 256) {
    const int t = e / a.R, j = e - t * a.R;
    lw[t][j] = to_f(low[t * a.ls + j]);
  }
  const float scale = 1.f / sqrtf((float)D);
  constexpr int V = 16 / sizeof(T);          // elements of 16 bytes
  if (a.ps % V == 0 && reinterpret_cast<uintptr_t>(a.proj) % 16 == 0) {
    typedef T TV __attribute__((ext_vector_type(V)));
    for (int e = tid * V; e < L * D; e += 256 * V) {
      const int t = e / D, c = e % D;
      const T* row = proj + min(t, nl - 1) * a.ps + h * D + c;
      const TV q = *reinterpret_cast<const TV*>(row), k = *reinterpret_cast<const TV*>(row + (int64_t)a.H * D);
#pragma unroll
      for (int i = 0; i < V; ++i) {
        qs[t][c + i] = t < nl ? to_f(q[i]) * scale : 0.f;
        ks[t][c + i] = t < nl ? to_f(k[i]) : 0.f;
      }
    }
  } else for (int e = tid; e < L * D; e += 256) {
    const int t = e / D, c = e % D;
    const T* row = proj + t * a.ps + h * D + c;
    qs[t][c] = t < nl ? to_f(row[0]) * scale : 0.f;
    ks[t][c] = t < nl ? to_f(row[(int64_t)a.H * D]) : 0.f;
  }
  __syncthreads();
  // thread (channel, half of the tokens): decays, their products up to and after each token
  const int c = tid % D, hf = tid / D, b = hf * (L / 2);
  {
    float acc[L / 2];
#pragma unroll
    for (int i = 0; i < L / 2; ++i) acc[i] = 0.f;
    const float* ar = a.a2 + ((int64_t)h * D + c) * a.R;
    int j = 0;
    if (a.R % 4 == 0)                        // four at a time: a quarter of the LDS reads
      for (; j < a.R; j += 4) {
        f32x4 w;
#pragma unroll
        for (int n = 0; n < 4; ++n) w[n] = ar[j + n];
#pragma unroll
        for (int i = 0; i < L / 2; ++i) {
          const f32x4 x = *reinterpret_cast<const f32x4*>(&lw[min(b + i, nl - 1)][j]);
#pragma unroll
          for (int n = 0; n < 4; ++n) acc[i] += w[n] * x[n];
        }
      }
    for (; j < a.R; ++j) {
      const float w = ar[j];
#pragma unroll
      for (int i = 0; i < L / 2; ++i) acc[i] += w * lw[min(b + i, nl - 1)][j];
    }
    const float bias = a.a2b[h * D + c];
    double p = 1.0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < L / 2; ++i) {
      const float x = acc[i] + bias;
      acc[i] = b + i < nl ? expf((fminf(x, 0.f) - log1pf(expf(-fabsf(x)))) * a.inv_tau) : 1.f;
      al[b + i][c] = acc[i];
      p *= acc[i];
    }
    if (hf == 0) half[c] = p;
    __syncthreads();
    const double first = half[c];            // the first half's product
    __syncthreads();
    if (hf == 1) half[c] = p;
    __syncthreads();
    const double second = half[c];
    float* qo = a.qp + at * L * D + c;
    float* ko = a.kr + at * L * D + c;
    p = hf ? first : 1.0;
#pragma unroll
    for (int i = 0; i < L / 2; ++i) {
      p *= acc[i];
      qo[(b + i) * D] = (float)(qs[b + i][c] * p);
    }
    double r = hf ? 1.0 : second;
#pragma unroll
    for (int i = L / 2 - 1; i >= 0; --i) {
      ko[(b + i) * D] = (float)(ks[b + i][c] * r);
      r *= acc[i];
    }
    if (hf == 0) a.pl[at * D + c] = (float)(first * second);
  }
  // A: thread (column s, channels 32 i + 4 g ..) carries k_s times the decays since s; eight threads read 128
  // bytes next to each other, and a wave begins at its first column
  {
    const int s = tid >> 3, g = (tid & 7) * 4;
    float w[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) w[i] = ks[s][(i >> 2) * 32 + g + (i & 3)];
    const int s0 = __builtin_amdgcn_readfirstlane(s & ~7);
    __syncthreads();
    for (int t = 0; t < s0; ++t)
      if ((tid & 7) == 0) X[t][s] = 0.f;
    for (int t = s0; t < L; ++t) {
      float a0 = 0.f, a1 = 0.f;
#pragma unroll
      for (int i = 0; i < 16; i += 4) {
        const f32x4 d = *reinterpret_cast<const f32x4*>(&al[t][i * 8 + g]);
        const f32x4 q = *reinterpret_cast<const f32x4*>(&qs[t][i * 8 + g]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          w[i + e] = t > s ? w[i + e] * d[e] : w[i + e];
          (e & 1 ? a1 : a0) += w[i + e] * q[e];
        }
      }
      const float x = sum8(a0 + a1);
      if ((tid & 7) == 0) X[t][s] = t >= s ? x : 0.f;
    }
  }
  __syncthreads();
  if (tid < L * 4) {                         // eight (permuted) columns per store
    const int t = tid >> 2, oct = tid & 3;
    const f32x4 x0 = *reinterpret_cast<const f32x4*>(&X[t][oct * 4]);
    const f32x4 x1 = *reinterpret_cast<const f32x4*>(&X[t][oct * 4 + 16]);
    const float x[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
    bf16x8 p[3];
    split8<3>(x, p);
#pragma unroll
    for (int i = 0; i < 3; ++i)
      *reinterpret_cast<bf16x8*>(a.am + at * MAT + i * L * L + t * L + oct * 8) = p[i];
  }
}

// MODE 0: whole sequences; 1: segments from zero (states only); 2: segments from the states that they start in
template <typename T, int MODE>
__global__ __launch_bounds__(NT) void gla_walk_kernel(const GlaArgs a) {
  __shared__ __align__(16) bf16 Qs[MODE == 1 ? 8 : 3 * L * DP], KT[3 * D * LP];
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
  f32x4 S[DT];
  float* Ss = a.S + ((int64_t)slot * a.H + h) * D * a.dv;
  float* mine = a.seg_state + ((int64_t)item * a.H + h) * D * a.dv;
  const bool own = MODE == 2 && seg_count > 1, zero = MODE == 1 || (pos0 == 0 && !own);
  const float* from = own ? mine : Ss;
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[i][r] = zero ? 0.f : from[(i * 16 + 4 * lg + r) * a.dv + colc];
  const T* vb = reinterpret_cast<const T*>(a.proj) + 2 * (int64_t)a.H * D + (int64_t)h * a.dv + colc;
  // Staging: a thread takes 8 columns of one row of q p, and 8 tokens of one column of k r, in both
  // cases the pieces 4 i .. and 16 + 4 i .. of 32: adjacent in the permuted order, one store.
  f32x4 rq[2], rt[2];
  const int ut = tid / 16, uc = (tid % 16 / 4) * 32 + (tid % 4) * 4, up_ = (tid % 16) * 8;
  const int ta = tid / D * 4, tc = tid % D;
  const int chunk0 = chunks_before<L>(seq, a.qsl) + (MODE != 0 ? seg_idx * (a.seg / L) : 0);
  auto fetch = [&](int ci) {
    const int64_t at = ((int64_t)ci * a.H + h) * L * D;
    if (MODE != 1) {
      rq[0] = *reinterpret_cast<const f32x4*>(a.qp + at + ut * D + uc);
      rq[1] = *reinterpret_cast<const f32x4*>(a.qp + at + ut * D + uc + 16);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) rt[i >> 2][i & 3] = a.kr[at + (ta + (i >> 2) * 16 + (i & 3)) * D + tc];
  };
  auto park = [&]() {
    float x[8];
    bf16x8 p[3];
    if (MODE != 1) {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = rq[i >> 2][i & 3];
      split8<3>(x, p);
#pragma unroll
      for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8*>(Qs + i * L * DP + ut * DP + up_) = p[i];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = rt[i >> 2][i & 3];
    split8<3>(x, p);
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8*>(KT + (i * D + tc) * LP + ta * 2) = p[i];
  };
  fetch(chunk0);
  for (int c0 = 0, ci = chunk0; c0 < len; c0 += L, ++ci) {
    const int nl = min(L, len - c0);
    park();
    __syncthreads();
    const int64_t t0 = start + c0, at = (int64_t)ci * a.H + h;
    // this lane's v (tokens 4 lg + r of each tile), its fragments of A, the channels' decays
    T v[LT][4];
#pragma unroll
    for (int ti = 0; ti < LT; ++ti)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[ti][r] = vb[(t0 + min(ti * 16 + lg * 4 + r, nl - 1)) * a.ps];
    bf16x8 fp[LT][3];
    if (MODE != 1)
#pragma unroll
    for (int ti = 0; ti < LT; ++ti)
#pragma unroll
      for (int i = 0; i < 3; ++i)
        fp[ti][i] = *reinterpret_cast<const bf16x8*>(a.am + at * MAT + i * L * L + (ti * 16 + lr) * L + lg * 8);
    f32x4 o[LT], ol[LT];
    bf16x8 fa[2][2][3];                      // two row tiles, a step ahead
    if (MODE != 1) {
#pragma unroll
      for (int ti = 0; ti < LT; ++ti) o[ti] = ol[ti] = f32x4{0.f, 0.f, 0.f, 0.f};
      bf16x8 sp[2][3];                       // parts of 32 rows of S, likewise
      auto load_q = [&](int j) {
#pragma unroll
        for (int ti = 0; ti < LT; ++ti)
#pragma unroll
          for (int i = 0; i < 3; ++i)
            fa[j & 1][ti][i] = *reinterpret_cast<const bf16x8*>(Qs + i * L * DP + (ti * 16 + lr) * DP + j * 32 + lg * 8);
      };
      auto split_s = [&](int j) {
        float x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = S[2 * j + (i >> 2)][i & 3];
        split8<3>(x, sp[j & 1]);
      };
      load_q(0);
      split_s(0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < KD; ++j) {
        if (j + 1 < KD) {
          load_q(j + 1);
          split_s(j + 1);
        }
        f32x4 main[LT];                      // (rounded into its sum once per step)
#pragma unroll
        for (int ti = 0; ti < LT; ++ti) main[ti] = f32x4{0.f, 0.f, 0.f, 0.f};
        mm3_add(fa[j & 1], sp[j & 1], main, ol);
#pragma unroll
        for (int ti = 0; ti < LT; ++ti) o[ti] += main[ti];
        __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
        interleave<12, 4>();
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    fetch(c0 + L < len ? ci + 1 : ci);       // (the last one again at the end: no branch)
    bf16x8 vp[3];
    int bad;
    {
      float x[8];
      auto tok = [&](int i) { return (i >> 2) * 16 + lg * 4 + (i & 3); };
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = tok(i) < nl ? to_f(v[i >> 2][i & 3]) : 0.f;
      bad = take_nonfinite(x, L, tok);
      split8<3>(x, vp);
    }
    const bool some_bad = __any(bad < L);
    float* oc = a.out + t0 * os + (int64_t)h * a.dv + col;
    if (MODE != 1)
#pragma unroll
    for (int ti = 0; ti < LT; ++ti) {
      f32x4 hi = {0.f, 0.f, 0.f, 0.f}, lo = hi;
      mm<true, 3, 3>(fp[ti], vp, hi, lo);
      if (some_bad)
#pragma unroll
        for (int e = 0; e < 4; ++e) hi[e] = ti * 16 + lg * 4 + e >= bad ? NAN : hi[e];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int t = ti * 16 + lg * 4 + e;
        if (colok && t < nl) oc[t * os] = (o[ti][e] + hi[e]) + (ol[ti][e] + lo[e]);
      }
    }
    f32x4 u[2][2], lo[2][2], pl[2][2];       // products of two row tiles, their corrections and decays
    auto load_k = [&](int q) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int i = 0; i < 3; ++i)
          fa[q & 1][t][i] = *reinterpret_cast<const bf16x8*>(KT + (i * D + (2 * q + t) * 16 + lr) * LP + lg * 8);
        pl[q & 1][t] = *reinterpret_cast<const f32x4*>(a.pl + at * D + (2 * q + t) * 16 + 4 * lg);
      }
    };
    auto add = [&](int q) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[2 * q + t][e] = __builtin_fmaf(S[2 * q + t][e], pl[q & 1][t][e], u[q & 1][t][e] + lo[q & 1][t][e]);
    };
    load_k(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < DT / 2; ++q) {
#pragma unroll
      for (int t = 0; t < 2; ++t) u[q & 1][t] = lo[q & 1][t] = f32x4{0.f, 0.f, 0.f, 0.f};
      mm3_add(fa[q & 1], vp, u[q & 1], lo[q & 1]);
      if (q > 0) add(q - 1);
      if (q + 1 < DT / 2) load_k(q + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    add(DT / 2 - 1);
    if (some_bad)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int e = 0; e < 4; ++e) S[dt][e] = bad < L ? NAN : S[dt][e];
    __syncthreads();
  }
  float* dst = MODE == 1 ? mine : Ss;
  if (colok && (MODE != 2 || seg_idx + 1 == seg_count))
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) dst[(i * 16 + 4 * lg + r) * a.dv + col] = S[i][r];
}

// ---- the states in which segments start, in place of the contributions: one element per thread ------------
__global__ __launch_bounds__(256) void gla_chain_kernel(const GlaArgs a) {
  const int seq = blockIdx.z, h = blockIdx.y, lane = threadIdx.x & 63;
  const int len = a.qsl[seq + 1] - a.qsl[seq], pos0 = a.seq_lens[seq] - len, slot = a.slots[seq];
  if (len <= a.seg || slot < 0 || slot >= a.num_slots || pos0 < 0) return;
  const int first = pieces_before(seq, a.qsl, a.seg);
  const int count = (len + a.seg - 1) / a.seg, per = a.seg / L, sh = D * a.dv;
  const int chunk0 = chunks_before<L>(seq, a.qsl);
  const int at = blockIdx.x * 256 + threadIdx.x;
  if (at >= sh) return;
  const int64_t step = (int64_t)a.H * sh;
  const float* pl = a.pl + ((int64_t)chunk0 * a.H + h) * D + at / a.dv;
  float* p = a.seg_state + ((int64_t)first * a.H + h) * sh + at;
  float S = pos0 == 0 ? 0.f : a.S[((int64_t)slot * a.H + h) * sh + at];
  for (int j = 0; j < count - 1; ++j) {
    const float c = p[j * step];
    double f = 1.0;                          // the segment's decay
#pragma unroll 8
    for (int k = 0; k < per; ++k) f *= pl[(int64_t)(j * per + k) * a.H * D];
    p[j * step] = S;
    S = __builtin_fmaf((float)f, S, c);
  }
  p[(count - 1) * step] = S;
}

template <typename T>
void run(const GlaArgs& a, int chunks, hipStream_t s) {
  gla_prep_kernel<T><<<dim3(chunks, a.H), 256, 0, s>>>(a);
  const int y = a.H * ((a.dv + 127) / 128);
  if (a.seg <= 0) {
    gla_walk_kernel<T, 0><<<dim3(a.P, y), NT, 0, s>>>(a);
  } else {
    gla_walk_kernel<T, 1><<<dim3(a.items, y), NT, 0, s>>>(a);
    gla_chain_kernel<<<dim3((D * a.dv + 255) / 256, a.H, a.P), 256, 0, s>>>(a);
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
  // 1 x 48 tokens 46 -> 35 us, 64 x 48 218 -> 120, 4 x 60 63 -> 42; fewer rows: chunk_rows.h
  return chunk_rows_pay(P, Tp, 32) && d == D && V >= 16 && R <= RMAX &&
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
