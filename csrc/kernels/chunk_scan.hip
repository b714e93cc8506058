// Chunkwise matrix-state recurrences of prompt rows on the matrix cores: the mLSTM (Beck et al., xLSTM, 2024)
// and the Mamba-2 (SSD) scan (Dao and Gu, 2024).  Both carry S [d, dv] per (sequence, head) and, with a log
// decay f_t and a log input weight i_t per token (SSD: i_t = ln of the step size),
//     S_t = e^(f_t) S_(t-1) + e^(i_t) k_t v_t^T,      o_t = S_t^T q_t .
// Over a chunk of L tokens with b_t the running sum of f and S_0 the state before it:
//     o_t = e^(b_t) S_0^T q_t + sum_(s <= t) e^(b_t - b_s + i_s) (q_t . k_s) v_s
//     S_L = e^(b_L) S_0      + sum_s        e^(b_L - b_s + i_s) k_s v_s^T
// (the mLSTM divides every weight by its running maximum e^(m_t), which is a maximum of
// i_s - b_s over s <= t, so all exponents are <= 0; running sums are kept in double, so the
// difference of two of them has no rounding of its own worth naming).
//
// A workgroup of 8 waves owns 128 value columns of one head (or 64 of each of two heads that
// share q and k) and walks the chunks of its sequence; a wave owns 16 columns, and its S stays in
// MFMA accumulators for the whole walk.  Per chunk q, k and k^T are staged in LDS (the next
// chunk's loads in flight), the masked and weighted score matrix is computed once per workgroup,
// and then every wave works on its own columns alone:
//     O = Q S_0 (rows scaled) + P V,     S = e^(b_L) S_0 + K^T (w V).
// An accumulator of S is the B operand of Q S_0 as it lies: the k index of an MFMA may be
// permuted as long as both operands agree, so q and k are stored with their columns permuted.
//
// Precision: everything the token-serial scan held in fp32 still carries 24 bits.  An fp32
// operand enters the bf16 MFMAs as up to three bf16 parts (value, remainder, remainder), the
// products of parts whose weight is at least 2^-16 are kept, and the sums are fp32.  bf16
// inputs are one exact part, f16 inputs two.
//
// Most bf16 rows of the mLSTM and SSD heads that share B and C have kernels of their own (chunk_mlstm.hip, chunk_ssd.hip).
//
// What bounds it (mLSTM, 4 heads with 256 x 512 states, 64-token chunks): a wave issues 1550 vector
// instructions per chunk, most of them splitting S, and 222 MFMAs; they fill 42 % and 24 % of a SIMD's
// cycles (SSD's second walk: 59 % and 26 %).  The rest is barriers and latency that two waves per SIMD do not
// cover; LDS (140 KB) allows no third.
//
// Few long sequences: the walk is serial, so a step of few workgroups is cut into segments.  A
// first launch computes every segment's contribution from a zero state, the second starts each
// segment from the sum of its predecessors' decayed contributions.  The second launch writes the slots,
// so it takes the states they held from copies (as n and m): the first launch's workgroups of a
// sequence's last segment, whose contribution nobody needs, put S in that segment's place.
#include "chunk.h"
#include "chunk_rows.h"
#include "device.h"
#include "launch.h"

namespace kgc {

namespace {

constexpr int NT = 512, NW = NT / 64;

template <typename E> struct PartsOf { static constexpr int n = 1; };
template <> struct PartsOf<f16> { static constexpr int n = 2; };
template <> struct PartsOf<float> { static constexpr int n = 3; };

// 8 consecutive elements as they lie in memory
template <typename E> struct Raw8 {
  u32x4 u;
  __device__ __forceinline__ void load(const E* p) { u = *reinterpret_cast<const u32x4*>(p); }
  __device__ __forceinline__ void zero() { u = u32x4{0, 0, 0, 0}; }
  __device__ __forceinline__ float get(int i) const {
    Pack8<E> k;
    k.u = u;
    return (float)k.h[i];
  }
};
template <> struct Raw8<float> {
  f32x4 a, b;
  __device__ __forceinline__ void load(const float* p) {
    a = *reinterpret_cast<const f32x4*>(p);
    b = *reinterpret_cast<const f32x4*>(p + 4);
  }
  __device__ __forceinline__ void zero() { a = b = f32x4{0.f, 0.f, 0.f, 0.f}; }
  __device__ __forceinline__ float get(int i) const { return i < 4 ? a[i] : b[i - 4]; }
};

struct ChunkArgs {
  float* out;                       // [T, H dv]
  const void *q, *k, *v;            // element (row, group / head, column) at row * stride + h * d + c
  int64_t stride;                   // elements, of all three
  const float* gates;               // mLSTM: [T, 2 H] log input | log forget gate
  const void* dt;                   // SSD: [T, H] step sizes before softplus, of type dt_type
  int64_t dts;
  int dt_type;
  const float *a_log, *dt_bias, *dskip;
  float *S, *n, *m;
  const float *n0, *m0;             // mLSTM: copies of n and m of the step's sequences
  const int *qsl, *seq_lens, *slots;
  int P, H, hpg, dv, num_slots;  // hpg: heads per q / k group
  int seg;                          // tokens per segment, a multiple of the chunk (0: not cut)
  // [items][H][d (dv + 1)]: S, n of a segment from zero; a cut sequence's last: S as the slot held it
  float* seg_state;
  double* seg_gate;                 // [items][H][2]: its log decay, its m
};

// E: element type of q, k, v; MLSTM or SSD; D: padded rows of S; L: chunk;
// HPW: heads per workgroup.  MODE 0: whole sequences, 1: segments from zero (states only),
// 2: segments from their predecessors' states.
template <typename E, bool MLSTM, int D, int L, int HPW, int MODE>
__global__ __launch_bounds__(NT) void chunk_scan_kernel(const ChunkArgs a) {
  constexpr int NP = PartsOf<E>::n;
  constexpr bool SEP = NP > 1;
  constexpr int DP = D + 8, LP = L + 8;      // padded LDS rows: 16-byte reads without bank conflicts
  constexpr int WPH = NW / HPW;              // waves (column tiles) per head
  constexpr int DT = D / 16, LT = L / 16, KD = D / 32, KL = L / 32;
  constexpr int NTILE = LT * (LT + 1) / 2;   // score tiles on and under the diagonal
  constexpr int NU = (L * D / 8 + NT - 1) / NT;                    // staged q (k) units per thread
  constexpr int TW = sizeof(E) == 2 ? 2 : 1;                       // columns per k^T unit
  constexpr int NUT = (L / 8 * D / TW + NT - 1) / NT;
  extern __shared__ __align__(16) char smem[];
  bf16* Qs = reinterpret_cast<bf16*>(smem);            // [NP][L][DP], columns permuted
  bf16* Ks = Qs + NP * L * DP;                         // [NP][L][DP], likewise
  bf16* KT = Ks + NP * L * DP;                         // [NP][D][LP]
  bf16* Ps = KT + NP * D * LP;                         // [HPW][3][L][LP]
  // per chunk, two of each: the gates run one chunk ahead
  double* rt = reinterpret_cast<double*>(Ps + HPW * 3 * L * LP);   // [2][HPW][L]
  double* cs = rt + 2 * HPW * L;                       // [2][HPW][L]
  float* inter = reinterpret_cast<float*>(cs + 2 * HPW * L);  // [2][HPW][L]: factor of a row of Q S_0
  float* wt = inter + 2 * HPW * L;                     // [2][HPW][L]: weight of a token in the update
  float* pw = wt + 2 * HPW * L;                        // [2][HPW][L]: weight of a score column
  float* sa = pw + 2 * HPW * L;                        // [2][HPW <= 2]: decay of S over the chunk
  float* em = sa + 4;                                  // mLSTM: [2][L] e^(-m_t)
  float* nq = em + 2 * L;                              //        [L] n_0 . q_t
  float* psum = nq + L;                                //        [LT][L] row sums of P by column tile
  float* ns = psum + LT * L;                           //        [D] n, in the permuted order
  float* rd = ns + D;                                  //        [NW][L] 1 / denominator

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int lr = lane & 15, lg = lane >> 4;
  int seq = blockIdx.x, seg_idx = 0, seg_first = 0, seg_count = 1;
  if (MODE != 0) {
    const SegItem it = seg_item(blockIdx.x, a.qsl, a.P, a.seg);
    if (it.seq < 0) return;
    seq = it.seq;
    seg_idx = it.idx;
    seg_first = it.first;
    seg_count = it.count;
  }
  const bool last_seg = MODE != 0 && seg_idx + 1 == seg_count;
  const int nct = (a.dv + 16 * WPH - 1) / (16 * WPH);
  const int hb = blockIdx.y / nct, ct = blockIdx.y - hb * nct;
  const int h0 = hb * HPW, hw = wave / WPH, h = h0 + hw, grp = h0 / a.hpg;
  const int col = (ct * WPH + (wave - hw * WPH)) * 16 + lr;
  const bool colok = col < a.dv;
  const int colc = colok ? col : a.dv - 1;   // rows and columns off the edge: read the last, use 0
  int start = a.qsl[seq], len = a.qsl[seq + 1] - start;
  const int pos0 = a.seq_lens[seq] - len;
  const int slot = a.slots[seq];
  const int64_t os = (int64_t)a.H * a.dv;
  if (MODE != 0) {
    start += seg_idx * a.seg;
    len = min(a.seg, len - seg_idx * a.seg);
  }
  if (len <= 0) return;
  if (slot < 0 || slot >= a.num_slots || pos0 < 0) {             // padding: defined zeros
    if (MODE != 1 && colok)
      for (int t = lg; t < len; t += 4) a.out[(start + t) * os + (int64_t)h * a.dv + col] = 0.f;
    return;
  }
  const bool fresh = pos0 == 0;
  if (MODE == 1 && last_seg && (fresh || seg_count == 1)) return;

  // ---- the state this walk starts from --------------------------------------------------
  const int64_t sh = (int64_t)D * a.dv, item_floats = sh + (MLSTM ? D : 0);
  float* Ss = a.S + ((int64_t)slot * a.H + h) * sh;
  float* copy = a.seg_state + ((int64_t)(seg_first + seg_count - 1) * a.H + h) * item_floats;
  const float* from = MODE == 2 && seg_count > 1 ? copy : Ss;
  f32x4 S[DT];
  double m0 = 0.0;                           // mLSTM: running maximum (kept by the gates' wave)
  const bool zero = (MODE == 1 && !last_seg) || fresh;
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = i * 16 + 4 * lg + r;
      S[i][r] = zero ? 0.f : from[row * a.dv + colc];
    }
  if (MODE == 1 && last_seg) {
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (colok) copy[(i * 16 + 4 * lg + r) * a.dv + col] = S[i][r];
    return;
  }
  if (MLSTM) {
    if (MODE == 1) m0 = -INFINITY;
    else if (!fresh) m0 = a.m0[(int64_t)seq * a.H + h];
  }
  float nreg = 0.f;                          // mLSTM: n[tid] for tid < D
  if (MLSTM && tid < D && !zero) nreg = a.n0[((int64_t)seq * a.H + h) * D + tid];
  if (MODE == 2) {
    // predecessors in order: S <- e^(b + m - m') S + e^(m_j - m') S_j, n likewise (SSD: m = 0)
    for (int j = 0; j < seg_idx; ++j) {
      const int64_t it = (int64_t)(seg_first + j) * a.H + h;
      const double b = a.seg_gate[2 * it], mj = a.seg_gate[2 * it + 1];
      const float* sp = a.seg_state + it * item_floats;
      float f, g = 1.f;
      int vj = a.dv;                          // opaque: see below
      asm volatile("" : "+s"(vj));
      if (MLSTM) {
        const double mn = fmax(b + m0, mj);
        f = exp_d(b + m0 - mn);
        g = exp_d(mj - mn);
        m0 = mn;
      } else {
        f = exp_d(b);
      }
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = i * 16 + 4 * lg + r;
          S[i][r] = f * S[i][r] + g * sp[row * vj + colc];
        }
      if (MLSTM && tid < D) nreg = f * nreg + g * sp[sh + tid];
    }
  }
  if (MLSTM && tid < D) ns[mfma_perm(tid)] = nreg;
  for (int i = tid; i < HPW * 3 * L * LP / 8; i += NT)           // tiles above the diagonal stay zero
    reinterpret_cast<u32x4*>(Ps)[i] = u32x4{0, 0, 0, 0};

  const E* qb = reinterpret_cast<const E*>(a.q) + (int64_t)grp * D;
  const E* kb = reinterpret_cast<const E*>(a.k) + (int64_t)grp * D;
  const E* vb = reinterpret_cast<const E*>(a.v) + (int64_t)h * a.dv + colc;
  const float skip = MLSTM ? 0.f : a.dskip[h];
  const float qscale = MLSTM ? 1.f / sqrtf((float)D) : 1.f;
  Raw8<E> rq[NU], rk[NU];
  uint32_t rkt[NUT][8];
  float gi = 0.f, gf = 0.f;
  double btot = 0.0;                         // log decay of the walk so far (likewise)

  // global -> registers for the chunk at token c0.  Rows past the end and columns past d read the
  // last one and become zero when they are stored or used: a test here would wait for the load.
  // Row offsets inside a chunk fit 32 bits; made opaque once per chunk, so that the offsets of all
  // staged rows are computed again and not kept in registers across the walk.
  int rs = (int)a.stride, ro = (int)os;
  auto fetch = [&](int c0) {
    const int nl = min(L, len - c0);
    const E* qc = qb + (int64_t)(start + c0) * a.stride;
    const E* kc = kb + (int64_t)(start + c0) * a.stride;
#pragma unroll
    for (int j = 0; j < NU; ++j) {
      const int u = tid + NT * j, t = u / (D / 8), c = (u % (D / 8)) * 8;
      if (MODE != 1) {
        const int at = min(t, nl - 1) * rs + c;
        rq[j].load(qc + at);
        rk[j].load(kc + at);
      }
    }
#pragma unroll
    for (int j = 0; j < NUT; ++j) {
      const int u = tid + NT * j, tg = u / (D / TW), c = (u % (D / TW)) * TW;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int t = tg * 8 + i;
        rkt[j][i] = *reinterpret_cast<const uint32_t*>(kc + min(t, nl - 1) * rs + c);
      }
    }
  };
  // The gates of the chunk at c0, one token per lane, and their running sums (and maxima): wave
  // NW - 1 - hh does them for head hh one chunk ahead, while the scores keep the others busy.
  const int hg = NW - 1 - wave;              // < HPW: the head of this wave's gates
  const double dt_bias = MLSTM || hg >= HPW ? 0.0 : a.dt_bias[h0 + hg];
  const double exp_a = MLSTM || hg >= HPW ? 0.0 : exp((double)a.a_log[h0 + hg]);
  auto fetch_gates = [&](int c0) {
    const int64_t t = start + c0 + min(lane, min(L, len - c0) - 1);
    if (MLSTM) {
      gi = a.gates[t * 2 * a.H + h0 + hg];
      gf = a.gates[t * 2 * a.H + a.H + h0 + hg];
    } else {
      const int64_t at = t * a.dts + h0 + hg;
      gi = a.dt_type == DT_F32 ? reinterpret_cast<const float*>(a.dt)[at]
           : a.dt_type == DT_F16 ? (float)reinterpret_cast<const f16*>(a.dt)[at]
                                 : (float)reinterpret_cast<const bf16*>(a.dt)[at];
    }
  };
  // registers -> LDS
  auto park = [&](int nl) {
    if (MODE != 1) {
#pragma unroll
      for (int j = 0; j < NU; ++j) {
        const int u = tid + NT * j, t = u / (D / 8), c = (u % (D / 8)) * 8;
        if (L * D / 8 % NT != 0 && t >= L) continue;
        if (nl < L && t >= nl) {
          rq[j].zero();
          rk[j].zero();
        }
        const int at0 = t * DP + mfma_perm(c), at1 = t * DP + mfma_perm(c + 4);
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          const Raw8<E>& x = w ? rk[j] : rq[j];
          bf16* base = w ? Ks : Qs;
          union { bf16x8 v; u32x2 h[2]; } o[NP];
          if constexpr (NP == 1) {
            o[0].v = __builtin_bit_cast(bf16x8, x.u);
          } else {
            float f[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) f[i] = x.get(i);
            bf16x8 p[NP];
            split8<NP>(f, p);
#pragma unroll
            for (int i = 0; i < NP; ++i) o[i].v = p[i];
          }
#pragma unroll
          for (int i = 0; i < NP; ++i) {
            *reinterpret_cast<u32x2*>(base + i * L * DP + at0) = o[i].h[0];
            *reinterpret_cast<u32x2*>(base + i * L * DP + at1) = o[i].h[1];
          }
        }
      }
    }
#pragma unroll
    for (int j = 0; j < NUT; ++j) {
      const int u = tid + NT * j, tg = u / (D / TW), c = (u % (D / TW)) * TW;
      if (L / 8 * D / TW % NT != 0 && tg >= L / 8) continue;
      if (nl < L)
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (tg * 8 + i >= nl) rkt[j][i] = 0;
#pragma unroll
      for (int w = 0; w < TW; ++w) {
        bf16x8 p[NP];
        if constexpr (NP == 1) {             // two columns of eight rows: byte permutes
          u32x4 o;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            o[i] = __builtin_amdgcn_perm(rkt[j][2 * i + 1], rkt[j][2 * i], w ? 0x07060302 : 0x05040100);
          p[0] = __builtin_bit_cast(bf16x8, o);
        } else {
          float f[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            if constexpr (sizeof(E) == 2)
              f[i] = (float)__builtin_bit_cast(E, (uint16_t)(rkt[j][i] >> (16 * w)));
            else
              f[i] = __builtin_bit_cast(float, rkt[j][i]);
          }
          split8<NP>(f, p);
        }
#pragma unroll
        for (int i = 0; i < NP; ++i)
          *reinterpret_cast<bf16x8*>(KT + i * D * LP + (c + w) * LP + tg * 8) = p[i];
      }
    }
  };
  auto scan_gates = [&](int nl, int buf) {
    const bool ok = lane < nl;
    // a decay of e^-1e6 is zero; a finite floor keeps the differences of running sums defined
    double f = gf;
    if (!MLSTM) {                            // step size and log decay, in double: two of a wave's
      const double z = (double)gi + dt_bias; // sixteen heads per token, and nobody waits for them
      const double size = z > 40.0 ? z : log1p(exp(z));
      gi = (float)size;
      f = -exp_a * size;
    }
    if (!ok) f = gi = 0.f;
    const double b = wave_scan<false>(f < -1e6 ? -1e6 : f);
    const double bL = lane63(b);
    const int at = (buf * HPW + hg) * L + lane;
    if (MLSTM) {
      const double c = ok ? (gi < -1e6f ? -1e6 : (double)gi) - b : -INFINITY;
      const double M = fmax(m0, wave_scan<true>(c)), ML = lane63(M);
      if (lane < L) {
        rt[at] = -M;
        cs[at] = c;
        pw[at] = qscale;
        inter[at] = exp_d(m0 - M) * qscale;
        wt[at] = exp_d(c - ML);
        em[buf * L + lane] = expf((float)-(b + M));
      }
      if (lane == 0) sa[buf * HPW + hg] = exp_d(m0 - ML);
      m0 = bL + ML;
    } else {
      if (lane < L) {
        rt[at] = b;
        cs[at] = -b;
        pw[at] = gi;
        inter[at] = exp_d(b);
        wt[at] = exp_d(bL - b) * gi;
      }
      if (lane == 0) sa[buf * HPW + hg] = exp_d(bL);
    }
    btot += bL;
  };

  fetch(0);
  if (hg < HPW) {
    fetch_gates(0);
    scan_gates(min(L, len), 0);
    if (L < len) fetch_gates(L);
  }
  int buf = 0;
  for (int c0 = 0; c0 < len; c0 += L, buf ^= 1) {
    const int nl = min(L, len - c0);
    const double *rtc = rt + buf * HPW * L, *csc = cs + buf * HPW * L;
    const float *ic = inter + buf * HPW * L, *wc = wt + buf * HPW * L, *pc = pw + buf * HPW * L;
    asm volatile("" : "+s"(rs), "+s"(ro));
    park(nl);
    __syncthreads();
    // this chunk's v (B operand: rows 8 lg .. of every 32, the lane's column), in flight while the
    // scores and Q S_0 are computed
    const E* vc = vb + (int64_t)(start + c0) * a.stride;
    E vr[KL * 8];
#pragma unroll
    for (int j = 0; j < KL; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int s = j * 32 + lg * 8 + i;
        vr[j * 8 + i] = vc[min(s, nl - 1) * rs];
      }
    float xr[LT][4];                         // SSD: x of this lane's outputs, for D x
    if (!MLSTM && MODE != 1)
#pragma unroll
      for (int ti = 0; ti < LT; ++ti)
#pragma unroll
        for (int r = 0; r < 4; ++r) xr[ti][r] = (float)vc[min(ti * 16 + lg * 4 + r, nl - 1) * rs];
    if (hg < HPW && c0 + L < len) {
      scan_gates(min(L, len - c0 - L), buf ^ 1);
      if (c0 + 2 * L < len) fetch_gates(c0 + 2 * L);
    }

    if (MODE != 1) {
      // ---- scores: tile (ti, si) as D[s][t], weighted, split, stored as rows of P ----------
      for (int tile = wave; tile < NTILE; tile += NW) {
        int ti = 0;
        while ((ti + 1) * (ti + 2) / 2 <= tile) ++ti;
        const int si = tile - ti * (ti + 1) / 2;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f}, low = acc;
#pragma unroll
        for (int ks = 0; ks < KD; ++ks) {
          bf16x8 fa[NP], fb[NP];
#pragma unroll
          for (int i = 0; i < NP; ++i) {
            fa[i] = *reinterpret_cast<const bf16x8*>(Ks + i * L * DP + (si * 16 + lr) * DP + ks * 32 + lg * 8);
            fb[i] = *reinterpret_cast<const bf16x8*>(Qs + i * L * DP + (ti * 16 + lr) * DP + ks * 32 + lg * 8);
          }
          mm<SEP, NP, NP>(fa, fb, acc, low);
          if (ks % 2 == 1) __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (SEP) acc += low;
        const int t = ti * 16 + lr, s0 = si * 16 + lg * 4;
#pragma unroll
        for (int hh = 0; hh < HPW; ++hh) {
          const double r0 = rtc[hh * L + t];
          float p[4], sum = 0.f;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int s = s0 + r;
            p[r] = s <= t ? acc[r] * (exp_d(r0 + csc[hh * L + s]) * pc[hh * L + s]) : 0.f;
            sum += p[r];
          }
          if (MLSTM) {
            sum += __shfl_xor(sum, 16, 64);
            sum += __shfl_xor(sum, 32, 64);
            if (lg == 0) psum[si * L + t] = sum;
          }
          bf16* row = Ps + (hh * 3 * L + t) * LP + s0;
          uint32_t lo2[3], hi2[3];
          split2<3>(p[0], p[1], lo2);
          split2<3>(p[2], p[3], hi2);
#pragma unroll
          for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x2*>(row + i * L * LP) = u32x2{lo2[i], hi2[i]};
        }
      }
      if (MLSTM) {                           // n_0 . q_t: NT / L threads per row
        constexpr int TPR = NT / L;
        const int t = tid / TPR, sub = tid % TPR;
        float x = 0.f;
#pragma unroll
        for (int c = sub * 8; c < D; c += TPR * 8)
#pragma unroll
          for (int i = 0; i < NP; ++i) {
            const bf16x8 f = *reinterpret_cast<const bf16x8*>(Qs + i * L * DP + t * DP + c);
#pragma unroll
            for (int e = 0; e < 8; ++e) x += (float)f[e] * ns[c + e];
          }
#pragma unroll
        for (int o = 1; o < TPR; o <<= 1) x += __shfl_xor(x, o, 64);
        if (sub == 0) nq[t] = x;
      }
    }
    f32x4 o[LT], ol[LT];
    if (MODE != 1) {                         // Q S_0 of this wave's columns
#pragma unroll
      for (int i = 0; i < LT; ++i) o[i] = ol[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KD; ++ks) {
        float x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = S[2 * ks + (i >> 2)][i & 3];
        bf16x8 sp[3];
        split8<3>(x, sp);
#pragma unroll
        for (int ti = 0; ti < LT; ++ti) {
          bf16x8 fa[NP];
#pragma unroll
          for (int i = 0; i < NP; ++i)
            fa[i] = *reinterpret_cast<const bf16x8*>(Qs + i * L * DP + (ti * 16 + lr) * DP + ks * 32 + lg * 8);
          mm<SEP, NP, 3>(fa, sp, o[ti], ol[ti]);
        }
        __builtin_amdgcn_sched_barrier(0);   // bounds the operands in flight: registers
      }
    }
    __syncthreads();

    // ---- the rest of this wave's columns --------------------------------------------------
    __builtin_amdgcn_s_waitcnt(0x0f70);      // vmcnt(0): v is here; what follows need not be
    if (MODE == 1 && c0 + L < len) fetch(c0 + L);
    if (nl < L)
#pragma unroll
      for (int j = 0; j < KL; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (j * 32 + lg * 8 + i >= nl) vr[j * 8 + i] = (E)0.f;
    const int bad = take_nonfinite(vr, L, [&](int i) { return (i >> 3) * 32 + lg * 8 + (i & 7); });
    const bool some_bad = __any(bad < L);
    if (MODE != 1 && c0 + L < len) fetch(c0 + L);      // lands while P V and the update run
    if (MODE != 1) {
      if (MLSTM && lane < L) {
        float dsum = nq[lane] * ic[lane];
#pragma unroll
        for (int si = 0; si < LT; ++si)
          if (si <= lane / 16) dsum += psum[si * L + lane];
        rd[wave * L + lane] = 1.f / (fmaxf(fabsf(dsum), em[buf * L + lane]) + 1e-6f);
      }
      float* oc = a.out + (int64_t)(start + c0) * os + (int64_t)h * a.dv + col;
#pragma unroll
      for (int ti = 0; ti < LT; ++ti) {
        const f32x4 f = *reinterpret_cast<const f32x4*>(ic + hw * L + ti * 16 + lg * 4);
#pragma unroll
        for (int r = 0; r < 4; ++r) o[ti][r] = (SEP ? o[ti][r] + ol[ti][r] : o[ti][r]) * f[r];
        ol[ti] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int j = 0; j < KL; ++j) {
        bf16x8 vp[NP];
        if constexpr (NP == 1) {
#pragma unroll
          for (int i = 0; i < 8; ++i) vp[0][i] = vr[j * 8 + i];
        } else {
          float x[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) x[i] = (float)vr[j * 8 + i];
          split8<NP>(x, vp);
        }
#pragma unroll
        for (int ti = 2 * j; ti < LT; ++ti) {
          bf16x8 fa[3];
#pragma unroll
          for (int i = 0; i < 3; ++i)
            fa[i] = *reinterpret_cast<const bf16x8*>(Ps + ((hw * 3 + i) * L + ti * 16 + lr) * LP + j * 32 + lg * 8);
          mm<SEP, 3, NP>(fa, vp, o[ti], ol[ti]);
        }
      }
      if (some_bad)
#pragma unroll
        for (int ti = 0; ti < LT; ++ti)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[ti][r] = ti * 16 + lg * 4 + r >= bad ? NAN : o[ti][r];
#pragma unroll
      for (int ti = 0; ti < LT; ++ti) {
        f32x4 f = {1.f, 1.f, 1.f, 1.f};
        if (MLSTM) f = *reinterpret_cast<const f32x4*>(rd + wave * L + ti * 16 + lg * 4);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int t = ti * 16 + lg * 4 + r;
          if (t < nl && colok)
            oc[t * ro] = MLSTM ? (SEP ? o[ti][r] + ol[ti][r] : o[ti][r]) * f[r]
                               : __builtin_fmaf(skip, xr[ti][r], o[ti][r] + ol[ti][r]);
        }
      }
    }
    const float decay = sa[buf * HPW + hw];
    bf16x8 vp[KL][3];
#pragma unroll
    for (int j = 0; j < KL; ++j) {
      float x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = (float)vr[j * 8 + i] * wc[hw * L + j * 32 + lg * 8 + i];
      split8<3>(x, vp[j]);
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      // three parts: the update's main product from zero, then one fused step; else it starts from
      // the decayed state
      f32x4 hi = {0.f, 0.f, 0.f, 0.f}, lo = hi;
      if (NP <= 2)
#pragma unroll
        for (int r = 0; r < 4; ++r) hi[r] = S[dt][r] * decay;
#pragma unroll
      for (int j = 0; j < KL; ++j) {
        bf16x8 fa[NP];
#pragma unroll
        for (int i = 0; i < NP; ++i)
          fa[i] = *reinterpret_cast<const bf16x8*>(KT + i * D * LP + (dt * 16 + lr) * LP + j * 32 + lg * 8);
        mm<(NP > 2), NP, 3>(fa, vp[j], hi, lo);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
        S[dt][r] = NP > 2 ? __builtin_fmaf(S[dt][r], decay, hi[r] + lo[r]) : hi[r];
      if (dt % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    if (some_bad)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[dt][r] = bad < L ? NAN : S[dt][r];
    if (MLSTM) {                             // n <- decay n + sum_t w_t k_t: NT / D threads per row
      constexpr int TPD = NT / D;
      const int c = tid / TPD, sub = tid % TPD;
      float x = 0.f;
#pragma unroll
      for (int t = sub * 8; t < L; t += TPD * 8)
#pragma unroll
        for (int i = 0; i < NP; ++i) {
          const bf16x8 f = *reinterpret_cast<const bf16x8*>(KT + i * D * LP + c * LP + t);
#pragma unroll
          for (int e = 0; e < 8; ++e) x += (float)f[e] * wc[t + e];
        }
#pragma unroll
      for (int o = 1; o < TPD; o <<= 1) x += __shfl_xor(x, o, 64);
      if (sub == 0) ns[mfma_perm(c)] = sa[buf * HPW] * ns[mfma_perm(c)] + x;
    }
    __syncthreads();
  }

  // ---- the state after the walk -----------------------------------------------------------
  int dw = a.dv;                             // opaque: addresses are not kept across the walk
  asm volatile("" : "+s"(dw));
  const bool to_slot = MODE == 0 || (MODE == 2 && last_seg);
  if (MODE == 1 || to_slot) {
    const int64_t it = (int64_t)(seg_first + seg_idx) * a.H + h;
    float* dst = MODE == 1 ? a.seg_state + it * item_floats : Ss;
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = i * 16 + 4 * lg + r;
        if (colok) dst[row * dw + col] = S[i][r];
      }
    if (ct == 0) {
      if (MLSTM && tid < D) {
        float* nd = MODE == 1 ? dst + sh : a.n + ((int64_t)slot * a.H + h) * D;
        nd[tid] = ns[mfma_perm(tid)];
      }
      if (hg < HPW && lane == 0) {
        const int64_t ih = (int64_t)(seg_first + seg_idx) * a.H + h0 + hg;
        if (MODE == 1) {
          a.seg_gate[2 * ih] = btot;
          a.seg_gate[2 * ih + 1] = m0;
        } else if (MLSTM) {
          a.m[(int64_t)slot * a.H + h0 + hg] = (float)m0;
        }
      }
    }
  }
}

template <typename E, int D, int L, int HPW>
constexpr size_t chunk_lds() {
  constexpr int NP = PartsOf<E>::n;
  return (size_t)2 * (2 * NP * L * (D + 8) + NP * D * (L + 8) + HPW * 3 * L * (L + 8)) +
         32 * HPW * L + 4 * (6 * HPW * L + 4 + 3 * L + L / 16 * L + D + NW * L);
}

template <typename E, bool MLSTM, int D, int L, int HPW, int MODE>
bool chunk_allowed() {
  static OncePerDevice once;
  return allow_lds(once, &chunk_scan_kernel<E, MLSTM, D, L, HPW, MODE>, chunk_lds<E, D, L, HPW>());
}
// the current device takes all launches of the form
template <typename E, bool MLSTM, int D, int L, int HPW>
bool chunk_form_ok() {
  return chunk_allowed<E, MLSTM, D, L, HPW, 0>() && chunk_allowed<E, MLSTM, D, L, HPW, 1>() &&
         chunk_allowed<E, MLSTM, D, L, HPW, 2>();
}

template <typename E, bool MLSTM, int D, int L, int HPW, int MODE>
void chunk_run(const ChunkArgs& a, int items, hipStream_t s) {
  const int nct = (a.dv + 16 * (NW / HPW) - 1) / (16 * (NW / HPW));
  chunk_scan_kernel<E, MLSTM, D, L, HPW, MODE>
      <<<dim3(items, a.H / HPW * nct), NT, chunk_lds<E, D, L, HPW>(), s>>>(a);
}

template <typename E, bool MLSTM, int D, int L, int HPW>
void chunk_dispatch(const ChunkArgs& a, int items, hipStream_t s) {
  if (a.seg <= 0) {
    chunk_run<E, MLSTM, D, L, HPW, 0>(a, a.P, s);
  } else {
    chunk_run<E, MLSTM, D, L, HPW, 1>(a, items, s);
    chunk_run<E, MLSTM, D, L, HPW, 2>(a, items, s);
  }
}

}  // namespace

// Segment length for a step of P sequences and Tp tokens whose walk has `wgs` workgroups per
// sequence, `least` chunks of L at least (0: sequences are not cut, as those of less than `shortest` chunks on
// average), and the number of segments it can come to.
static ChunkWork chunk_plan(int P, int Tp, int wgs, int L, int least, int shortest) {
  ChunkWork p;
  p.items = P;
  // a CU holds one of these workgroups; cut only where a good part of the CUs would idle
  // and the pieces are long enough to pay for computing every contribution twice
  const int want = (device_cus() + wgs - 1) / wgs;
  if (P * 2 > want) return p;
  const int seg = segment_rows(P, Tp, want, L, least);    // one round
  if (Tp / P < 2 * seg || Tp / P < shortest * L) return p;
  p.seg = seg;
  p.items = Tp / seg + P;
  return p;
}

// Chunkwise from 16 rows per sequence on or where the costs say so (of bf16 rows by a tenth: without, 4 rows were up to 12 %
// slower, 4 of 256 x 512 16 x 4 27.4 -> 30.7; chunk_mlstm.hip's kernel, which takes their larger steps, costs 0.7 of
// this file's), heads of 128 or 256 key channels in 16 bits (fp32 rows in
// three parts do not fit LDS).  32 x 512 tokens, 4 heads of 256 x 512: 1957 us token by token, 222 us
// chunkwise here and 128 to 136 in chunk_mlstm.hip, and nearer to float64 (3.5e-7 and 3.0e-7 against 5.0e-7).
bool mlstm_chunk_ok(int dtype, int64_t stride, const void* qkvg, int P, int Tp, int H, int d, int dv) {
  constexpr ChunkCost COST[2] = {{10.0, 0.0085, 0.0, 0.92, 0.0022, 13.5, 0.014, 10.8, 0.04, 0.0, 2},
                                 {12.5, 0.0185, 0.0, 1.45, 0.0034, 20.0, 0.029, 10.8, 0.068, 0.0, 2}};
  if (!((dtype == DT_BF16 || dtype == DT_F16) && P > 0 && (d == 128 || d == 256) &&
        (Tp >= 16 * P || chunk_pays(COST[d / 256], P, Tp, H, dv, dtype != DT_BF16 ? 1.0 : dv > 128 && Tp >= 1024 ? 0.7 : 1.1)) &&
        stride % 8 == 0 && (reinterpret_cast<uintptr_t>(qkvg) & 15) == 0 && dv >= 16 &&
        chunk_fits(stride, (long)H * dv, (long)H * ((dv + 127) / 128))))
    return false;
  if (dtype == DT_BF16) return d == 128 ? chunk_form_ok<bf16, true, 128, 64, 1>() : chunk_form_ok<bf16, true, 256, 64, 1>();
  return d == 128 ? chunk_form_ok<f16, true, 128, 32, 1>() : chunk_form_ok<f16, true, 256, 32, 1>();
}

// bf16 rows by DMA: heads of more than 128 columns, of which a workgroup there has twice as many, in sequences long enough
// to be cut and in steps of at least 1024 rows; with 128 key channels, whose walks gain less, the latter only where this
// file's do not all fit the CUs.  Heads of up to 128 columns leave half of its waves idle, which only shorter segments
// than this file's outweigh.  This file's kernel -> chunk_mlstm.hip's, us:
//   4 heads of 256 x 512   32 x 512, 24 x 700, 16 x 1000, 64 x 20   219 -> 136, 263 -> 147, 206 -> 185, 97 -> 75
//                          1 x 384, 512, 1000, 4000, 2 x 8192       72 -> 59, 74 -> 60, 84 -> 70, 122 -> 101, 318 -> 234
//                          16 x 64, 8 x 256, 4 x 300, 32 x 16       31.4 -> 31.0, 59.5 -> 58.7, 64.0 -> 64.6, 90.0 -> 89.8
//                          8 x 64, 4 x 64, 1 x 64, 1 x 256          23.9 -> 24.3, 22.4 -> 23.1, 20.5 -> 21.4, 52.7 -> 53.9
//   4 heads of 128 x 512   4 x 300, 8 x 200, 16 x 100, 300, 1000    39.5 -> 42.6, 34.0 -> 36.6, 23.2 -> 24.3, 42 -> 46, 114 -> 125
//                          32 x 64, 200, 64 x 20                    26 -> 21, 64 -> 40, 46 -> 32
//                          1 x 600, 5000, 8 x 600, 1500 (cut)       49 -> 41, 86 -> 74, 74 -> 64, 164 -> 116
//   4 heads of 256 x 128   32 x 200, 256 x 30                       56.0 -> 55.1, 77.9 -> 79.6
//                          1 x 600, 2 x 5000, 8 x 1500 (segments of 128, 192, 256)   71 -> 54, 114 -> 92, 91 -> 98
//   16 of 128 x 128        32 x 64, 16 x 300; 1 x 1500, 2 x 1000, 4 x 800 (128, 192, 320)   28 -> 29, 44 -> 48; 58 -> 47, 56 -> 56, 56 -> 69
ChunkWork mlstm_chunk_plan(int dtype, int P, int Tp, int H, int d, int dv) {
  const int wpi = H * ((dv + 127) / 128);
  if (mlstm_rows_ok(dtype, dv)) {
    const int cols = mlstm_rows_columns();
    ChunkWork p = chunk_plan(P, Tp, H * ((dv + cols - 1) / cols), 64, 2, 6);
    if (p.seg > 0) p.rows = dv > 128 || p.seg <= 192;
    else p.rows = Tp >= 1024 && dv > 128 && (d > 128 || (int64_t)P * wpi > device_cus());
    if (p.rows) return p;
  }
  return chunk_plan(P, Tp, wpi, dtype == DT_BF16 ? 64 : 32, 4, 8);
}

void launch_mlstm_chunk(int dtype, float* out, const void* qkvg, int64_t stride, const float* gates,
                        float* S, float* nst, float* mst, const float* n0, const float* m0,
                        const int* qsl, const int* seq_lens, const int* slots, int P, int H, int d,
                        int dv, int num_slots, const ChunkWork& work, hipStream_t s) {
  if (work.rows) {
    launch_mlstm_rows(out, qkvg, (const char*)qkvg + 2 * H * d, (const char*)qkvg + 4 * H * d, stride, gates, S, nst, mst,
                      n0, m0, qsl, seq_lens, slots, P, H, d, dv, num_slots, work, s);
    return;
  }
  ChunkArgs a{};
  a.out = out;
  const size_t es = 2;
  a.q = qkvg;
  a.k = (const char*)qkvg + es * H * d;
  a.v = (const char*)qkvg + es * 2 * H * d;
  a.stride = stride;
  a.gates = gates;
  a.S = S; a.n = nst; a.m = mst; a.n0 = n0; a.m0 = m0;
  a.qsl = qsl; a.seq_lens = seq_lens; a.slots = slots;
  a.P = P; a.H = H; a.hpg = 1; a.dv = dv; a.num_slots = num_slots;
  a.seg = work.seg; a.seg_state = work.state; a.seg_gate = work.gate;
  if (dtype == DT_BF16) {
    if (d <= 128) chunk_dispatch<bf16, true, 128, 64, 1>(a, work.items, s);
    else chunk_dispatch<bf16, true, 256, 64, 1>(a, work.items, s);
  } else {
    if (d <= 128) chunk_dispatch<f16, true, 128, 32, 1>(a, work.items, s);
    else chunk_dispatch<f16, true, 256, 32, 1>(a, work.items, s);
  }
}

// heads per workgroup
static int ssd_heads(int H, int V, int G) { return V <= 64 && (H / G) % 2 == 0 ? 2 : 1; }

// Mamba-2: 128 state rows, fp32 x | B | C (three bf16 parts each), 32-token chunks; two heads of up
// to 64 columns share a workgroup's B and C.  16 rows alone stay token by token (9.9 us against 10.3;
// 4 x 18: 12.8 and 10.9).  2 x 8192 tokens, 32 heads of 128 x 64: 4821 us token by
// token (a chain of 8192 steps in 64 workgroups), 359 us in chunks and segments of 1184 (130 the walk
// from zero, 255 the second); from float64 7.0e-8 (7.3e-8).
bool ssd_chunk_ok(const float* xbc, int P, int Tp, int H, int V, int N, int G) {
  return P > 0 && Tp >= 16 * P && Tp >= 20 && N == 128 && V >= 16 && ((int64_t)H * V) % 4 == 0 &&
         (reinterpret_cast<uintptr_t>(xbc) & 15) == 0 &&
         chunk_fits((long)H * V + 2L * G * N, (long)H * V, (long)H * ((V + 127) / 128)) &&
         (ssd_heads(H, V, G) == 2 ? chunk_form_ok<float, false, 128, 32, 2>() : chunk_form_ok<float, false, 128, 32, 1>());
}

ChunkWork ssd_chunk_plan(int P, int Tp, int H, int V, int G) {
  const int hpw = ssd_heads(H, V, G), cols = 16 * (NW / hpw);
  return chunk_plan(P, Tp, H / hpw * ((V + cols - 1) / cols), 32, 4, 8);
}

void launch_ssd_chunk(int dtype, float* out, const float* xbc, const void* dt, int64_t dts,
                      const float* a_log, const float* dt_bias, const float* dskip, float* S,
                      const int* qsl, const int* seq_lens, const int* slots, int P, int H, int V,
                      int N, int G, int num_slots, const ChunkWork& work, hipStream_t s) {
  ChunkArgs a{};
  a.out = out;
  a.v = xbc;
  a.k = xbc + (int64_t)H * V;
  a.q = xbc + (int64_t)H * V + (int64_t)G * N;
  a.stride = (int64_t)H * V + 2 * (int64_t)G * N;
  a.dt = dt; a.dts = dts; a.dt_type = dtype;
  a.a_log = a_log; a.dt_bias = dt_bias; a.dskip = dskip;
  a.S = S;
  a.qsl = qsl; a.seq_lens = seq_lens; a.slots = slots;
  a.P = P; a.H = H; a.hpg = H / G; a.dv = V; a.num_slots = num_slots;
  a.seg = work.seg; a.seg_state = work.state; a.seg_gate = work.gate;
  if (ssd_heads(H, V, G) == 2) chunk_dispatch<float, false, 128, 32, 2>(a, work.items, s);
  else chunk_dispatch<float, false, 128, 32, 1>(a, work.items, s);
}

}  // namespace kgc
