// The mLSTM (Beck et al., xLSTM, 2024) over prompt rows in bf16, chunkwise on the matrix cores: the recurrence,
// its weights and its precision are those of chunk_scan.hip, which keeps f16 rows, heads whose values do
// not come in 16-byte units, and small steps.
//
// A workgroup of 8 waves owns 256 value columns of one head, a wave 32 of them, whose S [D, 32] stays in the
// accumulators of 32 x 32 x 16 MFMAs for the whole walk: twice the columns for each operand read from LDS, each
// chunk's scores and each staged row, and half the MFMAs' issue.  q, k and v come by DMA as their rows lie (a wave
// brings its own columns of v, so that no barrier stands before them); k is read transposed by the LDS itself, and the
// rows of an S tile are numbered so that its accumulators are the operand of Q S_0 in the order of q's channels.
// n . q and the update of n are MFMAs too, n and the weights as three rows (or columns) of bf16 parts.
//
// Per chunk of 64 tokens:
//   scores P (one wave of each SIMD), Q S_0, the parts of v's weighted rows; v of the chunk and k of the next arrive
//   barrier
//   P V, the update, the outputs; q of the next chunk arrives
//   barrier (the outputs are still on their way)
//
// What bounds it: instruction issue, most of it the splitting of S, at the clock of full load (1.98 GHz where calls follow
// each other, 2.4 for lighter kernels).  Per wave and chunk 214 MFMAs of 32 cycles and 1800 vector instructions of 4, two
// waves per SIMD: the matrix core works in 49 % of the cycles, vector instructions are issued in 59 %; 126 to 132 us
// for 32 x 512 tokens, 4 heads of 256 x 512 (16 columns per
// wave: 222 us).  What it took: no spills (their reloads wait for every DMA before them; so lane numbers and places
// are computed where they are used), the vector work and one memory instruction at a time between the MFMAs,
// and barriers without the fence's wait for stores.
//
// Few long sequences are cut into segments: one walk makes every segment's contribution from a zero state, a
// small launch puts the states together in which the segments start, and the second walk has them all (1 x 4000: 202 us
// where each segment summed its predecessors itself, 101 so).
#include "chunk.h"
#include "chunk_rows.h"
#include "device.h"
#include "launch.h"

namespace kgc {

namespace {

constexpr int L = 64, NT = 512, NW = NT / 64;
constexpr int CW = 32, CB = NW * CW;         // columns per wave, per workgroup
constexpr double LOG2E = 1.4426950408889634074;
typedef int int32x4 __attribute__((ext_vector_type(4)));

struct MlstmArgs {
  float* out;                                // [T, H dv]
  const bf16 *q, *k, *v;                     // element (row, head, column) at row * stride + h * d (dv) + c
  int64_t stride;
  const float* gates;                        // [T, 2 H]: log input | log forget gate
  float *S, *n, *m;
  const float *n0, *m0;                      // copies of n and m of the step's sequences
  const int *qsl, *seq_lens, *slots;
  int P, H, dv, num_slots;
  int seg;                                   // tokens per segment (0: sequences are not cut)
  float* seg_state;                          // as in chunk_scan.hip
  double* seg_gate;
};

// Place of 16-byte unit u of row t (a row has 16 or 32): eight rows one below the other, and four rows' neighbouring
// units, lie in different banks.
__device__ __forceinline__ int sw(int t) { return (t & 3) << 1 | (t >> 2 & 1) | ((t >> 3 ^ t) & 1) << 3; }
// likewise the 8 units of P's rows
__device__ __forceinline__ int p_at(int t, int u) { return t * L + (u ^ (t >> 1 & 7)) * 8; }

__device__ __forceinline__ bf16x8 ld_tr8(const bf16* p0, const bf16* p1) {
  const u32x2 a = ld_tr4(p0), b = ld_tr4(p1);
  return __builtin_bit_cast(bf16x8, u32x4{a[0], a[1], b[0], b[1]});
}

// sum over the four lanes that share lane & 15
__device__ __forceinline__ float sum_rows(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  x = __builtin_bit_cast(float, (uint32_t)a[0]) + __builtin_bit_cast(float, (uint32_t)a[1]);
  const uint32_t w = __builtin_bit_cast(uint32_t, x);
  const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  return __builtin_bit_cast(float, (uint32_t)b[0]) + __builtin_bit_cast(float, (uint32_t)b[1]);
}
// 1024 bytes from each wave's 64 lanes to LDS
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t src, int at, void* dst) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (__attribute__((address_space(3))) void*)dst, 16, at, 0, 0, 0);
}

// what the waves share beside the rows
template <int D, int MODE> struct __align__(16) WalkLds {
  bf16 Ps[MODE == 1 ? 512 : 3 * L * L];      // parts of the weighted scores
  // per chunk, two of each: the gates run one chunk ahead
  int rtn[2 * L], csn[2 * L];                // score weights: 2^(rtn_t + csn_s + rtf_t + csf_s), whole numbers and rests
  float rtf[2 * L], csf[2 * L];
  float inter[2 * L], wt[2 * L], em[2 * L];  // factor of a row of Q S_0, weight of a token, e^(-m_t)
  bf16 Wb[2 * 3 * L];                        // parts of the weights
  float ns[D];                               // n
  bf16 Nb[3 * D];                            // its parts
  double m0;
  float nq[L], psum[10 * 16], rd[L], sa[2];  // n_0 . q_t, row sums of P by tile, 1 / denominator, decay of S
};

// the running maximum after segment `item`, from the one before it
__device__ __forceinline__ double next_m(const MlstmArgs& a, int item, int h, double m) {
  const double* g = a.seg_gate + 2 * ((int64_t)item * a.H + h);
  return fmax(g[0] + m, g[1]);
}

// MODE 0: whole sequences, 1: segments from zero (states only), 2: segments from the states that they start in.
template <int D, int MODE>
__global__ __launch_bounds__(NT) void mlstm_walk_kernel(const MlstmArgs a) {
  constexpr int UR = D / 8, DT = D / 32, KS = D / 16;
  constexpr int NQ = L * UR / NT, NV = L * CW / 8 / 64;   // DMAs of a wave for the rows of a chunk
  static_assert(NQ * NT == L * UR, "rows by DMA");
  __shared__ __align__(16) bf16 K0[L * D], K1[L * D], V0[L * CB];
  __shared__ __align__(16) bf16 QV[MODE == 1 ? L * CB : L * D];   // q; MODE 1: v of every other chunk
  __shared__ WalkLds<D, MODE> sm;

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), tid = threadIdx.x;
  // (a move that the compiler does not look through: what depends on it is computed where it is used and
  // not kept over the walk, where there are no registers left)
  auto opaque = [](int x) {
    asm volatile("" : "+v"(x));
    return x;
  };
  auto uniform64 = [](const void* p) -> const char* {
    const uint64_t x = reinterpret_cast<uint64_t>(p);
    return reinterpret_cast<const char*>((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(x >> 32)) << 32 |
                                         (uint32_t)__builtin_amdgcn_readfirstlane((int)x));
  };
  auto uniform = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
  const int c32 = lane & 31, hi = lane >> 5;
  int seq = blockIdx.x, seg_idx = 0, seg_first = 0, seg_count = 1;
  if (MODE != 0) {
    const SegItem it = seg_item(blockIdx.x, a.qsl, a.P, a.seg);
    if (it.seq < 0) return;
    seq = __builtin_amdgcn_readfirstlane(it.seq);
    seg_idx = __builtin_amdgcn_readfirstlane(it.idx);
    seg_first = __builtin_amdgcn_readfirstlane(it.first);
    seg_count = __builtin_amdgcn_readfirstlane(it.count);
  }
  const bool last_seg = MODE != 0 && seg_idx + 1 == seg_count;
  const int nct = (a.dv + CB - 1) / CB;
  const int h = uniform(blockIdx.y / nct), ct = blockIdx.y - h * nct;
  const int col0 = uniform(ct * CB + wave * CW), col = col0 + c32;
  const bool colok = col < a.dv;
  const int colc = colok ? col : a.dv - 1;
  int start = uniform(a.qsl[seq]), len = uniform(a.qsl[seq + 1]) - start;
  const int pos0 = uniform(a.seq_lens[seq]) - len;
  const int slot = uniform(a.slots[seq]);
  const int64_t os = (int64_t)a.H * a.dv;
  if (MODE != 0) {
    start += seg_idx * a.seg;
    len = min(a.seg, len - seg_idx * a.seg);
  }
  if (len <= 0) return;
  if (slot < 0 || slot >= a.num_slots || pos0 < 0) {      // padding: defined zeros
    if (MODE != 1 && colok)
      for (int t = hi; t < len; t += 2) a.out[(start + t) * os + (int64_t)h * a.dv + col] = 0.f;
    return;
  }
  const bool fresh = pos0 == 0;
  if (MODE == 1 && last_seg) return;

  // ---- the state this walk starts from: register (i, j) holds row 32 i + srow(j) --------------
  auto srow = [&](int j) { return 16 * (j >> 3) + 8 * hi + (j & 7); };
  const int64_t sh = (int64_t)D * a.dv, item_floats = sh + D;
  float* Ss = a.S + ((int64_t)slot * a.H + h) * sh;
  const bool own = MODE == 2 && seg_count > 1;            // the state is the segment's (mlstm_chain_kernel)
  const float* mine = a.seg_state + ((int64_t)(seg_first + seg_idx) * a.H + h) * item_floats;
  const float* from = own ? mine : Ss;
  f32x16 S[DT];
  double m0 = 0.0;                           // running maximum
  const bool zero = MODE == 1 || (fresh && !own);
  if (zero) {
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int j = 0; j < 16; ++j) S[i][j] = 0.f;
  } else {
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int j = 0; j < 16; ++j) S[i][j] = from[(i * 32 + srow(j)) * a.dv + colc];
  }
  if (MODE == 1) m0 = -INFINITY;
  else if (!fresh) m0 = a.m0[(int64_t)seq * a.H + h];
  float nreg = 0.f;                          // n[tid] for tid < D
  if (tid < D && !zero) nreg = own ? mine[sh + tid] : a.n0[((int64_t)seq * a.H + h) * D + tid];
  if (MODE == 2)
    for (int p = 0; p < seg_idx; ++p) m0 = next_m(a, seg_first + p, h, m0);
  const char* qb = uniform64(a.q + (int64_t)start * a.stride + (int64_t)h * D);
  const char* kb = uniform64(a.k + (int64_t)start * a.stride + (int64_t)h * D);
  const char* vb = uniform64(a.v + (int64_t)start * a.stride + (int64_t)h * a.dv);
  const char* ob = uniform64(a.out + (int64_t)start * os + (int64_t)h * a.dv);
  const char* gb = uniform64(a.gates + (int64_t)start * 2 * a.H + h);
  const float qscale = 1.f / sqrtf((float)D);
  // this lane's number, computed again wherever it is asked for
  auto lane_id = [&] { return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, opaque(0))); };
  auto uopaque = [](int x) {                 // a scalar's
    asm volatile("" : "+s"(x));
    return x;
  };
  // Rows of the chunk at c0 to LDS; those past the end are the last one again (their weights are zero,
  // their outputs not stored).  Offsets inside a chunk fit 32 bits, row numbers and strides 24.
  // (One at a time: a burst of them would hold up the wave.)
  auto rows_at = [&](const char* src, int c0) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(uniform64(src + (int64_t)c0 * a.stride * 2)), 0,
                                             0x7fffffff, 0x00027000);
  };
  // q, k: a wave brings 8 rows (sw is linear); v: its own columns of all rows, 4 units of each, two of them
  // exchanged in rows 2 and 3 of every 4, and the last one again past the edge
  struct Place { int r, u; };                // a lane's row and byte in it
  auto k_part = [&] {
    const int ln = lane_id(), r = ln / UR;
    return Place{r + wave * 8, ((ln & (UR - 1)) ^ sw(r) ^ sw(wave * 8)) * 16};
  };
  auto v_part = [&] {
    const int ln = lane_id(), r = ln >> 2, u = (ln & 3) ^ (r & 2);
    return Place{r, min(col0 * 2 + u * 16, a.dv * 2 - 16)};
  };
  auto dma_k = [&](__amdgpu_buffer_rsrc_t src, bf16* dst, const Place& p, int i, int nl) {
    constexpr int R = 64 / UR;
    dma16(src, (int)__umul24(min(i * R + p.r, nl - 1), 2 * (int)a.stride) + (p.u ^ (sw(i * R) * 16)), dst + (wave * NQ + i) * 512);
  };
  auto dma_v = [&](__amdgpu_buffer_rsrc_t src, bf16* dst, const Place& p, int i, int nl) {
    dma16(src, (int)__umul24(min(i * 16 + p.r, nl - 1), 2 * (int)a.stride) + p.u, dst + (wave * NV + i) * 512);
  };

  // The gates of the chunk at c0, one token per lane, their running sums and maxima: the last wave does
  // them one chunk ahead.
  float gi = 0.f, gf = 0.f;
  double btot = 0.0;                         // log decay of the walk so far
  auto fetch_gates = [&](int c0) {
    const auto g = (const __attribute__((address_space(1))) float*)uniform64(gb + (int64_t)c0 * a.H * 8);
    const uint32_t t = (uint32_t)__umul24(min(lane_id(), min(L, len - c0) - 1), 2 * a.H);
    gi = g[t];
    gf = g[t + a.H];
  };
  auto scan_gates = [&](int nl, int buf) {
    const int lane = lane_id();
    const double m0 = sm.m0;
    const bool ok = lane < nl;
    // a decay of e^-1e6 is zero; a finite floor keeps the differences of running sums defined
    double f = gf;
    if (!ok) f = gi = 0.f;
    const double b = wave_scan<false>(f < -1e6 ? -1e6 : f);
    const double bL = lane63(b);
    const int at = buf * L + lane;
    const double c = ok ? (gi < -1e6f ? -1e6 : (double)gi) - b : -INFINITY;
    const double M = fmax(m0, wave_scan<true>(c)), ML = lane63(M);
    const float w = exp_d(c - ML);
    // whole numbers of 30 bits: input gates beyond 7e8 weigh the same
    constexpr double B = 1 << 30;
    const double re = M * LOG2E > B ? -B : -M * LOG2E, rn = __builtin_rint(re);
    const double ce = !ok ? -B : c * LOG2E > B ? B : c * LOG2E, cn = __builtin_rint(ce);
    sm.rtn[at] = (int)rn;
    sm.rtf[at] = (float)(re - rn);
    sm.csn[at] = (int)cn;
    sm.csf[at] = (float)(ce - cn);
    sm.inter[at] = exp_d(m0 - M) * qscale;
    sm.wt[at] = w;
    sm.em[at] = expf((float)-(b + M));
    uint32_t p[3];
    split2<3>(w, 0.f, p);
#pragma unroll
    for (int i = 0; i < 3; ++i) sm.Wb[(buf * 3 + i) * L + lane] = __builtin_bit_cast(bf16, (uint16_t)p[i]);
    if (lane == 0) sm.sa[buf] = exp_d(m0 - ML);
    sm.m0 = bL + ML;
    if (MODE == 1) btot += bL;
  };

  // places of a lane's operands: rows of q; four rows of k (v) transposed, the columns of k in the order of S's rows
  auto q_place = [&] {
    const int ln = lane_id(), r = ln & 31;
    return r * D + ((ln >> 5) ^ sw(r)) * 8;
  };
  auto k_place = [&] {
    const int ln = lane_id(), t = (ln >> 5) * 8 + (ln >> 2 & 3);
    return t * D + (((ln >> 3 & 2) | (ln & 1)) ^ sw(t)) * 8 + (ln & 2) * 2;
  };
  auto v_place = [&] {
    const int ln = lane_id(), t = (ln >> 5) * 8 + (ln >> 2 & 3);
    return wave * L * CW + t * CW + (((ln >> 3 & 2) + (ln >> 1 & 1)) ^ (t & 2)) * 8 + (ln & 1) * 4;
  };
  // operand of the update: tokens 16 ks .. of S's 32 rows i
  auto load_k = [&](const bf16* K, int base, int i, int ks) {
    const int p0 = base ^ ((i & 3) * 32), p1 = p0 ^ 8, at = (i >> 2) * 128 + ks * 16 * D;
    return ld_tr8(K + at + p0, K + at + 4 * D + p1);
  };
  auto split_s = [&](bf16x8 (&p)[3], int ks) {
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = S[ks >> 1][(ks & 1) * 8 + i];
    split8<3>(x, p);
  };

  // One piece of what is no DMA's target otherwise, read nowhere: to the compiler a read of such memory
  // follows all DMAs, a read of a target its own.
  dma16(__builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(qb), 0, 16, 0x00027000), 0, sm.Ps);
  __builtin_amdgcn_s_waitcnt(0x0f70);
  __syncthreads();
  if (tid < D) {
    sm.ns[tid] = nreg;
    uint32_t p[3];
    split2<3>(nreg, 0.f, p);
#pragma unroll
    for (int i = 0; i < 3; ++i) sm.Nb[i * D + tid] = __builtin_bit_cast(bf16, (uint16_t)p[i]);
  }
  if (MODE != 1)                             // tiles above the diagonal stay zero
    for (int i = tid; i < 3 * L * L / 8; i += NT) reinterpret_cast<u32x4*>(sm.Ps)[i] = u32x4{0, 0, 0, 0};
  {
    const Place kp = k_part(), vp = v_part();
    const int n0 = min(L, len);
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      if (MODE != 1) dma_k(rows_at(qb, 0), QV, kp, i, n0);
      dma_k(rows_at(kb, 0), K0, kp, i, n0);
    }
    if (MODE == 1)
#pragma unroll
      for (int i = 0; i < NV; ++i) dma_v(rows_at(vb, 0), V0, vp, i, n0);
  }
  if (wave == NW - 1) {
    sm.m0 = m0;
    fetch_gates(0);
    scan_gates(min(L, len), 0);
    if (MODE == 1 && L < len) fetch_gates(L);
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);        // (the first chunk's are)
  auto chunk = [&](int c, int buf, const bf16* K, bf16* Kn, const bf16* V, bf16* Vn) {
    const int c0 = uniform(c), nl = min(L, len - c0);
    const bool more = c0 + L < len;
    const int cn = more ? c0 + L : c0;       // (after the last chunk the same again)
    int ro = (int)os;
    asm volatile("" : "+s"(ro));
    // q and k are here (32 outputs of the last chunk may still be on their way)
    meet<MODE == 1 ? 0 : 32>();
    if (MODE == 1 && wave == NW - 1 && more) scan_gates(min(L, len - c0 - L), buf ^ 1);
    const int nn = min(L, len - cn);
    if (MODE == 1) {
      const Place kp = k_part(), vp = v_part();
      const auto ksrc = rows_at(kb, cn), vsrc = rows_at(vb, cn);
#pragma unroll
      for (int i = 0; i < NQ; ++i) dma_k(ksrc, Kn, kp, i, nn);
#pragma unroll
      for (int i = 0; i < NV; ++i) dma_v(vsrc, Vn, vp, i, nn);
    }
    if (MODE == 1 && uopaque(wave) == NW - 1 && c0 + 2 * L < len) fetch_gates(c0 + 2 * L);
    // ---- v, and its weighted parts -----------------------------------------------------------------
    union { bf16x8 v[4]; bf16 e[32]; } vv;
    auto load_v = [&] {
      const int vbase = v_place();
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) vv.v[ks] = ld_tr8(V + ks * 16 * CW + vbase, V + (ks * 16 + 4) * CW + vbase);
    };
    const float* wrow = sm.wt + buf * L + (lane_id() >> 5) * 8;
    f32x4 w[2];
    auto load_w = [&](int ks) {
      w[0] = *reinterpret_cast<const f32x4*>(wrow + ks * 16);
      w[1] = *reinterpret_cast<const f32x4*>(wrow + ks * 16 + 4);
    };
    auto split_v = [&](bf16x8 (&p)[3], int ks) {
      float x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = (float)vv.e[ks * 8 + i] * w[i >> 2][i & 3];
      split8<3>(x, p);
    };
    bf16x8 vp[4][3];
    int bad;
    bool some_bad;
    auto find_bad = [&] {
      bad = take_nonfinite<true>(vv.e, L, [&](int i) { return (i >> 3) * 16 + (lane_id() >> 5) * 8 + (i & 7); });
      some_bad = __builtin_amdgcn_readfirstlane(__any(bad < L));
    };
    f32x16 o[2];
    if (MODE != 1) {
      // ---- scores: tile (ti, si) as D[s][t], weighted, split, stored as rows of P.  Tiles on the diagonal
      // also bring n_0 . q_t, the parts of n as rows of the other operand.
      auto scores = [&] {
        const int ln = lane_id(), lr = ln & 15, lg = ln >> 4;
        for (int pass = 0; pass < 3 - (uopaque(wave) >> 1); ++pass) {
          const int at = 16 * pass + 4 * wave, ti = 0x003203321231 >> at & 7, si = 0x002103101200 >> at & 7;
          // operands first, the weights while they come
          bf16x8 fk[D / 32], fq[D / 32];
          const int ks0 = (lg ^ sw(lr)) * 8, t = ti * 16 + lr, s0 = si * 16 + lg * 4;
          const bf16 *kr = K + (si * 16 + lr) * D, *qr = QV + (ti * 16 + lr) * D, *nr = sm.Nb + min(lr, 2) * D + lg * 8;
          const int rn = sm.rtn[buf * L + t];
          const float rf = sm.rtf[buf * L + t];
          const int32x4 cn = *reinterpret_cast<const int32x4*>(sm.csn + buf * L + s0);
          const f32x4 cf = *reinterpret_cast<const f32x4*>(sm.csf + buf * L + s0);
#pragma unroll
          for (int ks = 0; ks < D / 32; ++ks) {
            fk[ks] = *reinterpret_cast<const bf16x8*>(kr + (ks0 ^ (ks * 32)));
            fq[ks] = *reinterpret_cast<const bf16x8*>(qr + (ks0 ^ (ks * 32)));
          }
          float e[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            e[r] = __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(rf + cf[r]) * qscale, rn + cn[r]);
            asm volatile("" : "+v"(e[r]));   // (no branches)
          }
          __builtin_amdgcn_sched_barrier(0);
          f32x4 acc = {0.f, 0.f, 0.f, 0.f}, ac1 = acc;
#pragma unroll
          for (int ks = 0; ks < D / 32; ks += 2) {
            acc = mfma16x16x32(fk[ks], fq[ks], acc);
            ac1 = mfma16x16x32(fk[ks + 1], fq[ks + 1], ac1);
          }
          if (ti == si) {
            f32x4 an = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < D / 32; ++ks)
              an = mfma16x16x32(*reinterpret_cast<const bf16x8*>(nr + ks * 32), fq[ks], an);
            if (lg == 0) sm.nq[ti * 16 + lr] = an[2] + an[1] + an[0];
          }
          acc += ac1;
          float p[4], sum = 0.f;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            p[r] = s0 + r <= t ? acc[r] * e[r] : 0.f;
            sum += p[r];
          }
          sum = sum_rows(sum);
          if (lg == 0) sm.psum[(ti * (ti + 1) / 2 + si) * 16 + lr] = sum;
          uint32_t lo2[3], hi2[3];
          split2<3>(p[0], p[1], lo2);
          split2<3>(p[2], p[3], hi2);
  #pragma unroll
          for (int i = 0; i < 3; ++i)
            *reinterpret_cast<u32x2*>(sm.Ps + i * L * L + p_at(t, s0 >> 3) + (s0 & 4)) = u32x2{lo2[i], hi2[i]};
        }
      };
      // One wave of each SIMD does them, three tiles or two, while the other is at Q S_0.
      if (uopaque(wave) < NW / 2) scores();
      // ---- Q S_0 of this wave's columns, the parts of S a step ahead ------------------------------
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) o[i][j] = 0.f;
      bf16x8 fa[2][2], sp[2][3];
      const int qbase = q_place();
      auto load_q = [&](bf16x8 (&f)[2], int ks) {
        const bf16* p = QV + (qbase ^ ((ks & 7) * 16)) + (ks >> 3) * 128;
        f[0] = *reinterpret_cast<const bf16x8*>(p);
        f[1] = *reinterpret_cast<const bf16x8*>(p + 32 * D);
      };
      const auto vsrc = rows_at(vb, c0), ksrc = rows_at(kb, cn);
      const Place vpl = v_part(), kpl = k_part();
      load_q(fa[0], 0);
      split_s(sp[0], 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int k = ks & 1;
        if (ks + 1 < KS) {
          load_q(fa[k ^ 1], ks + 1);
          split_s(sp[k ^ 1], ks + 1);
        }
        // v and k, spread over the steps: all CUs ask at the same time
        constexpr int STEP = KS / (NV + NQ);
        if (ks % STEP == 0 && ks / STEP < NV) dma_v(vsrc, Vn, vpl, ks / STEP, nl);
        else if (ks % STEP == 0 && ks / STEP < NV + NQ) dma_k(ksrc, Kn, kpl, ks / STEP - NV, nn);
#pragma unroll
        for (int p = 2; p >= 0; --p)
#pragma unroll
          for (int i = 0; i < 2; ++i) o[i] = mfma32x32x16(fa[k][i], sp[k][p], o[i]);
        __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);   // addresses
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        interleave<6, 8, 0, 6>();
        __builtin_amdgcn_sched_barrier(0);
      }
      if (uopaque(wave) == NW - 1 && more) fetch_gates(c0 + L);
      // ---- the rows' factors; v, which the wave has brought for itself, and its weighted parts --------
      const float* fin = sm.inter + buf * L + (lane_id() >> 5) * 4;
      __builtin_amdgcn_s_waitcnt(0x0f70 | NQ);            // k of the next chunk need not be here
      load_v();
      load_w(0);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 f = *reinterpret_cast<const f32x4*>(fin + i * 32 + g * 8);
#pragma unroll
          for (int r = 0; r < 4; ++r) o[i][g * 4 + r] *= f[r];
        }
      find_bad();
      split_v(vp[0], 0);
      load_w(1);
      split_v(vp[1], 1);
      if (uopaque(wave) == NW - 1 && more) scan_gates(min(L, len - c0 - L), buf ^ 1);
      meet<NQ>();                            // v is here, k of the next chunk need not be
    }
    const float decay = sm.sa[buf];
    const int kbase = k_place();
    bf16x8 fk[2][2];                         // operands of the update: 32 rows, 32 tokens
    auto load_fk = [&](int q) {
#pragma unroll
      for (int k = 0; k < 2; ++k) fk[q & 1][k] = load_k(K, kbase, q & (DT - 1), q / DT * 2 + k);
    };
    // writes past the chunk's last row do nothing
    const auto od = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(uniform64(ob + (int64_t)c0 * os * 4)), 0,
        uniform(((nl - 1) * ro + a.dv) * 4), 0x00027000);
    const int ol = lane_id(), oc = col0 + (ol & 31);
    const uint32_t oat = oc < a.dv ? (uint32_t)(__mul24((ol >> 5) * 4, ro) + oc) * 4 : 1u << 30;
    const float* rds = sm.rd + (ol >> 5) * 4;
    constexpr int OS = DT / 4;               // steps of the update per group of four output rows
    f32x4 rdv;
    auto load_rd = [&](int g) { rdv = *reinterpret_cast<const f32x4*>(rds + (g >> 2) * 32 + (g & 3) * 8); };
    if (MODE != 1) {
      const auto qsrc = rows_at(qb, cn);
      const Place qpl = k_part();
      const int pl = lane_id(), prow = pl & 31, phi = pl >> 5;
      constexpr int PK[6] = {0, 0, 1, 1, 2, 3}, PI[6] = {0, 1, 0, 1, 1, 1};   // 16 tokens, 32 rows of the step
      bf16x8 fp[2][3];
      auto load_p = [&](int q) {
#pragma unroll
        for (int p = 0; p < 3; ++p)
          fp[q & 1][p] = *reinterpret_cast<const bf16x8*>(sm.Ps + p * L * L + p_at(PI[q] * 32 + prow, 2 * PK[q] + phi));
      };
      load_p(0);
      {                                      // every wave writes the same
        const int t = lane_id(), ti = t >> 4;
        const float* row = sm.psum + ti * (ti + 1) * 8 + (t & 15);
        float dsum = sm.nq[t] * sm.inter[buf * L + t] + row[0];
#pragma unroll
        for (int si = 1; si < 4; ++si) {
          const float x = row[min(si, ti) * 16];
          dsum += si <= ti ? x : 0.f;
        }
        sm.rd[t] = 1.f / (fmaxf(fabsf(dsum), sm.em[buf * L + t]) + 1e-6f);
      }
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        if (q < 5) load_p(q + 1);
        if (q < NQ) dma_k(qsrc, QV, qpl, q, nn);
        if (q == 4) load_fk(0);
        if (q == 5) {
          load_w(2);
          load_rd(0);
#pragma unroll
          for (int j = 0; j < 16; ++j) S[0][j] *= decay;
        }
#pragma unroll
        for (int p = 2; p >= 0; --p) o[PI[q]] = mfma32x32x16(fp[q & 1][p], vv.v[PK[q]], o[PI[q]]);
        __builtin_amdgcn_sched_barrier(0);
      }
      const int badr = bad - (lane_id() >> 5) * 4;
      if (some_bad)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            float x = o[i][j];
            asm volatile("" : "+v"(x));      // a branch, not selects in every chunk
            o[i][j] = i * 32 + (j >> 2) * 8 + (j & 3) >= badr ? NAN : x;
          }
    } else {
      load_v();
      find_bad();
      load_w(0);
      split_v(vp[0], 0);
      load_w(1);
      split_v(vp[1], 1);
      load_w(2);
      load_fk(0);
#pragma unroll
      for (int j = 0; j < 16; ++j) S[0][j] *= decay;
    }
    // (past the caches, which whole lines of results would fill: 32 x 512 tokens 131 -> 127.6 us, 1 x 4000 102.4 -> 101)
    auto put_o = [&](int i, int g, const f32x4& f) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float y = o[i][g * 4 + r] * f[r];
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, y), od, oat + (i * 32 + g * 8 + r) * ro * 4, 0, 2);
      }
    };
    // ---- n <- decay n + sum_t w_t k_t: 32 rows per wave, the weights' parts as columns ------------
    f32x16 nx;
    const int nd = wave & (DT - 1);
    auto sum_n = [&] {
      const bf16* wr = sm.Wb + (buf * 3 + min(lane_id() & 31, 2)) * L + (lane_id() >> 5) * 8;
#pragma unroll
      for (int j = 0; j < 16; ++j) nx[j] = 0.f;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        nx = mfma32x32x16(load_k(K, kbase, nd, ks), *reinterpret_cast<const bf16x8*>(wr + ks * 16), nx);
    };
    auto put_n = [&](int g) {                // the three columns, into the first; eight rows
      float y[8];
      const int row = nd * 32 + g * 16 + (lane_id() >> 5) * 8;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float x = nx[g * 8 + j];
        const float x1 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x101, 0xf, 0xf, true));
        const float x2 = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x102, 0xf, 0xf, true));
        y[j] = sm.ns[row + j] * decay + (x2 + x1 + x);
      }
      bf16x8 p[3];
      split8<3>(y, p);
      if ((lane_id() & 31) == 0 && wave < DT) {
#pragma unroll
        for (int j = 0; j < 8; ++j) sm.ns[row + j] = y[j];
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8*>(sm.Nb + i * D + row) = p[i];
      }
    };
    // ---- the update, 32 tokens at a time: in the first half the state decays, a step ahead; the outputs leave
    // on the way
#pragma unroll
    for (int q = 0; q < 2 * DT; ++q) {
      const int i = q & (DT - 1);
      if (q + 1 < 2 * DT) load_fk(q + 1);
      if (q + 1 < DT)
#pragma unroll
        for (int j = 0; j < 16; ++j) S[i + 1][j] *= decay;
      if (MODE != 1 && q % OS == 0) {
        put_o(q / OS >> 2, q / OS & 3, rdv);
        if (q / OS < 7) load_rd(q / OS + 1);
      }
      if (q == DT / 2) {
        split_v(vp[2], 2);
        load_w(3);
      }
      if (q == DT / 2 + 1) split_v(vp[3], 3);
      if (q == DT - 1) sum_n();
      if (q == DT + 1 || q == DT + 2) put_n(q - DT - 1);
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int p = 2; p >= 0; --p) S[i] = mfma32x32x16(fk[q & 1][k], vp[q / DT * 2 + k][p], S[i]);
      __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
      if (q < DT / 2) interleave<6, 4, 0, 1>();
      else if (q < DT) interleave<6, 12, 0, 1>();
      else interleave<6, 2, 0, 1>();
      __builtin_amdgcn_sched_barrier(0);
    }
    if (some_bad)
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          float x = S[i][j];
          asm volatile("" : "+v"(x));
          S[i][j] = bad < L ? NAN : x;
        }
  };
  for (int c0 = 0; c0 < len; c0 += 2 * L) {
    chunk(c0, 0, K0, K1, V0, MODE == 1 ? QV : V0);
    if (c0 + L < len) chunk(c0 + L, 1, K1, K0, MODE == 1 ? QV : V0, V0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

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
      for (int j = 0; j < 16; ++j)
        if (colok) dst[(i * 32 + srow(j)) * dw + col] = S[i][j];
    if (ct == 0) {
      if (tid < D) (MODE == 1 ? dst + sh : a.n + ((int64_t)slot * a.H + h) * D)[tid] = sm.ns[tid];
      if (wave == NW - 1 && lane == 0) {
        if (MODE == 1) {
          a.seg_gate[2 * it] = btot;
          a.seg_gate[2 * it + 1] = sm.m0;
        } else {
          a.m[(int64_t)slot * a.H + h] = (float)sm.m0;
        }
      }
    }
  }
}

// ---- the states (and n) in which segments start, in place of the contributions -----------------
__global__ __launch_bounds__(256) void mlstm_chain_kernel(const MlstmArgs a, int D) {
  const int seq = blockIdx.z, h = blockIdx.y, lane = threadIdx.x & 63;
  const int len = a.qsl[seq + 1] - a.qsl[seq], pos0 = a.seq_lens[seq] - len, slot = a.slots[seq];
  if (len <= a.seg || slot < 0 || slot >= a.num_slots || pos0 < 0) return;
  const int first = pieces_before(seq, a.qsl, a.seg);
  const int count = (len + a.seg - 1) / a.seg;
  const int64_t sh = (int64_t)D * a.dv, step = (int64_t)a.H * (sh + D);
  const int64_t at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;   // (a multiple of 4 elements each)
  if (at >= sh + D) return;
  f32x4 S = {0.f, 0.f, 0.f, 0.f};
  double m = 0.0;
  if (pos0 != 0) {
    S = *reinterpret_cast<const f32x4*>(at < sh ? a.S + ((int64_t)slot * a.H + h) * sh + at
                                                : a.n0 + ((int64_t)seq * a.H + h) * D + (at - sh));
    m = a.m0[(int64_t)seq * a.H + h];
  }
  float* p = a.seg_state + ((int64_t)first * a.H + h) * (sh + D) + at;
#pragma unroll 4
  for (int j = 0; j < count - 1; ++j) {
    // S <- e^(b + m - m') S + e^(m_j - m') S_j
    const f32x4 c = *reinterpret_cast<const f32x4*>(p + j * step);
    const double* g = a.seg_gate + 2 * ((int64_t)(first + j) * a.H + h);
    const double mn = next_m(a, first + j, h, m);
    const float f = exp_d(g[0] + m - mn), w = exp_d(g[1] - mn);
    *reinterpret_cast<f32x4*>(p + j * step) = S;
#pragma unroll
    for (int r = 0; r < 4; ++r) S[r] = f * S[r] + w * c[r];
    m = mn;
  }
  *reinterpret_cast<f32x4*>(p + (count - 1) * step) = S;
}

template <int D> void walk(const MlstmArgs& a, int items, hipStream_t s) {
  const dim3 whole(a.P, a.H * ((a.dv + CB - 1) / CB)), cut(items, whole.y);
  if (a.seg <= 0) {
    mlstm_walk_kernel<D, 0><<<whole, NT, 0, s>>>(a);
  } else {
    mlstm_walk_kernel<D, 1><<<cut, NT, 0, s>>>(a);
    mlstm_chain_kernel<<<dim3((D * (a.dv + 1) / 4 + 255) / 256, a.H, a.P), 256, 0, s>>>(a, D);
    mlstm_walk_kernel<D, 2><<<cut, NT, 0, s>>>(a);
  }
}

}  // namespace

bool mlstm_rows_ok(int dtype, int dv) {
  return dtype == DT_BF16 && dv % 8 == 0;
}

int mlstm_rows_columns() { return CB; }

void launch_mlstm_rows(float* out, const void* q, const void* k, const void* v, int64_t stride, const float* gates,
                       float* S, float* nst, float* mst, const float* n0, const float* m0, const int* qsl,
                       const int* seq_lens, const int* slots, int P, int H, int d, int dv, int num_slots,
                       const ChunkWork& work, hipStream_t s) {
  MlstmArgs a{};
  a.out = out;
  a.q = static_cast<const bf16*>(q);
  a.k = static_cast<const bf16*>(k);
  a.v = static_cast<const bf16*>(v);
  a.stride = stride;
  a.gates = gates;
  a.S = S; a.n = nst; a.m = mst; a.n0 = n0; a.m0 = m0;
  a.qsl = qsl; a.seq_lens = seq_lens; a.slots = slots;
  a.P = P; a.H = H; a.dv = dv; a.num_slots = num_slots;
  a.seg = work.seg; a.seg_state = work.state; a.seg_gate = work.gate;
  if (d == 128) walk<128>(a, work.items, s);
  else walk<256>(a, work.items, s);
}

}  // namespace kgc
