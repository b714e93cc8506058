// K2 varlen causal prefill attention over the paged KV cache (gfx950, bf16/f16).
//
// Each sequence contributes query rows [qsl[i], qsl[i+1]) at absolute positions
// seq_len-qlen .. seq_len-1 and attends causally to cache positions [0, seq_len):
// fresh prompts and chunked-prefill continuations run the same code.  The new
// tokens' K/V were already scattered into the cache by rope_kv_write.
//
// Grid: (work items, q-heads); a work item = (sequence, 128-row query block), listed
// heaviest-first by the host.  Workgroup = 4 waves x 32 query rows (two 16-row
// q-tiles per wave).  K/V advance in 64-key tiles staged global->VGPR->LDS,
// double-buffered, loads issued before the tile's MFMAs and written after them
// (one barrier per tile).
//
// MFMA orientation (v_mfma_f32_16x16x32): S^T = K.Q^T and O^T = V^T.P^T, so the
// query index is lane&15 in every accumulator: the online-softmax max/sum/rescale
// are lane-local (+ xor 16/32), and S^T's accumulator is already the B operand of
// the P.V product (row->key map key(m) = 8*(m>>2)+(m&3), +4 for the second tile of
// each 32-key pair).
// LDS images (16-byte chunk swizzles, conflict-free for the ds_read_b128 groups):
//   K   [64 keys][D]   chunk c of key k stored at c ^ f(k), f(k) = (k&3)|((k>>3)&3)<<2
//   V^T [D][64 keys]   chunk c of dim d stored at c ^ ((d>>1)&7)
#include "common.h"
#include "device.h"
#include "launch.h"
#include "prefill_items.h"
#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace kgc {

constexpr int PF_BM = 128;
constexpr int PF_BN = 64;

__device__ __forceinline__ int kswz(int k) { return (k & 3) | (((k >> 3) & 3) << 2); }

// over the four lanes that share lane & 15, without the LDS's latency (a shuffle's) in the chain
__device__ __forceinline__ float max_rows(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  x = __builtin_elementwise_maximum(__builtin_bit_cast(float, (uint32_t)a[0]), __builtin_bit_cast(float, (uint32_t)a[1]));
  const uint32_t w = __builtin_bit_cast(uint32_t, x);
  const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  return __builtin_elementwise_maximum(__builtin_bit_cast(float, (uint32_t)b[0]), __builtin_bit_cast(float, (uint32_t)b[1]));
}

// a barrier that leaves the newest N memory operations on their way
template <int N> __device__ __forceinline__ void pf_meet() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt((N & 15) | (N >> 4) << 14 | 0x70);   // vmcnt(N) lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// cos / sin of one row's dims as pf_load_q uses them, loaded ahead of the rotation
template <int D> struct PfRot { float4 c[D / 64][4]; };   // per fragment pair: cos lo / hi, sin lo / hi
template <int D>
__device__ __forceinline__ void pf_issue_rot(const float* __restrict__ cs_row, int qd, PfRot<D>& r) {
#pragma unroll
  for (int s = 0; s < D / 64; ++s) {
    const int col = 32 * s + 8 * qd;
    r.c[s][0] = *reinterpret_cast<const float4*>(cs_row + col);
    r.c[s][1] = *reinterpret_cast<const float4*>(cs_row + col + 4);
    r.c[s][2] = *reinterpret_cast<const float4*>(cs_row + D / 2 + col);
    r.c[s][3] = *reinterpret_cast<const float4*>(cs_row + D / 2 + col + 4);
  }
}
template <typename T, int D>
__device__ __forceinline__ void pf_rotate(const PfRot<D>& r, Pack8<T> (&t)[D / 32]) {
  constexpr int KS = D / 32;
#pragma unroll
  for (int s = 0; s < KS / 2; ++s) {
    const float cc[8] = {r.c[s][0].x, r.c[s][0].y, r.c[s][0].z, r.c[s][0].w,
                         r.c[s][1].x, r.c[s][1].y, r.c[s][1].z, r.c[s][1].w};
    const float sn[8] = {r.c[s][2].x, r.c[s][2].y, r.c[s][2].z, r.c[s][2].w,
                         r.c[s][3].x, r.c[s][3].y, r.c[s][3].z, r.c[s][3].w};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float ra, rb;
      neox_rot(to_f(t[s].h[j]), to_f(t[s + KS / 2].h[j]), cc[j], sn[j], ra, rb);
      t[s].h[j] = from_f<T>(ra);
      t[s + KS / 2].h[j] = from_f<T>(rb);
    }
  }
}

// q fragments of one 16-row q-tile: lane (r16, qd) holds dims 32 s + 8 qd .. + 7 of its
// row.  cos_sin != nullptr: the row is the unrotated q of the fused QKV projection and
// gets NeoX RoPE at position pos here -- dims i and i + D/2 sit in fragments s and
// s + KS/2 of the same lane, so the rotation is lane-local -- rounded to T exactly as
// rope_cache.hip rounds it.  (Prefill-only steps: rope_kv_write then writes only k / v,
// and q is neither stored nor re-read.)
template <typename T, int D>
__device__ __forceinline__ void pf_load_q(const T* qrow, const float* __restrict__ cos_sin,
                                          int cs_rows, int pos, int qd,
                                          typename Vec8<T>::type (&qf)[D / 32]) {
  constexpr int KS = D / 32;
  Pack8<T> t[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) t[s].u = *reinterpret_cast<const u32x4*>(qrow + 32 * s + 8 * qd);
  if (cos_sin != nullptr) {
    PfRot<D> r;
    // clamped: a bad sequence length gives wrong output, never a fault
    pf_issue_rot<D>(cos_sin + (int64_t)min(pos, cs_rows - 1) * D, qd, r);
    pf_rotate<T, D>(r, t);
  }
#pragma unroll
  for (int s = 0; s < KS; ++s) qf[s] = t[s].v;
}

// Lazy O rescale (log2 units): the running max m only moves when some row's tile max
// exceeds it by more than this, so P = exp2(s - m) stays <= 2^8 and the O / l rescale
// (DT*8 + 2 VALU per lane) runs on a few tiles per row instead of on every tile.  The
// decision covers the tile BEFORE its P is exponentiated and after the previous tile's
// P.V is complete, and O, l and m move together (no P at the old scale is pending).
constexpr float PF_RESCALE_THR = 8.f;

// keys behind a row's own position
__device__ __forceinline__ void pf_mask(f32x4 (&s)[2][4], const int (&qpos)[2], int key0, int qd) {
#pragma unroll
  for (int qt = 0; qt < 2; ++qt)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (key0 + (j >> 1) * 32 + 8 * qd + 4 * (j & 1) + i > qpos[qt]) s[qt][j][i] = -INFINITY;
}

// Lazy online softmax of a tile's scores (query = lane & 15: lane-local statistics): p = 2^(c s - m).  The maximum is the
// one that hands on a NaN, whose row is NaN either way: v_max first quiets every score that an MFMA has made.
template <typename T, int D>
__device__ __forceinline__ void pf_softmax(const f32x4 (&s)[2][4], typename Vec8<T>::type (&pf)[2][2], f32x4 (&o)[2][D / 16],
                                           float (&m)[2], float (&l)[2], float c) {
  constexpr int DT = D / 16;
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    float tmax = s[qt][0][0];
#pragma unroll
    for (int i = 1; i < 16; ++i) tmax = __builtin_elementwise_maximum(tmax, s[qt][i >> 2][i & 3]);
    tmax = max_rows(tmax);
    tmax *= c;                              // -inf stays -inf (a fully masked row)
    if (__any(tmax > m[qt] + PF_RESCALE_THR)) {
      const float mn = __builtin_elementwise_maximum(m[qt], tmax);
      const float alpha = __builtin_amdgcn_exp2f(m[qt] - mn);   // 0 on the first tile
      m[qt] = mn;
      l[qt] *= alpha;
#pragma unroll
      for (int t = 0; t < DT; ++t) o[qt][t] *= alpha;
    }
    const float nm = -m[qt];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      Pack8<T> pk;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float pa = __builtin_amdgcn_exp2f(__builtin_fmaf(s[qt][2 * kk][i], c, nm));
        const float pb = __builtin_amdgcn_exp2f(__builtin_fmaf(s[qt][2 * kk + 1][i], c, nm));
        l[qt] += pa + pb;
        pk.h[i] = from_f<T>(pa);
        pk.h[4 + i] = from_f<T>(pb);
      }
      pf[qt][kk] = pk.v;
    }
  }
}

// One 64-key tile for a wave's 32 query rows (two 16-row q-tiles), shared by both
// kernels.  K / V are the staged LDS images; key0 = the tile's first key.  Scores stay
// raw through the max (scale_log2 > 0 commutes with max) and enter the exponent as
// fma(s, scale_log2, -m): one VALU per score instead of a multiply and a subtract.
// exp2 is the bare v_exp_f32 (inputs <= PF_RESCALE_THR, -inf -> 0; no denormal
// range fix-up: exp2f() lowered to ~6 VALU per call).  MASK = the causal diagonal
// crosses this tile for some row of the wave; off-diagonal tiles skip the per-element
// key compare entirely.
template <typename T, int D, bool MASK>
__device__ __forceinline__ void pf_wave_tile(const T* __restrict__ K, const T* __restrict__ V,
                                             const typename Vec8<T>::type (&qf)[2][D / 32],
                                             f32x4 (&o)[2][D / 16], float (&m)[2], float (&l)[2],
                                             const int (&qpos)[2], int key0, float c, int r16,
                                             int qd) {
  typedef typename Vec8<T>::type V8;
  constexpr int NCH = D / 8, KS = D / 32, DT = D / 16;
  const int keyA = 8 * (r16 >> 2) + (r16 & 3);
  // ---- S^T tiles: [qt][a0, b0, a1, b1]
  f32x4 s[2][4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int key = (j >> 1) * 32 + keyA + 4 * (j & 1);
    const T* krow = K + key * D;
    f32x4 a0 = {0.f, 0.f, 0.f, 0.f}, a1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      Pack8<T> f;
      f.u = *reinterpret_cast<const u32x4*>(krow + (((4 * ks + qd) ^ (r16 & (NCH - 1))) * 8));
      a0 = mfma16x16x32(f.v, qf[0][ks], a0);
      a1 = mfma16x16x32(f.v, qf[1][ks], a1);
    }
    s[0][j] = a0;
    s[1][j] = a1;
  }
  V8 pf[2][2];
  if constexpr (MASK) pf_mask(s, qpos, key0, qd);
  pf_softmax<T, D>(s, pf, o, m, l, c);
  // ---- O^T += V^T . P^T
#pragma unroll
  for (int t = 0; t < DT; ++t) {
    const int d = 16 * t + r16;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      Pack8<T> f;
      f.u = *reinterpret_cast<const u32x4*>(V + d * PF_BN + (((4 * kk + qd) ^ ((d >> 1) & 7)) * 8));
      o[0][t] = mfma16x16x32(f.v, pf[0][kk], o[0][t]);
      o[1][t] = mfma16x16x32(f.v, pf[1][kk], o[1][t]);
    }
  }
}

// KV8: fp8 e4m3 cache; staged as 8-byte loads, widened to T on the way into LDS (the
// LDS image and everything after it is unchanged).  K scale folded into scale_log2,
// V scale applied in the epilogue.
template <typename T, int D, bool KV8>
__global__ __launch_bounds__(256, 2) void prefill_attn_kernel(
    const T* __restrict__ q, T* __restrict__ out, const void* __restrict__ kc_,
    const void* __restrict__ vc_, const int* __restrict__ block_tables, int bt_stride,
    const int* __restrict__ qsl, const int* __restrict__ seq_lens,
    const int* __restrict__ work_seq, const int* __restrict__ work_mblk, int nq, int nkv,
    int bs_log2, float scale_log2, float v_scale, int num_blocks, int64_t q_stride,
    const float* __restrict__ cos_sin, int cs_rows) {
  typedef typename Vec8<T>::type V8;
  typedef std::conditional_t<KV8, uint8_t, T> C;   // cache element
  typedef std::conditional_t<KV8, u32x2, u32x4> R; // staged raw fragment (8 elements)
  const C* __restrict__ kc = reinterpret_cast<const C*>(kc_);
  const C* __restrict__ vc = reinterpret_cast<const C*>(vc_);
  auto widen = [](R r) -> u32x4 {
    if constexpr (KV8) return fp8x8_widen<T>(r);
    else return r;
  };
  constexpr int NCH = D / 8;                 // 16-byte chunks per K row
  constexpr int KS = D / 32;                 // k-steps of QK^T
  constexpr int DT = D / 16;                 // d-tiles of O^T
  constexpr int KPT = PF_BN * NCH / 256;     // K chunks staged per thread
  constexpr int VPT = D * (PF_BN / 8) / 256; // V chunks staged per thread
  constexpr int TILE = PF_BN * D;            // elements per K (or V) image
  extern __shared__ __attribute__((aligned(16))) char smem[];
  T* lds = reinterpret_cast<T*>(smem);

  const int seq = work_seq[blockIdx.x], mb = work_mblk[blockIdx.x];
  const int hq = blockIdx.y;
  const int h = hq / (nq / nkv);
  const int q0 = qsl[seq];
  const int qlen = qsl[seq + 1] - q0;
  int L_in = seq_lens[seq];
  KGC_DCHECK_RANGE(L_in, 0, (bt_stride << bs_log2) + 1, "prefill seq_len");
  const int L = min(L_in, bt_stride << bs_log2);  // never index past the table
  const int ctx0 = L - qlen;
  if (qlen <= 0 || ctx0 < 0) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r16 = lane & 15, qd = lane >> 4;
  const int* bt = block_tables + (int64_t)seq * bt_stride;
  const int bsm = (1 << bs_log2) - 1;
  const int64_t hs = (int64_t)D << bs_log2;  // elements per (block, kv-head)

  V8 qf[2][KS];
  int qpos[2];
  // q is loaded (and, with cos_sin, rotated) AFTER the first K/V tile's loads are issued:
  // the rotation waits for q, and vmcnt retires in order, so q loaded first put its
  // latency in series with the block-table -> K/V chain of every workgroup's first tile
  auto load_q = [&]() {
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      const int qi = mb * PF_BM + wave * 32 + qt * 16 + r16;
      const int qc = min(qi, qlen - 1);
      qpos[qt] = ctx0 + qc;
      pf_load_q<T, D>(q + (int64_t)(q0 + qc) * q_stride + (int64_t)hq * D, cos_sin, cs_rows,
                      qpos[qt], qd, qf[qt]);
    }
  };
  const int last_q = ctx0 + min((mb + 1) * PF_BM, qlen) - 1;
  const int n_tiles = last_q / PF_BN + 1;

  // Block ids of a tile's chunks are fetched one tile AHEAD of its K/V loads: the
  // dependent block-table load would otherwise stall every tile's load issue for an
  // L2 round trip before the compute it is meant to overlap.
  R kreg[KPT], vreg[VPT];
  int kblk[KPT], vblk[VPT];
  auto fetch_bt = [&](int kt) {
#pragma unroll
    for (int u = 0; u < KPT; ++u) {
      const int key = (threadIdx.x + 256 * u) / NCH;
      kblk[u] = kgc_bt(bt, min(kt * PF_BN + key, L - 1) >> bs_log2, bt_stride, num_blocks);
    }
#pragma unroll
    for (int u = 0; u < VPT; ++u) {
      const int c = (threadIdx.x + 256 * u) / D;
      vblk[u] = kgc_bt(bt, (min(kt * PF_BN + 8 * c, L - 1) & ~7) >> bs_log2, bt_stride, num_blocks);
    }
  };
  auto load_tile = [&](int kt) {
#pragma unroll
    for (int u = 0; u < KPT; ++u) {
      const int ci = threadIdx.x + 256 * u;
      const int key = ci / NCH, c = ci % NCH;
      const int ka = min(kt * PF_BN + key, L - 1);
      const C* src = kc + ((int64_t)kblk[u] * nkv + h) * hs + (int64_t)(ka & bsm) * D + c * 8;
      kreg[u] = *reinterpret_cast<const R*>(src);
    }
#pragma unroll
    for (int u = 0; u < VPT; ++u) {       // 8-key group c of dim d: contiguous in d
      const int ci = threadIdx.x + 256 * u;
      const int c = ci / D, d = ci % D;
      const int ka = min(kt * PF_BN + 8 * c, L - 1) & ~7;
      const C* src = vc + ((int64_t)vblk[u] * nkv + h) * hs + ((ka & bsm) >> 3) * (D * 8) + d * 8;
      vreg[u] = *reinterpret_cast<const R*>(src);
    }
  };
  auto store_tile = [&](int buf) {
    T* K = lds + buf * 2 * TILE;
    T* V = K + TILE;
#pragma unroll
    for (int u = 0; u < KPT; ++u) {
      const int ci = threadIdx.x + 256 * u;
      const int key = ci / NCH, c = ci % NCH;
      *reinterpret_cast<u32x4*>(K + key * D + ((c ^ (kswz(key) & (NCH - 1))) * 8)) = widen(kreg[u]);
    }
#pragma unroll
    for (int u = 0; u < VPT; ++u) {
      const int ci = threadIdx.x + 256 * u;
      const int c = ci / D, d = ci % D;
      *reinterpret_cast<u32x4*>(V + d * PF_BN + ((c ^ ((d >> 1) & 7)) * 8)) = widen(vreg[u]);
    }
  };

  f32x4 o[2][DT];
#pragma unroll
  for (int qt = 0; qt < 2; ++qt)
#pragma unroll
    for (int t = 0; t < DT; ++t) o[qt][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m[2] = {-INFINITY, -INFINITY}, l[2] = {0.f, 0.f};

  fetch_bt(0);
  load_tile(0);
  load_q();
  if (n_tiles > 1) fetch_bt(1);
  store_tile(0);
  __syncthreads();
  for (int kt = 0; kt < n_tiles; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < n_tiles) {
      load_tile(kt + 1);
      fetch_bt(min(kt + 2, n_tiles - 1));   // unconditional: static vmcnt below
    }
    const T* K = lds + buf * 2 * TILE;
    const T* V = K + TILE;
    if ((kt + 1) * PF_BN - 1 > ctx0 + mb * PF_BM + wave * 32)
      pf_wave_tile<T, D, true>(K, V, qf, o, m, l, qpos, kt * PF_BN, scale_log2, r16, qd);
    else
      pf_wave_tile<T, D, false>(K, V, qf, o, m, l, qpos, kt * PF_BN, scale_log2, r16, qd);
    if (kt + 1 < n_tiles) store_tile(buf ^ 1);
    __syncthreads();
  }
  // ---- epilogue: O / l; lane holds O[query r16][16t + 4qd + i]
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    float tot = l[qt];
    tot += __shfl_xor(tot, 16, 64);
    tot += __shfl_xor(tot, 32, 64);
    const float inv = v_scale / tot;
    const int qi = mb * PF_BM + wave * 32 + qt * 16 + r16;
    if (qi < qlen) {
      T* orow = out + ((int64_t)(q0 + qi) * nq + hq) * D + 4 * qd;
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        Pack4<T> pk;
#pragma unroll
        for (int i = 0; i < 4; ++i) pk.h[i] = from_f<T>(o[qt][t][i] * inv);
        *reinterpret_cast<u32x2*>(orow + 16 * t) = pk.u;
      }
    }
  }
}

// GQA-shared variant (G = nq / nkv >= 4): one workgroup = GH q-heads of ONE kv head x
// QB = 128 / GH queries, 4 waves of 32 query rows (wave w: head w % GH, rows
// 32 * (w / GH) ..), two workgroups per CU.  Every K/V tile staged into LDS feeds 128 query rows of
// four heads instead of 128 rows of one head, and there is one staging pass per kv head instead of
// one per q-head.  The 128-row work items of the engine's work list split into 128 / QB sub-blocks; the
// blocks of an item run over the heads first (with 8 kv heads an XCD sees one of them).  The per-wave
// math is the single-head kernel's.
template <typename T, int D, bool KV8, int GH>
__global__ __launch_bounds__(256, 2) void prefill_attn_gqa_kernel(
    const T* __restrict__ q, T* __restrict__ out, const void* __restrict__ kc_,
    const void* __restrict__ vc_, const int* __restrict__ block_tables, int bt_stride,
    const int* __restrict__ qsl, const int* __restrict__ seq_lens,
    const int* __restrict__ work_seq, const int* __restrict__ work_mblk, int nq, int nkv,
    int bs_log2, float scale_log2, float v_scale, int num_blocks, int64_t q_stride,
    const float* __restrict__ cos_sin, int cs_rows) {
  typedef typename Vec8<T>::type V8;
  typedef std::conditional_t<KV8, uint8_t, T> C;
  typedef std::conditional_t<KV8, u32x2, u32x4> R;
  const C* __restrict__ kc = reinterpret_cast<const C*>(kc_);
  const C* __restrict__ vc = reinterpret_cast<const C*>(vc_);
  auto widen = [](R r) -> u32x4 {
    if constexpr (KV8) return fp8x8_widen<T>(r);
    else return r;
  };
  constexpr int NT_ = 256;
  constexpr int QB = 128 / GH;               // queries per workgroup
  static_assert(QB <= PF_BM && PF_BM % QB == 0, "sub-blocks of the 128-row work item");
  constexpr int NCH = D / 8, KS = D / 32, DT = D / 16;
  constexpr int KPT = PF_BN * NCH / NT_;
  constexpr int VPT = D * (PF_BN / 8) / NT_;
  constexpr int TILE = PF_BN * D;
  static_assert(KPT * NT_ == PF_BN * NCH && VPT * NT_ == D * (PF_BN / 8), "staging split");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  T* lds = reinterpret_cast<T*>(smem);

  const int G = nq / nkv, Y = nkv * (G / GH), w = blockIdx.x / (Y * (PF_BM / QB));
  const int y = blockIdx.x % Y, z = blockIdx.x / Y % (PF_BM / QB);
  const int seq = work_seq[w], mb = work_mblk[w];
  const int h = y / (G / GH);                          // kv head
  const int hg0 = h * G + (y % (G / GH)) * GH;         // first q-head of this workgroup
  const int q0 = qsl[seq];
  const int qlen = qsl[seq + 1] - q0;
  int L_in = seq_lens[seq];
  KGC_DCHECK_RANGE(L_in, 0, (bt_stride << bs_log2) + 1, "prefill seq_len");
  const int L = min(L_in, bt_stride << bs_log2);
  const int ctx0 = L - qlen;
  const int qbase = mb * PF_BM + z * QB;      // first query row of the workgroup
  if (qlen <= 0 || ctx0 < 0 || qbase >= qlen) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int hq = hg0 + wave % GH;
  const int wq0 = qbase + (wave / GH) * 32;            // first query row of this wave
  const int r16 = lane & 15, qd = lane >> 4;
  const int bsm = (1 << bs_log2) - 1;
  const int64_t hs = (int64_t)D << bs_log2;

  V8 qf[2][KS];
  int qpos[2];
  // q is loaded (and, with cos_sin, rotated) AFTER the first K/V tile's loads are issued:
  // the rotation waits for q, and vmcnt retires in order, so q loaded first put its
  // latency in series with the block-table -> K/V chain of every workgroup's first tile
  auto load_q = [&]() {
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      const int qi = wq0 + qt * 16 + r16;
      const int qc = min(qi, qlen - 1);
      qpos[qt] = ctx0 + qc;
      pf_load_q<T, D>(q + (int64_t)(q0 + qc) * q_stride + (int64_t)hq * D, cos_sin, cs_rows,
                      qpos[qt], qd, qf[qt]);
    }
  };
  const int last_q = ctx0 + min(qbase + QB, qlen) - 1;
  const int n_tiles = last_q / PF_BN + 1;

  // Block ids of a tile's chunks are fetched one tile AHEAD of its K/V loads: the
  // dependent block-table load would otherwise stall every tile's load issue for an
  // L2 round trip before the compute it is meant to overlap.
  // A wave's 64 chunks of one load are 4 whole keys (of a page: pages hold a multiple of 8) or half of
  // an 8-key group: block ids and the groups' places are scalar.
  static_assert(D == 128 && PF_BN == 64, "rows per wave");
  R kreg[KPT], vreg[VPT];
  int kblk[KPT], vblk[VPT];
  typedef const __attribute__((address_space(4))) int* TablePtr;
  const TablePtr bt = (TablePtr)(block_tables + (int64_t)seq * bt_stride);
  auto fetch_bt = [&](int kt) {
    auto id = [&](int key) {
      int i = min(key, L - 1) >> bs_log2;
      KGC_DCHECK_RANGE(i, 0, bt_stride, "block-table column");
      int v = bt[i];
      KGC_DCHECK_RANGE(v, 0, num_blocks, "block id");
      return v;
    };
#pragma unroll
    for (int u = 0; u < KPT; ++u) kblk[u] = id(kt * PF_BN + 4 * wave + (NT_ / 16) * u);
#pragma unroll
    for (int u = 0; u < VPT; ++u) vblk[u] = id(kt * PF_BN + 8 * ((wave >> 1) + (NT_ / 128) * u));
  };
  // (the lane index behind an opaque move: addresses that depend on it alone are not kept in
  // registers over the tile loop, where there are none left)
  auto opaque = [](int x) {
    asm volatile("" : "+v"(x));
    return x;
  };
  auto load_tile = [&](int kt) {
    const int lane = opaque(threadIdx.x & 63);
#pragma unroll
    for (int u = 0; u < KPT; ++u) {
      const C* page = kc + ((int64_t)kblk[u] * nkv + h) * hs;
      const int ka = min(kt * PF_BN + 4 * wave + (NT_ / 16) * u + (lane >> 4), L - 1);
      kreg[u] = *reinterpret_cast<const R*>(page + ((ka & bsm) * D + (lane & 15) * 8));
    }
#pragma unroll
    for (int u = 0; u < VPT; ++u) {
      const int ka = min(kt * PF_BN + 8 * ((wave >> 1) + (NT_ / 128) * u), L - 1);
      const C* group = vc + ((int64_t)vblk[u] * nkv + h) * hs + ((ka & bsm) >> 3) * (D * 8);
      vreg[u] = *reinterpret_cast<const R*>(group + ((wave & 1) * 64 + lane) * 8);
    }
  };
  auto store_tile = [&](int buf) {
    const int tid = opaque(threadIdx.x);
    T* K = lds + buf * 2 * TILE;
    T* V = K + TILE;
#pragma unroll
    for (int u = 0; u < KPT; ++u) {
      const int ci = tid + NT_ * u;
      const int key = ci / NCH, c = ci % NCH;
      *reinterpret_cast<u32x4*>(K + key * D + ((c ^ (kswz(key) & (NCH - 1))) * 8)) = widen(kreg[u]);
    }
#pragma unroll
    for (int u = 0; u < VPT; ++u) {
      const int ci = tid + NT_ * u;
      const int c = ci / D, d = ci % D;
      *reinterpret_cast<u32x4*>(V + d * PF_BN + ((c ^ ((d >> 1) & 7)) * 8)) = widen(vreg[u]);
    }
  };

  f32x4 o[2][DT];
#pragma unroll
  for (int qt = 0; qt < 2; ++qt)
#pragma unroll
    for (int t = 0; t < DT; ++t) o[qt][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m[2] = {-INFINITY, -INFINITY}, l[2] = {0.f, 0.f};
  // this wave's own last key tile (its rows end before the workgroup's last row)
  const int wave_tiles = (ctx0 + min(wq0 + 31, qlen - 1)) / PF_BN + 1;

  fetch_bt(0);
  load_tile(0);
  load_q();
  fetch_bt(n_tiles > 1);
  __builtin_amdgcn_s_waitcnt(0x0f70);        // vmcnt(0): q is there
  store_tile(0);
  __syncthreads();
  for (int kt = 0; kt < n_tiles; ++kt) {
    const int buf = kt & 1;
    load_tile(min(kt + 1, n_tiles - 1));
    if (kt < wave_tiles) {
      const T* K = lds + buf * 2 * TILE;
      const T* V = K + TILE;
      if ((kt + 1) * PF_BN - 1 > ctx0 + wq0)
        pf_wave_tile<T, D, true>(K, V, qf, o, m, l, qpos, kt * PF_BN, scale_log2, r16, qd);
      else
        pf_wave_tile<T, D, false>(K, V, qf, o, m, l, qpos, kt * PF_BN, scale_log2, r16, qd);
    }
    fetch_bt(min(kt + 2, n_tiles - 1));
    store_tile(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) {
    float tot = l[qt];
    tot += __shfl_xor(tot, 16, 64);
    tot += __shfl_xor(tot, 32, 64);
    const float inv = v_scale / tot;
    const int qi = wq0 + qt * 16 + r16;
    if (qi < qlen && qi < qbase + QB) {
      T* orow = out + ((int64_t)(q0 + qi) * nq + hq) * D + 4 * qd;
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        Pack4<T> pk;
#pragma unroll
        for (int i = 0; i < 4; ++i) pk.h[i] = from_f<T>(o[qt][t][i] * inv);
        *reinterpret_cast<u32x2*>(orow + 16 * t) = pk.u;
      }
    }
  }
}

// Persistent GQA variant (fp8 caches, pages of fewer than 32 keys): ONE workgroup per CU walks the work list (items = (128-row work
// item, kv-head group, QB-row sub-block), heaviest first, dealt round-robin), with the K / V
// tile stream running ACROSS items: the last tile of an item loads the next item's first
// tile into the free LDS buffer, so a new item starts with its tile already staged.
// Per-wave math, tile order and rounding are those of prefill_attn_gqa_kernel (results are
// bit-identical).  Why: at short prompts every workgroup of the one-shot grid paid its own
// pipeline fill -- the work_seq -> qsl / seq_lens -> block table -> K / V chain of dependent
// loads, the q load and the first LDS store, ~10 us -- against 1-8 tiles of ~2.5 us of
// work each.  What an item still costs beside its tiles
// are its q and output rows: q comes by DMA while the item before it computes, outputs leave as whole
// 256-byte rows (32 x 512 181 -> 162 us, 64 x 256 146 -> 126, 2 x 8192 1309 -> 1276).  At 32 x 512 vector
// instructions issue in 47 % of a SIMD's cycles, its matrix core works in 20 %; 300 MB of rows, 60 us at the
// rate of a copy, are what all CUs ask for at the same time.  Rotating the rows in LDS
// with each cos / sin row read once, and a stream of tiles without any wait before an item's compute,
// measured within 3 % of this and a tenth slower on long prompts.
template <typename T, int D, bool KV8, int GH>
__global__ __launch_bounds__(512, 1) void prefill_attn_gqa_persist_kernel(
    const T* __restrict__ q, T* __restrict__ out, const void* __restrict__ kc_,
    const void* __restrict__ vc_, const int* __restrict__ block_tables, int bt_stride,
    const int* __restrict__ qsl, const int* __restrict__ seq_lens,
    const int* __restrict__ work_seq, const int* __restrict__ work_mblk, int nq, int nkv,
    int bs_log2, float scale_log2, float v_scale, int num_blocks, int64_t q_stride,
    const float* __restrict__ cos_sin, int cs_rows, int n_items) {
  typedef typename Vec8<T>::type V8;
  typedef std::conditional_t<KV8, uint8_t, T> C;
  typedef std::conditional_t<KV8, u32x2, u32x4> R;
  const C* __restrict__ kc = reinterpret_cast<const C*>(kc_);
  const C* __restrict__ vc = reinterpret_cast<const C*>(vc_);
  auto widen = [](R r) -> u32x4 {
    if constexpr (KV8) return fp8x8_widen<T>(r);
    else return r;
  };
  constexpr int NT_ = 512;
  constexpr int QB = 256 / GH;
  constexpr int ZS = PF_BM / QB;                       // sub-blocks per 128-row work item
  constexpr int NCH = D / 8, KS = D / 32, DT = D / 16;
  constexpr int KPT = PF_BN * NCH / NT_;
  constexpr int VPT = D * (PF_BN / 8) / NT_;
  constexpr int TILE = PF_BN * D;
  static_assert(KPT * NT_ == PF_BN * NCH && VPT * NT_ == D * (PF_BN / 8), "staging split");
  // two objects: the compiler lets an LDS read follow every DMA into the object that it reads
  __shared__ __attribute__((aligned(16))) T lds[4 * TILE];
  __shared__ __attribute__((aligned(16))) T all_rows[256 * D];

  const int G = nq / nkv;
  const int Y = nkv * (G / GH);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r16 = lane & 15, qd = lane >> 4;
  const int bsm = (1 << bs_log2) - 1;
  const int64_t hs = (int64_t)D << bs_log2;
  const int cap = bt_stride << bs_log2;

  // an item's workgroup-uniform geometry (scalar registers); the per-wave values (q-head,
  // first row, last tile) are derived for the current item only (VGPRs are the limit
  // here: 256 at one workgroup of 8 waves per CU)
  struct Item {
    int q0, qlen, L, ctx0, qbase, hg0, h, n_tiles;
    const int* bt;
  };
  // item idx -> its geometry; false: nothing to do (empty / out-of-range sub-block)
  auto decode = [&](int idx, Item& I) -> bool {
    const int w = idx / (Y * ZS), r = idx - w * (Y * ZS);
    const int y = r / ZS, z = r - y * ZS;
    const int seq = work_seq[w], mb = work_mblk[w];
    I.h = y / (G / GH);
    I.hg0 = I.h * G + (y % (G / GH)) * GH;
    I.q0 = qsl[seq];
    I.qlen = qsl[seq + 1] - I.q0;
    int L_in = seq_lens[seq];
    KGC_DCHECK_RANGE(L_in, 0, cap + 1, "prefill seq_len");
    I.L = min(L_in, cap);
    I.ctx0 = I.L - I.qlen;
    I.qbase = mb * PF_BM + z * QB;
    if (I.qlen <= 0 || I.ctx0 < 0 || I.qbase >= I.qlen) return false;
    I.n_tiles = (I.ctx0 + min(I.qbase + QB, I.qlen) - 1) / PF_BN + 1;
    I.bt = block_tables + (int64_t)seq * bt_stride;
    return true;
  };
  // Items are dealt in rounds of gridDim.x, heaviest first (the host's work-list order),
  // alternating direction round to round: workgroup b takes item r * G + b in even rounds
  // and r * G + G - 1 - b in odd ones, so the workgroup dealt a round's heaviest item gets
  // the next round's lightest (plain round-robin left long prompts ~10 % imbalanced).
  const int G_ = gridDim.x, b_ = blockIdx.x;
  auto item_of = [&](int r) -> int { return r * G_ + ((r & 1) ? G_ - 1 - b_ : b_); };
  // the first round >= r whose item this workgroup has work in (its item in `I`), or a
  // round past the list
  auto next_valid = [&](int r, Item& I) -> int {
    while (r * G_ < n_items) {
      const int idx = item_of(r);
      if (idx < n_items && decode(idx, I)) break;
      ++r;
    }
    return r;
  };

  V8 qf[2][KS];
  int qpos[2];
  const int wrow = (wave / GH) * 32, whead = wave % GH;    // this wave's rows / head
  auto load_q = [&](const Item& I) {
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      const int qi = I.qbase + wrow + qt * 16 + r16;
      const int qc = min(qi, I.qlen - 1);
      qpos[qt] = I.ctx0 + qc;
      pf_load_q<T, D>(q + (int64_t)(I.q0 + qc) * q_stride + (int64_t)(I.hg0 + whead) * D,
                      cos_sin, cs_rows, qpos[qt], qd, qf[qt]);
    }
  };
  // The next item's q rows come into LDS by DMA while this item computes (as register loads they
  // would need 32 VGPRs more; issued after the last tile, their 5 us stood in every item).  A wave's
  // 32 rows of its head, 16-byte chunks permuted by the row; afterwards the place where its output
  // rows meet, so that they are stored 256 bytes at a time.
  static_assert(D == 128, "16 chunks per row");
  T* rows = all_rows + wave * 32 * D;
  // (the lane index behind an opaque move: addresses that depend on it alone are not kept in
  // registers over the tile loop, where there are none left)
  auto opaque = [](int x) {
    asm volatile("" : "+v"(x));
    return x;
  };
  auto issue_q = [&](const Item& I) {
    const int ln = opaque(lane), rl = ln >> 4, cl = ln & 15;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = 4 * i + rl, qc = min(I.qbase + wrow + row, I.qlen - 1);
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(
              q + (int64_t)(I.q0 + qc) * q_stride + (int64_t)(I.hg0 + whead) * D + ((cl ^ (row & 15)) * 8)),
          (__attribute__((address_space(3))) void*)(rows + 4 * i * D), 16, 0, 0);
    }
  };
  auto finish_q = [&](const Item& I) {
    const int ln = opaque(lane), r16 = ln & 15, qd = ln >> 4;
    PfRot<D> rot[2];
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      qpos[qt] = I.ctx0 + min(I.qbase + wrow + qt * 16 + r16, I.qlen - 1);
      if (cos_sin != nullptr)
        pf_issue_rot<D>(cos_sin + (int64_t)min(qpos[qt], cs_rows - 1) * D, qd, rot[qt]);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the wave's own DMAs: no barrier
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      Pack8<T> t[KS];
#pragma unroll
      for (int s = 0; s < KS; ++s)
        t[s].u = *reinterpret_cast<const u32x4*>(rows + (qt * 16 + r16) * D + (((4 * s + qd) ^ r16) * 8));
      if (cos_sin != nullptr) pf_rotate<T, D>(rot[qt], t);
#pragma unroll
      for (int s = 0; s < KS; ++s) qf[qt][s] = t[s].v;
    }
  };
  R kreg[KPT], vreg[VPT];
  int kblk[KPT], vblk[VPT];
  auto fetch_bt = [&](const int* bt, int L, int kt) {
#pragma unroll
    for (int u = 0; u < KPT; ++u) {
      const int key = (threadIdx.x + NT_ * u) / NCH;
      kblk[u] = kgc_bt(bt, min(kt * PF_BN + key, L - 1) >> bs_log2, bt_stride, num_blocks);
    }
#pragma unroll
    for (int u = 0; u < VPT; ++u) {
      const int c = (threadIdx.x + NT_ * u) / D;
      vblk[u] = kgc_bt(bt, (min(kt * PF_BN + 8 * c, L - 1) & ~7) >> bs_log2, bt_stride, num_blocks);
    }
  };
  auto load_tile = [&](int L, int h, int kt) {
#pragma unroll
    for (int u = 0; u < KPT; ++u) {
      const int ci = threadIdx.x + NT_ * u;
      const int key = ci / NCH, c = ci % NCH;
      const int ka = min(kt * PF_BN + key, L - 1);
      const C* src = kc + ((int64_t)kblk[u] * nkv + h) * hs + (int64_t)(ka & bsm) * D + c * 8;
      kreg[u] = *reinterpret_cast<const R*>(src);
    }
#pragma unroll
    for (int u = 0; u < VPT; ++u) {
      const int ci = threadIdx.x + NT_ * u;
      const int c = ci / D, d = ci % D;
      const int ka = min(kt * PF_BN + 8 * c, L - 1) & ~7;
      const C* src = vc + ((int64_t)vblk[u] * nkv + h) * hs + ((ka & bsm) >> 3) * (D * 8) + d * 8;
      vreg[u] = *reinterpret_cast<const R*>(src);
    }
  };
  auto store_tile = [&](int buf) {
    const int tid = opaque(threadIdx.x);
    T* K = lds + buf * 2 * TILE;
    T* V = K + TILE;
#pragma unroll
    for (int u = 0; u < KPT; ++u) {
      const int ci = tid + NT_ * u;
      const int key = ci / NCH, c = ci % NCH;
      *reinterpret_cast<u32x4*>(K + key * D + ((c ^ (kswz(key) & (NCH - 1))) * 8)) = widen(kreg[u]);
    }
#pragma unroll
    for (int u = 0; u < VPT; ++u) {
      const int ci = tid + NT_ * u;
      const int c = ci / D, d = ci % D;
      *reinterpret_cast<u32x4*>(V + d * PF_BN + ((c ^ ((d >> 1) & 7)) * 8)) = widen(vreg[u]);
    }
  };

  Item cur, nxt;
  int it = next_valid(0, cur);                    // `it`: the current item's round
  if (it * G_ >= n_items) return;                 // uniform: the whole workgroup leaves
  fetch_bt(cur.bt, cur.L, 0);
  load_tile(cur.L, cur.h, 0);
  fetch_bt(cur.bt, cur.L, min(1, cur.n_tiles - 1));
  load_q(cur);
  store_tile(0);
  __syncthreads();
  int buf = 0;
  bool ids_ready = cur.n_tiles > 1;          // kblk / vblk already hold the block ids of this item's tile 1
  for (;;) {
    const int nit = next_valid(it + 1, nxt);
    const bool has_next = nit * G_ < n_items;
    // an item of one tile: the block ids of the next item's tile 0
    if (!ids_ready && has_next) fetch_bt(nxt.bt, nxt.L, 0);
    const int wq0 = cur.qbase + wrow;
    const int wave_tiles = (cur.ctx0 + min(wq0 + 31, cur.qlen - 1)) / PF_BN + 1;
    f32x4 o[2][DT];
#pragma unroll
    for (int qt = 0; qt < 2; ++qt)
#pragma unroll
      for (int t = 0; t < DT; ++t) o[qt][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m[2] = {-INFINITY, -INFINITY}, l[2] = {0.f, 0.f};
    for (int kt = 0; kt < cur.n_tiles; ++kt) {
      // The tile after this one in the stream (this item's kt + 1, else the next item's tile 0) is loaded
      // while this one computes; then the block ids of the one after it.  Unconditional (at the end of the
      // stream the last tile once more): ids that branches merge are copied, and the copy waits for
      // everything loaded before them, the tile too (whole step, 32 x 512 195 us so and 189 without, 64 x 256
      // 158 and 150).
      const bool last = kt + 1 == cur.n_tiles, loaded = !last || has_next, to_next = last && has_next;
      load_tile(to_next ? nxt.L : cur.L, to_next ? nxt.h : cur.h, to_next ? 0 : min(kt + 1, cur.n_tiles - 1));
      const bool own = kt + 2 < cur.n_tiles || !has_next;
      fetch_bt(own ? cur.bt : nxt.bt, own ? cur.L : nxt.L,
               own ? min(kt + 2, cur.n_tiles - 1) : last ? min(1, nxt.n_tiles - 1) : 0);
      if (kt == 0 && has_next) issue_q(nxt);
      if (kt < wave_tiles) {
        const T* K = lds + buf * 2 * TILE;
        const T* V = K + TILE;
        if ((kt + 1) * PF_BN - 1 > cur.ctx0 + wq0)
          pf_wave_tile<T, D, true>(K, V, qf, o, m, l, qpos, kt * PF_BN, scale_log2, r16, qd);
        else
          pf_wave_tile<T, D, false>(K, V, qf, o, m, l, qpos, kt * PF_BN, scale_log2, r16, qd);
      }
      if (loaded) {
        store_tile(buf ^ 1);
        __syncthreads();
      }
      buf ^= 1;
    }
    const Item done = cur;
    if (has_next) finish_q(nxt);
    const int ln = opaque(lane), rl = ln >> 4, cl = ln & 15;
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      float tot = l[qt];
      tot += __shfl_xor(tot, 16, 64);
      tot += __shfl_xor(tot, 32, 64);
      const float inv = v_scale / tot;
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        Pack4<T> pk;
#pragma unroll
        for (int i = 0; i < 4; ++i) pk.h[i] = from_f<T>(o[qt][t][i] * inv);
        *reinterpret_cast<u32x2*>(rows + (qt * 16 + cl) * D + (((2 * t + (rl >> 1)) ^ cl) * 8) +
                                  4 * (rl & 1)) = pk.u;
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = 4 * i + rl, qi = done.qbase + wrow + row;
      const u32x4 v = *reinterpret_cast<const u32x4*>(rows + row * D + cl * 8);
      if (qi < done.qlen)
        __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(out + ((int64_t)(done.q0 + qi) * nq + done.hg0 + whead) * D +
                                  ((cl ^ (row & 15)) * 8)));
    }
    if (!has_next) break;
    // the next item's first tile is already staged in LDS buffer `buf`
    ids_ready = nxt.n_tiles > 1;
    cur = nxt;
    it = nit;
  }
}

// The walk for 16-bit caches with pages of 32 keys or more: as prefill_attn_gqa_persist_kernel, by workgroups of 4 waves
// (4 heads x 32 queries) of which two share a CU, so that one computes while the other is between two items or waits.
// K and V tiles come by DMA into two buffers each, in the order in which the MFMAs read them: unit c of key k at
// c ^ f(k), V^T in groups of 8 keys as the cache has them; one barrier per tile.  A tile is asked for while the one before
// it computes, its pages a tile before that, the next item's q in registers.  What only items need is read again from the
// arguments: there are no scalar registers left for it.  The order of the items: prefill_items.h.
//
// What bounds it: latency.  At 32 x 512 rows vector instructions issue in 47 % of a SIMD's busy cycles and its matrix core
// works in 24 % (4 x 4096: 54 and 41 %), at 2.4 GHz; LDS reads take 16 %, without conflicts.  The rest is waits.  Per
// MFMA, 32 x 512 takes 1.9 times as long as 4 x 4096: the ends of items (q's rows and rotation, the output rows) and unequal
// workgroups.  K / V write included, the 8-wave walk -> here, us: 32 x 512 187.1 -> 171.6, 64 x 256 152 -> 144, 8 x 2048 401 ->
// 341, 4 x 4096 726 -> 609, 20 x 300 79.3 -> 68.0, 8 x 500 after 3000 285 -> 243.  (Then 344:) items dealt over all XCDs, 8 x 2048
// 362; K by DMA a tile ahead and V within its tile: 373; operands read six steps ahead in the source: 377; indices drawn from a counter: 499.
struct WalkArgs {
  const void *q, *kc, *vc;
  void* out;
  const float* cos_sin;
  const int *block_tables, *qsl, *seq_lens, *work_seq, *work_mblk;
  int64_t q_stride;
  int bt_stride, nq, nkv, bs_log2, num_blocks, cs_rows, n_items;
  float scale_log2, v_scale;
};
// GR = 2: the tiles of one item per workgroup, every other one for each of two groups of 4 waves, whose sums meet at the
// end (the rule: at the launch).
template <typename T, int D, int GR>
__global__ __launch_bounds__(256 * GR, 2) void prefill_attn_walk_kernel(const WalkArgs) {
  static_assert(D == 128 && PF_BN == 64 && sizeof(T) == 2 && PF_BM == 32 * WALK_BLOCKS, "rows and groups per DMA");
  typedef typename Vec8<T>::type V8;
  typedef __attribute__((address_space(3))) void* LdsPtr;
  typedef const __attribute__((address_space(4))) WalkArgs* ArgPtr;
  typedef const __attribute__((address_space(4))) int* ScalarPtr;
  constexpr int GH = 4, QB = 32, KS = D / 32, DT = D / 16, RB = D * 2;   // RB: bytes of a row
  // (objects of their own: the compiler lets an LDS read follow every DMA into the object that it reads)
  constexpr int TE = PF_BN * D;              // elements of a tile
  __shared__ __attribute__((aligned(16))) T K0[GR * TE], K1[GR * TE], V0[GR * TE], V1[GR * TE], all_rows[4 * 16 * D];
  auto args = [] {                           // not kept: see above
    ArgPtr p = (ArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
  };
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wave = GR == 2 ? wv & 3 : wv, group = GR == 2 ? wv >> 2 : 0;
  const int r16 = lane & 15, qd = lane >> 4;
  T* rows = all_rows + wave * 16 * D;        // where 16 output rows meet, to be stored 256 bytes at a time
  // (lane and wave behind an opaque move: what depends on them alone is not kept over the tile loop)
  auto opaque = [](int x) {
    asm volatile("" : "+v"(x));
    return x;
  };
  auto uopaque = [](int x) {
    asm volatile("" : "+s"(x));
    return x;
  };

  // row0, nrow: rows of q; pos0: the first one's position; L: keys; k, v: the kv head's place in page 0
  struct Item {
    int row0, nrow, pos0, head, L, n_tiles;
    const int* bt;
    const char *k, *v;
  };
  auto decode = [&](int idx, Item& I) -> bool {
    const ArgPtr a = args();
    const int nkv = a->nkv, G = a->nq / nkv, Y = nkv * (G / GH), bs_log2 = a->bs_log2;
    int w, z, y;
    walk_item(idx, Y, w, z, y);
    const int h = y / (G / GH);
    const int seq = ((ScalarPtr)a->work_seq)[w], mb = ((ScalarPtr)a->work_mblk)[w];
    const int q0 = ((ScalarPtr)a->qsl)[seq], qlen = ((ScalarPtr)a->qsl)[seq + 1] - q0;
    int L_in = ((ScalarPtr)a->seq_lens)[seq];
    const int cap = a->bt_stride << bs_log2;
    KGC_DCHECK_RANGE(L_in, 0, cap + 1, "prefill seq_len");
    I.L = min(L_in, cap);
    const int ctx0 = I.L - qlen, qbase = mb * PF_BM + z * QB;
    if (qlen <= 0 || ctx0 < 0 || qbase >= qlen) return false;
    I.row0 = q0 + qbase;
    I.nrow = min(qlen - qbase, QB);
    I.pos0 = ctx0 + qbase;
    I.head = h * G + (y % (G / GH)) * GH;
    I.n_tiles = (I.pos0 + I.nrow - 1) / PF_BN + 1;
    I.bt = a->block_tables + (int64_t)seq * a->bt_stride;
    const int64_t at = (int64_t)h * ((int64_t)RB << bs_log2);
    I.k = static_cast<const char*>(a->kc) + at;
    I.v = static_cast<const char*>(a->vc) + at;
    return true;
  };
  const int G_ = gridDim.x, b_ = blockIdx.x, n_items = args()->n_items;
  const bool by_xcd = args()->nq / GH % 8 == 0;
  auto next_valid = [&](int r, Item& I) -> int {
    while (r * G_ < n_items) {
      const int idx = walk_index(r, b_, G_, by_xcd);
      if (idx < n_items && decode(idx, I)) break;
      ++r;
    }
    return r;
  };
  const int bs_log2 = args()->bs_log2, bsm = (1 << bs_log2) - 1;
  const uint32_t page_bytes = (uint32_t)args()->nkv * ((uint32_t)RB << bs_log2);
  // The two pages (or halves of one) of a tile, in even and odd lanes: a scalar load would make every LDS read
  // that is waited for beside it wait for it.
  auto page_ids = [&](const int* bt, int L, int kt) {
    int i = min(kt * PF_BN + 32 * (opaque(lane) & 1), L - 1) >> bs_log2;
    KGC_DCHECK_RANGE(i, 0, args()->bt_stride, "block-table column");
    int v = bt[i];
    KGC_DCHECK_RANGE(v, 0, args()->num_blocks, "block id");
    return v;
  };
  // (buffer loads: behind a flat one every wait is one for everything)
  auto dma = [&](__amdgpu_buffer_rsrc_t src, T* dst, int at) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (LdsPtr)dst, 16, at, 0, 0, 0);
  };
  // DMA u of a wave: keys 16 u + 4 wave .. + 3 of the tile, and half of the group of 8 keys that holds them
  auto ask_k = [&](const char* k, int L, int kt, const uint64_t (&at)[2], T* K, int u) {
    const int w = uopaque(wave), key = min(kt * PF_BN + 16 * u + 4 * w + qd, L - 1);
    const int c = r16 ^ (qd | ((2 * u + (w >> 1)) & 3) << 2);
    const auto src = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(k + at[u >> 1]), 0, RB << bs_log2, 0x00027000);
    dma(src, K + (16 * u + 4 * w) * D, (key & bsm) * RB + c * 16);
  };
  auto ask_v = [&](const char* v, int L, int kt, const uint64_t (&at)[2], T* V, int u) {
    const int w = uopaque(wave), g = 2 * u + (w >> 1), key = min(kt * PF_BN + 8 * g, L - 1) & ~7;
    const auto src = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(v + at[u >> 1]), 0, RB << bs_log2, 0x00027000);
    dma(src, V + g * 8 * D + (w & 1) * 4 * D, (key & bsm) * RB + (w & 1) * 1024 + lane * 16);
  };
  // the wave's 32 rows of q as they are; rows past the last: zeros
  Pack8<T> qn[2][KS];
  auto ask_q = [&](const Item& I) {
    const ArgPtr a = args();
    const int ln = opaque(lane), rs = (int)a->q_stride * 2;
    const auto src = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(static_cast<const char*>(a->q) + ((int64_t)I.row0 * a->q_stride + (int64_t)(I.head + wave) * D) * 2), 0,
        (I.nrow - 1) * rs + RB, 0x00027000);
    const int at = (ln & 15) * rs + (ln >> 4) * 16;
#pragma unroll
    for (int qt = 0; qt < 2; ++qt)
#pragma unroll
      for (int s = 0; s < KS; ++s)
        qn[qt][s].u = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(src, at + qt * 16 * rs + s * 64, 0, 0));
  };
  V8 qf[2][KS];
  int qpos[2];
  auto take_q = [&](const Item& I) {
    const ArgPtr a = args();
    const float* cos_sin = a->cos_sin;
    const int ln = opaque(lane), r16 = ln & 15, qd = ln >> 4;
    PfRot<D> rot[2];
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      qpos[qt] = I.pos0 + min(qt * 16 + r16, I.nrow - 1);
      if (cos_sin != nullptr) pf_issue_rot<D>(cos_sin + (int64_t)min(qpos[qt], a->cs_rows - 1) * D, qd, rot[qt]);
    }
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      if (cos_sin != nullptr) pf_rotate<T, D>(rot[qt], qn[qt]);
#pragma unroll
      for (int s = 0; s < KS; ++s) qf[qt][s] = qn[qt][s].v;
    }
  };

  Item cur, nxt;
  int it = next_valid(0, cur);
  if (it * G_ >= n_items) return;            // uniform: the whole workgroup leaves
  uint64_t at[2];                            // of the tile that computes next
  int id = page_ids(cur.bt, cur.L, group), page[2];       // pages of the one behind it
  auto pages = [&] {
#pragma unroll
    for (int p = 0; p < 2; ++p) page[p] = __builtin_amdgcn_readlane(id, p);
  };
  auto places = [&] {
#pragma unroll
    for (int p = 0; p < 2; ++p) at[p] = (uint64_t)(uint32_t)page[p] * page_bytes;
  };
  pages();
  places();
  ask_q(cur);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    ask_k(cur.k, cur.L, group, at, K0 + group * TE, u);
    ask_v(cur.v, cur.L, group, at, V0 + group * TE, u);
  }
  int nit = next_valid(it + 1, nxt);
  bool has_next = nit * G_ < n_items;
  if (!has_next) nxt = cur;
  id = GR == 2 || cur.n_tiles > 1 ? page_ids(cur.bt, cur.L, group + GR) : page_ids(nxt.bt, nxt.L, 0);
  pages();
  take_q(cur);
  f32x4 o[2][DT];
  float m[2], l[2];
  auto fresh = [&] {
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      // (rows may see none of the second group's keys: no score is below a maximum of the least number, and its sum is 0)
      m[qt] = group == 0 ? -INFINITY : -__FLT_MAX__, l[qt] = 0.f;
#pragma unroll
      for (int t = 0; t < DT; ++t) o[qt][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  fresh();
  const float c = args()->scale_log2;
  int kt = group;
  // One tile, in K and V (or on its way there); the one behind it goes to Kn and Vn.  True after the last tile of the last item.
  auto tile = [&](const T* K, const T* V, T* Kn, T* Vn) -> bool {
    const bool last = GR == 1 && kt + 1 == cur.n_tiles;
    // it is here (the output rows stored behind it need not be there), and everyone is done with the one before it
    if (GR == 1 && kt == 0) pf_meet<8>();
    else pf_meet<0>();
    if (GR == 1 || kt < cur.n_tiles) {
    places();
    if (GR == 1 && kt == 0) ask_q(nxt);
    const bool own = GR == 2 || kt + 2 < cur.n_tiles;
    id = page_ids(own ? cur.bt : nxt.bt, own ? cur.L : nxt.L, own ? kt + 2 * GR : last ? min(1, nxt.n_tiles - 1) : 0);
    // (behind the last item its rows again)
    const char *nk = last ? nxt.k : cur.k, *nv = last ? nxt.v : cur.v;
    const int nL = last ? nxt.L : cur.L, nkt = last ? 0 : kt + GR;
    f32x4 s[2][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const T* krow = K + ((j >> 1) * 32 + 8 * (r16 >> 2) + (r16 & 3) + 4 * (j & 1)) * D;
      f32x4 a0 = {0.f, 0.f, 0.f, 0.f}, a1 = a0;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const V8 f = *reinterpret_cast<const V8*>(krow + (((4 * ks + qd) ^ r16) * 8));
        a0 = mfma16x16x32(f, qf[0][ks], a0);
        a1 = mfma16x16x32(f, qf[1][ks], a1);
      }
      s[0][j] = a0;
      s[1][j] = a1;
      ask_k(nk, nL, nkt, at, Kn, j);         // (one DMA at a time: a burst holds the wave up)
    }
    V8 pf[2][2];
    if ((kt + 1) * PF_BN - 1 > cur.pos0) pf_mask(s, qpos, kt * PF_BN, qd);
    pf_softmax<T, D>(s, pf, o, m, l, c);
#pragma unroll
    for (int t = 0; t < DT; ++t) {
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const V8 f = *reinterpret_cast<const V8*>(V + (4 * kk + qd) * 8 * D + (16 * t + r16) * 8);
        o[0][t] = mfma16x16x32(f, pf[0][kk], o[0][t]);
        o[1][t] = mfma16x16x32(f, pf[1][kk], o[1][t]);
      }
      if (t & 1) ask_v(nv, nL, nkt, at, Vn, t >> 1);
    }
    pages();                                 // (older than the tile's DMAs)
    }
    kt += GR;
    if (GR == 1 ? !last : kt - group < cur.n_tiles) return false;
    if (GR == 2 && cur.n_tiles == 1) {       // the second group has none
      if (group == 1) return true;
    } else if constexpr (GR == 2) {          // the second group's sums join the first one's, by way of its own tiles
      f32x4* const in[4] = {reinterpret_cast<f32x4*>(K0 + TE), reinterpret_cast<f32x4*>(K1 + TE), reinterpret_cast<f32x4*>(V0 + TE),
                            reinterpret_cast<f32x4*>(V1 + TE)};
      f32x4* const ml = reinterpret_cast<f32x4*>(rows) + lane;
      const int to = wave * 64 + lane;
      static_assert(DT == 8 && TE * sizeof(T) == 4 * 256 * sizeof(f32x4), "four sums of a lane per tile");
      pf_meet<0>();
      if (group == 1) {
#pragma unroll
        for (int qt = 0; qt < 2; ++qt)
#pragma unroll
          for (int t = 0; t < DT; ++t) in[2 * qt + (t >> 2)][(t & 3) * 256 + to] = o[qt][t];
        *ml = f32x4{m[0], l[0], m[1], l[1]};
      }
      pf_meet<0>();
      if (group == 1) return true;
      const f32x4 other = *ml;
#pragma unroll
      for (int qt = 0; qt < 2; ++qt) {
        const float mn = __builtin_elementwise_maximum(m[qt], other[2 * qt]);
        const float a0 = __builtin_amdgcn_exp2f(m[qt] - mn), a1 = __builtin_amdgcn_exp2f(other[2 * qt] - mn);
        l[qt] = l[qt] * a0 + other[2 * qt + 1] * a1;
#pragma unroll
        for (int t = 0; t < DT; ++t) o[qt][t] = o[qt][t] * a0 + in[2 * qt + (t >> 2)][(t & 3) * 256 + to] * a1;
      }
    }
    // ---- the item's rows, and the next one's q
    if (GR == 1) take_q(nxt);
    const int ln = opaque(lane), r16 = ln & 15, qd = ln >> 4;
    const ArgPtr a = args();
    const int os = a->nq * RB;
    const auto od = __builtin_amdgcn_make_buffer_rsrc(
        static_cast<char*>(a->out) + (int64_t)cur.row0 * os + (int64_t)(cur.head + wave) * RB, 0, (cur.nrow - 1) * os + RB, 0x00027000);
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      float tot = l[qt];
      tot += __shfl_xor(tot, 16, 64);
      tot += __shfl_xor(tot, 32, 64);
      const float inv = a->v_scale / tot;
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        Pack4<T> pk;
#pragma unroll
        for (int i = 0; i < 4; ++i) pk.h[i] = from_f<T>(o[qt][t][i] * inv);
        *reinterpret_cast<u32x2*>(rows + r16 * D + (((2 * t + (qd >> 1)) ^ r16) * 8) + 4 * (qd & 1)) = pk.u;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {          // rows past the last are not written
        const u32x4 v = *reinterpret_cast<const u32x4*>(rows + (4 * i + qd) * D + r16 * 8);
        __builtin_amdgcn_raw_buffer_store_b128(v, od, (qt * 16 + 4 * i + qd) * os + ((r16 ^ qd) * 16 ^ i * 64), 0, 2);
      }
    }
    if (GR == 2 || !has_next) return true;
    cur = nxt;
    it = nit;
    nit = next_valid(it + 1, nxt);
    has_next = nit * G_ < n_items;
    if (!has_next) nxt = cur;
    if (cur.n_tiles == 1) {                  // (the pages behind it were taken to be its own)
      id = page_ids(nxt.bt, nxt.L, 0);
      pages();
    }
    fresh();
    kt = 0;
    return false;
  };
  if constexpr (GR == 1) {
    while (!tile(K0, V0, K1, V1) && !tile(K1, V1, K0, V0)) {}
  } else {
    T *const Ka = K0 + group * TE, *const Kb = K1 + group * TE, *const Va = V0 + group * TE, *const Vb = V1 + group * TE;
    while (!tile(Ka, Va, Kb, Vb) && !tile(Kb, Vb, Ka, Va)) {}
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);        // DMAs end before the LDS is another's
}

// KGC_PREFILL_GQA=0: the one-head-per-workgroup kernel everywhere (A/B and tests)
static int prefill_gqa_enabled() {
  const char* e = getenv("KGC_PREFILL_GQA");
  return e ? atoi(e) : 1;
}

// KGC_PREFILL_PERSIST=0: the one-shot GQA grid everywhere, =1: the persistent walks (A/B, tests)
static int prefill_persist_mode() {
  const char* e = getenv("KGC_PREFILL_PERSIST");
  return e ? atoi(e) : -1;
}

template <typename T, int D, bool KV8, int GH>
static void prefill_gqa_dispatch(const void* q, void* out, const void* kc, const void* vc,
                                 const int* bt, int bt_stride, const int* qsl, const int* sl,
                                 const int* ws, const int* wm, int n_work, const PromptShape& ps, int nq, int nkv,
                                 int bs_log2, float scale_log2, float v_scale, int num_blocks,
                                 int64_t q_stride, const float* cos_sin, int cs_rows, hipStream_t s) {
  constexpr size_t lds = 2 * 2 * PF_BN * D * sizeof(T);
  const int G = nq / nkv;
  const int64_t n_items = (int64_t)n_work * nkv * (G / GH) * (PF_BM / (256 / GH));
  const int n_cu = device_cus();
  const int mode = prefill_persist_mode();
  auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  const bool dma = aligned(q) && q_stride % 8 == 0;    // 16-byte DMAs
  if constexpr (!KV8) {
    // Few rows of short sequences are one tile each, for which the walk has nothing to overlap (K / V write included, one-shot grid
    // -> walk, us: 2 x 64 rows 14.5 -> 15.6, 1 x 30 16.3 -> 17.2, 8 x 128 20.2 -> 20.1; of many, those of up to 48 rows below 5
    // items per CU: attention alone 20 x 32 9.1 -> 9.8, 32 x 40 10.1 -> 10.7, 48 x 40 16.9 -> 15.9); all else is faster so: 512 rows
    // 31.1 -> 23.2, 1000 51.9 -> 39.1, 2000 after 2000 164 -> 128, 8 x 100 after 3000 127 -> 98, 4 x 300 30.1 -> 27.5.
    const int64_t n = (int64_t)n_work * nkv * (G / 4) * (PF_BM / 32);
    const int64_t table = (int64_t)bt_stride << bs_log2, length = ps.max_len > 0 ? std::min(ps.max_len, table) : table;
    const bool pays = length > 128 || (n > 2 * n_cu && (n > 5 * n_cu || ps.rows > (int64_t)48 * ps.seqs));
    if (dma && aligned(kc) && aligned(vc) && aligned(out) && bs_log2 >= 5 && (mode < 0 ? pays : mode != 0) &&
        n < ((int64_t)1 << 30) && q_stride < (1 << 24) && (int64_t)nq * D < (1 << 24) &&
        ((int64_t)nkv * D << bs_log2) < ((int64_t)1 << 31)) {       // offsets inside an item and a page in 32 bits
      const WalkArgs a{q, kc, vc, out, cos_sin, bt, qsl, sl, ws, wm, q_stride, bt_stride, nq, nkv, bs_log2, num_blocks,
                       cs_rows, (int)n, scale_log2, v_scale};
      // Two groups of waves per item where there is at most one item per CU, or one prompt's are two: its last rows' chain of
      // tiles outlasts the others.  us, one group -> two: 512 rows 27.8 -> 24.8, 1000 39.2 -> 33.0, 300 after 3000 85 -> 62, 4 x 200
      // after 1000 43.4 -> 36.9, 1500 52.6 -> 44.0, 2000 65.0 -> 58.3, 2000 after 2000 125 -> 116; other prompts beyond one item per CU 6 x 256
      // 28.3 -> 33.9, 4 x 500 after 1000 64.7 -> 65.8, 12 x 100 after 1000 56 -> 60; 16 x 128 28.9 -> 34.7, 4096 160 -> 170.
      if (mode < 0 && n <= (ps.seqs == 1 ? 2 : 1) * n_cu) prefill_attn_walk_kernel<T, D, 2><<<(int)n, 512, 0, s>>>(a);
      else prefill_attn_walk_kernel<T, D, 1><<<(int)std::min<int64_t>(n, 2 * n_cu), 256, 0, s>>>(a);
      return;
    }
  }
  // The 8-wave walk pays with more items than CUs (32 x 512 rows, 32 heads: 162 us against 185); with one item
  // per CU or less, twice as many workgroups of half the rows do (8 x 100 rows after 3000: 119 against
  // 128, 512 rows alone 26 against 28, 2000 after 2000 159 against 161).
  // One workgroup per CU: launch_bounds(512, 1), 128 KB of LDS (K / V tiles, the waves' q / output rows).
  const auto walk = &prefill_attn_gqa_persist_kernel<T, D, KV8, GH>;
  if (dma && (mode < 0 ? n_items > n_cu : mode != 0) && n_items < ((int64_t)1 << 30)) {
    walk<<<(int)std::min<int64_t>(n_items, n_cu), 512, 0, s>>>(
        (const T*)q, (T*)out, kc, vc, bt, bt_stride, qsl, sl, ws, wm, nq, nkv, bs_log2,
        scale_log2, v_scale, num_blocks, q_stride, cos_sin, cs_rows, (int)n_items);
    return;
  }
  prefill_attn_gqa_kernel<T, D, KV8, 4><<<nkv * (G / 4) * (PF_BM / 32) * n_work, 256, lds, s>>>(
      (const T*)q, (T*)out, kc, vc, bt, bt_stride, qsl, sl, ws, wm, nq, nkv, bs_log2,
      scale_log2, v_scale, num_blocks, q_stride, cos_sin, cs_rows);
}

template <typename T, int D, bool KV8>
static void prefill_dispatch(const void* q, void* out, const void* kc, const void* vc,
                             const int* bt, int bt_stride, const int* qsl, const int* sl,
                             const int* ws, const int* wm, int n_work, const PromptShape& ps, int nq, int nkv,
                             int bs_log2, float scale_log2, float v_scale, int num_blocks,
                             int64_t q_stride, const float* cos_sin, int cs_rows, hipStream_t s) {
  const int G = nkv > 0 ? nq / nkv : 1;
  if constexpr (D == 128) if (prefill_gqa_enabled() && nq % nkv == 0 && (G == 4 || G % 8 == 0)) {
    if (G == 4)
      prefill_gqa_dispatch<T, D, KV8, 4>(q, out, kc, vc, bt, bt_stride, qsl, sl, ws, wm, n_work, ps,
                                         nq, nkv, bs_log2, scale_log2, v_scale, num_blocks,
                                         q_stride, cos_sin, cs_rows, s);
    else
      prefill_gqa_dispatch<T, D, KV8, 8>(q, out, kc, vc, bt, bt_stride, qsl, sl, ws, wm, n_work, ps,
                                         nq, nkv, bs_log2, scale_log2, v_scale, num_blocks,
                                         q_stride, cos_sin, cs_rows, s);
    return;
  }
  const size_t lds = 2 * 2 * PF_BN * D * sizeof(T);
  prefill_attn_kernel<T, D, KV8><<<dim3(n_work, nq), 256, lds, s>>>(
      (const T*)q, (T*)out, kc, vc, bt, bt_stride, qsl, sl, ws, wm, nq,
      nkv, bs_log2, scale_log2, v_scale, num_blocks, q_stride, cos_sin, cs_rows);
}

void launch_prefill_attention(int dtype, const void* q, void* out, const void* k_cache,
                              const void* v_cache, const int* block_tables, int bt_stride,
                              const int* query_start_loc, const int* seq_lens,
                              const int* work_seq, const int* work_mblk, int n_work, const PromptShape& ps, int nq,
                              int nkv, int D, int bs_log2, float scale, bool kv_fp8,
                              float k_scale, float v_scale, int num_blocks, int64_t q_stride,
                              const float* cos_sin, int cs_rows, hipStream_t s) {
  if (n_work == 0) return;
  const float sl2 = scale * k_scale * 1.4426950408889634f;
#define KGC_PF(TT, DD, K8)                                                                 \
  prefill_dispatch<TT, DD, K8>(q, out, k_cache, v_cache, block_tables, bt_stride,          \
                               query_start_loc, seq_lens, work_seq, work_mblk, n_work, ps, \
                               nq, nkv, bs_log2, sl2, v_scale, num_blocks, q_stride, cos_sin, cs_rows, s)
#define KGC_PF_D(TT, K8) \
  if (D == 128) KGC_PF(TT, 128, K8); else KGC_PF(TT, 64, K8)
  if (dtype == DT_BF16) {
    if (kv_fp8) { KGC_PF_D(bf16, true); } else { KGC_PF_D(bf16, false); }
  } else {
    if (kv_fp8) { KGC_PF_D(f16, true); } else { KGC_PF_D(f16, false); }
  }
#undef KGC_PF_D
#undef KGC_PF
}

int prefill_block_m() { return PF_BM; }

KGC_DEBUG_TU(attention_prefill)

}  // namespace kgc
