// Windowed attention, decode rows of small steps (16-bit activations): a row's keys go to many one-wave
// workgroups, and a second launch puts the pieces together.
//
// A step of few requests has few (row, kv head) pairs -- four workgroups for one request -- and one
// workgroup is bound by the latency of its chain (block table, keys, scores, values, merge: 4 us for the first
// 32 keys of a wave, 3 us for each that follows) and by the 30 to 50 GB/s that one CU draws.
// Per 32-key chunk and wave, with the heads as columns (lane & 15):
//   S^T = K . Q^T   two 16-key tiles, A fragments straight from the cache rows (A row m is key
//                   8 (m >> 2) + (m & 3), + 4 in the second tile),
//   online softmax in fp32, statistics per head in the lane,
//   O^T += V^T . P^T with P^T straight from the S^T accumulators as a pair of values (value +
//                   remainder) and V^T by transposing reads of the value rows in the wave's LDS; where
//                   the values are columns of the key rows (SHARED) the key fragments are what is written.
// The next chunk's rows are in flight while a chunk is computed, its places one chunk before that.
#include <algorithm>

#include "window.h"

namespace kgc {

namespace {

struct SplitArgs {
  const void *q, *k, *v;
  void* out;
  const int *ctx_lens, *dbt;
  float* part;                      // [D][H][Z][dv]
  float2* stat;                     // [D][H][Z]: maximum, sum of weights
  int bt_stride, Tp, H, G, dk, dv, krs, vrs, bs, num_blocks, window, keep_first, Z;
  float scale;
  const float* gate;
  WindowExtra ex;
};

// keys that the row at `pos` sees: ns kept ones, then the span from lo
struct Span { int lo, ns, total; };
__device__ __forceinline__ Span span_of(const SplitArgs& a, int pos) {
  Span s;
  s.lo = first_visible(pos, a.window, a.ex.chunked);
  s.ns = min(a.keep_first, s.lo);
  s.total = s.ns + (pos - s.lo + 1);
  return s;
}

template <typename T, int KS, int DT, bool SHARED>
__global__ __launch_bounds__(64) void window_split_kernel(const SplitArgs a) {
  typedef typename Vec8<T>::type V8;
  constexpr int VST = DT * 16 + 8;                     // elements of a value row in LDS
  constexpr int NV = SHARED ? 1 : DT / 2;
  __shared__ __attribute__((aligned(16))) T vt[32 * VST];
  const int dd = blockIdx.x / a.Z, z = blockIdx.x - dd * a.Z, g = blockIdx.y, qpg = a.H / a.G;
  const int hq0 = blockIdx.z * 16, nh = min(16, qpg - hq0), h0 = g * qpg + hq0;
  const int lane = threadIdx.x, r16 = lane & 15, qd = lane >> 4;
  const int pos = a.ctx_lens[dd] - 1;
  if (pos < 0 || pos >= a.bt_stride * a.bs) return;    // a padding row
  const Span sp = span_of(a, pos);
  const int nch = (sp.total + 31) >> 5;
  if (z >= nch) return;
  const int* bt = a.dbt + (int64_t)dd * a.bt_stride;
  const T* kc = static_cast<const T*>(a.k);
  const T* vc = static_cast<const T*>(a.v);
  const int keyA = 8 * (r16 >> 2) + (r16 & 3);
  const u32x4 zero = {0u, 0u, 0u, 0u};
  auto locate = [&](int ch, int64_t (&row)[2]) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int idx = min(32 * ch + keyA + 4 * j, sp.total - 1);   // clamped: weight 0 below
      const int key = idx < sp.ns ? idx : sp.lo + (idx - sp.ns);
      int b = bt[key / a.bs];
      if (b < 0 || b >= a.num_blocks) b = 0;
      row[j] = ((int64_t)b * a.G + g) * a.bs + key % a.bs;
    }
  };
  auto fetch = [&](const int64_t (&row)[2], u32x4 (&kf)[2][KS], u32x4 (&vf)[2][NV]) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const T* kr = kc + row[j] * a.krs + 8 * qd;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        kf[j][s] = zero;
        if (32 * s + 8 * qd < a.dk) kf[j][s] = *reinterpret_cast<const u32x4*>(kr + 32 * s);
      }
    }
    if constexpr (!SHARED)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const T* vr = vc + row[j] * a.vrs + 8 * qd;
#pragma unroll
        for (int s = 0; s < NV; ++s) {
          vf[j][s] = zero;
          if (32 * s + 8 * qd < a.dv) vf[j][s] = *reinterpret_cast<const u32x4*>(vr + 32 * s);
        }
      }
  };
  int64_t row[2];
  locate(z, row);
  u32x4 kn[2][KS], vn[2][NV];
  fetch(row, kn, vn);
  V8 qf[KS];
  {
    const T* qrow = static_cast<const T*>(a.q) + ((int64_t)(a.Tp + dd) * a.H + h0 + min(r16, nh - 1)) * a.dk;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      u32x4 p = zero;
      if (32 * s + 8 * qd < a.dk) p = *reinterpret_cast<const u32x4*>(qrow + 32 * s + 8 * qd);
      qf[s] = __builtin_bit_cast(V8, p);
    }
  }
  if (z + a.Z < nch) locate(z + a.Z, row);
  float m = z == 0 ? a.ex.sink : -INFINITY;            // (the first wave always has keys)
  float l = qd == 0 && m > -INFINITY ? 1.f : 0.f;
  f32x4 o[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int ch = z; ch < nch; ch += a.Z) {
    u32x4 kf[2][KS], vf[2][NV];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int s = 0; s < KS; ++s) kf[j][s] = kn[j][s];
#pragma unroll
      for (int s = 0; s < NV; ++s) vf[j][s] = vn[j][s];
    }
    if (ch + a.Z < nch) {
      fetch(row, kn, vn);
      if (ch + 2 * a.Z < nch) locate(ch + 2 * a.Z, row);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");         // (the last chunk's values were read)
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int s = 0; s < DT / 2; ++s)
      if (32 * s + 8 * qd < a.dv)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          *reinterpret_cast<u32x4*>(vt + (keyA + 4 * j) * VST + 32 * s + 8 * qd) =
              SHARED ? kf[j][s < KS ? s : 0] : vf[j][SHARED ? 0 : s];
    f32x4 sc[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) acc = mfma16x16x32(__builtin_bit_cast(V8, kf[j][s]), qf[s], acc);
      sc[j] = acc;
    }
    float tmax = -INFINITY;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool ok = 32 * ch + 8 * qd + 4 * j + i < sp.total;
        sc[j][i] = ok ? cap_score(sc[j][i] * a.scale, a.ex.softcap) : -INFINITY;
        tmax = fmaxf(tmax, sc[j][i]);
      }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    const float mn = fmaxf(m, tmax);
    const float alpha = m == -INFINITY ? 0.f : __expf(m - mn);
    m = mn;
    l *= alpha;
    Pack8<T> ph, pl;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float pa = sc[0][i] == -INFINITY ? 0.f : __expf(sc[0][i] - mn);
      const float pb = sc[1][i] == -INFINITY ? 0.f : __expf(sc[1][i] - mn);
      l += pa + pb;
      ph.h[i] = from_f<T>(pa);
      ph.h[4 + i] = from_f<T>(pb);
      pl.h[i] = from_f<T>(pa - to_f(ph.h[i]));
      pl.h[4 + i] = from_f<T>(pb - to_f(ph.h[4 + i]));
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      if (16 * d < a.dv) {
        const T* at = vt + (8 * qd + (r16 >> 2)) * VST + 16 * d + 4 * (r16 & 3);
        const u32x2 v0 = ld_tr4(at), v1 = ld_tr4(at + 4 * VST);
        const V8 fr = __builtin_bit_cast(V8, u32x4{v0[0], v0[1], v1[0], v1[1]});
        f32x4 acc = o[d] * alpha;
        acc = mfma16x16x32(fr, ph.v, acc);
        o[d] = mfma16x16x32(fr, pl.v, acc);
      }
    }
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (r16 < nh) {
    const int64_t at = ((int64_t)dd * a.H + h0 + r16) * a.Z + z;
    if (qd == 0) a.stat[at] = make_float2(m, l);
#pragma unroll
    for (int d = 0; d < DT; ++d)
      if (16 * d + 4 * qd < a.dv) *reinterpret_cast<f32x4*>(a.part + at * a.dv + 16 * d + 4 * qd) = o[d];
  }
}

constexpr int SPLIT_MAX = 256, RNT = 256;

// One workgroup per (row, head): the pieces in groups of dv / 4 lanes, each piece scaled to the common maximum.
template <typename T>
__global__ __launch_bounds__(RNT) void window_split_sum_kernel(const SplitArgs a) {
  __shared__ float ws[RNT / 64][SPLIT_MAX];
  __shared__ __attribute__((aligned(16))) float red[RNT * 4];
  const int dd = blockIdx.x / a.H, h = blockIdx.x - dd * a.H, t = a.Tp + dd;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int pos = a.ctx_lens[dd] - 1;
  T* out = static_cast<T*>(a.out) + (int64_t)t * a.ex.ors + h * a.dv;
  if (pos < 0 || pos >= a.bt_stride * a.bs) {          // a padding row: zeros
    for (int c = tid; c < a.dv; c += RNT) out[c] = from_f<T>(0.f);
    return;
  }
  const int nz = min(a.Z, (span_of(a, pos).total + 31) >> 5);
  const int64_t at = ((int64_t)dd * a.H + h) * a.Z;
  float2 st[SPLIT_MAX / 64];                           // every wave has all statistics
  float M = -INFINITY, L = 0.f;
#pragma unroll
  for (int i = 0; i < SPLIT_MAX / 64; ++i) {
    st[i] = make_float2(-INFINITY, 0.f);
    if (64 * i + lane < nz) st[i] = a.stat[at + 64 * i + lane];
    M = fmaxf(M, st[i].x);
  }
  M = wave_max(M);
#pragma unroll
  for (int i = 0; i < SPLIT_MAX / 64; ++i) {
    const float f = st[i].x == -INFINITY ? 0.f : __expf(st[i].x - M);
    ws[wave][64 * i + lane] = f;
    if (st[i].x != -INFINITY) L += st[i].y * f;
  }
  L = wave_sum(L);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const int lpr = a.dv >> 2, ng = RNT / lpr, grp = tid / lpr, c4 = (tid - grp * lpr) * 4;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  if (grp < ng) {
    const float* p = a.part + at * a.dv + c4;
#pragma unroll 4
    for (int z = grp; z < nz; z += ng) acc += *reinterpret_cast<const f32x4*>(p + (int64_t)z * a.dv) * ws[wave][z];
    *reinterpret_cast<f32x4*>(red + grp * a.dv + c4) = acc;
  }
  __syncthreads();
  const float gt = (a.gate != nullptr ? a.gate[(int64_t)t * a.H + h] : 1.f) * a.ex.out_scale;
  for (int c = tid; c < a.dv; c += RNT) {
    float s = 0.f;
    for (int i = 0; i < min(ng, nz); ++i) s += red[i * a.dv + c];
    out[c] = from_f<T>(s * gt / L * elem_gate<T>(a.ex, t, h * a.dv + c));
  }
}

template <typename T>
void split_dispatch(const SplitArgs& a, int D, hipStream_t s) {
  const dim3 grid(D * a.Z, a.G, (a.H / a.G + 15) / 16);
  const bool shared = a.k == a.v && a.krs == a.vrs && a.dv <= a.dk;
#define KGC_WS(K, D_)                                                                  \
  do {                                                                                 \
    if (shared) window_split_kernel<T, K, D_, true><<<grid, 64, 0, s>>>(a);            \
    else window_split_kernel<T, K, D_, false><<<grid, 64, 0, s>>>(a);                  \
  } while (0)
  if (a.dk <= 128 && a.dv <= 128) KGC_WS(4, 8);
  else if (a.dv <= 192) KGC_WS(8, 12);
  else KGC_WS(8, 16);
#undef KGC_WS
  window_split_sum_kernel<T><<<D * a.H, RNT, 0, s>>>(a);
}

}  // namespace

// Pieces per row, from the longest context where the caller knows it, else from what the tables can hold (the contexts
// are on the device).  The second launch costs 1.5 us and workgroups without keys some more, so steps of few
// keys stay whole where a workgroup has 16 waves for them (128 / 128): up to 6 chunks of 32, 8 where that makes more
// than 768 workgroups and 12 from 1600 on (the CUs hold 1024 and take the rest later).  So do steps with workgroups for a
// quarter of the CUs.  One workgroup per row and kv head -> pieces, us:
//   128 / 128, 4 kv heads, window 1024, 33 (32) pieces whatever the contexts
//     1 x 64, 128, 200, 400, 1000      5.8 -> 7.4, 6.9 -> 7.6, 8.5 -> 7.7, 12.2 -> 7.9, 17.6 -> 7.8
//     8 x 64, 160, 200, 256, 1000      5.8 -> 8.1, 7.6 -> 8.3, 8.4 -> 8.4, 9.1 -> 8.4, 17.4 -> 10.8
//     16 x 64, 256, 320, 400, 1000     5.8 -> 10.9, 9.2 -> 11.2, 10.6 -> 11.5, 12.3 -> 11.6, 18.3 -> 13.4
//   pieces for the longest context: 4 x 160, 256 7.5 -> 7.8, 9.1 -> 7.9; 16 x 200, 256, 320 8.5 -> 8.5, 9.2 -> 9.1, 10.5 -> 9.3
//   long tables: 1 x 8192 84 -> 13.4, 8 x 4000 48 -> 21, 24 x 200 9.8 -> 10.0, 24 x 1000 20.4 -> 19.3, 32 x 2000 31 -> 33
//   256 / 192 latent rows (8 waves, one chunk 4 us)   1 x 20, 128, 1000: 10.9 -> 7.8, 12.9 -> 8.1, 27.2 -> 9.7; 64 x 64,
//                           300, 1000: 11.8 -> 12.2 (9.4 where the contexts are known), 17.5 -> 14.4, 29.3 -> 21.2; 128 x 500: 21.2 -> 22.0
// Waves in all: 2048 (1024 of the wide form, whose registers leave one per SIMD); 16 x 4000 with 1024, 2048, 4096:
// 42.0, 32.8, 33; 64 latent x 1000 with 1024, 2048: 21.2, 25.4.
int window_split_pieces(int D, int H, int G, int dk, int dv, int bt_stride, int bs, int window, int keep_first,
                        int64_t max_ctx) {
  const bool wide = dk > 128 || dv > 128;
  const int64_t wgs = (int64_t)D * G * ((H / G + 15) / 16);
  int64_t keys = (int64_t)bt_stride * bs;
  if (max_ctx > 0) keys = std::min(keys, max_ctx);
  if (window > 0) keys = std::min<int64_t>(keys, (int64_t)window + keep_first);
  const int64_t chunks = (keys + 31) / 32;
  if (wgs > 64 || chunks <= 0) return 0;
  const int64_t pieces = std::min<int64_t>(std::min<int64_t>(chunks, SPLIT_MAX), (wide ? 1024 : 2048) / wgs);
  const int64_t all = wgs * pieces;
  return wide || chunks > (all <= 768 ? 6 : all < 1600 ? 8 : 12) ? (int)pieces : 0;
}

int64_t window_split_floats(int D, int H, int dv, int Z) { return (int64_t)D * H * Z * (dv + 2); }

void launch_window_split(int dtype, void* out, const void* q, const void* k_cache, const void* v_cache,
                         const int* ctx_lens, const int* dbt, int bt_stride, int Tp, int D, int H, int G,
                         int dk, int dv, int krs, int vrs, int bs, int num_blocks, float scale, int window,
                         int keep_first, const float* gate, const WindowExtra& ex, int Z, float* work,
                         hipStream_t s) {
  SplitArgs a{};
  a.q = q; a.k = k_cache; a.v = v_cache; a.out = out;
  a.ctx_lens = ctx_lens; a.dbt = dbt;
  a.part = work;
  a.stat = reinterpret_cast<float2*>(work + (int64_t)D * H * Z * dv);
  a.bt_stride = bt_stride; a.Tp = Tp; a.H = H; a.G = G; a.dk = dk; a.dv = dv; a.krs = krs; a.vrs = vrs;
  a.bs = bs; a.num_blocks = num_blocks; a.window = window; a.keep_first = keep_first; a.Z = Z;
  a.scale = scale; a.gate = gate; a.ex = ex;
  if (dtype == DT_BF16) split_dispatch<bf16>(a, D, s);
  else split_dispatch<f16>(a, D, s);
}

}  // namespace kgc
