// Windowed attention of prompt rows where four query heads share a key/value head (attention_window.hip
// has the other shapes, pooled blocks and rotated values).
//
// A workgroup of 8 waves owns 64 query rows of four heads of one key/value group: a wave has 16 rows
// of two heads, as two MFMA column groups, so every key and value fragment read from LDS serves two
// products and every staged tile four heads.  Both groups see the same keys, and a wave leaves out the
// tiles of which it sees none: under weights of zero a value that is not finite would become NaN, so it
// reaches 16 rows (32 rows of one head per wave: equal times but for short prompts with an element gate, where
// a block of few rows then has fewer sigmoids per SIMD, 8 x 100 rows 18 us against 22).
//
// Key tiles are 64 rows -- first the kept first tokens that lie before the earliest window, then the span
// from that window to the last row -- copied as they lie (16 bytes a lane, rows padded by 8 elements) into
// one of two LDS buffers while the other is computed on; the page numbers are loaded a tile further ahead.
// Per tile and wave, as in the one-head kernel:
//   S^T = K Q^T, visibility, online softmax in fp32 (base 2), O^T += V^T P^T
// with P^T taken from the S^T accumulators as a pair of 16-bit values (value + remainder: the fp32
// weights keep ~16 bits).  V^T fragments come from the row-major tile by transposing LDS reads; where
// the values are columns of the key rows (latent rows) they come from the key tile itself.
//
// The waves of a SIMD take turns between MFMAs (raised priority: 1 % at long prompts, 18 -> 16 us for short
// ones) and the softmax.
//
// What bounds it: 8 x 2048 rows, window 1024, 198 us; the MFMAs (two thirds of them the pairs of P V) work in
// 36 % of a SIMD's cycles and vector instructions, most of them the softmax's, issue in 50 %, overlapping in
// part (capped and causal: 30 % and 73 %; latent rows: 29 % and 40 %).  Not the loads: a ring of four tiles
// filled by LDS-DMA three tiles ahead took 249 us where this took 229.
#include "device.h"
#include "window.h"
#include <type_traits>

namespace kgc {

namespace {

constexpr int BM = 64, BN = 64, HW = 4, NT = 512;     // rows, keys per tile, heads per workgroup

// two weights as value + remainder
template <typename T>
__device__ __forceinline__ void pair2(float a, float b, uint32_t& hi, uint32_t& lo) {
  typedef T T2 __attribute__((ext_vector_type(2)));
  typedef float F2 __attribute__((ext_vector_type(2)));
  const T2 h = __builtin_convertvector((F2{a, b}), T2);
  hi = __builtin_bit_cast(uint32_t, h);
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector((F2{a - (float)h[0], b - (float)h[1]}), T2));
}

// tanh of |y| <= 5/8: y + y^3 p(y^2), p fitted to the least relative error, 4e-9 of tanh.  (1 - 2 / (1 +
// e^(2 y)) has the error of a number near 1 where tanh is small: scores of deviation 2 under a cap of 30
// are off by up to 5.6e-6, 1.5e-6 rms; by 1.2e-6, 1.3e-7 here; by 1.1e-6, 0.9e-7 with a correctly rounded
// tanh.)
__device__ __forceinline__ float tanh_near(float y) {
  const float z = y * y;
  float p = __builtin_fmaf(z, -0.00570531f, 0.02063936f);
  p = __builtin_fmaf(z, p, -0.05373979f);
  p = __builtin_fmaf(z, p, 0.13331443f);
  p = __builtin_fmaf(z, p, -0.33333282f);
  return __builtin_fmaf(y * z, p, y);
}
__device__ __forceinline__ float tanh_far(float y) {
  return 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(y * 2.88539008177792681f));
}

// KS: dk / 32; DT: dv / 16; NJ: 16-key tiles per softmax step (fewer: fewer registers); ALIAS: values
// are the first dv columns of the key rows
template <typename T, int KS, int DT, int NJ, bool ALIAS, bool CAP>
__global__ __launch_bounds__(NT) void window_prefill_gqa_kernel(
    T* __restrict__ out, const T* __restrict__ q, const T* __restrict__ k_cache,
    const T* __restrict__ v_cache, const int* __restrict__ qsl, const int* __restrict__ seq_lens,
    const int* __restrict__ pbt, int bt_stride, const int* __restrict__ work_seq,
    const int* __restrict__ work_blk, int blk_rows, int H, int G, int krs, int vrs, int bs, int bs_shift,
    int num_blocks, float scale, int window, int keep_first, const float* __restrict__ gate,
    WindowExtra ex) {
  typedef typename Vec8<T>::type V8;
  constexpr int DK = KS * 32, DV = DT * 16, KST = DK + 8, VST = ALIAS ? KST : DV + 8;
  constexpr int NKU = BN * DK / 8 / NT, NVU = ALIAS ? 0 : BN * DV / 8 / NT;
  constexpr bool SAME = !ALIAS && DK == DV;           // a thread's key and value units: the same rows
  static_assert(BN * DK / 8 % NT == 0 && BN * DV / 8 % NT == 0, "whole units per thread");
  constexpr float LOG2E = 1.44269504088896340736f;
  extern __shared__ __align__(16) char smem[];
  T* Kb = reinterpret_cast<T*>(smem);                 // [2][BN][KST]
  T* Vb = ALIAS ? Kb : Kb + 2 * BN * KST;             // [2][BN][VST]
  // head groups run fastest: workgroups are dealt round-robin over the XCDs, so every XCD sees all
  // row blocks of its heads
  const int item = blockIdx.y / (blk_rows / BM), sub = blockIdx.y % (blk_rows / BM);
  const int seq = work_seq[item];
  const int q0 = qsl[seq], qlen = qsl[seq + 1] - q0, ctx0 = seq_lens[seq] - qlen;
  const int r0 = work_blk[item] * blk_rows + sub * BM;
  if (r0 >= qlen || ctx0 < 0) return;
  const int rows = min(BM, qlen - r0);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r16 = lane & 15, qd = lane >> 4;
  const int g = blockIdx.x * HW / (H / G);
  // column group c's head: c is swapped from one row group to the next, so that the waves write (and read
  // the gates of) all four heads at a time (1 %)
  auto head = [&](int c) { return (int)blockIdx.x * HW + 2 * (wave & 1) + (c ^ (wave >> 1 & 1)); };
  const int* bt = pbt + (int64_t)seq * bt_stride;
  const int wr = r0 + 16 * (wave >> 1);               // the wave's first row
  const int myrow = wr + r16, qpos = ctx0 + myrow;
  const bool rowok = myrow < qlen;
  const int row_lo = first_visible(qpos, window, ex.chunked);
  V8 qf[2][KS];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const T* qrow = q + ((int64_t)(q0 + min(myrow, qlen - 1)) * H + head(c)) * DK + 8 * qd;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      Pack8<T> t;
      t.u = *reinterpret_cast<const u32x4*>(qrow + 32 * s);
      qf[c][s] = t.v;
    }
  }
  f32x4 o[2][DT];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int t = 0; t < DT; ++t) o[c][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m[2], l[2];
  m[0] = m[1] = ex.sink * LOG2E;
  l[0] = l[1] = qd == 0 && ex.sink > -INFINITY ? 1.f : 0.f;
  const int p_min = ctx0 + r0, p_max = ctx0 + r0 + rows - 1;
  const int lo_min = first_visible(p_min, window, ex.chunked);
  const int ns = window > 0 ? min(keep_first, lo_min) : 0;
  const int nsink = (ns + BN - 1) / BN, ntile = nsink + (p_max - lo_min + BN) / BN;
  // the wave's own span of visible keys (tiles outside it are staged but not computed)
  const int wp_lo = ctx0 + wr, wp_hi = min(wp_lo + 15, p_max);
  const int w_lo = first_visible(wp_lo, window, ex.chunked);
  const int w_lo_hi = first_visible(wp_hi, window, ex.chunked);
  const bool live = wr < r0 + rows;

  auto first_key = [&](int t) { return t < nsink ? t * BN : lo_min + (t - nsink) * BN; };
  auto end_key = [&](int t, int kb) { return min(t < nsink ? ns : p_max + 1, kb + BN); };
  // a staging unit: 16 bytes of one key (value) row; keys past the end read the last one (their
  // weights are zero)
  int pgk[NKU], pgv[NVU > 0 ? NVU : 1];
  u32x4 rk[NKU], rv[NVU > 0 ? NVU : 1];
  auto unit_key = [&](int u, int per, int kb, int hi) { return min(kb + u / per, hi - 1); };
  auto pages = [&](int t) {
    const int kb = first_key(t), hi = end_key(t, kb);
#pragma unroll
    for (int i = 0; i < NKU; ++i) {
      const int key = unit_key(tid + NT * i, DK / 8, kb, hi);
      pgk[i] = bt[bs_shift >= 0 ? key >> bs_shift : key / bs];
    }
    if constexpr (!SAME)
#pragma unroll
      for (int i = 0; i < NVU; ++i) {
        const int key = unit_key(tid + NT * i, DV / 8, kb, hi);
        pgv[i] = bt[bs_shift >= 0 ? key >> bs_shift : key / bs];
      }
  };
  auto cache_row = [&](int key, int bl) -> int64_t {
    const int in = bs_shift >= 0 ? key & (bs - 1) : key % bs;
    if (bl < 0 || bl >= num_blocks) bl = 0;
    return (int64_t)(bl * G + g) * bs + in;
  };
  auto fetch = [&](int t) {
    const int kb = first_key(t), hi = end_key(t, kb);
#pragma unroll
    for (int i = 0; i < NKU; ++i) {
      const int u = tid + NT * i;
      const int64_t row = cache_row(unit_key(u, DK / 8, kb, hi), pgk[i]);
      rk[i] = *reinterpret_cast<const u32x4*>(k_cache + row * krs + u % (DK / 8) * 8);
      if constexpr (SAME) rv[i] = *reinterpret_cast<const u32x4*>(v_cache + row * vrs + u % (DV / 8) * 8);
    }
#pragma unroll
    for (int i = 0; i < (SAME ? 0 : NVU); ++i) {
      const int u = tid + NT * i;
      rv[i] = *reinterpret_cast<const u32x4*>(
          v_cache + cache_row(unit_key(u, DV / 8, kb, hi), pgv[i]) * vrs + u % (DV / 8) * 8);
    }
  };
  auto park = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NKU; ++i) {
      const int u = tid + NT * i;
      *reinterpret_cast<u32x4*>(Kb + (buf * BN + u / (DK / 8)) * KST + u % (DK / 8) * 8) = rk[i];
    }
#pragma unroll
    for (int i = 0; i < NVU; ++i) {
      const int u = tid + NT * i;
      *reinterpret_cast<u32x4*>(Vb + (buf * BN + u / (DV / 8)) * VST + u % (DV / 8) * 8) = rv[i];
    }
  };

  const float sl = CAP ? scale / ex.softcap : scale * LOG2E;
  const float fl = CAP ? ex.softcap * LOG2E : sl;  // what is left to multiply (> 0: see the launcher)
  pages(0);
  fetch(0);
  pages(min(1, ntile - 1));
  park(0);
  __syncthreads();
  for (int tile = 0; tile < ntile; ++tile) {
    const int buf = tile & 1;
    if (tile + 1 < ntile) {                  // in flight while this tile is computed
      fetch(tile + 1);
      pages(min(tile + 2, ntile - 1));
    }
    const bool sink = tile < nsink;
    const int kb = first_key(tile), hi = end_key(tile, kb);
    const T* Kt = Kb + buf * BN * KST;
    const T* Vt = Vb + buf * BN * VST;
    for (int st = 0; st < BN / 16 / NJ; ++st) {
      const int k0 = kb + st * 16 * NJ, k1 = k0 + 16 * NJ;         // this step's keys
      // nothing of them is visible to the wave's rows (kept first tokens can sit in a main tile
      // when the earliest window starts before them)
      if (!live || k0 > wp_hi || k0 >= hi || (!sink && min(hi, k1) <= w_lo && k0 >= keep_first)) continue;
      __builtin_amdgcn_s_setprio(1);
      f32x4 s[2][NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        s[0][j] = s[1][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        const T* krow = Kt + ((st * NJ + j) * 16 + r16) * KST + 8 * qd;
#pragma unroll
        for (int d = 0; d < KS; ++d) {
          Pack8<T> fr;
          fr.u = *reinterpret_cast<const u32x4*>(krow + 32 * d);
          s[0][j] = mfma16x16x32(fr.v, qf[0][d], s[0][j]);
          s[1][j] = mfma16x16x32(fr.v, qf[1][d], s[1][j]);
        }
      }
      __builtin_amdgcn_s_setprio(0);
      // keys that all are there, not after the wave's first row and inside the window of its last
      // are seen by every row: no test per element
      const bool full = k1 <= hi && k1 - 1 <= wp_lo && k0 >= w_lo_hi && wp_lo + 15 == wp_hi;
      V8 ph[2][NJ / 2], pl[2][NJ / 2];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        // (whole loops under each uniform test: a branch per element costs more than its work)
        if constexpr (CAP) {                 // tanh(score / cap); scores beyond 5/8 of the cap are rare
          float far = 0.f;
#pragma unroll
          for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              s[c][j][i] *= sl;
              far = fmaxf(far, fabsf(s[c][j][i]));
            }
          if (__any(far > 0.625f)) {
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const float y = s[c][j][i], near = tanh_near(y);
                float t = tanh_far(y);
                asm("" : "+v"(t));           // (no branch per element)
                s[c][j][i] = fabsf(y) > 0.625f ? t : near;
              }
          } else {
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
              for (int i = 0; i < 4; ++i) s[c][j][i] = tanh_near(s[c][j][i]);
          }
        }
        if (!full) {
          const int last = min(hi - 1, qpos) - k0 - 4 * qd, low = row_lo - k0 - 4 * qd,
                    kept = keep_first - k0 - 4 * qd;
#pragma unroll
          for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int key = 16 * j + i;
              const bool vis = (key <= last) & ((key >= low) | (key < kept)) & rowok;
              s[c][j][i] = vis ? s[c][j][i] : -INFINITY;
            }
        }
        float mx = -INFINITY;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[c][j][i]);
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * fl;
        const float mn = fmaxf(m[c], mx), ref = mn == -INFINITY ? 0.f : mn;
        if (__any(mn > m[c])) {
          const float alpha = __builtin_amdgcn_exp2f(m[c] - ref);
          m[c] = mn;
          l[c] *= alpha;
#pragma unroll
          for (int t = 0; t < DT; ++t) o[c][t] *= alpha;
        }
        float sum = 0.f;
#pragma unroll
        for (int kk = 0; kk < NJ / 2; ++kk) {
          u32x4 wh, wl;
#pragma unroll
          for (int i = 0; i < 4; ++i) {      // elements 0..3: tile 2 kk, 4..7: tile 2 kk + 1
            const int j = 2 * kk + (i >> 1), e = 2 * (i & 1);
            const float a = __builtin_amdgcn_exp2f(__builtin_fmaf(s[c][j][e], fl, -ref));
            const float b = __builtin_amdgcn_exp2f(__builtin_fmaf(s[c][j][e + 1], fl, -ref));
            sum += a + b;
            uint32_t x, y;
            pair2<T>(a, b, x, y);
            wh[i] = x;
            wl[i] = y;
          }
          ph[c][kk] = __builtin_bit_cast(V8, wh);
          pl[c][kk] = __builtin_bit_cast(V8, wl);
        }
        l[c] += sum;
      }
      __builtin_amdgcn_s_setprio(1);
      // ---- O^T += V^T P^T: lane (r16, qd) holds column 16 t + r16 of keys 4 qd .. and 16 + 4 qd ..
#pragma unroll
      for (int t = 0; t < DT; ++t) {
#pragma unroll
        for (int kk = 0; kk < NJ / 2; ++kk) {
          const T* vrow = Vt + ((st * NJ + 2 * kk) * 16 + 4 * qd + (r16 >> 2)) * VST + 16 * t + 4 * (r16 & 3);
          const u32x2 a = ld_tr4(vrow), b = ld_tr4(vrow + 16 * VST);
          const V8 fr = __builtin_bit_cast(V8, (u32x4{a[0], a[1], b[0], b[1]}));
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            o[c][t] = mfma16x16x32(fr, pl[c][kk], o[c][t]);
            o[c][t] = mfma16x16x32(fr, ph[c][kk], o[c][t]);
          }
        }
      }
      __builtin_amdgcn_s_setprio(0);
    }
    if (tile + 1 < ntile) {
      park(buf ^ 1);
      __syncthreads();                       // the next tile is there; this one was read
    }
  }
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    float ls = l[c] + __shfl_xor(l[c], 16, 64);
    ls += __shfl_xor(ls, 32, 64);
    if (!rowok || !live) continue;
    const int64_t t = q0 + myrow;
    const int h = head(c);
    const float gt = (gate != nullptr ? gate[t * H + h] : 1.f) * ex.out_scale;
    const float inv = ls > 0.f ? gt / ls : 0.f;
    T* orow = out + t * ex.ors + h * DV + 4 * qd;
    // the element gate, four columns at a time where its rows allow it
    const T* eg = static_cast<const T*>(ex.egate);
    if (eg != nullptr) {
      eg += t * ex.egs + h * DV + 4 * qd;
      if ((reinterpret_cast<uintptr_t>(eg) & 7) == 0) {
        Pack4<T> e[DT];
#pragma unroll
        for (int d = 0; d < DT; ++d) e[d].u = *reinterpret_cast<const u32x2*>(eg + 16 * d);
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[c][d][i] *= 1.f / (1.f + expf(-to_f(e[d].h[i])));
      } else {
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[c][d][i] *= 1.f / (1.f + expf(-to_f(eg[16 * d + i])));
      }
    }
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      Pack4<T> w;
#pragma unroll
      for (int i = 0; i < 4; ++i) w.h[i] = from_f<T>(o[c][d][i] * inv);
      *reinterpret_cast<u32x2*>(orow + 16 * d) = w.u;
    }
  }
}

template <typename T, int KS, int DT, int NJ, bool ALIAS, bool CAP>
bool run(T* out, const T* q, const T* kc, const T* vc, const int* qsl, const int* seq_lens, const int* pbt,
         int bt_stride, const int* work_seq, const int* work_blk, int n_work, int blk_rows, int H, int G,
         int krs, int vrs, int bs, int num_blocks, float scale, int window, int keep_first, const float* gate,
         const WindowExtra& ex, hipStream_t s) {
  constexpr size_t lds = sizeof(T) * 2 * BN * (KS * 32 + 8 + (ALIAS ? 0 : DT * 16 + 8));
  const auto kernel = &window_prefill_gqa_kernel<T, KS, DT, NJ, ALIAS, CAP>;
  static OncePerDevice once;
  if (!allow_lds(once, kernel, lds)) return false;
  const int shift = (bs & (bs - 1)) == 0 ? __builtin_ctz(bs) : -1;
  kernel<<<dim3(H / HW, n_work * (blk_rows / BM)), NT, lds, s>>>(
      out, q, kc, vc, qsl, seq_lens, pbt, bt_stride, work_seq, work_blk, blk_rows, H, G, krs, vrs, bs, shift,
      num_blocks, scale, window, keep_first, gate, ex);
  return true;
}

template <typename T, bool CAP, typename... A>
bool dispatch(int dk, int dv, bool alias, T* out, const T* q, const T* kc, const T* vc, A... a) {
  if (dk == 128 && dv == 128 && !alias) return run<T, 4, 8, 4, false, CAP>(out, q, kc, vc, a...);
  if (dk == 256 && dv == 192 && alias) return run<T, 8, 12, 2, true, CAP>(out, q, kc, vc, a...);
  return false;
}

}  // namespace

bool launch_window_prefill_gqa(int dtype, void* out, const void* q, const void* kc, const void* vc,
                               const int* qsl, const int* seq_lens, const int* pbt, int bt_stride,
                               const int* work_seq, const int* work_blk, int n_work, int blk_rows, int H,
                               int G, int dk, int dv, int krs, int vrs, int bs, int num_blocks, float scale,
                               int window, int keep_first, const float* gate, const WindowExtra& ex,
                               hipStream_t s) {
  // Four heads on one staged tile against one head per workgroup (bf16, 16 heads on 4 key/value heads): window
  // 1024 with 8 x 2048 rows 355 -> 198 us, causal and capped 577 -> 290, 48 rows after 3000 83 -> 68; latent rows
  // (one key/value head), 32 x 512 rows 380 -> 129 us, 4 x 2000 after 500 974 -> 390.  Up to 16 prompts of 33 to
  // 64 rows without context are slower, a wave having two heads of its one tile (8 x 64: 11.0 -> 11.8, capped
  // 16.2 -> 17.7, latent 12.8 -> 15.8); with 300 tokens of context they are faster (34.8 -> 27.3, 52.6 -> 35.9,
  // 47.4 -> 38.3), and the context is known on the device only.  The maximum is taken before
  // the scale, which has to be positive for that.
  if (n_work <= 0 || !(scale > 0.f) || H / G % HW != 0 || ex.pool > 0 || ex.vtab != nullptr ||
      blk_rows % BM != 0)
    return false;
  const bool alias = kc == vc && krs == vrs;
  auto go = [&](auto cap, auto* o) {
    typedef std::remove_pointer_t<decltype(o)> T;
    return dispatch<T, decltype(cap)::value>(dk, dv, alias, o, (const T*)q, (const T*)kc, (const T*)vc, qsl, seq_lens,
                                             pbt, bt_stride, work_seq, work_blk, n_work, blk_rows, H, G, krs, vrs,
                                             bs, num_blocks, scale, window, keep_first, gate, ex, s);
  };
  const bool capped = ex.softcap > 0.f;
  if (dtype == DT_BF16) return capped ? go(std::true_type(), (bf16*)out) : go(std::false_type(), (bf16*)out);
  if (dtype == DT_F16) return capped ? go(std::true_type(), (f16*)out) : go(std::false_type(), (f16*)out);
  return false;
}

}  // namespace kgc
