// Windowed attention of prompt rows where four query heads share a key/value head (attention_window.hip
// has the other shapes, pooled blocks and rotated values).
//
// A workgroup of 8 waves owns 64 query rows of four heads of one key/value group: a wave has 16 rows
// of two heads, the 32 columns of its MFMAs, so every key and value fragment read from LDS serves two
// heads and every staged tile four.  Both heads see the same keys, and a wave leaves out the
// tiles of which it sees none: under weights of zero a value that is not finite would become NaN, so it
// reaches 16 rows (32 rows of one head per wave: equal times but for short prompts with an element gate, where
// a block of few rows then has fewer sigmoids per SIMD).
//
// Key tiles are 64 rows -- first the kept first tokens that lie before the earliest window, then the span
// from that window to the last row -- copied as they lie (16 bytes a lane, rows padded by 8 elements) into
// one of two LDS buffers while the other is computed on; the page numbers are loaded a tile further ahead.
// Per tile and wave:
//   S^T = K Q^T, visibility, online softmax in fp32 (base 2), O^T += V^T P^T
// with P^T taken from the S^T accumulators as a pair of 16-bit values (value + remainder: the fp32
// weights keep ~16 bits).  V^T fragments come from the row-major tile by transposing LDS reads; where
// the values are columns of the key rows (latent rows) they come from the key tile itself.
//
// What bounds it: instruction issue.  MFMAs of 32 x 32 x 16 leave six vector instructions' time beside each (two
// of 16 x 16 x 32, the same work: four), so the next keys' weights, the maximum and the next tile's addresses stand
// between them in the order given below.  8 x 2048 rows, window 1024: per tile and wave 48 MFMAs and 380 vector
// instructions, in bf16 70 more where the maximum moves, 4000 cycles of two waves' issue of the 5800 that a tile
// takes; the rest is the barrier, and 3.5 rounds of workgroups that take 4.  bf16, in MFMAs of 16 x 16 x 32 -> so, us:
// 197 -> 179 to 184, 32 x 512 rows 90 -> 76, latent rows 124 -> 110 to 116, capped and causal with a gate 290 -> 261.
// (A ring of four tiles filled by LDS-DMA three tiles ahead: 249 us where this took 229.)
//
// That is ROWS64, one workgroup to a CU.  A step that does not fill the chip with them, or fills it just beyond a round, is
// bound by one workgroup's chain of tiles, 4 us each; two forms shorten it.  ROWS32: 4 waves own 32 rows, two workgroups
// to a CU (3 us for a tile where a workgroup has the CU for itself).  ROWS32X2: 8 waves own 32 rows, and of the tiles each
// 4 waves take every other one; their sums meet at the end.  Both copy tiles by DMA into unpadded buffers, without the
// registers and the instructions that eight units per thread would take (by registers: capped ones spill, latent rows
// at 32 rows 142 us where DMA takes 115).  Figures: at the rule below.
#include "device.h"
#include "chunk.h"
#include "window.h"
#include <algorithm>
#include <type_traits>

namespace kgc {

namespace {

enum { ROWS64, ROWS32, ROWS32X2 };                    // forms: see above
constexpr int BN = 64, HW = 4;                        // keys per tile, heads per workgroup

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

// KS: dk / 16; DT: dv / 32; NB: blocks of 32 keys per softmax step (fewer: fewer registers); ALIAS: values
// are the first dv columns of the key rows
template <typename T, int KS, int DT, int NB, bool ALIAS, bool CAP, int FORM>
__global__ __launch_bounds__(FORM == ROWS32 ? 256 : 512, 2) void window_prefill_gqa_kernel(
    T* __restrict__ out, const T* __restrict__ q, const T* __restrict__ k_cache,
    const T* __restrict__ v_cache, const int* __restrict__ qsl, const int* __restrict__ seq_lens,
    const int* __restrict__ pbt, int bt_stride, const int* __restrict__ work_seq,
    const int* __restrict__ work_blk, int blk_rows, int H, int G, int krs, int vrs, int bs, uint32_t bs_inv,
    int num_blocks, float scale, int window, int keep_first, const float* __restrict__ gate,
    WindowExtra ex) {
  typedef typename Vec8<T>::type V8;
  typedef __attribute__((address_space(3))) void* LdsPtr;
  constexpr bool DMA = FORM != ROWS64;
  constexpr int BM = DMA ? 32 : 64, NT = 512, GR = FORM == ROWS32X2 ? 2 : 1;   // GR: groups of 4 waves by DMA
  constexpr int DK = KS * 16, DV = DT * 32, KST = DMA ? DK : DK + 8, VST = ALIAS ? KST : DMA ? DV : DV + 8;
  constexpr int RPD = 512 / DK, NKD = BN / 4 / RPD, NVD = ALIAS ? 0 : NKD, LR = BN + RPD;   // rows per DMA, DMAs per wave and tile
  static_assert(!DMA || ((RPD == 4 && (ALIAS || DK == DV)) || (RPD == 2 && ALIAS)), "rows of a DMA");
  constexpr int NKU = BN * DK / 8 / NT, NVU = ALIAS ? 0 : BN * DV / 8 / NT;
  constexpr bool SAME = !ALIAS && DK == DV;           // a thread's key and value units: the same rows
  static_assert(BN * DK / 8 % NT == 0 && BN * DV / 8 % NT == 0, "whole units per thread");
  constexpr float LOG2E = 1.44269504088896340736f;
  // The maximum that weights refer to moves when a score passes it by more than FAR.  f16: weights up to 2^8 and few
  // rescalings of the sums.  bf16: always, since a pair of bf16 holds 17 bits of a weight, and all of the largest one
  // where that is 1: of 8 x 1024 rows 0.221 % of the results are not the exact ones' rounding so, 0.239 % where the maximum
  // stays 2^8 behind.  (f16, whose sums' own rounding counts: 0.165 % and 0.149 %.)  The sums then move in most tiles, so
  // they are scaled beside the first products of P V, whether they have to be or not: 4 x 300 rows after 2000 57.2 us where
  // the maximum stays behind, 59.2 with the scaling in a branch before the weights, 57.5 so; 32 x 512 76.0, 77.7, 76.6; 8 x
  // 2048, where the clock gives way, 184, 189, 187; latent 4 x 2000 after 500 165, 174, 173.
  constexpr float FAR = 8.f;
  constexpr bool EXACT = __is_same(T, bf16);
  extern __shared__ __align__(16) char smem[];
  // (objects of their own: the compiler lets an LDS read follow every DMA into the object that it reads)
  __shared__ __align__(16) T K0[DMA ? GR * LR * DK : 8], K1[DMA ? GR * LR * DK : 8],
      V0[DMA && NVD ? GR * LR * DV : 8], V1[DMA && NVD ? GR * LR * DV : 8];
  T* Kb = reinterpret_cast<T*>(smem);                 // [2][BN][KST]
  T* Vb = ALIAS ? Kb : Kb + 2 * BN * KST;             // [2][BN][VST]
  // head groups run fastest: workgroups are dealt round-robin over the XCDs, so every XCD sees all
  // row blocks of its heads
  const int hg = blockIdx.x, item = blockIdx.y / (blk_rows / BM), sub = blockIdx.y % (blk_rows / BM);
  const int seq = work_seq[item];
  const int q0 = qsl[seq], qlen = qsl[seq + 1] - q0, ctx0 = seq_lens[seq] - qlen;
  const int r0 = work_blk[item] * blk_rows + sub * BM;
  if (r0 >= qlen || ctx0 < 0) return;
  const int rows = min(BM, qlen - r0);
  const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, col = lane & 31, hh = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), wave = GR == 2 ? wv & 3 : wv, group = GR == 2 ? wv >> 2 : 0;
  const int g = hg * HW / (H / G);
  // a lane's column: a row of one of the wave's two heads (which is swapped from one row group to the next,
  // so that the waves write, and read the gates of, all four heads at a time: 1 %)
  const int head = hg * HW + 2 * (wave & 1) + ((col >> 4) ^ (wave >> 1 & 1));
  const int* bt = pbt + (int64_t)seq * bt_stride;
  const int wr = r0 + 16 * (wave >> 1);               // the wave's first row
  const int myrow = wr + r16, qpos = ctx0 + myrow;
  const bool rowok = myrow < qlen;
  const int row_lo = first_visible(qpos, window, ex.chunked);
  V8 qf[KS];
  {
    const T* qrow = q + ((int64_t)(q0 + min(myrow, qlen - 1)) * H + head) * DK + 8 * hh;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = __builtin_bit_cast(V8, *reinterpret_cast<const u32x4*>(qrow + 16 * s));
  }
  f32x16 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[t][i] = 0.f;
  float m = group == 0 ? ex.sink * LOG2E : -INFINITY, l = group == 0 && hh == 0 && ex.sink > -INFINITY ? 1.f : 0.f;
  // (tiles start where those of 64 rows do, so that both forms have the same results)
  const int p_min = ctx0 + (r0 & ~63), p_max = ctx0 + r0 + rows - 1;
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
  int pgk[NKU], ink[NKU], pgv[NVU > 0 ? NVU : 1], inv_[NVU > 0 ? NVU : 1];
  u32x4 rk[NKU], rv[NVU > 0 ? NVU : 1];
  // (whatever the page size, without a branch: it would end the region that the loads are placed in)
  auto page = [&](uint32_t key, int hi, int& pg, int& in) {
    key = min(key, (uint32_t)hi - 1);
    uint32_t at = __umulhi(key, bs_inv), r = key - at * bs;        // bs_inv = (2^32 - 1) / bs: at most one too few
    if (r >= (uint32_t)bs) {
      ++at;
      r -= bs;
    }
    pg = bt[at];
    in = r;
  };
  auto pages = [&](int t) {
    const int kb = first_key(t), hi = end_key(t, kb);
#pragma unroll
    for (int i = 0; i < NKU; ++i) page(kb + (tid + NT * i) / (DK / 8), hi, pgk[i], ink[i]);
    if constexpr (!SAME)
#pragma unroll
      for (int i = 0; i < NVU; ++i) page(kb + (tid + NT * i) / (DV / 8), hi, pgv[i], inv_[i]);
  };
  // element offset of a key's row, page by page (products of 32 bits each: a multiply-add)
  const uint32_t kpage = (uint32_t)G * bs * krs, vpage = (uint32_t)G * bs * vrs;
  auto place = [&](int bl, int in, uint32_t page, uint32_t stride) -> int64_t {
    if ((uint32_t)bl >= (uint32_t)num_blocks) bl = 0;
    return (uint64_t)(uint32_t)bl * page + (uint64_t)(uint32_t)(g * bs + in) * stride;
  };
  auto fetch = [&]() {                       // of the keys that pages() was last called for
#pragma unroll
    for (int i = 0; i < NKU; ++i) {
      const int u = tid + NT * i;
      rk[i] = *reinterpret_cast<const u32x4*>(k_cache + place(pgk[i], ink[i], kpage, krs) + u % (DK / 8) * 8);
      if constexpr (SAME)
        rv[i] = *reinterpret_cast<const u32x4*>(v_cache + place(pgk[i], ink[i], vpage, vrs) + u % (DV / 8) * 8);
    }
#pragma unroll
    for (int i = 0; i < (SAME ? 0 : NVU); ++i) {
      const int u = tid + NT * i;
      rv[i] = *reinterpret_cast<const u32x4*>(v_cache + place(pgv[i], inv_[i], vpage, vrs) + u % (DV / 8) * 8);
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

  // ---- tiles by DMA, RPD rows at a time that lie in one page: a tile's rows from the one before its first key whose
  // position is a multiple of RPD.  The unit c of 16 bytes of row k lies at c ^ f(k), f(k) = (k & 3) << 2 | (k >> 2 & 3): neither
  // the reads of 16 rows at one unit nor the transposing ones of 4 rows at four units meet in a bank.  Rows past the last
  // key are zeros (as are their weights).  Of the i-th RPD rows lane i keeps the place, from the head's first page
  // on, and the bytes that there are (0 past the last tile).
  int idn = 0, inn = 0, left = 0, bytes = 0;          // n: page and row in it, of the tile after the next
  uint32_t off0 = 0, off1 = 0;
  const int rb = krs * (int)sizeof(T);                // (values, if they are others, at the same places of theirs)
  auto page_ids = [&](int t) {
    const int kb = first_key(t), hi = end_key(t, kb), key = (kb & -RPD) + RPD * lane;
    left = t < ntile ? min(hi - key, RPD) : 0;
    page(key, hi, idn, inn);
  };
  auto take_pages = [&] {
    const uint64_t at = (uint64_t)((uint32_t)idn < (uint32_t)num_blocks ? idn : 0) * kpage + (uint64_t)(uint32_t)inn * (uint32_t)krs;
    off0 = (uint32_t)(at << 1);
    off1 = (uint32_t)(at >> 31);
    bytes = max(left, 0) * rb;
  };
  auto dma = [&](__amdgpu_buffer_rsrc_t src, T* dst, int off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (LdsPtr)dst, 16, off, 0, 0, 0);
  };
  const char *kg = reinterpret_cast<const char*>(k_cache + (int64_t)g * bs * krs), *vg = reinterpret_cast<const char*>(v_cache + (int64_t)g * bs * krs);
  const int rr = lane / (64 / RPD), row0 = RPD * wave + rr, lane_at = rr * rb + ((lane % (64 / RPD)) ^ ((row0 & 3) << 2 | (row0 >> 2 & 3))) * 16;
  // DMA u of the tile that take_pages() was last called for (rows 4 RPD u further: the unit's bit 1 turned over
  // where that is an odd multiple of 8)
  auto ask = [&](const char* from, T* dst, int u) {
    const int n = 4 * u + wave;
    const uint64_t at = (uint64_t)__builtin_amdgcn_readlane(off1, n) << 32 | (uint32_t)__builtin_amdgcn_readlane(off0, n);
    const auto src = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(from + at), 0, __builtin_amdgcn_readlane(bytes, n), 0x00027000);
    dma(src, dst + RPD * n * DK, RPD == 2 ? lane_at ^ (u & 1) * 32 : lane_at);
  };
  auto ask_k = [&](T* K, int u) { ask(kg, K, u); };
  auto ask_v = [&](T* V, int u) { ask(vg, V, u); };
  // where the operands lie: 8 elements of S^T's key row and depth 16 d, 4 of V^T's key row + .. and column 32 t .., from the
  // lane's place in bytes (by DMA its unit's bits are turned over)
  auto k_at = [&](const T* Kt, int ka, int row, int d) {
    const char* at = reinterpret_cast<const char*>(Kt + row * KST);
    if constexpr (!DMA) return at + ka + 32 * d;
    else return at + (ka ^ (d & 7) * 32) + (d >> 3) * 256;
  };
  auto v_at = [&](const T* Vt, int va, int row, int half, int t) {
    const char* at = reinterpret_cast<const char*>(Vt + (row + 8 * half) * VST);
    if constexpr (!DMA) return reinterpret_cast<const T*>(at + va + 64 * t);
    else return reinterpret_cast<const T*>(at + (va ^ ((t & 3) * 64 + half * 32)) + (t >> 2) * 256);
  };

  const float sl = CAP ? scale / ex.softcap : scale * LOG2E;
  const float fl = CAP ? ex.softcap * LOG2E : sl;  // what is left to multiply (> 0: see the launcher)
  // One tile, in Kt and Vt (by DMA: or on its way there; the one behind it goes to Kn and Vn)
  auto compute = [&](int tile, const T* Kt, const T* Vt, T* Kn, T* Vn) {
    // in flight while this tile is computed (the last one again at the end); where a tile is one step, the
    // addresses are made beside the products of S
    const auto next = [&] {
      if constexpr (!DMA) {
        fetch();
        pages(min(tile + 2, ntile - 1));
      }
    };
    if (!DMA && NB != 2 && tile + 1 < ntile) next();
    const bool sink = tile < nsink;
    const int kb = first_key(tile), hi = end_key(tile, kb);
#pragma unroll
    for (int st = 0; st < BN / 32 / NB; ++st) {
      const int k0 = kb + st * 32 * NB, k1 = k0 + 32 * NB;         // this step's keys
      // nothing of them is visible to the wave's rows (kept first tokens can sit in a main tile
      // when the earliest window starts before them)
      if (!live || k0 > wp_hi || k0 >= hi || (!sink && min(hi, k1) <= w_lo && k0 >= keep_first)) {
        if (NB == 2) next();
        if constexpr (DMA)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            ask_k(Kn, st * 4 + u);
            if (NVD) ask_v(Vn, u);
          }
        continue;
      }
      int ka, va;
      if constexpr (DMA) {
        const int off = kb & (RPD - 1), kr = col + off, vr = 4 * hh + (r16 >> 2) + off;
        ka = (kr * DK + (hh ^ ((kr & 3) << 2 | (kr >> 2 & 3))) * 8) * 2;
        va = (vr * VST + ((2 * (col >> 4) + (r16 >> 1 & 1)) ^ ((vr & 3) << 2 | (vr >> 2 & 3))) * 8 + 4 * (r16 & 1)) * 2;
        if (KS == 16) {                      // for want of registers: not kept over the tiles
          asm volatile("" : "+v"(ka));
          asm volatile("" : "+v"(va));
        }
      } else {
        ka = (col * KST + 8 * hh) * 2;
        va = ((4 * hh + (r16 >> 2)) * VST + 16 * (col >> 4) + 4 * (r16 & 3)) * 2;
      }
      f32x16 s[NB];
      float mx = -INFINITY;
      __builtin_amdgcn_sched_barrier(0);
      if (NB == 2 && CAP) next();
      if constexpr (NB == 2 && !CAP) {
        // S^T, four products at a time and the operands of the next four on their way; beside the first ones the next
        // tile's addresses and loads (operands read just in time: 8 x 2048 189.3 -> 187.5 us, 1 x 8192 130 -> 126)
        V8 kf[2][4];
        auto load_k = [&](int g) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            kf[g & 1][i] = __builtin_bit_cast(V8, *reinterpret_cast<const u32x4*>(k_at(Kt, ka, 32 * (st * NB + g * 4 / KS), g * 4 % KS + i)));
        };
        static_assert(KS % 4 == 0, "");
        load_k(0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int g = 0; g < NB * KS / 4; ++g) {
          const int b = g * 4 / KS;
          if (g + 1 < NB * KS / 4) load_k(g + 1);
          if (g == 0) next();
          if (g * 4 % KS == 0)
#pragma unroll
            for (int i = 0; i < 16; ++i) s[b][i] = 0.f;
#pragma unroll
          for (int i = 0; i < 4; ++i) s[b] = mfma32x32x16(kf[g & 1][i], qf[g * 4 % KS + i], s[b]);
          if (g == KS / 4 + 1)
#pragma unroll
            for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[0][i]);
          __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
          if constexpr (DMA) ask_k(Kn, g);
          interleave<4, 8, 0, DMA ? 4 : 1>();
          __builtin_amdgcn_sched_barrier(0);
        }
      } else
#pragma unroll
      for (int b = 0; b < NB; ++b) {         // S^T; beside a block's products the maximum of the one before it
#pragma unroll
        for (int i = 0; i < 16; ++i) s[b][i] = 0.f;
#pragma unroll
        for (int d = 0; d < KS; ++d)
          s[b] = mfma32x32x16(__builtin_bit_cast(V8, *reinterpret_cast<const u32x4*>(k_at(Kt, ka, 32 * (st * NB + b), d))), qf[d], s[b]);
        if constexpr (DMA)
#pragma unroll
          for (int u = 0; u < 4 / NB; ++u) ask_k(Kn, st * 4 + b * (4 / NB) + u);
        if (!CAP && b > 0)
#pragma unroll
          for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[b - 1][i]);
        // (whole loops under each uniform test: a branch per element costs more than its work)
        if constexpr (CAP) {                 // tanh(score / cap); scores beyond 5/8 of the cap are rare
          constexpr int CG = NB == 1 ? 4 : 16;            // at a time: registers
#pragma unroll
          for (int i0 = 0; i0 < 16; i0 += CG) {
            float far = 0.f;
#pragma unroll
            for (int i = i0; i < i0 + CG; ++i) {
              s[b][i] *= sl;
              far = fmaxf(far, fabsf(s[b][i]));
            }
            if (__any(far > 0.625f)) {
#pragma unroll
              for (int i = i0; i < i0 + CG; ++i) {
                const float y = s[b][i], near = tanh_near(y);
                float t = tanh_far(y);
                asm("" : "+v"(t));           // (no branch per element)
                s[b][i] = fabsf(y) > 0.625f ? t : near;
                if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
              }
            } else {
#pragma unroll
              for (int i = i0; i < i0 + CG; ++i) s[b][i] = tanh_near(s[b][i]);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      // keys that all are there, not after the wave's first row and inside the window of its last
      // are seen by every row: no test per element
      const bool full = k1 <= hi && k1 - 1 <= wp_lo && k0 >= w_lo_hi && wp_lo + 15 == wp_hi;
      if (!full) {
        const int last = min(hi - 1, qpos) - k0 - 4 * hh, low = row_lo - k0 - 4 * hh,
                  kept = keep_first - k0 - 4 * hh;
        mx = -INFINITY;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int key = 32 * b + 8 * (i >> 2) + (i & 3);
            const bool vis = (key <= last) & ((key >= low) | (key < kept)) & rowok;
            s[b][i] = vis ? s[b][i] : -INFINITY;
            if (!CAP && b + 1 < NB) mx = fmaxf(mx, s[b][i]);
          }
      }
#pragma unroll
      for (int b = CAP ? 0 : NB - 1; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[b][i]);
      {
        const auto both = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, mx), __builtin_bit_cast(uint32_t, mx), false, false);
        const uint32_t x = both[0], y = both[1];
        mx = fmaxf(__builtin_bit_cast(float, x), __builtin_bit_cast(float, y)) * fl;
      }
      float alpha = 1.f;
      if constexpr (EXACT) {
        const float mn = fmaxf(m, mx);
        alpha = __builtin_amdgcn_exp2f(m - (mn == -INFINITY ? 0.f : mn));
        m = mn;
        l *= alpha;
        o[0] *= alpha;
      } else if (__any(mx > m + FAR)) {
        const float mn = fmaxf(m, mx);
        alpha = __builtin_amdgcn_exp2f(m - (mn == -INFINITY ? 0.f : mn));
        m = mn;
        l *= alpha;
#pragma unroll
        for (int t = 0; t < DT; ++t) o[t] *= alpha;
      }
      const float ref = m == -INFINITY ? 0.f : m;
      // weights of 16 keys: the parts of a B operand as the accumulators lie
      V8 ph[2 * NB], pl[2 * NB];
      auto weigh = [&](int j) {
        u32x4 wh, wl;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float a = __builtin_amdgcn_exp2f(__builtin_fmaf(s[j >> 1][8 * (j & 1) + 2 * i], fl, -ref));
          const float c = __builtin_amdgcn_exp2f(__builtin_fmaf(s[j >> 1][8 * (j & 1) + 2 * i + 1], fl, -ref));
          l += a + c;
          uint32_t x, y;
          pair2<T>(a, c, x, y);
          wh[i] = x;
          wl[i] = y;
        }
        ph[j] = __builtin_bit_cast(V8, wh);
        pl[j] = __builtin_bit_cast(V8, wl);
      };
      weigh(0);
      __builtin_amdgcn_sched_barrier(0);
      // ---- O^T += V^T P^T, 16 keys at a time, the next ones' weights beside the products: lane (col, hh) holds
      // column 32 t + col of keys 4 hh .. and 8 + 4 hh ..
      // values one product ahead where registers are left: 8 x 2048 187.8 -> 181.7 us, capped 263 -> 254
      constexpr bool AHEAD = NB == 2;
      V8 vf[2];
      auto load_v = [&](int n) {             // 16 keys n / DT, columns n % DT
        const int row = 32 * NB * st + 16 * (n / DT);
        const u32x2 a = ld_tr4(v_at(Vt, va, row, 0, n % DT)), b = ld_tr4(v_at(Vt, va, row, 1, n % DT));
        vf[n & 1] = __builtin_bit_cast(V8, (u32x4{a[0], a[1], b[0], b[1]}));
      };
      if (AHEAD) {
        load_v(0);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int j = 0; j < 2 * NB; ++j) {
        if (j + 1 < 2 * NB) weigh(j + 1);
        if constexpr (DMA && NVD > 0) ask_v(Vn, j);
#pragma unroll
        for (int t = 0; t < DT; ++t) {
          const int n = j * DT + t;
          if (!AHEAD) load_v(n);
          else if (n + 1 < 2 * NB * DT) load_v(n + 1);
          o[t] = mfma32x32x16(vf[n & 1], pl[j], o[t]);
          o[t] = mfma32x32x16(vf[n & 1], ph[j], o[t]);
          if (EXACT && j == 0 && t + 1 < DT) o[t + 1] *= alpha;
        }
#pragma unroll
        for (int t = 0; t < DT; ++t) {
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (EXACT && j == 0) __builtin_amdgcn_sched_group_barrier(0x002, NB == 2 ? 12 : 8, 0);
          else __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (EXACT && j == 0) __builtin_amdgcn_sched_group_barrier(0x002, NB == 2 ? 12 : 8, 0);
          else __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  if constexpr (DMA) {
    auto rest = [&](int t, T* K, T* V) {     // the last rows of a tile that starts between two multiples of RPD
      if (wave == 0 && (first_key(t) & (RPD - 1)) != 0) {
        ask_k(K, NKD);
        if (NVD) ask_v(V, NKD);
      }
    };
    T *Ka = K0 + group * LR * DK, *Kz = K1 + group * LR * DK, *Va = ALIAS ? Ka : V0 + group * LR * DV, *Vz = ALIAS ? Kz : V1 + group * LR * DV;
    page_ids(group);
    take_pages();
    page_ids(group + GR);
#pragma unroll
    for (int u = 0; u < NKD; ++u) {
      ask_k(Ka, u);
      if (NVD) ask_v(Va, u);
    }
    rest(group, Ka, Va);
    take_pages();
    auto step = [&](int t, const T* K, const T* V, T* Kn, T* Vn) {
      meet<0>();                             // it is here, and everyone is done with the one before it
      page_ids(t + 2 * GR);
      rest(t + GR, Kn, Vn);
      if (GR == 1 || t < ntile) compute(t, K, V, Kn, Vn);
      take_pages();                          // (older than the tile's DMAs)
    };
    for (int t = 0; t < ntile; t += 2 * GR) {
      step(t + group, Ka, Va, Kz, Vz);
      if (t + GR < ntile) step(t + GR + group, Kz, Vz, Ka, Va);
    }
    if constexpr (GR == 1) {
      __builtin_amdgcn_s_waitcnt(0x0f70);    // DMAs end before the LDS is another's
    } else if (ntile == 1) {                 // the second group has none
      __builtin_amdgcn_s_waitcnt(0x0f70);
      if (group == 1) return;
    } else {                                 // the second group's sums join the first one's
      constexpr int N0 = DT == 4 ? 2 : 4;    // column blocks in K0; then K1
      static_assert(GR * LR * DK * sizeof(T) >= N0 * 16384 && GR * LR * DK * sizeof(T) >= (DT - N0) * 16384 + 2048, "");
      auto sums = [&](int t, int k) {
        return reinterpret_cast<f32x4*>(t < N0 ? K0 : K1) + ((t < N0 ? t : t - N0) * 4 + k) * 256 + (tid & 255);
      };
      float2* const ml = reinterpret_cast<float2*>(reinterpret_cast<char*>(K1) + (DT - N0) * 16384) + (tid & 255);
      meet<0>();
      if (group == 1) {
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int k = 0; k < 4; ++k) *sums(t, k) = f32x4{o[t][4 * k], o[t][4 * k + 1], o[t][4 * k + 2], o[t][4 * k + 3]};
        *ml = make_float2(m, l);
      }
      meet<0>();
      if (group == 1) return;
      const float2 other = *ml;
      const float mn = fmaxf(m, other.x), ref = mn == -INFINITY ? 0.f : mn;
      const float a0 = __builtin_amdgcn_exp2f(m - ref), a1 = __builtin_amdgcn_exp2f(other.x - ref);
      l = l * a0 + other.y * a1;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const f32x4 x = *sums(t, k);
#pragma unroll
          for (int i = 0; i < 4; ++i) o[t][4 * k + i] = o[t][4 * k + i] * a0 + x[i] * a1;
        }
    }
  } else {
    pages(0);
    fetch();
    pages(min(1, ntile - 1));
    park(0);
    __syncthreads();
    for (int t = 0; t < ntile; ++t) {
      const int buf = t & 1;
      compute(t, Kb + buf * BN * KST, Vb + buf * BN * VST, nullptr, nullptr);
      if (t + 1 < ntile) {
        park(buf ^ 1);
        __syncthreads();                     // the next tile is there; this one was read
      }
    }
  }
  l += __shfl_xor(l, 32, 64);
  if (!live) return;
  const int64_t t = q0 + min(myrow, qlen - 1);
  const float gt = (gate != nullptr ? gate[t * H + head] : 1.f) * ex.out_scale;
  const float inv = l > 0.f ? gt / l : 0.f;
  T* orow = out + t * ex.ors + head * DV;
  // the element gate, four columns at a time where its rows allow it
  const T* eg = static_cast<const T*>(ex.egate);
  if (eg != nullptr) {
    eg += t * ex.egs + head * DV + 4 * hh;
    if (__all((reinterpret_cast<uintptr_t>(eg) & 7) == 0)) {
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        Pack4<T> e[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) e[k].u = *reinterpret_cast<const u32x2*>(eg + 32 * d + 8 * k);
#pragma unroll
        for (int i = 0; i < 16; ++i) o[d][i] *= gate_sigmoid(to_f(e[i >> 2].h[i & 3]));
      }
    } else {
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[d][i] *= gate_sigmoid(to_f(eg[32 * d + 8 * (i >> 2) + (i & 3)]));
    }
  }
  // the halves of the wave trade columns: 16 bytes of a row per lane
  const bool wide = ((reinterpret_cast<uintptr_t>(out) | (uintptr_t)(ex.ors * sizeof(T))) & 15) == 0;
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int k = 0; k < 4; k += 2) {
      Pack4<T> x, y;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x.h[i] = from_f<T>(o[d][4 * k + i] * inv);
        y.h[i] = from_f<T>(o[d][4 * k + 4 + i] * inv);
      }
      const auto p0 = __builtin_amdgcn_permlane32_swap(x.u[0], y.u[0], false, false);
      const auto p1 = __builtin_amdgcn_permlane32_swap(x.u[1], y.u[1], false, false);
      T* to = orow + 32 * d + 8 * (k + hh);
      if (rowok) {
        if (wide) {
          *reinterpret_cast<u32x4*>(to) = u32x4{p0[0], p1[0], p0[1], p1[1]};
        } else {
          *reinterpret_cast<u32x2*>(to) = u32x2{p0[0], p1[0]};
          *reinterpret_cast<u32x2*>(to + 4) = u32x2{p0[1], p1[1]};
        }
      }
    }
}

template <typename T, int KS, int DT, int NB, bool ALIAS, bool CAP>
bool run(T* out, const T* q, const T* kc, const T* vc, const int* qsl, const int* seq_lens, const int* pbt,
         int bt_stride, const int* work_seq, const int* work_blk, int n_work, int blk_rows, int H, int G,
         int krs, int vrs, int bs, int num_blocks, float scale, int window, int keep_first, const float* gate,
         const WindowExtra& ex, const PromptShape& ps, hipStream_t s) {
  const int64_t wgs = (int64_t)(H / HW) * n_work * (blk_rows / 32);
  int64_t span = (int64_t)bt_stride * bs;
  if (ps.max_len > 0) span = std::min(span, ps.max_len);
  if (window > 0) span = std::min<int64_t>(span, (int64_t)window + keep_first + 64);
  auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  // 16-byte units of rows of one page per DMA, keys and values at the same places
  const bool dma = bs % (512 / (KS * 16)) == 0 && aligned(kc) && aligned(vc) && krs % 8 == 0 && krs == vrs && krs < 1 << 20 &&
                   n_work <= 65535 / (blk_rows / 32);
  auto go = [&](auto form) {
    constexpr int F = decltype(form)::value;
    const auto kernel = &window_prefill_gqa_kernel<T, KS, DT, NB, ALIAS, CAP, F>;
    constexpr size_t lds = F != ROWS64 ? 0 : sizeof(T) * 2 * BN * (KS * 16 + 8 + (ALIAS ? 0 : DT * 32 + 8));
    static OncePerDevice once;
    if (lds > 0 && !allow_lds(once, kernel, lds)) return false;
    kernel<<<dim3(H / HW, n_work * (blk_rows / (F == ROWS64 ? 64 : 32))), F == ROWS32 ? 256 : 512, lds, s>>>(
        out, q, kc, vc, qsl, seq_lens, pbt, bt_stride, work_seq, work_blk, blk_rows, H, G, krs, vrs, bs, 0xffffffffu / (uint32_t)bs,
        num_blocks, scale, window, keep_first, gate, ex);
    return true;
  };
  // In bf16, ROWS64 -> here, us (16 heads on 4 unless it says latent).
  // With no more workgroups of 32 rows than CUs two groups for each: window 1024, 1 x 512 rows 26.6 -> 18.9, 1 x 2048 55.3 -> 38.0,
  // 4 x 300 after 2000 57.8 -> 37.3, 1 x 60 after 3000 57.5 -> 36.1, causal and capped 1 x 100 after 4000 229 -> 137, latent 2 x 1000
  // 77.3 -> 49.1.  Three tiles at most: one group (4 x 64 8.9 -> 7.5, two groups 9.4; 2 x 100 10.8 -> 9.4; latent 4 x 64 12.2 -> 9.7, 13.0);
  // ROWS64 itself where a prompt ends in a block of at most 35 rows, the waves of the others being idle there (1 x 30
  // 7.0, 7.3 by one group; 20 after 160 11.2, 11.9; 2 x 150 11.4, 12.1).
  // Without a window a prompt's rows have one tile to as many as its length, and the longest rows' chain lasts past the
  // others: two groups up to two rounds for prompts of 500 rows and more (capped 1 x 3000 175 -> 113, 2 x 1500 92 -> 59, 2 x 2048 114 ->
  // 88, 4 x 1000 67.5 -> 55; 8 x 500 after 2000 161 -> 161), of which fewer lose: 16 x 140 13.8 -> 21.8, 10 x 256 19.0 -> 20.4, 31 x 106
  // after 3583 221 -> 243; windowed 1 x 3000 61 -> 65.
  // Beyond, one group where 64 rows each are no more than 11/8 of a round, of windowed prompts or ones of up to 128 rows: window
  // 1024, 1 x 5000 103 -> 90, 12 x 300 23.4 -> 22.0, 7 x 546 after 1500 107 -> 91 (2 x 2500 69.2 -> 70.6), causal 40 x 100 24.4 -> 22.4, 36 x
  // 128 32.1 -> 23.2, 40 x 60 after 2000 208 -> 189.  Where the last round is fuller two workgroups to a CU are no faster than one
  // of twice the rows (24 x 300 38.0 -> 41, 6 x 1000 capped 66.4 -> 67.5), and of longer causal prompts as many lose as gain: 5 x 1000
  // 56.6 -> 52, 3 x 2134 104 -> 94, but 2 x 2500 111 -> 117, 5 x 1000 after 1000 124 -> 131, capped 17 x 181 21.8 -> 23.6, 1 x 6000 after
  // 1000 369 -> 402.
  // Latent rows beyond one round: 32 x 250 50.7 -> 48.4, 5 x 1000 83 -> 73, 4 x 2048 155 -> 142, 8 x 2048 260 -> 254, 80 x 64 48 -> 36 (16 x
  // 380 46.1 -> 47.2, 12 x 512 54.2 -> 55); but causal 1 x 8000 613 -> 641.  Within one: 1 x 4096 86 -> 89, 30 x 100 17.5 -> 18.8.
  const int64_t n_cu = device_cus(), mean = ps.rows / std::max(1, ps.seqs);
  // blocks of 64 rows that have rows: of the last 128 of a prompt the second 64 have none where those rows are 64 at most
  const double tail = 128. - ((double)n_work * blk_rows - (double)ps.rows) / std::max(1, ps.seqs);
  const int64_t full = (H / HW) * (int64_t)(n_work * (blk_rows / 64) - ps.seqs * std::min(1., std::max(0., 0.5 + (64 - tail) / 16)));
  const bool pairs = wgs <= n_cu ? span > 192 : wgs <= 2 * n_cu && window <= 0 && mean >= 500;
  const bool ends = KS == 16 || mean > 192 || (mean - 1) % 64 >= 35;
  const bool spare = wgs / 2 > n_cu && (KS == 16 ? window > 0 || mean <= 6000 || full > 2 * n_cu
                                                 : ends && 8 * full <= 11 * n_cu && span <= 4096 && (window > 0 || mean <= 128));
  const int form = !dma ? ROWS64 : pairs ? ROWS32X2 : (wgs <= n_cu && ends) || spare ? ROWS32 : ROWS64;
  if (form == ROWS32X2) return go(std::integral_constant<int, ROWS32X2>());
  if (form == ROWS32) return go(std::integral_constant<int, ROWS32>());
  return go(std::integral_constant<int, ROWS64>());
}

template <typename T, bool CAP, typename... A>
bool dispatch(int dk, int dv, bool alias, T* out, const T* q, const T* kc, const T* vc, A... a) {
  if (dk == 128 && dv == 128 && !alias) return run<T, 8, 4, 2, false, CAP>(out, q, kc, vc, a...);
  if (dk == 256 && dv == 192 && alias) return run<T, 16, 6, 1, true, CAP>(out, q, kc, vc, a...);
  return false;
}

}  // namespace

bool launch_window_prefill_gqa(int dtype, void* out, const void* q, const void* kc, const void* vc,
                               const int* qsl, const int* seq_lens, const int* pbt, int bt_stride,
                               const int* work_seq, const int* work_blk, int n_work, int blk_rows, int H,
                               int G, int dk, int dv, int krs, int vrs, int bs, int num_blocks, float scale,
                               int window, int keep_first, const float* gate, const WindowExtra& ex,
                               const PromptShape& ps, hipStream_t s) {
  // Four heads on one staged tile against one head per workgroup (bf16, 16 heads on 4 key/value heads): window
  // 1024 with 8 x 2048 rows 355 -> 182 us, causal and capped 577 -> 261, 48 rows after 3000 83 -> 54; latent rows
  // (one key/value head), 32 x 512 rows 380 -> 116 us; 8 x 64 rows 11.0 -> 10.2, latent 12.8 -> 12.4.  The maximum
  // is taken before the scale, which has to be positive for that.
  if (n_work <= 0 || !(scale > 0.f) || H / G % HW != 0 || ex.pool > 0 || ex.vtab != nullptr ||
      blk_rows % 64 != 0)
    return false;
  if ((int64_t)G * bs * std::max(krs, vrs) >= (int64_t)1 << 32) return false;   // pages are 32-bit factors of the offsets
  const bool alias = kc == vc && krs == vrs;
  auto go = [&](auto cap, auto* o) {
    typedef std::remove_pointer_t<decltype(o)> T;
    return dispatch<T, decltype(cap)::value>(dk, dv, alias, o, (const T*)q, (const T*)kc, (const T*)vc, qsl, seq_lens,
                                             pbt, bt_stride, work_seq, work_blk, n_work, blk_rows, H, G, krs, vrs,
                                             bs, num_blocks, scale, window, keep_first, gate, ex, ps, s);
  };
  const bool capped = ex.softcap > 0.f;
  if (dtype == DT_BF16) return capped ? go(std::true_type(), (bf16*)out) : go(std::false_type(), (bf16*)out);
  if (dtype == DT_F16) return capped ? go(std::true_type(), (f16*)out) : go(std::false_type(), (f16*)out);
  return false;
}

}  // namespace kgc
