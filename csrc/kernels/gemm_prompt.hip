// act(x W^T) of prompt rows on the matrix cores: the feed-forward's first projection with its activation, so that
// the projection's output, two to three times as wide as the model, is neither written nor read again.
//     SILU: W = gate | up [2 I, K], out [M, I] = silu(x gate^T) * (x up^T);   XIELU: out [M, N] = xIELU(x W^T)
//
// A workgroup of 4 waves, one per SIMD, owns 256 rows x 256 columns of the product (SILU: 128 gates and the same 128
// ups), a wave 128 x 128 of them in 256 accumulator registers: 8 + 8 operands for 64 MFMAs.  Per step of 64 columns of K
// the rows of x and W come by DMA as whole lines (8 rows of 128 bytes per instruction: half lines ask the L2 twice and
// cost a fifth), unit c of row r at c ^ (r & 7).  x's operands of a whole step are read during the second half of the step
// before it, so that the rows of x two steps ahead arrive in the first half of a step and those of W in the second,
// evenly; a barrier follows each half and waits for what was asked for two halves before, not for the newest.
// One workgroup per CU walks over the tiles, and the steps run on across them: the next tile's first rows arrive
// during the last steps and its outputs' conversion.  The MFMAs are written with their accumulators tied: left to the
// compiler, 256 of 256 accumulators in flight are copied around (half the rate).
//
// What bounds it: the power limit at long K (8192^3 plain products 1.58 PFLOP/s at 1.79 GHz, the library 1.60), the
// outputs' conversion besides at K = 2048, beside which the matrix cores idle (one wave per SIMD): of 419 us of XIELU about 70.
// Library and activation launch -> here, us: 14336 x 2048 -> 2 x 5504 SILU 566 -> 459, 14336 x 2048 -> 8256 XIELU 467 -> 419,
// 16384 x 4096 -> 2 x 14336 SILU 2746 -> 2540.  (The activations are those of their own launches, to the bit; a quotient by
// v_rcp and a series of two terms took 442 and 398 us and were less exact.)  A last round of few tiles goes over the CUs in
// pieces (plan_of).
#include <type_traits>

#include "activation.h"
#include "common.h"
#include "device.h"
#include "launch.h"

namespace kgc {

namespace {

constexpr int NTHR = 256, BK = 64;           // threads, columns of K per step
constexpr int BT = 256;                      // rows and weight rows of a whole tile
constexpr int GROUP = 8;                     // row tiles that neighbouring workgroups share the weights of

struct PromptArgs {
  const void *x, *w;
  void* out;
  const float* ab;                           // XIELU's two parameters
  int M, N, K, ldx, ldo, wrows;              // N: output columns; wrows: rows of w
  int tm, tn;                                // tiles
  int whole, pieces;                         // tiles walked as a whole; 1, 2 or 4 pieces of each that follows
};

// c += a b, in place.  (The compiler does not see an MFMA here: whoever reads c waits for it, settle.)
template <typename T> __device__ __forceinline__ void mfma_tied(f32x4& c, typename Vec8<T>::type a, typename Vec8<T>::type b) {
  if constexpr (std::is_same_v<T, bf16>) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
template <typename T> __device__ __forceinline__ void mfma_new(f32x4& c, typename Vec8<T>::type a, typename Vec8<T>::type b) {
  if constexpr (std::is_same_v<T, bf16>) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
}
// 24 wait states (an MFMA of eight passes wants 11 before its result is read)
__device__ __forceinline__ void settle(f32x4& a, f32x4& b, f32x4& c, f32x4& d) {
  asm volatile("s_nop 15\n\ts_nop 7" : "+a"(a), "+a"(b), "+a"(c), "+a"(d));
}

// a barrier that leaves the newest N memory operations on their way
template <int N> __device__ __forceinline__ void meet() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt((N & 15) | (N >> 4) << 14 | 0x70);   // vmcnt(N) lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Walks over tiles (or pieces) of 2 MT x 2 NT 16-row tiles, MT x NT per wave: numbers first, first + step, .. < count.
template <typename T, int ACT, int MT, int NT>
__device__ __forceinline__ void walk(const PromptArgs& g, T* x0, T* x1, T* w0, T* w1, T* out_rows, int first, int step, int count) {
  typedef typename Vec8<T>::type V8;
  typedef __attribute__((address_space(3))) void* LdsPtr;
  constexpr bool SILU = ACT == PROMPT_SILU;
  constexpr int CW = NT * 16 / (SILU ? 2 : 1), CN = 2 * CW;       // output columns of a wave, of the workgroup
  constexpr int U = CW / 8, R = 64 / U, NS = MT * U / 4;          // 16-byte units of its rows, rows per store, stores
  constexpr int PM = 16 / (2 * MT), PN = 16 / (2 * NT);           // pieces of a tile
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, qd = lane >> 4, wm = wave >> 1, wn = wave & 1;
  const int rowb = g.K * 2, nk = g.K / BK;
  auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  auto uniform64 = [](const void* p) -> char* {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    return reinterpret_cast<char*>((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32 |
                                   (uint32_t)__builtin_amdgcn_readfirstlane((int)v));
  };
  // Piece `at`: its first row and output column.  Tiles run down GROUP row tiles before the next column.
  auto place = [&](int at, int& m0, int& n0) {
    const int tile = at / (PM * PN) + (PM * PN > 1 ? g.whole : 0), sub = at % (PM * PN);
    const int per = GROUP * g.tn, grp = tile / per, rem = tile - grp * per;
    const int gm = min(GROUP, g.tm - grp * GROUP), col = rem / gm;
    m0 = uniform((grp * GROUP + rem - col * gm) * BT + sub / PN * (MT * 32));
    n0 = uniform(col * CN * PN + sub % PN * CN);
  };
  auto next = [&](int at, int& m0, int& n0) {                     // the first from `at` on that is not past the edges
    for (; at < count; at += step) {
      place(at, m0, n0);
      if (m0 < g.M && n0 < g.N) break;
    }
    return at;
  };
  // rows past the last are read as zeros
  auto src_x = [&](int m0) {
    return __builtin_amdgcn_make_buffer_rsrc(uniform64(static_cast<const char*>(g.x) + (int64_t)m0 * g.ldx * 2), 0,
                                             uniform(((min(g.M - m0, BT) - 1) * g.ldx + g.K) * 2), 0x00027000);
  };
  auto src_w = [&](int n0) {
    return __builtin_amdgcn_make_buffer_rsrc(uniform64(static_cast<const char*>(g.w) + (int64_t)n0 * rowb), 0,
                                             uniform((g.wrows - n0) * rowb), 0x00027000);
  };
  // A lane's 16 bytes of DMA i: row 8 i + (lane >> 3) of the wave's share.  Row r of w's 16-row tile t is column 32 (t / 2) + 8
  // (r / 4) + 4 (t & 1) + r % 4, so that a lane's accumulators of two tiles are eight neighbouring columns; SILU: the first
  // half of a wave's tiles are gates, the others their ups.
  int vx[MT], vw[NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
    vx[i] = (wave * MT * 8 + 8 * i + (lane >> 3)) * g.ldx * 2 + ((lane & 7) ^ (lane >> 3)) * 16;
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int lr = wave * NT * 8 + 8 * i + (lane >> 3), t = lr >> 4, r = lr & 15, in = 8 * (r >> 2) + 4 * (t & 1) + (r & 3);
    const int tt = t % NT, n = SILU ? t / NT * CW + 32 * (tt % (NT / 2) / 2) + in + (tt >= NT / 2 ? g.N : 0) : 32 * (t >> 1) + in;
    vw[i] = n * rowb + ((lane & 7) ^ (lane >> 3)) * 16;
  }
  auto dma_x = [&](__amdgpu_buffer_rsrc_t src, int k, T* dst, int i) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (LdsPtr)(dst + (wave * MT * 8 + 8 * i) * BK), 16, vx[i], k * (BK * 2), 0, 0);
  };
  auto dma_w = [&](__amdgpu_buffer_rsrc_t src, int k, T* dst, int i) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (LdsPtr)(dst + (wave * NT * 8 + 8 * i) * BK), 16, vw[i], k * (BK * 2), 0, 0);
  };
  // operands: 16 rows, 32 columns of K, the first (0) or second (1) of a step
  const int at0 = r16 * BK + ((qd ^ (r16 & 7)) * 8), at1 = r16 * BK + (((4 + qd) ^ (r16 & 7)) * 8);
  const int ax0 = wm * MT * 16 * BK + at0, ax1 = wm * MT * 16 * BK + at1;
  const int aw0 = wn * NT * 16 * BK + at0, aw1 = wn * NT * 16 * BK + at1;
  auto ld = [&](const T* p, int at, int i) { return *reinterpret_cast<const V8*>(p + at + i * 16 * BK); };
  V8 fx0[MT], fx1[2][MT], fw0[NT], fw1[NT];
  f32x4 acc[NT][MT];
  T* rows = out_rows + wave * 32 * 128;

  int m0, n0, at = next(first, m0, n0);
  if (at >= count) return;                   // (the same for all waves)
  meet<0>();                                 // a walk before this one is done with the LDS
  {
    const auto sx = src_x(m0);
    const auto sw = src_w(n0);
#pragma unroll
    for (int i = 0; i < MT; ++i) { dma_x(sx, 0, x0, i); dma_x(sx, 1, x1, i); }
#pragma unroll
    for (int i = 0; i < NT; ++i) { dma_w(sw, 0, w0, i); dma_w(sw, 1, w1, i); }
  }
  meet<0>();
#pragma unroll
  for (int i = 0; i < MT; ++i) { fx0[i] = ld(x0, ax0, i); fx1[0][i] = ld(x0, ax1, i); }
#pragma unroll
  for (int i = 0; i < NT; ++i) fw0[i] = ld(w0, aw0, i);
  meet<0>();                                 // x's rows of step 0 are read
  for (;;) {
    int m1 = m0, n1 = n0;                    // (after the last tile the same rows again)
    const int nat = next(at + step, m1, n1);
    const bool more = nat < count;
    if (!more) m1 = m0, n1 = n0;
    // Step k from x / w, whose rows those of step k + 2 (of the next tile) replace; xn / wn: step k + 1.
    auto steps = [&](auto begins, auto parity, int k, T* x, T* w, const T* xn, const T* wn) {
      constexpr bool BEGIN = decltype(begins)::value;
      constexpr int P = decltype(parity)::value, NM = MT * NT;
      const bool own = k + 2 < nk;
      const auto sx = src_x(own ? m0 : m1);
      const auto sw = src_w(own ? n0 : n1);
      const int kk = own ? k + 2 : k + 2 - nk;
#pragma unroll
      for (int n = 0; n < NM; ++n) {
        if constexpr (BEGIN) mfma_new<T>(acc[n / MT][n % MT], fw0[n / MT], fx0[n % MT]);
        else mfma_tied<T>(acc[n / MT][n % MT], fw0[n / MT], fx0[n % MT]);
        constexpr int SR = MT / 2, SD = NT;
        if (n % SR == 0 && n / SR < NT) fw1[n / SR] = ld(w, aw1, n / SR);
        if (n % SD == SD / 4) dma_x(sx, kk, x, n / SD);
        __builtin_amdgcn_sched_barrier(0);
      }
      // the rows of step k + 1 are here (a tile's first step: its predecessor's stores need not be done)
      meet<MT + (BEGIN ? NS : 0)>();
#pragma unroll
      for (int n = 0; n < NM; ++n) {
        mfma_tied<T>(acc[n / MT][n % MT], fw1[n / MT], fx1[P][n % MT]);
        constexpr int NR = NT + 2 * MT, SR = NM / NR, SD = MT;
        if (n % SR == 0 && n / SR < NR) {
          const int i = n / SR;
          if (i < NT) fw0[i] = ld(wn, aw0, i);
          else if (i < NT + MT) fx0[i - NT] = ld(xn, ax0, i - NT);
          else fx1[P ^ 1][i - NT - MT] = ld(xn, ax1, i - NT - MT);
        }
        if (n % SD == 3) dma_w(sw, kk, w, n / SD);
        __builtin_amdgcn_sched_barrier(0);
      }
      meet<63>();                            // x's rows of step k + 1 and w's of step k are read
    };
    constexpr std::integral_constant<int, 0> even;
    constexpr std::integral_constant<int, 1> odd;
    steps(std::true_type(), even, 0, x0, w0, x1, w1);
    steps(std::false_type(), odd, 1, x1, w1, x0, w0);
    for (int k = 2; k < nk; k += 2) {
      steps(std::false_type(), even, k, x0, w0, x1, w1);
      steps(std::false_type(), odd, k + 1, x1, w1, x0, w0);
    }
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < MT; j += 4) settle(acc[i][j], acc[i][j + 1], acc[i][j + 2], acc[i][j + 3]);
    __builtin_amdgcn_sched_barrier(0);
    // ---- outputs: 32 rows at a time through the wave's own LDS, so that they leave as whole lines (past the caches: the
    // next launch reads them in another order); a store past the edges writes nothing, but counts
    const auto od = __builtin_amdgcn_make_buffer_rsrc(uniform64(static_cast<char*>(g.out) + (int64_t)m0 * g.ldo * 2), 0,
                                                      uniform(min(g.M - m0, BT) * g.ldo * 2), 0x00027000);
    float pa = 0.f, pb = 0.f;
    if constexpr (!SILU) pa = g.ab[0], pb = g.ab[1];
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      const int rr = (j & 1) * 16 + r16;
#pragma unroll
      for (int p = 0; p < CW / 32; ++p) {
        Pack8<T> o;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          // (of the projection as rounded to T, as a launch of the activation reads it)
          const float z = to_f(from_f<T>(acc[2 * p + (e >> 2)][j][e & 3]));
          if constexpr (SILU) o.h[e] = from_f<T>(silu_mul_of(z, to_f(from_f<T>(acc[NT / 2 + 2 * p + (e >> 2)][j][e & 3]))));
          else o.h[e] = from_f<T>(xielu_of(z, pa, pb));
        }
        *reinterpret_cast<u32x4*>(rows + rr * CW + (((p * 4 + qd) ^ (rr & (U - 1))) * 8)) = o.u;
        __builtin_amdgcn_sched_barrier(0);
      }
      if (j & 1) {
#pragma unroll
        for (int i = 0; i < 32 / R; ++i) {
          const int row = i * R + lane / U, u = lane % U, col = n0 + wn * CW + u * 8;
          const u32x4 v = *reinterpret_cast<const u32x4*>(rows + row * CW + ((u ^ (row & (U - 1))) * 8));
          const int to = col < g.N ? ((wm * MT * 16 + (j - 1) * 16 + row) * g.ldo + col) * 2 : 0x7ffffff0;
          __builtin_amdgcn_raw_buffer_store_b128(v, od, to, 0, 2);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (!more) break;
    m0 = m1, n0 = n1, at = nat;
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);        // DMAs end before the LDS is another's
}

template <typename T, int ACT>
__global__ __launch_bounds__(NTHR) __attribute__((amdgpu_waves_per_eu(1, 1))) void prompt_gemm_kernel(const PromptArgs g) {
  // (objects of their own: the compiler lets an LDS read follow every DMA into the object that it reads)
  __shared__ __align__(16) T x0[BT * BK], x1[BT * BK], w0[BT * BK], w1[BT * BK], rows[4 * 32 * 128];
  // neighbouring workgroups run on eight XCDs: each takes neighbouring tiles of a round
  const int nb = gridDim.x, b = blockIdx.x, me = nb % 8 == 0 ? (b & 7) * (nb >> 3) + (b >> 3) : b;
  walk<T, ACT, 8, 8>(g, x0, x1, w0, w1, rows, me, nb, g.whole);
  const int rest = g.tm * g.tn - g.whole;
  if (g.pieces == 2) walk<T, ACT, 4, 8>(g, x0, x1, w0, w1, rows, me, nb, rest * 2);
  else if (g.pieces == 4) walk<T, ACT, 4, 4>(g, x0, x1, w0, w1, rows, me, nb, rest * 4);
}

template <typename T>
void launch_act(int act, const PromptArgs& g, int grid, hipStream_t s) {
  if (act == PROMPT_SILU) prompt_gemm_kernel<T, PROMPT_SILU><<<grid, NTHR, 0, s>>>(g);
  else prompt_gemm_kernel<T, PROMPT_XIELU><<<grid, NTHR, 0, s>>>(g);
}

// Tiles of the launch, and how those behind the last whole round over the CUs are cut: into quarters (128 x 128 weight rows) or
// halves (128 x 256) where the pieces come to one round.  A quarter takes 0.43 of a tile's time and a half 0.62, so that two
// rounds of either are no faster than one of tiles: 2048 -> 2 x 5504, rows: us whole, halves, quarters: 256 (43 tiles) 43, 28,
// 21; 320 (86) 42, 26, 34; 768 (129) 48, 47, 49; 1024 (172) 47, 51, 52; 1536 (258) 78, 67, 61; 8192 (5 rounds, 96) 262, 246, 258.
struct Plan { int tm, tn, whole, pieces; };
Plan plan_of(int act, int M, int N) {
  const int cn = act == PROMPT_SILU ? BT / 2 : BT, cus = device_cus();
  Plan p{(M + BT - 1) / BT, (N + cn - 1) / cn, 0, 1};
  const int tiles = p.tm * p.tn, last = tiles % cus;
  if (last != 0 && last * 2 <= cus) p.pieces = last * 4 <= cus ? 4 : 2;
  p.whole = p.pieces == 1 ? tiles : tiles - last;
  return p;
}

}  // namespace

// Whether it is faster than the library's projection and a launch of the activation, which fill small or odd numbers of tiles
// better: by the useful part of the time of the rounds (quarters and halves as above).  From 512 rows on for SILU and 1024 for
// XIELU, whose outputs' conversion takes a sixth of a tile's time at K = 2048 and whose activation launch moves less.
// K <= 2048, where the library takes 26 us at least: one round of quarters from 65 rows on; else half (a single round of tiles
// 0.54), XIELU 0.7, and not below K = 2048, where the conversion takes as long as the products.  Longer K: 0.77.  Over 19 shapes
// of 1024 to 8192 columns and 80 to 16384 rows with weights from memory, what the rule takes is 1.23 times as fast in the
// geometric mean, 0.976 at worst; half of the rounds' time for all K took as many shapes again at 0.79 to 1.05.
// us, library and activation -> here:
//   SILU  K 2048 -> 2 x 5504, 256 rows 29 -> 20, 512 36 -> 29, 1024 58 -> 49, 2048 94 -> 78, 2700 134 -> 96, 6000 299 -> 202,
//         14336 566 -> 459;  -> 2 x 2752, 256 29 -> 20, 1024 37 -> 29, 3072 84 -> 66, 14336 357 -> 237
//         K 4096 -> 2 x 14336, 512 105 -> 91, 768 170 -> 139, 2700 577 -> 432, 16384 2746 -> 2540; not 320 75 -> 82, 640 145 -> 156;
//         -> 2 x 5504, 3072 315 -> 206, 16384 1206 -> 995; not 768 79 -> 93;  -> 2 x 3584, 2700 250 -> 123; not 1280 83 -> 94
//         K 8192 -> 2 x 7168, 1024 217 -> 180, 5120 950 -> 827; not 512 119 -> 132, 640 141 -> 171
//   XIELU K 2048 -> 8256, 256 29 -> 23, 1536 70 -> 60, 2048 93 -> 78, 3000 113 -> 113, 4096 150 -> 135, 8192 319 -> 250, 14336 467 ->
//         419; not 512 34 -> 35, 1024 53 -> 58
//         K 4096 -> 21504, 2560 472 -> 361, 4096 586 -> 529, 8192 1219 -> 1030; not 512 88 -> 100, 1152 184 -> 198
bool prompt_gemm_pays(int act, int M, int N, int K) {
  const Plan p = plan_of(act, M, N);
  const int cus = device_cus(), rest = p.tm * p.tn - p.whole;
  const bool silu = act == PROMPT_SILU, pieces = p.whole == 0;
  if (M > 64 && pieces && p.pieces == 4 && K <= 2048) return true;
  if (M < (silu ? 512 : 1024)) return false;
  const double rounds = (p.whole + cus - 1) / cus + (rest == 0 ? 0. : p.pieces == 4 ? 0.43 : 0.62);
  const double useful = (double)M * N / (BT * (silu ? BT / 2 : BT)) / cus;
  if (K > 2048) return useful >= rounds * 0.77;
  if (silu) return useful >= rounds * (rounds == 1. ? 0.54 : 0.5);
  return (K == 2048 || pieces) && useful >= rounds * 0.7;
}

void launch_prompt_gemm(int dtype, int act, void* out, const void* x, const void* w, const float* ab, int M, int N,
                        int K, int ldx, hipStream_t s) {
  const Plan p = plan_of(act, M, N);
  const PromptArgs g{x, w, out, ab, M, N, K, ldx, N, act == PROMPT_SILU ? 2 * N : N, p.tm, p.tn, p.whole, p.pieces};
  if (dtype == DT_BF16) launch_act<bf16>(act, g, device_cus(), s);
  else launch_act<f16>(act, g, device_cus(), s);
}

}  // namespace kgc
