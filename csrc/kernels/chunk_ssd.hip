// Mamba-2 (SSD, Dao and Gu, 2024) scan of prompt rows, chunkwise on the matrix cores.  Per (sequence, head) with a
// log decay f_t = -e^a size_t and the step size size_t,
//     S_t = e^(f_t) S_(t-1) + size_t B_t x_t^T,      y_t = S_t^T C_t + D x_t .
// Over a chunk of L = 32 tokens, b_t the running sum of f and S_0 the state before it:
//     Y   = e^(b_t) C S_0 + P X,      P_ts = e^(b_t - b_s) size_s (C_t . B_s) for s <= t, + D where s = t
//     S_L = e^(b_L) S_0 + sum_s e^(b_L - b_s) size_s B_s x_s^T
// Heads share B and C, so a first launch makes once per chunk and group what every head would: the bf16
// parts of C and of B^T in the order in which the walk's MFMAs read them from LDS, and the products C_t . B_s; and per
// head the running sums and weights of the tokens.  In the walk a workgroup of 4 waves owns 128 value
// columns (two heads of up to 64, or 128 of one), a wave 32 of them, whose S stays in MFMA accumulators: two
// column tiles for each operand read.  The parts arrive by DMA, C's while the state is updated and B^T's while
// the outputs are computed; two workgroups share a CU.
//
// What bounds it: instruction issue.  An MFMA takes 8 cycles of a SIMD's issue and 16 of its matrix core, a vector
// instruction 4, so both fill only where a wave's own vector work (splitting S) stands between its MFMAs: the
// regions below say in which order.  Per wave and chunk 226 MFMAs and 950 vector instructions, in 44 and 58 % of the
// cycles at two waves per SIMD (before the order was given: the same work in 1.5 times the time), 2.16 GHz in a loop of calls.  2 x 8192 tokens, 32 heads of
// 128 x 64, us: 220 in all (chunk_scan.hip 357); kernel by kernel in a trace, whose clocks are not warm, images 23,
// contributions 60, states 11, walk 145 (130 and 255 there).
//
// Precision: fp32 operands enter the bf16 MFMAs as three bf16 parts each (24 bits), six products of parts.  The
// corrections of C S_0 and of C . B have sums of their own; those of P X and of the update are summed first and the main
// products on top of them.  Exponents are differences of running sums kept in double.
//
// Workspace: 52 KB per chunk and group, 1 KB per chunk and head, and 4 D V bytes per segment and head: 76 MB for 2 x 8192
// tokens with one group (27, 17 and 32; chunk_scan.hip 16), 268 MB with eight.
//
// Few long sequences are cut into segments: one walk makes every segment's contribution from a zero state
// (B^T only), a small launch puts the states together in which the segments start, and the second walk has them all.
#include "chunk.h"
#include "chunk_rows.h"
#include "device.h"
#include "launch.h"

namespace kgc {

namespace {

constexpr int L = 32, D = 128;               // tokens per chunk, state rows
constexpr int NT = 256, NW = NT / 64;
constexpr int DT = D / 16, LT = L / 16, KD = D / 32;
constexpr int PART = L * D;                  // elements of a part of C or B^T
constexpr int IMG = 2 * 3 * PART * 2 + L * L * 4;   // bytes of a chunk's image: C, B^T, C . B
constexpr double LOG2E = 1.4426950408889634074;

// what a chunk's tokens carry, per head; zero weights past the sequence's end
struct TokenRec {
  int bn[L];                                 // running sum of f, times log2 e: nearest whole number
  float bf[L];                               // and what is left
  float size[L];
  int none[L];                               // (a part is a whole number of 16-byte units of 32 lanes)
  float in[L];                               // e^(b_t)
  float wt[L];                               // e^(b_L - b_t) size_t
  double total;                              // b_L times log2 e
  int none2[2 * L - 2];
};
static_assert(sizeof(TokenRec) == 1024, "two parts of 512 bytes");

struct SsdArgs {
  float* out;                                // [T, H dv]
  const float* xbc;                          // [T, H dv + 2 G D]: x | B | C
  int64_t stride;
  const void* dt;                            // [T, H]: step sizes before softplus
  int64_t dts;
  int dt_type;
  const float *a_log, *dt_bias, *dskip;
  float* S;
  const int *qsl, *seq_lens, *slots;
  int P, H, G, dv, num_slots, hpw;
  int seg;                                   // tokens per segment (0: sequences are not cut)
  int items;
  char* img;                                 // [chunks][G][IMG]
  TokenRec* rec;                             // [chunks][H]
  float* seg_state;                          // [items][H][D][dv]: contribution, then state a segment starts from
  double* seg_gate;                          // [items][H]: log2 of a segment's decay
};

// 2^y for y <= 0 held in double: the reduction is exact to fp32 however large y is
__device__ __forceinline__ float exp2_d(double y) {
  const double n = __builtin_rint(y);
  return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f((float)(y - n)), (int)n);
}

// places of 16-byte units in the image, so that 16 lanes read 16 different bank groups
__device__ __forceinline__ int c_unit(int t, int u) { return t * (D / 8) + (u ^ (t & 15)); }
__device__ __forceinline__ int c_unit32(int t, int u) { return t * (L / 4) + (u ^ ((t >> 1) & 7)); }   // C . B
__device__ __forceinline__ int b_unit(int d, int u) { return d * (L / 8) + (u ^ ((d >> 2) & 3)); }

// ---- images of a chunk (blockIdx.y < G) and its tokens' weights, 8 heads per workgroup -------
__global__ __launch_bounds__(NT) void ssd_prep_kernel(const SsdArgs a) {
  __shared__ __align__(16) bf16 Cs[3 * PART], Bs[3 * PART];
  const SegItem it = seg_item(blockIdx.x, a.qsl, a.P, L);
  if (it.seq < 0) return;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int c0 = it.idx * L, len = a.qsl[it.seq + 1] - a.qsl[it.seq], nl = min(L, len - c0);
  const int slot = a.slots[it.seq];
  if (nl <= 0 || slot < 0 || slot >= a.num_slots || a.seq_lens[it.seq] < len) return;
  const int64_t t0 = a.qsl[it.seq] + c0;
  if (blockIdx.y >= a.G) {
    const int t = lane & 31, h = (blockIdx.y - a.G) * 8 + wave * 2 + (lane >> 5);
    const int hc = min(h, a.H - 1);
    const int64_t at = (t0 + min(t, nl - 1)) * a.dts + hc;
    const float raw = a.dt_type == DT_F32 ? reinterpret_cast<const float*>(a.dt)[at]
                      : a.dt_type == DT_F16 ? (float)reinterpret_cast<const f16*>(a.dt)[at]
                                            : (float)reinterpret_cast<const bf16*>(a.dt)[at];
    const double z = (double)raw + (double)a.dt_bias[hc];
    const double size = z > 40.0 ? z : log1p(exp(z));
    const double f = -exp((double)a.a_log[hc]) * size;
    const bool ok = t < nl;
    // a decay of e^-1e6 is zero; a finite floor keeps the differences of running sums defined
    double b = !ok ? 0.0 : (f < -1e6 ? -1e6 : f) * LOG2E;
    b = scan_step<0x111, 0xf, false>(b);     // within each half of the wave
    b = scan_step<0x112, 0xf, false>(b);
    b = scan_step<0x114, 0xf, false>(b);
    b = scan_step<0x118, 0xf, false>(b);
    b = scan_step<0x142, 0xa, false>(b);
    const double bL = __shfl(b, lane | 31, 64);
    const float s = ok ? (float)size : 0.f;
    if (h < a.H) {
      TokenRec& r = a.rec[(int64_t)blockIdx.x * a.H + h];
      const double n = __builtin_rint(b);
      r.bn[t] = (int)n;
      r.bf[t] = (float)(b - n);
      if (t == L - 1) r.total = b;
      r.size[t] = s;
      r.in[t] = exp2_d(b);
      r.wt[t] = exp2_d(bL - b) * s;
    }
    return;
  }
  const float* kb = a.xbc + t0 * a.stride + (int64_t)a.H * a.dv + (int64_t)blockIdx.y * D;
  const float* qb = kb + (int64_t)a.G * D;
  char* img = a.img + ((int64_t)blockIdx.x * a.G + blockIdx.y) * IMG;
  u32x4* ci = reinterpret_cast<u32x4*>(img);
  u32x4* bi = reinterpret_cast<u32x4*>(img + 3 * PART * 2);
  const int64_t rs = a.stride;
  // rows of C and B: the columns 4 j .. and 16 + 4 j .. of 32 make a unit of the permuted order
#pragma unroll
  for (int i = 0; i < L * D / 8 / NT; ++i) {
    const int e = tid + NT * i, t = e / (D / 8), u = e % (D / 8), c = (u >> 2) * 32 + (u & 3) * 4;
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const float* row = (w ? kb : qb) + min(t, nl - 1) * rs + c;
      const f32x4 x0 = *reinterpret_cast<const f32x4*>(row), x1 = *reinterpret_cast<const f32x4*>(row + 16);
      float x[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
      if (t >= nl)
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = 0.f;
      bf16x8 p[3];
      split8<3>(x, p);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const u32x4 o = __builtin_bit_cast(u32x4, p[j]);
        reinterpret_cast<u32x4*>(w ? Bs : Cs)[j * (PART / 8) + c_unit(t, u)] = o;
        if (w == 0) ci[j * (PART / 8) + c_unit(t, u)] = o;
      }
    }
  }
  // B^T: eight tokens of a column
#pragma unroll
  for (int i = 0; i < L * D / 8 / NT; ++i) {
    const int e = tid + NT * i, d = e % D, u = e / D;
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int t = u * 8 + j;
      const float y = kb[min(t, nl - 1) * rs + d];
      x[j] = t < nl ? y : 0.f;
    }
    bf16x8 p[3];
    split8<3>(x, p);
#pragma unroll
    for (int j = 0; j < 3; ++j) bi[j * (PART / 8) + b_unit(d, u)] = __builtin_bit_cast(u32x4, p[j]);
  }
  __syncthreads();
  if (wave < LT * (LT + 1) / 2) {            // C . B: tiles (0, 0), (1, 0), (1, 1) as [s][t]
    const int ti = wave > 0, si = wave > 1;
    f32x4 hi = {0.f, 0.f, 0.f, 0.f}, lo = hi;
#pragma unroll
    for (int ks = 0; ks < KD; ++ks) {
      bf16x8 fa[3], fb[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        fa[j] = *reinterpret_cast<const bf16x8*>(Bs + j * PART + c_unit(si * 16 + lr, ks * 4 + lg) * 8);
        fb[j] = *reinterpret_cast<const bf16x8*>(Cs + j * PART + c_unit(ti * 16 + lr, ks * 4 + lg) * 8);
      }
      mm<true, 3, 3>(fa, fb, hi, lo);
    }
    reinterpret_cast<f32x4*>(img + 2 * 3 * PART * 2)[c_unit32(ti * 16 + lr, si * 4 + lg)] = hi + lo;
  }
}

// 1024 bytes from each wave's 64 lanes to LDS
__device__ __forceinline__ void dma16(const void* src, void* dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                   (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

// ---- the walk.  MODE 0: whole sequences; 1: segments from zero (states only); 2: segments from
// the states that they start in ------------------------------------------------------------------
// PAIRS: an even number of value columns
template <int MODE, bool PAIRS>
__global__ __launch_bounds__(NT, 2) void ssd_walk_kernel(const SsdArgs a) {
  __shared__ __align__(16) bf16 Bs[3 * PART];
  __shared__ __align__(16) bf16 Cs[3 * PART];             // (MODE 1: B^T of every other chunk)
  __shared__ __align__(16) bf16 Ps[MODE == 1 ? 8 : 2 * 3 * L * L];
  __shared__ __align__(16) float Gs[MODE == 1 ? 4 : L * L];
  __shared__ __align__(16) char Rp[2 * 512], Rw[2 * 512];   // both parts of the heads' records (MODE 1: the second of two chunks)
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // workgroups of one item on one XCD: they read the same images
  const int nct = a.hpw == 2 ? 1 : (a.dv + 127) / 128, wpi = a.H / a.hpw * nct;
  const int q8 = blockIdx.x / 8, y = q8 % wpi, bx = q8 / wpi * 8 + blockIdx.x % 8;
  if (bx >= a.items) return;
  int seq = bx, seg_idx = 0, item = 0, seg_count = 1;
  if (MODE != 0) {
    const SegItem it = seg_item(bx, a.qsl, a.P, a.seg);
    if (it.seq < 0) return;
    seq = __builtin_amdgcn_readfirstlane(it.seq);
    seg_idx = __builtin_amdgcn_readfirstlane(it.idx);
    seg_count = __builtin_amdgcn_readfirstlane(it.count);
    item = __builtin_amdgcn_readfirstlane(it.first) + seg_idx;
    if (MODE == 1 && seg_idx + 1 == seg_count) return;
  }
  const int hb = y / nct, ct = y - hb * nct;
  const int hw = a.hpw == 2 ? wave >> 1 : 0;              // this wave's head of the workgroup's
  const int h = hb * a.hpw + hw, grp = h / (a.H / a.G);
  // this lane's columns: 2 lr and 2 lr + 1 of the wave's 32
  const int col = (a.hpw == 2 ? (wave & 1) * 32 : ct * 128 + wave * 32) + 2 * lr;
  const bool ok0 = col < a.dv, ok1 = col + 1 < a.dv;
  const int cc0 = min(col, a.dv - 1 - (int)PAIRS), cc1 = min(col + 1, a.dv - 1);   // off the edge: read the last
  const int seq0 = a.qsl[seq];
  int start = seq0, len = a.qsl[seq + 1] - start;
  const int pos0 = a.seq_lens[seq] - len, slot = a.slots[seq];
  const int64_t os = (int64_t)a.H * a.dv;
  const int chunk0 = __builtin_amdgcn_readfirstlane(chunks_before<L>(seq, a.qsl)) + (MODE != 0 ? seg_idx * (a.seg / L) : 0);
  if (MODE != 0) {
    start += seg_idx * a.seg;
    len = min(a.seg, len - seg_idx * a.seg);
  }
  if (len <= 0) return;
  if (slot < 0 || slot >= a.num_slots || pos0 < 0) {      // padding: defined zeros
    if (MODE != 1)
      for (int t = lg; t < len; t += 4) {
        float* o = a.out + (start + t) * os + (int64_t)h * a.dv;
        if (ok0) o[col] = 0.f;
        if (ok1) o[col + 1] = 0.f;
      }
    return;
  }
  const int64_t sh = (int64_t)D * a.dv;
  float* Ss = a.S + ((int64_t)slot * a.H + h) * sh;
  f32x4 S[DT][2];
  {
    const bool own = MODE == 2 && seg_count > 1;
    const float* from = own ? a.seg_state + ((int64_t)item * a.H + h) * sh : Ss;
    if (MODE == 1 || (!own && pos0 == 0)) {
#pragma unroll
      for (int i = 0; i < DT; ++i) S[i][0] = S[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    } else {
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float* row = from + (i * 16 + 4 * lg + r) * a.dv;
          S[i][0][r] = row[cc0];
          S[i][1][r] = row[cc1];
        }
    }
  }
  const float* vb = a.xbc + (int64_t)h * a.dv;
  const float skip = a.dskip[h];
  int rs = (int)a.stride, ro = (int)os;
  auto image = [&](int ci) { return a.img + ((int64_t)ci * a.G + grp) * IMG; };
  // one of the six pieces that a wave brings of the parts of C or B^T
  auto dma = [&](const char* src, bf16* dst, int i) {
    dma16(src + lane * 16 + (wave * 6 + i) * 1024, reinterpret_cast<char*>(dst) + (wave * 6 + i) * 1024);
  };
  float v[2][8];                             // x of tokens 8 lg .., both columns
  // Rows past the end and columns off the edge: through a descriptor that ends with the chunk's last value,
  // reads beyond it give zero, and writes do nothing.
  const uint32_t vat = (__mul24(8 * lg, rs) + col) * 4;
  const uint32_t out_at = (__mul24(4 * lg, ro) + col) * 4, oat0 = ok0 ? out_at : 1u << 30, oat1 = ok1 ? out_at + 4 : 1u << 30;
  auto span = [&](const float* p, int rows, int row) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, ((rows - 1) * row + a.dv) * 4, 0x00027000);
  };
  auto fetch_v = [&](int c0, int i0, int i1) {
    const auto r = span(vb + (int64_t)(start + c0) * a.stride, min(L, len - c0), rs);
#pragma unroll
    for (int i = i0; i < i1; ++i) {
      if constexpr (PAIRS) {
        const f32x2 p = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, vat + i * rs * 4, 0, 0));
        v[0][i] = p[0];
        v[1][i] = p[1];
      } else {
        v[0][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, vat + i * rs * 4, 0, 0));
        v[1][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, vat + i * rs * 4 + 4, 0, 0));
      }
    }
  };
  // records of the workgroup's heads, a part of 32 lanes each (one head: twice); every wave brings the same
  auto dma_rec = [&](int ci, int part, char* dst) {
    const int hh = hb * a.hpw + (a.hpw == 2 ? lane >> 5 : 0);
    dma16(reinterpret_cast<const char*>(a.rec + (int64_t)ci * a.H + hh) + part * 512 + (lane & 31) * 16, dst);
  };
  auto dma_p = [&](int ci) {                 // C . B and the weights of P
    dma16(image(ci) + 2 * 3 * PART * 2 + wave * 1024 + lane * 16, reinterpret_cast<char*>(Gs) + wave * 1024);
    dma_rec(ci, 0, Rp);
  };
  auto dma_w = [&](int ci, char* dst) {
    dma_rec(ci, 1, dst);
  };
  // Weighted products P of one row tile of this wave's head; the head's waves share the tiles in LDS
  // (four waves of one head: two and two write the same).
  const int trow = (wave & 1) * 16 + lr;
  auto put_p = [&]() {
    const TokenRec& rec = *reinterpret_cast<const TokenRec*>(Rp + hw * 512);
    const int tn = rec.bn[trow];
    const float tf = rec.bf[trow];
    int before = trow - 8 * lg;              // masks are made where they are used, not kept
    asm volatile("" : "+v"(before));
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      // 2^(b_t - b_s): the whole numbers' difference is exact, the rest's within [-1, 1]
      const int s = 8 * lg + i;
      const float e = __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(tf - rec.bf[s]), tn - rec.bn[s]);
      const float p = Gs[c_unit32(trow, 2 * lg + (i >> 2)) * 4 + (i & 3)] * (e * rec.size[s]);
      x[i] = i < before ? p : i == before ? p + skip : 0.f;
    }
    bf16x8 fp[3];
    split8<3>(x, fp);
#pragma unroll
    for (int i = 0; i < 3; ++i)
      *reinterpret_cast<bf16x8*>(Ps + (hw * 3 + i) * L * L + b_unit(trow, lg) * 8) = fp[i];
  };
  auto arrived = [] { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };

  double btot = 0.0;
  fetch_v(0, 0, 8);
#pragma unroll
  for (int i = 0; i < 6; ++i) dma(image(chunk0) + (MODE == 1 ? 3 * PART * 2 : 0), Cs, i);
  dma_w(chunk0, Rw);
  if (MODE != 1) {
    dma_p(chunk0);
    arrived();
    __syncthreads();
    put_p();
  }
  auto load_a = [&](bf16x8 (&f)[2][3], const bf16* cur, int ks) {
#pragma unroll
    for (int ti = 0; ti < LT; ++ti)
#pragma unroll
      for (int i = 0; i < 3; ++i)
        f[ti][i] = *reinterpret_cast<const bf16x8*>(cur + i * PART + c_unit(ti * 16 + lr, ks * 4 + lg) * 8);
  };
  auto load_b = [&](bf16x8 (&f)[2][3], const bf16* cur, int dt) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 3; ++i)
        f[j][i] = *reinterpret_cast<const bf16x8*>(cur + i * PART + b_unit((dt + j) * 16 + lr, lg) * 8);
  };
  auto split_s = [&](bf16x8 (&sp)[2][3], int ks) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      float x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = S[2 * ks + (i >> 2)][c][i & 3];
      split8<3>(x, sp[c]);
    }
  };
  bf16x8 sp[2][2][3];                        // parts of 32 rows of S; the first ones of the next chunk
  if (MODE != 1) split_s(sp[0], 0);
  // One chunk; its C (MODE 1: B^T) is in or on its way to `cur`.
  auto chunk = [&](int c0, int ci, bf16* cur, bf16* other, char* rcur, char* rother) {
    // (after the last chunk the same again: a branch would end the regions that the order is made in)
    const bool more = c0 + L < len;
    const int cn = more ? c0 + L : c0, in = more ? ci + 1 : ci;
    asm volatile("" : "+s"(rs), "+s"(ro));   // row offsets are computed per chunk, not kept
    bf16x8 wp[2][3];
    f32x4 o[LT][2];
    int bad[2];
    arrived();
    __syncthreads();
    if (MODE == 1) {
#pragma unroll
      for (int i = 0; i < 6; ++i) dma(image(in) + 3 * PART * 2, other, i);
      dma_w(in, rother);
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) bad[c] = take_nonfinite(v[c], L, [&](int i) { return lg * 8 + i; });
    const bool some_bad = __builtin_amdgcn_readfirstlane(__any(min(bad[0], bad[1]) < L));
    const TokenRec& rec = *reinterpret_cast<const TokenRec*>(rcur + hw * 512 - 512);
    const float decay = rec.in[L - 1];
    if (MODE == 1) btot += rec.total;
    auto split_w = [&]() {                   // weighted x of the update
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        float x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = v[c][i] * rec.wt[8 * lg + i];
        split8<3>(x, wp[c]);
      }
    };
    if (MODE != 1) {
      // C S_0, the parts of S a step ahead
      f32x4 ol[LT][2];
#pragma unroll
      for (int ti = 0; ti < LT; ++ti)
#pragma unroll
        for (int c = 0; c < 2; ++c) o[ti][c] = ol[ti][c] = f32x4{0.f, 0.f, 0.f, 0.f};
      dma_p(in);
      bf16x8 fa[2][2][3];
      load_a(fa[0], cur, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < KD; ++ks) {
        if (ks + 1 < KD) {
          load_a(fa[(ks + 1) & 1], cur, ks + 1);
          split_s(sp[(ks + 1) & 1], ks + 1);
        } else {                             // P and x
#pragma unroll
          for (int ti = 0; ti < LT; ++ti)
#pragma unroll
            for (int i = 0; i < 3; ++i)
              fa[0][ti][i] = *reinterpret_cast<const bf16x8*>(Ps + (hw * 3 + i) * L * L + b_unit(ti * 16 + lr, lg) * 8);
#pragma unroll
          for (int c = 0; c < 2; ++c) split8<3>(v[c], sp[0][c]);
        }
        if (ks < 3) {
          dma(image(ci) + 3 * PART * 2, other, 2 * ks);
          dma(image(ci) + 3 * PART * 2, other, 2 * ks + 1);
        }
        mm3_add(fa[ks & 1], sp[ks & 1], o, ol);
        __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
        interleave<24, 4, 0, 8>();
        __builtin_amdgcn_sched_barrier(0);
      }
      f32x4 px[LT][2];
      mm3(fa[0], sp[0], px);
      split_w();
      f32x4 fin[LT];
#pragma unroll
      for (int ti = 0; ti < LT; ++ti) fin[ti] = *reinterpret_cast<const f32x4*>(rec.in + ti * 16 + 4 * lg);
#pragma unroll
      for (int ti = 0; ti < LT; ++ti)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[ti][c][r] = __builtin_fmaf(o[ti][c][r] + ol[ti][c][r], fin[ti][r], px[ti][c][r]);
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
      interleave<24, 4, 0, 8>();
      __builtin_amdgcn_sched_barrier(0);
      arrived();
      __syncthreads();
      if (some_bad)
#pragma unroll
        for (int ti = 0; ti < LT; ++ti)
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              asm volatile("" : "+v"(o[ti][c][r]));       // a branch, not selects in every chunk
              if (ti * 16 + lg * 4 + r >= bad[c]) o[ti][c][r] = NAN;
            }
    } else {
      split_w();
    }
    const auto od = span(a.out + (int64_t)(start + c0) * os + (int64_t)h * a.dv, min(L, len - c0), ro);
    auto put_o = [&](int ti, int r) {
      const uint32_t row = (ti * 16 + r) * ro * 4;
      if constexpr (PAIRS) {
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, f32x2{o[ti][0][r], o[ti][1][r]}), od, oat0 + row, 0, 0);
      } else {
        const float y0 = o[ti][0][r], y1 = o[ti][1][r];   // (a bit_cast of a vector's element takes the first)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, y0), od, oat0 + row, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, y1), od, oat1 + row, 0, 0);
      }
    };
    const bf16* bsrc = MODE == 1 ? cur : other;
    bf16x8 fb[2][2][3];
    f32x4 u[2][2][2];
    load_b(fb[0], bsrc, 0);
    auto add = [&](int dt) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            S[dt + j][c][r] = __builtin_fmaf(S[dt + j][c][r], decay, u[dt >> 1 & 1][j][c][r]);
    };
#pragma unroll
    for (int dt = 0; dt < DT; dt += 2) {
      const int k = dt >> 1 & 1;
      if (dt + 2 < DT) load_b(fb[k ^ 1], bsrc, dt + 2);
      if (dt < 4) fetch_v(cn, dt * 2, dt * 2 + 4);
      if (MODE != 1) {                       // C, its weights, and the outputs on the way
        if (dt < 6) {
          dma(image(in), cur, dt);
          dma(image(in), cur, dt + 1);
        } else {
          dma_w(in, Rw);
        }
        put_o(dt >> 2, dt & 2);
        put_o(dt >> 2, (dt & 2) + 1);
        if (dt == 4) put_p();                // of the next chunk (the last one's again: nobody reads it)
        if (dt == 6) split_s(sp[0], 0);
      }
      mm3(fb[k], wp, u[k]);
      if (dt > 0) add(dt - 2);
      if (MODE != 1) {
        __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
        if (dt == 4) interleave<24, 6, 0, 4>();
        else if (dt == 6) interleave<24, 4, 0, 6>();
        else interleave<24, 2, 0, 3>();
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    add(DT - 2);
    if (some_bad) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            asm volatile("" : "+v"(S[dt][c][r]));
            S[dt][c][r] = bad[c] < L ? NAN : S[dt][c][r];
          }
      if (MODE != 1) split_s(sp[0], 0);
    }
  };
  if (MODE == 1) {
    for (int c0 = 0, ci = chunk0; c0 < len; c0 += 2 * L, ci += 2) {
      chunk(c0, ci, Cs, Bs, Rw, Rp);
      if (c0 + L < len) chunk(c0 + L, ci + 1, Bs, Cs, Rp, Rw);
    }
  } else {
    for (int c0 = 0, ci = chunk0; c0 < len; c0 += L, ++ci) chunk(c0, ci, Cs, Bs, Rw, Rw);
  }
  if (MODE == 1 || MODE == 0 || seg_idx + 1 == seg_count) {
    int dw = a.dv;                           // opaque: addresses are not kept across the walk
    asm volatile("" : "+s"(dw));
    float* dst = MODE == 1 ? a.seg_state + ((int64_t)item * a.H + h) * sh : Ss;
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float* row = dst + (i * 16 + 4 * lg + r) * dw + col;
        if (ok0) row[0] = S[i][0][r];
        if (ok1) row[1] = S[i][1][r];
      }
    if (MODE == 1 && lane == 0) a.seg_gate[(int64_t)item * a.H + h] = btot;   // (all waves of a head: the same)
  }
}

// ---- the states in which segments start, in place of the contributions --------------------------
__global__ __launch_bounds__(NT) void ssd_chain_kernel(const SsdArgs a) {
  const int seq = blockIdx.z, h = blockIdx.y, lane = threadIdx.x & 63;
  const int len = a.qsl[seq + 1] - a.qsl[seq], pos0 = a.seq_lens[seq] - len, slot = a.slots[seq];
  if (len <= a.seg || slot < 0 || slot >= a.num_slots || pos0 < 0) return;
  const int first = pieces_before(seq, a.qsl, a.seg);
  const int count = (len + a.seg - 1) / a.seg, sh = D * a.dv;
  const int64_t step = (int64_t)a.H * sh;
  const int at = (blockIdx.x * NT + threadIdx.x) * 4;     // (128 rows: a multiple of 4 elements)
  if (at >= sh) return;
  f32x4 S = {0.f, 0.f, 0.f, 0.f};
  if (pos0 != 0) S = *reinterpret_cast<const f32x4*>(a.S + ((int64_t)slot * a.H + h) * sh + at);
  float* p = a.seg_state + ((int64_t)first * a.H + h) * sh + at;
  const double* gate = a.seg_gate + (int64_t)first * a.H + h;
#pragma unroll 4
  for (int j = 0; j < count - 1; ++j) {
    const f32x4 c = *reinterpret_cast<const f32x4*>(p + j * step);
    const float f = exp2_d(gate[(int64_t)j * a.H]);
    *reinterpret_cast<f32x4*>(p + j * step) = S;
#pragma unroll
    for (int r = 0; r < 4; ++r) S[r] = __builtin_fmaf(f, S[r], c[r]);
  }
  *reinterpret_cast<f32x4*>(p + (count - 1) * step) = S;
}

template <bool PAIRS> void walk(const SsdArgs& a, int grid, hipStream_t s) {
  if (a.seg <= 0) {
    ssd_walk_kernel<0, PAIRS><<<grid, NT, 0, s>>>(a);
  } else {
    ssd_walk_kernel<1, PAIRS><<<grid, NT, 0, s>>>(a);
    ssd_chain_kernel<<<dim3((D * a.dv / 4 + NT - 1) / NT, a.H, a.P), NT, 0, s>>>(a);
    ssd_walk_kernel<2, PAIRS><<<grid, NT, 0, s>>>(a);
  }
}

// heads per workgroup
int heads_per_wg(int H, int V, int G) { return V <= 64 && (H / G) % 2 == 0 ? 2 : 1; }

// workgroups of a sequence's walk
int walk_wgs(int H, int V, int G) { return H / heads_per_wg(H, V, G) * (heads_per_wg(H, V, G) == 2 ? 1 : (V + 127) / 128); }

}  // namespace

// Segments for two workgroups per CU, of at least four chunks.  Sequences of two to three segments are cut only where
// every workgroup then has a CU of its own: the second walk's start costs 13 us (32 heads of 128 x 64, one group, whole ->
// cut: 1 x 256, 272, 340 42.0 -> 46.0, 45.8 -> 44.1, 53.0 -> 44.5; 4 x 300, 380 50.3 -> 52.8, 58.0 -> 52.3; 8 x 300 51 -> 67).
SsdWork ssd_shared_plan(int P, int Tp, int H, int V, int G) {
  SsdWork w;
  w.items = P;
  const int64_t chunks = Tp / L + P;
  w.bytes = chunks * G * IMG + chunks * H * (int64_t)sizeof(TokenRec);
  const int cus = device_cus(), wpi = walk_wgs(H, V, G), want = (2 * cus + wpi - 1) / wpi;   // items for two workgroups per CU
  if (P * 2 > want) return w;
  const int seg = segment_rows(P, Tp, want, L, 4);    // one round
  const int rows = Tp / P;
  const int64_t wgs = (int64_t)P * ((rows + seg - 1) / seg) * wpi;
  if (rows < 3 * seg && (wgs > cus || rows <= 2 * seg + (2 * wgs > cus ? 2 * L : 0))) return w;
  w.seg = seg;
  w.items = Tp / seg + P;
  w.state_at = w.bytes;
  w.gate_at = w.state_at + 4 * (int64_t)w.items * H * D * V;
  w.bytes = w.gate_at + 8 * (int64_t)w.items * H;
  return w;
}

// Of the calls that ssd_chunk_ok takes: at least four heads to a group, and rows enough for the images (52 KB per chunk
// and group, written and read once more) and the launch that makes them.  chunk_scan.hip, one workgroup per CU where
// this has two -> this, in us, 128 x 64 and (V 128) 128 x 128 states; a sequence has 16 workgroups:
//   workgroups for up to all CUs: from four chunks a sequence on, from six where there are many images or heads of 128
//   columns; which of the two walks is cut into segments decides between 256 and 1000 rows
//     32 heads, 1 group    1 x 96, 144, 256, 1000   21.1 -> 22.6, 32.4 -> 30.3, 45.2 -> 42.0, 58 -> 51; 16 x 500 98 -> 79
//                          (not cut here) 4 x 300, 380 50.1 -> 50.3, 52.8 -> 58.0
//     32 heads, 4 groups   1 x 128, 144, 256   26.7 -> 27.5, 32.5 -> 31.6, 45.2 -> 43.2; 4 x 128 27.8 -> 29.2; 16 x 500 99 -> 89
//                          cut: 1 x 340, 1000 45.6 -> 45.8, 58 -> 52; 4 x 380 51 -> 54; 3 x 700 62 -> 66
//     V 128, 2 groups      1 x 128, 144, 200   25.1 -> 26.8, 30.4 -> 30.7, 40.6 -> 38.6; cut: 1 x 340 43.7 -> 44.9, 3 x 700 61 -> 64
//     V 128, 8 heads, 1 group   1 x 128, 200   24.9 -> 25.8, 40.5 -> 36.9; cut: 1 x 300, 500 42.5 -> 41.1, 45.9 -> 43.7; 4 x 300 44.9 -> 47.4
//   for more: from a second chunk on, with few images also one that is full
//     1 group   17 x 20, 33 20.9 -> 21.0, 26.1 -> 22.7; 20 x 20 21.5 -> 22.4; 33 x 20, 48 30.9 -> 28.9, 50 -> 38; 256 x 20 154 -> 137
//     4 groups  24 x 20 21.7 -> 23.7, 48 x 20 32.1 -> 34.0, 17 x 33 26.5 -> 24.7, 64 x 60 66 -> 55; V 128 32 x 64 33.6 -> 34.7
//   an image for less than four workgroups (32 heads, 8 groups): where half the CUs are idle, or the images stay in the caches
//     4 x 160, 256 33.1 -> 34.9, 51 -> 45; 16 x 200, 500 47 -> 51, 99 -> 116; 20 x 40 32.7 -> 33.4, 30 x 100 56 -> 48; 64 x 33,
//     64, 120 56 -> 46, 67 -> 63, 112 -> 115
//   2 x 8192, 32 heads, 1, 4, 8 and 16 groups   356 -> 222, 358 -> 258, 366 -> 317, 368 -> 459
bool ssd_shared_ok(int P, int Tp, int H, int V, int G) {
  if (H / G < 4 || G + (H + 7) / 8 > 65535) return false;
  const int wpi = walk_wgs(H, V, G), cus = device_cus();
  const int64_t wgs = (int64_t)P * wpi;
  const bool light = G <= 2 && V <= 64, whole = wpi >= 4 * G;     // few images; shared by four workgroups
  const auto rows = [&](int n) { return Tp > n * (int64_t)P; };
  if (wgs <= cus) {
    if (!(whole || 2 * wgs <= cus) || !rows(light ? 112 : 160)) return false;
    const int seg = ssd_shared_plan(P, Tp, H, V, G).seg;
    if (seg == 0) return !rows(256) || ssd_chunk_plan(P, Tp, H, V, G).seg == 0;
    return rows(999) || ((light || G == 1) && (P <= 2 || rows(3 * seg - 1)));
  }
  if (!whole) return rows(wgs > 2 * cus ? 24 : 80) && ((int64_t)Tp / L + P) * G * IMG <= 96 << 20;
  return rows(V > 64 && G > 2 && wgs <= 2 * cus ? 64 : 24) || (G <= 2 && wgs > 2 * cus);
}

void launch_ssd_shared(int dtype, float* out, const float* xbc, const void* dt, int64_t dts,
                      const float* a_log, const float* dt_bias, const float* dskip, float* S,
                      const int* qsl, const int* seq_lens, const int* slots, int P, int Tp, int H, int V,
                      int G, int num_slots, const SsdWork& work, void* ws, hipStream_t s) {
  SsdArgs a{};
  a.out = out;
  a.xbc = xbc;
  a.stride = (int64_t)H * V + 2 * (int64_t)G * D;
  a.dt = dt; a.dts = dts; a.dt_type = dtype;
  a.a_log = a_log; a.dt_bias = dt_bias; a.dskip = dskip;
  a.S = S;
  a.qsl = qsl; a.seq_lens = seq_lens; a.slots = slots;
  a.P = P; a.H = H; a.G = G; a.dv = V; a.num_slots = num_slots;
  a.hpw = heads_per_wg(H, V, G);
  a.seg = work.seg;
  a.items = work.items;
  const int64_t chunks = Tp / L + P;
  char* w = static_cast<char*>(ws);
  a.img = w;
  a.rec = reinterpret_cast<TokenRec*>(w + chunks * G * IMG);
  a.seg_state = reinterpret_cast<float*>(w + work.state_at);
  a.seg_gate = reinterpret_cast<double*>(w + work.gate_at);
  ssd_prep_kernel<<<dim3(chunks, G + (H + 7) / 8), NT, 0, s>>>(a);
  const int grid = (work.items + 7) / 8 * 8 * walk_wgs(H, V, G);
  if (V % 2 == 0) walk<true>(a, grid, s);
  else walk<false>(a, grid, s);
}

}  // namespace kgc
