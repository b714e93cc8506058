// Row kernels of the hybrid decoders over an fp32 residual stream:
//   residual_group_norm  x += y (optional); h = grouped RMSNorm(x) * w
//   depth_mix_norm       the end of a depth-averaged layer: store the layer's result,
//                        form the weighted sum of all results so far, norm it for the
//                        next layer -- one pass over the row instead of three kernels
//   head_norm_gate       per-head RMS norm of a recurrence output, weight, sigmoid gate
//   xielu                the xIELU activation
//   gate_proj            a few fp32 gate outputs per row: act(h . w^T + b)
//   residual_norm        x += mult * (add, or RMS-normed add * weight); h = RMSNorm(x) * w
//   residual_sum_norm    x += up to three results, each plain or RMS-normed; h = RMSNorm(x) * w
//   gate_mul, relu_sq, side_gate   element-wise epilogues between GEMMs
// All arithmetic is fp32; T is the activation dtype of h / y (bf16, f16 or fp32).
// One workgroup per row.  Rows of any width are walked twice (sum of squares, then scale), the second
// walk re-reading what the same thread wrote in the first; where vectors fit, the row stays in
// registers.
#include "activation.h"
#include "common.h"
#include "launch.h"

namespace kgc {

namespace {

constexpr int NT = 256;
constexpr int MAX_GROUPS = 64;

// sum of squares per group -> rsqrt(mean + eps), in rs[0..groups)
template <typename F>
__device__ __forceinline__ void group_scales(F&& value, int W, int groups, float eps, float* rs,
                                             float* scratch) {
  const int gw = W / groups;
  for (int g = 0; g < groups; ++g) {
    float ss = 0.f;
    for (int c = g * gw + threadIdx.x; c < (g + 1) * gw; c += NT) {
      const float v = value(c);
      ss += v * v;
    }
    ss = block_sum<NT>(ss, scratch);
    if (threadIdx.x == 0) rs[g] = 1.f / sqrtf(ss / (float)gw + eps);
  }
  __syncthreads();
}

template <typename T>
__global__ __launch_bounds__(NT) void residual_group_norm_kernel(
    T* __restrict__ out, float* __restrict__ x, const T* __restrict__ y,
    const float* __restrict__ w, int W, int groups, float eps) {
  __shared__ float rs[MAX_GROUPS];
  __shared__ float scratch[NT / 64];
  const int64_t row = blockIdx.x;
  float* xr = x + row * W;
  if (y != nullptr) {
    const T* yr = y + row * W;
    for (int c = threadIdx.x; c < W; c += NT) xr[c] += to_f(yr[c]);
  }
  group_scales([&](int c) { return xr[c]; }, W, groups, eps, rs, scratch);
  const int gw = W / groups;
  T* o = out + row * W;
  for (int c = threadIdx.x; c < W; c += NT) o[c] = from_f<T>(xr[c] * rs[c / gw] * w[c]);
}

// hist [L + 1, Tcap, W]; layer result -> hist[layer + 1]; x = sum_j coef[j] hist[j], from sums m.from over
// the results before m.first where an earlier layer began it; A = m.n later layers' sums are begun
template <typename T, int A>
__global__ __launch_bounds__(NT) void depth_mix_norm_kernel(
    T* __restrict__ out, float* __restrict__ x, float* __restrict__ hist,
    const T* __restrict__ y, const float* __restrict__ coef, const float* __restrict__ w,
    int layer, int64_t hist_stride, int W, int groups, float eps, DepthAhead m) {
  __shared__ float rs[MAX_GROUPS];
  __shared__ float scratch[NT / 64];
  const int64_t row = blockIdx.x;
  float* xr = x + row * W;
  const T* yr = y + row * W;
  float* hr = hist + row * W;
  const float own = coef[layer + 1];
  for (int c = threadIdx.x; c < W; c += NT) {
    const float r = xr[c] + to_f(yr[c]);
    hr[(int64_t)(layer + 1) * hist_stride + c] = r;
    float acc = A == 0 && m.from != nullptr ? m.from[row * W + c] : 0.f, ahead[A + 1] = {};
    for (int j = A == 0 ? m.first : 0; j <= layer; ++j) {
      const float h = hr[(int64_t)j * hist_stride + c];
      acc += coef[j] * h;
#pragma unroll
      for (int a = 0; a < A; ++a) ahead[a] += m.coef[a][j] * h;
    }
    xr[c] = acc + own * r;
#pragma unroll
    for (int a = 0; a < A; ++a) m.to[a][row * W + c] = ahead[a] + m.coef[a][layer + 1] * r;
  }
  group_scales([&](int c) { return xr[c]; }, W, groups, eps, rs, scratch);
  const int gw = W / groups;
  T* o = out + row * W;
  for (int c = threadIdx.x; c < W; c += NT) o[c] = from_f<T>(xr[c] * rs[c / gw] * w[c]);
}

// ---- the same by vectors: thread t holds the V float4 at columns 4 (t + 256 k), x and what is added to
// it are read once and the row stays in registers.  Groups of a multiple of 256 columns: a wave's
// float4 of one k lie in one group, so its sums meet in a table behind one barrier, whatever the
// number of groups.  Bound by bytes; 16384 rows of 2048, by elements -> by vectors (us): residual and
// norm 80 -> 58 (8 groups 102 -> 58), depth average over 2 / 7 / 13 results 187 / 362 / 573 -> 118 /
// 243 / 409 (4.6 TB/s; 32 rows, 13 results 15 -> 9), head norm and gate 82 -> 48, xIELU of 8192
// columns 144 -> 99.
template <typename T>
__device__ __forceinline__ float4 ld4(const T* p) {
  if constexpr (sizeof(T) == 4) return *reinterpret_cast<const float4*>(p);
  else {
    Pack4<T> v;
    v.u = *reinterpret_cast<const u32x2*>(p);
    return make_float4(to_f(v.h[0]), to_f(v.h[1]), to_f(v.h[2]), to_f(v.h[3]));
  }
}
template <typename T>
__device__ __forceinline__ void st4(T* p, float4 v) {
  if constexpr (sizeof(T) == 4) *reinterpret_cast<float4*>(p) = v;
  else {
    Pack4<T> o;
    o.h[0] = from_f<T>(v.x);
    o.h[1] = from_f<T>(v.y);
    o.h[2] = from_f<T>(v.z);
    o.h[3] = from_f<T>(v.w);
    *reinterpret_cast<u32x2*>(p) = o.u;
  }
}

// out = x / rms(group of x) * w for the row held in xv (zeros past W)
template <typename T, int V>
__device__ __forceinline__ void group_norm_out(T* o, const float4 (&xv)[V], const float* __restrict__ w,
                                               int W, int gw, float eps, float (&tab)[V * NT / 64]) {
  const int wave = threadIdx.x >> 6;
  float4 wv[V];
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const int c = 4 * (threadIdx.x + NT * k);
    wv[k] = c < W ? ld4(w + c) : make_float4(0.f, 0.f, 0.f, 0.f);
    const float ss = wave_sum((xv[k].x * xv[k].x + xv[k].y * xv[k].y) + (xv[k].z * xv[k].z + xv[k].w * xv[k].w));
    if ((threadIdx.x & 63) == 0) tab[k * (NT / 64) + wave] = ss;
  }
  __syncthreads();
  const int per = gw >> 8;
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const int c = 4 * (threadIdx.x + NT * k), g = (k * (NT / 64) + wave) / per;
    if (c >= W) break;
    float ss = 0.f;
    for (int i = 0; i < per; ++i) ss += tab[g * per + i];
    const float r = 1.f / sqrtf(ss / (float)gw + eps);
    st4(o + c, make_float4(xv[k].x * r * wv[k].x, xv[k].y * r * wv[k].y, xv[k].z * r * wv[k].z,
                           xv[k].w * r * wv[k].w));
  }
}

template <typename T, int V>
__global__ __launch_bounds__(NT) void residual_group_norm_vec_kernel(
    T* __restrict__ out, float* __restrict__ x, const T* __restrict__ y,
    const float* __restrict__ w, int W, int gw, float eps) {
  __shared__ float tab[V * NT / 64];
  const int64_t row = blockIdx.x;
  float* xr = x + row * W;
  float4 xv[V];
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const int c = 4 * (threadIdx.x + NT * k);
    xv[k] = c < W ? ld4(xr + c) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  if (y != nullptr) {
    const T* yr = y + row * W;
#pragma unroll
    for (int k = 0; k < V; ++k) {
      const int c = 4 * (threadIdx.x + NT * k);
      if (c >= W) break;
      const float4 a = ld4(yr + c);
      xv[k] = make_float4(xv[k].x + a.x, xv[k].y + a.y, xv[k].z + a.z, xv[k].w + a.w);
      st4(xr + c, xv[k]);
    }
  }
  group_norm_out<T, V>(out + row * W, xv, w, W, gw, eps, tab);
}

// The averages of A later layers are begun on the way (``m.to``), over the results that exist now: what is read
// here is not read again by them.  A 12-layer stack so reads 26 rows of results and 7 of sums and writes 7
// instead of reading 78, and every sum has the order it has without (14544 rows of 2048 through 12 layers: 2650
// -> 1940 us).  A sum that was begun (FROM) has an instance of its own: asked for in the loop that loads x and y, it made each of their
// loads wait for the one before (16384 rows of 8192 through 2 layers, which begin none, 1167 -> 1282 us).
template <typename T, int V, int A, bool FROM>
__global__ __launch_bounds__(NT) void depth_mix_norm_vec_kernel(
    T* __restrict__ out, float* __restrict__ x, float* __restrict__ hist,
    const T* __restrict__ y, const float* __restrict__ coef, const float* __restrict__ w,
    int layer, int64_t hist_stride, int W, int gw, float eps, DepthAhead m) {
  __shared__ float tab[V * NT / 64];
  const int64_t row = blockIdx.x;
  float* xr = x + row * W;
  const T* yr = y + row * W;
  float* hr = hist + row * W;
  float4 r[V], acc[1 + A][V];
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const int c = min(4 * (int)(threadIdx.x + NT * k), W - 4);
    const float4 a = ld4(xr + c), b = ld4(yr + c);
    r[k] = make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
#pragma unroll
    for (int i = 0; i <= A; ++i) acc[i][k] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (FROM) acc[0][k] = ld4(m.from + row * W + c);
  }
  auto add = [&](float4& s, float cj, const float4& h) {
    s = make_float4(s.x + cj * h.x, s.y + cj * h.y, s.z + cj * h.z, s.w + cj * h.w);
  };
  constexpr int U = V * A > 12 ? 2 : 4;   // rows of 8192 with sums ahead: a second wave per SIMD
#pragma unroll U
  for (int j = FROM ? m.first : 0; j <= layer; ++j) {
#pragma unroll
    for (int k = 0; k < V; ++k) {
      const int c = min(4 * (int)(threadIdx.x + NT * k), W - 4);
      const float4 h = ld4(hr + (int64_t)j * hist_stride + c);
      add(acc[0][k], coef[j], h);
#pragma unroll
      for (int i = 0; i < A; ++i) add(acc[1 + i][k], m.coef[i][j], h);
    }
  }
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const int c = 4 * (threadIdx.x + NT * k);
    add(acc[0][k], coef[layer + 1], r[k]);
#pragma unroll
    for (int i = 0; i < A; ++i) add(acc[1 + i][k], m.coef[i][layer + 1], r[k]);
    if (c < W) {
      st4(hr + (int64_t)(layer + 1) * hist_stride + c, r[k]);
      st4(xr + c, acc[0][k]);
#pragma unroll
      for (int i = 0; i < A; ++i) st4(m.to[i] + row * W + c, acc[1 + i][k]);
    } else {
      acc[0][k] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  group_norm_out<T, V>(out + row * W, acc[0], w, W, gw, eps, tab);
}

// one wave per head vector of dv <= 256 V columns, four of them per workgroup
template <typename T, int V>
__global__ __launch_bounds__(NT) void head_norm_gate_vec_kernel(
    T* __restrict__ out, const float* __restrict__ o, const T* __restrict__ g, int64_t g_stride,
    const float* __restrict__ w, int64_t n, int H, int dv, float eps) {
  const int64_t i = (int64_t)blockIdx.x * (NT / 64) + (threadIdx.x >> 6);
  if (i >= n) return;
  const int64_t row = i / H;
  const int h = (int)(i - row * H), lane = threadIdx.x & 63;
  const T* gr = g + row * g_stride + h * dv;
  float4 ov[V], gv[V], wv[V];
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const int c = 4 * (lane + 64 * k), cc = min(c, dv - 4);
    ov[k] = ld4(o + i * dv + cc);
    gv[k] = ld4(gr + cc);
    wv[k] = ld4(w + h * dv + cc);
    if (c < dv) ss += (ov[k].x * ov[k].x + ov[k].y * ov[k].y) + (ov[k].z * ov[k].z + ov[k].w * ov[k].w);
  }
  const float r = 1.f / sqrtf(wave_sum(ss) / (float)dv + eps);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const int c = 4 * (lane + 64 * k);
    if (c >= dv) break;
    auto f = [&](float a, float b, float z) { return a * r * b * (1.f / (1.f + expf(-z))); };
    st4(out + i * dv + c, make_float4(f(ov[k].x, wv[k].x, gv[k].x), f(ov[k].y, wv[k].y, gv[k].y),
                                      f(ov[k].z, wv[k].z, gv[k].z), f(ov[k].w, wv[k].w, gv[k].w)));
  }
}

// grid (rows, H), 64 threads: o fp32 [rows, H * dv]; g [rows, g_stride] (column slice)
template <typename T>
__global__ __launch_bounds__(64) void head_norm_gate_kernel(
    T* __restrict__ out, const float* __restrict__ o, const T* __restrict__ g, int64_t g_stride,
    const float* __restrict__ w, int H, int dv, float eps) {
  const int64_t row = blockIdx.x;
  const int h = blockIdx.y;
  const float* orow = o + (row * H + h) * dv;
  float ss = 0.f;
  for (int c = threadIdx.x; c < dv; c += 64) ss += orow[c] * orow[c];
  ss = wave_sum(ss);
  const float r = 1.f / sqrtf(ss / (float)dv + eps);
  const T* gr = g + row * g_stride + h * dv;
  T* orr = out + (row * H + h) * dv;
  for (int c = threadIdx.x; c < dv; c += 64) {
    const float gate = 1.f / (1.f + expf(-to_f(gr[c])));
    orr[c] = from_f<T>(orow[c] * r * w[h * dv + c] * gate);
  }
}

template <typename T>
__global__ __launch_bounds__(NT) void xielu_kernel(T* __restrict__ out, const T* __restrict__ z,
                                                   const float* __restrict__ ab, int64_t n) {
  const float a = ab[0], b = ab[1];
  for (int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x; i < n; i += (int64_t)gridDim.x * NT) {
    const float v = to_f(z[i]);
    const float r = v > 0.f ? a * v * v + 0.5f * v : b * (expm1f(v) - v) + 0.5f * v;
    out[i] = from_f<T>(r);
  }
}

// eight 16-bit elements per thread and step
template <typename T>
__global__ __launch_bounds__(NT) void xielu_vec_kernel(T* __restrict__ out, const T* __restrict__ z,
                                                       const float* __restrict__ ab, int64_t n8) {
  const float a = ab[0], b = ab[1];
  for (int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x; i < n8; i += (int64_t)gridDim.x * NT) {
    Pack8<T> v, o;
    v.u = reinterpret_cast<const u32x4*>(z)[i];
#pragma unroll
    for (int j = 0; j < 8; ++j) o.h[j] = from_f<T>(xielu_of(to_f(v.h[j]), a, b));
    reinterpret_cast<u32x4*>(out)[i] = o.u;
  }
}

__device__ __forceinline__ float gate_act(float y, int kind, float cap) {
  if (kind == 0) return 1.f / (1.f + expf(-y));
  if (kind == 3) return y;                            // the plain projection (router logits)
  y = cap * tanhf(y / cap);
  if (kind == 1) return y;
  // logsigmoid(y) = min(y, 0) - log1p(exp(-|y|))
  return fminf(y, 0.f) - log1pf(expf(-fabsf(y)));
}

// Few rows: grid (rows, ceil(N / 4)); the row of h sits in LDS as fp32 and each of the four
// waves computes one output, eight independent 64-column strips at a time so that the
// weight loads of a strip group are all in flight together.
template <typename T>
__global__ __launch_bounds__(NT) void gate_proj_kernel(
    float* __restrict__ out, const T* __restrict__ h, const T* __restrict__ w,
    const float* __restrict__ bias, int W, int N, int kind_a, int kind_b, int split, float cap) {
  extern __shared__ float hrow[];
  const int64_t row = blockIdx.x;
  const T* hr = h + row * W;
  for (int c = threadIdx.x; c < W; c += NT) hrow[c] = to_f(hr[c]);
  __syncthreads();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int n = blockIdx.y * (NT / 64) + wave;
  if (n >= N) return;
  const T* wr = w + (int64_t)n * W;
  float acc = 0.f;
  for (int c0 = lane; c0 < W; c0 += 64 * 8) {
    float wv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int c = c0 + 64 * u;
      wv[u] = c < W ? to_f(wr[c]) : 0.f;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int c = c0 + 64 * u;
      if (c < W) acc += hrow[c] * wv[u];
    }
  }
  acc = wave_sum(acc);
  if (lane == 0) {
    if (bias != nullptr) acc += bias[n];
    out[row * N + n] = gate_act(acc, n < split ? kind_a : kind_b, cap);
  }
}

// Many rows: a workgroup keeps 8 rows of w in registers (thread t: columns t, t + 256, ...)
// and walks rows bx, bx + gridDim.x, ...; per row each thread multiplies its columns of h
// into 8 partial sums, which meet through wave shuffles and a double-buffered LDS table.
template <typename T, int CPT>
__global__ __launch_bounds__(NT) void gate_proj_rows_kernel(
    float* __restrict__ out, const T* __restrict__ h, const T* __restrict__ w,
    const float* __restrict__ bias, int rows, int W, int N, int kind_a, int kind_b, int split,
    float cap) {
  constexpr int NB = 8;
  __shared__ float red[2][NT / 64][NB];
  const int n0 = blockIdx.y * NB;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  float wr[NB][CPT];
#pragma unroll
  for (int n = 0; n < NB; ++n)
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      const int c = threadIdx.x + NT * j;
      wr[n][j] = (n0 + n < N && c < W) ? to_f(w[(int64_t)(n0 + n) * W + c]) : 0.f;
    }
  int it = 0;
  for (int row = blockIdx.x; row < rows; row += gridDim.x, ++it) {
    const T* hr = h + (int64_t)row * W;
    float acc[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) acc[n] = 0.f;
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      const int c = threadIdx.x + NT * j;
      const float hv = c < W ? to_f(hr[c]) : 0.f;
#pragma unroll
      for (int n = 0; n < NB; ++n) acc[n] += hv * wr[n][j];
    }
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      const float t = wave_sum(acc[n]);
      if (lane == 0) red[it & 1][wave][n] = t;
    }
    __syncthreads();
    if (threadIdx.x < NB && n0 + threadIdx.x < N) {
      const int n = n0 + threadIdx.x;
      float t = 0.f;
#pragma unroll
      for (int wv = 0; wv < NT / 64; ++wv) t += red[it & 1][wv][threadIdx.x];
      if (bias != nullptr) t += bias[n];
      out[(int64_t)row * N + n] = gate_act(t, n < split ? kind_a : kind_b, cap);
    }
  }
}

// Many rows of 16-bit activations on the matrix cores: a workgroup takes 16 outputs, its NW waves
// W / NW columns each, and keeps that part of w in registers (S k-steps of 32) while it walks blocks of
// 16 rows: one MFMA per k-step where the kernel above takes 8 cross-lane sums per row and 8 outputs.
// Every product starts from zero and is added in fp32, to four sums in turn: a chain inside the MFMA
// loses more (from float64: 7.4e-8 with the shuffles, 7.35e-8 here).  W a multiple of 32 NW.  Bound by reading h.
template <typename T, int S, int NW>
__global__ __launch_bounds__(NW * 64) void gate_proj_mfma_kernel(
    float* __restrict__ out, const T* __restrict__ h, const T* __restrict__ w,
    const float* __restrict__ bias, int rows, int W, int N, int kind_a, int kind_b, int split,
    float cap) {
  typedef typename Vec8<T>::type V8;
  __shared__ __align__(16) float red[2][NW][16][20];           // [wave][row][output], padded
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r16 = lane & 15, qd = lane >> 4;
  const int n0 = blockIdx.y * 16, steps = W / (32 * NW), c0 = wave * (W / NW) + 8 * qd;
  V8 wf[S];
#pragma unroll
  for (int j = 0; j < S; ++j) {
    Pack8<T> t;
    t.u = u32x4{0u, 0u, 0u, 0u};
    if (j < steps && n0 + r16 < N) t.u = *reinterpret_cast<const u32x4*>(w + (int64_t)(n0 + r16) * W + c0 + 32 * j);
    wf[j] = t.v;
  }
  int it = 0;
  for (int b = blockIdx.x * 16; b < rows; b += gridDim.x * 16, ++it) {
    const T* hr = h + (int64_t)min(b + r16, rows - 1) * W + c0;
    V8 hf[S];
#pragma unroll
    for (int j = 0; j < S; ++j) {
      Pack8<T> t;
      t.u = *reinterpret_cast<const u32x4*>(hr + 32 * min(j, steps - 1));
      hf[j] = t.v;
    }
    f32x4 acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < S; ++j)
      if (j < steps) acc[j & 3] += mfma16x16x32(wf[j], hf[j], f32x4{0.f, 0.f, 0.f, 0.f});
    *reinterpret_cast<f32x4*>(&red[it & 1][wave][r16][4 * qd]) = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    __syncthreads();
    const int row = b + (threadIdx.x >> 4), n = n0 + (threadIdx.x & 15);
    if (threadIdx.x < 256 && row < rows && n < N) {
      const auto& t = red[it & 1];
      const int i = threadIdx.x >> 4, j = threadIdx.x & 15;
      float y = (t[0][i][j] + t[1][i][j]) + (t[2][i][j] + t[3][i][j]);
      if constexpr (NW == 8) y += (t[4][i][j] + t[5][i][j]) + (t[6][i][j] + t[7][i][j]);
      if (bias != nullptr) y += bias[n];
      out[(int64_t)row * N + n] = gate_act(y, n < split ? kind_a : kind_b, cap);
    }
  }
}

}  // namespace

#define KGC_DISPATCH_T(dtype, ...)                          \
  do {                                                      \
    if ((dtype) == DT_BF16) { typedef bf16 T; __VA_ARGS__; } \
    else if ((dtype) == DT_F16) { typedef f16 T; __VA_ARGS__; } \
    else { typedef float T; __VA_ARGS__; }                  \
  } while (0)

static bool al16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }
// rows that 256 threads hold as at most eight float4 each, in groups that waves do not straddle
static bool row_vectors(int W, int gw) { return W <= 8 * 4 * NT && gw % 256 == 0; }
#define KGC_ROW_V(W, GO)         \
  do {                           \
    if ((W) <= 4 * NT) GO(1);    \
    else if ((W) <= 8 * NT) GO(2); \
    else if ((W) <= 16 * NT) GO(4); \
    else GO(8);                  \
  } while (0)

void launch_residual_group_norm(int dtype, void* out, float* x, const void* y, const float* w,
                                int rows, int W, int groups, float eps, hipStream_t s) {
  if (rows <= 0) return;
  const int gw = W / groups;
  if (row_vectors(W, gw) && al16(out) && al16(x) && al16(y) && al16(w)) {
#define KGC_RGN(V)                                                                          \
  KGC_DISPATCH_T(dtype, residual_group_norm_vec_kernel<T, V><<<rows, NT, 0, s>>>(           \
      (T*)out, x, (const T*)y, w, W, gw, eps))
    KGC_ROW_V(W, KGC_RGN);
#undef KGC_RGN
    return;
  }
  KGC_DISPATCH_T(dtype, residual_group_norm_kernel<T><<<rows, NT, 0, s>>>(
      (T*)out, x, (const T*)y, w, W, groups, eps));
}

void launch_depth_mix_norm(int dtype, void* out, float* x, float* hist, const void* y,
                           const float* coef, const float* w, int layer, int64_t hist_stride,
                           int rows, int W, int groups, float eps, const DepthAhead& m, hipStream_t s) {
  if (rows <= 0) return;
  const int gw = W / groups;
  bool vec = row_vectors(W, gw) && hist_stride % 4 == 0 && al16(out) && al16(x) && al16(y) && al16(w) &&
             al16(hist) && al16(m.from);
  for (int i = 0; i < m.n; ++i) vec = vec && al16(m.to[i]);
  if (vec) {
#define KGC_DMN_A(V, A, FROM)                                                               \
  KGC_DISPATCH_T(dtype, depth_mix_norm_vec_kernel<T, V, A, FROM><<<rows, NT, 0, s>>>(       \
      (T*)out, x, hist, (const T*)y, coef, w, layer, hist_stride, W, gw, eps, m))
#define KGC_DMN(V)                                                                          \
  do {                                                                                      \
    if (m.n == 1) KGC_DMN_A(V, 1, false);                                                   \
    else if (m.n == 2) KGC_DMN_A(V, 2, false);                                              \
    else if (m.n == 3) KGC_DMN_A(V, 3, false);                                              \
    else if (m.from != nullptr) KGC_DMN_A(V, 0, true);                                      \
    else KGC_DMN_A(V, 0, false);                                                            \
  } while (0)
    KGC_ROW_V(W, KGC_DMN);
#undef KGC_DMN
#undef KGC_DMN_A
    return;
  }
#define KGC_DMN(A)                                                                          \
  KGC_DISPATCH_T(dtype, depth_mix_norm_kernel<T, A><<<rows, NT, 0, s>>>(                    \
      (T*)out, x, hist, (const T*)y, coef, w, layer, hist_stride, W, groups, eps, m))
  if (m.n == 0) KGC_DMN(0);
  else if (m.n == 1) KGC_DMN(1);
  else if (m.n == 2) KGC_DMN(2);
  else KGC_DMN(3);
#undef KGC_DMN
}

void launch_head_norm_gate(int dtype, void* out, const float* o, const void* g, int64_t g_stride,
                           const float* w, int rows, int H, int dv, float eps, hipStream_t s) {
  if (rows <= 0) return;
  if (dv % 4 == 0 && dv <= 1024 && g_stride % 4 == 0 && al16(out) && al16(o) && al16(w) &&
      reinterpret_cast<uintptr_t>(g) % (dtype == DT_F32 ? 16 : 8) == 0) {
    const int64_t n = (int64_t)rows * H;
#define KGC_HNG(V)                                                                              \
  KGC_DISPATCH_T(dtype, head_norm_gate_vec_kernel<T, V><<<(n + NT / 64 - 1) / (NT / 64), NT, 0, s>>>( \
      (T*)out, o, (const T*)g, g_stride, w, n, H, dv, eps))
    if (dv <= 256) KGC_HNG(1);
    else if (dv <= 512) KGC_HNG(2);
    else KGC_HNG(4);
#undef KGC_HNG
    return;
  }
  KGC_DISPATCH_T(dtype, head_norm_gate_kernel<T><<<dim3(rows, H), 64, 0, s>>>(
      (T*)out, o, (const T*)g, g_stride, w, H, dv, eps));
}

void launch_xielu(int dtype, void* out, const void* z, const float* ab, int64_t n,
                  hipStream_t s) {
  if (n <= 0) return;
  const bool vec = dtype != DT_F32 && n % 8 == 0 && al16(out) && al16(z);
  const int grid = (int)std::min<int64_t>(((vec ? n / 8 : n) + NT - 1) / NT, 256 * 32);
  if (vec) {
    if (dtype == DT_BF16) xielu_vec_kernel<bf16><<<grid, NT, 0, s>>>((bf16*)out, (const bf16*)z, ab, n / 8);
    else xielu_vec_kernel<f16><<<grid, NT, 0, s>>>((f16*)out, (const f16*)z, ab, n / 8);
    return;
  }
  KGC_DISPATCH_T(dtype, xielu_kernel<T><<<grid, NT, 0, s>>>((T*)out, (const T*)z, ab, n));
}

void launch_gate_proj(int dtype, float* out, const void* h, const void* w, const float* bias,
                      int rows, int W, int N, int kind_a, int kind_b, int split, float cap,
                      hipStream_t s) {
  if (rows <= 0) return;
  // at 64 rows as fast as a workgroup per row (8.5 us; 64 outputs at 256 rows 15 -> 8), at 16384 rows of
  // 2048, 16 outputs, 182 -> 19 us against the registers-and-shuffles kernel (64 outputs 571 -> 58)
  if (dtype != DT_F32 && rows >= 64 && W % (W > 2048 ? 256 : 128) == 0 && W <= 4096 && al16(h) && al16(w)) {
    const dim3 grid(std::min((rows + 15) / 16, 512), (N + 15) / 16);
#define KGC_GPM(S, NW)                                                                      \
  do {                                                                                      \
    if (dtype == DT_BF16)                                                                   \
      gate_proj_mfma_kernel<bf16, S, NW><<<grid, NW * 64, 0, s>>>(                          \
          out, (const bf16*)h, (const bf16*)w, bias, rows, W, N, kind_a, kind_b, split, cap); \
    else                                                                                    \
      gate_proj_mfma_kernel<f16, S, NW><<<grid, NW * 64, 0, s>>>(                           \
          out, (const f16*)h, (const f16*)w, bias, rows, W, N, kind_a, kind_b, split, cap); \
  } while (0)
    if (W <= 1024) KGC_GPM(8, 4);
    else if (W <= 2048) KGC_GPM(16, 4);
    else KGC_GPM(16, 8);
#undef KGC_GPM
    return;
  }
  if (rows >= 1024 && W <= 16 * NT) {
    // enough rows to amortise holding w in registers: 8 outputs per workgroup column
    const dim3 grid(1024, (N + 7) / 8);
#define KGC_GP(C)                                                                      \
  KGC_DISPATCH_T(dtype, gate_proj_rows_kernel<T, C><<<grid, NT, 0, s>>>(               \
      out, (const T*)h, (const T*)w, bias, rows, W, N, kind_a, kind_b, split, cap))
    if (W <= 4 * NT) KGC_GP(4);
    else if (W <= 8 * NT) KGC_GP(8);
    else KGC_GP(16);
#undef KGC_GP
    return;
  }
  const size_t lds = (size_t)W * sizeof(float);
  const dim3 grid(rows, (N + NT / 64 - 1) / (NT / 64));
  KGC_DISPATCH_T(dtype, gate_proj_kernel<T><<<grid, NT, lds, s>>>(
      out, (const T*)h, (const T*)w, bias, W, N, kind_a, kind_b, split, cap));
}

// ---- scaled residual + plain RMS norm, head gate, squared ReLU, side-input gate ----------
namespace {

// x += mult * a, a = add or add / rms(add) * anw; then out = x / rms(x) * w (w null: x;
// out null: none).  out may be x itself (O = float).  A thread owns columns threadIdx.x +
// k NT; with EPT > 0 (W <= EPT * NT) it keeps them in registers, so x and add are read once
// and x written once; EPT = 0 walks the row in passes, re-reading only what it wrote.
template <typename T, typename O, int EPT>
__global__ __launch_bounds__(NT) void residual_norm_kernel(
    O* out, float* x, const T* __restrict__ add, const float* __restrict__ anw,
    const float* __restrict__ w, float mult, int W, float eps) {
  __shared__ float scratch[NT / 64];
  const int64_t row = blockIdx.x;
  float* xr = x + row * W;
  if constexpr (EPT > 0) {
    float xv[EPT];
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
      const int c = threadIdx.x + k * NT;
      xv[k] = c < W ? xr[c] : 0.f;
    }
    if (add != nullptr) {
      const T* ar = add + row * W;
      float av[EPT];
#pragma unroll
      for (int k = 0; k < EPT; ++k) {
        const int c = threadIdx.x + k * NT;
        av[k] = c < W ? to_f(ar[c]) : 0.f;
      }
      if (anw != nullptr) {
        float ss = 0.f;
#pragma unroll
        for (int k = 0; k < EPT; ++k) ss += av[k] * av[k];
        ss = block_sum<NT>(ss, scratch);
        const float ra = 1.f / sqrtf(ss / (float)W + eps);
#pragma unroll
        for (int k = 0; k < EPT; ++k) {
          const int c = threadIdx.x + k * NT;
          if (c < W) av[k] = av[k] * ra * anw[c];
        }
      }
#pragma unroll
      for (int k = 0; k < EPT; ++k) {
        const int c = threadIdx.x + k * NT;
        xv[k] += mult * av[k];
        if (c < W) xr[c] = xv[k];
      }
    }
    if (out == nullptr) return;
    O* o = out + row * W;
    float r = 1.f;
    if (w != nullptr) {
      float ss = 0.f;
#pragma unroll
      for (int k = 0; k < EPT; ++k) ss += xv[k] * xv[k];
      ss = block_sum<NT>(ss, scratch);
      r = 1.f / sqrtf(ss / (float)W + eps);
    }
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
      const int c = threadIdx.x + k * NT;
      if (c < W) o[c] = from_f<O>(w != nullptr ? xv[k] * r * w[c] : xv[k]);
    }
    return;
  }
  if (add != nullptr) {
    const T* ar = add + row * W;
    if (anw != nullptr) {
      float ss = 0.f;
      for (int c = threadIdx.x; c < W; c += NT) {
        const float v = to_f(ar[c]);
        ss += v * v;
      }
      ss = block_sum<NT>(ss, scratch);
      const float ra = 1.f / sqrtf(ss / (float)W + eps);
      for (int c = threadIdx.x; c < W; c += NT) xr[c] += mult * (to_f(ar[c]) * ra * anw[c]);
    } else {
      for (int c = threadIdx.x; c < W; c += NT) xr[c] += mult * to_f(ar[c]);
    }
  }
  if (out == nullptr) return;
  O* o = out + row * W;
  if (w == nullptr) {
    for (int c = threadIdx.x; c < W; c += NT) o[c] = from_f<O>(xr[c]);
    return;
  }
  float ss = 0.f;
  for (int c = threadIdx.x; c < W; c += NT) ss += xr[c] * xr[c];
  ss = block_sum<NT>(ss, scratch);
  const float r = 1.f / sqrtf(ss / (float)W + eps);
  for (int c = threadIdx.x; c < W; c += NT) o[c] = from_f<O>(xr[c] * r * w[c]);
}

// x += sum_j a_j, or a_j / rms(a_j) * aw_j where aw_j is given; then out = x / rms(x) * w (out
// null: none).  A thread keeps EPT columns in registers, VEC adjacent ones at a time, so every
// addend and x are read once and x written once; EPT = 0 walks the row in passes.
template <typename T, int VEC>
__device__ __forceinline__ void ld_cols(const T* p, float (&v)[VEC]) {
  if constexpr (VEC == 1) {
    v[0] = to_f(p[0]);
  } else if constexpr (std::is_same_v<T, float>) {
    const float4 t = *reinterpret_cast<const float4*>(p);
    v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
  } else {
    Pack4<T> t;
    t.u = *reinterpret_cast<const u32x2*>(p);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = to_f(t.h[e]);
  }
}
template <typename T, int VEC>
__device__ __forceinline__ void st_cols(T* p, const float (&v)[VEC]) {
  if constexpr (VEC == 1) {
    p[0] = from_f<T>(v[0]);
  } else if constexpr (std::is_same_v<T, float>) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  } else {
    Pack4<T> t;
#pragma unroll
    for (int e = 0; e < 4; ++e) t.h[e] = from_f<T>(v[e]);
    *reinterpret_cast<u32x2*>(p) = t.u;
  }
}

template <typename T, typename O, int EPT, int VEC>
__global__ __launch_bounds__(NT) void residual_sum_norm_kernel(O* __restrict__ out,
                                                               float* __restrict__ x,
                                                               ResidualAdds adds,
                                                               const float* __restrict__ w, int W,
                                                               float eps) {
  __shared__ float scratch[3][NT / 64];
  const int64_t row = blockIdx.x;
  float* xr = x + row * W;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // three sums over the workgroup with one barrier
  auto sums3 = [&](float (&ss)[3]) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      ss[j] = wave_sum(ss[j]);
      if (lane == 0) scratch[j][wave] = ss[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      ss[j] = 0.f;
#pragma unroll
      for (int v = 0; v < NT / 64; ++v) ss[j] += scratch[j][v];
    }
    __syncthreads();
  };
  const bool normed = adds.w[0] != nullptr || adds.w[1] != nullptr || adds.w[2] != nullptr;
  if constexpr (EPT > 0) {
    constexpr int NC = EPT / VEC;
    float xv[NC][VEC], av[3][NC][VEC], ss[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const int c = (threadIdx.x + k * NT) * VEC;
#pragma unroll
      for (int e = 0; e < VEC; ++e) xv[k][e] = 0.f;
      if (c < W) ld_cols<float, VEC>(xr + c, xv[k]);
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const T* ar = static_cast<const T*>(adds.a[j]);
#pragma unroll
      for (int k = 0; k < NC; ++k) {
        const int c = (threadIdx.x + k * NT) * VEC;
#pragma unroll
        for (int e = 0; e < VEC; ++e) av[j][k][e] = 0.f;
        if (ar != nullptr && c < W) ld_cols<T, VEC>(ar + row * W + c, av[j][k]);
#pragma unroll
        for (int e = 0; e < VEC; ++e) ss[j] += av[j][k][e] * av[j][k][e];
      }
    }
    if (normed) sums3(ss);
    float sx = 0.f;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const int c = (threadIdx.x + k * NT) * VEC;
      if (c < W) {
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          if (adds.w[j] != nullptr) {
            const float ra = 1.f / sqrtf(ss[j] / (float)W + eps);
            float wv[VEC];
            ld_cols<float, VEC>(adds.w[j] + c, wv);
#pragma unroll
            for (int e = 0; e < VEC; ++e) xv[k][e] += av[j][k][e] * ra * wv[e];
          } else {
#pragma unroll
            for (int e = 0; e < VEC; ++e) xv[k][e] += av[j][k][e];
          }
        }
        if (adds.a[0] != nullptr) st_cols<float, VEC>(xr + c, xv[k]);
      }
#pragma unroll
      for (int e = 0; e < VEC; ++e) sx += xv[k][e] * xv[k][e];
    }
    if (out == nullptr) return;
    sx = block_sum<NT>(sx, scratch[0]);
    const float r = 1.f / sqrtf(sx / (float)W + eps);
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const int c = (threadIdx.x + k * NT) * VEC;
      if (c < W) {
        float wv[VEC], o[VEC];
        ld_cols<float, VEC>(w + c, wv);
#pragma unroll
        for (int e = 0; e < VEC; ++e) o[e] = xv[k][e] * r * wv[e];
        st_cols<O, VEC>(out + row * W + c, o);
      }
    }
    return;
  }
  float ss[3] = {0.f, 0.f, 0.f};
  if (normed) {
    for (int c = threadIdx.x; c < W; c += NT)
#pragma unroll
      for (int j = 0; j < 3; ++j)
        if (adds.w[j] != nullptr) {
          const float v = to_f(static_cast<const T*>(adds.a[j])[row * W + c]);
          ss[j] += v * v;
        }
    sums3(ss);
  }
  float sx = 0.f;
  for (int c = threadIdx.x; c < W; c += NT) {
    float v = xr[c];
#pragma unroll
    for (int j = 0; j < 3; ++j)
      if (adds.a[j] != nullptr) {
        float a = to_f(static_cast<const T*>(adds.a[j])[row * W + c]);
        if (adds.w[j] != nullptr) a = a * (1.f / sqrtf(ss[j] / (float)W + eps)) * adds.w[j][c];
        v += a;
      }
    xr[c] = v;
    sx += v * v;
  }
  if (out == nullptr) return;
  sx = block_sum<NT>(sx, scratch[0]);
  const float r = 1.f / sqrtf(sx / (float)W + eps);
  for (int c = threadIdx.x; c < W; c += NT) out[row * W + c] = from_f<O>(xr[c] * r * w[c]);
}

// out [T, H * dv] (row stride so) = o[t, h, :] (strides st, sh) * sigmoid(g[t, h * dv + :])
// (row stride sg) * scale
template <typename T>
__global__ __launch_bounds__(NT) void gate_mul_kernel(
    T* __restrict__ out, int64_t so, const T* __restrict__ o, int64_t st, int64_t sh,
    const T* __restrict__ g, int64_t sg, int H, int dv, float scale) {
  const int64_t t = blockIdx.x;
  const int n = H * dv;
  for (int e = threadIdx.x; e < n; e += NT) {
    const int h = e / dv, c = e - h * dv;
    const float gate = 1.f / (1.f + expf(-to_f(g[t * sg + e])));
    out[t * so + e] = from_f<T>(to_f(o[t * st + h * sh + c]) * gate * scale);
  }
}

template <typename T>
__global__ __launch_bounds__(NT) void relu_sq_kernel(T* __restrict__ out, const T* __restrict__ z,
                                                     int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x; i < n; i += (int64_t)gridDim.x * NT) {
    const float v = fmaxf(to_f(z[i]), 0.f);
    out[i] = from_f<T>(v * v);
  }
}

// out [T, n] = gelu_tanh(pre [T, n]) * table[ids[t], col0 + :] (table row stride ts)
template <typename T>
__global__ __launch_bounds__(NT) void side_gate_kernel(
    T* __restrict__ out, const T* __restrict__ pre, const int64_t* __restrict__ ids,
    const T* __restrict__ table, int64_t ts, int vocab, int col0, int n) {
  const int64_t t = blockIdx.x;
  int64_t id = ids[t];
  if (id < 0 || id >= vocab) id = 0;                  // never read outside the table
  const T* e = table + id * ts + col0;
  for (int c = threadIdx.x; c < n; c += NT) {
    const float z = to_f(pre[t * n + c]);
    const float gl = 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
    out[t * n + c] = from_f<T>(gl * to_f(e[c]));
  }
}

// The per-token side input of a layer for a few rows (decode steps), one workgroup per row:
//   x += mult * y;  pre = W_g x;  g = gelu_tanh(pre) * table[id, col0 + :];  v = W_p g;
//   x += mult * v / rms(v) * sw;  out = x / rms(x) * w  (w null: no output)
// in one kernel instead of a cast, two small GEMMs, the gate and the add + norm.  Products
// accumulate in fp32 and are rounded to T where the GEMM path rounds (its inputs and
// outputs), so rows that take this kernel agree with rows that take the GEMMs to rounding
// order.  16-bit T, W % 8 == 0, W <= EPT * 1024 threads, n % 8 == 0, n <= 512.
constexpr int SI_NT = 1024, SI_JB = 4;

template <typename T, typename O, int EPT>
__global__ __launch_bounds__(SI_NT) void side_input_rows_kernel(
    O* out, float* x, const T* __restrict__ y, const T* __restrict__ wg,
    const T* __restrict__ wp, const int64_t* __restrict__ ids, const T* __restrict__ table,
    int64_t ts, int vocab, int col0, const float* __restrict__ sw, const float* __restrict__ w,
    float mult, int W, int n, float eps) {
  extern __shared__ float lds[];
  float* xb = lds;                 // [W]: x as the GEMM reads it (rounded to T)
  float* gs = lds + W;             // [n]
  __shared__ float scratch[SI_NT / 64];
  const int64_t row = blockIdx.x;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  float* xr = x + row * W;
  float xv[EPT];
#pragma unroll
  for (int k = 0; k < EPT; ++k) {
    const int c = threadIdx.x + k * SI_NT;
    xv[k] = 0.f;
    if (c < W) {
      xv[k] = xr[c] + (y != nullptr ? mult * to_f(y[row * W + c]) : 0.f);
      xb[c] = to_f(from_f<T>(xv[k]));
    }
  }
  __syncthreads();
  int64_t id = ids[row];
  if (id < 0 || id >= vocab) id = 0;
  const T* e = table + id * ts + col0;
  const int chunks = W >> 3;
  // a wave takes SI_JB outputs at a time, their weight rows' loads all in flight
  constexpr int NWV = SI_NT / 64;
  for (int j0 = wave * SI_JB; j0 < n; j0 += NWV * SI_JB) {
    float acc[SI_JB];
#pragma unroll
    for (int b = 0; b < SI_JB; ++b) acc[b] = 0.f;
    for (int ch = lane; ch < chunks; ch += 64) {
      Pack8<T> p[SI_JB];
#pragma unroll
      for (int b = 0; b < SI_JB; ++b)
        p[b].u = *reinterpret_cast<const u32x4*>(wg + (int64_t)min(j0 + b, n - 1) * W + 8 * ch);
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const float xq = xb[8 * ch + q];
#pragma unroll
        for (int b = 0; b < SI_JB; ++b) acc[b] += xq * to_f(p[b].h[q]);
      }
    }
#pragma unroll
    for (int b = 0; b < SI_JB; ++b) {
      const float tot = wave_sum(acc[b]);
      const int j = j0 + b;
      if (lane == 0 && j < n) {
        const float z = to_f(from_f<T>(tot));
        const float gl = 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
        gs[j] = to_f(from_f<T>(gl * to_f(e[j])));
      }
    }
  }
  __syncthreads();
  float vv[EPT], ss = 0.f;
#pragma unroll
  for (int k = 0; k < EPT; ++k) {
    const int c = threadIdx.x + k * SI_NT;
    vv[k] = 0.f;
    if (c < W) {
      const T* pr = wp + (int64_t)c * n;
      float acc = 0.f;
      for (int j0 = 0; j0 < n; j0 += 8) {
        Pack8<T> p;
        p.u = *reinterpret_cast<const u32x4*>(pr + j0);
#pragma unroll
        for (int q = 0; q < 8; ++q) acc += gs[j0 + q] * to_f(p.h[q]);
      }
      vv[k] = to_f(from_f<T>(acc));
      ss += vv[k] * vv[k];
    }
  }
  ss = block_sum<SI_NT>(ss, scratch);
  const float ra = 1.f / sqrtf(ss / (float)W + eps);
  float s2 = 0.f;
#pragma unroll
  for (int k = 0; k < EPT; ++k) {
    const int c = threadIdx.x + k * SI_NT;
    if (c < W) {
      xv[k] += mult * (vv[k] * ra * sw[c]);
      xr[c] = xv[k];
      s2 += xv[k] * xv[k];
    }
  }
  if (out == nullptr || w == nullptr) return;
  s2 = block_sum<SI_NT>(s2, scratch);
  const float r = 1.f / sqrtf(s2 / (float)W + eps);
  O* o = out + row * W;
#pragma unroll
  for (int k = 0; k < EPT; ++k) {
    const int c = threadIdx.x + k * SI_NT;
    if (c < W) o[c] = from_f<O>(xv[k] * r * w[c]);
  }
}

}  // namespace

bool side_input_rows_ok(int dtype, int rows, int W, int n) {
  return (dtype == DT_BF16 || dtype == DT_F16) && rows <= 256 && W % 8 == 0 && W <= 4 * SI_NT &&
         n % 8 == 0 && n <= 512;
}

void launch_side_input_rows(int dtype, int out_dtype, void* out, float* x, const void* y,
                            const void* wg, const void* wp, const int64_t* ids,
                            const void* table, int64_t ts, int vocab, int col0, const float* sw,
                            const float* w, float mult, int rows, int W, int n, float eps,
                            hipStream_t s) {
  if (rows <= 0) return;
  const size_t lds = (size_t)(W + n) * sizeof(float);
#define KGC_SI(T, O, EPT)                                                                     \
  side_input_rows_kernel<T, O, EPT><<<rows, SI_NT, lds, s>>>(                                  \
      (O*)out, x, (const T*)y, (const T*)wg, (const T*)wp, ids, (const T*)table, ts, vocab,   \
      col0, sw, w, mult, W, n, eps)
#define KGC_SI_W(T, O)                     \
  do {                                     \
    if (W <= SI_NT) KGC_SI(T, O, 1);          \
    else if (W <= 2 * SI_NT) KGC_SI(T, O, 2); \
    else KGC_SI(T, O, 4);                     \
  } while (0)
  const bool f32out = out == nullptr || out_dtype == DT_F32;
  if (dtype == DT_BF16) {
    if (f32out) KGC_SI_W(bf16, float); else KGC_SI_W(bf16, bf16);
  } else {
    if (f32out) KGC_SI_W(f16, float); else KGC_SI_W(f16, f16);
  }
#undef KGC_SI_W
#undef KGC_SI
}

void launch_residual_norm(int dtype, int out_dtype, void* out, float* x, const void* add,
                          const float* anw, const float* w, float mult, int rows, int W,
                          float eps, hipStream_t s) {
  if (rows <= 0) return;
#define KGC_RN(O, EPT)                                                          \
  residual_norm_kernel<T, O, EPT><<<rows, NT, 0, s>>>((O*)out, x, (const T*)add, anw, w, mult, \
                                                      W, eps)
#define KGC_RN_W(O)                      \
  do {                                   \
    if (W <= 4 * NT) KGC_RN(O, 4);       \
    else if (W <= 8 * NT) KGC_RN(O, 8);  \
    else if (W <= 16 * NT) KGC_RN(O, 16); \
    else KGC_RN(O, 0);                   \
  } while (0)
  if (out == nullptr || out_dtype == DT_F32) {
    KGC_DISPATCH_T(dtype, KGC_RN_W(float));
  } else {
    KGC_DISPATCH_T(dtype, KGC_RN_W(T));
  }
#undef KGC_RN_W
#undef KGC_RN
}

void launch_residual_sum_norm(int dtype, int out_dtype, void* out, float* x, ResidualAdds adds,
                              const float* w, int rows, int W, float eps, hipStream_t s) {
  if (rows <= 0) return;
  bool vec = W % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
             reinterpret_cast<uintptr_t>(out) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0;
  for (int j = 0; j < 3; ++j)
    vec = vec && reinterpret_cast<uintptr_t>(adds.a[j]) % 16 == 0 &&
          reinterpret_cast<uintptr_t>(adds.w[j]) % 16 == 0;
#define KGC_RSN(O, EPT, V) \
  residual_sum_norm_kernel<T, O, EPT, V><<<rows, NT, 0, s>>>((O*)out, x, adds, w, W, eps)
#define KGC_RSN_W(O)                                 \
  do {                                               \
    if (vec && W <= 4 * NT) KGC_RSN(O, 4, 4);        \
    else if (vec && W <= 8 * NT) KGC_RSN(O, 8, 4);   \
    else if (vec && W <= 16 * NT) KGC_RSN(O, 16, 4); \
    else if (W <= 4 * NT) KGC_RSN(O, 4, 1);          \
    else KGC_RSN(O, 0, 1);                           \
  } while (0)
  if (out == nullptr || out_dtype == DT_F32) {
    KGC_DISPATCH_T(dtype, KGC_RSN_W(float));
  } else {
    KGC_DISPATCH_T(dtype, KGC_RSN_W(T));
  }
#undef KGC_RSN_W
#undef KGC_RSN
}

void launch_gate_mul(int dtype, void* out, int64_t so, const void* o, int64_t st, int64_t sh,
                     const void* g, int64_t sg, int rows, int H, int dv, float scale,
                     hipStream_t s) {
  if (rows <= 0) return;
  KGC_DISPATCH_T(dtype, gate_mul_kernel<T><<<rows, NT, 0, s>>>((T*)out, so, (const T*)o, st, sh,
                                                              (const T*)g, sg, H, dv, scale));
}

void launch_relu_sq(int dtype, void* out, const void* z, int64_t n, hipStream_t s) {
  if (n <= 0) return;
  const int grid = (int)std::min<int64_t>((n + NT - 1) / NT, 256 * 32);
  KGC_DISPATCH_T(dtype, relu_sq_kernel<T><<<grid, NT, 0, s>>>((T*)out, (const T*)z, n));
}

void launch_side_gate(int dtype, void* out, const void* pre, const int64_t* ids,
                      const void* table, int64_t ts, int vocab, int col0, int rows, int n,
                      hipStream_t s) {
  if (rows <= 0) return;
  KGC_DISPATCH_T(dtype, side_gate_kernel<T><<<rows, NT, 0, s>>>(
      (T*)out, (const T*)pre, ids, (const T*)table, ts, vocab, col0, n));
}

}  // namespace kgc
