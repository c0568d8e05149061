// Kernels of the fused training regions on gfx950: the frozen-feature (perceptual) loss of
// the reference's xdna_train/regions.py:1-425 (its host kernels: _native/region_kernels.cpp:
// 51-340), re-designed for device memory.  The region's convolutions are the 3x3 conv path
// with a fused ReLU epilogue; what is left for these kernels is one pass per tensor:
//
//   * 2x2 / stride-2 max-pool (PyTorch's rule: the first maximum of the window in row-major
//     order wins, a NaN wins over any number);
//   * tap loss terms as fp32 partial sums over a fixed partition of the elements (one slab
//     per tap, each pre-scaled), and one fixed-order finish into the scalar loss, so the
//     loss never leaves the device and the same inputs give the same bits;
//   * the backward of ReLU, max-pool and the tap terms in one elementwise pass:
//       out = mask ? bf16(base + extra + scale * go * (a - b)) : 0
//     with base the incoming gradient or, through a max-pool, the pooled gradient routed
//     to the window's maximum (recomputed from the pool input, same rule as the forward),
//     and mask the ReLU result's positivity (threshold_backward: a NaN result passes);
//   * the Gram-matrix style term: sum of (G / chw - T)^2, and the symmetric matrix S with
//     which the gradient with respect to the features F (G = F F^T) is one product, S F.
//
// bf16 storage, fp32 arithmetic, one rounding per output, as the reference's region
// contract states (regions.py:29-32).  Scalars that come from autograd (the loss's
// incoming gradient) are read on the device, so a region's backward needs no host sync and
// can be captured in a graph.
#include "common.h"

#include <algorithm>
#include <cmath>
#include "../../include/xdna_hip.h"

namespace xdna {
namespace {

constexpr int kRegionThreads = 256;
constexpr int kLossParts = 2048;  // partial sums per tap term (fixed partition)

__device__ inline float go_value(const void* go, int go_dtype) {
  if (go_dtype == 1) return *static_cast<const float*>(go);
  if (go_dtype == 2) return bf16_to_f32(*static_cast<const uint16_t*>(go));
  return 1.0f;
}

// Row-major index (0..3) of the window maximum: (0,0), (0,1), (1,0), (1,1); a value
// replaces the running maximum when it is larger or NaN (PyTorch's max_pool2d rule).
__device__ inline int argmax4(const float (&v)[4], float* max = nullptr) {
  float m = -INFINITY;
  int k = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (v[j] > m || v[j] != v[j]) {
      m = v[j];
      k = j;
    }
  if (max) *max = m;
  return k;
}

__global__ __launch_bounds__(kRegionThreads) void maxpool2_kernel(const uint16_t* __restrict__ x,
                                                                  uint16_t* __restrict__ y, int64_t planes, int H,
                                                                  int W, int Ho, int Wo) {
  const int64_t n = planes * Ho * Wo;
  for (int64_t i = int64_t(blockIdx.x) * kRegionThreads + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * kRegionThreads) {
    const int64_t p = i / (int64_t(Ho) * Wo);
    const int r = int(i - p * Ho * Wo);
    const int oy = r / Wo, ox = r - oy * Wo;
    const uint16_t* w0 = x + (p * H + 2 * oy) * W + 2 * ox;
    const float v[4] = {bf16_to_f32(w0[0]), bf16_to_f32(w0[1]), bf16_to_f32(w0[W]), bf16_to_f32(w0[W + 1])};
    float m;
    argmax4(v, &m);
    y[i] = f32_to_bf16(m);
  }
}

struct BwdArgs {
  const uint16_t* r;      // ReLU result (mask), or null
  const uint16_t* g;      // incoming gradient at this shape, or null
  const uint16_t* gp;     // incoming gradient at the pooled shape, or null
  const uint16_t* px;     // max-pool input (for the window maxima), with gp
  const uint16_t* extra;  // another gradient term at this shape, or null
  const uint16_t* ta;     // tap term a - b, or null
  const uint16_t* tb;
  const void* go;
  int go_dtype;
  float scale;
  uint16_t* out;
  int64_t planes;
  int H, W, Ho, Wo;
};

// The four elements from i of a tensor of `total` in the low bits on (past the last: anything).  The
// load is whole and unconditional, so that a kernel's loads fly together: one that ends past the
// tensor is moved back and shifted.  Tensors of fewer than four elements are read one by one.
__device__ inline uint64_t load4(const uint16_t* p, int64_t i, int64_t total) {
  if (total < 4) {
    uint64_t v = 0;
    for (int u = 0; i + u < total; ++u) v |= uint64_t(p[i + u]) << (16 * u);
    return v;
  }
  const int64_t b = i < total - 4 ? i : total - 4;
  const Pix4 a = *reinterpret_cast<const Pix4*>(p + b);
  return (a.lo | (uint64_t(a.hi) << 32)) >> (16 * int(i - b));
}

__device__ inline float val4(uint64_t v, int u) { return bf16_to_f32(uint16_t(v >> (16 * u))); }

__device__ inline void store4(uint16_t* p, int n, const float (&v)[4]) {
  uint16_t h[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) h[u] = f32_to_bf16(v[u]);
  if (n >= 4) {
    *reinterpret_cast<Pix4*>(p) = Pix4{h[0] | (uint32_t(h[1]) << 16), h[2] | (uint32_t(h[3]) << 16)};
  } else {
#pragma unroll
    for (int u = 0; u < 3; ++u)
      if (u < n) p[u] = h[u];
  }
}

// The mask and the terms beside the base gradient of four elements: loaded, then applied.
struct Terms4 {
  uint64_t extra, ta, tb, r;
};

__device__ inline Terms4 load_terms(const BwdArgs& a, int64_t i, int64_t total) {
  Terms4 t = {0, 0, 0, 0};
  if (a.extra) t.extra = load4(a.extra, i, total);
  if (a.ta) t.ta = load4(a.ta, i, total), t.tb = load4(a.tb, i, total);
  if (a.r) t.r = load4(a.r, i, total);
  return t;
}

__device__ inline void region_terms(const BwdArgs& a, float s, const Terms4& t, float (&v)[4]) {
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    if (a.extra) v[u] += val4(t.extra, u);
    if (a.ta) v[u] += s * (val4(t.ta, u) - val4(t.tb, u));
    if (a.r) v[u] = val4(t.r, u) <= 0.0f ? 0.0f : v[u];
  }
}

// Memory bound: four elements per thread, the loads of all terms in flight before the mask is
// known (one element per thread, masked before its other loads, was a chain of two or three
// latencies on 2-byte loads; us on 40 x 64 x 36 x 36, a tensor 1.3: r and g 9.7 -> 4.6, with
// extra and a tap 10.3 -> 5.7).
__global__ __launch_bounds__(kRegionThreads) void region_bwd_kernel(BwdArgs a) {
  const int64_t n = a.planes * a.H * a.W;
  const float s = a.ta ? a.scale * go_value(a.go, a.go_dtype) : 0.0f;
  for (int64_t i = (int64_t(blockIdx.x) * kRegionThreads + threadIdx.x) * 4; i < n;
       i += int64_t(gridDim.x) * kRegionThreads * 4) {
    const uint64_t g = a.g ? load4(a.g, i, n) : 0;
    const Terms4 t = load_terms(a, i, n);
    float v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = val4(g, u);
    region_terms(a, s, t, v);
    store4(a.out + i, int(std::min<int64_t>(4, n - i)), v);
  }
}

// One element per thread, through the max-pool too: small tensors, where the other forms' longer
// code, not memory, is the time (with the pool, extra and a mask 3.1 us against 4.1 up to 100k
// elements, level at 400k; without the pool, with extra and a tap, 2.9 against 3.2, level at 200k).
__global__ __launch_bounds__(kRegionThreads) void region_bwd_small_kernel(BwdArgs a) {
  const int n = int(a.planes * a.H * a.W), i = int(blockIdx.x) * kRegionThreads + int(threadIdx.x);
  if (i >= n) return;
  const float s = a.ta ? a.scale * go_value(a.go, a.go_dtype) : 0.0f;
  if (a.r && bf16_to_f32(a.r[i]) <= 0.0f) {
    a.out[i] = 0;
    return;
  }
  float v = 0.0f;
  if (a.g) {
    v = bf16_to_f32(a.g[i]);
  } else if (a.gp) {
    const int row = i / a.W, x = i - row * a.W, p = row / a.H, y = row - p * a.H;
    const int oy = y >> 1, ox = x >> 1;
    if (oy < a.Ho && ox < a.Wo) {
      const uint16_t* w0 = a.px + (p * a.H + 2 * oy) * a.W + 2 * ox;
      const float w[4] = {bf16_to_f32(w0[0]), bf16_to_f32(w0[1]), bf16_to_f32(w0[a.W]), bf16_to_f32(w0[a.W + 1])};
      if (argmax4(w) == ((y & 1) << 1) + (x & 1)) v = bf16_to_f32(a.gp[(p * a.Ho + oy) * a.Wo + ox]);
    }
  }
  if (a.extra) v += bf16_to_f32(a.extra[i]);
  if (a.ta) v += s * (bf16_to_f32(a.ta[i]) - bf16_to_f32(a.tb[i]));
  a.out[i] = f32_to_bf16(v);
}

// Through the max-pool: a thread takes four columns of the two rows of a window row, so a
// window's maximum is found once, not by each of its pixels (40 x 64 x 36 x 36 with extra: 14.4
// -> 6.2 us).  I: the index type that holds the item count.
template <class I>
__global__ __launch_bounds__(kRegionThreads) void region_bwd_pool_kernel(BwdArgs a) {
  const I wq = I((a.W + 3) / 4), hq = I((a.H + 1) / 2), n = I(a.planes) * hq * wq;
  const int64_t total = a.planes * a.H * a.W, pooled = a.planes * a.Ho * a.Wo;
  const float s = a.ta ? a.scale * go_value(a.go, a.go_dtype) : 0.0f;
  for (I i = I(blockIdx.x) * kRegionThreads + threadIdx.x; i < n; i += I(gridDim.x) * kRegionThreads) {
    const I row = i / wq;
    const int x = 4 * int(i - row * wq);
    const I p = row / hq;
    const int oy = int(row - p * hq), y = 2 * oy, m = min(4, a.W - x);
    const int64_t at = (int64_t(p) * a.H + y) * a.W + x;
    const bool two = y + 1 < a.H;
    const int64_t below = two ? at + a.W : at;
    const uint64_t r0 = load4(a.px, at, total), r1 = load4(a.px, below, total);
    const Terms4 t0 = load_terms(a, at, total), t1 = load_terms(a, below, total);
    // (the windows of the two column pairs; past the last one: anything)
    const int64_t gi = (int64_t(p) * a.Ho + oy) * a.Wo + (x >> 1);
    const float g[2] = {pooled ? bf16_to_f32(a.gp[gi < pooled ? gi : pooled - 1]) : 0.0f,
                        pooled ? bf16_to_f32(a.gp[gi + 1 < pooled ? gi + 1 : pooled - 1]) : 0.0f};
    float v[2][4] = {};
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (!two || 2 * j + 1 >= m) continue;  // no window (an odd last row or column)
      const float w[4] = {val4(r0, 2 * j), val4(r0, 2 * j + 1), val4(r1, 2 * j), val4(r1, 2 * j + 1)};
      const int k = argmax4(w);
      v[0][2 * j] = k == 0 ? g[j] : 0.0f;
      v[0][2 * j + 1] = k == 1 ? g[j] : 0.0f;
      v[1][2 * j] = k == 2 ? g[j] : 0.0f;
      v[1][2 * j + 1] = k == 3 ? g[j] : 0.0f;
    }
    region_terms(a, s, t0, v[0]);
    store4(a.out + at, m, v[0]);
    if (two) {
      region_terms(a, s, t1, v[1]);
      store4(a.out + below, m, v[1]);
    }
  }
}

struct __attribute__((packed, aligned(4))) F32x4 {
  float v[4];
};

// part[blockIdx.x] = scale * the block's sum of s, by a fixed tree
__device__ inline void block_part(float s, float scale, float* part) {
  __shared__ float red[kRegionThreads];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = kRegionThreads / 2; w > 0; w >>= 1) {
    if (int(threadIdx.x) < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = scale * red[0];
}

// part[blockIdx.x] = scale * sum over this block's elements of (a - b)^2.  Block b sums
// elements b * 256 + tid + k * gridDim.x * 256 in that order per thread, then a fixed tree.
// (Wider runs per thread leave half of the blocks without work at 3.3M elements: 3.8 us so,
// 4.4 with eight.)
__global__ __launch_bounds__(kRegionThreads) void sqdiff_kernel(const uint16_t* __restrict__ a,
                                                                const uint16_t* __restrict__ b, int64_t n,
                                                                float scale, float* __restrict__ part) {
  float s = 0.0f;
  for (int64_t i = int64_t(blockIdx.x) * kRegionThreads + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * kRegionThreads) {
    const float d = bf16_to_f32(a[i]) - bf16_to_f32(b[i]);
    s = fmaf(d, d, s);
  }
  block_part(s, scale, part);
}

// The same of (G / chw - t)^2: G the bf16 Gram matrices [batch][cc], t fp32 targets with batch
// stride t_bstride, 0 for one target broadcast over the batch.  A thread sums runs of eight (at
// 8 (b * 256 + tid) + k * gridDim.x * 2048) in order, each divided once, in 32 bits where it fits (a
// 64-bit division per element held 40 matrices of 512 x 512 to 14.2 us; now 8.0, the bytes' time is
// 4; 30 of 471 x 471 10.7).  A run that crosses into the next matrix, or ends the last, is read
// element by element, all loads in flight.
// kSmall: no more elements than threads, one each (3.3 us; the runs' code alone 0.2-0.9 more).
template <bool kSmall>
__global__ __launch_bounds__(kRegionThreads) void gram_sqdiff_kernel(const uint16_t* __restrict__ G,
                                                                     const float* __restrict__ t, int64_t t_bstride,
                                                                     int64_t cc, float chw, int64_t n, float scale,
                                                                     float* __restrict__ part) {
  float s = 0.0f;
  if constexpr (kSmall) {
    const uint32_t i = blockIdx.x * kRegionThreads + threadIdx.x;
    if (i < n) {
      const uint32_t bi = i / uint32_t(cc);
      const float d = bf16_to_f32(G[i]) / chw - t[bi * t_bstride + (i - bi * cc)];
      s = d * d;
    }
    block_part(s, scale, part);
    return;
  }
  for (int64_t i = (int64_t(blockIdx.x) * kRegionThreads + threadIdx.x) * 8; i < n;
       i += int64_t(gridDim.x) * kRegionThreads * 8) {
    const int64_t bi = (i | cc) >> 32 ? i / cc : uint32_t(i) / uint32_t(cc);
    const float* tp = t + bi * t_bstride;
    int64_t r = i - bi * cc;
    float g[8], w[8];
    if (r + 8 <= cc) {  // (then i + 8 <= n)
      const Pix8 x = *reinterpret_cast<const Pix8*>(G + i);
      const F32x4 lo = *reinterpret_cast<const F32x4*>(tp + r), hi = *reinterpret_cast<const F32x4*>(tp + r + 4);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        g[u] = bf16_to_f32(uint16_t(x.v[u >> 1] >> (16 * (u & 1))));
        w[u] = u < 4 ? lo.v[u & 3] : hi.v[u & 3];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float d = g[u] / chw - w[u];
        s = fmaf(d, d, s);
      }
    } else {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const bool in = i + u < n;  // (past the end: the run's first element again)
        const float* tu = in ? tp + r : t;
        g[u] = bf16_to_f32(G[in ? i + u : i]);
        w[u] = *tu;
        if (++r == cc) r = 0, tp += t_bstride;
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float d = g[u] / chw - w[u];
        if (i + u < n) s = fmaf(d, d, s);
      }
    }
  }
  block_part(s, scale, part);
}

// loss = sum of part[0 .. n) in fp64, thread-strided then a fixed tree; written as fp32
// and bf16 scalars (either may be null).
constexpr int kFinishThreads = 1024;

__global__ __launch_bounds__(kFinishThreads) void finish_kernel(const float* __restrict__ part, int n,
                                                                float* __restrict__ out_f32,
                                                                uint16_t* __restrict__ out_bf16) {
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += kFinishThreads) s += double(part[i]);
  __shared__ double red[kFinishThreads];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = kFinishThreads / 2; w > 0; w >>= 1) {
    if (int(threadIdx.x) < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    if (out_f32) *out_f32 = float(red[0]);
    if (out_bf16) *out_bf16 = f32_to_bf16(float(red[0]));
  }
}

// S = bf16(coef * go * (d_ij + d_ji) / chw), d = G / chw - t, over C x C matrices: with
// G = F F^T, the gradient of coef / 2 * sum d^2 with respect to F is S F (both operands of
// the Gram product carry F), so one product gives it (coef = 2 w / N for w times a mean).
// S is symmetric, so a block takes the 32 x 32 tile at (ti, tj) of matrix blockIdx.z and
// its mirror image: d is read once, four elements per thread, exchanged through LDS, and
// both tiles are written.  The grid folds tile row y onto row nt - 1 - y: nt + 1 tiles on or
// above the diagonal per pair of rows (x first the row's, then its partner's).  40 matrices of
// 512 x 512: 25.2 us with every tile and its mirror read by its own block -> 13.9 (bytes: 8).
constexpr int kGT = 32;

__global__ __launch_bounds__(kRegionThreads) void gram_grad_kernel(const uint16_t* __restrict__ G,
                                                                   const float* __restrict__ t, int64_t t_bstride,
                                                                   int C, float chw, float coef, const void* go,
                                                                   int go_dtype, uint16_t* __restrict__ S) {
  const int nt = (C + kGT - 1) / kGT;
  int ti = blockIdx.y, tj = ti + int(blockIdx.x);
  if (tj >= nt) {
    if (nt - 1 - ti == ti) return;  // the middle row has no partner
    tj = int(blockIdx.x) - (nt - ti);
    ti = nt - 1 - ti;
    tj += ti;
  }
  const float c = coef * go_value(go, go_dtype);
  const int64_t cc = int64_t(C) * C;
  const uint16_t* Gb = G + blockIdx.z * cc;
  const float* tb = t + blockIdx.z * t_bstride;
  uint16_t* Sb = S + blockIdx.z * cc;
  __shared__ float tile[2][kGT][kGT + 1];
  const int y = threadIdx.x / 8, x = 4 * (threadIdx.x % 8);
  float d[2][4];
  const bool whole = (tj + 1) * kGT <= C;  // (ti <= tj) else elements, clamped: what is past the matrix is not stored
#pragma unroll
  for (int h = 0; h < 2; ++h) {  // the tile, its mirror
    const int r = (h ? tj : ti) * kGT + y, col = (h ? ti : tj) * kGT + x;
    float g[4], w[4];
    if (whole) {
      const int64_t e = int64_t(r) * C + col;
      const Pix4 q = *reinterpret_cast<const Pix4*>(Gb + e);
      const F32x4 f = *reinterpret_cast<const F32x4*>(tb + e);
#pragma unroll
      for (int u = 0; u < 4; ++u) g[u] = bf16_to_f32(uint16_t((u < 2 ? q.lo : q.hi) >> (16 * (u & 1)))), w[u] = f.v[u];
    } else {
      const int64_t row = int64_t(min(r, C - 1)) * C;
#pragma unroll
      for (int u = 0; u < 4; ++u) g[u] = bf16_to_f32(Gb[row + min(col + u, C - 1)]), w[u] = tb[row + min(col + u, C - 1)];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) tile[h][y][x + u] = d[h][u] = g[u] / chw - w[u];
  }
  __syncthreads();
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (h && ti == tj) break;
    const int r = (h ? tj : ti) * kGT + y, col = (h ? ti : tj) * kGT + x;
    float v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = c * (d[h][u] + tile[h ^ 1][x + u][y]) / chw;
    store4(Sb + int64_t(r) * C + col, r < C ? C - col : 0, v);
  }
}

unsigned grid_for(int64_t n) { return unsigned(std::max<int64_t>(1, std::min<int64_t>(ceil_div(n, kRegionThreads), 16384))); }

}  // namespace
}  // namespace xdna

using namespace xdna;

extern "C" {

int xdna_region_maxpool2_bf16(const uint16_t* x, uint16_t* y, int64_t planes, int H, int W, void* stream) {
  if (planes < 0 || H < 0 || W < 0) {
    set_error("xdna_region_maxpool2_bf16: invalid arguments");
    return -1;
  }
  const int Ho = H / 2, Wo = W / 2;
  if (planes == 0 || Ho == 0 || Wo == 0) return 0;  // nothing to write
  if (!x || !y) {
    set_error("xdna_region_maxpool2_bf16: null operand");
    return -1;
  }
  if (!admit_launch("xdna_region_maxpool2_bf16")) return -1;
  maxpool2_kernel<<<grid_for(planes * Ho * Wo), kRegionThreads, 0, as_stream(stream)>>>(x, y, planes, H, W, Ho, Wo);
  return check_launch("xdna_region_maxpool2_bf16");
}

int xdna_region_backward_bf16(const uint16_t* r, const uint16_t* g, const uint16_t* gp, const uint16_t* px,
                              const uint16_t* extra, const uint16_t* ta, const uint16_t* tb, float scale,
                              const void* go, int go_dtype, uint16_t* out, int64_t planes, int H, int W,
                              void* stream) {
  if (planes < 0 || H < 0 || W < 0 || (g && gp) || (gp && !px) || (!ta != !tb) || go_dtype < 0 || go_dtype > 2 ||
      (go_dtype != 0 && !go)) {
    set_error("xdna_region_backward_bf16: invalid arguments");
    return -1;
  }
  const int64_t n = planes * H * W;
  if (n == 0) return 0;
  if (!out) {
    set_error("xdna_region_backward_bf16: null output");
    return -1;
  }
  if (!admit_launch("xdna_region_backward_bf16")) return -1;
  BwdArgs a{r, g, gp, px, extra, ta, tb, go, go_dtype, scale, out, planes, H, W, H / 2, W / 2};
  if (n <= (!g && gp ? 400000 : 200000)) {
    region_bwd_small_kernel<<<unsigned(ceil_div(n, kRegionThreads)), kRegionThreads, 0, as_stream(stream)>>>(a);
  } else if (!g && gp) {
    const int64_t items = planes * ceil_div(H, 2) * ceil_div(W, 4);
    if (items < (int64_t(1) << 31))
      region_bwd_pool_kernel<uint32_t><<<grid_for(items), kRegionThreads, 0, as_stream(stream)>>>(a);
    else
      region_bwd_pool_kernel<int64_t><<<grid_for(items), kRegionThreads, 0, as_stream(stream)>>>(a);
  } else {
    region_bwd_kernel<<<grid_for(ceil_div(n, 4)), kRegionThreads, 0, as_stream(stream)>>>(a);
  }
  return check_launch("xdna_region_backward_bf16");
}

int xdna_region_loss_parts(void) { return kLossParts; }

int xdna_region_sqdiff_bf16(const uint16_t* a, const uint16_t* b, int64_t n, float scale, float* part,
                            void* stream) {
  if (!a || !b || !part || n < 0) {
    set_error("xdna_region_sqdiff_bf16: invalid arguments");
    return -1;
  }
  if (!admit_launch("xdna_region_sqdiff_bf16")) return -1;
  sqdiff_kernel<<<kLossParts, kRegionThreads, 0, as_stream(stream)>>>(a, b, n, scale, part);
  return check_launch("xdna_region_sqdiff_bf16");
}

int xdna_region_gram_sqdiff_bf16(const uint16_t* G, const float* t, int64_t t_bstride, int64_t batch, int64_t cc,
                                 float chw, float scale, float* part, void* stream) {
  if (!G || !t || !part || batch < 0 || cc < 1 || t_bstride < 0 || !(chw > 0.0f)) {
    set_error("xdna_region_gram_sqdiff_bf16: invalid arguments");
    return -1;
  }
  if (!admit_launch("xdna_region_gram_sqdiff_bf16")) return -1;
  const int64_t n = batch * cc;
  if (n <= int64_t(kLossParts) * kRegionThreads)
    gram_sqdiff_kernel<true><<<kLossParts, kRegionThreads, 0, as_stream(stream)>>>(G, t, t_bstride, cc, chw, n, scale, part);
  else
    gram_sqdiff_kernel<false><<<kLossParts, kRegionThreads, 0, as_stream(stream)>>>(G, t, t_bstride, cc, chw, n, scale, part);
  return check_launch("xdna_region_gram_sqdiff_bf16");
}

int xdna_region_loss_finish(const float* part, int n, float* out_f32, uint16_t* out_bf16, void* stream) {
  if (!part || n < 0 || (!out_f32 && !out_bf16)) {
    set_error("xdna_region_loss_finish: invalid arguments");
    return -1;
  }
  if (!admit_launch("xdna_region_loss_finish")) return -1;
  finish_kernel<<<1, kFinishThreads, 0, as_stream(stream)>>>(part, n, out_f32, out_bf16);
  return check_launch("xdna_region_loss_finish");
}

int xdna_region_gram_grad_bf16(const uint16_t* G, const float* t, int64_t t_bstride, int64_t batch, int C,
                               float chw, float coef, const void* go, int go_dtype, uint16_t* S, void* stream) {
  if (!G || !t || !S || batch < 0 || C < 1 || t_bstride < 0 || !(chw > 0.0f) || go_dtype < 0 || go_dtype > 2 ||
      (go_dtype != 0 && !go)) {
    set_error("xdna_region_gram_grad_bf16: invalid arguments");
    return -1;
  }
  if (batch == 0) return 0;
  if (batch > 65535) {
    set_error("xdna_region_gram_grad_bf16: batch too large");
    return -1;
  }
  if (!admit_launch("xdna_region_gram_grad_bf16")) return -1;
  const unsigned nt = unsigned(ceil_div(C, kGT));
  gram_grad_kernel<<<dim3(nt + 1, (nt + 1) / 2, unsigned(batch)), kRegionThreads, 0, as_stream(stream)>>>(G, t, t_bstride, C, chw,
                                                                                        coef, go, go_dtype, S);
  return check_launch("xdna_region_gram_grad_bf16");
}

}  // extern "C"
