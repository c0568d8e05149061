// 1x1 convolutions (no padding, stride 1 or 2) read and written where they are.
//
// y[n][co][p] = sum over ci of w[co][ci] x[n][ci][s p]: a product per image whose inner sides
// are pixels.  With few channels it is bound by memory (64 -> 128 channels on 128 images of
// 64 x 64: 101 MB against 2.1 GFLOP), so a stride costs no pass of its own here: the forward
// and the weight gradient sample x in their loads, and the input gradient writes its zeros
// from its epilogue.
//
// Forward and input gradient: a workgroup makes 32 MW output channels x 64 (4 / MW) pixels of
// one image (4 waves, each 32 channels x 64 pixels).  The pixels of 64 input channels are
// stored as they come, [64 k][pieces of 8 pixels], and transposed by the fragment reads; the
// forward's weights are k-contiguous and go from memory to fragments, the input gradient's
// (rows are input channels) through LDS like the pixels.  The result is staged in LDS, so each
// channel's pixels leave in 16-byte stores.
//
// Weight gradient: k runs over the pixels of all images, which both operands hold
// contiguously; each split takes a range of 64-pixel steps (a plane's last one is padded with
// zeros) and leaves fp32 partials that a second kernel adds in order.
//
// us, against sampled, spread and channel-major copies around batched products: 64 -> 128 stride
// 2 on 128 images of 64 x 64 (memory alone 10 / 19 / 10): forward 37 -> 19, input gradient
// 31 -> 23, weight gradient 85 -> 21; 61 x 67 planes 73 -> 28, 85 -> 45, 100 -> 34; 64 -> 256
// stride 1 on 128 x 56 x 56 (50 each): 137 -> 57, 47 -> 48, 241 -> 57.  What is left is the
// latency of a workgroup's few load rounds: one 64-channel step is in flight at a time.
#include "common.h"
#include "mfma.h"
#include "../../include/xdna_hip.h"

#include <algorithm>

namespace xdna {
namespace {

struct C1Args {
  const uint16_t* x;     // the input of this direction
  const uint16_t* w;     // [Cout][Cin] of the conv
  const uint16_t* bias;  // or null
  uint16_t* y;
  int B, M, K;           // images, output and input channels of this direction
  int P, Wo;             // strided pixels of a plane and of a row
  int H, W;              // the full plane
  int tpi;               // pixel tiles of an image
};

// 8 strided pixels from (oy, ox), the p-th, of a full plane (stride 2), zeros past the plane:
// 16 full-plane pixels per row that the 8 touch, read where that row's pixels fall on their
// places.  `end`: pixels from the plane's start to the end of the tensor; a row whose 16 pixels
// would start before the plane or end past the tensor is read pixel by pixel.
__device__ inline u32x4_t c1_load8_s2(const uint16_t* plane, int64_t end, int p, int oy, int ox, int P, int Wo, int W) {
  u32x4_t r = {0, 0, 0, 0};
  for (int u0 = 0; u0 < 8 && p + u0 < P;) {
    const int n = min(min(8 - u0, Wo - ox), P - p - u0);  // this row's pixels: places u0 .. u0 + n - 1
    const int64_t base = int64_t(2 * oy) * W + 2 * ox - 2 * u0;
    if (base >= 0 && base + 16 <= end) {
      const Pix8 a = *reinterpret_cast<const Pix8*>(plane + base), b = *reinterpret_cast<const Pix8*>(plane + base + 8);
      const uint32_t v[4] = {(a.v[0] & 0xFFFFu) | (a.v[1] << 16), (a.v[2] & 0xFFFFu) | (a.v[3] << 16),
                             (b.v[0] & 0xFFFFu) | (b.v[1] << 16), (b.v[2] & 0xFFFFu) | (b.v[3] << 16)};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t lo = 2 * u >= u0 && 2 * u < u0 + n ? 0xFFFFu : 0u;
        const uint32_t hi = 2 * u + 1 >= u0 && 2 * u + 1 < u0 + n ? 0xFFFF0000u : 0u;
        r[u] |= v[u] & (lo | hi);
      }
    } else {
      const uint16_t* src = plane + base;
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (u >= u0 && u < u0 + n) r[u >> 1] |= uint32_t(src[2 * u]) << (16 * (u & 1));
    }
    u0 += n;
    ox = 0;
    ++oy;
  }
  return r;
}

// 8 values from i of a run of n, zeros past its end
__device__ inline u32x4_t c1_load8(const uint16_t* run, int i, int n) {
  u32x4_t r = {0, 0, 0, 0};
  if (i + 8 <= n) {
    const Pix8 a = *reinterpret_cast<const Pix8*>(run + i);
    return u32x4_t{a.v[0], a.v[1], a.v[2], a.v[3]};
  }
#pragma unroll
  for (int u = 0; u < 8; ++u)
    if (i + u < n) r[u >> 1] |= uint32_t(run[i + u]) << (16 * (u & 1));
  return r;
}

// Piece q of k row k of a [64 k][NP pieces] tile: four k rows x 64 bytes of a transposing read
// lie on 64 distinct banks.
template <int NP>
__device__ inline int c1_piece(int k, int q) {
  return k * NP * 8 + ((NP == 8 ? q ^ (4 * ((k >> 1) & 1)) : q ^ (4 * (k & 3))) << 3);
}

typedef uint32_t c1u2 __attribute__((ext_vector_type(2)));
typedef int16_t c1i16x4 __attribute__((ext_vector_type(4)));

// MFMA fragment (rows rb + lane % 32, k = 16 ks + 8 (lane / 32) .. + 7) of such a tile
template <int NP>
__device__ inline u32x4_t c1_frag(const uint16_t* lds, int rb, int ks, int lane) {
  const int g = lane >> 4, j = lane & 15;
  const int k = 16 * ks + 8 * (g >> 1) + (j >> 2), r = rb + 16 * (g & 1) + 4 * (j & 3);
  const uint16_t* lo = lds + c1_piece<NP>(k, r >> 3) + (r & 7);
  const uint16_t* hi = lds + c1_piece<NP>(k + 4, r >> 3) + (r & 7);
  const c1u2 a = __builtin_bit_cast(
      c1u2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) c1i16x4*)(lo)));
  const c1u2 b = __builtin_bit_cast(
      c1u2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) c1i16x4*)(hi)));
  return u32x4_t{a[0], a[1], b[0], b[1]};
}

// S: the conv's stride.  kDx: the input gradient (w transposed; S = 2 spreads the result).
template <int S, bool kDx, int MW>
__global__ __launch_bounds__(256) void conv1x1_kernel(C1Args g) {
  constexpr int kPx = 64 * (4 / MW), kNp = kPx / 8, kRows = 32 * MW, kOp = kPx + 4;
  constexpr int kXT = 64 * kPx, kWT = kDx ? 64 * kRows : 0, kXl = kXT / 8 / 256, kWl = 64 * kRows / 8 / 256;
  constexpr int kOut = kRows * kOp, kLds = 2 * (kXT + kWT) > kOut ? 2 * (kXT + kWT) : kOut;
  __shared__ __attribute__((aligned(16))) uint16_t smem[kLds];
  uint16_t* xs = smem;             // [2][kXT]
  uint16_t* wsm = smem + 2 * kXT;  // [2][kWT]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int img = blockIdx.x / g.tpi, p0 = (blockIdx.x - img * g.tpi) * kPx;
  const int m0 = blockIdx.y * kRows;
  const int q = tid & (kNp - 1), kr = tid / kNp;  // this thread's piece and first k row
  const int p = p0 + 8 * q;
  const int oy = S == 2 ? p / g.Wo : 0, ox = S == 2 ? p - oy * g.Wo : 0;
  const int64_t in_plane = S == 2 && !kDx ? int64_t(g.H) * g.W : g.P;
  const uint16_t* x = g.x + int64_t(img) * g.K * in_plane;
  const int64_t left = int64_t(g.B - img) * g.K * in_plane;  // to the end of the tensor
  u32x4_t rx[kXl], rw[kWl];
  u32x4_t fa[4];  // forward: this wave's weight fragments of a k-tile
  const int wm = wave % MW, wp = wave / MW;
  const int frow = min(m0 + 32 * wm + (lane & 31), g.M - 1);

  const auto load = [&](int k0) {
#pragma unroll
    for (int j = 0; j < kXl; ++j) {
      const int k = k0 + kr + j * (256 / kNp);
      if (k >= g.K) rx[j] = u32x4_t{0, 0, 0, 0};
      else if (S == 2 && !kDx) rx[j] = c1_load8_s2(x + k * in_plane, left - k * in_plane, p, oy, ox, g.P, g.Wo, g.W);
      else rx[j] = c1_load8(x + k * in_plane, p, g.P);
    }
    if constexpr (kDx) {  // w[co = k][ci = row]
#pragma unroll
      for (int j = 0; j < kWl; ++j) {
        const int i = tid + j * 256, k = k0 + i / (kRows / 8), r = m0 + 8 * (i & (kRows / 8 - 1));
        rw[j] = k < g.K ? c1_load8(g.w + int64_t(k) * g.M, r, g.M)  : u32x4_t{0, 0, 0, 0};
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        fa[ks] = c1_load8(g.w + int64_t(frow) * g.K, k0 + 16 * ks + 8 * (lane >> 5), g.K);
    }
  };
  const auto store = [&](int buf) {
#pragma unroll
    for (int j = 0; j < kXl; ++j)
      *reinterpret_cast<u32x4_t*>(xs + buf * kXT + c1_piece<kNp>(kr + j * (256 / kNp), q)) = rx[j];
    if constexpr (kDx) {
#pragma unroll
      for (int j = 0; j < kWl; ++j) {
        const int i = tid + j * 256;
        *reinterpret_cast<u32x4_t*>(wsm + buf * kWT + c1_piece<kRows / 8>(i / (kRows / 8), i & (kRows / 8 - 1))) = rw[j];
      }
    }
  };

  f32x16_t acc[2] = {zero_acc(), zero_acc()};  // rows: pixels, columns: output channels
  load(0);
  store(0);
  __syncthreads();
  int buf = 0;
  for (int k0 = 0; k0 < g.K; k0 += 64, buf ^= 1) {
    const bool more = k0 + 64 < g.K;
    u32x4_t wf[4];
    if constexpr (!kDx) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) wf[ks] = fa[ks];
    }
    if (more) load(k0 + 64);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if constexpr (kDx) wf[ks] = c1_frag<kRows / 8>(wsm + buf * kWT, 32 * wm, ks, lane);
#pragma unroll
      for (int n = 0; n < 2; ++n)
        acc[n] = mfma_32x32x16(as_bf16x8(c1_frag<kNp>(xs + buf * kXT, 64 * wp + 32 * n, ks, lane)),
                               as_bf16x8(wf[ks]), acc[n]);
    }
    if (more) store(buf ^ 1);  // its last reads ended before the previous barrier
    __syncthreads();
  }

  // [channel][kPx + 4] in LDS (8-byte writes of 32 channels on distinct banks)
  const float bv = !kDx && g.bias ? bf16_to_f32(g.bias[frow]) : 0.0f;
  const int row = 32 * wm + (lane & 31);
#pragma unroll
  for (int n = 0; n < 2; ++n)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      uint16_t h[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) h[u] = f32_to_bf16(acc[n][4 * t + u] + bv);
      *reinterpret_cast<uint2*>(smem + row * kOp + 64 * wp + 32 * n + 8 * t + 4 * (lane >> 5)) =
          make_uint2(h[0] | (uint32_t(h[1]) << 16), h[2] | (uint32_t(h[3]) << 16));
    }
  __syncthreads();
  if (p >= g.P) return;
  for (int r = kr; r < kRows && m0 + r < g.M; r += 256 / kNp) {
    const uint2 a = *reinterpret_cast<const uint2*>(smem + r * kOp + 8 * q);
    const uint2 b = *reinterpret_cast<const uint2*>(smem + r * kOp + 8 * q + 4);
    const uint32_t v[4] = {a.x, a.y, b.x, b.y};
    if (S == 2 && kDx) {
      uint16_t* o = g.y + (int64_t(img) * g.M + m0 + r) * g.H * g.W;
      if (2 * ox + 16 <= g.W) {  // all 16 full-plane pixels in this row
        o += int64_t(2 * oy) * g.W + 2 * ox;
        *reinterpret_cast<Pix8*>(o) = Pix8{{v[0] & 0xFFFFu, v[0] >> 16, v[1] & 0xFFFFu, v[1] >> 16}};
        *reinterpret_cast<Pix8*>(o + 8) = Pix8{{v[2] & 0xFFFFu, v[2] >> 16, v[3] & 0xFFFFu, v[3] >> 16}};
        if (2 * oy + 1 < g.H) {
          *reinterpret_cast<Pix8*>(o + g.W) = Pix8{{0, 0, 0, 0}};
          *reinterpret_cast<Pix8*>(o + g.W + 8) = Pix8{{0, 0, 0, 0}};
        }
      } else {
        int yy = 2 * oy, xx = 2 * ox;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          if (p + u >= g.P) break;
          uint16_t* d = o + int64_t(yy) * g.W + xx;
          const bool below = yy + 1 < g.H;
          if (xx + 1 < g.W) {
            *reinterpret_cast<Pix2*>(d) = Pix2{(v[u >> 1] >> (16 * (u & 1))) & 0xFFFFu};
            if (below) *reinterpret_cast<Pix2*>(d + g.W) = Pix2{0};
          } else {
            d[0] = uint16_t(v[u >> 1] >> (16 * (u & 1)));
            if (below) d[g.W] = 0;
          }
          xx += 2;
          if (xx >= g.W) xx = 0, yy += 2;
        }
      }
    } else {
      uint16_t* o = g.y + (int64_t(img) * g.M + m0 + r) * g.P + p;
      if (p + 8 <= g.P) {
        *reinterpret_cast<Pix8*>(o) = Pix8{{v[0], v[1], v[2], v[3]}};
      } else {
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (p + u < g.P) o[u] = uint16_t(v[u >> 1] >> (16 * (u & 1)));
      }
    }
  }
}

struct C1WgArgs {
  const uint16_t* x;
  const uint16_t* dy;
  float* part;  // [nsplit][Cout][Cin]
  int B, Ci, Co, P, Wo, H, W;
  int spi;      // 64-pixel steps of an image
  int steps, per;
};

constexpr int kWgP = 72;  // LDS pitch of a row of 64 pixels: fragment reads free of conflicts

// MW waves along the output channels, 4 / MW along the input channels, 32 x 64 each.
template <int S, int MW>
__global__ __launch_bounds__(256) void conv1x1_wgrad_kernel(C1WgArgs g) {
  constexpr int kA = 32 * MW, kB = 64 * (4 / MW), kAl = kA / 32, kBl = kB / 32;
  __shared__ __attribute__((aligned(16))) uint16_t as[2][kA * kWgP], bs[2][kB * kWgP];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = blockIdx.y * kA, n0 = blockIdx.z * kB;
  const int wm = wave % MW, wn = wave / MW;
  const int q = tid & 7, rr = tid >> 3;  // this thread's pixel piece and first row
  const int64_t xplane = S == 2 ? int64_t(g.H) * g.W : g.P;
  u32x4_t ra[kAl], rb[kBl];
  const auto load = [&](int t) {
    const int img = t / g.spi, p = (t - img * g.spi) * 64 + 8 * q;
    const int oy = S == 2 ? p / g.Wo : 0, ox = S == 2 ? p - oy * g.Wo : 0;
#pragma unroll
    for (int j = 0; j < kAl; ++j) {
      const int r = min(m0 + rr + 32 * j, g.Co - 1);
      ra[j] = c1_load8(g.dy + (int64_t(img) * g.Co + r) * g.P, p, g.P);
    }
#pragma unroll
    for (int j = 0; j < kBl; ++j) {
      const uint16_t* plane = g.x + (int64_t(img) * g.Ci + min(n0 + rr + 32 * j, g.Ci - 1)) * xplane;
      rb[j] = S == 2 ? c1_load8_s2(plane, g.x + int64_t(g.B) * g.Ci * xplane - plane, p, oy, ox, g.P, g.Wo, g.W)
                     : c1_load8(plane, p, g.P);
    }
  };
  const auto store = [&](int b) {
#pragma unroll
    for (int j = 0; j < kAl; ++j)
      *reinterpret_cast<u32x4_t*>(as[b] + (rr + 32 * j) * kWgP + 8 * q) = ra[j];
#pragma unroll
    for (int j = 0; j < kBl; ++j)
      *reinterpret_cast<u32x4_t*>(bs[b] + (rr + 32 * j) * kWgP + 8 * q) = rb[j];
  };
  f32x16_t acc[2] = {zero_acc(), zero_acc()};
  const int t0 = blockIdx.x * g.per, t1 = min(t0 + g.per, g.steps);
  load(t0);  // (every split has a step)
  store(0);
  __syncthreads();
  int buf = 0;
  for (int t = t0; t < t1; ++t, buf ^= 1) {
    const bool more = t + 1 < t1;
    if (more) load(t + 1);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int k = 16 * ks + 8 * (lane >> 5);
      const bf16x8_t a = as_bf16x8(*reinterpret_cast<const u32x4_t*>(as[buf] + (32 * wm + (lane & 31)) * kWgP + k));
#pragma unroll
      for (int n = 0; n < 2; ++n)
        acc[n] = mfma_32x32x16(
            a, as_bf16x8(*reinterpret_cast<const u32x4_t*>(bs[buf] + (64 * wn + 32 * n + (lane & 31)) * kWgP + k)),
            acc[n]);
    }
    if (more) store(buf ^ 1);
    __syncthreads();
  }
  float* part = g.part + int64_t(blockIdx.x) * g.Co * g.Ci;
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const int c = n0 + 64 * wn + 32 * n + (lane & 31);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = m0 + 32 * wm + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
      if (m < g.Co && c < g.Ci) part[int64_t(m) * g.Ci + c] = acc[n][r];
    }
  }
}

// gw = the splits' partials added in a fixed order: 32 elements x 8 interleaved runs of splits
// per workgroup.
__global__ __launch_bounds__(256) void conv1x1_wgrad_reduce_kernel(const float* __restrict__ part,
                                                                   uint16_t* __restrict__ gw, int n, int nsplit) {
  __shared__ float sums[8][32];
  const int e = blockIdx.x * 32 + (threadIdx.x & 31), z = threadIdx.x >> 5;
  sums[z][threadIdx.x & 31] = e < n ? sum_strided8(0.0f, part + e, n, z, 8, nsplit) : 0.0f;
  __syncthreads();
  if (z > 0 || e >= n) return;
  float s = sums[0][threadIdx.x];
#pragma unroll
  for (int u = 1; u < 8; ++u) s += sums[u][threadIdx.x];
  gw[e] = f32_to_bf16(s);
}

struct C1Geom {
  int Ho, Wo, P;
};

bool c1_geom(const char* who, const void* a, const void* b, const void* c, int B, int Cin, int Cout, int H, int W,
             int stride, C1Geom& o) {
  if (!a || !b || !c || B < 1 || Cin < 1 || Cout < 1 || H < 1 || W < 1 || (stride != 1 && stride != 2) ||
      int64_t(H) * W >= (int64_t(1) << 30)) {
    set_error(std::string(who) + ": invalid arguments");
    return false;
  }
  o.Ho = (H + stride - 1) / stride;
  o.Wo = (W + stride - 1) / stride;
  o.P = o.Ho * o.Wo;
  return true;
}

// up to 64 output channels: two waves along them, twice the pixels
bool c1_narrow(int M) { return M <= 64; }

int c1_launch(const char* who, bool dx, const uint16_t* x, const uint16_t* w, const uint16_t* bias, uint16_t* y, int B,
              int Cin, int Cout, int H, int W, int stride, void* stream) {
  C1Geom q;
  if (!c1_geom(who, x, w, y, B, Cin, Cout, H, W, stride, q)) return -1;
  C1Args g;
  g.x = x;
  g.w = w;
  g.bias = bias;
  g.y = y;
  g.B = B;
  g.M = dx ? Cin : Cout;
  g.K = dx ? Cout : Cin;
  g.P = q.P;
  g.Wo = q.Wo;
  g.H = H;
  g.W = W;
  const bool narrow = c1_narrow(g.M);
  g.tpi = int(ceil_div(q.P, narrow ? 128 : 64));
  const int64_t gx = int64_t(B) * g.tpi, gy = ceil_div(g.M, narrow ? 64 : 128);
  if (gx > kMaxGridX256 || gy > 65535) {
    set_error(std::string(who) + ": grid too large");
    return -1;
  }
  if (!admit_launch(who)) return -1;
  const dim3 grid(unsigned(gx), unsigned(gy), 1);
  const hipStream_t st = as_stream(stream);
  if (dx) {
    if (stride == 2) {
      if (narrow) conv1x1_kernel<2, true, 2><<<grid, 256, 0, st>>>(g);
      else conv1x1_kernel<2, true, 4><<<grid, 256, 0, st>>>(g);
    } else {
      if (narrow) conv1x1_kernel<1, true, 2><<<grid, 256, 0, st>>>(g);
      else conv1x1_kernel<1, true, 4><<<grid, 256, 0, st>>>(g);
    }
  } else if (stride == 2) {
    if (narrow) conv1x1_kernel<2, false, 2><<<grid, 256, 0, st>>>(g);
    else conv1x1_kernel<2, false, 4><<<grid, 256, 0, st>>>(g);
  } else {
    if (narrow) conv1x1_kernel<1, false, 2><<<grid, 256, 0, st>>>(g);
    else conv1x1_kernel<1, false, 4><<<grid, 256, 0, st>>>(g);
  }
  return check_launch(who);
}

struct C1WgPlan {
  int64_t steps;
  int spi, per, nsplit, mt, nt;
  bool narrow;
};

C1WgPlan c1_wgrad_plan(int B, int Cin, int Cout, int P) {
  C1WgPlan p;
  p.narrow = Cout <= 64;
  p.mt = int(ceil_div(Cout, p.narrow ? 64 : 128));
  p.nt = int(ceil_div(Cin, p.narrow ? 128 : 64));
  p.spi = int(ceil_div(P, 64));
  p.steps = int64_t(B) * p.spi;
  // two workgroups per CU, each with at least two steps to stream
  const int64_t want = std::max<int64_t>(1, std::min(ceil_div(512, int64_t(p.mt) * p.nt), p.steps / 2));
  p.per = int(ceil_div(p.steps, want));
  p.nsplit = int(ceil_div(p.steps, p.per));
  return p;
}

// Modelled times, us, of these kernels and of the products they stand beside, fitted to 2500
// random shapes (1 - 256 images, 4 - 2048 channels, planes from 1 x 1 to 100 x 100, both strides;
// 20 - 30 % off at one standard deviation).  A workgroup is a chain of ceil(K / 64) rounds of about
// one load latency each, so a long k on few workgroups belongs to the GEMM, whose k groups and
// splits cut the chain (512 -> 64 stride 2 on 39 x 7 x 10: 53 in place, 12 as a product; input
// gradient of 85 -> 2048 on 12 x 2 x 2: 101 / 13.5), and many workgroups, or planes whose
// pixels fill no GEMM tile, belong here (64 -> 128 stride 2 on 128 x 64 x 64 19 / 37; input gradient
// of 1024 -> 1483 on 190 x 4 x 2 81 / 275).
// Used below two workgroups per CU and for strided planes of short rows; the choice asks for 12 %
// in favour of these kernels.
double c1_mb(int64_t elements) { return 2e-6 * double(elements); }

// rows beyond the first that 8 consecutive pixels of the strided plane touch
int c1_row_breaks(const C1Geom& q) { return std::min(int(ceil_div(8, std::min(q.Wo, 8))), q.Ho) - 1; }

// forward / input gradient, `wgs` workgroups of M outputs over K
double c1_us(bool dx, int64_t wgs, int B, int M, int K, int Cin, int H, int W, const C1Geom& q, int stride) {
  const double rounds = double(ceil_div(K, 64)), waves = std::max(1.0, double(wgs) / 256);
  const bool narrow = c1_narrow(M), odd_px = q.P % 8 != 0, s2 = stride == 2;
  const double mb = c1_mb(int64_t(B) * q.P * (M + K) + int64_t(M) * K);
  if (!dx) {
    const double round = 0.92 + 0.52 * narrow + 0.40 * odd_px + 0.28 * (K % 8 != 0) + s2 * (0.28 + 0.49 * c1_row_breaks(q));
    return 3.8 + rounds * round * (1 + 0.54 * (waves - 1)) + 0.22 * mb;
  }
  const double round = 1.1 + 0.29 * narrow + 0.45 * odd_px + 1.0 * (M % 8 != 0);
  // a spread piece that crosses a row's end is stored pixel by pixel
  const double crossing = q.Wo % 8 == 0 ? 0.0 : std::min(1.5, 8.0 / q.Wo);
  return 3.8 + rounds * round * (1 + 0.34 * (waves - 1)) + 0.19 * mb +
         s2 * (1.1 * waves + (0.22 + 0.8 * crossing) * c1_mb(int64_t(B) * Cin * H * W));
}

// the batched product (and, stride 2, the sampling or spreading pass)
double c1_gemm_us(bool dx, int B, int M, int K, int Cin, int H, int W, const C1Geom& q, int stride) {
  const double rounds = double(ceil_div(K, 64)), tiles = double(B) * double(ceil_div(q.P, 64)) * double(ceil_div(M, 64));
  const double gf = 2e-9 * B * double(q.P) * M * K, full = stride == 2 ? c1_mb(int64_t(B) * Cin * H * W) : 0.0;
  const bool odd_px = q.P % 8 != 0, odd_w = Cin % 8 != 0, s2 = stride == 2;  // operands staged by elements
  if (!dx)
    return 4.9 + s2 * 2.1 + 0.42 * full + 2.0 * odd_px + 4.5 * odd_w + 2.2 * gf * (odd_px + odd_w) + 0.39 * std::min(rounds, 4.0) +
           1.7 * tiles * rounds / 512;
  return 3.8 + s2 * 1.7 + 1.1 * full + 2.0 * odd_px + 3.5 * odd_w + gf * (0.66 + 0.98 * (odd_px + odd_w)) +
         0.81 * std::min(rounds, 4.0) + 2.0 * tiles * rounds / 512;
}

// weight gradient: a chain of 64-pixel steps, then the partials' sum (505 -> 1024 on 200 x 3 x 3, steps
// of 9 pixels, loses: the product's copies are contiguous over images)
double c1_wgrad_us(const C1WgPlan& p, int B, int Cin, int Cout, int H, int W, const C1Geom& q, int stride) {
  const double step = 1.3 + 0.93 * (q.P % 8 != 0) + (stride == 2) * (0.72 + 0.86 * c1_row_breaks(q));
  const double n = 1e-6 * Cin * double(Cout);
  return 7.4 + p.per * step + 2.7 * p.nsplit * n + 3.1 * n + 0.09 * c1_mb(int64_t(B) * q.P * (Cin + Cout));
}

// channel-major copies (none of a single image) and one product over the pixels
double c1_wgrad_gemm_us(int B, int Cin, int Cout, int H, int W, const C1Geom& q, int stride) {
  const double k = double(B) * q.P, n = 1e-6 * Cin * double(Cout);
  const double odd = int64_t(B) * q.P % 8 != 0, padded = 2e-9 * 128 * double(ceil_div(Cin, 128)) * 128 * double(ceil_div(Cout, 128)) * k;
  return 7.2 + (stride == 2) * (2.0 + 0.38 * c1_mb(int64_t(B) * Cin * H * W)) +
         (B > 1) * (7.8 + c1_mb(int64_t(B) * q.P * (Cin + Cout))) + 4.5e-3 * n * k * odd + 1.1 * n + 0.24 * std::min(k / 64, 16.0) +
         5.9 * odd + 3.8 * padded;
}

}  // namespace
}  // namespace xdna

using namespace xdna;

extern "C" {

int xdna_conv1x1_pick(int op, int B, int Cin, int Cout, int H, int W, int stride) {
  C1Geom q;
  static const char one = 0;
  if (op < 0 || op > 2) {
    set_error("xdna_conv1x1_pick: invalid op");
    return -1;
  }
  if (!c1_geom("xdna_conv1x1_pick", &one, &one, &one, B, Cin, Cout, H, W, stride, q)) return -1;
  if (op == 2) {
    const C1WgPlan p = c1_wgrad_plan(B, Cin, Cout, q.P);
    const int64_t n = int64_t(Cin) * Cout;
    if (n > 0x7FFFFFFF || p.steps > 0x7FFFFFFF || p.mt > 65535 || p.nt > 65535) return 0;
    // Many outputs from few pixels: 2 copies to channel-major rows and one product on 256 x 256
    // tiles (us, this form / that one: 512 -> 2048 on 128 x 7 x 7 130 / 74, 512 -> 1024 on
    // 64 x 7 x 7 46 / 43; but 1024 -> 1024 on 32 x 32 x 32 127 / 172).
    if (n >= (int64_t(1) << 19) && int64_t(B) * q.P < 16384) return 0;
    return c1_wgrad_us(p, B, Cin, Cout, H, W, q, stride) < 0.88 * c1_wgrad_gemm_us(B, Cin, Cout, H, W, q, stride);
  }
  const int M = op == 1 ? Cin : Cout, K = op == 1 ? Cout : Cin;
  const bool narrow = c1_narrow(M);
  const int64_t gx = int64_t(B) * ceil_div(q.P, narrow ? 128 : 64), gy = ceil_div(M, narrow ? 64 : 128);
  if (gx > kMaxGridX256 || gy > 65535) return 0;
  // A long k on planes whose rows the large GEMM tiles fill and load whole (1024 -> 1024 on
  // 32 x 32 x 32: 160 / 96 forward, 124 / 74 input gradient; 1024 -> 2048 on 50 x 16 x 16, 400
  // tiles, 127 / 90, but input gradient of 256 -> 1024 on 43 x 16 x 16, 43 tiles, 21 / 73).
  if (K >= 1024 && q.P % 8 == 0 && (q.P > 256 || (q.P == 256 && int64_t(B) * ceil_div(M, 256) >= 200))) return 0;
  // Few workgroups on a long k (forward, 2048 -> 512 on 8 x 7 x 7: 41 / 16; 2048 -> 2048 on 4 x 14 x 14
  // 66 / 43; input gradient of 256 -> 512 stride 2 on 8 x 8 x 8: 11.4 / 8.5).
  if (gx * gy < 256 && (op == 0 ? K >= 1024 : stride == 2 && K >= 512)) return 0;
  // From 512 workgroups the chains overlap and these kernels win (half the product's time) but for
  // strided planes of short rows.
  if (gx * gy >= 512 && (stride == 1 || (op == 0 ? c1_row_breaks(q) < 3 : W >= 16))) return 1;
  return c1_us(op == 1, gx * gy, B, M, K, Cin, H, W, q, stride) < 0.88 * c1_gemm_us(op == 1, B, M, K, Cin, H, W, q, stride);
}

int xdna_conv1x1_fwd_bf16(const uint16_t* x, const uint16_t* w, const uint16_t* bias, uint16_t* y, int B, int Cin,
                          int Cout, int H, int W, int stride, void* stream) {
  return c1_launch("xdna_conv1x1_fwd_bf16", false, x, w, bias, y, B, Cin, Cout, H, W, stride, stream);
}

int xdna_conv1x1_dgrad_bf16(const uint16_t* dy, const uint16_t* w, uint16_t* dx, int B, int Cin, int Cout, int H,
                            int W, int stride, void* stream) {
  return c1_launch("xdna_conv1x1_dgrad_bf16", true, dy, w, nullptr, dx, B, Cin, Cout, H, W, stride, stream);
}

size_t xdna_conv1x1_wgrad_workspace_bytes(int B, int Cin, int Cout, int H, int W, int stride) {
  C1Geom q;
  static const char one = 0;
  if (!c1_geom("xdna_conv1x1_wgrad_workspace_bytes", &one, &one, &one, B, Cin, Cout, H, W, stride, q)) return 0;
  return size_t(c1_wgrad_plan(B, Cin, Cout, q.P).nsplit) * size_t(Cout) * size_t(Cin) * sizeof(float);
}

int xdna_conv1x1_wgrad_bf16(const uint16_t* x, const uint16_t* dy, uint16_t* gw, int B, int Cin, int Cout, int H,
                            int W, int stride, void* workspace, size_t workspace_bytes, void* stream) {
  C1Geom q;
  if (!c1_geom("xdna_conv1x1_wgrad_bf16", x, dy, gw, B, Cin, Cout, H, W, stride, q)) return -1;
  const C1WgPlan p = c1_wgrad_plan(B, Cin, Cout, q.P);
  const size_t need = size_t(p.nsplit) * size_t(Cout) * size_t(Cin) * sizeof(float);
  const int64_t n = int64_t(Cout) * Cin;
  if (!workspace || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 3)) {
    set_error("xdna_conv1x1_wgrad_bf16: workspace too small or misaligned");
    return -1;
  }
  if (n > 0x7FFFFFFF || p.steps > 0x7FFFFFFF || p.mt > 65535 || p.nt > 65535) {
    set_error("xdna_conv1x1_wgrad_bf16: too many channels or pixels");
    return -1;
  }
  if (!admit_launch("xdna_conv1x1_wgrad_bf16")) return -1;
  C1WgArgs g;
  g.x = x;
  g.dy = dy;
  g.part = static_cast<float*>(workspace);
  g.B = B;
  g.Ci = Cin;
  g.Co = Cout;
  g.P = q.P;
  g.Wo = q.Wo;
  g.H = H;
  g.W = W;
  g.spi = p.spi;
  g.steps = int(p.steps);
  g.per = p.per;
  const dim3 grid(unsigned(p.nsplit), unsigned(p.mt), unsigned(p.nt));
  const hipStream_t st = as_stream(stream);
  if (stride == 2) {
    if (p.narrow) conv1x1_wgrad_kernel<2, 2><<<grid, 256, 0, st>>>(g);
    else conv1x1_wgrad_kernel<2, 4><<<grid, 256, 0, st>>>(g);
  } else {
    if (p.narrow) conv1x1_wgrad_kernel<1, 2><<<grid, 256, 0, st>>>(g);
    else conv1x1_wgrad_kernel<1, 4><<<grid, 256, 0, st>>>(g);
  }
  conv1x1_wgrad_reduce_kernel<<<unsigned(ceil_div(n, 32)), 256, 0, st>>>(g.part, gw, int(n), p.nsplit);
  return check_launch("xdna_conv1x1_wgrad_bf16");
}

}  // extern "C"
