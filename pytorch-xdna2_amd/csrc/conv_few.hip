// Stride-1 convolutions with few channels on one side: the 9x9 image layers of a style
// network (3 -> 32, 32 -> 3), an RGB stem, and their gradients.  Implicit GEMM over (channel,
// tap) pads such a layer's 3 channels to a 32-wide MFMA tile and reads every operand element
// once per tap; these layers move a few MB and need microseconds of matrix work, so what
// bounds them is the latency of load -> LDS -> MFMA -> store and the LDS reads per MFMA.
// Each kernel therefore puts taps, not padding, beside the few channels:
//
//  few outputs (few_out_kernel): rows m = (output channel, kx) of the MFMA hold one output
//    channel's kx taps; K runs over (ky, input channel) only.  z[(co, kx)][column] is summed
//    along the diagonal, y[co][ox] = sum over kx of z[(co, kx)][ox + kx], in LDS.
//  few inputs (few_in_kernel): k runs over (ky, two kx x four channels): positions of four
//    channels (8 bytes) in LDS, so a lane's 8 k are two neighbouring positions.
//  weight gradient (few_wgrad_kernel): rows m = (few channel, kx) are copies of the few side
//    shifted by kx, the wide side's channels are the columns, K runs over pixels, and each ky
//    is a row offset into the same LDS tile: one accumulator per ky.
//
// 40 x 36 x 36 pixels, 9x9, us in a graph on an MI355X, against the direct, gather and
// sliding-window kernels of conv_gather.hip: 32 -> 3 forward 27.7 -> 11.7, input gradient
// 21.4 -> 8.2, weight and bias gradients 51.0 -> 20.8; 3 -> 32 23.1 -> 8.5, 25.9 -> 11.4,
// 33.0 -> 17.8; 3x3 3 -> 64 at 128 x 64 x 64 44 -> 30, 82 -> 51, 153 -> 76.  The rules beside the plans
// say where the general kernels stay ahead.
#include "conv_few.h"

#include "common.h"
#include "mfma.h"
#include "../../include/xdna_hip.h"

namespace xdna {
namespace {

constexpr int kFewPitch = 40;             // LDS elements of 32 channels (80 bytes: 16-byte reads without conflicts)
constexpr size_t kFewLds = 80 * 1024;     // two workgroups per CU
constexpr size_t kFewLdsMax = 156 * 1024;  // a CU's 160 KiB less the block reductions' own
constexpr int kFewThreads = 512;          // weight gradient: its staging is latency, so more loads per workgroup
constexpr int kFewWeights = 16;           // weight loads in flight per thread

// Every kernel below may use up to a CU's LDS.
bool raise_lds(const void* fn) {
  const bool ok = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, int(kFewLdsMax)) == hipSuccess;
  if (!ok) (void)hipGetLastError();  // (the general kernels take the call)
  return ok;
}

// Calls put(row, chan, tap, value) for `rows` x `chans` x `taps` weights from row0, chan0 on;
// a channel past nchan gives 0.  The weight (row, chan, tap) is w[(row * Cin + chan) * taps +
// tap], or, flipped, w[(chan * Cout + row) * taps + taps - 1 - tap].  A thread keeps its tap
// and steps over (row, chan) pairs, so consecutive threads read consecutive taps and an
// element costs no division by a run-time value; kFewWeights loads are in flight.
template <class Put>
__device__ inline void each_weight(const uint16_t* __restrict__ w, int row0, int rows, int chan0, int chans, int nchan,
                                   int taps, int Cin, int Cout, int flip, Put put) {
  const int tp = min(taps, 256), step = 256 / tp;
  const int first = threadIdx.x / tp;
  if (first >= step) return;
  const uint32_t mc = chans > 1 ? 0xFFFFFFFFu / uint32_t(chans) + 1 : 0;
  const int pairs = rows * chans;
  const int64_t srow = int64_t(flip ? 1 : Cin) * taps, schan = int64_t(flip ? Cout : 1) * taps;
  for (int tap = threadIdx.x - first * tp; tap < taps; tap += tp) {
    const uint16_t* wt = w + row0 * srow + chan0 * schan + (flip ? taps - 1 - tap : tap);
    for (int p0 = first; p0 < pairs; p0 += step * kFewWeights) {
      uint16_t v[kFewWeights];
      int row[kFewWeights], chan[kFewWeights];
#pragma unroll
      for (int j = 0; j < kFewWeights; ++j) {
        const int p = min(p0 + j * step, pairs - 1);
        row[j] = chans > 1 ? fast_div(p, mc) : p;
        chan[j] = p - row[j] * chans;
        const int c = min(chan[j], nchan - chan0 - 1);
        v[j] = wt[row[j] * srow + c * schan];
        if (c < chan[j]) v[j] = 0;
      }
#pragma unroll
      for (int j = 0; j < kFewWeights; ++j)
        if (p0 + j * step < pairs) put(row[j], chan[j], tap, v[j]);
    }
  }
}

// ---------------------------------------------------------------------------------------
// Few outputs: Cout * KW <= 32
// ---------------------------------------------------------------------------------------
struct FewOutArgs {
  const uint16_t* x;     // [B][Cin][H][W]
  const uint16_t* w;
  const uint16_t* bias;  // [Cout] or null
  uint16_t* out;         // [B][Cout][Ho][Wo]
  int B, Cin, Cout, H, W, KH, KW, ph, pw, Ho, Wo, flip, act;
  int Wp;      // Wo + KW - 1: columns of the zero-padded grid
  int R;       // output rows per workgroup
  int rtiles;  // ceil(Ho / R)
  int nb;      // blocks of 32 grid positions: ceil(R * Wp / 32)
  int xpos;    // staged positions: nb * 32 + (KH - 1) * Wp
};

// Workgroup = (image, R output rows).  LDS: the R + KH - 1 input rows as a zero-padded grid of
// Wp columns, 32 channels per position, and the weights as [ky][(co, kx)][32 channels].
// NBW: position blocks per wave (blocks wave, wave + 4, ...; a wave past the last block
// computes it again and drops it).
template <int NBW>
__global__ __launch_bounds__(256) void few_out_kernel(FewOutArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  uint16_t* xs = smem;                       // [xpos][kFewPitch]
  uint16_t* ws = smem + a.xpos * kFewPitch;  // [KH][32][kFewPitch]
  const int b = blockIdx.x / a.rtiles, oy0 = (blockIdx.x % a.rtiles) * a.R;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 31, lk = (lane >> 5) * 8;
  const int iy0 = oy0 - a.ph;
  const int ylo = max(iy0, 0), yhi = min(iy0 + a.R + a.KH - 1, a.H);
  const int npix = max(yhi - ylo, 0) * a.W;  // one run of pixels per channel (a multiple of W >= 4)
  const int ngrp = (npix + 3) >> 2;
  const int64_t plane = int64_t(a.H) * a.W;
  const uint32_t mw = 0xFFFFFFFFu / uint32_t(a.W) + 1;

  // staging item: 4 pixels x 16 channels of chunk ch; the run's last group ends with the run
  auto load_x = [&](int ch, int it, uint32_t (&d)[16][2]) {
    const int seg = it >= ngrp ? 1 : 0;
    const int pix0 = min((it - seg * ngrp) * 4, npix - 4);
    const uint16_t* sp = a.x + (int64_t(b) * a.Cin + ch * 32) * plane + int64_t(ylo) * a.W + pix0;
    const int cc = a.Cin - ch * 32 - seg * 16;  // channels of this item
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const Pix4 t = *reinterpret_cast<const Pix4*>(sp + min(seg * 16 + k, a.Cin - ch * 32 - 1) * plane);
      d[k][0] = k < cc ? t.lo : 0u;
      d[k][1] = k < cc ? t.hi : 0u;
    }
  };
  auto store_x = [&](int it, const uint32_t (&d)[16][2]) {
    const int seg = it >= ngrp ? 1 : 0;
    const int pix0 = min((it - seg * ngrp) * 4, npix - 4);
    int y = fast_div(pix0, mw), x = pix0 - y * a.W;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t o[8];
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        const uint32_t u = d[2 * m][i >> 1], v = d[2 * m + 1][i >> 1];
        o[m] = (i & 1) ? __builtin_amdgcn_perm(v, u, 0x07060302u) : __builtin_amdgcn_perm(v, u, 0x05040100u);
      }
      u32x4_t* p = reinterpret_cast<u32x4_t*>(xs + ((ylo - iy0 + y) * a.Wp + x + a.pw) * kFewPitch + seg * 16);
      p[0] = u32x4_t{o[0], o[1], o[2], o[3]};
      p[1] = u32x4_t{o[4], o[5], o[6], o[7]};
      if (++x == a.W) {
        x = 0;
        ++y;
      }
    }
  };

  f32x16_t acc[NBW];
  int bpos[NBW];
#pragma unroll
  for (int j = 0; j < NBW; ++j) {
    acc[j] = zero_acc();
    bpos[j] = (min(wave + 4 * j, a.nb - 1) * 32 + lr) * kFewPitch + lk;
  }
  const int chunks = (a.Cin + 31) >> 5;
  for (int ch = 0; ch < chunks; ++ch) {
    // the first item's loads are in flight while the grid is cleared and the weights staged
    uint32_t d[16][2];
    const bool mine = tid < 2 * ngrp;
    if (mine) load_x(ch, tid, d);
    if (ch == 0) {
      for (int i = tid; i < a.xpos * (kFewPitch / 8); i += 256)
        reinterpret_cast<u32x4_t*>(xs)[i] = u32x4_t{0, 0, 0, 0};
    } else {
      __syncthreads();  // the previous chunk's reads are done
    }
    each_weight(a.w, 0, a.Cout, ch * 32, 32, a.Cin, a.KH * a.KW, a.Cin, a.Cout, a.flip,
                [&](int co, int cl, int tap, uint16_t v) {
                  const int ky = tap / a.KW, kx = tap - ky * a.KW;
                  ws[(ky * 32 + co * a.KW + kx) * kFewPitch + cl] = v;
                });
    __syncthreads();
    if (mine) store_x(tid, d);
    for (int it = tid + 256; it < 2 * ngrp; it += 256) {
      load_x(ch, it, d);
      store_x(it, d);
    }
    __syncthreads();
    const uint16_t* wa = ws + lr * kFewPitch + lk;
    const uint16_t* xb = xs;
    for (int ky = 0; ky < a.KH; ++ky, wa += 32 * kFewPitch, xb += a.Wp * kFewPitch) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const bf16x8_t af = as_bf16x8(*reinterpret_cast<const u32x4_t*>(wa + ks * 16));
#pragma unroll
        for (int j = 0; j < NBW; ++j) {
          const bf16x8_t bf = as_bf16x8(*reinterpret_cast<const u32x4_t*>(xb + bpos[j] + ks * 16));
          acc[j] = mfma_32x32x16(af, bf, acc[j]);
        }
      }
    }
  }
  // z[(co, kx)][position] to LDS, then each output sums its diagonal
  __syncthreads();
  float* zs = reinterpret_cast<float*>(smem);
  const int zp = a.nb * 32 + 1, rows = a.Cout * a.KW;
#pragma unroll
  for (int j = 0; j < NBW; ++j) {
    const int nbk = wave + 4 * j;
    if (nbk < a.nb) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = mfma_row(r, lane);
        if (m < rows) zs[m * zp + nbk * 32 + lr] = acc[j][r];
      }
    }
  }
  __syncthreads();
  const int per = a.R * a.Wo;
  for (int i = tid; i < a.Cout * per; i += 256) {
    const int co = i / per, rem = i - co * per;
    const int row = rem / a.Wo, ox = rem - row * a.Wo;
    if (oy0 + row >= a.Ho) continue;
    const float* z = zs + co * a.KW * zp + row * a.Wp + ox;
    float v = 0.0f;
    for (int kx = 0; kx < a.KW; ++kx) v += z[kx * (zp + 1)];
    if (a.bias) v += bf16_to_f32(a.bias[co]);
    a.out[((int64_t(b) * a.Cout + co) * a.Ho + oy0 + row) * a.Wo + ox] = f32_to_bf16(act_forward(a.act, 0.0f, v));
  }
}

size_t few_out_lds(const FewOutArgs& a) {
  return std::max(size_t(a.xpos + a.KH * 32) * kFewPitch * 2, size_t(a.Cout) * a.KW * (a.nb * 32 + 1) * 4);
}

// Fills in the geometry; false where the kernel does not apply or (unless `any`) loses.
bool few_out_plan(FewOutArgs& a, bool any) {
  // at least 8 input channels (below, the 32-channel chunk is mostly padding)
  if (a.KH > 16 || a.KH < 1 || a.KW < 1 || a.Cout * a.KW > 32 || a.Cin < 8 || a.W < 4) return false;
  a.Wp = a.Wo + a.KW - 1;
  // rows per workgroup: the fewest rounds of workgroups (two per CU in half its LDS) times
  // rows staged in each
  int best = 0;
  int64_t cost = 0;
  for (int R = 1; R <= std::min(a.Ho, 16); ++R) {
    a.R = R;
    a.nb = int(ceil_div(int64_t(R) * a.Wp, 32));
    a.xpos = a.nb * 32 + (a.KH - 1) * a.Wp;
    const size_t lds = few_out_lds(a);
    if (a.nb > 16 || lds > kFewLdsMax) break;
    const int64_t slots = lds > kFewLds ? 256 : 512;
    const int64_t c = ceil_div(a.B * ceil_div(a.Ho, R), slots) * (R + a.KH - 1);
    if (!best || c < cost) {
      best = R;
      cost = c;
    }
  }
  if (!best) return false;
  a.R = best;
  a.nb = int(ceil_div(int64_t(a.R) * a.Wp, 32));
  a.xpos = a.nb * 32 + (a.KH - 1) * a.Wp;
  a.rtiles = int(ceil_div(a.Ho, a.R));
  // A batch of planes of up to 64 pixels over more than two workgroups per CU: the gather's tiles
  // run over the images, and up to four of its k-tiles are no chain (9 -> 3 on 2032 x 3 x 3 15.8
  // against 8.0 us; longer ones gain all the same: 16 -> 1 9x9 on 657 x 4 x 4 8.5 against 29.9).
  if (!any && int64_t(a.Ho) * a.Wo <= 64 && int64_t(a.B) * a.rtiles > 512 && int64_t(a.Cin) * a.KH * a.KW <= 128)
    return false;
  return int64_t(a.B) * a.rtiles <= kMaxGridX256;
}

int run_few_out(FewOutArgs a, bool any, hipStream_t st) {
  if (!few_out_plan(a, any)) return 1;
  static const bool ok = raise_lds(reinterpret_cast<const void*>(&few_out_kernel<1>)) &&
                         raise_lds(reinterpret_cast<const void*>(&few_out_kernel<2>)) &&
                         raise_lds(reinterpret_cast<const void*>(&few_out_kernel<3>)) &&
                         raise_lds(reinterpret_cast<const void*>(&few_out_kernel<4>));
  if (!ok) return 1;
  const unsigned grid = unsigned(a.B * a.rtiles);
  const size_t lds = few_out_lds(a);
  if (a.nb <= 4) few_out_kernel<1><<<grid, 256, lds, st>>>(a);
  else if (a.nb <= 8) few_out_kernel<2><<<grid, 256, lds, st>>>(a);
  else if (a.nb <= 12) few_out_kernel<3><<<grid, 256, lds, st>>>(a);
  else few_out_kernel<4><<<grid, 256, lds, st>>>(a);
  return check_launch("conv few outputs");
}

// ---------------------------------------------------------------------------------------
// Few inputs: Cin <= 4, KW in {3, 5, 7, 9}
// ---------------------------------------------------------------------------------------
struct FewInArgs {
  const uint16_t* x;
  const uint16_t* w;
  const uint16_t* bias;
  uint16_t* out;
  int B, Cin, Cout, H, W, KH, ph, pw, Ho, Wo, flip, act;
  int Wp;     // Wo + KW - 1
  int tiles;  // pixel tiles of 128 NP per image
};

constexpr int kFewInPad = 16;   // positions a pair may read past the grid (masked)

// Workgroup = (image, 128 NP consecutive output pixels, 32 MT output channels).  LDS: the
// input rows those pixels read as a zero-padded grid of four channels per position, and the
// weights as [ky][kx pair][channel m][2 kx x 4 ci].  A k-step takes one pair per lane half.
// The last pair's second half lies past the kernel: its weights are 0 and its positions are
// replaced by 0, since a value there may be infinite.
template <int KW, int MT, int NP>
__global__ __launch_bounds__(256) void few_in_kernel(FewInArgs a) {
  constexpr int NST = (KW + 3) / 4;  // k-steps per kernel row
  constexpr int kM = 32 * MT, kPix = 128 * NP;
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  const int b = blockIdx.x / a.tiles, p0 = (blockIdx.x % a.tiles) * kPix;
  const int m0 = blockIdx.y * kM;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 31, half = lane >> 5;
  const int npix = a.Ho * a.Wo;
  const int oy0 = p0 / a.Wo;
  const int rows = min(p0 + kPix - 1, npix - 1) / a.Wo - oy0 + a.KH;
  uint16_t* ws = smem;                             // [KH * NST * 2][kM][8]
  uint16_t* xs = smem + a.KH * NST * 2 * kM * 8;   // [rows * Wp + kFewInPad][4]
  const int64_t plane = int64_t(a.H) * a.W;

  const uint16_t* xb = a.x + int64_t(b) * a.Cin * plane;
  const uint32_t mwp = 0xFFFFFFFFu / uint32_t(a.Wp) + 1;
  const int npos = rows * a.Wp + kFewInPad;
#pragma unroll 4
  for (int i = tid; i < npos; i += 256) {
    const int r = fast_div(i, mwp), c = i - r * a.Wp;
    const int iy = oy0 - a.ph + r, ix = c - a.pw;
    const bool ok = r < rows && iy >= 0 && iy < a.H && ix >= 0 && ix < a.W;
    const int64_t off = ok ? int64_t(iy) * a.W + ix : 0;
    uint32_t v[4];
#pragma unroll
    for (int c4 = 0; c4 < 4; ++c4) {
      const uint32_t u = xb[min(c4, a.Cin - 1) * plane + off];
      v[c4] = ok && c4 < a.Cin ? u : 0u;
    }
    *reinterpret_cast<uint2*>(xs + i * 4) = make_uint2(v[0] | (v[1] << 16), v[2] | (v[3] << 16));
  }
  // weights: a thread keeps its tap and writes the four channels of its rows; the positions
  // kx >= KW of the last pairs are zeros
  {
    const int taps = a.KH * KW, tp = min(taps, 256), step = 256 / tp, first = tid / tp;
    const int rows_w = min(kM, a.Cout - m0);
    const int64_t srow = int64_t(a.flip ? 1 : a.Cin) * taps, schan = int64_t(a.flip ? a.Cout : 1) * taps;
    if (first < step) {
      for (int tap = tid - first * tp; tap < taps; tap += tp) {
        const int ky = tap / KW, kx = tap - ky * KW;
        const uint16_t* wt = a.w + m0 * srow + (a.flip ? taps - 1 - tap : tap);
        uint16_t* d = ws + (ky * NST * 2 + (kx >> 1)) * kM * 8 + (kx & 1) * 4;
#pragma unroll 4
        for (int m = first; m < rows_w; m += step) {
          uint32_t v[4];
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const uint32_t u = wt[m * srow + min(c, a.Cin - 1) * schan];
            v[c] = c < a.Cin ? u : 0u;
          }
          *reinterpret_cast<uint2*>(d + m * 8) = make_uint2(v[0] | (v[1] << 16), v[2] | (v[3] << 16));
        }
      }
    }
    for (int i = tid; i < a.KH * (4 * NST - KW) * kM; i += 256) {
      const int m = i % kM, t = i / kM, ky = t / (4 * NST - KW), kx = KW + t - ky * (4 * NST - KW);
      *reinterpret_cast<uint2*>(ws + ((ky * NST * 2 + (kx >> 1)) * kM + m) * 8 + (kx & 1) * 4) = make_uint2(0, 0);
    }
  }
  __syncthreads();

  const uint16_t* xp[NP];
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    const int p = min(p0 + (j * 4 + wave) * 32 + lr, npix - 1);
    const int oy = p / a.Wo, ox = p - oy * a.Wo;
    xp[j] = xs + ((oy - oy0) * a.Wp + ox + 2 * half) * 4;
  }
  const uint16_t* wp = ws + (half * kM + lr) * 8;
  f32x16_t acc[NP][MT];
#pragma unroll
  for (int j = 0; j < NP; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[j][i] = zero_acc();
  for (int ky = 0; ky < a.KH; ++ky, wp += NST * 2 * kM * 8) {
#pragma unroll
    for (int s = 0; s < NST; ++s) {
      bf16x8_t wf[MT];
#pragma unroll
      for (int i = 0; i < MT; ++i) wf[i] = as_bf16x8(*reinterpret_cast<const u32x4_t*>(wp + (s * 2 * kM + i * 32) * 8));
#pragma unroll
      for (int j = 0; j < NP; ++j) {
        // this lane half's pair: kx = 4 s + 2 half and the next
        uint2 lo = *reinterpret_cast<const uint2*>(xp[j] + s * 16);
        uint2 hi = *reinterpret_cast<const uint2*>(xp[j] + s * 16 + 4);
        if (4 * s + 2 >= KW && half) lo = make_uint2(0, 0);
        if (4 * s + 1 >= KW || (4 * s + 3 >= KW && half)) hi = make_uint2(0, 0);
        const bf16x8_t bf = as_bf16x8(u32x4_t{lo.x, lo.y, hi.x, hi.y});
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[j][i] = mfma_32x32x16(bf, wf[i], acc[j][i]);
      }
    }
#pragma unroll
    for (int j = 0; j < NP; ++j) xp[j] += a.Wp * 4;
  }
  // a lane holds runs of 4 pixels of channel i * 32 + lr: the tile goes through LDS so that
  // each store is 16 bytes of a channel's contiguous run (2-byte stores of 32-pixel runs
  // bound this kernel: 45 against 30 us at 128 x 3 -> 64 x 64 x 64)
  constexpr int kOut = kPix + 8;  // elements per channel row in LDS
  __syncthreads();
  uint16_t* os = smem;
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int co = m0 + i * 32 + lr;
    const float bias = a.bias && co < a.Cout ? bf16_to_f32(a.bias[co]) : 0.0f;
#pragma unroll
    for (int j = 0; j < NP; ++j)
#pragma unroll
      for (int r = 0; r < 16; r += 4) {
        uint32_t h[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          h[e] = f32_to_bf16(act_forward(a.act, 0.0f, a.bias ? acc[j][i][r + e] + bias : acc[j][i][r + e]));
        *reinterpret_cast<uint2*>(os + (i * 32 + lr) * kOut + (j * 4 + wave) * 32 + mfma_row(r, lane)) =
            make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
      }
  }
  __syncthreads();
  const int nco = min(kM, a.Cout - m0);
  for (int i = tid; i < nco * (kPix / 8); i += 256) {
    const int co = i / (kPix / 8), p = p0 + (i % (kPix / 8)) * 8;
    const uint16_t* src = os + co * kOut + (p - p0);
    uint16_t* o = a.out + (int64_t(b) * a.Cout + m0 + co) * npix + p;
    if (p + 8 <= npix) {
      *reinterpret_cast<Pix8*>(o) = *reinterpret_cast<const Pix8*>(src);
    } else {
      for (int e = 0; p + e < npix; ++e) o[e] = src[e];
    }
  }
}

// The tile of a conv of KW columns: 32 mt channels x 128 np pixels; np 0 where the kernel does
// not apply or loses.
struct FewInPlan {
  int mt = 0, np = 0;
  size_t lds = 0;
};

// Where the kernel is the better one, in `wgs` tiles of 64 channels x 128 pixels (us, this one /
// the gather): planes that fill less than half of a tile only while two workgroups per CU hold
// them all (3 -> 102 3x3 on 1859 x 4 x 4 45 / 9.2, 1 -> 254 7x7 on 445 x 4 x 4, 46 / 11.3; on up to
// 512 workgroups 0.4-0.9 of its time).  With a bias, which the gather adds element by element,
// everything else (0.3-0.9).  Without one, a lone input channel leaves three of four channel slots
// empty, so not 5 columns (25 taps are one k-tile of the gather: 1.0-1.5 of its time) nor many
// workgroups (1 -> 228 9x9 on 73 x 63 x 9 41 / 23); and taps that fill one k-tile of the gather (3x3
// of 3 channels) leave nothing to gain but the wide stores of more than 64 channels on a few
// hundred workgroups (0.93; 1.09 past 1024) or of many pixels on fewer channels.
bool few_in_pays(const FewInArgs& a, int KW) {
  const int64_t px = int64_t(a.Ho) * a.Wo, wgs = a.B * ceil_div(px, 128) * ceil_div(a.Cout, 64);
  if (px <= 64 && wgs > 512) return false;
  if (a.bias) return true;
  if (a.Cin == 1 && (KW == 5 || wgs > 1024)) return false;
  if (a.Cin * a.KH * KW <= 32) return a.Cout > 64 ? wgs <= 1024 : wgs > 512;
  return true;
}

FewInPlan few_in_plan(const FewInArgs& a, int KW, bool any) {
  FewInPlan p;
  if (a.KH > 16 || a.KH < 1 || (KW != 3 && KW != 5 && KW != 7 && KW != 9) || a.Cin > 4 || ceil_div(a.Cout, 32) > 65535 ||
      !(any || few_in_pays(a, KW)))
    return p;
  p.mt = a.Cout > 32 ? 2 : 1;
  const int64_t px = int64_t(a.Ho) * a.Wo;
  // 256 pixels per workgroup where that still gives two workgroups per CU (a workgroup's
  // weights and halo rows are staged once per tile), else 128.
  for (int np = a.B * ceil_div(px, 256) * ceil_div(a.Cout, 64) >= 512 ? 2 : 1; np > 0 && !p.np; --np) {
    const int pix = 128 * np;
    // the most input rows `pix` consecutive pixels read
    const int rows = std::min((pix - 2) / a.Wo + 2, a.Ho) + a.KH - 1;
    p.lds = std::max(size_t(a.KH) * ((KW + 3) / 4) * 2 * 32 * p.mt * 16 +
                         size_t(int64_t(rows) * (a.Wo + KW - 1) + kFewInPad) * 8,
                     size_t(32 * p.mt) * (pix + 8) * 2);
    if (p.lds <= kFewLdsMax && a.B * ceil_div(px, pix) <= kMaxGridX256) p.np = np;
  }
  return p;
}

template <int KW, int MT, int NP>
int launch_few_in_np(FewInArgs a, size_t lds, hipStream_t st) {
  static const bool ok = raise_lds(reinterpret_cast<const void*>(&few_in_kernel<KW, MT, NP>));
  if (!ok) return 1;
  a.tiles = int(ceil_div(int64_t(a.Ho) * a.Wo, 128 * NP));
  const dim3 grid(unsigned(a.B * a.tiles), unsigned(ceil_div(a.Cout, 32 * MT)));
  few_in_kernel<KW, MT, NP><<<grid, 256, lds, st>>>(a);
  return check_launch("conv few inputs");
}

template <int KW>
int launch_few_in(const FewInArgs& a, const FewInPlan& p, hipStream_t st) {
  if (p.mt == 2) return p.np == 2 ? launch_few_in_np<KW, 2, 2>(a, p.lds, st) : launch_few_in_np<KW, 2, 1>(a, p.lds, st);
  return p.np == 2 ? launch_few_in_np<KW, 1, 2>(a, p.lds, st) : launch_few_in_np<KW, 1, 1>(a, p.lds, st);
}

int run_few_in(FewInArgs a, int KW, bool any, hipStream_t st) {
  const FewInPlan p = few_in_plan(a, KW, any);
  if (!p.np) return 1;
  a.Wp = a.Wo + KW - 1;
  switch (KW) {
    case 3: return launch_few_in<3>(a, p, st);
    case 5: return launch_few_in<5>(a, p, st);
    case 7: return launch_few_in<7>(a, p, st);
    default: return launch_few_in<9>(a, p, st);
  }
}

// ---------------------------------------------------------------------------------------
// Weight gradient: few = dy (few outputs) or few = x (few inputs), few channels * KW <= 32
// ---------------------------------------------------------------------------------------
struct FewWgArgs {
  const uint16_t* wide;  // x (few = dy) or dy (few = x): [B][Cw][Hw][Ww]
  const uint16_t* few;   // [B][Cf][Hf][Wf]
  float* part;           // [workgroups][total]
  int Cw, Cf, Hw, Ww, Hf, Wf, Ho, Wo, KH, KW, ph, pw;
  int Wq;            // staged row: the wide side's columns, rounded up to 8
  int R;             // output rows per tile
  int tpi, ntiles;   // tiles per image, tiles
  int wrows, frows;  // staged rows of the wide and the few side
  int PW, PF;        // LDS elements per wide channel / few row (odd multiples of 8)
  int RP;            // LDS elements per raw few row: KW zeros, Wq columns, KW + 2 zeros (even)
  int M;             // Cf * KW
  int wblks;         // blocks of 32 wide channels
  int total;         // wblks * KH * M * 32 + output channels
  int bias;
};

constexpr int kFewMaxKy = 2;  // kernel rows per wave: KH <= 16
constexpr int kFewStage = 6;  // wide loads in flight per thread

// Workgroup = (32 wide channels, a strided set of tiles of R output rows of one image).  Per
// tile: the wide rows as [channel][row * Wq + column], zero outside the image, and the few
// side as [(channel, kx)][row * Wq + q] = few[channel][row][q -+ kx +- pw], zero outside its
// rows.  Output (channel, kx), wide channel, ky sums few * wide over the R * Wq positions,
// with ky * Wq added on the side that is x.
//
// The products include x values against zeros that stand for no pair (columns past the few
// side's, rows past the last output row, the k pad), which an infinity or NaN in x would turn
// into NaN: a tile with one in its x is summed over the real pairs only, by scalar FMAs.
template <bool kFewDy>
__global__ __launch_bounds__(kFewThreads) void few_wgrad_kernel(FewWgArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  uint16_t* xw = smem;               // [32][PW]
  uint16_t* xf = smem + 32 * a.PW;   // [32][PF]
  uint16_t* xr = xf + 32 * a.PF;     // [Cf * frows][RP]: the few side's rows
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 31, lk = (lane >> 5) * 8;
  const int wb = blockIdx.y, c0 = wb * 32;
  const int64_t planew = int64_t(a.Hw) * a.Ww, planef = int64_t(a.Hf) * a.Wf;
  const int K = (a.R * a.Wq + 15) & ~15;  // past R * Wq: zeros of both sides' pads
  for (int i = tid; i < 32 * 8; i += kFewThreads) {
    xw[(i >> 3) * a.PW + a.wrows * a.Wq + (i & 7)] = 0;
    xf[(i >> 3) * a.PF + a.frows * a.Wq + (i & 7)] = 0;
  }

  f32x16_t acc[kFewMaxKy];
#pragma unroll
  for (int i = 0; i < kFewMaxKy; ++i) acc[i] = zero_acc();
  int koff[kFewMaxKy];  // this wave's kernel rows wave, wave + 8, ... (past the last: computed, dropped)
#pragma unroll
  for (int i = 0; i < kFewMaxKy; ++i) koff[i] = min(wave + 8 * i, a.KH - 1) * a.Wq;
  float bsum = 0.0f;

  const int ng = a.Wq >> 2, nv = a.Wq >> 3;
  const uint32_t mrp = 0xFFFFFFFFu / uint32_t(a.RP) + 1, mkw = 0xFFFFFFFFu / uint32_t(a.KW) + 1;
  const uint32_t mfr = a.frows > 1 ? 0xFFFFFFFFu / uint32_t(a.frows) + 1 : 0;
  const uint32_t mnv = nv > 1 ? 0xFFFFFFFFu / uint32_t(nv) + 1 : 0;
  const uint32_t mng = 0xFFFFFFFFu / uint32_t(ng) + 1;
  const uint32_t mwr = a.wrows > 1 ? 0xFFFFFFFFu / uint32_t(a.wrows) + 1 : 0;
  for (int tile = blockIdx.x; tile < a.ntiles; tile += gridDim.x) {
    const int b = tile / a.tpi, oy0 = (tile - b * a.tpi) * a.R;
    if (tile != int(blockIdx.x)) __syncthreads();  // the previous tile's reads are done
    // wide side: items of 4 columns; a row's last group is loaded to end with the row and
    // shifted, so every load is whole and every LDS write aligned
    const int wy0 = kFewDy ? oy0 - a.ph : oy0;
    const int wylim = kFewDy ? a.Hw : a.Ho;
    int odd = 0;
    for (int it0 = tid; it0 < 32 * a.wrows * ng; it0 += kFewThreads * kFewStage) {
      uint64_t v[kFewStage];
      int dst[kFewStage];
#pragma unroll
      for (int j = 0; j < kFewStage; ++j) {
        const int it = it0 + j * kFewThreads;
        const int rc = fast_div(it, mng), g = it - rc * ng;
        const int ch = a.wrows > 1 ? fast_div(rc, mwr) : rc, row = rc - ch * a.wrows;
        const int y = wy0 + row, col = g * 4;
        const bool in = it < 32 * a.wrows * ng;
        const bool ok = in && c0 + ch < a.Cw && y >= 0 && y < wylim && col < a.Ww;
        const int cl = min(col, a.Ww - 4);
        const Pix4 t = *reinterpret_cast<const Pix4*>(
            a.wide + (ok ? (int64_t(b) * a.Cw + c0 + ch) * planew + int64_t(y) * a.Ww + cl : 0));
        const uint64_t u = (uint64_t(t.lo) | (uint64_t(t.hi) << 32)) >> (ok ? 16 * (col - cl) : 0);
        v[j] = ok ? u : 0;
        dst[j] = in ? ch * a.PW + row * a.Wq + col : -1;
        if (kFewDy && ok)
          odd |= ((u & 0x7F80) == 0x7F80) | (((u >> 16) & 0x7F80) == 0x7F80) | (((u >> 32) & 0x7F80) == 0x7F80) |
                 (((u >> 48) & 0x7F80) == 0x7F80);
      }
#pragma unroll
      for (int j = 0; j < kFewStage; ++j)
        if (dst[j] >= 0) *reinterpret_cast<uint64_t*>(xw + dst[j]) = v[j];
    }
    // few side: its rows between KW zeros on either side, ...
    const int fy0 = kFewDy ? oy0 : oy0 - a.ph;
    for (int it = tid; it < a.Cf * a.frows * a.RP; it += kFewThreads) {
      const int rc = fast_div(it, mrp), col = it - rc * a.RP - a.KW;
      const int cf = a.frows > 1 ? fast_div(rc, mfr) : rc, y = fy0 + rc - cf * a.frows;
      const bool ok = y >= 0 && y < a.Hf && col >= 0 && col < a.Wf;
      const uint32_t u = a.few[ok ? (int64_t(b) * a.Cf + cf) * planef + int64_t(y) * a.Wf + col : 0];
      if (!kFewDy) odd |= ok && (u & 0x7F80) == 0x7F80;
      xr[it] = ok ? uint16_t(u) : uint16_t(0);
    }
    __syncthreads();
    // ... then 8 columns of one shifted row per item: 4 dwords, or 5 moved by one element
    for (int it = tid; it < a.M * a.frows * nv; it += kFewThreads) {
      const int mr = nv > 1 ? fast_div(it, mnv) : it, q8 = it - mr * nv;
      const int m = a.frows > 1 ? fast_div(mr, mfr) : mr, row = mr - m * a.frows;
      const int cf = fast_div(m, mkw), kx = m - cf * a.KW;
      const int at = (cf * a.frows + row) * a.RP + q8 * 8 + (kFewDy ? a.pw - kx : kx - a.pw) + a.KW;
      const uint32_t* d = reinterpret_cast<const uint32_t*>(xr) + (at >> 1);
      uint32_t u[5], o[4];
#pragma unroll
      for (int e = 0; e < 5; ++e) u[e] = d[e];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (at & 1) ? __builtin_amdgcn_alignbit(u[e + 1], u[e], 16) : u[e];
      *reinterpret_cast<u32x4_t*>(xf + m * a.PF + row * a.Wq + q8 * 8) = u32x4_t{o[0], o[1], o[2], o[3]};
    }
    odd = __syncthreads_or(odd);
    const int nr = min(a.R, a.Ho - oy0);
    if (a.bias) {
      // bias gradient: the tile's sum of dy
      if (kFewDy) {
        if (wave < a.Cf && wb == 0) {
          const uint16_t* d = a.few + (int64_t(b) * a.Cf + wave) * planef + int64_t(oy0) * a.Wf;
          for (int i = lane; i < nr * a.Wf; i += 64) bsum += bf16_to_f32(d[i]);
        }
      } else if (tid < 256) {
        const uint16_t* d = xw + (tid >> 3) * a.PW;
        for (int i = tid & 7; i < nr * a.Wq; i += 8) bsum += bf16_to_f32(d[i]);
      }
    }
    if (odd) {
      // D[m][c]: row m = mfma_row(r, lane), column lr
#pragma unroll
      for (int i = 0; i < kFewMaxKy; ++i)
        for (int r = 0; r < 16; ++r) {
          const int m = mfma_row(r, lane);
          if (m >= a.M) continue;
          const int kx = m % a.KW, s = kFewDy ? a.pw - kx : kx - a.pw;
          const uint16_t* f = xf + m * a.PF + (kFewDy ? 0 : koff[i]);
          const uint16_t* w = xw + lr * a.PW + (kFewDy ? koff[i] : 0);
          float t = acc[i][r];
          for (int row = 0; row < nr; ++row)
            for (int q = 0; q < a.Ww; ++q)
              if (q + s >= 0 && q + s < a.Wf)
                t = fmaf(bf16_to_f32(f[row * a.Wq + q]), bf16_to_f32(w[row * a.Wq + q]), t);
          acc[i][r] = t;
        }
      continue;
    }
    const uint16_t* fa = xf + lr * a.PF + lk;
    const uint16_t* wa = xw + lr * a.PW + lk;
    for (int k = 0; k < K; k += 16) {
      if (kFewDy) {
        const bf16x8_t f = as_bf16x8(*reinterpret_cast<const u32x4_t*>(fa + k));
#pragma unroll
        for (int i = 0; i < kFewMaxKy; ++i)
          acc[i] = mfma_32x32x16(f, as_bf16x8(*reinterpret_cast<const u32x4_t*>(wa + koff[i] + k)), acc[i]);
      } else {
        const bf16x8_t w = as_bf16x8(*reinterpret_cast<const u32x4_t*>(wa + k));
#pragma unroll
        for (int i = 0; i < kFewMaxKy; ++i)
          acc[i] = mfma_32x32x16(as_bf16x8(*reinterpret_cast<const u32x4_t*>(fa + koff[i] + k)), w, acc[i]);
      }
    }
  }

  float* out = a.part + int64_t(blockIdx.x) * a.total;
#pragma unroll
  for (int i = 0; i < kFewMaxKy; ++i) {
    const int ky = wave + 8 * i;
    if (ky >= a.KH) continue;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = mfma_row(r, lane);
      if (m < a.M) out[((wb * a.KH + ky) * a.M + m) * 32 + lr] = acc[i][r];
    }
  }
  if (a.bias) {
    float* ob = out + a.wblks * a.KH * a.M * 32;
    if (kFewDy) {
      for (int o = 32; o > 0; o >>= 1) bsum += __shfl_xor(bsum, o);
      if (lane == 0 && wave < a.Cf && wb == 0) ob[wave] = bsum;
    } else {
      for (int o = 4; o > 0; o >>= 1) bsum += __shfl_xor(bsum, o);
      if (tid < 256 && (tid & 7) == 0 && c0 + (tid >> 3) < a.Cw) ob[c0 + (tid >> 3)] = bsum;
    }
  }
}

// gw / gb from the workgroups' partials: 8 groups of 32 consecutive entries per block, group
// z summing partials z, z + 8, ..., the groups added in order (a fixed association).
__global__ __launch_bounds__(256) void few_wgrad_reduce_kernel(const float* __restrict__ part, uint16_t* __restrict__ gw,
                                                               uint16_t* __restrict__ gb, int nwg, FewWgArgs a,
                                                               int few_dy, int n) {
  const int z = threadIdx.x >> 5, e = threadIdx.x & 31;
  const int i = blockIdx.x * 32 + e;
  __shared__ float red[8][33];
  float s = i < n ? sum_strided8(0.0f, part + i, a.total, z, 8, nwg) : 0.0f;
  red[z][e] = s;
  __syncthreads();
  if (z || i >= n) return;
  for (int q = 1; q < 8; ++q) s += red[q][e];
  const int nw = a.wblks * a.KH * a.M * 32;
  if (i >= nw) {
    gb[i - nw] = f32_to_bf16(s);
    return;
  }
  int t = i >> 5;
  const int m = t % a.M;
  t /= a.M;
  const int ky = t % a.KH, cw = (t / a.KH) * 32 + (i & 31);
  if (cw >= a.Cw) return;
  const int cf = m / a.KW, kx = m - cf * a.KW;
  const int64_t at = few_dy ? int64_t(cf) * a.Cw + cw : int64_t(cw) * a.Cf + cf;
  gw[(at * a.KH + ky) * a.KW + kx] = f32_to_bf16(s);
}

// The weight gradient's geometry (operands and outputs left out); 0 LDS bytes where the kernel
// does not apply or (unless `any`) loses.
size_t few_wgrad_plan(FewWgArgs& a, int B, int Cin, int Cout, int H, int W, int KH, int KW, int ph, int pw, bool bias,
                      bool any) {
  a.Ho = H + 2 * ph - KH + 1;
  a.Wo = W + 2 * pw - KW + 1;
  const bool few_dy = Cout <= Cin;
  a.Cw = few_dy ? Cin : Cout;
  a.Cf = few_dy ? Cout : Cin;
  a.Hw = few_dy ? H : a.Ho;
  a.Ww = few_dy ? W : a.Wo;
  a.Hf = few_dy ? a.Ho : H;
  a.Wf = few_dy ? a.Wo : W;
  a.KH = KH; a.KW = KW; a.ph = ph; a.pw = pw;
  a.M = a.Cf * KW;
  // (pw <= KW: a shifted row then stays within the zeros kept around it)
  if (pw > KW || a.Cf > 4 || a.Cw < 8 || KH > 8 * kFewMaxKy || KH < 1 || KW < 3 || a.M > 32 || a.Ww < 4) return 0;
  // Few inputs: a tile is one image's, so planes of up to 64 pixels (3 -> 254 5x5 on 1266 x 4 x 4 94
  // against the general kernels' 29 us; from 7x7 on up to 25) and up to 64 channels on a few thousand
  // pixels, one tile's latency against splits over the chip (3 -> 22 9x9 on 4 x 45 x 22 14.8 / 10.3),
  // stay there.  A bias, whose gradient is a pass of its own there, draws the two level; it has no
  // say, so that the weight gradient has the same bits with and without.  Few outputs gain
  // throughout (0.2-0.9).
  const int64_t px = int64_t(a.Ho) * a.Wo;
  if (!any && !few_dy && (px <= (KH * KW >= 49 ? 25 : 64) || (Cout <= 64 && B * px < 8000))) return 0;
  a.Wq = (a.Ww + 7) & ~7;
  a.wblks = int(ceil_div(a.Cw, 32));
  const int64_t total = int64_t(a.wblks) * KH * a.M * 32 + Cout;
  if (total > (1 << 24) || a.wblks > 65535) return 0;
  a.total = int(total);
  a.bias = bias;
  auto geometry = [&](int R) {
    a.R = R;
    a.wrows = few_dy ? R + KH - 1 : R;
    a.frows = few_dy ? R : R + KH - 1;
    auto pitch = [](int n) { return (n & 8) ? n : n + 8; };  // an odd multiple of 8
    a.PW = pitch(a.wrows * a.Wq + 8);
    a.PF = pitch(a.frows * a.Wq + 8);
    a.RP = (a.Wq + 2 * KW + 3) & ~1;
    return size_t(32) * (a.PW + a.PF) * 2 + size_t(a.Cf) * a.frows * a.RP * 2 + 16;
  };
  // rows per tile: the fewest rounds of one workgroup per CU times rows staged in each (4
  // more for what a tile costs besides)
  int best = 0;
  int64_t cost = 0;
  for (int R = 1; R <= std::min(a.Ho, 16); ++R) {
    if (geometry(R) > kFewLdsMax) break;
    const int64_t c = ceil_div(int64_t(B) * ceil_div(a.Ho, R) * a.wblks, 256) * (R + KH - 1 + 4);
    if (!best || c < cost) {
      best = R;
      cost = c;
    }
  }
  if (!best) return 0;
  const size_t lds = geometry(best);
  a.tpi = int(ceil_div(a.Ho, a.R));
  if (int64_t(B) * a.tpi > 0x7fffffff) return 0;
  a.ntiles = B * a.tpi;
  return lds;
}

FewOutArgs few_out_args(int B, int Cin, int Cout, int H, int W, int KH, int KW, int ph, int pw) {
  FewOutArgs a{};
  a.B = B; a.Cin = Cin; a.Cout = Cout; a.H = H; a.W = W; a.KH = KH; a.KW = KW; a.ph = ph; a.pw = pw;
  a.Ho = H + 2 * ph - KH + 1;
  a.Wo = W + 2 * pw - KW + 1;
  return a;
}

FewInArgs few_in_args(const FewOutArgs& o) {
  FewInArgs a{};
  a.x = o.x; a.w = o.w; a.bias = o.bias; a.out = o.out;
  a.B = o.B; a.Cin = o.Cin; a.Cout = o.Cout; a.H = o.H; a.W = o.W; a.KH = o.KH; a.ph = o.ph; a.pw = o.pw;
  a.Ho = o.Ho; a.Wo = o.Wo; a.flip = o.flip; a.act = o.act;
  return a;
}

}  // namespace

int conv_few_fwd(const uint16_t* x, const uint16_t* w, const uint16_t* bias, uint16_t* out, int B, int Cin, int Cout,
                 int H, int W, int KH, int KW, int ph, int pw, int flip, int act, bool any,
                 hipStream_t st) {
  FewOutArgs a = few_out_args(B, Cin, Cout, H, W, KH, KW, ph, pw);
  a.x = x; a.w = w; a.bias = bias; a.out = out; a.flip = flip; a.act = act;
  const int rc = run_few_out(a, any, st);
  return rc <= 0 ? rc : run_few_in(few_in_args(a), KW, any, st);
}

int conv_few_wgrad(const uint16_t* x, const uint16_t* dy, uint16_t* gw, uint16_t* gb, int B, int Cin, int Cout, int H,
                   int W, int KH, int KW, int ph, int pw, bool any, hipStream_t st) {
  FewWgArgs a{};
  const size_t lds = few_wgrad_plan(a, B, Cin, Cout, H, W, KH, KW, ph, pw, gb != nullptr, any);
  if (!lds) return 1;
  const bool few_dy = Cout <= Cin;
  a.wide = few_dy ? x : dy;
  a.few = few_dy ? dy : x;
  static const bool ok = raise_lds(reinterpret_cast<const void*>(&few_wgrad_kernel<true>)) &&
                         raise_lds(reinterpret_cast<const void*>(&few_wgrad_kernel<false>));
  if (!ok) return 1;
  const int nwg = std::min(a.ntiles, std::max(1, 256 / a.wblks));
  a.part = static_cast<float*>(xdna_hip_cache_alloc(size_t(nwg) * a.total * sizeof(float)));
  if (!a.part) return -1;
  const dim3 grid{unsigned(nwg), unsigned(a.wblks)};
  if (few_dy) few_wgrad_kernel<true><<<grid, kFewThreads, lds, st>>>(a);
  else few_wgrad_kernel<false><<<grid, kFewThreads, lds, st>>>(a);
  const int n = gb ? a.total : a.total - Cout;
  few_wgrad_reduce_kernel<<<unsigned(ceil_div(n, 32)), 256, 0, st>>>(a.part, gw, gb, nwg, a, few_dy ? 1 : 0, n);
  xdna_hip_cache_free(a.part);  // stream-ordered reuse: the next user of the block runs after the reduce
  return check_launch("conv few-channel weight gradient");
}

int conv_few_pick(int op, int B, int Cin, int Cout, int H, int W, int KH, int KW, int ph, int pw, bool bias,
                  bool any) {
  if (op == 2) {
    FewWgArgs a{};
    return few_wgrad_plan(a, B, Cin, Cout, H, W, KH, KW, ph, pw, bias, any) ? 3 : 0;
  }
  // (the input gradient as a forward conv of dy)
  static const uint16_t one = 0;
  const bool dx = op == 1;
  if (dx && (ph > KH - 1 || pw > KW - 1)) return 0;
  FewOutArgs a = dx ? few_out_args(B, Cout, Cin, H + 2 * ph - KH + 1, W + 2 * pw - KW + 1, KH, KW, KH - 1 - ph, KW - 1 - pw)
                    : few_out_args(B, Cin, Cout, H, W, KH, KW, ph, pw);
  a.bias = bias && !dx ? &one : nullptr;
  return few_out_plan(a, any) ? 1 : few_in_plan(few_in_args(a), KW, any).np ? 2 : 0;
}

}  // namespace xdna
