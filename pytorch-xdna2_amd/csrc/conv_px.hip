// 3x3 convolutions as implicit GEMMs over real output pixels.
//
// C[co][n] = sum over (input chunk, tap) of W[co][chunk, tap][64] . X[row(n) + tap offset]
// [chunk][64]: the packed rows of conv3x3.hip, one k-tile of 64 channels per (chunk, tap).
// Both operands reach LDS by the 16-byte LDS DMA, whose source address is per lane: a lane
// keeps the row of its pixel and adds the (chunk, tap) offset, a scalar.  So the columns of
// a tile are any pixels, and three things cost nothing that the window kernels pay for:
//   - border rows and columns of the padded grid (a third of its rows at 9 x 9);
//   - a stride: the columns of a stride-2 conv are the packed rows of its even pixels, a
//     quarter of the stride-1 form's products;
//   - the input gradient of a stride-2 conv: its output pixels of one parity (y % 2, x % 2)
//     read 1, 2, 2 or 4 of the taps, from the half-resolution gradient packed as it is.
// The price is that a tap's rows are loaded again for each tap (from L2) where a window is
// loaded once, so large stride-1 grids stay on the window kernels.
//
// LDS: a ring of NS k-tiles, each [rows][8 pieces of 8 k], piece c of row r at c ^ ((r >> 1) &
// 7): the DMA writes 8 whole rows per instruction, fragment reads (32 rows, one piece) are
// free of bank conflicts under the probed lane groups.  One barrier per k-tile: it publishes
// the next k-tile, whose loads every wave has waited for, and frees this one's slot, whose
// fragments every wave has read; the next k-tile's fragments and the loads of the one NS ahead
// are issued between this one's MFMAs.
#include "conv_px.h"

#include "mfma.h"
#include "../../include/xdna_hip.h"

#include <algorithm>
#include <cmath>

namespace xdna {
namespace {

constexpr int kPxSkip = 0x40000000;  // past every valid output offset (host-checked)

struct PxTaps {
  int n;         // taps
  int w[9];      // tap in the prepared weights
  int off[9];    // packed row offset from the output row
};

struct PxArgs {
  const uint16_t* xp;
  const uint16_t* wt;
  const uint16_t* bias;
  uint16_t* out;
  float* part;   // split-K: [nsplit][cout][N] fp32, else null
  int x_bytes, w_bytes, out_bytes;
  int chunks, cout, wp, first, S, So, img, oH, oW;
  int gs;        // packed pixel of lattice pixel (i, j): (i gs, j gs)
  int os;        // output pixel of it: (i os + phase / 2, j os + phase % 2)
  int Ly[4], Lx[4], N[4];  // the phase's lattice
  PxTaps taps[4];
  int npt, nct;  // pixel tiles (of the largest phase), channel tiles
  int nsplit, ch_per, act;
};

// lds_dma16_m0 with a scalar byte offset beside the lane's
__device__ inline void lds_dma16_soff(const i32x4_t& rs, uint32_t m0, int voff, int soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(m0), "v"(voff), "s"(rs), "s"(soff)
               : "m0");
}

__device__ inline void px_pixel(const PxArgs& a, int phase, int n, int& b, int& i, int& j) {
  const int per = a.Ly[phase] * a.Lx[phase];
  b = n / per;
  const int rem = n - b * per;
  i = rem / a.Lx[phase];
  j = rem - i * a.Lx[phase];
}

// Tiles of 64 MI channels x 64 NJ pixels, stored by waves 2 x 2, each MI x NJ blocks of 32 x 32.
// KW 1: each wave multiplies its own blocks over all of K.  KW 4: each wave multiplies the
// whole tile over a quarter of every k-tile (k-step = wave) and the four partial tiles are
// added in wave order through LDS: every fragment is read once per workgroup instead of
// twice, and consecutive MFMAs are independent, for one exchange per tile.
//
// kPair (the stride-2 input gradient, KW 1): a workgroup multiplies both column parities of its
// lattice pixels, one after the other on one ring, and stores them as pairs.  One parity alone
// stores every other pixel, 2 bytes each: half lines, written twice.
template <int MI, int NJ, int NS, int KW, bool kPair>
__global__ __launch_bounds__(256) void conv_px_kernel(PxArgs a) {
  constexpr int TM = 64 * MI, TN = 64 * NJ;
  constexpr int kStage = (TM + TN) * 64;          // elements of one k-tile
  constexpr int kLoads = 2 * MI + 2 * NJ;         // DMA instructions per wave per k-tile
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int lr = lane & 31, half = lane >> 5;
  const int phase = kPair ? 2 * blockIdx.y : blockIdx.y, split = blockIdx.z;
  // XCD x (workgroup L on XCD L % 8) takes every channel tile of its pixel tiles
  const int L = blockIdx.x, k8 = L >> 3;
  const int pt = (k8 / a.nct) * 8 + (L & 7), ct = k8 % a.nct;
  const int N = a.N[phase];
  const int n0 = pt * TN, co0 = ct * TM;
  if (n0 >= N) return;

  const int c_beg = split * a.ch_per, c_end = min(a.chunks, c_beg + a.ch_per);
  const int nkt = (c_end - c_beg) * a.taps[phase].n;
  const int nkt1 = kPair ? (c_end - c_beg) * a.taps[phase + 1].n : 0;  // the odd columns'
  const i32x4_t rsw = uniform_rsrc(lds_dma_rsrc(a.wt, a.w_bytes)), rsx = uniform_rsrc(lds_dma_rsrc(a.xp, a.x_bytes));
  // this wave's DMA blocks of 8 rows: lane L at row 8 blk + L / 8, position L % 8
  int va[2 * MI], vb[2 * NJ];
  const int wrow = a.chunks * 9 * 64;
#pragma unroll
  for (int q = 0; q < 2 * MI; ++q) {
    const int r = (wave * 2 * MI + q) * 8 + (lane >> 3);
    va[q] = ((co0 + r) * wrow + (((lane & 7) ^ ((r >> 1) & 7)) << 3)) * 2;
  }
#pragma unroll
  for (int q = 0; q < 2 * NJ; ++q) {
    const int r = (wave * 2 * NJ + q) * 8 + (lane >> 3);
    int b, i, j;
    px_pixel(a, phase, min(n0 + r, N - 1), b, i, j);
    const int y = i * a.gs, x = j * a.gs;
    const int s = a.S == 1 ? 0 : x / a.So;
    const int p = (b * a.S + s) * a.img + y * a.wp + a.first + x - s * a.So;
    const int row = (p >> 11) * a.chunks * kGroupRows + (p & (kGroupOutRows - 1));
    vb[q] = (row * 64 + (((lane & 7) ^ ((r >> 1) & 7)) << 3)) * 2;
  }
  const uint32_t lds0 = lds_addr(smem);
  // the k-tile to issue next; past the last one it stays there (its loads are never read)
  int ic = c_beg, it = 0, in = 0, iph = phase;
  int soa = (ic * 9 + a.taps[iph].w[0]) * 128, sob = (ic * kGroupRows + a.taps[iph].off[0]) * 128;
  auto issue = [&](int slot, int q) {
    const uint32_t m0 = lds0 + uint32_t(slot * kStage * 2);
    if (q < 2 * MI)
      lds_dma16_soff(rsw, m0 + uint32_t((wave * 2 * MI + q) * 1024), va[q], soa);
    else
      lds_dma16_soff(rsx, m0 + uint32_t(TM * 128 + (wave * 2 * NJ + q - 2 * MI) * 1024), vb[q < 2 * MI ? 0 : q - 2 * MI], sob);
  };
  auto issued = [&] {
    if (++in < nkt + nkt1) {
      if (++it == a.taps[iph].n) {
        it = 0;
        ++ic;
        if (kPair && ic == c_end) {
          ic = c_beg;
          iph = phase + 1;
        }
      }
      soa = (ic * 9 + a.taps[iph].w[it]) * 128;
      sob = (ic * kGroupRows + a.taps[iph].off[it]) * 128;
    }
  };
#pragma unroll
  for (int t = 0; t < NS; ++t) {
#pragma unroll
    for (int q = 0; q < kLoads; ++q) issue(t, q);
    issued();
  }

  constexpr int BI = KW == 4 ? 2 * MI : MI, BJ = KW == 4 ? 2 * NJ : NJ;  // blocks a wave multiplies
  constexpr int KS = KW == 4 ? 1 : 4;                                    // k-steps of a k-tile it takes
  f32x16_t acc[BI][BJ], acc1[kPair ? BI : 1][kPair ? BJ : 1];
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j) {
      acc[i][j] = zero_acc();
      if (kPair) acc1[kPair ? i : 0][kPair ? j : 0] = zero_acc();
    }
  float bias[MI][16];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int co = co0 + (wm * MI + i) * 32 + mfma_row(r, lane);
      bias[i][r] = a.bias && !a.part ? bf16_to_f32(a.bias[min(co, a.cout - 1)]) : 0.0f;
    }
  // fragments: row lr of a 32-row block, piece 2 ks + half
  const int sw = (lr >> 1) & 7;
  struct Frags {
    u32x4_t a[KS][BI], b[KS][BJ];
  };
  const int rm = KW == 4 ? 0 : wm * MI * 32, rn = KW == 4 ? 0 : wn * NJ * 32;
  auto read = [&](Frags& f, int slot, int ks) {
    const int c = ((2 * (KW == 4 ? wave : ks) + half) ^ sw) << 3;
    const uint16_t* ta = smem + slot * kStage + (rm + lr) * 64 + c;
    const uint16_t* tb = smem + slot * kStage + (TM + rn + lr) * 64 + c;
#pragma unroll
    for (int i = 0; i < BI; ++i) f.a[ks][i] = *reinterpret_cast<const u32x4_t*>(ta + i * 32 * 64);
#pragma unroll
    for (int j = 0; j < BJ; ++j) f.b[ks][j] = *reinterpret_cast<const u32x4_t*>(tb + j * 32 * 64);
  };
  // k-tile t from `cur`, read before; k-tile t + 1's fragments into `nxt` and the loads of
  // k-tile t + NS into this one's slot between the MFMAs
  int slot = 0;
  auto ktile = [&](const Frags& cur, Frags& nxt, auto& sum) {
    lds_reads_wait();                     // this wave's reads of k-tile t are done: its slot is free
    lds_dma_wait<(NS - 2) * kLoads>();    // this wave's loads of k-tile t + 1 have landed
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    const int next = slot == NS - 1 ? 0 : slot + 1;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int i = 0; i < BI; ++i)
#pragma unroll
        for (int j = 0; j < BJ; ++j) {
          sum[i][j] = mfma_32x32x16(as_bf16x8(cur.a[ks][i]), as_bf16x8(cur.b[ks][j]), sum[i][j]);
          if (i == 0 && j == 0) read(nxt, next, ks);
          constexpr int kPer = (kLoads + KS * BI * BJ - 1) / (KS * BI * BJ);
#pragma unroll
          for (int q = 0; q < kPer; ++q) {
            const int l = ((ks * BI + i) * BJ + j) * kPer + q;
            if (l < kLoads) issue(slot, l);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
    }
    issued();
    slot = next;
  };
  Frags f0, f1;
  lds_dma_wait<(NS - 1) * kLoads>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) read(f0, 0, ks);
  for (int t = 0; t < nkt; t += 2) {
    ktile(f0, f1, acc);
    if (t + 1 < nkt) ktile(f1, f0, acc);
  }
  if constexpr (kPair) {
    if (nkt & 1) f0 = f1;
    for (int t = 0; t < nkt1; t += 2) {
      ktile(f0, f1, acc1);
      if (t + 1 < nkt1) ktile(f1, f0, acc1);
    }
  }
  lds_dma_wait<0>();
  if constexpr (KW == 4) {
    // [block][wave][register][lane]: every wave's share of a block, added in wave order
    lds_reads_wait();
    __syncthreads();
    float* red = reinterpret_cast<float*>(smem) + lane;
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int j = 0; j < BJ; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) red[(((i * BJ + j) * 4 + wave) * 16 + r) * 64] = acc[i][j][r];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const float* src = red + ((wm * MI + i) * BJ + wn * NJ + j) * 4 * 16 * 64;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          acc[i][j][r] = ((src[r * 64] + src[(16 + r) * 64]) + src[(32 + r) * 64]) + src[(48 + r) * 64];
      }
  }

#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int n = n0 + (wn * NJ + j) * 32 + lr;
    if (a.part) {
      float* P = a.part + int64_t(split) * a.cout * N + n;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int co = co0 + (wm * MI + i) * 32 + mfma_row(r, lane);
          if (n < N && co < a.cout) P[int64_t(co) * N] = acc[i][j][r];
        }
      continue;
    }
    const auto rs = uniform_buffer_rsrc(a.out, a.out_bytes);
    int b, y, x;
    px_pixel(a, phase, min(n, N - 1), b, y, x);
    const int plane = a.oH * a.oW;
    if constexpr (kPair) {
      uint16_t* o = a.out + int64_t(b) * a.cout * plane + (2 * y + (phase >> 1)) * a.oW + 2 * x;
      const bool both = 2 * x + 1 < a.oW;  // (an odd width's last column has no odd neighbour)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int co = co0 + (wm * MI + i) * 32 + mfma_row(r, lane);
          if (n >= N || co >= a.cout) continue;
          const uint32_t lo = f32_to_bf16(act_forward(a.act, 0.0f, acc[i][j][r] + bias[i][r]));
          const uint32_t hi = f32_to_bf16(act_forward(a.act, 0.0f, acc1[i][j][r] + bias[i][r]));
          uint16_t* p = o + int64_t(co) * plane;
          if (both) *reinterpret_cast<Pix2*>(p) = Pix2{lo | (hi << 16)};
          else *p = uint16_t(lo);
        }
      continue;
    }
    const int po =
        n < N ? (b * a.cout * plane + (y * a.os + (phase >> 1)) * a.oW + x * a.os + (phase & 1)) * 2 : kPxSkip;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int co = co0 + (wm * MI + i) * 32 + mfma_row(r, lane);
        const float v = act_forward(a.act, 0.0f, acc[i][j][r] + bias[i][r]);
        __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16(v), rs, po + (co < a.cout ? co * plane * 2 : kPxSkip), 0, 0);
      }
  }
}

// Split-K: out = act(bias + the splits' partials in split order); lattices that are the whole
// output (n is image-major: image, then pixel).
__global__ __launch_bounds__(256) void px_reduce_kernel(PxArgs a) {
  const int plane = a.oH * a.oW;
  const int co = blockIdx.y;
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n >= a.N[0]) return;
  const float bias = a.bias ? bf16_to_f32(a.bias[co]) : 0.0f;
  const float v = sum_strided8(bias, a.part + int64_t(co) * a.N[0] + n, int64_t(a.cout) * a.N[0], 0, 1, a.nsplit);
  const int b = n / plane, pix = n - b * plane;
  a.out[(int64_t(b) * a.cout + co) * plane + pix] = f32_to_bf16(act_forward(a.act, 0.0f, v));
}

template <int MI, int NJ, int NS, int KW, bool kPair = false>
int launch_px(PxArgs a, int phases, hipStream_t st) {
  constexpr int kRing = NS * (64 * MI + 64 * NJ) * 64 * 2, kRed = KW == 4 ? 4 * 64 * MI * 64 * NJ * 4 : 0;
  constexpr int kLds = kRing > kRed ? kRing : kRed;
  static const bool ok = hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_px_kernel<MI, NJ, NS, KW, kPair>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, kLds) == hipSuccess;
  if (!ok) {
    set_error("conv3x3 pixels: cannot enable the kernel's LDS size");
    return -1;
  }
  a.npt = int(ceil_div(*std::max_element(a.N, a.N + 4), 64 * NJ));
  a.nct = int(ceil_div(a.cout, 64 * MI));
  const dim3 grid(unsigned(ceil_div(a.npt, 8) * 8 * a.nct), unsigned(phases), unsigned(a.nsplit));
  conv_px_kernel<MI, NJ, NS, KW, kPair><<<grid, 256, kLds, st>>>(a);
  if (a.part) px_reduce_kernel<<<dim3(unsigned(ceil_div(a.N[0], 256)), unsigned(a.cout)), 256, 0, st>>>(a);
  return check_launch("conv3x3 pixels");
}

// ---------------------------------------------------------------------------------------
// Weight gradient over real output pixels: gw[co][tap][ci] = sum over pixels n of dy[n][co] *
// x[row(n) + tap offset][ci].  K runs over pixels; both sides reach LDS by the DMA as tiles of
// [32 pixels][64 channels] whose rows are any packed rows (a table of them, made once per
// workgroup, sits in LDS), and are read as MFMA fragments by the transposing LDS reads.  A
// workgroup takes 64 MC output channels x 64 input channels x the three taps of one kernel
// row over one split of the pixels: a third of the accumulators, and of the fp32 partials,
// that all nine taps cost, so more splits fit the chip before the partials' traffic does not
// pay; dy is loaded once per kernel row.
// ---------------------------------------------------------------------------------------
struct PxWgArgs {
  const uint16_t* xp;  // packed x, H x W
  const uint16_t* dp;  // packed dY, Ho x Wo
  float* part;         // [splits][co_pad][9][ci_pad]
  float* bpart;        // [splits][co_pad] or null
  int x_bytes, d_bytes;
  int ci_chunks, co_chunks, ci_pad, co_pad;
  int gs, Ly, Lx, N;                       // output lattice: oy, ox; x's pixel (oy gs, ox gs)
  int wp, first, S, So, img;               // x's grid
  int dwp, dfirst, dS, dSo, dimg;          // dY's grid
  int kt_per, splits, ntiles;
};

constexpr int kPwK = 32;                   // pixels per k-tile
constexpr int kPwTile = kPwK * 64;         // elements of a [32][64] tile
constexpr int kPwStages = 3;
constexpr int kPwMaxKt = 80;               // k-tiles per split: the table beside the ring leaves two workgroups per CU
constexpr int kPwMaxSplits = 1024;
constexpr int kPwOob = 0x7FFFFE00;         // a row past both operands: the DMA writes zeros

// 16-byte piece q of pixel row r sits at q ^ 4 ((r >> 1) & 1): the four rows x 64 bytes of a
// half-wave's transposing read fall on 64 distinct banks.
//
// Two workgroups per CU (the second bound: 228 registers; left alone, MC 2 took 279 and one
// workgroup, whose loads nothing covered): 64 -> 256 on 40 x 72 x 72 96 -> 82 us, 512ch
// 1024 x 8 x 8 431 -> 349, 512ch 16 x 18 x 18 43.4 -> 38.3.
template <int MC>
__global__ __launch_bounds__(256, 2) void px_wgrad_kernel(PxWgArgs a) {
  constexpr int kTiles = MC + 3;           // [32][64] tiles per k-tile: dY's, one per tap
  constexpr int kStage = kTiles * kPwTile;
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  int2* table = reinterpret_cast<int2*>(smem + kPwStages * kStage);  // [kt_per * 32]: byte offsets of x's and dY's row
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // XCD x (workgroup L on XCD L % 8) takes every tile of its splits, which read the same rows
  const int L = blockIdx.x, k8 = L >> 3;
  const int split = a.splits % 8 ? L / a.ntiles : (k8 / a.ntiles) * 8 + (L & 7);
  int tile = a.splits % 8 ? L - split * a.ntiles : k8 % a.ntiles;
  const int ky = tile % 3;
  tile /= 3;
  const int cit = tile % a.ci_chunks, cot = tile / a.ci_chunks;  // 64 input channels, 64 MC output channels
  const int n_beg = split * a.kt_per * kPwK, n_end = min(a.N, n_beg + a.kt_per * kPwK);
  const int nkt = max(1, (n_end - n_beg + kPwK - 1) / kPwK);  // a split past the last pixel: one k-tile of zeros
  const int per = a.Ly * a.Lx;
  for (int i = tid; i < nkt * kPwK; i += 256) {
    const int n = n_beg + i;
    int2 v = make_int2(kPwOob, kPwOob);
    if (n < n_end) {
      const int b = n / per, rem = n - b * per, oy = rem / a.Lx, ox = rem - oy * a.Lx;
      const int x = ox * a.gs, xs = a.S == 1 ? 0 : x / a.So, ds = a.dS == 1 ? 0 : ox / a.dSo;
      const int p = (b * a.S + xs) * a.img + oy * a.gs * a.wp + a.first + x - xs * a.So;
      const int q = (b * a.dS + ds) * a.dimg + oy * a.dwp + a.dfirst + ox - ds * a.dSo;
      v.x = ((p >> 11) * a.ci_chunks * kGroupRows + (p & (kGroupOutRows - 1))) * 128;
      v.y = ((q >> 11) * a.co_chunks * kGroupRows + (q & (kGroupOutRows - 1)) + a.dwp + 1) * 128;
    }
    table[i] = v;
  }
  __syncthreads();

  const i32x4_t rsx = uniform_rsrc(lds_dma_rsrc(a.xp, a.x_bytes)), rsd = uniform_rsrc(lds_dma_rsrc(a.dp, a.d_bytes));
  const uint32_t lds0 = lds_addr(smem) + uint32_t(wave * 1024);
  // this wave loads rows 8 wave .. + 7 of every tile: lane L row 8 wave + L / 8, position L % 8
  const int drow = wave * 8 + (lane >> 3);
  const int piece = ((lane & 7) ^ (4 * ((drow >> 1) & 1))) * 16;
  const int last = (nkt - 1) * kPwK + drow;
  int2 rows = table[drow];
  const int sox = (cit * kGroupRows + ky * a.wp) * 128;
  int sod[MC];
#pragma unroll
  for (int c = 0; c < MC; ++c) sod[c] = min(cot * MC + c, a.co_chunks - 1) * kGroupRows * 128;
  auto issue = [&](int slot, int q) {
    const uint32_t m0 = lds0 + uint32_t((slot * kStage + q * kPwTile) * 2);
    if (q < MC)
      lds_dma16_soff(rsd, m0, rows.y + piece, sod[q < MC ? q : 0]);
    else
      lds_dma16_soff(rsx, m0, rows.x + piece, sox + (q - MC) * 128);
  };
  int inext = drow;
  auto issued = [&] {
    inext = min(inext + kPwK, last);
    rows = table[inext];
  };
#pragma unroll
  for (int t = 0; t < kPwStages; ++t) {
#pragma unroll
    for (int q = 0; q < kTiles; ++q) issue(t, q);
    issued();
  }

  // wave (wc, wi): output channel blocks wc * MC .. + MC - 1 of 32, input channel block wi
  const int wc = wave & 1, wi = wave >> 1;
  const int g = lane >> 4, j = lane & 15;
  struct Frags {
    u32x4_t d[2][MC], x[2][3];
  };
  // transposing read of 32 channels from ch0 x 16 pixels from 16 ks of a tile
  auto frag = [&](const uint16_t* tl, int ch0, int ks) {
    const int kr = 16 * ks + 8 * (g >> 1) + (j >> 2), ch = ch0 + 16 * (g & 1) + 4 * (j & 3);
    const uint16_t* p = tl + kr * 64 + (((ch >> 3) ^ (4 * ((kr >> 1) & 1))) << 3) + (ch & 7);
    typedef short i16x4 __attribute__((ext_vector_type(4)));
    typedef unsigned int u2 __attribute__((ext_vector_type(2)));
    const u2 lo = __builtin_bit_cast(
        u2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(p)));
    const u2 hi = __builtin_bit_cast(
        u2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(p + 4 * 64)));
    return u32x4_t{lo[0], lo[1], hi[0], hi[1]};
  };
  auto read = [&](Frags& f, int slot, int ks) {
    const uint16_t* st = smem + slot * kStage;
#pragma unroll
    for (int i = 0; i < MC; ++i) {
      const int blk = wc * MC + i;
      f.d[ks][i] = frag(st + (blk >> 1) * kPwTile, (blk & 1) * 32, ks);
    }
#pragma unroll
    for (int t = 0; t < 3; ++t) f.x[ks][t] = frag(st + (MC + t) * kPwTile, wi * 32, ks);
  };
  f32x16_t acc[MC][3], bacc[MC];
#pragma unroll
  for (int i = 0; i < MC; ++i) {
    bacc[i] = zero_acc();
#pragma unroll
    for (int t = 0; t < 3; ++t) acc[i][t] = zero_acc();
  }
  const bool bias = a.bpart && cit == 0 && ky == 0 && wi == 0;
  const u32x4_t ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
  int slot = 0;
  auto ktile = [&](const Frags& cur, Frags& nxt) {
    lds_reads_wait();
    lds_dma_wait<(kPwStages - 2) * kTiles>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    const int next = slot == kPwStages - 1 ? 0 : slot + 1;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < MC; ++i)
#pragma unroll
        for (int t = 0; t < 3; ++t) {
          acc[i][t] = mfma_32x32x16(as_bf16x8(cur.d[ks][i]), as_bf16x8(cur.x[ks][t]), acc[i][t]);
          if (i == 0 && t == 0) read(nxt, next, ks);
          const int l = (ks * MC + i) * 3 + t;
          if (l < kTiles) issue(slot, l);
          __builtin_amdgcn_sched_barrier(0);
        }
    if (bias) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int i = 0; i < MC; ++i) bacc[i] = mfma_32x32x16(as_bf16x8(cur.d[ks][i]), as_bf16x8(ones), bacc[i]);
    }
    issued();
    slot = next;
  };
  Frags f0, f1;
  lds_dma_wait<(kPwStages - 1) * kTiles>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) read(f0, 0, ks);
  for (int t = 0; t < nkt; t += 2) {
    ktile(f0, f1);
    if (t + 1 < nkt) ktile(f1, f0);
  }
  lds_dma_wait<0>();

  const int lr = lane & 31;
#pragma unroll
  for (int i = 0; i < MC; ++i) {
    const int co0 = cot * 64 * MC + (wc * MC + i) * 32;
    float* P = a.part + (int64_t(split) * a.co_pad + co0) * 9 * a.ci_pad + ky * 3 * a.ci_pad + cit * 64 + wi * 32 + lr;
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) P[(mfma_row(r, lane) * 9 + t) * a.ci_pad] = acc[i][t][r];
    if (bias && lr == 0) {
#pragma unroll
      for (int r = 0; r < 16; ++r) a.bpart[int64_t(split) * a.co_pad + co0 + mfma_row(r, lane)] = bacc[i][r];
    }
  }
}

}  // namespace

bool conv_px_fits(int form, int B, int cin, int cout, int H, int W, int layout) {
  const int Hp = form == kPxS2Dgrad ? (H + 1) / 2 : H, Wp = form == kPxS2Dgrad ? (W + 1) / 2 : W;
  const ConvGeom g = conv_geom(B, Hp, Wp, layout);
  const int64_t chunks = ceil_div(cin, kKStep);
  const int64_t oH = form == kPxStride2 ? (H + 1) / 2 : H, oW = form == kPxStride2 ? (W + 1) / 2 : W;
  // (packed rows end before the weight gradient's out-of-range row offset)
  return int64_t(g.groups) * chunks * kGroupRows * kKStep * 2 < kPwOob - 4096 &&
         int64_t(B) * cout * oH * oW * 2 < kPxSkip && g.m_total < (int64_t(1) << 31) &&
         ceil_div(cout, 256) * 256 * chunks * 9 * kKStep * 2 < (int64_t(1) << 31) && cout <= 65535;
}

int conv_px(int form, const uint16_t* xp, const uint16_t* wt, const uint16_t* bias, uint16_t* out, int B, int cin,
            int cout, int H, int W, int layout, int act, int tile, hipStream_t st) {
  const int Hp = form == kPxS2Dgrad ? (H + 1) / 2 : H, Wp = form == kPxS2Dgrad ? (W + 1) / 2 : W;
  const ConvGeom g = conv_geom(B, Hp, Wp, layout);
  PxArgs a{};
  a.xp = xp;
  a.wt = wt;
  a.bias = bias;
  a.out = out;
  a.chunks = int(ceil_div(cin, kKStep));
  a.cout = cout;
  a.wp = g.st.wp;
  a.first = g.st.first;
  a.S = g.st.S;
  a.So = g.st.So;
  a.img = int(g.img);
  a.oH = form == kPxStride2 ? (H + 1) / 2 : H;
  a.oW = form == kPxStride2 ? (W + 1) / 2 : W;
  a.gs = form == kPxStride2 ? 2 : 1;
  a.os = form == kPxS2Dgrad ? 2 : 1;
  a.act = act;
  a.x_bytes = int(int64_t(g.groups) * a.chunks * kGroupRows * kKStep * 2);
  a.w_bytes = int((cout <= 128 ? 128 : ceil_div(cout, 256) * 256) * a.chunks * 9 * kKStep * 2);
  a.out_bytes = int(int64_t(B) * cout * a.oH * a.oW * 2);
  const int phases = form == kPxS2Dgrad ? 4 : 1;
  for (int p = 0; p < phases; ++p) {
    const int py = p >> 1, px = p & 1;
    a.Ly[p] = form == kPxS2Dgrad ? (H + 1 - py) / 2 : a.oH;
    a.Lx[p] = form == kPxS2Dgrad ? (W + 1 - px) / 2 : a.oW;
    a.N[p] = B * a.Ly[p] * a.Lx[p];
    PxTaps& t = a.taps[p];
    t.n = 0;
    for (int dy = 0; dy < 3; ++dy)
      for (int dx = 0; dx < 3; ++dx) {
        // tap (dy, dx) reads padded-grid row y + dy - 1; the spread gradient has values at
        // even pixels only: parity 0 meets the centre tap, parity 1 taps 0 and 2, whose
        // gradient pixels are the lattice's own and the next
        if (form == kPxS2Dgrad && (((dy + 1 + py) & 1) || ((dx + 1 + px) & 1))) continue;
        const int ry = form == kPxS2Dgrad ? (dy == 2 ? 2 : 1) : dy, rx = form == kPxS2Dgrad ? (dx == 2 ? 2 : 1) : dx;
        t.w[t.n] = dy * 3 + dx;
        t.off[t.n] = ry * a.wp + rx;
        ++t.n;
      }
  }
  a.nsplit = 1;
  a.ch_per = a.chunks;
  const int64_t wgs = ceil_div(a.N[0], 64) * ceil_div(cout, 64);
  if (tile == 0) {
    // 128 x 128 tiles, then 64 x 128, where they give two workgroups per CU; below, 64 x 64, the
    // waves splitting K from 36 k-tiles on (326 channels, 11 x 13 x 13: 15.2 against 17.2 us).
    // The input gradient in column pairs where half as many, longer workgroups still cover
    // the chip: 64 x 128 from 320 of them on (us, without / with pairs: 128 -> 64 channels on
    // 128 x 64 x 64 72 / 57, on 24 x 61 x 67 22 / 17, 32 -> 16 on 16 x 72 x 72 13.1 / 9.7), 64 x 64 from
    // 400 (64 -> 32 on 40 x 36 x 36 10.1 / 8.4; 128 -> 64 on 40 x 18 x 18, 102 of them, 6.9 / 9.0).
    // 128 x 128 leaves no registers for a pair's sums and wins on weights read once (512 -> 512
    // on 64 x 24 x 24 73 / 80).
    const int64_t wide = ceil_div(a.N[0], 128) * phases, ct = ceil_div(cout, 64);
    const bool dx = form == kPxS2Dgrad;
    tile = cout > 64 && wide * ceil_div(cout, 128) >= 512 ? 4
           : dx && ceil_div(a.N[0], 128) * 2 * ct >= 320  ? 6
           : dx && ceil_div(a.N[0], 64) * 2 * ct >= 400   ? 5
           : wide * ct >= 512                             ? 3
           : a.chunks * a.taps[phases - 1].n >= 36        ? 1
                                                          : 2;
  }
  // one lattice of few 64 x 64 tiles: K split over workgroups, at least 18 k-tiles each (the
  // reduce costs what 10 take)
  const int ns = int(std::min<int64_t>(256 / std::max<int64_t>(wgs, 1), a.chunks / 2));
  if (form != kPxS2Dgrad && tile <= 2 && ns >= 2) {
    a.ch_per = int(ceil_div(a.chunks, ns));
    a.nsplit = int(ceil_div(a.chunks, a.ch_per));
    if (a.nsplit > 1) {
      a.part = static_cast<float*>(xdna_hip_cache_alloc(size_t(a.nsplit) * cout * a.N[0] * sizeof(float)));
      if (!a.part) return -1;
    }
  }
  int rc;
  switch (tile) {
    case 1: rc = launch_px<1, 1, 4, 4>(a, phases, st); break;
    case 2: rc = launch_px<1, 1, 4, 1>(a, phases, st); break;
    case 3: rc = launch_px<1, 2, 3, 1>(a, phases, st); break;
    case 4: rc = launch_px<2, 2, 2, 1>(a, phases, st); break;
    case 5: rc = launch_px<1, 1, 4, 1, true>(a, 2, st); break;
    case 6: rc = launch_px<1, 2, 3, 1, true>(a, 2, st); break;
    default: set_error("conv3x3 pixels: unknown tile"); rc = -1;
  }
  // stream-ordered reuse: the next user of the block runs after the reduce
  if (a.part) xdna_hip_cache_free(a.part);
  return rc;
}

bool conv_px_wgrad_fits(int form, int B, int Cin, int Cout, int H, int W, int layout) {
  const int Ho = form == kPxStride2 ? (H + 1) / 2 : H, Wo = form == kPxStride2 ? (W + 1) / 2 : W;
  const ConvGeom g = conv_geom(B, H, W, layout), d = conv_geom(B, Ho, Wo, layout);
  const int64_t ci = ceil_div(Cin, 64), co = ceil_div(Cout, 64);
  // What it addresses: the packed rows of x and of dY, both ending before the out-of-range row
  // offset, and partials the size of the weight.  A split's table holds kPwMaxKt k-tiles, so more
  // pixels than kPwMaxSplits of them have no plan.
  return int64_t(g.groups) * ci * kGroupRows * kKStep * 2 < kPwOob - 4096 &&
         int64_t(d.groups) * co * kGroupRows * kKStep * 2 < kPwOob - 4096 && g.m_total < (int64_t(1) << 31) &&
         ci * 64 * co * 64 * 9 * 2 < (int64_t(1) << 31) &&
         ceil_div(int64_t(B) * Ho * Wo, kPwK) <= int64_t(kPwMaxSplits) * kPwMaxKt;
}

PxWgradPlan conv_px_wgrad_plan(int form, int B, int Cin, int Cout, int H, int W, int forced_splits) {
  PxWgradPlan p;
  const int Ho = form == kPxStride2 ? (H + 1) / 2 : H, Wo = form == kPxStride2 ? (W + 1) / 2 : W;
  p.N = B * Ho * Wo;
  p.MC = Cout > 64 ? 2 : 1;
  p.ci_pad = int(ceil_div(Cin, 64) * 64);
  p.co_pad = int(ceil_div(Cout, 64 * p.MC) * 64 * p.MC);
  const int64_t ktiles = ceil_div(p.N, kPwK);
  const int64_t tiles = int64_t(p.co_pad / (64 * p.MC)) * (p.ci_pad / 64) * 3;
  const double out_bytes = double(p.co_pad) * 9 * p.ci_pad * 4;
  // splits: a multiple of 8 gives every XCD whole splits, tiles * s / 8 workgroups on its 32
  // CUs (21 splits of 12 tiles, 36 workgroups on some XCDs, took 51 us where 16 took 39).  A
  // k-tile costs a CU about 0.3 us of DMA for each of its workgroups (one alone 0.36), a
  // workgroup 2 us of prologue and epilogue, and the partials are written and read once.
  int64_t best = 1;
  double best_t = 1e30;
  for (int64_t s = 1; s <= std::min<int64_t>(ktiles, kPwMaxSplits); s += s < 32 ? 1 : 8) {
    const int64_t kt = ceil_div(ktiles, s);
    if (kt > kPwMaxKt) continue;
    const double per_cu = double(s % 8 ? ceil_div(tiles * s, 256) : ceil_div(s / 8 * tiles, 32));
    // (splits between multiples of 8: 9 of 24 tiles, 256ch B16 36 x 36, 39.7 us; 16 47.4)
    const double t = (per_cu + 0.2) * kt * 0.30e-6 + std::ceil(per_cu / 2) * 2e-6 + 2.0 * s * out_bytes / 5e12;
    if (t < best_t) {
      best_t = t;
      best = s;
    }
  }
  if (forced_splits > 0) best = std::min<int64_t>(std::max<int64_t>(forced_splits, ceil_div(ktiles, kPwMaxKt)), ktiles);
  p.kt_per = int(ceil_div(ktiles, best));
  p.splits = best % 8 ? int(ceil_div(ktiles, p.kt_per)) : int(best);  // a split past the last pixel adds zeros
  p.part_bytes = size_t(p.splits) * p.co_pad * 9 * p.ci_pad * 4;
  p.bpart_bytes = size_t(p.splits) * p.co_pad * 4;
  return p;
}

int conv_px_wgrad(const PxWgradPlan& pl, int form, const uint16_t* xp, const uint16_t* dp, float* part, float* bpart, int B,
                  int Cin, int Cout, int H, int W, int layout, hipStream_t st) {
  const int Ho = form == kPxStride2 ? (H + 1) / 2 : H, Wo = form == kPxStride2 ? (W + 1) / 2 : W;
  const ConvGeom g = conv_geom(B, H, W, layout), d = conv_geom(B, Ho, Wo, layout);
  PxWgArgs a{};
  a.xp = xp;
  a.dp = dp;
  a.part = part;
  a.bpart = bpart;
  a.ci_chunks = int(ceil_div(Cin, 64));
  a.co_chunks = int(ceil_div(Cout, 64));
  a.ci_pad = pl.ci_pad;
  a.co_pad = pl.co_pad;
  a.x_bytes = int(int64_t(g.groups) * a.ci_chunks * kGroupRows * kKStep * 2);
  a.d_bytes = int(int64_t(d.groups) * a.co_chunks * kGroupRows * kKStep * 2);
  a.gs = form == kPxStride2 ? 2 : 1;
  a.Ly = Ho;
  a.Lx = Wo;
  a.N = pl.N;
  a.wp = g.st.wp; a.first = g.st.first; a.S = g.st.S; a.So = g.st.So; a.img = int(g.img);
  a.dwp = d.st.wp; a.dfirst = d.st.first; a.dS = d.st.S; a.dSo = d.st.So; a.dimg = int(d.img);
  a.kt_per = pl.kt_per;
  a.splits = pl.splits;
  a.ntiles = (pl.co_pad / (64 * pl.MC)) * a.ci_chunks * 3;
  static const bool ok =
      hipFuncSetAttribute(reinterpret_cast<const void*>(&px_wgrad_kernel<1>), hipFuncAttributeMaxDynamicSharedMemorySize,
                          160 * 1024) == hipSuccess &&
      hipFuncSetAttribute(reinterpret_cast<const void*>(&px_wgrad_kernel<2>), hipFuncAttributeMaxDynamicSharedMemorySize,
                          160 * 1024) == hipSuccess;
  if (!ok) {
    set_error("conv3x3 pixel weight gradient: cannot raise the dynamic LDS limit");
    return -1;
  }
  const size_t lds = size_t(kPwStages) * (pl.MC + 3) * kPwTile * 2 + size_t(pl.kt_per) * kPwK * 8;
  const unsigned grid = unsigned(pl.splits * a.ntiles);
  if (pl.MC == 2) px_wgrad_kernel<2><<<grid, 256, lds, st>>>(a);
  else px_wgrad_kernel<1><<<grid, 256, lds, st>>>(a);
  return check_launch("conv3x3 pixel weight gradient");
}

}  // namespace xdna
