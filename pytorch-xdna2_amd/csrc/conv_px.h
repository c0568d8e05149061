// 3x3 convolutions as implicit GEMMs over real output pixels (conv_px.hip), reading the
// packed rows and the prepared weights of conv3x3.hip.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "common.h"

namespace xdna {

// Which pixels and taps a launch computes.
enum PxForm {
  kPxStride1 = 0,   // out H x W from packed H x W
  kPxStride2 = 1,   // out ceil(H/2) x ceil(W/2) (3x3, stride 2, padding 1) from packed H x W
  kPxS2Dgrad = 2    // out H x W, the input gradient of that conv, from packed ceil(H/2) x ceil(W/2)
};

// Whether the operands fit the kernel's 32-bit offsets.  H x W: the stride-1 image.
bool conv_px_fits(int form, int B, int cin, int cout, int H, int W, int layout);

// y (or, kPxS2Dgrad, dx) = act(conv + bias).  xp: packed rows of `layout`; wt: the prepared
// weights [co_pad][chunks * 9 * 64].  tile: 0 automatic; 1 64 x 64 (channels x pixels),
// K split over the waves; 2 64 x 64; 3 64 x 128; 4 128 x 128; kPxS2Dgrad in column pairs
// 5 64 x 64, 6 64 x 128 (measurements).  0 when launched, -1 with the error set.
int conv_px(int form, const uint16_t* xp, const uint16_t* wt, const uint16_t* bias, uint16_t* out, int B, int cin,
            int cout, int H, int W, int layout, int act, int tile, hipStream_t st);

// Weight gradient partials [splits][co_pad][9][ci_pad] (and bias partials [splits][co_pad])
// of a stride-1 or stride-2 conv, from the packed rows of x (H x W) and of dY.
struct PxWgradPlan {
  int N = 0, MC = 1, ci_pad = 0, co_pad = 0, kt_per = 0, splits = 0;
  size_t part_bytes = 0, bpart_bytes = 0;
};
// Whether the operands fit the offsets and the pixels a plan (2.6 million).
bool conv_px_wgrad_fits(int form, int B, int Cin, int Cout, int H, int W, int layout);
PxWgradPlan conv_px_wgrad_plan(int form, int B, int Cin, int Cout, int H, int W, int forced_splits);
int conv_px_wgrad(const PxWgradPlan& p, int form, const uint16_t* xp, const uint16_t* dp, float* part, float* bpart, int B,
                  int Cin, int Cout, int H, int W, int layout, hipStream_t st);

}  // namespace xdna
