// Stride-1 convolutions with few channels on one side (conv_few.hip).  Each returns 1 where
// it does not apply or loses to the general kernels (any: only where it does not apply), 0
// when launched, -1 with the error set.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace xdna {

// y = act(conv(x, w) + bias) for few outputs or few inputs (act 0 none, 1 ReLU).  flip: w is the forward conv's
// weight, [Cin][Cout][KH][KW] in this direction's terms, and its taps are reversed (the
// input gradient as a forward conv of dy).
int conv_few_fwd(const uint16_t* x, const uint16_t* w, const uint16_t* bias, uint16_t* out, int B, int Cin, int Cout,
                 int H, int W, int KH, int KW, int ph, int pw, int flip, int act, bool any, hipStream_t st);

// gw (and gb where not null) of such a conv.
int conv_few_wgrad(const uint16_t* x, const uint16_t* dy, uint16_t* gw, uint16_t* gb, int B, int Cin, int Cout, int H,
                   int W, int KH, int KW, int ph, int pw, bool any, hipStream_t st);

// Which of these kernels takes a stride-1 conv (op 0 forward, 1 input gradient, 2 weight gradient; Cin, Cout, H, W
// and the paddings are the conv's): 1 few outputs, 2 few inputs, 3 weight gradient, 0 none.
int conv_few_pick(int op, int B, int Cin, int Cout, int H, int W, int KH, int KW, int ph, int pw, bool bias,
                  bool any);

}  // namespace xdna
