// Host-side interface of the few-channel 3x3x3 stem on the matrix cores (the network's first convolution).
#pragma once
#include "common.hpp"
#include "gn_stats.hpp"

namespace sfh {

// y[n][od][oh][ow][cw] = conv3x3x3(x[n][td][th][tw][ct]), stride 1, dilation 1, padding (pd, ph, pw), ct = 1..4.
struct StemArgs {
  int n, od, oh, ow, cw;
  int td, th, tw, ct;
  int pd, ph, pw;
  int64_t ws_wide, ws_thin, ws_kd, ws_kh, ws_kw;  // element strides of the weight (forward)
};

// 16-bit types, 32 or 64 output channels, 32-bit offsets inside a sample.
bool stem_supported(const StemArgs& a, int dtype);
// GroupNorm records per sample the forward leaves (0: not offered for this group count).
int stem_gn_records(const StemArgs& a, int groups);
int stem_fwd(const StemArgs& a, int dtype, const void* x, const void* w, const void* bias, void* y, hipStream_t st, const GnPartialOut& gn);
// Weight gradient [cw][27][ct] through fp32 slices in `ws`.
int stem_wgrad_splits(const StemArgs& a);
size_t stem_wgrad_workspace_bytes(const StemArgs& a);
int stem_wgrad(const StemArgs& a, int dtype, const void* x, const void* gy, void* gw, int gw_dtype, void* ws, hipStream_t st);

}  // namespace sfh
