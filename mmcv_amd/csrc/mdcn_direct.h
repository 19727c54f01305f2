// Direct DCNv2 forward: one thread per output element, any shape, NCHW input
// read in place.  It covers the shapes the fused MFMA kernel does not
// (channel counts that are not a multiple of its K slab, very large kernels)
// and gives the tests a second, independent device implementation.  The kernels
// that make an fp32 product of bf16 planes take single outputs from here.
#pragma once

#include "mdcn_common.h"

namespace mdcn {

// One output element before the bias, an fp32 sum over the group's (channel, tap) in order: output channel co at pixel
// (ho, wo) of image n.  `im0`: the image, its channels in_c elements and its pixels in_px elements apart.
// SKIP: a position outside the image adds nothing (else zero times the weight, which is NaN for an infinite one).
template <typename E, bool SKIP>
__device__ __forceinline__ float direct_sum(const Geom &g, const E *im0, long in_c, int in_px, const OffMaskView &om,
                                            const E *weight, int n, int co, int ho, int wo) {
  const int grp = co / g.cout_g;
  const long pix = (long)ho * g.Wo + wo;
  float acc = 0.0f;
  for (int cl = 0; cl < g.cin_g; ++cl) {
    const int c = grp * g.cin_g + cl;
    const int dgi = c / g.ch_per_dg;
    const E *im = im0 + (long)c * in_c;
    const E *off = (const E *)om.off + (long)n * om.off_n + pix * om.off_px +
                   (long)(dgi * 2 * g.taps) * om.off_ch;
    const E *msk = (const E *)om.msk + (long)n * om.msk_n + pix * om.msk_px +
                   (long)(dgi * g.taps) * om.msk_ch;
    const E *wrow = weight + ((long)co * g.cin_g + cl) * g.taps;
    for (int i = 0; i < g.kh; ++i) {
      for (int j = 0; j < g.kw; ++j) {
        const int tap = i * g.kw + j;
        const float dy = to_f32(off[(long)(2 * tap) * om.off_ch]);
        const float dx = to_f32(off[(long)(2 * tap + 1) * om.off_ch]);
        const float m = mask_value<E>(msk[(long)tap * om.msk_ch], om.logit);
        const TapSample s =
            make_tap_sample(ho * g.sh - g.ph + i * g.dh,
                            wo * g.sw - g.pw + j * g.dw, dy, dx, m, g.H, g.W);
        if (SKIP && !s.inside) continue;
        const int y1 = s.y0 + 1, x1 = s.x0 + 1;
        float v = 0.0f;
        if (SKIP || s.inside) {
          if (s.y0 >= 0 && s.x0 >= 0) v += s.w00 * to_f32(im[(s.y0 * g.W + s.x0) * in_px]);
          if (s.y0 >= 0 && x1 <= g.W - 1) v += s.w01 * to_f32(im[(s.y0 * g.W + x1) * in_px]);
          if (y1 <= g.H - 1 && s.x0 >= 0) v += s.w10 * to_f32(im[(y1 * g.W + s.x0) * in_px]);
          if (y1 <= g.H - 1 && x1 <= g.W - 1) v += s.w11 * to_f32(im[(y1 * g.W + x1) * in_px]);
        }
        acc += to_f32(wrow[tap]) * v;
      }
    }
    if (acc != acc) break;  // (it stays NaN)
  }
  return acc;
}

template <typename E>
__global__ __launch_bounds__(256) void direct_kernel(
    Geom g, const E *__restrict__ input, OffMaskView om, const E *__restrict__ weight,
    const E *__restrict__ bias, E *__restrict__ output, long total) {
  const long plane_out = (long)g.Ho * g.Wo;
  const long plane_in = (long)g.H * g.W;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (long)gridDim.x * blockDim.x) {
    const int wo = (int)(idx % g.Wo);
    const int ho = (int)((idx / g.Wo) % g.Ho);
    const int co = (int)((idx / plane_out) % g.Cout);
    const int n = (int)(idx / (plane_out * g.Cout));
    float acc = direct_sum<E, true>(g, input + (long)n * g.Cin * plane_in, plane_in, 1, om, weight, n, co, ho, wo);
    if (bias) acc += to_f32(bias[co]);
    output[idx] = from_f32<E>(acc);
  }
}

}  // namespace mdcn
