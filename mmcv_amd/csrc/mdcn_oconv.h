// The offset/mask producer of ModulatedDeformConv2dPack: the plain convolution
// conv_offset (mmcv/ops/modulated_deform_conv.py:297-305,328) from Cin to
// 3 * deform_groups * kh * kw channels with the geometry of the deformable
// convolution itself.  It reads the same zero-bordered slab-major input copy as
// the main kernel and writes its result pixel-major, [pixel][CO_pad], so that the
// main kernel's table builder finds the 27 values of a pixel in one or two cache
// lines instead of 27.
#pragma once

#include "mdcn_common.h"
#include "mdcn_fused.h"

namespace mdcn {

struct OconvArgs {
  Geom g;
  const void *xt;     // zero-bordered slab-major input copy
  const void *owp;    // packed conv_offset weights, see pack_offset_chunks
  const void *obias;  // (CO) or null
  void *raw;          // [N * Ho * Wo][CO_pad]
  long total_px;      // N * Ho * Wo
  int CO;             // 3 * DG * taps
  int CO_pad;         // CO rounded up to 32
  int slabs_total;    // Cin / KC
  int plane_px;       // Hp * Wp
  // tiled kernel: a workgroup computes TH x 32 output pixels of one image from a
  // PH x PW patch of the input copy, `stage` slabs of it at a time
  int tiles_x, tiles_y, PH, PW, stage;
  long tiles;
};

// conv_offset weight (CO, Cin, kh, kw) -> MFMA B fragments: for every
// (slab, tap, ksub, 32-channel block) the 64 lanes' 16-byte operands back to
// back, i.e. one fully coalesced 1 KiB load per fragment.  Lane l holds output
// channel 32 * block + l % 32 and the input channels of 16-byte chunk
// 2 * ksub + l / 32 of the slab.  Rows past CO are zero.  16-byte chunk first, first + stride, ...
struct OffsetPack {
  const void *ow;
  void *owp;
  int CO, cof;
  long total;    // 16-byte chunks
  int blocks;    // workgroups of the pre-pass that do this
};

template <typename E>
__device__ __forceinline__ void pack_offset_chunks(const Geom &g, const OffsetPack &o, long first, long stride) {
  constexpr int EPC = 16 / (int)sizeof(E);  // elements per 16-byte chunk
  for (long idx = first; idx < o.total; idx += stride) {
    long r = idx;
    const int lane = (int)(r & 63);
    r >>= 6;
    const int blk = (int)(r % o.cof);
    r /= o.cof;
    const int ksub = (int)(r & 3);
    r >>= 2;
    const int tap = (int)(r % g.taps);
    const int slab = (int)(r / g.taps);
    const int co = blk * 32 + (lane & 31);
    const int ch = slab * 8 * EPC + (ksub * 2 + (lane >> 5)) * EPC;
    const E *src = (const E *)o.ow + ((long)min(co, o.CO - 1) * g.Cin + ch) * g.taps + tap;
    E v[EPC];
#pragma unroll
    for (int e = 0; e < EPC; ++e) v[e] = co < o.CO ? src[(long)e * g.taps] : from_f32<E>(0.0f);
    uint4 c;
    __builtin_memcpy(&c, v, 16);
    ((uint4 *)o.owp)[idx] = c;
  }
}

// a.tiles_*, PH, PW, stage are filled in here.  dtype: enum mdcn_dtype; CO_pad / 32 blocks of channels, at most 4.
hipError_t oconv_forward(int dtype, OconvArgs a, hipStream_t st);

// The same convolution for shapes the slab-major copy does not cover: one thread
// per output element, NCHW in, NCHW out.
template <typename E>
__global__ __launch_bounds__(256) void oconv_direct_kernel(Geom g, const E *__restrict__ input,
                                                           const E *__restrict__ ow,
                                                           const E *__restrict__ ob,
                                                           E *__restrict__ raw, int CO, long total) {
  const long plane_out = (long)g.Ho * g.Wo;
  const long plane_in = (long)g.H * g.W;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (long)gridDim.x * blockDim.x) {
    const int wo = (int)(idx % g.Wo);
    const int ho = (int)((idx / g.Wo) % g.Ho);
    const int co = (int)((idx / plane_out) % CO);
    const int n = (int)(idx / (plane_out * CO));
    float acc = 0.0f;
    for (int c = 0; c < g.Cin; ++c) {
      const E *im = input + ((long)n * g.Cin + c) * plane_in;
      const E *wrow = ow + ((long)co * g.Cin + c) * g.taps;
      for (int i = 0; i < g.kh; ++i) {
        const int y = ho * g.sh - g.ph + i * g.dh;
        if (y < 0 || y >= g.H) continue;
        for (int j = 0; j < g.kw; ++j) {
          const int x = wo * g.sw - g.pw + j * g.dw;
          if (x < 0 || x >= g.W) continue;
          acc += to_f32(wrow[i * g.kw + j]) * to_f32(im[(long)y * g.W + x]);
        }
      }
    }
    if (ob) acc += to_f32(ob[co]);
    raw[idx] = from_f32<E>(acc);
  }
}

// [pixel][CO_pad] -> dense (N, CO, Ho, Wo), for callers that want to see the
// conv_offset output.
template <typename E>
__global__ __launch_bounds__(256) void raw_to_nchw_kernel(const E *__restrict__ raw_pm,
                                                          E *__restrict__ raw, int CO, int CO_pad,
                                                          long plane_out, long total) {
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (long)gridDim.x * blockDim.x) {
    const long rem = idx % plane_out;
    const int co = (int)((idx / plane_out) % CO);
    const long n = idx / (plane_out * CO);
    raw[idx] = raw_pm[(n * plane_out + rem) * CO_pad + co];
  }
}

// raw, dense (N, n_off + n_msk channels), by images: the first run_off elements of an image are offsets, copied, the
// other run_msk mask logits.  A thread has 16 bytes of raw.
template <typename E>
__global__ __launch_bounds__(256) void raw_split_kernel(const E *__restrict__ raw, E *__restrict__ off, E *__restrict__ msk,
                                                        long run_off, long run_msk, long total) {
  constexpr int EPV = 16 / (int)sizeof(E);
  const long i0 = ((long)blockIdx.x * 256 + threadIdx.x) * EPV;
  if (i0 >= total) return;
  const long run = run_off + run_msk, n = i0 / run, r0 = i0 - n * run;
  E *o = off + n * run_off, *m = msk + n * run_msk - run_off;
  if (i0 + EPV <= total && (r0 + EPV <= run_off || (r0 >= run_off && r0 + EPV <= run))) {
    E v[EPV];
    __builtin_memcpy(v, raw + i0, 16);
    if (r0 < run_off) {
      __builtin_memcpy(o + r0, v, 16);
    } else {
#pragma unroll
      for (int k = 0; k < EPV; ++k) v[k] = from_f32<E>(mask_value<E>(v[k], kMaskLogit));
      __builtin_memcpy(m + r0, v, 16);
    }
    return;
  }
  for (int k = 0; k < EPV && i0 + k < total; ++k) {
    const long nk = (i0 + k) / run, r = i0 + k - nk * run;
    if (r < run_off)
      off[nk * run_off + r] = raw[i0 + k];
    else
      msk[nk * run_msk + r - run_off] = from_f32<E>(mask_value<E>(raw[i0 + k], kMaskLogit));
  }
}

}  // namespace mdcn
