// Forward for the shapes whose channels do not come in whole 128-byte slabs of
// one deformable group: narrow or uneven channel counts, many deformable groups
// of few channels (mdcn_segment.hip holds the kernels).
#pragma once

#include "mdcn_common.h"

namespace mdcn {

constexpr int kSegPairsMax = 2048;   // (channel group, tap) pairs of one convolution group: 32 KB of LDS

// How the channels of a convolution group are laid out: in segments of `seg`
// channels that belong to one deformable group, each padded to `cps` 16-byte
// chunks, which are read cq at a time.
struct SegPlan {
  int seg;        // channels per segment: gcd(Cin / groups, Cin / dgroups)
  int cps;        // chunks per segment, a multiple of cq
  int cq;         // chunks per channel group: 1, 2 or 4
  int nseg_g;     // segments per convolution group
  int pairs;      // (channel group, tap) pairs per convolution group
  int iters;      // pairs are taken two at a time
  int nb;         // 32-channel blocks of output channels per tile
  int n_ctiles;   // tiles of output channels per group
  int kshare;     // waves of a workgroup that share a pixel block's K range: 1, 2 or 4
  bool rounded;   // 16 bits: samples are rounded to the tensors' type, as the fused kernels do
  size_t xt_bytes, wp_bytes;
};

struct SegArgs {
  Geom g;
  const void *xt;   // [N][chunks][H + 2][W + 2][16 bytes], chunks in order of the padded channels
  const void *wp;   // [G][n_ctiles][iters][fragments of 8 channels x bf16 planes, fp32 with cq = 1: 4 channels][nb][64 lanes][16 bytes]
  OffMaskView om;
  const void *bias;
  void *out;
  // the call's own tensors (a.g.N images of the input), for outputs that are made again one by one
  const void *in, *weight;
  long total_px;
  long n_work;        // pixel tiles x n_ctiles x G
  uint32_t plane_bytes, row_bytes;
  uint32_t img_bytes;
  SegPlan s;
};

// Fills *s for images of *g of type dtype (enum mdcn_dtype); false when the shape is not covered.  rounded: see
// SegPlan, for 64 output channels a tile at most.
bool seg_plan(const Geom &g, int dtype, bool rounded, int n_images, bool may_share, int cus, SegPlan *s);
// The pre-pass writes a.xt from the dense NCHW images a.in (a.g.N of them)
// and, when told to, a.wp from a.weight.
hipError_t seg_prepass(int dtype, const SegArgs &a, bool pack, hipStream_t st);
hipError_t seg_forward(int dtype, const SegArgs &a, hipStream_t st);

}  // namespace mdcn
