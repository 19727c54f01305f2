// Backward of conv_offset, the plain convolution in front of the deformable one
// (mmcv/ops/modulated_deform_conv.py:297-305,328; mmcv/ops/deform_conv.py:381-389,406):
// from the gradients of offset and mask to those of the input, of conv_offset.weight
// and of conv_offset.bias.  Four launches: oconv_bwd_prep_kernel, oconv_dgrad_kernel,
// oconv_wgrad_kernel, oconv_bwd_finish_kernel.  In us, 27 channels of conv_offset, 3x3, and before them the fifteen
// launches of torch's convolution, sigmoid, cat, chunk, their backward and the sum of the two gradients of the input:
//   bf16 N=16 256 channels 100x152: 25 + 111 + 93 + 6; a training call 3010 instead of 3474
//   bf16 N=2 256 channels 50x84: 6 + 10 + 10 + 6; 358 instead of 440
//   fp32 N=2 256 channels 50x84: 6 + 26 + 31 + 5; 560 instead of 600
#pragma once

#include "mdcn_common.h"

namespace mdcn {

constexpr int kOdLdsSmall = 32 * 1024;                // gradient halo of the data kernel: four workgroups per CU
constexpr int kOdLds = 64 * 1024 - 2048;              // ... or two
constexpr int kOdMaxKw = 16;                          // columns of the data kernel's table
constexpr int kOwLds3 = 52 * 1024, kOwLds2 = 80 * 1024, kOwLds1 = 156 * 1024;  // weight kernel, by workgroups per CU
constexpr int kOwTaps = 9, kOwWaves = 3;              // taps of a workgroup of the weight kernel, its waves

struct OconvBwdPlan {
  int CO, cob;            // conv_offset channels, blocks of 32 of them
  int Wp;                 // row pitch of the channel-major gradient: whole runs of 32 pixels
  int d_th, d_waves, d_cper, gh, gw, d_lds;   // data kernel: input rows per wave, waves, blocks of 32 channels, rows and columns of its gradient halo, LDS bytes of that
  int w_th, lw, plane_chunks, w_lds;  // weight kernel: output rows per tile, columns of its input halo, its planes in LDS
  int tgroups, splits;    // ... groups of kOwTaps taps, shares of its tiles
  bool data, weight;
  size_t gpm_bytes, gcm_bytes, owf_bytes, part_bytes, bpart_bytes, xt_bytes;
  size_t total() const { return gpm_bytes + gcm_bytes + owf_bytes + part_bytes + bpart_bytes + xt_bytes; }
};

// False where the halos of its kernels do not fit LDS, or channels do not come in whole 128 bytes.
// data / weight: gradients of the input / of weight and bias wanted; own_copy: nobody has made OconvBwdArgs::xt.
bool oconv_bwd_plan(const Geom &g, int dtype, bool unmodulated, bool data, bool weight, bool own_copy, int cus,
                    OconvBwdPlan *pl);

// Whether a training call of the layers is not slower for it than with torch's convolution backward (for shapes that
// oconv_bwd_plan covers).
bool oconv_bwd_pays(const Geom &g, int dtype, bool unmodulated);

struct OconvBwdArgs {
  Geom g;
  int CO, cob, Wp;
  // dense: input (N, Cin, H, W), weight (CO, Cin, kh, kw), gradients of offset and mask, mask (null when unmodulated)
  const void *x, *ow, *goff, *gmask, *mask;
  void *gin;              // added into; null: not wanted
  void *gw, *gb;          // null: not wanted
  void *gpm;              // [N][Ho * Wo][32 * cob]
  void *gcm;              // [N][32 * cob][Ho][Wp]
  void *owf;              // data kernel's operand, see oconv_bwd_prep_kernel
  float *part;            // [splits][taps][32 * cob][Cin]
  float *bpart;           // [splits][32 * cob]
  const void *xt;         // zero-bordered copy of the input in 32-byte records, [N][Cin * element size / 32][Hp][Wp]
  void *own_xt;           // ... where none is given
  int tiles_y, tiles_x, gh, gw_cols, lw;
  int g_blocks, segs;     // pre-pass: blocks of the gradients, runs of 64 pixels per row
  uint32_t lw_inv;        // 2^20 / lw, rounded up
  int plane_chunks;
  long d_work;            // tiles times blocks of channels of the data kernel
  int tgroups, splits, tiles;
  int waves, c_per, c_groups;  // data kernel: waves, blocks of 32 input channels per workgroup, workgroups per tile
};

hipError_t oconv_backward(int dtype, const OconvBwdPlan &pl, OconvBwdArgs a, unsigned char *ws, hipStream_t st);

}  // namespace mdcn
