// Host helpers the library's sources share.
#pragma once

#include "../../include/mdcn.h"
#include "mdcn_common.h"

namespace mdcn {

constexpr size_t kAlign = 256;
// Column gradient (and columns) held in memory per pass of the backward's matrix-core paths.
constexpr uint64_t kBwdColGradCap = (uint64_t)3 << 29;  // 1.5 GiB each (of one image: an fp32 d beside 16-bit columns 3)
inline size_t align_up(size_t v) { return (v + kAlign - 1) / kAlign * kAlign; }

inline size_t elem_size(int dtype) { return dtype == MDCN_F64 ? 8 : dtype == MDCN_F32 ? 4 : 2; }

inline bool forced_fused(int path) {
  return path == MDCN_PATH_FUSED || path == MDCN_PATH_FUSED_SPLIT || path == MDCN_PATH_FUSED_WIDE ||
         path == MDCN_PATH_FUSED_NARROW;
}

// compute units of the current device
int num_cus();

// ---- backward (mdcn_backward.hip) ----
struct BwdPlan {
  size_t gin_bytes, gw_bytes;  // fp32 staging (0 for fp32 tensors)
  // grad_input / grad_offset / grad_mask by bwd_data_tiled_kernel (else, without
  // `gemm`, one workgroup per tap):
  bool tiled;
  int R, WH, WW;   // its window margin and size
  // matrix-core paths (bwd_colgrad_kernel + bwd_scatter_kernel, bwd_wgrad_kernel):
  bool gemm;       // data gradients
  bool wgemm;      // grad_weight from stored columns
  bool fused;      // ... by bwd_fused_kernel, column gradient in registers (else fp32 in memory, a window of doubles)
  int sR, sWH, sWW;  // window of the scatter kernel
  int sCH;         // channels per pass over that window
  int fR, fWH, fWW;  // window for far offsets (fWH = 0: none), with half as many channels a pass, or 8
  int tw_log;      // fused: log2 of the width of a tile of 256 pixels
  int n_chunk;     // images per pass
  int cg_tile;     // tile of the column-gradient product (kCgTile or kCgTileBig)
  // Padded channel orders of its copies: segments of the input's channels to whole passes of sCH, a group's to
  // a multiple of 32, the output channels of a group to 128 bytes
  ChanMap im, om;
  int M_pad;       // rows of the transposed weight matrix per group
  long P_pad;      // row pitch of the columns matrix
  int parts;       // workgroups of the scatter kernel per tile (shares of the channels)
  FusedSchedule sched;  // fused: of a whole pass of images
  size_t xt_bytes, gt_bytes, wt_bytes, d_bytes, col_bytes, part_bytes;
  int w_tile, w_splits;  // weight-gradient product: tile, shares of the K range
  size_t wpart_bytes;    // ... and their partial sums
  size_t gpad_bytes;     // grad_output with padded rows, when its own rows cannot be copied 16 bytes at a time
  size_t gb_bytes;  // sums of grad_bias
  int bsplits;      // ... shares of a channel's pixels (matrix-core paths)
  size_t mx_bytes;  // the counts of far offsets
  // where the matrix-core paths have their copy of the input, and whether its channels are the input's own
  size_t xt_at() const { return gin_bytes + gb_bytes + mx_bytes; }
  bool plain_copy() const { return (gemm || wgemm) && im.segp == im.seg && im.cgp == im.cg; }
  // fp32 column gradient of fp16 pairs: magnitudes of grad_output's pixels, exponents of the weights' rows and these as pairs, at max_at of the workspace (0: not
  // there, bf16 triples)
  size_t gmax_bytes, wexp_bytes, wpair_bytes, max_at;
  size_t max_bytes() const { return gmax_bytes + wexp_bytes + wpair_bytes; }
  size_t total() const {
    return gin_bytes + gw_bytes + gb_bytes + mx_bytes + xt_bytes + gt_bytes + wt_bytes + d_bytes + col_bytes + part_bytes +
           wpart_bytes + gpad_bytes;
  }
};

// pass_bytes: column gradient (and columns) held at a time
void make_bwd_plan(const mdcn_bwd_params *bp, const Geom &g, uint64_t pass_bytes, BwdPlan *pl);
int run_backward(const mdcn_bwd_params *bp, const Geom &g, const BwdPlan &pl, hipStream_t st);

}  // namespace mdcn
