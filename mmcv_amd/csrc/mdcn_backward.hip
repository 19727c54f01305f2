// Backward: plan, workspace carving and kernel launches.
#include <algorithm>
#include <type_traits>

#include "mdcn_backward.h"
#include "mdcn_backward_ends.h"
#include "mdcn_backward_fused.h"
#include "mdcn_backward_gemm.h"
#include "mdcn_f64.h"
#include "mdcn_fused.h"
#include "mdcn_host.h"
#include "mdcn_prepass.h"

namespace mdcn {

namespace {

// Largest margin R (up to `most`) for which the LDS window of a th x tw output-pixel
// tile fits max_px pixels; -1 if even R = 0 does not.
int window_margin(const Geom &g, int th, int tw, long max_px, int *WH, int *WW, int most = 8) {
  const long base_h = (long)(th - 1) * g.sh + (long)(g.kh - 1) * g.dh + 2;
  const long base_w = (long)(tw - 1) * g.sw + (long)(g.kw - 1) * g.dw + 2;
  int R = -1;
  while (R < most && (base_h + 2 * (R + 1)) * (base_w + 2 * (R + 1)) <= max_px) ++R;
  *WH = (int)base_h + 2 * std::max(R, 0);
  *WW = (int)base_w + 2 * std::max(R, 0);
  return R;
}

// Workgroups that share a tile's passes over the window in bwd_scatter_kernel.  Two fit a CU but take nearly twice as long
// there -- LDS adds and VALU are busy with either --, so what counts is the longest share times the workgroups that a CU gets; a share
// costs some 0.4 of a pass beside its passes (offsets and mask, first loads, its sums for bwd_finish_kernel to add).  A power of two up to
// eight, until the launch fills the chip eight times over, is where it starts from and what calls of many tiles stay with: there any number is within 2 %.
// Whole training calls in us, parts as powers of two / as this has them: bf16 N=4 96 -> 72 channels 37x53, 2 deformable groups (80
// tiles, 6 passes each) 4 129 / 6 110 (3: 115); fp32 N=2 256 50x84 (42, 32) 8 438 / 12 407 (6: 436, 16: 423, 32: 411); N=1 256 50x84 (21, 32)
// 8 266 / 12 249; N=1 512 25x42 (8, 64) 8 390 / 32 294 (12: 354, 16: 321, 64: 308); N=2 128 60x80 stride 2 (16, 32) 8 159 / 16 138; N=4 512
// 25x42 (32, 64) 8 667 / 16 646; bf16 N=2 200 -> 160 40x60 (20, 25) 8 168 / 25 134.
int scatter_parts(long tiles, int passes) {
  constexpr int kCus = 256, kMost = 32;
  auto cost = [&](int parts) {
    const long wgs = tiles * parts, longest = (passes + parts - 1) / parts;
    if (wgs <= kCus) return (double)longest + 0.4;
    if (wgs <= 2 * kCus) return 1.7 * ((double)longest + 0.4);
    return 0.85 * (double)wgs / kCus * ((double)passes / parts + 0.4) + 0.3 * (double)longest;
  };
  int best = 1;
  while (best < 8 && tiles * best < 4096 && 2 * best <= passes) best *= 2;
  double least = 0.9 * cost(best);   // (what changes for less than a tenth may as well be noise)
  for (int parts = best + 1; parts <= kMost && parts <= passes && tiles * parts <= 4 * kCus; ++parts)
    if (cost(parts) <= least) least = cost(best = parts);
  return best;
}

}  // namespace

void make_bwd_plan(const mdcn_bwd_params *bp, const Geom &g, uint64_t pass_bytes, BwdPlan *pl) {
  const bool f64 = bp->conv.dtype == MDCN_F64;
  const bool staged = bp->conv.dtype != MDCN_F32 && !f64;
  const size_t es = elem_size(bp->conv.dtype);
  pl->gin_bytes = (staged && bp->grad_input) ? align_up((size_t)g.N * g.Cin * g.H * g.W * 4) : 0;
  pl->gw_bytes = (staged && bp->grad_weight) ? align_up((size_t)g.Cout * g.cin_g * g.taps * 4) : 0;
  pl->gb_bytes = (staged && bp->grad_bias) ? align_up((size_t)g.Cout * 4) : 0;
  pl->mx_bytes = 0;
  pl->tiled = pl->gemm = pl->wgemm = pl->fused = false;
  pl->tw_log = 0;
  pl->xt_bytes = pl->gt_bytes = pl->wt_bytes = pl->d_bytes = pl->col_bytes = pl->part_bytes = pl->wpart_bytes = 0;
  pl->w_tile = kCgTile;
  pl->w_splits = 1;
  pl->gpad_bytes = 0;
  pl->gmax_bytes = pl->wexp_bytes = pl->wpair_bytes = pl->max_at = 0;
  pl->bsplits = 0;
  pl->im = pl->om = ChanMap{1, 1, 1, 1, 1};
  pl->parts = 1;
  pl->sched = FusedSchedule{0, 1};
  pl->n_chunk = g.N;
  pl->M_pad = 0;
  pl->cg_tile = kCgTile;
  pl->P_pad = 0;
  pl->R = pl->sR = -1;
  pl->WH = pl->WW = pl->sWH = pl->sWW = 0;
  pl->fR = pl->fWH = pl->fWW = 0;
  const int path = forced_fused(bp->conv.path) ? MDCN_PATH_FUSED : bp->conv.path;
  if (path == MDCN_PATH_DIRECT || g.taps > kBwdTapsMax || f64) return;
  const bool forced = path == MDCN_PATH_FUSED;
  const size_t plane_out = (size_t)g.Ho * g.Wo;

  // Matrix-core paths, for every channel count (padded in the copies) and any number of tiles: a call of 42
  // tiles (fp32, N=2, 256 channels, 50x84) takes 0.41 ms here and took 2.57 ms with a workgroup per tap, one
  // whose channels fill nothing (bf16, N=4, 96 -> 72, 37x53) 0.12 ms instead of 0.90.
  const int KC = (int)(128 / es);
  const long s_tiles = (long)g.N * g.DG * ((g.Ho + kScTH - 1) / kScTH) * ((g.Wo + kScTW - 1) / kScTW);
  // 16-bit tensors whose channels come in whole 128-byte slabs, and 64 or more tiles of them: the data side in one kernel,
  // d in registers and grad_input summed in fixed point.  What is smaller or uneven, and fp32, goes through memory with
  // an fp32 d and sums in doubles.
  // (The 64 is a line of precision, not of speed: small calls have had sums in doubles since before this kernel, and fixed point takes
  // bits from gradients beside much larger ones of the same tile -- error of the others by themselves, beside one
  // pixel of 1e3 / 1e5 times their gradient: fp16 2.2e-3 / 0.18 of their norm, bf16 3.1e-3 / 0.20, where sums in doubles leave one
  // rounding, 2.1e-4 and 1.7e-3.  Whole training calls in us, this
  // kernel / the other path: bf16 N=1 512 channels 25x42, 8 tiles, 130 / 163; fp16 N=2 256 50x84, 42, 178 / 226; bf16 N=4 512 25x42, 32, 239 /
  // 316; N=3 512 40x60 stride 2, 4 deformable groups, 36, 192 / 220; N=1 128 56x56, 14, 82 to 111 / 94.)
  const bool whole = g.Cin % KC == 0 && g.cout_g % KC == 0 && g.cin_g % 32 == 0 && g.ch_per_dg % 8 == 0;
  pl->fused = staged && bp->grad_input && whole && (s_tiles >= 64 || forced) && (g.kh - 1) * g.dh < 255 && (g.kw - 1) * g.dw < 255 &&
              s_tiles < (1L << 28) && (long)g.Ho * g.Wo < kBfPlaneMax && (long)g.Hp * g.Wp < kBfPlaneMax;
  const bool columns_only = staged && !bp->grad_input;
  const size_t ds = pl->fused || columns_only ? es : 4;  // bytes of an element of d, or of the columns
  int u = g.cin_g, v = g.ch_per_dg;
  while (v) {
    const int t = u % v;
    u = v;
    v = t;
  }
  const int seg = u;
  auto padded = [](int n, int to) { return (n + to - 1) / to * to; };
  // Channels per pass over the window, and its margins: fewer channels at a time buy a wider window.  A second, wider one
  // is for calls whose offsets leave the first.
  if (pl->fused) {
    // the tile shape that fewer tiles cover the plane with
    const long n32 = (long)((g.Ho + 7) / 8) * ((g.Wo + 31) / 32), n16 = (long)((g.Ho + 15) / 16) * ((g.Wo + 15) / 16);
    pl->tw_log = n16 < n32 ? 4 : 5;
    const int TW = 1 << pl->tw_log, TH = 256 / TW;
    pl->sCH = 16;
    pl->sR = seg % 16 == 0 ? window_margin(g, TH, TW, bf_window_px(16), &pl->sWH, &pl->sWW) : -1;
    if (pl->sR < 2) {
      pl->sCH = 8;
      pl->sR = window_margin(g, TH, TW, bf_window_px(8), &pl->sWH, &pl->sWW);
    }
    pl->fR = window_margin(g, TH, TW, bf_window_px(8), &pl->fWH, &pl->fWW, kScFarMargin);
    if (pl->fR <= pl->sR) pl->fWH = 0;
  } else {
    const int ch_big = columns_only ? 16 : 8;  // doubles: 8 or 4
    pl->sCH = ch_big;
    pl->sR = window_margin(g, kScTH, kScTW, kScWindowPx, &pl->sWH, &pl->sWW);
    // (half the channels also mean less padding where segments are short)
    const bool pads_less = 4 * padded(seg, ch_big) > 5 * padded(seg, ch_big / 2);
    if (pl->sR < 2 || pads_less) {
      int wh, ww;
      const int r = window_margin(g, kScTH, kScTW, 2 * kScWindowPx, &wh, &ww);
      if (r > pl->sR || pads_less) {
        pl->sCH = ch_big / 2;
        pl->sR = r;
        pl->sWH = wh;
        pl->sWW = ww;
      }
    }
    pl->fR = window_margin(g, kScTH, kScTW, (long)kScWindowPx * (2 * ch_big / pl->sCH), &pl->fWH, &pl->fWW, kScFarMargin);
    if (pl->fR <= pl->sR || pl->sCH * es < 16) pl->fWH = 0;  // (a pass reads 8 bytes of channels at least)
  }
  ChanMap &im = pl->im, &om = pl->om;
  im.seg = seg;
  im.segp = padded(seg, pl->sCH);
  im.nseg = g.cin_g / seg;
  im.cg = g.cin_g;
  im.cgp = padded(im.nseg * im.segp, 32);
  om.seg = om.cg = g.cout_g;
  om.nseg = 1;
  om.segp = om.cgp = padded(g.cout_g, KC);
  const int cin_p = g.G * im.cgp;
  const size_t d_img = (size_t)g.taps * cin_p * plane_out * ds;
  // (the limit goes by the columns; an fp32 d beside 16-bit ones has twice their bytes)
  const bool mfma_ok = pl->sR >= 1 && d_img / ds * es <= kBwdColGradCap && plane_out <= ((size_t)1 << 30) &&
                       (size_t)g.H * g.W <= ((size_t)1 << 30);  // (plane offsets held in 32 bits)
  pl->fused = pl->fused && mfma_ok;
  if (mfma_ok) {
    pl->gemm = bp->grad_input != nullptr;
    pl->wgemm = bp->grad_weight != nullptr;
  }
  if (pl->gemm || pl->wgemm) {
    pl->n_chunk = (int)std::min<uint64_t>((uint64_t)g.N, std::max<uint64_t>(1, pass_bytes / d_img));
    pl->xt_bytes = align_up((size_t)g.N * cin_p * g.Hp * g.Wp * es);
    pl->gw_bytes = 0;
    const int passes = g.ch_per_dg / seg * (im.segp / pl->sCH);
    if (pl->fused) {
      pl->sched.passes = passes;
      pl->sched.tiles = pl->n_chunk * g.DG * ((g.Ho + (256 >> pl->tw_log) - 1) / (256 >> pl->tw_log)) *
                        ((g.Wo + (1 << pl->tw_log) - 1) >> pl->tw_log);
    } else {
      pl->parts = scatter_parts(s_tiles, passes);
    }
    pl->bsplits = 1;
    if (bp->grad_bias) {
      const long runs = (long)g.N * (((long)plane_out + kBiasRun - 1) / kBiasRun);
      pl->bsplits = (int)std::min<long>(runs, 64);
      pl->gb_bytes = align_up((size_t)g.Cout * pl->bsplits * 4);
    }
  }
  if (pl->gemm) {
    // Tiles of 256 for calls that have more than two and a half rounds of them, in fp32 if the rounds are full: what they are filled
    // with, in tiles of 128, is 7 in 8 or more with 16 K steps and more, 15 in 16 with 8, 1 - steps / 128.  Otherwise of 128, two
    // workgroups a CU: the last round is fuller, one's products cover the other's barriers, and what fp32 splits behind its LDS reads costs
    // it no more.  Training calls in us, 256 / 128:
    // fp32 of few tiles of 256: N=2 256 channels 50x84 (306) 404 / 380; N=1 512 25x42 (90) 284 / 260; N=8 512 13x21 424 / 380;
    // fp32 256 channels, 8 K steps, by how full: 0.87 (N=12 50x84) 1 790 / 1 765, 0.90 (N=8 64x64) 1 077 / 1 060, 0.93 (N=16 50x84) 2 300 /
    // 2 283, 0.93 (N=4 100x152) 2 028 / 2 011, 0.97 (N=6 100x152) 2 922 / 2 994, 1 (N=16 64x64) 2 014 / 2 020;
    // fp32 512 channels, 16: 0.75 (N=8 32x32) 915 / 891, 0.90 (N=16 32x32) 1 614 / 1 626, 0.94 (N=10 32x32, 720 tiles) 1 093 / 1 120, 0.90 (N=4
    // 64x64) 1 630 / 1 647, 0.93 (N=8 50x84) 3 487 / 3 566, 0.95 (N=6 48x48) 1 596 / 1 625;
    // (triples; with pairs, of all calls of more than 128 tiles of 256, by this rule: N=8 256 64x64 872 / 863, N=8 512 32x32 709 / 695, N=3 512 25x42 479 / 450, N=4 256 50x84 605 / 594,
    // N=16 128 100x152 2 721 / 2 751.)
    // 16 bits: N=4 96 -> 72 37x53 (128 tiles) 113 / 110; N=4 240 60x60 (540) 336 / 331; N=8 104 -> 96 100x100 (1 280) 713 / 720; N=8 312 -> 300
    // 90x100 (3 168) 2 092 / 2 133.
    auto tiles_of = [&](long tile) {
      return (long)pl->n_chunk * g.G * (((long)plane_out + tile - 1) / tile) * ((g.taps * im.cgp + tile - 1) / tile);
    };
    const long big_tiles = tiles_of(kCgTileBig), rounds = (big_tiles + 255) / 256, k_steps = om.cgp * (long)es / 128;
    const bool full = tiles_of(kCgTile) * 128 >= rounds * 4 * 256 * (128 - std::min<long>(16, k_steps));
    pl->cg_tile = (g.taps * im.cgp >= kCgTileBig && plane_out >= (size_t)kCgTileBig && big_tiles > 640 && (es == 2 || full)) ? kCgTileBig : kCgTile;
    pl->M_pad = pl->fused ? g.taps * im.cgp : padded(g.taps * im.cgp, pl->cg_tile);
    pl->gt_bytes = align_up((size_t)g.N * g.G * om.cgp * plane_out * es);
    pl->wt_bytes = align_up((size_t)g.G * pl->M_pad * om.cgp * es);
    pl->d_bytes = pl->fused ? 0 : align_up(d_img * pl->n_chunk);
    pl->mx_bytes = kAlign;
    // fp32: the column gradient as fp16 pairs (tile_products), with sums of up to 64 products as bf16 triples: their error is as large (grad_input against
    // float64, triples / pairs: 64 output channels 1.23e-7 / 1.26e-7, 72 1.43e-7 / 1.37e-7, 256 2.49e-7 / 1.99e-7, 512 3.57e-7 / 2.66e-7).
    if (es == 4 && om.cgp > 64) {
      pl->gmax_bytes = align_up((size_t)g.N * g.G * (om.cgp / KC) * plane_out * 2);
      pl->wexp_bytes = align_up((size_t)g.G * pl->M_pad * 4);
      pl->wpair_bytes = pl->wt_bytes;
    }
    if (pl->fused)
      pl->part_bytes = align_up((size_t)((g.N + pl->n_chunk - 1) / pl->n_chunk) * FusedSchedule::kGroups * 3 * g.taps * 256 * 4);
    else if (pl->parts > 1)
      pl->part_bytes = align_up((size_t)pl->parts * g.N * g.DG * 3 * g.taps * plane_out * 4);
  }
  if (pl->wgemm) {
    const long kpx = 128 / (long)es;  // pixels per K step
    pl->P_pad = ((long)plane_out + kpx - 1) / kpx * kpx;
    pl->col_bytes = align_up((size_t)pl->n_chunk * g.taps * cin_p * pl->P_pad * es);
    const int M = g.taps * im.cgp;
    const long work = (long)pl->n_chunk * (pl->P_pad / kpx);
    // Tiles of 256 where a workgroup's share is long enough: K steps of it were the chip filled evenly.  Shorter ones are mostly
    // their first copies and the partial sums, of which two workgroups of 128 a CU do one beside the other's products.
    // Training calls in us, 256 / 128: fp32 steps of 4.7 (N=1 256 channels 50x84) 245 / 234, 9.3 (N=2) 385 / 380, 10.1 (N=8 512 13x21) 380 / 383,
    // 16.7 (N=1 256 100x152) 587 / 589, 23.7 (N=3 256 72x100) 835 / 842; bf16 and fp16 steps of 0.4 (N=1 512 13x13) 108 / 101, 2.4 (N=1 512
    // 25x42) 132 / 121, 4.6 (N=2 256 50x84) 174 / 166, 9.3 (N=4) 272 / 260, 19.1 (N=8 512 25x42) 351 / 345, 22.8 (N=8 256 72x72) 508 / 507,
    // 25.1 (N=3 256 100x152) 525 / 537, 28.7 (N=12 512 25x42) 482 / 473, 33.5 (N=4 256 100x152) 637 / 653, 66.9 (N=8) 1 203 / 1 246.
    // (28.7 goes the other way, why is not known; fp32 is even from 9 to 24.)
    const long big_steps = work * g.G * ((g.cout_g + kCgTileBig - 1) / kCgTileBig) * ((M + kCgTileBig - 1) / kCgTileBig);
    pl->w_tile = (g.cout_g >= 192 && M >= kCgTileBig && big_steps > 256L * (es == 4 ? 10 : 20)) ? kCgTileBig : kCgTile;
    const long tiles = (long)g.G * ((g.cout_g + pl->w_tile - 1) / pl->w_tile) * ((M + pl->w_tile - 1) / pl->w_tile);
    // one round of workgroups (256-tiles: one per CU, 128-tiles: two), shares of at least 8 K steps
    const long slots = pl->w_tile == kCgTileBig ? 256 : 512;
    pl->w_splits = (int)std::max<long>(1, std::min<long>(std::min<long>(work / 8, 64), slots / tiles));
    pl->wpart_bytes = align_up((size_t)pl->w_splits * g.Cout * M * 4);
    // grad_output rows go to LDS 16 bytes at a time: in place when they start aligned
    if (plane_out % (16 / es) != 0 || ((uintptr_t)bp->grad_output % 16) != 0)
      pl->gpad_bytes = align_up((size_t)g.N * g.Cout * pl->P_pad * es);
  }
  if (bp->grad_input && !pl->gemm) {
    // (small problems keep the per-tap kernel: it has taps x more workgroups)
    pl->R = window_margin(g, kBwdTile, kBwdTile, kBwdWindowBytes / (4 * kBwdChunk), &pl->WH, &pl->WW);
    const long n_tiles = (long)g.N * g.DG * ((g.Ho + kBwdTile - 1) / kBwdTile) * ((g.Wo + kBwdTile - 1) / kBwdTile);
    pl->tiled = pl->R >= 1 && (n_tiles >= 512 || forced);
  }
}

namespace {

// Any shape: tiled or per-tap kernels on the VALU, grad_weight by sampling on the fly.
template <typename E>
int run_backward_general(const mdcn_bwd_params *bp, const Geom &g, const BwdPlan &pl, hipStream_t st) {
  const mdcn_params *p = &bp->conv;
  const long plane_out = (long)g.Ho * g.Wo;
  const OffMaskView om = dense_view(p->offset, p->mask, g);
  unsigned char *ws = (unsigned char *)p->workspace;
  auto blocks_for = [](long n) { return (int)std::max<long>(1, std::min<long>((n + 255) / 256, 1L << 20)); };
  int rc = MDCN_OK;
  auto check = [&]() { if (hipGetLastError() != hipSuccess) rc = MDCN_ERR_LAUNCH; };

  const long n_in = (long)g.N * g.Cin * g.H * g.W;
  const long n_w = (long)g.Cout * g.cin_g * g.taps;
  float *gin32 = pl.gin_bytes ? (float *)ws : (float *)bp->grad_input;
  float *gw32 = pl.gw_bytes ? (float *)(ws + pl.gin_bytes) : (float *)bp->grad_weight;
  float *gb32 = pl.gb_bytes ? (float *)(ws + pl.gin_bytes + pl.gw_bytes) : (float *)bp->grad_bias;

  if (bp->grad_input) {
    hipLaunchKernelGGL(fill_zero_kernel<float>, dim3(blocks_for(n_in / 4 + 1)), dim3(256), 0, st, gin32, n_in);  // (16 bytes per thread)
    check();
  }
  if (bp->grad_weight) {
    hipLaunchKernelGGL(fill_zero_kernel<float>, dim3(blocks_for(n_w / 4 + 1)), dim3(256), 0, st, gw32, n_w);
    check();
  }

  if (bp->grad_input) {
    if (pl.tiled) {
      BwdDataTiledArgs da;
      da.g = g;
      da.input = p->input;
      da.om = om;
      da.weight = p->weight;
      da.gout = bp->grad_output;
      da.gin32 = gin32;
      da.goff = bp->grad_offset;
      da.gmask = bp->grad_mask;
      da.tiles_x = (g.Wo + kBwdTile - 1) / kBwdTile;
      da.tiles_y = (g.Ho + kBwdTile - 1) / kBwdTile;
      da.R = pl.R;
      da.WH = pl.WH;
      da.WW = pl.WW;
      const long blocks = (long)g.N * g.DG * da.tiles_y * da.tiles_x;
      hipLaunchKernelGGL(bwd_data_tiled_kernel<E>, dim3((unsigned)blocks), dim3(256), 0, st, da);
      check();
    } else {
      const int rows = g.N * g.DG * g.taps;  // (image, deformable group, tap)
      const dim3 grid((unsigned)((plane_out + 255) / 256), (unsigned)std::min(rows, 65535));
      hipLaunchKernelGGL(bwd_data_kernel<E>, grid, dim3(256), 0, st, g, (const E *)p->input, om,
                         (const E *)p->weight, (const E *)bp->grad_output, gin32,
                         (E *)bp->grad_offset, (E *)bp->grad_mask, rows);
      check();
    }
    if (pl.gin_bytes) {
      hipLaunchKernelGGL(round_kernel<E>, dim3(blocks_for(n_in / 8 + 1)), dim3(256), 0, st, gin32,  // (8 elements per thread)
                         (E *)bp->grad_input, n_in);
      check();
    }
  }
  if (bp->grad_weight) {
    {
      BwdWeightArgs wa;
      wa.g = g;
      wa.input = p->input;
      wa.om = om;
      wa.gout = bp->grad_output;
      wa.gw32 = gw32;
      wa.k_tiles = (g.cin_g * g.taps + 63) / 64;
      wa.co_tiles = (g.cout_g + 255) / 256;
      wa.px_chunks = (int)((plane_out + 63) / 64);
      const long tiles = (long)wa.k_tiles * wa.co_tiles * g.G;
      const long work = (long)g.N * wa.px_chunks;
      wa.splits = (int)std::max<long>(1, std::min<long>(work, (4L * num_cus() + tiles - 1) / tiles));
      wa.g_vec_ok = (plane_out % (16 / (long)sizeof(E)) == 0) && (((uintptr_t)bp->grad_output % 16) == 0);
      hipLaunchKernelGGL(bwd_weight_kernel<E>, dim3((unsigned)tiles, (unsigned)wa.splits), dim3(256), 0,
                         st, wa);
      check();
    }
    if (pl.gw_bytes) {
      hipLaunchKernelGGL(round_kernel<E>, dim3(blocks_for(n_w / 8 + 1)), dim3(256), 0, st, gw32,
                         (E *)bp->grad_weight, n_w);
      check();
    }
  }
  if (bp->grad_bias) {
    hipLaunchKernelGGL(fill_zero_kernel<float>, dim3(blocks_for(g.Cout)), dim3(256), 0, st, gb32, (long)g.Cout);
    check();
    const int runs = (int)((plane_out + kBiasRun - 1) / kBiasRun);
    const int splits = (int)std::min<long>((long)g.N * runs, 64);
    hipLaunchKernelGGL(bwd_bias_kernel<E>, dim3(g.Cout, splits), dim3(256), 0, st, g,
                       (const E *)bp->grad_output, gb32, runs, splits);
    check();
    if (pl.gb_bytes) {
      hipLaunchKernelGGL(round_kernel<E>, dim3(blocks_for(g.Cout)), dim3(256), 0, st, gb32,
                         (E *)bp->grad_bias, (long)g.Cout);
      check();
    }
  }
  return rc;
}

// The matrix-core path: pre-pass, then per pass of images column gradient, scatter / columns and weight product, then the
// finishing pass.
template <typename E>
int run_backward_matrix(const mdcn_bwd_params *bp, const Geom &g, const BwdPlan &pl, hipStream_t st) {
  const mdcn_params *p = &bp->conv;
  constexpr int KC = 128 / (int)sizeof(E);
  constexpr int EPV = 16 / (int)sizeof(E);
  constexpr bool staged = sizeof(E) == 2;  // grad_input is summed in fp32 and rounded at the end
  const long plane_out = (long)g.Ho * g.Wo;
  const OffMaskView om = dense_view(p->offset, p->mask, g);
  unsigned char *ws = (unsigned char *)p->workspace;
  auto take = [&](size_t bytes) {
    unsigned char *q = ws;
    ws += bytes;
    return q;
  };
  int rc = MDCN_OK;
  auto check = [&]() { if (hipGetLastError() != hipSuccess) rc = MDCN_ERR_LAUNCH; };
  const bool gemm = pl.gemm, wgemm = pl.wgemm;
  const int cin_p = g.G * pl.im.cgp, cout_p = g.G * pl.om.cgp;

  float *gin_staging = (float *)take(pl.gin_bytes);
  float *gin32 = staged ? gin_staging : (float *)bp->grad_input;
  float *bpart = (float *)take(pl.gb_bytes);
  uint32_t *far = (uint32_t *)take(pl.mx_bytes);
  unsigned char *xt = take(pl.xt_bytes), *gT = take(pl.gt_bytes), *wT = take(pl.wt_bytes);
  unsigned char *D = take(pl.d_bytes), *col = take(pl.col_bytes);
  const long off_total = (long)g.N * g.DG * 2 * g.taps * plane_out, mask_total = off_total / 2;
  float *poff = (float *)take(pl.part_bytes);
  float *pmask = poff + (long)pl.parts * off_total;
  float *wpart = (float *)take(pl.wpart_bytes);
  unsigned char *gpad = take(pl.gpad_bytes);
  uint16_t *gmax = pl.max_at ? (uint16_t *)((unsigned char *)p->workspace + pl.max_at) : nullptr;
  int *wexp = pl.max_at ? (int *)((unsigned char *)p->workspace + pl.max_at + pl.gmax_bytes) : nullptr;
  void *wpair = (unsigned char *)wexp + pl.wexp_bytes;
  const long n_in = (long)g.N * g.Cin * g.H * g.W;

  // a sample of the offsets, 64 Ki of them at most, decides which window the scatter kernel uses
  const long off_step = std::max<long>(1, (off_total >> 16) | 1);
  const int far_blocks = (int)std::max<long>(1, std::min<long>(off_total / off_step / 1024, 64));

  // Share of offset components beyond the margin from which the far window is taken: its passes of fewer channels against
  // the samples beyond the other one.  Backward in us, near / far window, by the offsets' sigma:
  // - bwd_fused_kernel, 16 channels a pass or 8.  A pass's products take as long for half the channels, so the line goes by their
  //   K.  bf16, margins 7 and 12: N=8 256 channels 50x84 3.5 433 / 558, 4.0 462 / 563, 4.5 514 / 565, 5.0 608 / 570; N=2 256 135x224 3.5
  //   622 / 679, 4.0 702 / 695, 4.5 819 / 714; margins 8 and 12: N=16 512 25x42 4.0 554 / 730, 6.0 600 / 731.  (Shares: 0.045 for 3.5
  //   and a margin of 7, 0.080 for 4.0, 0.119 for 4.5.)  N=8 64 96x160 3.0 278 / 288, 3.5 302 / 296, 4.0 336 / 306; N=8 128 60x60 3.5
  //   172 / 176, 4.0 184 / 179.
  // - ... 8 or 8, over another window: fp16 N=7 128 118x196 stride 2, margins 8 and 12: 3.0 351 / 353, 4.0 379 / 368, 6.0 480 / 425.
  // - Doubles, 8 or 4, margins 5 and 11: fp32 N=2 256 50x84 2.0 321 / 331, 3.0 328 / 332, 4.0 351 / 338, 6.0 539 / 366; bf16 N=2 128 60x80 3.0
  //   121 / 124, 4.0 131 / 126, 6.0 240 / 138; N=4 96 -> 72 37x53 2.0 116 / 105, 4.0 118 / 103.
  // - ... 4 or 2, margins 3 and 12: fp32 N=4 128 60x80 stride 2 2.0 131 / 164, 4.0 147 / 173, 6.0 178 / 181.  (The line is from when every
  //   sample beyond the window cost more.)
  const int far_share = pl.fused && pl.sCH == 16 && g.cout_g > kBfK ? 11 : pl.fused || pl.sCH == 8 ? 32 : 5;
  const uint32_t far_min = (uint32_t)(off_total / off_step / far_share);
  auto up = [](long n, long per) { return (int)((n + per - 1) / per); };
  {
    BwdPreArgs a;
    a.g = g;
    a.im = pl.im;
    a.om = pl.om;
    a.cin_p = cin_p;
    a.cout_p = cout_p;
    a.in = p->input;
    a.gout = bp->grad_output;
    a.w = p->weight;
    a.xt = xt;
    a.gT = gT;
    a.wT = wT;
    a.gmax = gmax;
    a.wexp = wexp;
    a.wpair = wpair;
    a.gpad = gpad;
    a.col = col;
    a.gin32 = gin32;
    a.n_in = n_in;
    a.x_chunks = up((long)g.H * g.W, 32 * EPV);
    a.g_chunks = up(plane_out, 32 * EPV);
    a.P_pad = pl.P_pad;
    a.run = pl.sCH;
    a.col_rows = (long)pl.n_chunk * g.taps * cin_p;
    a.M_pad = pl.M_pad;
    a.wt_run = pl.fused ? kBfK : 0;
    a.off = p->offset;
    a.n_off = off_total;
    a.off_step = off_step;
    a.far_from = (float)pl.sR;
    a.far = far;
    a.bpart = bpart;
    a.bsplits = pl.bsplits;
    // The bias sums read grad_output a second time.  At the end of the launch they find it in the last-level cache (256 MB) unless
    // what the jobs between move -- its re-layout, the zeros of grad_input -- is more than that holds; right behind the re-layout
    // they find its end.  Whole launch in us at the end / behind the re-layout: bf16, 256 channels 100x152, N=8 (249 MB
    // between) 76 / 79, N=9 (280) 87.6 / 85.9, N=10 (311) 98 / 95, N=16 (498) 175 / 163; 128 channels 200x200, N=16 (655) 230 / 194; fp32,
    // 256 channels 100x152, N=6 (280) 88 / 91, N=8 (374) 128 / 124; N=2 50x84 14.4 / 16.7.
    const bool early = 2.0 * g.N * g.Cout * plane_out * sizeof(E) + 4.0 * n_in > 300e6;
    const int bias_blocks = bp->grad_bias ? g.Cout * pl.bsplits : 0;
    const int jobs[kPreJobs] = {
        g.N * up(cin_p, KC) * a.x_chunks,
        gemm ? g.N * (cout_p / KC) * a.g_chunks : 0,
        early ? bias_blocks : 0,
        pl.gpad_bytes ? up((long)g.N * g.Cout * (pl.P_pad / EPV), 256) : 0,
        gemm ? up(n_in, kPreZeroPerBlock) : 0,
        wgemm && pl.P_pad > plane_out ? up(a.col_rows * (pl.P_pad - plane_out), kPrePadPerBlock) : 0,
        gemm ? wexp ? up((long)g.G * pl.M_pad, kPrePairRows) : up((long)g.G * pl.M_pad * pl.om.cgp, 256) : 0,
        gemm && pl.fWH ? far_blocks : 0,
        early ? 0 : bias_blocks,
    };
    int total = 0;
    for (int j = 0; j < kPreJobs; ++j) a.end[j] = total += jobs[j];
    hipLaunchKernelGGL(bwd_prepass_kernel<E>, dim3((unsigned)total), dim3(256), 0, st, a);
    check();
  }
  for (int n0 = 0; n0 < g.N; n0 += pl.n_chunk) {
    const int nb = std::min(pl.n_chunk, g.N - n0);
    if (gemm && !pl.fused) {
      ColGradArgs ca;
      ca.wT = wT;
      ca.gT = gT;
      ca.gmax = gmax;
      ca.wexp = wexp;
      ca.wpair = wpair;
      ca.D = (float *)D;
      ca.P = (int)plane_out;
      ca.px_tiles = (int)((plane_out + pl.cg_tile - 1) / pl.cg_tile);
      ca.m_tiles = pl.M_pad / pl.cg_tile;
      ca.M = g.taps * pl.im.cgp;
      ca.M_pad = pl.M_pad;
      ca.cin_g = pl.im.cgp;
      ca.cout_g = pl.om.cgp;
      ca.taps = g.taps;
      ca.G = g.G;
      ca.Cin = cin_p;
      ca.Cout = cout_p;
      ca.kslabs = pl.om.cgp / KC;
      ca.n0 = n0;
      ca.total = (long)nb * g.G * ca.px_tiles * ca.m_tiles;
      const dim3 grid((unsigned)((ca.total + 7) / 8 * 8));
      auto launch = [&](auto pairs) {
        if (pl.cg_tile == kCgTileBig)
          hipLaunchKernelGGL((bwd_colgrad_kernel<E, kCgTileBig, decltype(pairs)::value>), grid, dim3(2 * kCgTileBig), 0, st, ca);
        else
          hipLaunchKernelGGL((bwd_colgrad_kernel<E, kCgTile, decltype(pairs)::value>), grid, dim3(2 * kCgTile), 0, st, ca);
      };
      if constexpr (sizeof(E) == 4) {
        if (gmax) launch(std::true_type());
        else launch(std::false_type());
      } else {
        launch(std::false_type());
      }
      check();
    }
    if (pl.fused) {
      if constexpr (staged) {
        BwdFusedArgs fa;
        fa.g = g;
        fa.xt = xt;
        fa.gT = gT;
        fa.wT = wT;
        fa.om = om;
        fa.gin32 = gin32;
        fa.goff = bp->grad_offset;
        fa.gmask = bp->grad_mask;
        fa.col = wgemm ? col : nullptr;
        fa.P_pad = pl.P_pad;
        fa.tw_log = pl.tw_log;
        fa.tiles_x = (g.Wo + (1 << pl.tw_log) - 1) >> pl.tw_log;
        fa.tiles_y = (g.Ho + (256 >> pl.tw_log) - 1) / (256 >> pl.tw_log);
        fa.win = ScatterWindow{pl.sR, pl.sWH, pl.sWW};
        fa.win_far = ScatterWindow{pl.fR, pl.fWH, pl.fWW};
        fa.far = far;
        fa.n_far = far_blocks;
        fa.far_min = far_min;
        fa.n0 = n0;
        fa.sched = pl.sched;
        fa.sched.tiles = pl.sched.tiles / pl.n_chunk * nb;
        fa.part = poff + (long)(n0 / pl.n_chunk) * FusedSchedule::kGroups * 3 * g.taps * 256;
        launch_fused<E>(fa, pl.sCH, st);
        check();
      }
    } else {
    BwdScatterArgs sa;
    sa.g = g;
    sa.xt = xt;
    sa.om = om;
    sa.D = gemm ? D : nullptr;
    sa.gin32 = gin32;
    sa.goff = bp->grad_offset;
    sa.gmask = bp->grad_mask;
    sa.col = wgemm ? col : nullptr;
    sa.run = pl.sCH;
    sa.P_pad = pl.P_pad;
    sa.tiles_x = (g.Wo + kScTW - 1) / kScTW;
    sa.tiles_y = (g.Ho + kScTH - 1) / kScTH;
    sa.win = ScatterWindow{pl.sR, pl.sWH, pl.sWW};
    sa.win_far = ScatterWindow{pl.fR, pl.fWH, pl.fWW};
    sa.far = far;
    sa.n_far = far_blocks;
    sa.far_min = far_min;
    sa.n0 = n0;
    sa.parts = pl.parts;
    sa.im = pl.im;
    sa.cin_p = cin_p;
    sa.poff = poff;
    sa.pmask = pmask;
    sa.off_total = off_total;
    sa.mask_total = mask_total;
    const long sblocks = (long)nb * g.DG * sa.tiles_y * sa.tiles_x;
    const dim3 sgrid((unsigned)sblocks, (unsigned)sa.parts);
    auto launch = [&](auto chv) {
      constexpr int CHS = decltype(chv)::value;
      if (!gemm) {
        if constexpr (staged || CHS <= 8) hipLaunchKernelGGL((bwd_scatter_kernel<E, CHS, false, true>), sgrid, dim3(256), 0, st, sa);
      } else if constexpr (CHS <= 8) {
        if (wgemm)
          hipLaunchKernelGGL((bwd_scatter_kernel<E, CHS, true, true>), sgrid, dim3(256), 0, st, sa);
        else
          hipLaunchKernelGGL((bwd_scatter_kernel<E, CHS, true, false>), sgrid, dim3(256), 0, st, sa);
      }
    };
    if (pl.sCH == 16)
      launch(std::integral_constant<int, 16>());
    else if (pl.sCH == 8)
      launch(std::integral_constant<int, 8>());
    else
      launch(std::integral_constant<int, 4>());
    check();
    }
    if (wgemm) {
      WGradArgs wa;
      wa.gout = pl.gpad_bytes ? (const void *)gpad : bp->grad_output;
      wa.a_pitch = pl.gpad_bytes ? pl.P_pad : plane_out;
      wa.col = col;
      wa.part = wpart;
      wa.P = (int)plane_out;
      wa.P_pad = pl.P_pad;
      wa.ksteps = (int)(pl.P_pad / KC);
      wa.nb = nb;
      wa.n0 = n0;
      wa.M = g.taps * pl.im.cgp;
      wa.cgp = pl.im.cgp;
      wa.rows = pl.im.nseg * pl.im.segp;
      wa.accumulate = n0 > 0;
      wa.cout_g = g.cout_g;
      wa.taps = g.taps;
      wa.G = g.G;
      wa.Cin = cin_p;
      wa.Cout = g.Cout;
      const int wtile = pl.w_tile;
      wa.co_tiles = (g.cout_g + wtile - 1) / wtile;
      wa.m_tiles = (wa.M + wtile - 1) / wtile;
      const long tiles = (long)g.G * wa.co_tiles * wa.m_tiles;
      wa.splits = pl.w_splits;
      wa.total = tiles * wa.splits;
      auto launch_w = [&](auto runv) {
        constexpr int RUN = decltype(runv)::value;
        const dim3 wgrid((unsigned)((wa.total + 7) / 8 * 8));
        if (wtile == kCgTileBig)
          hipLaunchKernelGGL((bwd_wgrad_kernel<E, kCgTileBig, RUN>), wgrid, dim3(2 * kCgTileBig), 0, st, wa);
        else
          hipLaunchKernelGGL((bwd_wgrad_kernel<E, kCgTile, RUN>), wgrid, dim3(2 * kCgTile), 0, st, wa);
      };
      if (!staged || pl.sCH == 16)
        launch_w(std::integral_constant<int, 16>());
      else if constexpr (staged) {
        if (pl.sCH == 8)
          launch_w(std::integral_constant<int, 8>());
        else
          launch_w(std::integral_constant<int, 4>());
      }
      check();
    }
  }

  {
    BwdFinArgs a;
    a.g = g;
    a.im = pl.im;
    a.gin32 = gin32;
    a.gin = bp->grad_input;
    a.n_in = n_in;
    a.poff = poff;
    a.pmask = pmask;
    a.goff = bp->grad_offset;
    a.gmask = bp->grad_mask;
    a.off_total = off_total;
    a.mask_total = mask_total;
    a.parts = pl.parts;
    a.wpart = wpart;
    a.gw = bp->grad_weight;
    a.splits = pl.w_splits;
    a.bpart = bpart;
    a.gb = bp->grad_bias;
    a.bsplits = pl.bsplits;
    a.fpart = poff;
    a.tw_log = pl.tw_log;
    a.n_chunk = pl.n_chunk;
    a.chunks = pl.fused ? (g.N + pl.n_chunk - 1) / pl.n_chunk : 0;
    a.sched = a.sched_last = pl.sched;
    a.sched_last.tiles = pl.sched.tiles / pl.n_chunk * (g.N - (a.chunks - 1) * pl.n_chunk);
    auto cut_tiles = [](const FusedSchedule &sc) {
      int n = 0;
      for (int x = 0; x < FusedSchedule::kXcds; ++x) n += sc.shares(x) > 1 ? sc.rest(x) : 0;
      return n;
    };
    a.cut = cut_tiles(a.sched);
    a.cut_last = cut_tiles(a.sched_last);
    const int jobs[kFinJobs] = {
        gemm && staged ? up(n_in, 1024) : 0,
        pl.fused ? ((a.chunks - 1) * a.cut + a.cut_last) * 3 * g.taps : gemm && pl.parts > 1 ? up(off_total, 1024) : 0,
        gemm && pl.parts > 1 && bp->grad_mask ? up(mask_total, 1024) : 0,
        wgemm ? g.Cout * up(pl.im.cgp, kFinWeightCh) : 0,
        bp->grad_bias ? up(g.Cout, 256) : 0,
    };
    int total = 0;
    for (int j = 0; j < kFinJobs; ++j) a.end[j] = total += jobs[j];
    if (total > 0) {
      hipLaunchKernelGGL(bwd_finish_kernel<E>, dim3((unsigned)total), dim3(256), 0, st, a);
      check();
    }
  }
  return rc;
}

template <typename E>
int run_backward_typed(const mdcn_bwd_params *bp, const Geom &g, const BwdPlan &pl, hipStream_t st) {
  return pl.gemm || pl.wgemm ? run_backward_matrix<E>(bp, g, pl, st) : run_backward_general<E>(bp, g, pl, st);
}

// Double precision: grad_input by atomics into the zeroed tensor, everything else
// has one owner; no workspace.
int run_backward_f64(const mdcn_bwd_params *bp, const Geom &g, hipStream_t st) {
  const mdcn_params *p = &bp->conv;
  const long plane_out = (long)g.Ho * g.Wo;
  auto blocks_for = [](long n) { return (int)std::max<long>(1, std::min<long>((n + 255) / 256, 1L << 20)); };
  int rc = MDCN_OK;
  auto check = [&]() { if (hipGetLastError() != hipSuccess) rc = MDCN_ERR_LAUNCH; };
  if (bp->grad_input) {
    const long n_in = (long)g.N * g.Cin * g.H * g.W;
    hipLaunchKernelGGL(f64_zero_kernel, dim3(blocks_for(n_in)), dim3(256), 0, st, (double *)bp->grad_input, n_in);
    check();
    const long total = (long)g.N * g.DG * g.taps * plane_out;
    hipLaunchKernelGGL(f64_bwd_data_kernel, dim3(blocks_for(total)), dim3(256), 0, st, g, (const double *)p->input,
                       (const double *)p->offset, (const double *)p->mask, (const double *)p->weight,
                       (const double *)bp->grad_output, (double *)bp->grad_input, (double *)bp->grad_offset,
                       (double *)bp->grad_mask, total);
    check();
  }
  if (bp->grad_weight) {
    const long n_w = (long)g.Cout * g.cin_g * g.taps;
    hipLaunchKernelGGL(f64_bwd_weight_kernel, dim3((unsigned)std::min<long>(n_w, 1L << 20)), dim3(256), 0, st, g,
                       (const double *)p->input, (const double *)p->offset, (const double *)p->mask,
                       (const double *)bp->grad_output, (double *)bp->grad_weight);
    check();
  }
  if (bp->grad_bias) {
    hipLaunchKernelGGL(f64_bwd_bias_kernel, dim3((unsigned)std::min(g.Cout, 65535)), dim3(256), 0, st, g,
                       (const double *)bp->grad_output, (double *)bp->grad_bias);
    check();
  }
  return rc;
}

}  // namespace

int run_backward(const mdcn_bwd_params *bp, const Geom &g, const BwdPlan &pl, hipStream_t st) {
  switch (bp->conv.dtype) {
    case MDCN_F64: return run_backward_f64(bp, g, st);
    case MDCN_F32: return run_backward_typed<float>(bp, g, pl, st);
    case MDCN_F16: return run_backward_typed<f16_t>(bp, g, pl, st);
    default: return run_backward_typed<bf16_t>(bp, g, pl, st);
  }
}

}  // namespace mdcn
