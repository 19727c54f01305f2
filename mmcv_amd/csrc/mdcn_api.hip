// C ABI of libmdcn_hip.so (see include/mdcn.h): parameter checks, path choice,
// workspace carving and kernel launches.  No allocation, no synchronisation
// (mdcn_forward_timed excepted, which exists to measure).
#include "../../include/mdcn.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <mutex>
#include <numeric>
#include <type_traits>

#include "mdcn_common.h"
#include "mdcn_direct.h"
#include "mdcn_f64.h"
#include "mdcn_fused.h"
#include "mdcn_fused2.h"
#include "mdcn_fused3.h"
#include "mdcn_fused_f32.h"
#include "mdcn_oconv.h"
#include "mdcn_oconv_backward.h"
#include "mdcn_host.h"
#include "mdcn_pairs.h"
#include "mdcn_prepass.h"
#include "mdcn_segment.h"

namespace mdcn {

int num_cus() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}

}  // namespace mdcn

namespace {

using namespace mdcn;

constexpr size_t kMaxLds = 160 * 1024;
// Device byte offsets into the channels-last copy are 32-bit.
constexpr uint64_t kMaxXtBytes = 0xF0000000ull;
// Per-pass limits in force (mdcn_set_pass_limits lowers them; process wide).  Atomic, so that a
// call that runs while another thread changes them reads one of the two values; a workspace that was
// sized under one value and used under another is still the caller's to avoid.
std::atomic<uint64_t> g_fwd_pass_bytes{kMaxXtBytes};
std::atomic<uint64_t> g_bwd_pass_bytes{kBwdColGradCap};

// Scratch of mdcn_forward_noalloc(): the input copy and the packed weights of one
// call, held by every device the library runs on until the process ends.  Host
// code never uses the array's name as an address: scratch_of_current_device()
// asks the runtime where the current device keeps its copy.
static __device__ __align__(256) unsigned char scratch[MDCN_NOALLOC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void *g_scratch_ptr[kMaxDevices] = {nullptr};

int scratch_of_current_device(void **out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return MDCN_ERR_LAUNCH;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void *ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return MDCN_ERR_LAUNCH;
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return MDCN_OK;
}

int check_params(const mdcn_params *p, Geom *g, bool need_ptrs, bool need_offsets = true) {
  if (!p) return MDCN_ERR_NULL;
  if (p->dtype != MDCN_F32 && p->dtype != MDCN_F16 && p->dtype != MDCN_BF16 && p->dtype != MDCN_F64)
    return MDCN_ERR_DTYPE;
  if (p->N <= 0 || p->Cin <= 0 || p->H <= 0 || p->W <= 0 || p->Cout <= 0 ||
      p->kh <= 0 || p->kw <= 0 || p->sh <= 0 || p->sw <= 0 || p->ph < 0 ||
      p->pw < 0 || p->dh <= 0 || p->dw <= 0 || p->groups <= 0 || p->dgroups <= 0)
    return MDCN_ERR_SHAPE;
  if (p->Cin % p->groups || p->Cout % p->groups || p->Cin % p->dgroups)
    return MDCN_ERR_SHAPE;
  const long Ho = ((long)p->H + 2L * p->ph - ((long)p->dh * (p->kh - 1) + 1)) / p->sh + 1;
  const long Wo = ((long)p->W + 2L * p->pw - ((long)p->dw * (p->kw - 1) + 1)) / p->sw + 1;
  if ((long)p->H + 2L * p->ph < (long)p->dh * (p->kh - 1) + 1 ||
      (long)p->W + 2L * p->pw < (long)p->dw * (p->kw - 1) + 1 || Ho <= 0 || Wo <= 0)
    return MDCN_ERR_SHAPE;
  if (need_ptrs && (!p->input || !p->weight || !p->output)) return MDCN_ERR_NULL;
  if (need_ptrs && need_offsets && !p->offset) return MDCN_ERR_NULL;  // mask NULL: unmodulated
  g->N = p->N; g->Cin = p->Cin; g->H = p->H; g->W = p->W;
  g->Cout = p->Cout; g->kh = p->kh; g->kw = p->kw;
  g->sh = p->sh; g->sw = p->sw; g->ph = p->ph; g->pw = p->pw;
  g->dh = p->dh; g->dw = p->dw; g->G = p->groups; g->DG = p->dgroups;
  g->Ho = (int)Ho; g->Wo = (int)Wo;
  g->cin_g = p->Cin / p->groups;
  g->cout_g = p->Cout / p->groups;
  g->ch_per_dg = p->Cin / p->dgroups;
  g->taps = p->kh * p->kw;
  g->Hp = p->H + 2; g->Wp = p->W + 2;
  return MDCN_OK;
}

// channels per K step: 128 bytes
inline int slab_channels(int dtype) { return dtype == MDCN_F32 ? 32 : 64; }

inline int table_capacity(int taps) { return taps <= kTapsSmall ? kTapsSmall : kTapsLarge; }

// Output-channel tile of the fused kernel for a group of cout_g channels; the
// 256-wide tile leaves LDS room for the 9-tap table only.
inline int pick_ct(int cout_g, int taps) {
  if (cout_g > 128 && taps <= kTapsSmall) return 256;
  return cout_g > 64 ? 128 : 64;
}

bool fused_ok(const mdcn_params *p, const Geom &g) {
  if (p->dtype == MDCN_F64) return false;  // double precision: the one-thread-per-output kernels only
  const int KC = slab_channels(p->dtype);
  if (p->input_nhwc && (g.H < 2 || g.W < 2 || ((uintptr_t)p->input % 16) != 0)) return false;
  if (g.cin_g % KC || g.ch_per_dg % KC) return false;
  if (g.taps > kTapsLarge) return false;
  const int ct = pick_ct(g.cout_g, g.taps), tmax = table_capacity(g.taps);
  if ((p->dtype == MDCN_F32 ? fused_f32_lds_bytes(tmax) : fused_lds_bytes(ct, tmax)) > kMaxLds) return false;
  // one padded image must fit the 32-bit offsets
  const uint64_t img = (uint64_t)g.Hp * g.Wp * g.Cin * elem_size(p->dtype);
  if (img > kMaxXtBytes) return false;
  if ((uint64_t)g.N * g.Ho * g.Wo > 0x7fffffffull) return false;
  return true;
}

// Length of the fp32 kernel's persistent schedule of `tiles` tiles of nk K steps in tile times, as PartSchedule lays
// it out: whole rounds, then the last round's tiles whole, in equal parts or (*even) in even shares, whichever is shorter with what it costs that
// parts meet.  (More than four parts count as four: with the sum of all of them they take no less.  N=1 256
// channels 50x84, six parts of 256-channel tiles 84 us a call, three of 128-channel ones 69.)
// kEvenCost: steps that even shares cost beyond equal parts' or a whole tile's: a second unit, and twice the parts through memory.
constexpr double kEvenCost = 14.0;
double schedule_rounds(long tiles, int nk, bool may_cut, bool *even = nullptr) {
  const int stride = std::max(1, num_cus() / 8);
  if (even) *even = false;
  const long chunk = (tiles + 7) / 8;  // the fullest XCD
  const long full = chunk / stride, rest = chunk % stride;
  if (rest == 0) return (double)full;
  const int rounds = (nk + kGatherAhead - 1) / kGatherAhead, min_rounds = 8 / kGatherAhead;
  if (!may_cut) return (double)full + 1.0;
  const long parts = std::max<long>(1, std::min<long>(std::min<long>(stride / rest, 4), rounds / min_rounds));
  const double equal = 1.0 / (double)parts, shares = (double)rest / stride + kEvenCost / nk;
  if (shares >= equal || rest * rounds < 3L * min_rounds * stride) return (double)full + equal;
  if (even) *even = true;
  return (double)full + shares;
}

struct Plan {
  bool fused;
  int CT, KC, n_ctiles, slabs;
  int n_chunk;       // images per launch of the fused path
  size_t xt_bytes;   // channels-last copy of one chunk
  size_t wp_bytes;   // packed weights
  // fp32 as fp16 pairs (may be left out: bf16 triples): magnitudes of the input's pixels, exponents of weights and of samples
  size_t max_bytes, wexp_bytes, rexp_bytes, tpix_bytes;   // (four weights to an offset)
  size_t pair_bytes() const { return max_bytes + wexp_bytes + rexp_bytes + 5 * tpix_bytes; }
  size_t cut_bytes;  // eight-wave kernel: buffers and counters of the tiles it cuts along K (may be left out)
  int cut_wgs;     // ... one buffer (cut_even: two) and one counter per workgroup of its grid
  bool cut_even;   // fp32: even shares of the last round
  bool seg;          // segment kernel: the shapes the fused kernels do not cover
  bool seg_small;    // ... or small calls of those they do
  SegPlan sp;
  // pack-level call only
  int CO, CO_pad;    // conv_offset channels: 3 (2 when unmodulated) * DG * taps, rounded up to 32
  int mask_kind;     // kMaskLogit, or kMaskNone when unmodulated
  size_t owp_bytes;  // packed conv_offset weights (fused path, conv_offset run here)
  size_t raw_bytes;  // conv_offset output kept in the workspace
};

size_t part_buffers(const Plan &pl) { return align_up((size_t)pl.cut_wgs * (pl.cut_even ? 2 : 1) * kPT * kF2CT * 4); }
size_t cut_region(const Plan &pl) { return part_buffers(pl) + align_up((size_t)pl.cut_wgs * 4); }

// What a pack-level call adds to the plain one.
struct PackExtra {
  const void *offset_weight, *offset_bias;
  void *raw;
};

// 16-bit tensors, 256- or 128-channel tiles, one deformable group, enough K steps: the eight-wave
// kernels (mdcn_fused2.h; mdcn_fused3.h beside it where wide_ok() says so)
bool uses_fused2(const mdcn_params *p, const Geom &g, const Plan &pl) {
  if ((pl.CT != 256 && pl.CT != 128) || g.taps > kTapsSmall || elem_size(p->dtype) != 2 || g.DG != 1 ||
      p->path == MDCN_PATH_FUSED_SPLIT)
    return false;
  const int nk_pad = (pl.slabs * g.taps + kF2Unroll - 1) / kF2Unroll * kF2Unroll;
  return nk_pad >= kF2MinSteps;
}

// ... and the kernel with 256-pixel tiles for whole tiles of such a call: an even
// number of K steps, output planes of whole 16-byte runs (the caller checks the pointer's alignment), groups of
// whole channel tiles
bool wide_ok(const mdcn_params *p, const Geom &g, const Plan &pl) {
  if (!pl.fused || !uses_fused2(p, g, pl) || p->path == MDCN_PATH_FUSED_NARROW)
    return false;
  const int nk = pl.slabs * g.taps;
  const long plane_out = (long)g.Ho * g.Wo;
  return nk >= kF3MinSteps && nk % 2 == 0 && g.taps >= kF3MinTaps && plane_out % 8 == 0 && plane_out >= 64 &&
         g.cout_g % pl.CT == 0 && g.Cout <= kF3MaxBias;
}

// Rounds of the 128-pixel kernel's schedule for `tiles` tiles of nk K steps, in tile times (its last round's
// tiles are cut along K when that is allowed; the sixth part of a tile and the sum of all six take a quarter of its time).
double narrow_rounds(long tiles, int nk, bool may_cut) {
  if (tiles <= 0) return 0.0;
  const int stride = std::max(1, num_cus() / 8);
  const long chunk = (tiles + 7) / 8;
  const long full = chunk / stride, rest = chunk % stride;
  if (rest == 0) return (double)full;
  const long steps6 = (nk + kF2Unroll - 1) / kF2Unroll;
  long parts = 1;
  if (may_cut) parts = std::max<long>(1, std::min<long>(std::min<long>(stride / rest, 4), steps6));
  return (double)full + 1.0 / (double)parts;
}

// How many of a launch's pixel tiles of 256 go to the wide kernel: all of them (`all`), or whole rounds of
// its one-workgroup-per-CU grid when that and the 128-pixel kernel on the rest come out shorter than the
// 128-pixel kernel alone.  wide_cost: time of a 256-pixel tile in units of a 128-pixel one (measured).
// 256 channels, stride 1 (N=16, 100x152): 79.7 us per round of 256-pixel tiles against 46.6 us.
// 128 channels, stride 1 (N=16, 100x168): 29.4 us against 19.4 us.
// Stride 2 (128 channels, 200x336 input): the wide kernel's main stage takes as long as the narrow one's;
// neighbouring pixels share no input rows there and the time goes with the rows the L2 delivers.
inline double wide_tile_cost(int CT, bool unit_stride) { return !unit_stride ? 2.0 : CT == 256 ? 1.71 : 1.52; }
constexpr double kSecondKernelCost = 0.45;  // what launching the 128-pixel kernel behind it costs (ramps, table, tail)
long wide_tiles(long total_px, int n_ctiles_groups, int nk, bool may_cut, bool all, double wide_cost) {
  const long full = total_px / kF3PT;
  if (all || full == 0) return full;
  const long grid = std::max(8, num_cus() / 8 * 8);
  auto cost = [&](long n3) {
    const long wg_tiles = (n3 * n_ctiles_groups + grid - 1) / grid;  // tiles of the busiest workgroup
    const long px2 = total_px - n3 * kF3PT;
    const long tiles2 = (px2 + kPT - 1) / kPT * n_ctiles_groups;
    return wg_tiles * wide_cost + narrow_rounds(tiles2, nk, may_cut) + ((n3 && tiles2) ? kSecondKernelCost : 0.0);
  };
  const long rounds = full * n_ctiles_groups / grid;
  const long whole = rounds * grid / n_ctiles_groups;  // pixel tiles of the whole rounds
  long best = 0;
  double best_cost = cost(0);
  for (long n3 : {whole, full})
    if (n3 > 0 && cost(n3) < best_cost) best = n3, best_cost = cost(n3);
  return best;
}

// ... for a launch of total_px pixels of the call *p
long wide_tiles_of_call(const mdcn_params *p, const Geom &g, const Plan &pl, long total_px, bool out_vec_ok) {
  if (!wide_ok(p, g, pl) || !out_vec_ok) return 0;
  return wide_tiles(total_px, pl.n_ctiles * g.G, pl.slabs * g.taps, pl.cut_bytes != 0, p->path == MDCN_PATH_FUSED_WIDE,
                    wide_tile_cost(pl.CT, g.sh == 1 && g.sw == 1));
}

// The segment kernel for a call the fused kernels do not take, in passes of n_chunk images.  small: one that they do
// take, whose 16-bit samples it rounds as they do.
void plan_segments(const mdcn_params *p, const Geom &g, Plan *pl, bool small = false) {
  pl->seg = false;
  if (p->path == MDCN_PATH_DIRECT || p->dtype == MDCN_F64 || p->input_nhwc) return;
  if ((uint64_t)g.N * g.Ho * g.Wo > 0x7fffffffull || !seg_plan(g, p->dtype, small, 1, false, num_cus(), &pl->sp)) return;
  pl->n_chunk = (int)std::min<uint64_t>((uint64_t)g.N, std::max<uint64_t>(1, g_fwd_pass_bytes.load() / pl->sp.xt_bytes));
  pl->seg = seg_plan(g, p->dtype, small, pl->n_chunk, !p->no_k_split, num_cus(), &pl->sp);
  pl->xt_bytes = align_up(pl->sp.xt_bytes);
  pl->wp_bytes = align_up(pl->sp.wp_bytes);
}

// ... without it: one thread per output element, no workspace of its own
void drop_segments(Plan *pl) {
  pl->seg = false;
  pl->xt_bytes = pl->wp_bytes = 0;
}

// Small calls of few terms, which the fused kernels cover too: there a tile's table, its first gathers and the sum
// of its parts are most of the time, and a wavefront of the segment kernel has none of these.  Up to 18 iterations
// (64 input channels of 3x3) and 64 output channels, until it has three waves per CU before they share K.  Whole
// call, us, fused / segment kernel: fp32 64 -> 64 28x28 24.1 / 18.4, 56x56 26.6 / 19.4, 120x120 37.4 / 29.6, 150x150
// 43.6 / 43.0; 64 -> 256 56x56 37 / 44, 128 -> 64 32.1 / 34.8 (fp32 MFMAs); bf16 64 -> 64 56x56 19.5 / 14.4, 150x150
// 26.2 / 21.5, 200x200 34.1 / 34.5.
// Never with more scratch than the fused kernels ask for.
bool small_call(const mdcn_params *p, const Geom &g, const Plan &fused, Plan *alt) {
  if (p->path != MDCN_PATH_AUTO || p->input_nhwc || !fused.fused) return false;
  *alt = fused;
  alt->fused = false;
  plan_segments(p, g, alt, true);
  if (!alt->seg || alt->n_chunk != g.N || alt->sp.iters > 18 || alt->sp.nb > 2) return false;
  const long waves = ((long)g.N * g.Ho * g.Wo + 31) / 32 * alt->sp.n_ctiles * g.G;
  if (waves > 3L * num_cus() || alt->xt_bytes + alt->wp_bytes > fused.xt_bytes + fused.wp_bytes) return false;
  alt->seg_small = true;
  alt->max_bytes = alt->wexp_bytes = alt->rexp_bytes = alt->tpix_bytes = 0;
  alt->cut_bytes = 0;
  alt->cut_wgs = 0;
  return true;
}

// Products of fp16 pairs or of bf16 triples (mdcn_fused_f32.h): pairs cost a launch in front of the main kernel's, 4 to 5 us, and
// save so much a K step of 256 channels that any schedule makes up for it, less with 128 and little with 64, whose steps the
// gathers bound.  Whole call, us, triples / pairs.  256 channels a tile: 256 channels 50x84 N=2 (24 steps a workgroup) 94.9 / 69.3, 512 channels
// 25x42 N=4 162.7 / 118.1; 128: 128 channels 64x64 N=2 (9) 36.7 / 35.8, 256 channels 50x84 (24) 55.5 / 50.5; 64: 256 channels 28x28
// (8) 31.1 / 34.3, 64 channels 200x200 (22) 51.5 / 54.9, N=8 (176) 256 / 254.
bool pairs_pay(const mdcn_params *p, const Geom &g, const Plan &pl) {
  const int nk = pl.slabs * g.taps;
  const long px_tiles = ((long)pl.n_chunk * g.Ho * g.Wo + kPT - 1) / kPT;
  const double steps = schedule_rounds(px_tiles * pl.n_ctiles * g.G, nk, !p->no_k_split) * nk;
  return steps >= (pl.CT == 256 ? 4 : pl.CT == 128 ? 9 : 140);
}

int make_plan(const mdcn_params *p, const Geom &g, Plan *pl, bool may_be_small = true) {
  const bool ok = fused_ok(p, g);
  if (forced_fused(p->path) && !ok) return MDCN_ERR_PATH;
  if (p->input_nhwc && (!ok || p->path == MDCN_PATH_DIRECT || p->path == MDCN_PATH_SEGMENT)) return MDCN_ERR_PATH;  // in-place reads: fused kernel only
  pl->fused = ok && p->path != MDCN_PATH_DIRECT && p->path != MDCN_PATH_SEGMENT;
  pl->seg = pl->seg_small = false;
  pl->CT = pl->KC = pl->n_ctiles = pl->slabs = pl->n_chunk = 0;
  pl->xt_bytes = pl->wp_bytes = pl->owp_bytes = pl->raw_bytes = pl->cut_bytes = pl->max_bytes = pl->wexp_bytes = pl->rexp_bytes = pl->tpix_bytes = 0;
  pl->cut_wgs = 0;
  pl->cut_even = false;
  pl->CO = 3 * g.DG * g.taps;
  pl->CO_pad = (pl->CO + 31) / 32 * 32;
  pl->mask_kind = kMaskLogit;
  if (!pl->fused) {
    plan_segments(p, g, pl);
    return MDCN_OK;
  }
  const size_t es = elem_size(p->dtype);
  pl->KC = slab_channels(p->dtype);
  pl->CT = pick_ct(g.cout_g, g.taps);
  pl->slabs = g.cin_g / pl->KC;
  const uint64_t img = (uint64_t)g.Hp * g.Wp * g.Cin * es;
  pl->n_chunk = (int)std::min<uint64_t>((uint64_t)g.N, std::max<uint64_t>(1, g_fwd_pass_bytes.load() / img));
  if (p->dtype == MDCN_F32 && pl->CT == 256) {
    // What counts is how evenly the tiles fill the workgroups, and a tile's time, which goes with its width: a K step of 128 channels takes
    // 0.72 of one of 256 (1 910 and 2 650 clocks); where all tiles are cut what parts cost each other goes with the width too (N=1 256
    // channels 50x84: 33 tiles of 256 channels in six parts 61.2 us a call, 66 of 128 in three 50.5).
    const long px_tiles = ((long)pl->n_chunk * g.Ho * g.Wo + kPT - 1) / kPT;
    const int nk = pl->slabs * g.taps;
    auto cost = [&](int ct) {
      const long tiles = px_tiles * ((g.cout_g + ct - 1) / ct) * g.G;
      const double rounds = schedule_rounds(tiles, nk, !p->no_k_split);
      return rounds * (ct == 256 ? 1.0 : rounds < 1.0 ? 0.56 : 0.72);
    };
    if (cost(128) < 0.95 * cost(256)) pl->CT = 128;
  }
  // Few tiles: narrower ones, so that more workgroups have a part of one and its sum is shorter.  16 bits: the narrowest
  // that still leaves two workgroups a tile (eight-wave kernel: 128 channels at least).  fp32, whose waves
  // split the samples again for every tile of channels: 64, where that leaves four.  Whole call, us, wide / narrow:
  // bf16 256 channels 14x14 30 / 23 (128), 90x90 37.4 / 34.0, 100x100 (a workgroup a tile) 38.2 / 42.2; 512 channels 25x42 41 / 34;
  // 4 deformable groups, 256 channels 28x28 N=2 50 / 29 (64), 512 channels 25x42 76 / 50, N=2 79 / 70 (128) / 90 (64);
  // fp32 256 channels 14x14 42 / 36, 28x28 48 / 43, 512 channels 25x42 (three a tile) 84 / 89.
  if (!p->no_k_split) {
    const long px_tiles = ((long)pl->n_chunk * g.Ho * g.Wo + kPT - 1) / kPT;
    const bool f32 = p->dtype == MDCN_F32;
    for (int ct : {64, 128}) {
      const long tiles = px_tiles * ((g.cout_g + ct - 1) / ct) * g.G;
      if (ct < pl->CT && (ct == 64 ? f32 || !uses_fused2(p, g, *pl) : !f32) && tiles * (f32 ? 4 : 2) <= num_cus()) {
        pl->CT = ct;
        break;
      }
    }
  }
  pl->n_ctiles = (g.cout_g + pl->CT - 1) / pl->CT;
  pl->xt_bytes = p->input_nhwc ? 0 : align_up((size_t)img * pl->n_chunk);
  // (fp32: three bf16 planes, 6 bytes an element)
  pl->wp_bytes = align_up((size_t)g.G * pl->n_ctiles * pl->slabs * g.taps * pl->CT * pl->KC * (es == 4 ? 6 : es));
  if (p->dtype == MDCN_F32 && !p->input_nhwc && pairs_pay(p, g, *pl)) {
    pl->max_bytes = align_up((size_t)pl->n_chunk * g.H * g.W * (g.Cin / pl->KC) * 2);
    pl->wexp_bytes = align_up((size_t)g.G * pl->n_ctiles * pl->CT * 4);
    pl->rexp_bytes = align_up((size_t)g.G * pl->n_chunk * g.Ho * g.Wo * 4);
    pl->tpix_bytes = align_up((size_t)g.DG * g.taps * pl->n_chunk * g.Ho * g.Wo * 4);
  }
  // Tiles of the 128-pixel kernels' last round are cut along K where workgroups would otherwise idle: one
  // 128 x 256 fp32 tile and a counter per workgroup of the persistent grid -- asked for only when a launch
  // of this call has such a round (the 256-pixel kernel never cuts; what it leaves to the 128-pixel one may)
  if (!p->no_k_split) {
    const int stride = std::max(1, num_cus() / 8);
    auto may_cut = [&](long tiles) {  // an XCD's run of tiles ends in a round that fills at most half of its workgroups
      if (tiles <= 0) return false;
      const long chunk = (tiles + 7) / 8;
      for (long run : {chunk, tiles - 7 * chunk}) {
        const long rest = run > 0 ? run % stride : 0;
        if (rest > 0 && stride / rest >= 2) return true;
      }
      return false;
    };
    const long plane_out = (long)g.Ho * g.Wo;
    bool cuts = false;
    for (int n0 = 0; n0 < g.N && !cuts; n0 += pl->n_chunk) {
      const long total_px = (long)std::min(pl->n_chunk, g.N - n0) * plane_out;
      long px = total_px;
      if (wide_ok(p, g, *pl)) {
        // (the split itself looks at whether cutting is allowed: take the answer for "allowed")
        pl->cut_bytes = 1;
        px -= wide_tiles_of_call(p, g, *pl, total_px, plane_out % 8 == 0) * kF3PT;
        pl->cut_bytes = 0;
      }
      cuts = may_cut((px + kPT - 1) / kPT * pl->n_ctiles * g.G);
    }
    if (p->dtype == MDCN_F32) {   // (by the first pass's schedule, which all have but the last)
      const long tiles = ((long)pl->n_chunk * plane_out + kPT - 1) / kPT * pl->n_ctiles * g.G;
      (void)schedule_rounds(tiles, pl->slabs * g.taps, true, &pl->cut_even);
      cuts = cuts || pl->cut_even;
    }
    if (cuts) {
      pl->cut_wgs = num_cus() / 8 * 8;
      pl->cut_bytes = cut_region(*pl);
    }
  }
  if (p->path == MDCN_PATH_FUSED_WIDE && !wide_ok(p, g, *pl)) return MDCN_ERR_PATH;
  Plan alt;
  if (may_be_small && small_call(p, g, *pl, &alt)) *pl = alt;
  return MDCN_OK;
}

// Workspace of a pack-level call: [xt][wp][owp][raw] on the fused path, [raw] on
// the direct one (nothing when the caller's own raw buffer serves).
int make_pack_plan(const mdcn_pack_params *pp, const Geom &g, Plan *pl) {
  const mdcn_params *p = &pp->conv;
  if (p->input_nhwc) return MDCN_ERR_PATH;
  const int rc = make_plan(p, g, pl, false);
  if (rc != MDCN_OK) return rc;
  if (pp->unmodulated) {
    pl->CO = 2 * g.DG * g.taps;
    pl->CO_pad = (pl->CO + 31) / 32 * 32;
    pl->mask_kind = kMaskNone;
  }
  const size_t es = elem_size(p->dtype);
  const size_t plane = (size_t)g.Ho * g.Wo;
  if (pp->offset_weight) {
    if (pl->fused) {
      if (pl->CO_pad > 128) {  // accumulator blocks of the conv_offset kernel
        if (forced_fused(p->path)) return MDCN_ERR_PATH;
        pl->fused = false;
        pl->xt_bytes = pl->wp_bytes = pl->cut_bytes = pl->max_bytes = pl->wexp_bytes = pl->rexp_bytes = pl->tpix_bytes = 0;
        pl->cut_wgs = 0;
        plan_segments(p, g, pl);
      } else {
        pl->owp_bytes = align_up((size_t)(g.Cin / pl->KC) * g.taps * 4 * (pl->CO_pad / 32) * 64 * 16);
        pl->raw_bytes = align_up((size_t)pl->n_chunk * plane * pl->CO_pad * es);
      }
    }
    if (!pl->fused && !pp->raw) pl->raw_bytes = align_up((size_t)g.N * pl->CO * plane * es);
  }
  return MDCN_OK;
}

template <typename E, int CT, int TMAX, bool MULTI_DG>
hipError_t launch_fused_ct(const FusedArgs &fa, bool unbordered, hipStream_t st) {
  // persistent workgroups: one per CU, a multiple of the 8 XCDs
  // (with tiles cut along K, workgroups beyond the tile count take parts of tiles: the whole chip)
  const int total_wg = fa.n_ptiles * fa.n_ctiles * fa.g.G;
  const int per_xcd = fa.cut_max > 1 ? std::max(1, num_cus() / 8)
                                       : std::max(1, std::min((total_wg + 7) / 8, num_cus() / 8));
  const dim3 grid(per_xcd * 8), block(kThreads);
  if constexpr (sizeof(E) == 4) {
    if (unbordered)
      hipLaunchKernelGGL((fused_f32_kernel<CT, TMAX, MULTI_DG, true, 3>), grid, block, 0, st, fa);
    else if (fa.row_exp)
      hipLaunchKernelGGL((fused_f32_kernel<CT, TMAX, MULTI_DG, false, 2>), grid, block, 0, st, fa);
    else
      hipLaunchKernelGGL((fused_f32_kernel<CT, TMAX, MULTI_DG, false, 3>), grid, block, 0, st, fa);
  } else {
    if (unbordered)
      hipLaunchKernelGGL((fused_kernel<E, CT, TMAX, MULTI_DG, true>), grid, block, 0, st, fa);
    else
      hipLaunchKernelGGL((fused_kernel<E, CT, TMAX, MULTI_DG, false>), grid, block, 0, st, fa);
  }
  return hipGetLastError();
}

// 16-bit tensors, 256- and 128-channel tiles: the eight-wave kernel of mdcn_fused2.h
template <typename E, int CT>
hipError_t launch_fused2(const FusedArgs &fa, bool unbordered, hipStream_t st) {
  const int total_wg = fa.n_ptiles * fa.n_ctiles * fa.g.G;
  const int per_xcd = fa.cut_max > 1 ? std::max(1, num_cus() / 8)
                                       : std::max(1, std::min((total_wg + 7) / 8, num_cus() / 8));
  if (unbordered)
    hipLaunchKernelGGL((fused2_kernel<E, CT, true>), dim3(per_xcd * 8), dim3(kF2Threads), 0, st, fa);
  else
    hipLaunchKernelGGL((fused2_kernel<E, CT, false>), dim3(per_xcd * 8), dim3(kF2Threads), 0, st, fa);
  return hipGetLastError();
}

// 16-bit tensors, 256- or 128-channel tiles, whole tiles of 256 pixels: mdcn_fused3.h
template <typename E>
hipError_t launch_fused3(const FusedArgs &fa, int CT, bool nhwc, hipStream_t st) {
  const int total_wg = fa.n_ptiles * fa.n_ctiles * fa.g.G;
  const int per_xcd = std::max(1, std::min((total_wg + 7) / 8, num_cus() / 8));
  const dim3 grid(per_xcd * 8), block(kF3Threads);
  if (CT == 256) {
    if (nhwc)
      hipLaunchKernelGGL((fused3_kernel<E, 256, true>), grid, block, 0, st, fa);
    else
      hipLaunchKernelGGL((fused3_kernel<E, 256, false>), grid, block, 0, st, fa);
  } else {
    if (nhwc)
      hipLaunchKernelGGL((fused3_kernel<E, 128, true>), grid, block, 0, st, fa);
    else
      hipLaunchKernelGGL((fused3_kernel<E, 128, false>), grid, block, 0, st, fa);
  }
  return hipGetLastError();
}

template <typename E, int CT>
hipError_t launch_fused_tm(const FusedArgs &fa, bool ub, bool eight_wave, hipStream_t st) {
  const bool small = fa.g.taps <= kTapsSmall;
  if constexpr (sizeof(E) == 2 && (CT == 256 || CT == 128)) {
    if (eight_wave) return launch_fused2<E, CT>(fa, ub, st);
  }
  if constexpr (CT == 256) {  // (pick_ct never pairs the 256-wide tile with the large table)
    return fa.g.DG > 1 ? launch_fused_ct<E, CT, kTapsSmall, true>(fa, ub, st)
                       : launch_fused_ct<E, CT, kTapsSmall, false>(fa, ub, st);
  } else {
    if (fa.g.DG > 1)
      return small ? launch_fused_ct<E, CT, kTapsSmall, true>(fa, ub, st)
                   : launch_fused_ct<E, CT, kTapsLarge, true>(fa, ub, st);
    return small ? launch_fused_ct<E, CT, kTapsSmall, false>(fa, ub, st)
                 : launch_fused_ct<E, CT, kTapsLarge, false>(fa, ub, st);
  }
}

template <typename E>
hipError_t launch_fused(const FusedArgs &fa, int CT, bool ub, bool eight_wave, hipStream_t st) {
  switch (CT) {
    case 64: return launch_fused_tm<E, 64>(fa, ub, eight_wave, st);
    case 128: return launch_fused_tm<E, 128>(fa, ub, eight_wave, st);
    default: return launch_fused_tm<E, 256>(fa, ub, eight_wave, st);
  }
}

template <typename E>
int run_typed(const mdcn_params *p, const Geom &g, const Plan &pl, hipStream_t st,
              float *ms, const PackExtra *px) {
  hipEvent_t ev[2] = {nullptr, nullptr};
  auto tic = [&]() { if (ms) (void)hipEventRecord(ev[0], st); };
  auto toc = [&](int slot) {
    if (!ms) return;
    (void)hipEventRecord(ev[1], st);
    (void)hipEventSynchronize(ev[1]);
    float t = 0.f;
    (void)hipEventElapsedTime(&t, ev[0], ev[1]);
    ms[slot] += t;
  };
  if (ms) {
    ms[0] = ms[1] = ms[2] = ms[3] = 0.f;
    if (px) ms[4] = 0.f;
    if (hipEventCreate(&ev[0]) != hipSuccess || hipEventCreate(&ev[1]) != hipSuccess)
      return MDCN_ERR_LAUNCH;
  }
  int rc = MDCN_OK;
  const size_t es = sizeof(E);
  const long plane_out = (long)g.Ho * g.Wo;

  // the conv_offset output of a pack-level call as dense (N, CO, Ho, Wo)
  auto nchw_raw_view = [&](const E *raw) {
    OffMaskView v;
    v.off = raw;
    v.msk = raw + (long)2 * g.DG * g.taps * plane_out;
    v.off_n = v.msk_n = (long)pl.CO * plane_out;
    v.off_ch = v.msk_ch = plane_out;
    v.off_px = v.msk_px = 1;
    v.logit = pl.mask_kind;
    if (pl.mask_kind == kMaskNone) v.msk = raw;
    return v;
  };

  if (!pl.fused) {
    OffMaskView om = dense_view(p->offset, p->mask, g);
    if (px) {
      E *raw = (E *)px->raw;
      if (px->offset_weight) {
        if (!raw) raw = (E *)((unsigned char *)p->workspace + pl.xt_bytes + pl.wp_bytes);
        const long total = (long)g.N * pl.CO * plane_out;
        const int grid = (int)std::min<long>((total + 255) / 256, 1L << 20);
        tic();
        hipLaunchKernelGGL(oconv_direct_kernel<E>, dim3(grid), dim3(256), 0, st, g,
                           (const E *)p->input, (const E *)px->offset_weight,
                           (const E *)px->offset_bias, raw, pl.CO, total);
        if (hipGetLastError() != hipSuccess) rc = MDCN_ERR_LAUNCH;
        toc(4);
      }
      om = nchw_raw_view(raw);
    }
    if (pl.seg) {
      SegArgs sa;
      sa.s = pl.sp;
      sa.xt = p->workspace;
      sa.wp = (unsigned char *)p->workspace + pl.xt_bytes;
      sa.bias = p->bias;
      sa.row_bytes = (uint32_t)g.Wp * 16u;
      sa.plane_bytes = (uint32_t)g.Hp * sa.row_bytes;
      sa.img_bytes = (uint32_t)(g.G * pl.sp.nseg_g * pl.sp.cps) * sa.plane_bytes;
      for (int n0 = 0; n0 < g.N && rc == MDCN_OK; n0 += pl.n_chunk) {
        sa.g = g;
        sa.g.N = std::min(pl.n_chunk, g.N - n0);
        sa.om = om;
        sa.om.off = (const E *)om.off + (long)n0 * om.off_n;
        sa.om.msk = (const E *)om.msk + (long)n0 * om.msk_n;
        sa.out = (E *)p->output + (size_t)n0 * g.Cout * plane_out;
        sa.total_px = (long)sa.g.N * plane_out;
        const long tile_px = 32 * (4 / pl.sp.kshare);
        sa.n_work = (sa.total_px + tile_px - 1) / tile_px * pl.sp.n_ctiles * g.G;
        tic();
        sa.in = (const E *)p->input + (size_t)n0 * g.Cin * g.H * g.W;
        sa.weight = p->weight;
        if (seg_prepass(p->dtype, sa, n0 == 0, st) != hipSuccess)
          rc = MDCN_ERR_LAUNCH;
        toc(0);
        tic();
        if (rc == MDCN_OK && seg_forward(p->dtype, sa, st) != hipSuccess) rc = MDCN_ERR_LAUNCH;
        toc(2);
      }
    } else {
    const long total = (long)g.N * g.Cout * plane_out;
    const int grid = (int)std::min<long>((total + 255) / 256, 1L << 20);
    tic();
    hipLaunchKernelGGL(direct_kernel<E>, dim3(grid), dim3(256), 0, st, g,
                       (const E *)p->input, om, (const E *)p->weight,
                       (const E *)p->bias, (E *)p->output, total);
    if (hipGetLastError() != hipSuccess) rc = MDCN_ERR_LAUNCH;
    toc(2);
    }
  } else {
    unsigned char *ws = (unsigned char *)p->workspace;
    E *xt = (E *)ws;
    E *wp = (E *)(ws + pl.xt_bytes);
    E *owp = (E *)(ws + pl.xt_bytes + pl.wp_bytes);
    E *raw_pm = (E *)(ws + pl.xt_bytes + pl.wp_bytes + pl.owp_bytes);
    const bool own_oconv = px && px->offset_weight;
    const int cof = pl.CO_pad / 32;
    unsigned char *opt = ws + pl.xt_bytes + pl.wp_bytes + pl.owp_bytes + pl.raw_bytes;
    const bool pairs = pl.max_bytes != 0;
    PairArgs pa{};
    pa.w = (const float *)p->weight;
    pa.wp = wp;
    pa.row_max = (uint16_t *)opt;
    pa.wexp = (int *)(opt + pl.max_bytes);
    pa.row_exp = (int *)(opt + pl.max_bytes + pl.wexp_bytes);
    pa.tab_pix = (uint32_t *)((unsigned char *)pa.row_exp + pl.rexp_bytes);
    pa.tab_w = (float4 *)((unsigned char *)pa.tab_pix + pl.tpix_bytes);
    pa.unit = std::max(1, std::gcd(g.cin_g, g.ch_per_dg) / pl.KC);
    pa.CT = pl.CT;
    pa.n_ctiles = pl.n_ctiles;
    pa.slabs = pl.slabs;
    pa.slabs_total = g.Cin / pl.KC;
    float *cut_part = (float *)(opt + pl.pair_bytes());
    uint32_t *cut_cnt = (uint32_t *)((unsigned char *)cut_part + part_buffers(pl));
    if (!pl.cut_bytes) cut_part = nullptr, cut_cnt = nullptr;

    // weights: once per call -- inside the launch that re-lays the first batch chunk; on their own when
    // there is no such launch (channels-last input read in place)
    constexpr int EPV = 16 / (int)sizeof(E);
    const bool vec_relayout = !p->input_nhwc;
    const long wtotal = (long)g.G * pl.n_ctiles * pl.slabs * g.taps * pl.CT * pl.KC;
    bool packed = false;
    {
      tic();
      if (!vec_relayout) {
        const int grid = (int)std::min<long>((wtotal + 255) / 256, 1L << 16);
        hipLaunchKernelGGL(pack_weight_kernel<E>, dim3(grid), dim3(256), 0, st, g,
                           (const E *)p->weight, wp, pl.CT, pl.KC, pl.n_ctiles,
                           pl.slabs, wtotal, cut_cnt, pl.cut_wgs);
        if (hipGetLastError() != hipSuccess) rc = MDCN_ERR_LAUNCH;
        packed = true;
      }
      toc(1);
    }
    for (int n0 = 0; n0 < g.N && rc == MDCN_OK; n0 += pl.n_chunk) {
      Geom gc = g;
      gc.N = std::min(pl.n_chunk, g.N - n0);
      const E *in = (const E *)p->input + (size_t)n0 * g.Cin * g.H * g.W;
      const bool nhwc = p->input_nhwc != 0;
      if (!nhwc && vec_relayout) {
        const int n_pchunks = (gc.H * gc.W + 32 * EPV - 1) / (32 * EPV);
        const long blocks = (long)gc.N * (gc.Cin / pl.KC) * n_pchunks;
        tic();
        OffsetPack op = {nullptr, nullptr, 0, 1, 0, 0};
        if (!packed && own_oconv) {
          const long chunks = (long)(g.Cin / pl.KC) * g.taps * 4 * cof * 64;
          op = OffsetPack{px->offset_weight, owp, pl.CO, cof, chunks, (int)std::min<long>((chunks + 255) / 256, 512)};
        }
        if constexpr (sizeof(E) == 4) {
          if (pairs) {
            pa.g = gc;
            pa.zero_ptr = cut_cnt;
            pa.zero_n = packed ? 0 : pl.cut_wgs;
            const int wmax_blocks = packed ? 0 : pair_col_groups(g, pl.n_ctiles, pl.CT);
            hipLaunchKernelGGL(pair_relayout_kernel, dim3((unsigned)(blocks + wmax_blocks + op.blocks)), dim3(256), 0, st, pa,
                               in, xt, n_pchunks, wmax_blocks, op);
          }
        }
        if (pairs) {
        } else if (!packed) {
          const int pack_blocks = (int)std::max<long>(1, std::min<long>(wtotal / (256 * 8), 512));
          hipLaunchKernelGGL(prepass_kernel<E>, dim3((unsigned)(blocks + pack_blocks + op.blocks)), dim3(256), 0, st, gc,
                             in, xt, n_pchunks, g, (const E *)p->weight, wp, pl.CT, pl.KC, pl.n_ctiles, pl.slabs, wtotal,
                             pack_blocks, cut_cnt, pl.cut_wgs, op);
          packed = true;
        } else {
          hipLaunchKernelGGL((relayout_vec_kernel<E, true>), dim3((unsigned)blocks), dim3(256), 0, st, gc, in, xt,
                             n_pchunks);
        }
        if (hipGetLastError() != hipSuccess) rc = MDCN_ERR_LAUNCH;
        toc(0);
      }
      FusedArgs fa;
      fa.g = gc;
      fa.xt = nhwc ? (const void *)in : (const void *)xt;
      fa.wp = wp;
      fa.in = in;
      fa.row_exp = pairs ? pa.row_exp : nullptr;
      fa.wexp = pa.wexp;
      fa.tab_pix = pa.tab_pix;
      fa.tab_w = pa.tab_w;
      fa.weight = p->weight;
      fa.in_c = nhwc ? 1 : (long)g.H * g.W;
      fa.in_px = nhwc ? g.Cin : 1;
      if (nhwc) {
        fa.px_bytes = (uint32_t)(g.Cin * es);
        fa.row_bytes = (uint32_t)g.W * fa.px_bytes;
        fa.slab_bytes = (uint32_t)kRowB;
        fa.img_bytes = (uint32_t)g.H * fa.row_bytes;
      } else {
        fa.px_bytes = (uint32_t)kRowB;
        fa.row_bytes = (uint32_t)g.Wp * (uint32_t)kRowB;
        fa.slab_bytes = (uint32_t)(g.Hp * g.Wp) * (uint32_t)kRowB;
        fa.img_bytes = (uint32_t)(g.Cin / pl.KC) * fa.slab_bytes;
      }
      if (own_oconv) {
        OconvArgs oa;
        oa.g = gc;
        oa.xt = xt;
        oa.owp = owp;
        oa.obias = px->offset_bias;
        oa.raw = raw_pm;
        oa.total_px = (long)gc.N * plane_out;
        oa.CO = pl.CO;
        oa.CO_pad = pl.CO_pad;
        oa.slabs_total = g.Cin / pl.KC;
        oa.plane_px = g.Hp * g.Wp;
        tic();
        const hipError_t e = oconv_forward(p->dtype, oa, st);
        if (e != hipSuccess) rc = MDCN_ERR_LAUNCH;
        if (px->raw) {
          const long total = (long)gc.N * pl.CO * plane_out;
          const int grid = (int)std::min<long>((total + 255) / 256, 1L << 20);
          hipLaunchKernelGGL(raw_to_nchw_kernel<E>, dim3(grid), dim3(256), 0, st, raw_pm,
                             (E *)px->raw + (size_t)n0 * pl.CO * plane_out, pl.CO, pl.CO_pad,
                             plane_out, total);
          if (hipGetLastError() != hipSuccess) rc = MDCN_ERR_LAUNCH;
        }
        toc(4);
        // pixel-major: the values of one pixel are CO_pad consecutive elements
        fa.om.off = raw_pm;
        fa.om.msk = raw_pm + 2 * g.DG * g.taps;
        fa.om.off_n = fa.om.msk_n = plane_out * pl.CO_pad;
        fa.om.off_ch = fa.om.msk_ch = 1;
        fa.om.off_px = fa.om.msk_px = pl.CO_pad;
        fa.om.logit = pl.mask_kind;
        if (pl.mask_kind == kMaskNone) fa.om.msk = raw_pm;
      } else if (px) {
        fa.om = nchw_raw_view((const E *)px->raw + (size_t)n0 * pl.CO * plane_out);
      } else {
        fa.om = dense_view((const E *)p->offset + (size_t)n0 * g.DG * 2 * g.taps * plane_out,
                           p->mask ? (const E *)p->mask + (size_t)n0 * g.DG * g.taps * plane_out : nullptr, g);
      }
      fa.cut_max = !pl.cut_bytes ? 0 : sizeof(E) == 4 ? kF32CutMax : uses_fused2(p, g, pl) ? kF2CutMax : kCutMax;
      fa.cut_even = pl.cut_even;
      fa.cut_part = cut_part;
      fa.cut_cnt = cut_cnt;
      fa.bias = p->bias;
      fa.out = (E *)p->output + (size_t)n0 * g.Cout * plane_out;
      fa.total_px = (long)gc.N * plane_out;
      fa.n_ptiles = (int)((fa.total_px + kPT - 1) / kPT);
      fa.n_ctiles = pl.n_ctiles;
      fa.slabs = pl.slabs;
      fa.slabs_total = g.Cin / pl.KC;
      fa.plane_px = g.Hp * g.Wp;
      fa.out_vec_ok = (plane_out % (long)(16 / es) == 0) && (((uintptr_t)fa.out % 16) == 0);
      fa.px0 = 0;
      if constexpr (sizeof(E) == 4) {
        if (pairs && rc == MDCN_OK) {
          tic();
          pa.g = gc;
          pa.om = fa.om;
          pa.img_bytes = fa.img_bytes;
          pa.row_bytes = fa.row_bytes;
          const int pack_blocks = packed ? 0 : pair_col_groups(g, pl.n_ctiles, pl.CT) * pl.slabs;
          const int sample_blocks = g.G * (int)((fa.total_px + 63) / 64);
          hipLaunchKernelGGL(pair_exponent_kernel, dim3((unsigned)(sample_blocks + pack_blocks)), dim3(256), 0, st, pa, sample_blocks);
          packed = true;
          if (hipGetLastError() != hipSuccess) rc = MDCN_ERR_LAUNCH;
          toc(0);
        }
      }
      tic();
      const bool eight_wave = uses_fused2(p, g, pl);
      bool rest = true;
      if constexpr (sizeof(E) == 2) {
        {
          // whole tiles of 256 pixels to the wide kernel, what is left to the 128-pixel one
          const long n3 = wide_tiles_of_call(p, g, pl, fa.total_px, fa.out_vec_ok != 0);
          if (n3 > 0) {
            FusedArgs fw = fa;
            fw.n_ptiles = (int)n3;
            if (launch_fused3<E>(fw, pl.CT, nhwc, st) != hipSuccess) rc = MDCN_ERR_LAUNCH;
            fa.px0 = (int)(n3 * kF3PT);
            fa.n_ptiles = (int)((fa.total_px - fa.px0 + kPT - 1) / kPT);
            rest = fa.n_ptiles > 0;
          }
        }
      }
      if (rest && launch_fused<E>(fa, pl.CT, nhwc, eight_wave, st) != hipSuccess) rc = MDCN_ERR_LAUNCH;
      toc(2);
    }
  }
  if (ms) {
    ms[3] = ms[0] + ms[1] + ms[2] + (px ? ms[4] : 0.f);
    (void)hipEventDestroy(ev[0]);
    (void)hipEventDestroy(ev[1]);
  }
  return rc;
}

// Double precision: one kernel, no workspace.
int run_f64(const mdcn_params *p, const Geom &g, hipStream_t st, float *ms) {
  hipEvent_t ev[2] = {nullptr, nullptr};
  if (ms) {
    ms[0] = ms[1] = ms[2] = ms[3] = 0.f;
    if (hipEventCreate(&ev[0]) != hipSuccess || hipEventCreate(&ev[1]) != hipSuccess) return MDCN_ERR_LAUNCH;
    (void)hipEventRecord(ev[0], st);
  }
  const long total = (long)g.N * g.Cout * g.Ho * g.Wo;
  const int grid = (int)std::min<long>((total + 255) / 256, 1L << 20);
  hipLaunchKernelGGL(f64_forward_kernel, dim3(grid), dim3(256), 0, st, g, (const double *)p->input,
                     (const double *)p->offset, (const double *)p->mask, (const double *)p->weight,
                     (const double *)p->bias, (double *)p->output, total);
  const int rc = hipGetLastError() == hipSuccess ? MDCN_OK : MDCN_ERR_LAUNCH;
  if (ms) {
    (void)hipEventRecord(ev[1], st);
    (void)hipEventSynchronize(ev[1]);
    (void)hipEventElapsedTime(&ms[2], ev[0], ev[1]);
    ms[3] = ms[2];
    (void)hipEventDestroy(ev[0]);
    (void)hipEventDestroy(ev[1]);
  }
  return rc;
}

int run(const mdcn_params *p, void *stream, float *ms, const mdcn_pack_params *pp = nullptr) {
  Geom g;
  int rc = check_params(p, &g, true, pp == nullptr);
  if (rc != MDCN_OK) return rc;
  Plan pl;
  PackExtra px_store, *px = nullptr;
  if (pp) {
    if (!pp->offset_weight && !pp->raw) return MDCN_ERR_NULL;
    rc = make_pack_plan(pp, g, &pl);
    px_store.offset_weight = pp->offset_weight;
    px_store.offset_bias = pp->offset_bias;
    px_store.raw = pp->raw;
    px = &px_store;
  } else {
    rc = make_plan(p, g, &pl);
  }
  if (rc != MDCN_OK) return rc;
  if (p->dtype == MDCN_F64) {
    if (pp) return MDCN_ERR_DTYPE;  // the pack-level call has no double-precision form
    return run_f64(p, g, (hipStream_t)stream, ms);
  }
  // (the split-tile buffers come last and are optional: a workspace without them runs unsplit)
  // a call whose workspace does not hold the segment kernel's copies runs without that kernel, as it may
  if (pl.seg && !pl.seg_small && (p->workspace_bytes < pl.xt_bytes + pl.wp_bytes + pl.raw_bytes || !p->workspace ||
                 ((uintptr_t)p->workspace % kAlign) != 0))
    drop_segments(&pl);
  const size_t need = pl.xt_bytes + pl.wp_bytes + pl.owp_bytes + pl.raw_bytes;
  if (need > 0 && (!p->workspace || p->workspace_bytes < need ||
                   ((uintptr_t)p->workspace % kAlign) != 0))
    return MDCN_ERR_WORKSPACE;
  if (p->workspace_bytes < need + pl.pair_bytes()) pl.max_bytes = pl.wexp_bytes = pl.rexp_bytes = pl.tpix_bytes = 0;
  if (pl.cut_even && p->workspace_bytes < need + pl.pair_bytes() + pl.cut_bytes) {  // equal parts have half of the buffers
    pl.cut_even = false;
    pl.cut_bytes = cut_region(pl);
  }
  if (p->workspace_bytes < need + pl.pair_bytes() + pl.cut_bytes) pl.cut_bytes = 0, pl.cut_wgs = 0;
  hipStream_t st = (hipStream_t)stream;
  switch (p->dtype) {
    case MDCN_F32: return run_typed<float>(p, g, pl, st, ms, px);
    case MDCN_F16: return run_typed<f16_t>(p, g, pl, st, ms, px);
    default: return run_typed<bf16_t>(p, g, pl, st, ms, px);
  }
}

template <typename E>
int split_raw(const mdcn_pack_params *pp, const Geom &g, E *offset, E *mask, hipStream_t st) {
  const long plane = (long)g.Ho * g.Wo * g.DG * g.taps, total = 3 * plane * g.N, per = 256 * (16 / (long)sizeof(E));
  hipLaunchKernelGGL(raw_split_kernel<E>, dim3((unsigned)((total + per - 1) / per)), dim3(256), 0, st, (const E *)pp->raw, offset,
                     mask, 2 * plane, plane, total);
  return hipGetLastError() == hipSuccess ? MDCN_OK : MDCN_ERR_LAUNCH;
}

// Workspace: the convolution's, then conv_offset's, which reads the copy of the input the former leaves, then (optional) the maxima.
bool plan_pack_backward(const mdcn_pack_bwd_params *pb, const Geom &g, BwdPlan *pl, OconvBwdPlan *ol) {
  make_bwd_plan(&pb->bwd, g, g_bwd_pass_bytes.load(), pl);
  return oconv_bwd_plan(g, pb->bwd.conv.dtype, pb->unmodulated != 0, pb->through_input != 0,
                        pb->grad_offset_weight || pb->grad_offset_bias, !pl->plain_copy(), num_cus(), ol);
}

int check_bwd(const mdcn_bwd_params *bp, Geom *g, bool need_ptrs) {
  if (!bp) return MDCN_ERR_NULL;
  const mdcn_params *p = &bp->conv;
  int rc = check_params(p, g, false);
  if (rc != MDCN_OK) return rc;
  if (p->input_nhwc) return MDCN_ERR_PATH;
  if (!need_ptrs) return MDCN_OK;
  if (!p->input || !p->offset || !p->weight || !bp->grad_output) return MDCN_ERR_NULL;
  // grad_input and the offset/mask gradients come out of one kernel
  const bool data = bp->grad_input != nullptr;
  if (data != (bp->grad_offset != nullptr)) return MDCN_ERR_NULL;
  if (p->mask ? (data != (bp->grad_mask != nullptr)) : (bp->grad_mask != nullptr)) return MDCN_ERR_NULL;
  if ((uint64_t)g->N * g->DG * g->taps > 0x7fffffffull) return MDCN_ERR_TOO_LARGE;
  if (p->dtype == MDCN_F64 && forced_fused(p->path)) return MDCN_ERR_PATH;
  if (forced_fused(p->path)) {  // asked for the tiled kernels: the shape must allow them
    BwdPlan pl;
    make_bwd_plan(bp, *g, g_bwd_pass_bytes.load(), &pl);
    if ((data && !pl.tiled && !pl.gemm) || (!data && bp->grad_weight && !pl.wgemm)) return MDCN_ERR_PATH;
  }
  return MDCN_OK;
}

}  // namespace

extern "C" {

int mdcn_abi_version(void) { return MDCN_ABI_VERSION; }

void mdcn_set_pass_limits(uint64_t forward_bytes, uint64_t backward_bytes) {
  g_fwd_pass_bytes.store(forward_bytes ? std::min<uint64_t>(forward_bytes, kMaxXtBytes) : kMaxXtBytes);
  g_bwd_pass_bytes.store(backward_bytes ? std::min<uint64_t>(backward_bytes, kBwdColGradCap) : kBwdColGradCap);
}

const char *mdcn_status_string(int status) {
  switch (status) {
    case MDCN_OK: return "ok";
    case MDCN_ERR_NULL: return "a required pointer is NULL";
    case MDCN_ERR_SHAPE: return "invalid shape (non-positive size or channels not divisible by groups)";
    case MDCN_ERR_DTYPE: return "unsupported dtype";
    case MDCN_ERR_WORKSPACE: return "workspace missing, misaligned or too small";
    case MDCN_ERR_PATH: return "shape not covered by the fused path";
    case MDCN_ERR_TOO_LARGE: return "tensor too large for 32-bit device offsets";
    case MDCN_ERR_LAUNCH: return "HIP launch error";
    case MDCN_ERR_SCRATCH_LIMIT: return "call needs more scratch than the library's built-in buffer holds";
    default: return "unknown status";
  }
}

int mdcn_output_size(const mdcn_params *p, int32_t *Ho, int32_t *Wo) {
  Geom g;
  const int rc = check_params(p, &g, false);
  if (rc != MDCN_OK) return rc;
  if (Ho) *Ho = g.Ho;
  if (Wo) *Wo = g.Wo;
  return MDCN_OK;
}

int mdcn_fused_eligible(const mdcn_params *p) {
  Geom g;
  if (check_params(p, &g, false) != MDCN_OK) return 0;
  return fused_ok(p, g) ? 1 : 0;
}

const char *mdcn_forward_kernels(const mdcn_params *p) {
  Geom g;
  if (check_params(p, &g, false) != MDCN_OK) return "";
  Plan pl;
  if (make_plan(p, g, &pl) != MDCN_OK) return "";
  if (p->dtype == MDCN_F64) return "f64_forward_kernel";
  if (pl.seg) return "segment_kernel";
  if (!pl.fused) return "direct_kernel";
  if (p->dtype == MDCN_F32) return "fused_f32_kernel";
  if (!uses_fused2(p, g, pl)) return "fused_kernel";
  const size_t es = elem_size(p->dtype);
  const long plane_out = (long)g.Ho * g.Wo;
  const bool out_vec_ok = (plane_out % (long)(16 / es) == 0) && (((uintptr_t)p->output % 16) == 0);
  const long total_px = (long)std::min(pl.n_chunk, g.N) * plane_out;
  const long n3 = wide_tiles_of_call(p, g, pl, total_px, out_vec_ok);
  if (n3 == 0) return "fused2_kernel";
  return total_px - n3 * kF3PT > 0 ? "fused3_kernel+fused2_kernel" : "fused3_kernel";
}

size_t mdcn_workspace_bytes(const mdcn_params *p) {
  Geom g;
  if (check_params(p, &g, false) != MDCN_OK) return 0;
  Plan pl;
  if (make_plan(p, g, &pl) != MDCN_OK) return 0;
  return pl.seg && !pl.seg_small ? 0 : pl.xt_bytes + pl.wp_bytes + pl.pair_bytes() + pl.cut_bytes;
}

size_t mdcn_workspace_wanted(const mdcn_params *p) {
  Geom g;
  if (check_params(p, &g, false) != MDCN_OK) return 0;
  Plan pl;
  if (make_plan(p, g, &pl) != MDCN_OK) return 0;
  return pl.xt_bytes + pl.wp_bytes + pl.pair_bytes() + pl.cut_bytes;
}

int mdcn_forward(const mdcn_params *p, void *hip_stream) {
  return run(p, hip_stream, nullptr);
}

int mdcn_forward_noalloc(const mdcn_params *p, void *hip_stream) {
  Geom g;
  int rc = check_params(p, &g, true);
  if (rc != MDCN_OK) return rc;
  Plan pl;
  rc = make_plan(p, g, &pl);
  if (rc != MDCN_OK) return rc;
  mdcn_params q = *p;
  if (pl.seg && !pl.seg_small) {  // needs no scratch: the kernel, and the bits, of a mdcn_forward() with mdcn_workspace_bytes()
    q.workspace = nullptr;
    q.workspace_bytes = 0;
    return run(&q, hip_stream, nullptr);
  }
  if (pl.xt_bytes + pl.wp_bytes > (size_t)MDCN_NOALLOC_SCRATCH_BYTES) return MDCN_ERR_SCRATCH_LIMIT;
  void *ptr = nullptr;
  rc = scratch_of_current_device(&ptr);
  if (rc != MDCN_OK) return rc;
  q.workspace = ptr;
  q.workspace_bytes = (size_t)MDCN_NOALLOC_SCRATCH_BYTES;
  return run(&q, hip_stream, nullptr);
}

int mdcn_forward_timed(const mdcn_params *p, void *hip_stream, float ms[4]) {
  if (!ms) return MDCN_ERR_NULL;
  return run(p, hip_stream, ms);
}

size_t mdcn_pack_workspace_bytes(const mdcn_pack_params *pp) {
  Geom g;
  if (!pp || check_params(&pp->conv, &g, false) != MDCN_OK) return 0;
  Plan pl;
  if (make_pack_plan(pp, g, &pl) != MDCN_OK) return 0;
  return pl.xt_bytes + pl.wp_bytes + pl.owp_bytes + pl.raw_bytes + pl.pair_bytes() + pl.cut_bytes;
}

int mdcn_pack_forward(const mdcn_pack_params *pp, void *hip_stream) {
  if (!pp) return MDCN_ERR_NULL;
  return run(&pp->conv, hip_stream, nullptr, pp);
}

size_t mdcn_backward_workspace_bytes(const mdcn_bwd_params *bp) {
  Geom g;
  if (check_bwd(bp, &g, false) != MDCN_OK) return 0;
  BwdPlan pl;
  make_bwd_plan(bp, g, g_bwd_pass_bytes.load(), &pl);
  return pl.total() + pl.max_bytes();
}

int mdcn_backward(const mdcn_bwd_params *bp, void *hip_stream) {
  Geom g;
  const int rc = check_bwd(bp, &g, true);
  if (rc != MDCN_OK) return rc;
  BwdPlan pl;
  make_bwd_plan(bp, g, g_bwd_pass_bytes.load(), &pl);
  const size_t need = pl.total();
  const mdcn_params *p = &bp->conv;
  if (need > 0 && (!p->workspace || p->workspace_bytes < need || ((uintptr_t)p->workspace % kAlign) != 0))
    return MDCN_ERR_WORKSPACE;
  if (pl.max_bytes() && p->workspace_bytes >= need + pl.max_bytes()) pl.max_at = need;
  return run_backward(bp, g, pl, (hipStream_t)hip_stream);
}

int mdcn_pack_trains(const mdcn_pack_params *pp) {
  Geom g;
  if (!pp || check_params(&pp->conv, &g, false) != MDCN_OK || pp->conv.input_nhwc) return 0;
  OconvBwdPlan ol;
  return oconv_bwd_plan(g, pp->conv.dtype, pp->unmodulated != 0, true, true, false, num_cus(), &ol) &&
         oconv_bwd_pays(g, pp->conv.dtype, pp->unmodulated != 0);
}

int mdcn_pack_split(const mdcn_pack_params *pp, void *offset, void *mask, void *hip_stream) {
  if (!pp || !pp->raw || !offset || !mask) return MDCN_ERR_NULL;
  if (pp->unmodulated) return MDCN_ERR_PATH;  // (all of raw is offsets: there is nothing to split)
  Geom g;
  const int rc = check_params(&pp->conv, &g, false);
  if (rc != MDCN_OK) return rc;
  hipStream_t st = (hipStream_t)hip_stream;
  switch (pp->conv.dtype) {
    case MDCN_F32: return split_raw<float>(pp, g, (float *)offset, (float *)mask, st);
    case MDCN_F16: return split_raw<f16_t>(pp, g, (f16_t *)offset, (f16_t *)mask, st);
    case MDCN_BF16: return split_raw<bf16_t>(pp, g, (bf16_t *)offset, (bf16_t *)mask, st);
    default: return MDCN_ERR_DTYPE;
  }
}

size_t mdcn_pack_backward_workspace_bytes(const mdcn_pack_bwd_params *pb) {
  Geom g;
  if (!pb || check_bwd(&pb->bwd, &g, false) != MDCN_OK) return 0;
  BwdPlan pl;
  OconvBwdPlan ol;
  return plan_pack_backward(pb, g, &pl, &ol) ? pl.total() + ol.total() + pl.max_bytes() : 0;
}

int mdcn_pack_backward(const mdcn_pack_bwd_params *pb, void *hip_stream) {
  if (!pb) return MDCN_ERR_NULL;
  Geom g;
  int rc = check_bwd(&pb->bwd, &g, true);
  if (rc != MDCN_OK) return rc;
  const mdcn_params *p = &pb->bwd.conv;
  if (!pb->offset_weight || !pb->bwd.grad_input || (!pb->unmodulated) != (p->mask != nullptr)) return MDCN_ERR_NULL;
  BwdPlan pl;
  OconvBwdPlan ol;
  if (!plan_pack_backward(pb, g, &pl, &ol)) return MDCN_ERR_PATH;
  const size_t need = pl.total() + ol.total();
  if (need > 0 && (!p->workspace || p->workspace_bytes < need || ((uintptr_t)p->workspace % kAlign) != 0))
    return MDCN_ERR_WORKSPACE;
  if (pl.max_bytes() && p->workspace_bytes >= need + pl.max_bytes()) pl.max_at = need;
  rc = run_backward(&pb->bwd, g, pl, (hipStream_t)hip_stream);
  if (rc != MDCN_OK || (!ol.data && !ol.weight)) return rc;
  unsigned char *ws = (unsigned char *)p->workspace;
  OconvBwdArgs a{};
  a.g = g;
  a.x = p->input;
  a.ow = pb->offset_weight;
  a.goff = pb->bwd.grad_offset;
  a.gmask = pb->bwd.grad_mask;
  a.mask = p->mask;
  a.gin = pb->bwd.grad_input;
  a.gw = pb->grad_offset_weight;
  a.gb = pb->grad_offset_bias;
  a.xt = pl.plain_copy() ? ws + pl.xt_at() : nullptr;
  return oconv_backward(p->dtype, ol, a, ws + pl.total(), (hipStream_t)hip_stream) == hipSuccess ? MDCN_OK : MDCN_ERR_LAUNCH;
}

int mdcn_pack_forward_timed(const mdcn_pack_params *pp, void *hip_stream, float ms[5]) {
  if (!pp || !ms) return MDCN_ERR_NULL;
  return run(&pp->conv, hip_stream, ms, pp);
}

}  // extern "C"
