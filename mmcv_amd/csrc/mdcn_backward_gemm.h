// Backward on the matrix cores, for fp32 tensors and for 16-bit calls of few tiles or uneven channels (the others have
// bwd_fused_kernel for the data side, and bwd_wgrad_kernel here): the column
// gradient  d[pixel, (tap, c)] = sum_co grad_output[co, pixel] * weight[co, c, tap]
// (the reference's first GEMM, mmcv/ops/csrc/pytorch/modulated_deform_conv.cpp:199-206)
// is a plain matrix product, so it runs on the matrix cores
// (bwd_colgrad_kernel) and is handed to the scatter kernel through memory in a
// layout made for that kernel: d[image][16-channel chunk][tap][pixel][16].  The
// scatter kernel (bwd_scatter_kernel) then is the reference's three element-wise
// kernels in one pass (cpu/modulated_deform_conv.cpp:34-107,170-320): a thread
// owns an output pixel, reads 4 or 8 channels of d and of the four corners (from
// the zero-bordered pixel-major input copy, 8 to 32 contiguous bytes per corner,
// one tap ahead of their use), forms its share of grad_offset / grad_mask from
// the four sums of d times a corner's values, and adds the grad_input
// contributions into an LDS window around its 8 x 32 pixel tile, which is flushed
// with one global atomic per non-zero entry.  On the way it can
// store the forward's columns, from which grad_weight is a second plain product
// (bwd_wgrad_kernel).
// Both operands of the product are pixel-major / K-contiguous copies written by
// the pre-pass (mdcn_backward_ends.h), which with the finishing pass holds
// everything else a call needs: five launches in all.
//
// Channels that do not fill the tiles are padded in these copies: a segment of
// the input's channels (those of one group and one deformable group) to whole
// passes of the scatter kernel, a group's to a multiple of 32, the output
// channels of a group to 128 bytes.  Padding is zero in every copy, so it adds nothing
// and its gradients -- zero, or NaN where grad_output is not finite -- are never written.
#pragma once

#include <type_traits>

#include "mdcn_backward.h"
#include "mdcn_fused_f32.h"

namespace mdcn {

// Rows of either operand per workgroup tile of the two products: 256 (8
// wavefronts, each 128 x 64, a workgroup a CU) or 128 (4 wavefronts, each 64 x 64,
// two).  Per K step a 256-tile moves 64 KB for 2 048 MFMA
// clocks, a 128-tile 32 KB for 512: with two K steps in flight the small tile is
// bound by the latency of its copies, the large one is not.  Which of them a call has goes
// by how full its rounds and how long its shares are (make_bwd_plan, with both sides measured).
constexpr int kCgTile = 128;
constexpr int kCgTileBig = 256;

struct ColGradArgs {
  // (channel counts are those of the padded orders, see BwdPlan)
  const void *wT;  // [G][M_pad][cout_g]
  const void *gT;  // [N][Cout / KC][P][KC], KC = 128 bytes of channels
  // fp32 as fp16 pairs: those of wT (pack_weight_row_pairs), exponents of its rows, [G][M_pad], and the largest
  const void *wpair;
  const int *wexp;
  const uint16_t *gmax;  // magnitude of each 128 bytes of gT, as relayout_vec_block's row_max, [N][Cout / KC][P]
  float *D;        // [images of the pass][Cin / 16][taps][P][16]
  int P;           // output pixels per image
  int px_tiles, m_tiles;
  int M, M_pad;    // taps * cin_g and its padded size
  int cin_g, cout_g, taps, G, Cin, Cout;
  int kslabs;      // cout_g / KC
  int n0;          // first image of the pass
  long total;      // workgroups with work: images of the pass x G x px_tiles x m_tiles
};

// A wave's products of one K step of either kernel: TILE / 64 x 2 blocks of 32 x 32 over 128 bytes of K, operand tiles
// [row][8 chunks of 16 bytes, swizzled by the row number].
//
// fp32 runs on the 16-bit matrix pipe, as in fused_f32_kernel, with an error that is that of fp32 arithmetic: of bf16 triples (six of the nine products
// of three planes; the weight gradient, whose rows have no exponents at hand) or of fp16 pairs (three products of two planes; the column
// gradient of more than 64 output channels).  Pairs are scaled row by row: a pixel's channels of grad_output and a weight row's output
// channels by the largest of them.  The weights are split by the pre-pass, a row at a time, beside wT, which the fp32 sweep reads; for grad_output it writes the largest of each 128 bytes
// beside its copy.  What is not split before is split behind the LDS reads, every wave for itself: some 290 VALU instructions per 16 of K for triples,
// beside 48 MFMAs of 32 clocks, a third of that for pairs in tiles of 256, half in tiles of 128, beside 24.  An infinity, or a number that the
// scale takes to one (kSplitScale), leaves NaN in the planes and so in the sums: a workgroup
// that finds any goes over its K range again with fp32 MFMAs (PLANES = 0).
// Column gradient in us, triples / pairs split behind the reads / weights split before: N=8 256 -> 256 64x64 279 / 202 / 188, N=4 512 64x64 484 / 338 / 300 (tiles of
// 256), N=4 128 60x80 54 / 45 / 43; whole training calls, pairs, weights split behind the reads / before: N=1 512 25x42 235 / 223, N=8 512 13x21 332 / 317, N=4 512 64x64 1 308 / 1 275.
// Weight gradient, N=2 256 50x84, fp32 MFMAs / triples: 107 / 70.  Errors against float64 (2-norm) there: grad_input
// 2.9e-7 with fp32 MFMAs, 2.5e-7, 2.0e-7 pairs; grad_weight 3.3e-7 / 3.0e-7.
// PLANES: 3, 2 (fp16 pairs, rows scaled by the powers of two ea and eb of the lane's), 0 (products of E itself).
// SPLIT_A: A holds fp16 pairs (pack_weight_row_pairs).
template <typename E, int TILE, int PLANES, bool SPLIT_A = false>
__device__ __forceinline__ void tile_products(f32x16 (&acc)[TILE / 64][2], const uint4 *A, const uint4 *B, int wm, int wn,
                                              int frow, int fhalf, const int (&ea)[TILE / 64], const int (&eb)[2]) {
  using TR = ElemTraits<E>;
  constexpr int MB = TILE / 64;
  // (the rows of a lane's fragments are multiples of 32 apart: one swizzle for all of them)
  const uint4 *a0 = A + (wm * (TILE / 2) + frow) * 8, *b0 = B + (wn * 64 + frow) * 8;
  auto load_a = [&](int mb, int ksub) { return a0[mb * 256 + ((ksub * 2 + fhalf) ^ (frow & 7))]; };
  auto load_b = [&](int nb, int ksub) { return b0[nb * 256 + ((ksub * 2 + fhalf) ^ (frow & 7))]; };
  if constexpr (sizeof(E) == 2 || PLANES == 0) {
#pragma unroll
    for (int ksub = 0; ksub < 4; ++ksub) {
      uint4 af[MB], bf[2];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) af[mb] = load_a(mb, ksub);
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) bf[nb] = load_b(nb, ksub);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) TR::mma(acc[mb][nb], af[mb], bf[nb]);
    }
  } else {
    using TB = ElemTraits<std::conditional_t<PLANES == 2, f16_t, bf16_t>>;
    // 8 values of K as the planes of an operand
    auto split8 = [](const uint4 (&v)[2], uint4 (&p)[PLANES], int e) {
      uint2 lo[PLANES], hi[PLANES];
      auto scaled = [&](uint32_t x) {
        return PLANES == 2 ? __builtin_amdgcn_ldexpf(__uint_as_float(x), e) : __uint_as_float(x) * kSplitScale;
      };
      const float s0[4] = {scaled(v[0].x), scaled(v[0].y), scaled(v[0].z), scaled(v[0].w)};
      const float s1[4] = {scaled(v[1].x), scaled(v[1].y), scaled(v[1].z), scaled(v[1].w)};
      if constexpr (PLANES == 2) {
        split2(s0, lo);
        split2(s1, hi);
      } else {
        split3(s0, lo);
        split3(s1, hi);
      }
#pragma unroll
      for (int s = 0; s < PLANES; ++s) p[s] = make_uint4(lo[s].x, lo[s].y, hi[s].x, hi[s].y);
    };
#pragma unroll
    for (int half = 0; half < 2; ++half) {  // (any order of K will do: both operands have the same)
      uint4 bp[2][PLANES];
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) split8({load_b(nb, half * 2), load_b(nb, half * 2 + 1)}, bp[nb], eb[nb]);
      uint4 af[2] = {load_a(0, half * 2), load_a(0, half * 2 + 1)};
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        uint4 ap[PLANES];
        if constexpr (SPLIT_A) ap[0] = af[0], ap[1] = af[1];
        else split8(af, ap, ea[mb]);
        if (mb + 1 < MB) af[0] = load_a(mb + 1, half * 2), af[1] = load_a(mb + 1, half * 2 + 1);
        __builtin_amdgcn_sched_barrier(0);  // (or every block's planes are made ahead and spilled)
        auto products = [&](int pa, int pb) {
#pragma unroll
          for (int nb = 0; nb < 2; ++nb) TB::mma(acc[mb][nb], ap[pa], bp[nb][pb]);
        };
        if constexpr (PLANES == 3) {
          products(2, 0);  // smallest terms first
          products(0, 2);
          products(1, 1);
        }
        products(1, 0);
        products(0, 1);
        products(0, 0);
      }
    }
  }
}

// Takes the scale of split operands out of the sums; whether one of them is infinite or NaN.
template <int MB>
__device__ __forceinline__ bool unscale(f32x16 (&acc)[MB][2]) {
  float t = 0.0f;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[mb][nb][r] *= kSplitUnscale;
        t = fmaf(acc[mb][nb][r], 0.0f, t);
      }
  return t != t;
}

// Workgroup = TILE rows of wT (one group) x TILE pixels of one image, reduction
// over the group's output channels in slabs of 128 bytes; TILE / 32 waves as
// 2 x TILE / 64, each TILE / 64 x 2 MFMA blocks of 32 x 32.  Both operand tiles of a slab go to LDS with
// 16-byte direct-to-LDS copies (rows of 128 bytes, the 16-byte chunks of a row
// swizzled by the row number on the source side, so that fragment reads are
// conflict free), double buffered.  A rows = (tap, channel), B rows = pixels:
// a lane ends up with 4 x 4 consecutive channels of one pixel, which is what the
// d layout wants (16-byte stores).
// PAIRS: fp32 as fp16 pairs (see tile_products).
template <typename E, int TILE, bool PAIRS>
__global__ __launch_bounds__(TILE * 2, TILE == 128 ? 2 : 1) void bwd_colgrad_kernel(ColGradArgs a) {
  using TR = ElemTraits<E>;
  constexpr int ES = (int)sizeof(E);
  constexpr int KC = 128 / ES;
  constexpr int MB = TILE / 64;            // 32-row blocks of A per wave
  constexpr uint32_t kBuf = TILE * 128u;   // bytes of one operand tile
  __shared__ uint4 As[2][TILE * 8];
  __shared__ uint4 Bs[2][TILE * 8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int frow = lane & 31, fhalf = lane >> 5;
  const int wm = wave & 1, wn = wave >> 1;
  // (the row tiles of one pixel tile are neighbours: they share the grad_output tile)
  long b = xcd_work_index(a.total);
  if (b < 0) return;
  const int mt = (int)(b % a.m_tiles);
  b /= a.m_tiles;
  const int pt = (int)(b % a.px_tiles);
  b /= a.px_tiles;
  const int grp = (int)(b % a.G);
  const int nl = (int)(b / a.G);
  const int n = a.n0 + nl;

  // this lane's share of the copies: 4 of the 16 one-KiB blocks (8 rows) of each tile
  const unsigned char *a_src[4], *b_src[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int row = (wave * 4 + c) * 8 + (lane >> 3);
    const int ch = (lane & 7) ^ (row & 7);
    a_src[c] = (const unsigned char *)(PAIRS ? a.wpair : a.wT) +
               ((long)grp * a.M_pad + (long)mt * TILE + row) * a.cout_g * ES + ch * 16;
    // rows past the image repeat its last pixel; they are never stored
    const int px = min(pt * TILE + row, a.P - 1);
    b_src[c] = (const unsigned char *)a.gT +
               (((long)n * (a.Cout / KC) + (long)grp * a.kslabs) * a.P + px) * 128 + ch * 16;
  }
  const long b_step = (long)a.P * 128;
  const uint32_t lds_a = (uint32_t)(uintptr_t)(lptr_t)(&As[0][0]) +
                         (uint32_t)__builtin_amdgcn_readfirstlane(wave) * 4096u;
  const uint32_t lds_b = (uint32_t)(uintptr_t)(lptr_t)(&Bs[0][0]) +
                         (uint32_t)__builtin_amdgcn_readfirstlane(wave) * 4096u;
  auto issue = [&](int ks, int buf) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      copy16_global_to_lds(a_src[c] + (long)ks * 128, lds_a + (uint32_t)buf * kBuf + (uint32_t)c * 1024u);
      copy16_global_to_lds(b_src[c] + (long)ks * b_step, lds_b + (uint32_t)buf * kBuf + (uint32_t)c * 1024u);
    }
  };

  // pairs: exponents of the tile's rows of A, then of B
  __shared__ __align__(16) int exps[PAIRS ? 2 * TILE : 4];
  int ea[MB] = {}, eb[2] = {};
  issue(0, 0);
  if constexpr (PAIRS) {
    const int row = tid & (TILE - 1);
    if (tid < TILE) {
      exps[tid] = a.wexp[(long)grp * a.M_pad + (long)mt * TILE + row];
    } else {
      const uint16_t *src = a.gmax + ((long)n * (a.Cout / KC) + (long)grp * a.kslabs) * a.P + min(pt * TILE + row, a.P - 1);
      uint32_t top = 0;
#pragma unroll 8
      for (int s = 0; s < a.kslabs; ++s) top = max(top, (uint32_t)src[(long)s * a.P]);
      exps[tid] = pair_exponent(__uint_as_float(top << 16));
    }
    __syncthreads();
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) ea[mb] = exps[wm * (TILE / 2) + mb * 32 + frow];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) eb[nb] = exps[TILE + wn * 64 + nb * 32 + frow];
  }

  f32x16 acc[MB][2];
  auto sweep = [&](auto planes) {
    constexpr int PLANES = decltype(planes)::value;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    for (int ks = 0; ks < a.kslabs; ++ks) {
      const int buf = ks & 1;
      if (ks + 1 < a.kslabs) {
        issue(ks + 1, buf ^ 1);  // (its buffer was last read before the barrier that ended step ks - 1)
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
      } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      __syncthreads();
      tile_products<E, TILE, PLANES, PAIRS && PLANES == 2>(acc, As[buf], Bs[buf], wm, wn, frow, fhalf, ea, eb);
      __syncthreads();
    }
  };
  sweep(std::integral_constant<int, PAIRS ? 2 : 3>());
  if constexpr (sizeof(E) == 4) {
    bool bad;
    if constexpr (PAIRS) {
      float t = 0.0f;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int4 e4 = *(const int4 *)&exps[wm * (TILE / 2) + mb * 32 + j * 8 + fhalf * 4];
          const int e[4] = {e4.x, e4.y, e4.z, e4.w};
#pragma unroll
          for (int nb = 0; nb < 2; ++nb)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float c = __builtin_amdgcn_ldexpf(acc[mb][nb][j * 4 + i], -(e[i] + eb[nb]));
              acc[mb][nb][j * 4 + i] = c;
              t = fmaf(c, 0.0f, t);
            }
        }
      bad = t != t;
    } else {
      bad = unscale(acc);
    }
    if (__syncthreads_or(bad)) {
      if constexpr (PAIRS) {
        const long to_whole = (const unsigned char *)a.wT - (const unsigned char *)a.wpair;
#pragma unroll
        for (int c = 0; c < 4; ++c) a_src[c] += to_whole;
      }
      issue(0, 0);
      sweep(std::integral_constant<int, 0>());
    }
  }

  // register r of lane l: A row (r/4)*8 + (l/32)*4 + r%4 of the block, B row l%32
  const int chunks = a.Cin / 16;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int m0 = mt * TILE + wm * (TILE / 2) + mb * 32;  // a block = one tap, 32 consecutive channels
    if (m0 >= a.M) continue;
    const int tap = m0 / a.cin_g;
    const int cb = grp * a.cin_g + (m0 - tap * a.cin_g);
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      const int px = pt * TILE + wn * 64 + nb * 32 + frow;
      if (px >= a.P) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int c = cb + j * 8 + fhalf * 4;
        float *dst = a.D + ((((long)nl * chunks + (c >> 4)) * a.taps + tap) * a.P + px) * 16 + (c & 15);
        *(float4 *)dst = make_float4(acc[mb][nb][4 * j], acc[mb][nb][4 * j + 1], acc[mb][nb][4 * j + 2],
                                     acc[mb][nb][4 * j + 3]);
      }
    }
  }
}

// Bytes of the scatter kernel's window (two workgroups per CU).  It holds CH
// channels of a WH x WW pixel neighbourhood of the tile; kScWindowPx pixels fit
// with 8 channels of doubles, twice as many -- stride 2, dilation -- with 4.  (A 48 KB window with 8 channels and three
// workgroups per CU was slower: the passes over the window double.)
constexpr int kScWindowBytes = 60 * 1024;
constexpr int kScWindowPx = kScWindowBytes / 64;
// Largest margin of the window for far offsets.
constexpr int kScFarMargin = 12;
// Samples beyond the window that a wavefront adds at a time, and the floats each has in LDS: position and channels.
template <int CH>
constexpr int kLoneAtOnce = CH >= 16 ? 1 : 16 / CH;
template <int CH>
constexpr int kLoneStride = (CH + 4 + 3) / 4 * 4;
template <int CH>
constexpr int kLoneFloats = kLoneAtOnce<CH> * kLoneStride<CH>;

// CH consecutive channels (8 to 32 bytes) as floats.
template <typename E, int CH>
struct VecCh {
  static constexpr int NW = CH * (int)sizeof(E) / 4;  // 32-bit words
  uint32_t raw[NW];
  __device__ __forceinline__ void load(const E *p) {
    if constexpr (NW % 4 == 0) {
#pragma unroll
      for (int i = 0; i < NW / 4; ++i) {
        const uint4 v = ((const uint4 *)p)[i];
        raw[4 * i] = v.x;
        raw[4 * i + 1] = v.y;
        raw[4 * i + 2] = v.z;
        raw[4 * i + 3] = v.w;
      }
    } else {
      static_assert(NW == 2, "8 bytes");
      const uint2 v = *(const uint2 *)p;
      raw[0] = v.x;
      raw[1] = v.y;
    }
  }
  // channels 2 i and 2 i + 1
  __device__ __forceinline__ void pair(int i, float &lo, float &hi) const {
    if constexpr (sizeof(E) == 4) {
      lo = __uint_as_float(raw[2 * i]);
      hi = __uint_as_float(raw[2 * i + 1]);
    } else {
      ElemTraits<E>::unpack2(raw[i], lo, hi);
    }
  }
  // acc + this's channels 2 i and 2 i + 1 times o's
  template <typename D>
  __device__ __forceinline__ float dot_pair(const VecCh<D, CH> &o, int i, float acc) const {
    if constexpr (sizeof(D) == 4) {
      float lo, hi;
      pair(i, lo, hi);
      acc = fmaf(lo, __uint_as_float(o.raw[2 * i]), acc);
      return fmaf(hi, __uint_as_float(o.raw[2 * i + 1]), acc);
    } else {
      return ElemTraits<E>::dot2(raw[i], o.raw[i], acc);
    }
  }
  __device__ __forceinline__ void unpack(float (&out)[CH]) const {
    if constexpr (sizeof(E) == 4) {
#pragma unroll
      for (int i = 0; i < CH; ++i) out[i] = __uint_as_float(raw[i]);
    } else {
#pragma unroll
      for (int i = 0; i < NW; ++i) ElemTraits<E>::unpack2(raw[i], out[2 * i], out[2 * i + 1]);
    }
  }
};

// Output-pixel tile of the scatter kernel: 8 rows x 32 columns, one thread per
// pixel (rows of 32 keep the loads of d and the stores of the columns in 64-byte
// or longer runs, and the window around it stays under 48 KiB for a margin of 3).
constexpr int kScTH = 8;
constexpr int kScTW = 32;

// A workgroup's window of grad_input in LDS: WH x WW input pixels, R of margin around the tile's undeformed footprint.
struct ScatterWindow {
  int R, WH, WW;
};

struct BwdScatterArgs {
  Geom g;
  const void *xt;  // zero-bordered input copy in 32-byte records [N][Cin / RC][H + 2][W + 2][RC], RC = 32 bytes of channels
  OffMaskView om;
  const void *D;   // column gradient of the pass, layout of ColGradArgs::D; null: columns only
  float *gin32;
  void *goff;
  void *gmask;     // null when unmodulated
  void *col;       // columns of the pass (WGradArgs::col), or null
  int run;
  ChanMap im;      // padded order of the input channels
  int cin_p;       // ... how many there are
  long P_pad;      // row pitch of col in elements
  int tiles_x, tiles_y;
  ScatterWindow win;      // with CH channels a pass
  ScatterWindow win_far;  // with CH / 2: twice the pixels, for offsets that leave the other one (WH = 0: none)
  const uint32_t *far;    // n_far counts of sampled offsets beyond win's margin; above far_min in all, win_far is used
  int n_far;
  uint32_t far_min;
  int n0;          // first image of the pass
  // A deformable group's channels are shared among `parts` workgroups per tile
  // (blockIdx.y): up to 8 of them where that makes the last of many rounds short, up
  // to 32 where tiles are few (scatter_parts); with parts > 1 each writes its
  // share of the offset / mask sums as floats to poff / pmask ([part][layout of
  // grad_offset / grad_mask]), which bwd_finish_kernel adds up.
  int parts;
  float *poff, *pmask;
  long off_total, mask_total;  // elements of grad_offset / grad_mask
};

// The window is not fp32: LDS single-precision atomic adds are slow on this
// hardware (measured per wavefront instruction per CU: ds_add_f32 170 clocks,
// ds_add_f64 26, ds_add_u64 14, ds_add_u32 11, whatever the addresses), so it holds doubles.  16-bit
// tensors that fill the tiles have bwd_fused_kernel, whose window is fixed point.
// DATA: the gradient part (a.D, window, offset / mask sums).  COL: the kernel
// stores the forward's columns (mask * bilinear sample, rounded to E as the
// reference's columns tensor is) to a.col for the weight-gradient product.  At
// least one of the two.
template <typename E, int CH, bool DATA, bool COL>
__device__ __forceinline__ void scatter_tile(const BwdScatterArgs &a, const ScatterWindow &wd, double *win, float *lone) {
  constexpr int RC = 32 / (int)sizeof(E);   // channels per record of the input copy
  static_assert(DATA || COL, "nothing to do");
  static_assert(CH <= RC && RC % CH == 0, "a pass reads a record or a whole fraction of one");
  static_assert(kScTH * kScTW == 256, "one thread per pixel of the tile");
  const Geom &g = a.g;
  const long plane_out = (long)g.Ho * g.Wo;
  const long plane_in = (long)g.H * g.W;
  const long slab_px = (long)g.Hp * g.Wp;
  const int tid = threadIdx.x;
  int b = blockIdx.x;
  const int tx = b % a.tiles_x;
  b /= a.tiles_x;
  const int ty = b % a.tiles_y;
  b /= a.tiles_y;
  const int dgi = b % g.DG;
  const int nl = b / g.DG;
  const int n = a.n0 + nl;
  const int ho = ty * kScTH + tid / kScTW, wo = tx * kScTW + tid % kScTW;
  const bool valid = ho < g.Ho && wo < g.Wo;
  const long pix = valid ? (long)ho * g.Wo + wo : 0;
  const int wy0 = ty * kScTH * g.sh - g.ph - wd.R, wx0 = tx * kScTW * g.sw - g.pw - wd.R;
  const int win_px = wd.WH * wd.WW;

  const E *off = (const E *)a.om.off + (long)n * a.om.off_n + pix * a.om.off_px +
                 (long)(dgi * 2 * g.taps) * a.om.off_ch;
  const E *msk = (const E *)a.om.msk + (long)n * a.om.msk_n + pix * a.om.msk_px +
                 (long)(dgi * g.taps) * a.om.msk_ch;

  float acc_m[kBwdTapsMax], acc_y[kBwdTapsMax], acc_x[kBwdTapsMax];
#pragma unroll
  for (int t = 0; t < kBwdTapsMax; ++t) acc_m[t] = acc_y[t] = acc_x[t] = 0.0f;
  // this pixel's offsets and mask, fetched once: every channel pass needs them before it can
  // address its corners
  E t_dy[kBwdTapsMax], t_dx[kBwdTapsMax], t_m[kBwdTapsMax];
#pragma unroll
  for (int t = 0; t < kBwdTapsMax; ++t) {
    const int tc = min(t, g.taps - 1);
    t_dy[t] = off[(long)(2 * tc) * a.om.off_ch];
    t_dx[t] = off[(long)(2 * tc + 1) * a.om.off_ch];
    t_m[t] = msk[(long)tc * a.om.msk_ch];
  }

  // This workgroup's passes of CH channels.  Pass i of the deformable group: segment i / (segp / CH) of the
  // group, from padded channel c0 on; the tensor's channel cs, of which `room` are left in the segment.
  const int part = blockIdx.y;
  const int passes = g.ch_per_dg / a.im.seg * (a.im.segp / CH);
  const int ps_begin = (int)((long)passes * part / a.parts), ps_end = (int)((long)passes * (part + 1) / a.parts);
  struct Pass {
    int c0, cs, room, grp;
  };
  auto pass_at = [&](int i) {
    const int per = a.im.segp / CH;
    const int k = i / per, w = (i - k * per) * CH;
    const int S = dgi * (g.ch_per_dg / a.im.seg) + k;   // segment of the tensor
    Pass p;
    p.grp = S / a.im.nseg;
    p.c0 = p.grp * a.im.cgp + (S - p.grp * a.im.nseg) * a.im.segp + w;
    p.cs = S * a.im.seg + w;
    p.room = a.im.seg - w;
    return p;
  };

  // Window pixels this thread flushes (tid, tid + 256, ...) as offsets into an image plane, the same
  // in every pass; -1 for one outside the image or past the window (it only ever receives zeros).
  constexpr int kSlots = DATA ? (kScWindowBytes / (CH * 8) + 255) / 256 : 1;
  int flush_at[kSlots];
  if constexpr (DATA) {
#pragma unroll
    for (int j = 0; j < kSlots; ++j) {
      const int q = tid + 256 * j;
      const int y = wy0 + q / wd.WW, x = wx0 + q % wd.WW;
      flush_at[j] = (q < win_px && y >= 0 && y < g.H && x >= 0 && x < g.W) ? y * g.W + x : -1;
    }
    // (the flush leaves the window zeroed for the next pass)
    for (int i = tid; i < kScWindowBytes / 16; i += 256) ((uint4 *)win)[i] = make_uint4(0u, 0u, 0u, 0u);
  }

  // One tap's sampling position and what was loaded there.  No branch around a tap's body: a
  // position outside the sampling range (or a lane past the image) samples four pixels of the
  // border with weights, mask and d of zero, so it stores a column of zeros and adds zeros.
  // Per-corner conditions become weights of zero too: a wavefront pays for an LDS atomic
  // whether or not a lane sits it out, and a branch per corner and channel was most of the
  // instructions this kernel issued.
  struct Sample {
    int y0, x0;
    float ly, lx, m;
    bool inside;
    VecCh<E, CH> r00, r01, r10, r11;
    VecCh<float, CH> rd;
  };
  auto fetch = [&](int c0, int tap, E e_dy, E e_dx, E e_m, Sample &s) {
    const int ti = tap / g.kw, tj = tap - ti * g.kw;
    float dy = to_f32(e_dy);
    float dx = to_f32(e_dx);
    // (opaque to the optimiser: it would otherwise move the position arithmetic of all taps
    // out of the channel loop and spill what that keeps alive)
    asm volatile("" : "+v"(dy), "+v"(dx));
    const float py = (float)(ho * g.sh - g.ph + ti * g.dh) + dy;
    const float px = (float)(wo * g.sw - g.pw + tj * g.dw) + dx;
    s.inside = valid && (py > -1.0f) && (px > -1.0f) && (py < (float)g.H) && (px < (float)g.W);
    const float fy = floorf(py), fx = floorf(px);
    s.y0 = s.inside ? (int)fy : -1;
    s.x0 = s.inside ? (int)fx : g.W;   // (nothing sampled: four zeros, the right border's above the image and the pixel behind each)
    s.ly = s.inside ? py - fy : 0.0f;
    s.lx = s.inside ? px - fx : 0.0f;
    s.m = s.inside ? mask_value<E>(e_m, a.om.logit) : 0.0f;
    // corners outside the image read the copy's zero border
    const E *xp = (const E *)a.xt + (((long)n * (a.cin_p / RC) + c0 / RC) * slab_px) * RC + (c0 % RC) +
                  ((long)(s.y0 + 1) * g.Wp + (s.x0 + 1)) * RC;
    s.r00.load(xp);
    s.r01.load(xp + RC);
    s.r10.load(xp + (long)g.Wp * RC);
    s.r11.load(xp + (long)(g.Wp + 1) * RC);
    if constexpr (DATA)
      s.rd.load((const float *)a.D + (((long)nl * (a.cin_p / 16) + (c0 >> 4)) * g.taps + tap) * plane_out * 16 + pix * 16 +
                (c0 & 15));
  };
  // A tap's loads are issued one tap ahead, in front of the previous tap's stores and atomics
  // (a wait for loads also waits for every older store, and the compiler cannot move a load
  // above a store that might alias it); the last tap of a pass fetches the first of the next.
  // Two samples take turns: copying the next one over the current one would wait for its loads at the end of every tap
  // (backward of fp32, N=2, 256 channels, 50x84: 329 against 322 us; N=8, 128 channels, 60x80, stride 2: 196 / 187).
  Sample smp[2];
  Pass ps = pass_at(ps_begin);
  fetch(ps.c0, 0, t_dy[0], t_dx[0], t_m[0], smp[0]);

  for (int pi = ps_begin; pi < ps_end; ++pi) {
    if constexpr (DATA) __syncthreads();  // the window is zero: first fill or the previous pass's flush
    const int c0 = ps.c0, cs = ps.cs;
    // this pixel's columns of channel c0 at tap 0, and the way to the next tap (a pass stays inside one group)
    E *cbase;
    long ctap;
    if constexpr (sizeof(E) == 2) {
      cbase = (E *)a.col + (((long)nl * (a.cin_p / a.run) + c0 / a.run) * g.taps * a.P_pad + pix) * a.run + c0 % a.run;
      ctap = a.P_pad * a.run;
    } else {
      cbase = (E *)a.col + (((long)nl * a.cin_p + (long)ps.grp * a.im.cgp) * g.taps + (c0 - ps.grp * a.im.cgp)) * a.P_pad + pix;
      ctap = (long)a.im.cgp * a.P_pad;
    }
    const Pass nps = pass_at(min(pi + 1, ps_end - 1));  // (the last pass fetches its own first tap again: unused)
    const int c_next = nps.c0;
#pragma unroll
    for (int tap = 0; tap < kBwdTapsMax; ++tap) {
      if (tap < g.taps) {
        Sample &cur = smp[tap & 1], &nxt = smp[(tap + 1) & 1];
        {
          const bool more = tap + 1 < g.taps;  // workgroup uniform
          const int tn = tap + 1 < kBwdTapsMax ? tap + 1 : 0;  // (a constant once the loop is unrolled)
          fetch(more ? c0 : c_next, more ? tn : 0, more ? t_dy[tn] : t_dy[0], more ? t_dx[tn] : t_dx[0],
                more ? t_m[tn] : t_m[0], nxt);
        }
        __builtin_amdgcn_sched_barrier(0);   // (these loads first, then the wait for the current sample's)
        const bool inside = cur.inside;
        const int y0 = cur.y0, x0 = cur.x0, y1 = y0 + 1, x1 = x0 + 1;
        const float ly = cur.ly, lx = cur.lx, hy = 1.0f - ly, hx = 1.0f - lx, m = cur.m;
        const bool ok00 = y0 >= 0 && x0 >= 0, ok01 = y0 >= 0 && x1 <= g.W - 1;
        const bool ok10 = y1 <= g.H - 1 && x0 >= 0, ok11 = y1 <= g.H - 1 && x1 <= g.W - 1;
        const float w00 = hy * hx, w01 = hy * lx, w10 = ly * hx, w11 = ly * lx;
        VecCh<float, CH> &rd = cur.rd;
        if constexpr (DATA) {
          const uint32_t keep = inside ? ~0u : 0u;  // (whatever d holds where nothing is sampled)
#pragma unroll
          for (int i = 0; i < VecCh<float, CH>::NW; ++i) rd.raw[i] &= keep;
        }
        const int ry = y0 - wy0, rx = x0 - wx0;
        const bool in_win = ry >= 0 && ry + 1 < wd.WH && rx >= 0 && rx + 1 < wd.WW;
        const bool to_win = inside && in_win;
        // window is [channel][WH][WW]: neighbouring pixels, neighbouring banks; a lane with nothing
        // for the window adds its zeros at an entry of its own
        const int wbase = to_win ? ry * wd.WW + rx : (tid & 63);
        const float s00 = (to_win && ok00) ? w00 : 0.0f, s01 = (to_win && ok01) ? w01 : 0.0f;
        const float s10 = (to_win && ok10) ? w10 : 0.0f, s11 = (to_win && ok11) ? w11 : 0.0f;
        // sums over the pass's channels of d times each corner's value: the offset and mask
        // gradients are combinations of these four
        float S00 = 0.0f, S01 = 0.0f, S10 = 0.0f, S11 = 0.0f;
        E cv[CH];
        // two channels at a time, straight from the loaded words
#pragma unroll
        for (int cp = 0; cp < CH / 2; ++cp) {
          if constexpr (DATA) {
            S00 = cur.r00.dot_pair(rd, cp, S00);
            S01 = cur.r01.dot_pair(rd, cp, S01);
            S10 = cur.r10.dot_pair(rd, cp, S10);
            S11 = cur.r11.dot_pair(rd, cp, S11);
          }
          if constexpr (COL) {
            float v00[2], v01[2], v10[2], v11[2];
            cur.r00.pair(cp, v00[0], v00[1]);
            cur.r01.pair(cp, v01[0], v01[1]);
            cur.r10.pair(cp, v10[0], v10[1]);
            cur.r11.pair(cp, v11[0], v11[1]);
#pragma unroll
            for (int h = 0; h < 2; ++h)
              cv[2 * cp + h] = from_f32<E>(m * (w00 * v00[h] + w01 * v01[h] + w10 * v10[h] + w11 * v11[h]));
          }
          if constexpr (DATA) {
            float d[2];
            rd.pair(cp, d[0], d[1]);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              // (a lane with nothing for the window adds zeros to an entry that may be somebody's: also where its own
              // d is infinite, which a weight of zero would make NaN)
              const float t = to_win ? d[h] * m : 0.0f;
              double *wp = win + (2 * cp + h) * win_px + wbase;
              atomicAdd(wp, (double)(s00 * t));
              atomicAdd(wp + 1, (double)(s01 * t));
              atomicAdd(wp + wd.WW, (double)(s10 * t));
              atomicAdd(wp + wd.WW + 1, (double)(s11 * t));
            }
          }
        }
        if constexpr (COL) {
          if (valid) {
            E *crow = cbase + tap * ctap;
            if constexpr (sizeof(E) == 2) {
              __builtin_memcpy(__builtin_assume_aligned(crow, CH >= 8 ? 16 : 8), cv, sizeof(cv));
            } else {
#pragma unroll
              for (int cc = 0; cc < CH; ++cc) crow[(long)cc * a.P_pad] = cv[cc];
            }
          }
        }
        if constexpr (DATA) {
          acc_m[tap] += w00 * S00 + w01 * S01 + w10 * S10 + w11 * S11;
          acc_y[tap] += m * (hx * (S10 - S00) + lx * (S11 - S01));
          acc_x[tap] += m * (hy * (S01 - S00) + ly * (S11 - S10));
          // Samples beyond the window go to memory directly, a lane for every channel and corner of kLoneAtOnce<CH> samples at a
          // time: what a lane takes part in comes through LDS, position first, then the channels.  Backward in us, every lane its own
          // sample with 4 CH atomics / one sample at a time / this: bf16 N=2 C=128 60x80 stride 2 (4 channels a pass, margin 3)
          // sigma 3 116 / 128 / 112, 5 125 / 159 / 122, 10 210 / 214 / 150; bf16 N=2 C=256 50x84 (8 channels, margin 5) sigma 6
          // 277 / 256 / 248, 20 1 049 / 716 / 659.
          constexpr int S = kLoneAtOnce<CH>, LS = kLoneStride<CH>;
          const unsigned long long beyond = __ballot(inside && !in_win);
          if (beyond != 0ull) {
            const int lane = tid & 63, total = __popcll(beyond), mine = lane / (4 * CH);
            const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(beyond >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)beyond, 0u));
            const int k = lane % CH, corner = lane / CH % 4;
            for (int done = 0; done < total; done += S) {
              if (inside && !in_win && rank >= done && rank < done + S) {
                float *q = lone + (rank - done) * LS, d[CH];
                *(float4 *)q = make_float4(__int_as_float(y0), __int_as_float(x0), ly, lx);
                rd.unpack(d);
#pragma unroll
                for (int cc = 0; cc < CH; ++cc) q[4 + cc] = d[cc] * m;
              }
              __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
              const float4 at = *(const float4 *)(lone + mine * LS);
              const float t = lone[mine * LS + 4 + k];
              const int yy = __float_as_int(at.x) + (corner >> 1), xx = __float_as_int(at.y) + (corner & 1);
              const float w = ((corner & 2) ? at.z : 1.0f - at.z) * ((corner & 1) ? at.w : 1.0f - at.w);
              if (done + mine < total && k < ps.room && yy >= 0 && yy < g.H && xx >= 0 && xx < g.W)
                unsafeAtomicAdd(a.gin32 + ((long)n * g.Cin + cs + k) * plane_in + ((long)yy * g.W + xx), w * t);
              __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
          }
        }
      }
    }
    if constexpr (DATA) {
      __syncthreads();  // every add into the window has landed
      // (Padding channels have no plane of their own: d is zero there, but NaN where grad_output is not finite, and what
      // follows is another segment, the next image, or the end of the tensor.  A fixed-point call has none.)
      const int room = ps.room;
      float *gplane = a.gin32 + ((long)n * g.Cin + cs) * plane_in;
#pragma unroll
      for (int j = 0; j < kSlots; ++j) {
        if (flush_at[j] >= 0) {
          const int q = tid + 256 * j;
          float *gi = gplane + flush_at[j];
#pragma unroll
          for (int cc = 0; cc < CH; ++cc) {
            const double v = win[cc * win_px + q];
            if (v != 0.0) {
              win[cc * win_px + q] = 0.0;
              if (cc < room) unsafeAtomicAdd(gi + (long)cc * plane_in, (float)v);
            }
          }
        }
      }
    }
    if (g.taps & 1) smp[0] = smp[1];   // (the next pass's first)
    ps = nps;
  }
  if constexpr (DATA) {
    if (valid) {
      const long ob = ((long)n * g.DG + dgi) * 2 * g.taps;
      const long mb = ((long)n * g.DG + dgi) * g.taps;
      if (a.parts == 1) {
        E *goff = (E *)a.goff, *gmask = (E *)a.gmask;
#pragma unroll
        for (int tap = 0; tap < kBwdTapsMax; ++tap) {
          if (tap < g.taps) {
            goff[(ob + 2 * tap) * plane_out + pix] = from_f32<E>(acc_y[tap]);
            goff[(ob + 2 * tap + 1) * plane_out + pix] = from_f32<E>(acc_x[tap]);
            if (gmask) gmask[(mb + tap) * plane_out + pix] = from_f32<E>(acc_m[tap]);
          }
        }
      } else {
        float *poff = a.poff + (long)part * a.off_total;
        float *pmask = a.gmask ? a.pmask + (long)part * a.mask_total : nullptr;
#pragma unroll
        for (int tap = 0; tap < kBwdTapsMax; ++tap) {
          if (tap < g.taps) {
            poff[(ob + 2 * tap) * plane_out + pix] = acc_y[tap];
            poff[(ob + 2 * tap + 1) * plane_out + pix] = acc_x[tap];
            if (pmask) pmask[(mb + tap) * plane_out + pix] = acc_m[tap];
          }
        }
      }
    }
  }
}

// Few offsets beyond the margin of the wide pass's window: CH channels a pass.  Many: half as many channels over a
// window twice as large, since a corner outside the window costs CH global atomics.  (Which of the two is
// decided on the device, from a sample of the offsets that the pre-pass has looked at.)
template <typename E, int CH, bool DATA, bool COL>
__global__ __launch_bounds__(256, 2) void bwd_scatter_kernel(BwdScatterArgs a) {
  __shared__ __align__(16) double win[DATA ? kScWindowBytes / 8 : 4];
  constexpr int kLone = kLoneFloats<CH> > kLoneFloats<CH / 2> ? kLoneFloats<CH> : kLoneFloats<CH / 2>;
  __shared__ __align__(16) float lone[4 * kLone];   // of each wavefront
  float *mine = lone + (threadIdx.x >> 6) * kLone;
  if constexpr (DATA && CH * (int)sizeof(E) >= 16) {
    if (a.win_far.WH > 0) {
      uint32_t n = (int)(threadIdx.x & 63) < a.n_far ? a.far[threadIdx.x & 63] : 0u;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o);
      if (__builtin_amdgcn_readfirstlane((int)n) > (int)a.far_min) {
        scatter_tile<E, CH / 2, DATA, COL>(a, a.win_far, win, mine);
        return;
      }
    }
  }
  scatter_tile<E, CH, DATA, COL>(a, a.win, win, mine);
}

struct WGradArgs {
  const void *gout;  // [N][Cout][a_pitch]: grad_output in place (a_pitch = P) or its padded copy (P_pad)
  long a_pitch;
  // Columns: 16-bit tensors [images of the pass][padded channel / run][taps][P_pad][run], run = 16, 8 or 4 channels, those that
  // are stored together (runs of 16 half filled by each of two passes: 173 -> 184 us for the backward of bf16 N=2, 32 channels,
  // 150x200, 4 deformable groups); fp32 [images of the pass][G][taps][padded channels of a group][P_pad]
  const void *col;
  float *part;       // partial sums [split][G][cout_g][M], every element written
  int accumulate;    // 0: the first pass writes them; 1: a later one adds to them
  int P;
  long P_pad;
  int ksteps;        // P_pad / (pixels per 128 bytes)
  int nb, n0;        // images of the pass, first image
  int M;             // taps * padded channels of a group
  int cgp, rows;     // padded channels of a group, and how many of them have rows in col: its segments'
  int cout_g, taps, G, Cin, Cout;   // (Cin: padded)
  int co_tiles, m_tiles;
  int splits;        // workgroups sharing the (image, K step) range of one tile
  long total;        // workgroups with work: G x co_tiles x m_tiles x splits
};

// Where an element of run `run` of a block of 16 columns lies among the 64 x RUN of that run: at its index with these bits
// toggled.  A transposing read takes four pixels of all of a block's runs at once, whole multiples of 512 bytes apart: on the
// same banks, unless each run has its fours of pixels in another order.  (Weight gradient in us, in order / so: bf16 N=12 64 channels
// 16x25 stride 2, runs of 4, 14.0 / 11.7; N=4 96 -> 72 37x53, runs of 8, 14.6 / 14.1.)
template <int RUN>
__device__ __forceinline__ int tr_swizzle(int run) {
  return run * (4 * RUN);
}

// A wave's products of one K step with the second operand pixel major: B holds, for every 16 columns, 16 / run runs of 64 pixels x
// run columns.  An LDS read that transposes gives a lane four consecutive pixels of one column: 16 lanes
// read 8 bytes each, four pixels of every four columns.
template <typename E, int TILE, int RUN>
__device__ __forceinline__ void tile_products_tr(f32x16 (&acc)[TILE / 64][2], const uint4 *A, const uint4 *B, int wm, int wn,
                                                 int lane) {
  using TR = ElemTraits<E>;
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4 *lds4_t;
  constexpr int MB = TILE / 64;
  const int frow = lane & 31, fhalf = lane >> 5;
  const uint4 *a0 = A + (wm * (TILE / 2) + frow) * 8;
  // the four columns and the pixel whose 8 bytes this lane reads; four pixels of a run lie where tr_swizzle has put them
  constexpr int per = RUN / 4, pitch = RUN * 2;
  const int quad = lane & 3, run = quad / per, px = fhalf * 8 + ((lane & 15) >> 2), sw = 2 * tr_swizzle<RUN>(run);
  const unsigned char *b0 = (const unsigned char *)B + (wn * 4 + ((lane >> 4) & 1)) * 2048 + run * (64 * pitch) + quad % per * 8;
  const unsigned char *b_lo = b0 + ((px * pitch) ^ sw), *b_hi = b0 + (((px + 4) * pitch) ^ sw);
#pragma unroll
  for (int ksub = 0; ksub < 4; ++ksub) {
    uint4 af[MB], bf[2];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) af[mb] = a0[mb * 256 + ((ksub * 2 + fhalf) ^ (frow & 7))];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      const int at = nb * 4096 + ksub * 16 * pitch;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4_t)(lptr_t)(void *)(b_lo + at));
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4_t)(lptr_t)(void *)(b_hi + at));
      const uint2 l2 = __builtin_bit_cast(uint2, lo), h2 = __builtin_bit_cast(uint2, hi);
      bf[nb] = make_uint4(l2.x, l2.y, h2.x, h2.y);
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) TR::mma(acc[mb][nb], af[mb], bf[nb]);
  }
}

// grad_weight[co, (c, tap)] += sum over the pass's images and pixels of
// grad_output[co, pixel] * col[(tap, c), pixel]: a plain product with the pixels
// as reduction dimension (the reference's second GEMM,
// mmcv/ops/csrc/pytorch/modulated_deform_conv.cpp:227-237).  Workgroup = TILE
// output channels x TILE columns of one group over a share of the (image,
// 128-byte pixel run) steps; both operand tiles go to LDS with direct copies as
// in bwd_colgrad_kernel (grad_output is read in place: its rows are pixel
// contiguous; columns of 16-bit tensors are pixel major and transposed on the way out of LDS).  Runs of pixels past the end
// of an image read the row's last 16 bytes again; the zero padding of col cancels them.  Rows past the group's
// channels repeat its last ones and are dropped at the end.  Each share of the K
// range stores its partial tile (plain stores, rows of M contiguous);
// bwd_finish_kernel adds the shares up in a fixed order, so grad_weight does
// not vary from run to run.
// RUN: run of 16-bit columns.
template <typename E, int TILE, int RUN>
__global__ __launch_bounds__(TILE * 2, TILE == 128 ? 2 : 1) void bwd_wgrad_kernel(WGradArgs a) {
  constexpr int ES = (int)sizeof(E);
  constexpr int PXC = 16 / ES;  // pixels per 16-byte chunk
  constexpr int MB = TILE / 64;
  constexpr uint32_t kBuf = TILE * 128u;
  __shared__ uint4 As[2][TILE * 8];
  __shared__ uint4 Bs[2][TILE * 8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int frow = lane & 31, fhalf = lane >> 5;
  const int wm = wave & 1, wn = wave >> 1;
  // (all tiles of one share of the K range are neighbours: those of a row of
  // tiles share the grad_output tile, those of a column the columns tile)
  long b = xcd_work_index(a.total);
  if (b < 0) return;
  const int ct = (int)(b % a.co_tiles);
  b /= a.co_tiles;
  const int mt = (int)(b % a.m_tiles);
  b /= a.m_tiles;
  const int grp = (int)(b % a.G);
  const int split = (int)(b / a.G);

  // this lane's rows and 16-byte chunk of the copies
  long a_row[4], b_row[4];
  int chunk[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int row = (wave * 4 + c) * 8 + (lane >> 3);
    chunk[c] = (lane & 7) ^ (row & 7);
    const int co = min(ct * TILE + row, a.cout_g - 1);
    a_row[c] = ((long)grp * a.cout_g + co) * a.a_pitch;      // + n * Cout * a_pitch
    // (+ nl * taps * Cin * P_pad)
    if constexpr (sizeof(E) == 2) {
      // This lane's 16 bytes of the 2 KiB of 16 columns.  (Columns that only fill up a group may hold anything: each is
      // an accumulator column of its own, which is not looked at.)
      const int blk = wave * 4 + c;
      const int m = min(mt * TILE + (blk >> 1) * 16, a.M - 16);
      const int tap = m / a.cgp;
      const int at = (blk & 1) * 512 + lane * 8;   // element of the 64 pixels x 16 columns
      const int sub = at / (64 * RUN), in = (at - sub * 64 * RUN) ^ tr_swizzle<RUN>(sub);   // (whole fours of pixels trade places)
      b_row[c] = ((long)((grp * a.cgp + m - tap * a.cgp) / RUN + sub) * a.taps + tap) * a.P_pad * RUN + in;
    } else {
      // (the rows of the channels that only fill up a group are never written: they would hold what was there before, NaN
      // for instance, and the call then goes over its K range a second time)
      int m = min(mt * TILE + row, a.M - 1);
      const int tap = m / a.cgp;
      m = min(m, tap * a.cgp + a.rows - 1);
      b_row[c] = ((long)grp * a.M + m) * a.P_pad + chunk[c] * PXC;
    }
  }
  const uint32_t lds_a = (uint32_t)(uintptr_t)(lptr_t)(&As[0][0]) +
                         (uint32_t)__builtin_amdgcn_readfirstlane(wave) * 4096u;
  const uint32_t lds_b = (uint32_t)(uintptr_t)(lptr_t)(&Bs[0][0]) +
                         (uint32_t)__builtin_amdgcn_readfirstlane(wave) * 4096u;
  const E *gout = (const E *)a.gout, *col = (const E *)a.col;
  const int last_chunk_px = (int)a.a_pitch - PXC;  // (the pitch is a multiple of PXC)
  auto issue = [&](long wi, int buf) {
    const int nl = (int)(wi / a.ksteps);
    const int p0 = (int)(wi - (long)nl * a.ksteps) * (8 * PXC);
    const E *ga = gout + (long)(a.n0 + nl) * a.Cout * a.a_pitch;
    const E *cb = col + (long)nl * a.taps * a.Cin * a.P_pad;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int px = p0 + chunk[c] * PXC;
      copy16_global_to_lds(ga + a_row[c] + min(px, last_chunk_px), lds_a + (uint32_t)buf * kBuf + (uint32_t)c * 1024u);
      copy16_global_to_lds(cb + b_row[c] + (sizeof(E) == 2 ? (long)p0 * RUN : p0), lds_b + (uint32_t)buf * kBuf + (uint32_t)c * 1024u);
    }
  };

  // this workgroup's contiguous share of the (image, K step) range
  const long work = (long)a.nb * a.ksteps;
  const long per = (work + a.splits - 1) / a.splits;
  const long w_begin = (long)split * per, w_end = min(work, w_begin + per);
  f32x16 acc[MB][2];
  const int unused[MB] = {}, unused2[2] = {};
  auto sweep = [&](auto planes) {
    constexpr int PLANES = decltype(planes)::value;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    if (w_begin < w_end) {
      issue(w_begin, 0);
      int buf = 0;
      for (long wi = w_begin; wi < w_end; ++wi, buf ^= 1) {
        if (wi + 1 < w_end) {
          issue(wi + 1, buf ^ 1);
          asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        } else {
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        __syncthreads();
        if constexpr (sizeof(E) == 2)
          tile_products_tr<E, TILE, RUN>(acc, As[buf], Bs[buf], wm, wn, lane);
        else
          tile_products<E, TILE, PLANES>(acc, As[buf], Bs[buf], wm, wn, frow, fhalf, unused, unused2);
        __syncthreads();
      }
    }
  };
  sweep(std::integral_constant<int, 3>());
  if constexpr (sizeof(E) == 4) {
    if (__syncthreads_or(unscale(acc))) sweep(std::integral_constant<int, 0>());
  }

  // register r of lane l: A row (output channel) (r/4)*8 + (l/32)*4 + r%4 of the block, B row (column row) l%32
  float *part = a.part + ((long)split * a.G + grp) * a.cout_g * a.M;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      const int m = mt * TILE + wn * 64 + nb * 32 + frow;
      if (m >= a.M) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int co = ct * TILE + wm * (TILE / 2) + mb * 32 + (r >> 2) * 8 + fhalf * 4 + (r & 3);
        if (co < a.cout_g) {
          float *p = part + (long)co * a.M + m;
          *p = a.accumulate ? *p + acc[mb][nb][r] : acc[mb][nb][r];
        }
      }
    }
}

}  // namespace mdcn
