// Backward, data side, of 16-bit tensors in one kernel: the column gradient
// d[pixel, (tap, c)] = sum_co grad_output[co, pixel] * weight[co, c, tap] comes
// out of the matrix cores into registers and is used there -- for the offset and
// mask gradients, for grad_input through a window in LDS, beside the sampling of
// the forward's columns for the weight gradient (the reference's first GEMM and
// its three element-wise kernels, mmcv/ops/csrc/pytorch/modulated_deform_conv.cpp:199-206,
// cpu/modulated_deform_conv.cpp:34-107,170-320).  d never exists in memory and is
// never rounded to 16 bits.
#pragma once

#include "mdcn_backward_gemm.h"

namespace mdcn {

constexpr int kBfThreads = 512, kBfWaves = kBfThreads / 64;
constexpr int kBfItems = (kBwdTapsMax + 1) / 2;     // pairs of taps
constexpr int kBfK = 128;                           // of K at a time
// Blocks of products of a pass of CH channels, bytes of LDS of a stage of weights (32 rows a block, kBfK of K; two stages are
// held) and pixels of the window beside them.
constexpr int bf_blocks(int ch) { return (kBfItems * ch + 15) / 16; }
constexpr int bf_stage_bytes(int ch) { return bf_blocks(ch) * 32 * kBfK * 2; }
constexpr int kBfLdsBytes = 163072;
constexpr int bf_window_px(int ch) { return (kBfLdsBytes - 2 * bf_stage_bytes(ch)) / (4 * ch); }
constexpr long kBfPlaneMax = 1L << 24;              // pixels of a plane, its zero border included
constexpr float kRoundMagic = 12582912.0f;          // 1.5 * 2^23: adding it leaves an integer in the mantissa
constexpr uint32_t kRoundBits = 0x4B400000u;        // ... on top of these bits

struct BwdFusedArgs {
  Geom g;
  const void *xt;   // zero-bordered input copy in 32-byte records [N][Cin / 16][H + 2][W + 2][16]
  const void *gT;   // grad_output, pixel major [N][Cout / 64][P][64]
  const void *wT;   // [G][chunk of kBfK output channels][taps * cin_g][of the chunk], row tap * cin_g + channel
  OffMaskView om;   // (dense tensors: logit is kMaskPlain or kMaskNone)
  float *gin32;
  void *goff;
  void *gmask;      // null when unmodulated
  void *col;        // columns of the pass [image][Cin / CH][taps][P_pad][CH], or null: CH the kernel's
  long P_pad;
  int tw_log;       // a tile of 256 pixels is 1 << tw_log wide (16 or 32)
  int tiles_x, tiles_y;
  ScatterWindow win, win_far;   // (win_far.WH = 0: none)
  const uint32_t *far;          // counts of sampled offsets beyond win's margin; above far_min in all, win_far is used
  int n_far;
  uint32_t far_min;
  int n0;           // first image of the pass
  FusedSchedule sched;
  float *part;      // [workgroup][3 taps][256]: sums of the offset (y and x of a tap) and mask gradients of a share of a tile
};

// The largest value of a wavefront's lanes.
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
  // (within rows of 16 lanes, rotated by 8, 4, 2 and 1)
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x128, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x124, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x122, 0xf, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x121, 0xf, 0xf, false));
  return max(max((uint32_t)__builtin_amdgcn_readlane((int)v, 0), (uint32_t)__builtin_amdgcn_readlane((int)v, 16)),
             max((uint32_t)__builtin_amdgcn_readlane((int)v, 32), (uint32_t)__builtin_amdgcn_readlane((int)v, 48)));
}

// One tile of 256 output pixels (tile b), channels [c_first, c_last) of its deformable group; part: where the sums of a share go,
// or null.  Eight wavefronts, 32 pixels each.  Per pass of CH channels:
//
// Products: blocks of 32 rows of weights -- two taps of 16 channels, or four of 8 -- times the wavefront's 32 pixels, K in chunks
// of 128.  The weights of a pass go to LDS for all wavefronts (two chunks; copied during the scatter of the pass before), rows in
// an order that gives a lane consecutive channels of one (pixel, tap) of the result.  grad_output comes in registers, 16
// bytes a lane and 16 of K, each half chunk loaded into the registers of the one before it, a pass's first during the last tap of the
// scatter before it.  These loads take 2 to 5 thousand clocks (a round's tiles have more grad_output than an L2 holds), so no
// branch and no wait for something else lies between them and their products.  More than 256 output channels: a chunk's copies are
// on their way during the products of the one before.
// Scatter: a lane takes its pixel's taps of one parity, 8 channels at a time, their corners loaded two such units ahead.
// Every wait among its items is for loads that are due: whatever the compiler keeps in scratch or fetches from the argument
// block again there makes it wait for all loads, or all LDS adds, under way (the kernel took 2.1 ms in the shape below with either,
// 1.35 without).  Hence the asm statements without text below: they hold a sum where it is, and a value in its register.
// Window: 32-bit fixed point in LDS.  Its scale is the pass's own: from the largest |d| of its products over the tile, the largest
// mask value and the number of adds the busiest entry sees, so that no contribution leaves 2^21 and no sum of them 2^30.  The
// first decides where no entry sees more than 512, and the quantum is then 2^-20 or 2^-21 of the largest contribution there could
// be.  Where the largest |d * mask| of a sample gives three bits or more, the scale is from that instead: else one large gradient
// under a small mask takes bits from its whole tile (fp16, one pixel of a mask of 0 and 1 000 times the gradient: error of grad_input
// 3.3e-3 of its norm, so 2.1e-4, its one rounding).  Below three bits (inputs whose large gradients and open masks meet somewhere in a
// tile) results stay those of the first scale, bit for bit.  The second costs training calls of N=16 256 channels 100x152 in bf16 0.3 %
// (2 377 -> 2 383 us).  (Bounds of |d| from norms of grad_output and weights instead: 0.4 % less there, 2 % more for N=8 512 channels 25x42 in
// fp16.  But such a scale goes by gradients that the weights do not carry on: fp16, 256 output channels, one of them without weights and with 300 times the gradient: error of grad_input
// 8.6e-4 of its norm, where its one rounding is 2.1e-4 and this stays at that.)
// What is added to an entry is the bit pattern of fmaf(weight, d, 1.5 * 2^23), for two channels at
// once: every tap of every pixel adds to four entries, the same ones for all channels, so the number of adds an entry has
// seen is known from a count made once per tile, and what the patterns hold beside the integers is subtracted when the entry is
// read.  (Two instructions per channel and corner, where taking it off each contribution was six per two.)  In a pass where d or
// the mask is not finite, or so small or large that no scale fits, nothing goes through the window.
// Samples beyond the window are added to memory one at a time, a lane for every channel and corner.  (Backward of fp16 N=8 256
// channels 50x84: 0.42 ms, with one infinity in grad_output -- no window in 1 tile's passes -- 2.1; where every lane added its own samples 7.3.)
//
// bf16, N=16, 256 -> 256 channels, 100x152: 1.29 ms for what took 0.52 (column gradient to memory) + 1.50 (scatter kernel reading
// it); a pass takes a CU 40 thousand clocks: 25 scatter (VALU busy in 16, LDS adds 18), 6 products (MFMA 5), 7 flush, the rest
// waits at the barriers.  fp16 without modulation, N=8, 512 -> 512 channels, 25x42: 0.17 ms.  (Whole training calls with
// grad_output loaded within branches and behind the scatter, the argument block kept as it was loaded, 64-bit addresses in each lane and the
// largest of a pass found with integers, two instructions a value, took 0.4 to 4 % longer, by the card: on four of them, before / now, us,
// 2 333 / 2 246, 2 349 / 2 261, 2 335 / 2 277, 2 414 / 2 386, and 397 / 364, 363 / 344.)
// No scratch but with more than 256 output channels and 16 of the input's a pass: 20 (bf16) and 8 bytes (fp16), read at a tile's start.
template <typename E, int CH, int RUN, bool DEEP>
__device__ __forceinline__ void fused_tile(const BwdFusedArgs &a, const ScatterWindow &wd, int b, int c_first, int c_last, float *part, uint4 *lds,
                                           float *red) {
  using TR = ElemTraits<E>;
  constexpr int NP = CH / 2;
  constexpr int PLANE = bf_window_px(CH);
  constexpr int PER = 16 / CH;                        // items per block of products
  constexpr int U = CH / 8;                           // units of 8 channels an item has
  constexpr int LA = 2 / U;                           // items between a unit and the loads for it
  constexpr int kBlocks = bf_blocks(CH);
  constexpr int kStage = bf_stage_bytes(CH);
  constexpr int kSlots = (PLANE + kBfThreads - 1) / kBfThreads;
  uint4 *wst = lds;
  unsigned long long *win = (unsigned long long *)(lds + 2 * kStage / 16);
  // What a pass reads of the argument block, a scalar each: as parts of its sixteen-register loads they would be put away and fetched
  // back sixteen at a time (366 of the scatter's 2 679 VALU instructions).
  Geom g = a.g;
  auto apart = [](const void *p) {
    auto q = (const __attribute__((address_space(1))) unsigned char *)p;   // (or nothing would say that it is global memory)
    asm volatile("" : "+s"(q));
    return (const unsigned char *)q;
  };
  const unsigned char *wt = apart(a.wT), *gt = apart(a.gT), *xt = apart(a.xt);
  unsigned char *cols = (unsigned char *)apart(a.col);
  float *gin = (float *)apart(a.gin32);
  uint32_t col_px = (uint32_t)a.P_pad;
  asm volatile("" : "+s"(g.H), "+s"(g.W), "+s"(g.Wp), "+s"(g.Cin), "+s"(g.cin_g), "+s"(g.cout_g), "+s"(g.taps), "+s"(g.G), "+s"(col_px));
  const long plane_out = (long)g.Ho * g.Wo, plane_in = (long)g.H * g.W, slab_px = (long)g.Hp * g.Wp;
  int tid = threadIdx.x, lane = tid & 63, frow = lane & 31, half = lane >> 5;
  asm volatile("" : "+v"(lane), "+v"(frow), "+v"(half), "+v"(tid));   // (or addresses of all copies are kept over the tiles, in scratch)
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tx = b % a.tiles_x;
  b /= a.tiles_x;
  const int ty = b % a.tiles_y;
  b /= a.tiles_y;
  const int dgi = b % g.DG, nl = b / g.DG;
  const int n = a.n0 + nl;
  const int TW = 1 << a.tw_log, TH = 256 >> a.tw_log;
  const int ho = ty * TH + ((wave * 32 + frow) >> a.tw_log), wo = tx * TW + (frow & (TW - 1));
  const bool valid = ho < g.Ho && wo < g.Wo;
  // (lanes past the image: any pixel of it.  Addresses are a scalar base and a lane's 32 bits wherever a pass needs them: planes have
  // fewer than kBfPlaneMax pixels.)
  const uint32_t pix = (uint32_t)(min(ho, g.Ho - 1) * g.Wo + min(wo, g.Wo - 1));
  const int wy0 = ty * TH * g.sh - g.ph - wd.R, wx0 = tx * TW * g.sw - g.pw - wd.R;
  int WW = wd.WW, WH = wd.WH;
  asm volatile("" : "+s"(WW), "+s"(WH));   // (kept: fetched again for every use, each wait for one would be for all LDS adds)
  const int win_px = WH * WW;
  const uint32_t inv_ww = (1u << 22) / (uint32_t)WW + 1u;   // k / WW = k * inv_ww >> 22 for every pixel k of a window

  // This lane's taps 2 i + half: offsets, mask and place in the kernel
  uint32_t t_off[kBfItems], t_m[kBfItems];   // dy | dx << 16; mask | row << 16 | column << 24, a row of 255: no such tap
  float *lone = red + 5 * kBfWaves + wave * 16;   // of this wavefront
  const int items = (g.taps + 1) / 2, blocks = (items + PER - 1) / PER;

  // (zero where nothing is sampled, once the tile has begun)
  auto mask_of = [&](int i) { return to_f32(__builtin_bit_cast(E, (uint16_t)t_m[i])); };
  auto has_tap = [&](int i) { return ((t_m[i] >> 16) & 255u) != 255u; };
  int base_y = ho * g.sh - g.ph, base_x = wo * g.sw - g.pw;
  struct Place {
    int y0, x0;
    float ly, lx;
    bool inside;
  };
  auto place = [&](int i) {
    Place p;
    float dy, dx;
    TR::unpack2(t_off[i], dy, dx);
    const int row = (int)(t_m[i] >> 16) & 255;
    const float py = (float)(base_y + row) + dy;
    const float px = (float)(base_x + (int)(t_m[i] >> 24)) + dx;
    p.inside = valid && row != 255 && py > -1.0f && px > -1.0f && py < (float)g.H && px < (float)g.W;
    const float fy = floorf(py), fx = floorf(px);
    p.y0 = p.inside ? (int)fy : -1;
    // (nothing sampled: the right border of the row above the image, whose next pixel is the left one of the image's first: four
    // zeros.  At -1 the last corner would be the image's first pixel, and d times it an infinity where neither is.)
    p.x0 = p.inside ? (int)fx : g.W;
    p.ly = p.inside ? py - fy : 0.0f;
    p.lx = p.inside ? px - fx : 0.0f;
    return p;
  };

  // Passes of CH channels each.  (The copies hold the tensors' own channels; a pass lies in one group.)
  const int c_begin = dgi * g.ch_per_dg + c_first, c_end = dgi * g.ch_per_dg + c_last;
  auto group_of = [&](int c0) { return g.G == 1 ? 0 : c0 / g.cin_g; };

  // Copies of a stage of weights: 32 rows a block, 128 (or what is left: 64) of K, pieces of 16 bytes swizzled by the row.  Chunk kh of K goes to buffer
  // kh % 2.
  const int nkh = (g.cout_g + kBfK - 1) / kBfK;
  const uint32_t lds_w = (uint32_t)(uintptr_t)(lptr_t)wst + (uint32_t)wave * 1024u;
  const uint32_t rows_g = (uint32_t)(g.taps * g.cin_g);
  auto issue = [&](int c0, int kh) {
    const int sh = g.cout_g - kh * kBfK >= kBfK ? 4 : 3;
    const int grp = group_of(c0);
    const uint32_t row_bytes = 16u << sh;
    const unsigned char *base = wt + ((long)grp * g.cout_g + kh * kBfK) * rows_g * 2 + (long)(c0 - grp * g.cin_g) * row_bytes;
    const int copies = blocks << (sh - 1);   // of 1 KiB
    // Copies are 32 or 64 rows apart, so all of a lane's are the same row of their blocks: result register 4 * r8 + r4 of the lanes of half hh
    const uint32_t row0 = (uint32_t)(wave * 64 + lane) >> sh, s = (uint32_t)lane & ((1u << sh) - 1u);
    const uint32_t r8 = (row0 >> 3) & 3u, hh = (row0 >> 2) & 1u, r4 = row0 & 3u;
    const uint32_t ch = 4 * (PER == 2 ? r8 & 1 : r8) + r4, at = ch * row_bytes + ((s ^ (row0 & 7u)) * 16u);
    const uint32_t tap0 = PER * 2 * (row0 >> 5) + (PER == 2 ? 2 * (r8 >> 1) : 0) + hh, tap_bytes = (uint32_t)g.cin_g * row_bytes;
    const uint32_t lds = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds_w + (uint32_t)(kh & 1) * (uint32_t)kStage));
#pragma unroll
    for (int c = 0; c < 8 * kBlocks / kBfWaves; ++c) {
      if (wave + kBfWaves * c < copies) {
        const uint32_t tap = min(tap0 + (uint32_t)(PER * 2 * c) * (sh == 4 ? 1u : 2u), (uint32_t)g.taps - 1u);
        copy16_global_to_lds(base + (tap * tap_bytes + at), lds + (uint32_t)c * (kBfWaves * 1024u));
      }
    }
  };
  // This lane's grad_output of chunk kh of K, the products' second operand: j-th 16 of it (j < 4, or < 8 where the chunk is whole)
  const unsigned char *gbase = gt + (long)n * (g.Cout / 64) * plane_out * 128;
  auto whole_chunk = [&](int kh) { return g.cout_g - kh * kBfK >= kBfK; };
  uint4 gf[8];
  // (the second half of a half chunk is the first once more: read, and not used)
  auto load_g_half = [&](int grp, int kh, int s) {
    const unsigned char *p = gbase + ((long)(grp * (g.cout_g / 64) + kh * 2 + (whole_chunk(kh) ? s : 0)) * plane_out) * 128;
    uint32_t at = pix * 128u + (uint32_t)half * 16u;
    asm volatile("" : "+v"(at));
#pragma unroll
    for (int j = 0; j < 4; ++j) gf[4 * s + j] = *(const uint4 *)(p + j * 32 + at);
  };
  // Whether a pass's first chunk has its second half loaded.  Passes of 8 channels leave it out with 64 output channels (bf16 training calls,
  // loaded / left out, us: N=4 64 channels, 8 deformable groups, 120x160 304 / 296, N=8 96x128 356 / 345).  The branch costs those of 128 output
  // channels that take it and load all the same (N=4 128, 16 deformable groups, 120x160 610 / 620, 90x150 469 / 479); with 16 channels a pass
  // it would be 44 reloads of spilled registers, more than it saves (N=4 256 channels 50x84: 260 / 269).
  auto first_second = [&]() { return CH == 16 || whole_chunk(0); };
  // the first two stages of a pass
  auto issue_first = [&](int c0) {
    issue(c0, 0);
    if (nkh > 1) issue(c0, 1);
  };
  issue_first(c_begin);
  {
    const E *off = (const E *)a.om.off + (long)n * a.om.off_n + (long)pix * a.om.off_px + (long)(dgi * 2 * g.taps) * a.om.off_ch;
    const E *msk = (const E *)a.om.msk + (long)n * a.om.msk_n + (long)pix * a.om.msk_px + (long)(dgi * g.taps) * a.om.msk_ch;
    int row = 0, col = 0;
    auto tap_at = [&](int tap) {   // (one after the other)
      const uint32_t at = tap < g.taps ? (uint32_t)(row * g.dh) | (uint32_t)(col * g.dw) << 8 : 255u;
      if (++col == g.kw) {
        col = 0;
        ++row;
      }
      return at;
    };
#pragma unroll
    for (int i = 0; i < kBfItems; ++i) {
      const int tap = 2 * i + half, tc = min(tap, g.taps - 1);
      const uint32_t at0 = tap_at(2 * i), at1 = tap_at(2 * i + 1);
      t_off[i] = (uint32_t)__builtin_bit_cast(uint16_t, off[(long)(2 * tc) * a.om.off_ch]) |
                 (uint32_t)__builtin_bit_cast(uint16_t, off[(long)(2 * tc + 1) * a.om.off_ch]) << 16;
      t_m[i] = (uint32_t)__builtin_bit_cast(uint16_t, msk[(long)tc * a.om.msk_ch]) | (half ? at1 : at0) << 16;
    }
  }

  // (The barrier ends the tile before: nobody is at the window any more.)
  __syncthreads();
  load_g_half(group_of(c_begin), 0, 0);
  if (first_second()) load_g_half(group_of(c_begin), 0, 1);
  // (the counts of adds go where the window will be)
  for (int i = tid; i < win_px; i += kBfThreads) ((uint32_t *)win)[i] = 0u;
  // Largest mask value and the sum of all of the tile's; then a mask of zero where nothing is sampled
  {
    float top = 0.0f, sum = 0.0f;
#pragma unroll
    for (int i = 0; i < kBfItems; ++i) {
      const uint32_t one = (uint32_t)__builtin_bit_cast(uint16_t, from_f32<E>(1.0f));
      const uint32_t m = a.om.logit == kMaskNone ? one : t_m[i] & 0xffffu;   // (1: unmodulated)
      const float v = valid && has_tap(i) ? fabsf(to_f32(__builtin_bit_cast(E, (uint16_t)m))) : 0.0f;
      top = fmaxf(top, v);   // (NaN is left out: where it is sampled, the largest |d * mask| has it)
      sum += v;
      t_m[i] = (t_m[i] & 0xffff0000u) | (place(i).inside ? m : 0u);
      asm volatile("" : "+v"(t_off[i]), "+v"(t_m[i]));   // (here and now, or the halves they are made of are kept)
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    const uint32_t bits = wave_max(__float_as_uint(top));
    if (lane == 0) {
      red[wave] = __uint_as_float(bits);
      red[kBfWaves + wave] = sum;
    }
  }
  __syncthreads();
  auto window_at = [&](const Place &p, bool &in_win) {
    const int ry = p.y0 - wy0, rx = p.x0 - wx0;
    in_win = ry >= 0 && ry + 1 < WH && rx >= 0 && rx + 1 < WW;
    // a lane with nothing for the window adds its zeros at an entry of its own
    return p.inside && in_win ? ry * WW + rx : lane;
  };
  // How many adds the window pixels that this thread flushes (tid, tid + 512, ...) see in a pass, 16 bits each
  uint32_t adds[(kSlots + 1) / 2];
  // Largest mask value, a bound on the sum of those of an entry, largest number of adds.  (In LDS: as scalars of the whole tile they cost
  // registers that are then short elsewhere.)
  float *tops = red + (5 + 16) * kBfWaves;
  {
#pragma unroll
    for (int i = 0; i < kBfItems; ++i) {
      if (i < items) {
        bool in_win;
        uint32_t *c = (uint32_t *)win + window_at(place(i), in_win);
        atomicAdd(c, 1u);
        atomicAdd(c + 1, 1u);
        atomicAdd(c + WW, 1u);
        atomicAdd(c + WW + 1, 1u);
      }
    }
    __syncthreads();
    uint32_t most = 0u;
#pragma unroll
    for (int j = 0; j < kSlots; ++j) {
      const int q = tid + kBfThreads * j;
      const uint32_t c = q < win_px ? ((const uint32_t *)win)[q] : 0u;
      adds[j / 2] = j % 2 ? adds[j / 2] | c << 16 : c;
      most = max(most, c);
    }
    most = wave_max(most);
    if (lane == 0) red[2 * kBfWaves + wave] = __uint_as_float(most);
    __syncthreads();
    float top = 0.0f, sum = 0.0f;
    most = 0u;
#pragma unroll
    for (int w = 0; w < kBfWaves; ++w) {
      top = fmaxf(top, red[w]);
      sum += red[kBfWaves + w];
      most = max(most, __float_as_uint(red[2 * kBfWaves + w]));
    }
    if (tid == 0) {
      tops[0] = top;
      tops[1] = fminf(sum, (float)most * top);
      tops[2] = (float)most;
    }
    for (int i = tid; i < PLANE * NP / 2; i += kBfThreads) ((uint4 *)win)[i] = make_uint4(0u, 0u, 0u, 0u);
  }
  // The scale of the pass in the window, and whether there is one
  bool fits = false;
  float scale = 1.0f, inv_scale = 1.0f;
  // Corners of 8 channels of an item, loaded one unit of work ahead: first channel c0 of the pass, half h of its channels
  struct Corners {
    VecCh<E, 8> r00, r01, r10, r11;
  };
  auto fetch = [&](int c0, const Place &p, int h, Corners &s) {
    // corners outside the image read the copy's zero border
    const unsigned char *xp = xt + (((long)n * (g.Cin / 16) + c0 / 16) * slab_px) * 32 + (c0 % 16) * 2 + h * 16;
    uint32_t top = (uint32_t)((p.y0 + 1) * g.Wp + (p.x0 + 1)) * 32u, bot = top + (uint32_t)g.Wp * 32u;
    asm volatile("" : "+v"(top), "+v"(bot));   // (these beside a scalar base, and no sums of the two)
    s.r00.load((const E *)(xp + top));
    s.r01.load((const E *)(xp + 32 + top));
    s.r10.load((const E *)(xp + bot));
    s.r11.load((const E *)(xp + 32 + bot));
  };

  float acc_m[kBfItems], acc_y[kBfItems], acc_x[kBfItems];
#pragma unroll
  for (int i = 0; i < kBfItems; ++i) acc_m[i] = acc_y[i] = acc_x[i] = 0.0f;

  // every copy of a stage has landed, and every wavefront is past whatever it did before
  auto settle = [&]() {
    asm volatile("s_waitcnt vmcnt(0) ; lds-copies" ::: "memory");
    __syncthreads();
  };
  f32x16 d[kBlocks];
  // Products of half s of chunk kh of K.
  auto products_half = [&](int kh, int s, int pitch) {
    const uint4 *w0 = wst + (kh & 1) * (kStage / 16) + frow * pitch;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint4 *wj = w0 + 8 * s + ((2 * j + half) ^ (frow & 7));
      uint4 f[kBlocks];
#pragma unroll
      for (int blk = 0; blk < kBlocks; ++blk) f[blk] = wj[blk * 32 * pitch];
#pragma unroll
      for (int blk = 0; blk < kBlocks; ++blk) TR::mma(d[blk], f[blk], gf[4 * s + j]);
    }
    // fragments are read three products ahead of theirs
    __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
    for (int j = 0; j < 4 * kBlocks - 3; ++j) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
  };
  // All of a pass's products; the first two stages are in LDS.
  auto products_of = [&](int c0) {
    const int grp = group_of(c0);
#pragma unroll
    for (int blk = 0; blk < kBlocks; ++blk)
#pragma unroll
      for (int r = 0; r < 16; ++r) d[blk][r] = 0.0f;
    // A chunk's grad_output goes into the registers of what has been used.  (No branch between a load and its product: the
    // waits are for the half chunk that is due, with the next one under way.)
    auto chunk_and_load = [&](int kh, auto between) {
      products_half(kh, 0, 16);
      load_g_half(grp, kh + 1, 0);
      products_half(kh, 1, 16);
      between();
      load_g_half(grp, kh + 1, 1);
    };
    auto last_chunk = [&](int kh) {
      products_half(kh, 0, whole_chunk(kh) ? 16 : 8);
      if (whole_chunk(kh)) products_half(kh, 1, 16);
    };
    if constexpr (DEEP) {
      chunk_and_load(0, [] { __syncthreads(); });   // (nobody reads the first stage any more)
      issue(c0, 2);
      for (int kh = 1; kh + 1 < nkh; ++kh) {
        chunk_and_load(kh, settle);   // (every wavefront is past this stage, and the next one has landed)
        if (kh + 2 < nkh) issue(c0, kh + 2);
      }
      last_chunk(nkh - 1);
    } else if (nkh > 1) {
      chunk_and_load(0, [] {});
      last_chunk(1);
    } else {
      last_chunk(0);
    }
    // (No load is under way here.  The compiler, which follows each branch above by itself, is told so, or it waits for
    // whatever is under way at the next use of these registers.)
#pragma unroll
    for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(gf[j].x), "+v"(gf[j].y), "+v"(gf[j].z), "+v"(gf[j].w));
  };
  // Leaves the largest |d| and the largest |d * mask| of this wavefront, as bits (NaN above all), where the others find them behind a
  // barrier.
  auto put_largest = [&]() {
    float largest_d = 0.0f, largest = 0.0f;
#pragma unroll
    for (int i = 0; i < kBfItems; ++i) {
      float c = 0.0f;
#pragma unroll
      for (int k = 0; k < CH; ++k) c = __builtin_elementwise_maximum(c, fabsf(d[i / PER][(i % PER) * CH + k]));
      largest_d = __builtin_elementwise_maximum(largest_d, i < items ? c : 0.0f);
      // (what is not finite makes this NaN where the mask is zero)
      c *= mask_of(i);
      largest = __builtin_elementwise_maximum(largest, i < items ? fabsf(c) : 0.0f);
    }
    const uint32_t bits_d = wave_max(__float_as_uint(largest_d) & 0x7fffffffu);
    const uint32_t bits = wave_max(__float_as_uint(largest) & 0x7fffffffu);
    if (lane == 0) {
      red[3 * kBfWaves + wave] = __uint_as_float(bits_d);
      red[4 * kBfWaves + wave] = __uint_as_float(bits);
    }
  };
  auto take_scale = [&]() {
    // (the waves' eight words of either, a lane each, and the largest of eight lanes: sixteen reads at once are more registers than there
    // are here)
    uint32_t bits = __float_as_uint(red[3 * kBfWaves + (lane & 15)]);
    bits = max(bits, (uint32_t)__builtin_amdgcn_mov_dpp((int)bits, 0xB1, 0xf, 0xf, true));    // of two
    bits = max(bits, (uint32_t)__builtin_amdgcn_mov_dpp((int)bits, 0x4E, 0xf, 0xf, true));    // of four
    bits = max(bits, (uint32_t)__builtin_amdgcn_mov_dpp((int)bits, 0x141, 0xf, 0xf, true));   // of eight
    const float dmax = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)bits, 0));
    const float one = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)bits, 8));
    // exponent of a scale, from a bound of a sum and one of a contribution
    auto exponent = [](float all, float one) {   // (positive and finite where it counts: frexp's exponent is ilogb's + 1)
      const int e = min(30 - __builtin_amdgcn_frexp_expf(all), one > 0.0f ? 21 - __builtin_amdgcn_frexp_expf(one) : 120);
      return (all > 0.0f && all < 3.0e38f) ? e : 0;
    };
    const float mask_top = tops[0];
    const float apart = dmax * tops[1], all = one * tops[2];
    const int e_apart = exponent(apart, dmax * mask_top), e_one = exponent(all, one);
    const int e = !(apart < 3.0e38f) || e_one >= e_apart + 3 ? e_one : e_apart;
    scale = __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(ldexpf(1.0f, min(120, e)))));
    inv_scale = 1.0f / scale;
    fits = __builtin_amdgcn_readfirstlane(all < 3.0e38f && e <= 120 && mask_top * scale < 3.0e38f) != 0;  // (false for NaN)
  };
  // Adds what the window holds of the CH channels from cf on to grad_input, and clears it.
  auto flush = [&](int cf) {
    float *gplane = gin + ((long)n * g.Cin + cf) * plane_in;
#pragma unroll
    for (int j = 0; j < kSlots; ++j) {
      const uint32_t seen = j % 2 ? adds[j / 2] >> 16 : adds[j / 2] & 0xffffu;
      if (seen != 0u) {
        const int k = tid + kBfThreads * j, r = (int)(((uint32_t)k * inv_ww) >> 22);
        const int y = wy0 + r, x = wx0 + k - r * WW;
        unsigned long long *e = win + k;
        unsigned long long v[NP];
#pragma unroll
        for (int cp = 0; cp < NP; ++cp) v[cp] = e[cp * PLANE];
#pragma unroll
        for (int cp = 0; cp < NP; ++cp) e[cp * PLANE] = 0ull;
        if (fits && y >= 0 && y < g.H && x >= 0 && x < g.W) {
          const unsigned long long bias = (unsigned long long)seen * kRoundBits;
          uint32_t at = (uint32_t)(y * g.W + x) * 4u;
          long step = plane_in;
          asm volatile("" : "+s"(step));   // (or its multiples are kept, and put away)
          auto into = [&](int c) {
            asm volatile("" : "+v"(at));   // (a plane's address stays a scalar, and this beside it)
            return (float *)((unsigned char *)(gplane + c * step) + at);
          };
#pragma unroll
          for (int cp = 0; cp < NP; ++cp) {
            const long long s = (long long)(v[cp] - (bias + (bias << 32)));
            const int lo = (int)(uint32_t)s, hi = (int)((s - (long long)lo) >> 32);
            unsafeAtomicAdd(into(2 * cp), (float)lo * inv_scale);
            unsafeAtomicAdd(into(2 * cp + 1), (float)hi * inv_scale);
          }
        }
      }
    }
  };
  settle();
  for (int c0 = c_begin; c0 < c_end; c0 += CH) {
    // (Opaque to the optimiser: it would otherwise move what follows from these in every pass -- positions, addresses of
    // all stages -- out of this loop, and spill it.)
#pragma unroll
    for (int i = 0; i < kBfItems; ++i) asm volatile("" : "+v"(t_off[i]), "+v"(t_m[i]));
#pragma unroll
    for (int j = 0; j < (kSlots + 1) / 2; ++j) asm volatile("" : "+v"(adds[j]));
    asm volatile("" : "+v"(lane), "+v"(frow), "+v"(half), "+v"(tid), "+v"(base_y), "+v"(base_x));
    products_of(c0);
    put_largest();
    Place p[LA + 1];
#pragma unroll
    for (int i = 0; i < LA; ++i) p[i] = place(i);
    Corners q[3];
    fetch(c0, p[0], 0, q[0]);
    fetch(c0, p[LA - 1], U - 1, q[1]);
    if (c0 > c_begin) flush(c0 - CH);   // (behind these loads: a wavefront's loads wait for every add in front of them)
    __syncthreads();   // the window is zero and the stages are free
    if (c0 + CH < c_end) issue_first(c0 + CH);
    take_scale();
    const int grp_next = group_of(min(c0 + CH, c_end - 1));
    __builtin_amdgcn_sched_barrier(0);
    unsigned char *cbase = cols + (((long)nl * (g.Cin / RUN) + c0 / RUN) * g.taps * col_px * RUN + c0 % RUN) * 2;
    uint32_t cat = ((uint32_t)half * col_px + pix) * (RUN * 2u);
#pragma unroll
    for (int i = 0; i < kBfItems; ++i) {
      // The next pass's grad_output, where the products were that are through.  (Not within the branch: the registers
      // would be kept for the way round it.)
      if (i == kBfItems - 3 + U) {
        load_g_half(grp_next, 0, 0);
        if (first_second()) load_g_half(grp_next, 0, 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (i < items) {
        Place &next = p[(i + LA) % (LA + 1)];
        const Place c = p[i % (LA + 1)];
        if (i + LA < kBfItems) next = place(i + LA);
        const float ly = c.ly, lx = c.lx, hy = 1.0f - ly, hx = 1.0f - lx;
        const float m = mask_of(i);
        const int y0 = c.y0, x0 = c.x0, y1 = y0 + 1, x1 = x0 + 1;
        const bool ok00 = y0 >= 0 && x0 >= 0, ok01 = y0 >= 0 && x1 <= g.W - 1;
        const bool ok10 = y1 <= g.H - 1 && x0 >= 0, ok11 = y1 <= g.H - 1 && x1 <= g.W - 1;
        const float w00 = hy * hx, w01 = hy * lx, w10 = ly * hx, w11 = ly * lx;
        bool in_win;
        const int wbase = window_at(c, in_win);
        in_win = in_win && fits;
        const bool to_win = c.inside && in_win;
        const float s00 = (to_win && ok00) ? w00 : 0.0f, s01 = (to_win && ok01) ? w01 : 0.0f;
        const float s10 = (to_win && ok10) ? w10 : 0.0f, s11 = (to_win && ok11) ? w11 : 0.0f;
        const float mts = m * scale;
        const float v00 = m * w00, v01 = m * w01, v10 = m * w10, v11 = m * w11;
        float S00 = 0.0f, S01 = 0.0f, S10 = 0.0f, S11 = 0.0f;
        // (What a pass without a scale adds to the window is dropped by the flush.)
        if (!fits) {  // (then d may be anything where nothing is sampled; otherwise it is finite and meets zeros there)
#pragma unroll
          for (int k = 0; k < CH; ++k)
            d[i / PER][(i % PER) * CH + k] = c.inside ? d[i / PER][(i % PER) * CH + k] : 0.0f;
        }
#pragma unroll
        for (int h = 0; h < U; ++h) {
          const Corners &cur = q[(i * U + h) % 3];
          if (i + LA < kBfItems) fetch(c0, next, h, q[(i * U + h + 2) % 3]);
          unsigned long long *wp0 = win + h * 4 * PLANE + wbase, *wp1 = wp0 + WW;
          uint32_t cv[4];
#pragma unroll
          for (int cp = 0; cp < 4; ++cp) {
            const float d0 = d[i / PER][(i % PER) * CH + h * 8 + 2 * cp], d1 = d[i / PER][(i % PER) * CH + h * 8 + 2 * cp + 1];
            float q00[2], q01[2], q10[2], q11[2];
            cur.r00.pair(cp, q00[0], q00[1]);
            cur.r01.pair(cp, q01[0], q01[1]);
            cur.r10.pair(cp, q10[0], q10[1]);
            cur.r11.pair(cp, q11[0], q11[1]);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const float dd = e ? d1 : d0;
              S00 = fmaf(dd, q00[e], S00);
              S01 = fmaf(dd, q01[e], S01);
              S10 = fmaf(dd, q10[e], S10);
              S11 = fmaf(dd, q11[e], S11);
            }
            auto column = [&](int e) { return fmaf(v00, q00[e], fmaf(v01, q01[e], fmaf(v10, q10[e], v11 * q11[e]))); };
            cv[cp] = TR::pack2(column(0), column(1));
            // (Here and now: the optimiser would move these sums behind the branches below and keep all corners until then.)
            asm volatile("" : "+v"(cv[cp]), "+v"(S00), "+v"(S01), "+v"(S10), "+v"(S11));
            const float tl = d0 * mts, th = d1 * mts;
            auto entry = [&](float w) {
              return (unsigned long long)__float_as_uint(fmaf(w, tl, kRoundMagic)) |
                     (unsigned long long)__float_as_uint(fmaf(w, th, kRoundMagic)) << 32;
            };
            atomicAdd(wp0 + cp * PLANE, entry(s00));
            atomicAdd(wp0 + cp * PLANE + 1, entry(s01));
            atomicAdd(wp1 + cp * PLANE, entry(s10));
            atomicAdd(wp1 + cp * PLANE + 1, entry(s11));
            __builtin_amdgcn_sched_barrier(0);
          }
          asm volatile("" : "+v"(cat));
          if (cols && valid && has_tap(i))
            *(uint4 *)(cbase + (long)(2 * i) * col_px * (RUN * 2) + h * 16 + cat) = make_uint4(cv[0], cv[1], cv[2], cv[3]);
          __builtin_amdgcn_sched_barrier(0);
        }
        acc_m[i] += w00 * S00 + w01 * S01 + w10 * S10 + w11 * S11;
        acc_y[i] += m * (hx * (S10 - S00) + lx * (S11 - S01));
        acc_x[i] += m * (hy * (S01 - S00) + ly * (S11 - S10));
        // Samples beyond the window go to memory directly, one at a time: a lane for every channel and corner.
        for (unsigned long long rest = __ballot(c.inside && !in_win); rest != 0ull; rest &= rest - 1ull) {
          const int l = __ffsll((long long)rest) - 1;
          if (lane == l) {
#pragma unroll
            for (int k = 0; k < CH; ++k) lone[k] = d[i / PER][(i % PER) * CH + k] * m;
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          const int fy = __builtin_amdgcn_readlane(c.y0, l), fx = __builtin_amdgcn_readlane(c.x0, l);
          const float gy = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(c.ly), l));
          const float gx = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(c.lx), l));
          const int k = lane % CH, corner = lane / CH;
          const int yy = fy + (corner >> 1), xx = fx + (corner & 1);
          const float w = ((corner & 2) ? gy : 1.0f - gy) * ((corner & 1) ? gx : 1.0f - gx);
          const float t = lone[k];
          if (corner < 4 && yy >= 0 && yy < g.H && xx >= 0 && xx < g.W)
            unsafeAtomicAdd(gin + ((long)n * g.Cin + c0 + k) * plane_in + ((long)yy * g.W + xx), w * t);
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // Every add into the window has landed behind this barrier, and so have the copies of the next pass's weights.  (What is
    // waited for beside them are the loads of grad_output, which the products are about to use, and the last stores of columns.  A count
    // of the loads issued since the copies instead would have nothing to spare: 16 with 8 channels a pass, 5 taps and 64 output
    // channels.)
    settle();
  }
  flush(c_end - CH);
  if (part) {
    const int px = wave * 32 + frow;
#pragma unroll
    for (int i = 0; i < kBfItems; ++i) {
      const int tap = 2 * i + half;
      if (tap < g.taps) {
        part[(2 * tap) * 256 + px] = acc_y[i];
        part[(2 * tap + 1) * 256 + px] = acc_x[i];
        part[(2 * g.taps + tap) * 256 + px] = acc_m[i];
      }
    }
  } else if (valid) {
    const long ob = ((long)n * g.DG + dgi) * 2 * g.taps, mb = ob / 2;
    E *goff = (E *)a.goff, *gmask = (E *)a.gmask;
#pragma unroll
    for (int i = 0; i < kBfItems; ++i) {
      const int tap = 2 * i + half;
      if (tap < g.taps) {
        goff[(ob + 2 * tap) * plane_out + pix] = from_f32<E>(acc_y[i]);
        goff[(ob + 2 * tap + 1) * plane_out + pix] = from_f32<E>(acc_x[i]);
        if (gmask) gmask[(mb + tap) * plane_out + pix] = from_f32<E>(acc_m[i]);
      }
    }
  }
}

// CH channels a pass over the window; CHF when many offsets lie beyond its margin (decided on the device, from a sample of the
// offsets that the pre-pass has looked at).
template <typename E, int CH, int CHF, bool DEEP>
__global__ __launch_bounds__(kBfThreads, 2) void bwd_fused_kernel(BwdFusedArgs a) {
  __shared__ uint4 lds[kBfLdsBytes / 16];
  __shared__ float red[(5 + 16) * kBfWaves + 3];
  asm volatile("; mdcn-counted-waits");
  bool far = false;
  if (a.win_far.WH > 0) {
    uint32_t n = (int)(threadIdx.x & 63) < a.n_far ? a.far[threadIdx.x & 63] : 0u;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o);
    far = __builtin_amdgcn_readfirstlane((int)n) > (int)a.far_min;
  }
  const FusedSchedule &sc = a.sched;
  const int xcd = blockIdx.x % FusedSchedule::kXcds, j = blockIdx.x / FusedSchedule::kXcds;
  const int rounds = sc.count(xcd) / FusedSchedule::kPerXcd, rest = sc.rest(xcd);
  for (int r = 0; r <= rounds; ++r) {
    int tile = sc.first(xcd) + r * FusedSchedule::kPerXcd + j;
    int first = 0, last = sc.passes;
    float *part = nullptr;
    if (r == rounds) {
      const int shares = sc.shares(xcd), k = j / shares, share = j - k * shares;
      if (k >= rest) break;
      tile += k - j;
      first = sc.passes * share / shares;
      last = sc.passes * (share + 1) / shares;
      if (shares > 1) part = a.part + (long)(xcd * FusedSchedule::kPerXcd + j) * 3 * a.g.taps * 256;
    }
    if constexpr (CHF == CH) {
      fused_tile<E, CH, CH, DEEP>(a, far ? a.win_far : a.win, tile, first * CH, last * CH, part, lds, red);
    } else {
      if (far)
        fused_tile<E, CHF, CH, DEEP>(a, a.win_far, tile, first * CH, last * CH, part, lds, red);
      else
        fused_tile<E, CH, CH, DEEP>(a, a.win, tile, first * CH, last * CH, part, lds, red);
    }
  }
}

// Adds up the shares of cut tile `b / (3 taps)` (counted over the XCDs' last rounds), row b % (3 taps) of its sums: one thread a pixel.
template <typename E>
__device__ __forceinline__ void fused_sums_block(const Geom &g, const FusedSchedule &sc, int tw_log, int n0, const float *part, E *goff,
                                                 E *gmask, int b) {
  const int rows = 3 * g.taps, row = b % rows;
  int k = b / rows, xcd = 0;
  while (xcd < FusedSchedule::kXcds - 1 && (sc.shares(xcd) < 2 || k >= sc.rest(xcd))) {
    if (sc.shares(xcd) > 1) k -= sc.rest(xcd);
    ++xcd;
  }
  const int shares = sc.shares(xcd);
  const float *p = part + ((long)(xcd * FusedSchedule::kPerXcd + k * shares) * rows + row) * 256 + threadIdx.x;
  float s = p[0];
  for (int i = 1; i < shares; ++i) s += p[(long)i * rows * 256];
  int t = sc.first(xcd) + sc.count(xcd) - sc.rest(xcd) + k;
  const int TW = 1 << tw_log, TH = 256 >> tw_log, tiles_x = (g.Wo + TW - 1) / TW, tiles_y = (g.Ho + TH - 1) / TH;
  const int tx = t % tiles_x;
  t /= tiles_x;
  const int ty = t % tiles_y;
  t /= tiles_y;
  const int ho = ty * TH + ((int)threadIdx.x >> tw_log), wo = tx * TW + ((int)threadIdx.x & (TW - 1));
  if (ho >= g.Ho || wo >= g.Wo) return;
  const long nd = (long)n0 * g.DG + t, plane = (long)g.Ho * g.Wo, pix = (long)ho * g.Wo + wo;   // (t: image of the pass, deformable group)
  if (row < 2 * g.taps)
    goff[(nd * 2 * g.taps + row) * plane + pix] = from_f32<E>(s);
  else if (gmask)
    gmask[(nd * g.taps + row - 2 * g.taps) * plane + pix] = from_f32<E>(s);
}

// Launches the kernel with ch (16 or 8) channels a pass.  (Defined in a source per element type.)
template <typename E>
void launch_fused(const BwdFusedArgs &a, int ch, hipStream_t st);
template <>
void launch_fused<bf16_t>(const BwdFusedArgs &a, int ch, hipStream_t st);
template <>
void launch_fused<f16_t>(const BwdFusedArgs &a, int ch, hipStream_t st);

template <typename E>
void launch_fused_impl(const BwdFusedArgs &a, int ch, hipStream_t st) {
  const dim3 grid(FusedSchedule::kGroups);
  const bool deep = a.g.cout_g > 2 * kBfK;
  if (ch == 16 && !deep)
    hipLaunchKernelGGL((bwd_fused_kernel<E, 16, 8, false>), grid, dim3(kBfThreads), 0, st, a);
  else if (ch == 16)
    hipLaunchKernelGGL((bwd_fused_kernel<E, 16, 8, true>), grid, dim3(kBfThreads), 0, st, a);
  else if (!deep)
    hipLaunchKernelGGL((bwd_fused_kernel<E, 8, 8, false>), grid, dim3(kBfThreads), 0, st, a);
  else
    hipLaunchKernelGGL((bwd_fused_kernel<E, 8, 8, true>), grid, dim3(kBfThreads), 0, st, a);
}

}  // namespace mdcn
