// fp32 forward: the implicit GEMM of mdcn_fused.h, its products on the 16-bit
// matrix pipe.
//
// The fp32 MFMA (32x32x2) runs at a sixteenth of the 16-bit rate, and an fp32 tile
// was bound by it.  Two ways to make an fp32 product of 16-bit ones:
//
// Pairs (PLANES = 2).  h = fp16(x), l = fp16(x - h): what is left of x is at most 2^-23 |x|, half of that for most.  Three products,
// hl, lh and hh, are summed in fp32; ll, at most 2^-22 of the product and a ninth of it on average, is left out.  fp16 has
// few exponents, so rows are scaled by powers of two: an output channel's weights by the largest of them, an output pixel's samples by the
// largest there can be, from the magnitudes of the input pixels its corners lie on (mdcn_pairs.h); sums are scaled back at the end.  A number
// keeps its 22 bits down to 2^-17 of the largest of its row, below that what lies above 2^-40 of it.
// Triples (PLANES = 3), for calls that pairs do not pay for (pairs_pay), channels-last input, and workspaces without room for the exponents.
// An fp32 number is the sum of three bf16 numbers exactly: h = bf16(x), m = bf16(x - h), l = x - h - m, 8 mantissa bits each
// (both differences are exact).  Six of nine products are summed -- hh, hm, mh, mm, hl, lh; |m| <= 2^-8 |x| and |l| <= 2^-17 |x|, so that ml, lm
// and ll are at most (2^-24 + 2^-34) of the product together, as much as an fp32 multiplication may round by.
//
// What a sum of many terms loses it loses for the most part where it is added up: an MFMA adds sixteen terms at a time, and pairs have half as many of
// them.  Against float64, with positions that fp32 holds exactly, the relative error (2-norm) is 2.8e-7 (pairs) and 3.6e-7 (triples)
// for 2 304 terms, 3.2e-7 and 4.2e-7 for 4 608; with fp32 MFMAs it was 4.3e-7 and 5.9e-7.  Channels whose magnitudes span six decades, the
// weights the same the other way round: 7.0e-7 / 3.6e-7.  For K = 16 six bf16 MFMAs take 192 clocks, three fp16 ones 96, eight fp32 ones 512.
//
// Roles, tables, schedule, cut tiles and epilogue are those of fused_kernel.  What
// differs: a K step (32 channels of a tap) is two half steps of 16 channels; sample and
// weight tiles are kept in fragment order ([half step][plane][32-row block][lane half]
// [32 rows][8 channels], 1 KiB per fragment), so that every access of the loop is
// sequential; the producers split their samples when they write them, the pre-pass splits
// the weights; the consumer waves lie along the channels, so that each weight fragment has one
// reader, which loads it from L2 into registers.
//
// What bounds it (N=8 256 -> 256 64x64, pairs, clocks in the kernel): a K step of a 128 x 256 tile takes 2 650 at the 1.8 GHz that the card runs it at.
// The consumers' half is 2 050 of them, 1 536 MFMAs; the producers' 2 480, and the barrier waits for them: 150 VALU instructions, which make no progress while
// MFMAs are issued on their SIMD, between gathers.  Main kernel, us: 325 with fp32 MFMAs, 213 triples, 131 pairs (MFMAs alone: 58); whole call
// 230 -> 148.  N=2 50x84, whole call: 103 -> 69.  Without weights' loads, gathers, MFMAs (each alone, at 146): 132, 120, 128.
// Tried and not faster: weights through LDS, producers at a higher or lower wave priority (triples), weights' loads a half step
// earlier (pairs, 152 against 149).
#pragma once

#include <type_traits>

#include "mdcn_direct.h"
#include "mdcn_fused.h"

namespace mdcn {

constexpr int kF32Planes = 3;
// ... or two fp16 planes (see the head of the file): fp16 pairs are scaled row by row so that the largest number there can be
// in a row of either operand lies in [2^14, 2^15).
constexpr int kPairTop = 14;
// Both operands are multiplied by this before they are split, and the sums by its inverse squared: the third plane holds bits
// down to 2^-23 of a number, and bf16, with the exponents of fp32, ends at 2^-126.  Unscaled, numbers below 2^-103 lose
// some of their bits (2e-6 of a number of 2^-115, 2e-3 at 2^-125); scaled, the smallest normal number has
// all of its 24.  In exchange numbers from 2^104 and sums from 2^80 on overflow, and are made again.
constexpr float kSplitScale = 16777216.0f;
constexpr float kSplitUnscale = 1.0f / (kSplitScale * kSplitScale);
// K steps a gather is in flight, bf16 triples: one register set, refilled behind its use, so that every load has a whole step
// (some 3 000 clocks) to land.  (With two sets the compiler copies them into each other at the loop's
// end and waits for all of their loads to do so.)
constexpr int kF32Ahead = 1;
// ... fp16 pairs, whose steps are shorter: two sets, taken in turn by a loop of two steps.
constexpr int kPairAhead = 2;
// Sample tiles: one being read, one ready, so that the consumers fetch their first fragments of a step ahead of the
// barrier that ends the one before, and one being written.
constexpr int kF32Tiles = 3;
// LDS of one workgroup (three planes; of two it is less): sample tiles, table.
constexpr size_t fused_f32_lds_bytes(int tmax) {
  return (size_t)kF32Tiles * kPT * 192 + (size_t)kPT * tmax * 20 + 16;
}

// Units of one workgroup: as UnitSchedule's, tiles round robin within the XCD's run and then the last round's tiles in parts.  These
// `rest` tiles lie end to end, rest * rounds rounds of K steps, and workgroup w of the XCD's `stride` has those from pos(w) to
// pos(w + 1): an equal part of one tile (`parts` workgroups each, some may have nothing), or, `even`, the same number of rounds for
// everybody, wherever tiles begin; a workgroup then has parts of up to two tiles, and a tile up to three.  Parts of less than min_rounds
// are not made.  host: the same arithmetic for the plan.
struct PartSchedule {
  int xcd, wg, stride, tile0, full, rest, rounds, round, min_rounds, parts, per_wg;
  int begin, end;   // this workgroup's rounds of the last round
  bool even;

  __host__ __device__ __forceinline__ void init(int xcd_, int wg_, int stride_, int total_tiles, int nk_pad, int round_, int min_rounds_,
                                                int cut_max, bool even_) {
    xcd = xcd_, wg = wg_, stride = stride_, round = round_, min_rounds = min_rounds_;
    per_wg = even_ ? 2 : 1;
    const int chunk = (total_tiles + 7) >> 3;
    tile0 = xcd * chunk;
    const int left = total_tiles - tile0, count = left < 0 ? 0 : left < chunk ? left : chunk;
    full = count / stride;
    rest = count - full * stride;
    rounds = nk_pad / round;
    even = even_ && rest * rounds >= 3 * min_rounds * stride;   // (no share may vanish between two tiles)
    parts = 1;
    if (even) {
      begin = pos(wg), end = pos(wg + 1);
      return;
    }
    if (cut_max > 1 && rest > 0) {
      parts = stride / rest < cut_max ? stride / rest : cut_max;
      parts = parts < rounds / min_rounds ? parts : rounds / min_rounds;
      parts = parts > 1 ? parts : 1;
    }
    const int t = wg / parts, i = wg - t * parts;
    begin = t * rounds + i * rounds / parts, end = t * rounds + (i + 1) * rounds / parts;
    if (t >= rest) end = begin;
  }
  __host__ __device__ __forceinline__ int pos(int w) const {   // even shares
    const int x = w * rest * rounds / stride, r = x % rounds;
    return r < min_rounds ? x - r : rounds - r < min_rounds ? x - r + rounds : x;
  }
  __host__ __device__ __forceinline__ int units() const {
    if (begin == end) return full;
    return full + (even && (end - 1) / rounds > begin / rounds ? 2 : 1);
  }
  struct Unit {
    int tile, kb, pad;          // K steps kb .. kb + pad - 1 of a tile
    bool is_part;
    int slot;                   // of its tile among the last round's
    int first, n, idx;          // first workgroup with a part of the tile, number of parts, which one this is
    bool first_behind;          // the first part is its workgroup's second
  };
  __host__ __device__ __forceinline__ Unit unit(int u) const {
    Unit r;
    r.tile = tile0 + wg + u * stride;
    r.kb = 0, r.pad = rounds * round;
    r.is_part = false;
    r.slot = r.first = r.idx = 0, r.n = 1;
    r.first_behind = false;
    if (u < full) return r;
    if (!even) {
      r.slot = wg / parts;
      r.first = r.slot * parts, r.n = parts, r.idx = wg - r.first;
    } else {
      r.slot = begin / rounds + u - full;
      int f = wg, l = wg;
      while (f > 0 && pos(f) > r.slot * rounds) --f;
      while (l + 1 < stride && pos(l + 1) < (r.slot + 1) * rounds) ++l;
      r.first = f, r.n = l - f + 1, r.idx = wg - f;
      r.first_behind = pos(f) < r.slot * rounds;
    }
    const int t0 = r.slot * rounds, lo = begin > t0 ? begin : t0, hi = end < t0 + rounds ? end : t0 + rounds;
    r.tile = tile0 + full * stride + r.slot;
    r.kb = (lo - t0) * round, r.pad = (hi - lo) * round;
    r.is_part = hi - lo < rounds;
    return r;
  }
  // buffer of part i of a unit's tile (one for each workgroup; even: two), and the counter of the tile
  __host__ __device__ __forceinline__ int buffer(const Unit &r, int i) const {
    return (xcd * stride + r.first + i) * per_wg + (i == 0 && r.first_behind ? 1 : 0);
  }
  __host__ __device__ __forceinline__ int counter(const Unit &r) const { return xcd * stride + r.slot; }
};

// Four floats, scaled already, as three bf16 planes of 8 bytes each.  An infinity, or a number that bf16 rounds to one
// (from 2^128 (1 - 2^-9) on), leaves NaN in the planes, and so in every sum that it is part of: sums that are not
// finite are not used, but made again from the tensors themselves.
__device__ __forceinline__ void split3(const float (&x)[4], uint2 (&p)[3]) {
  float r[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = x[i];
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    uint32_t lo = ElemTraits<bf16_t>::pack2(r[0], r[1]), hi = ElemTraits<bf16_t>::pack2(r[2], r[3]);
    asm("" : "+v"(lo), "+v"(hi));  // (or the compiler converts the first of each pair a second time)
    p[s] = make_uint2(lo, hi);
    if (s < 2) {
      r[0] -= __uint_as_float(lo << 16);
      r[1] -= __uint_as_float(lo & 0xffff0000u);
      r[2] -= __uint_as_float(hi << 16);
      r[3] -= __uint_as_float(hi & 0xffff0000u);
    }
  }
}

// Four floats, scaled already, as an fp16 number and the fp16 number nearest to what that leaves.  An infinity, and what is beyond
// fp16, leaves NaN or an infinity.
__device__ __forceinline__ void split2(const float (&x)[4], uint2 (&p)[2]) {
  f16x2 h[2], l[2];
  float minus = -1.0f;
  asm("" : "+s"(minus));     // (... and makes two instructions of the mixed multiply-add below)
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    uint32_t hw = __builtin_bit_cast(uint32_t, f16x2{(f16_t)x[2 * i], (f16_t)x[2 * i + 1]});
    asm("" : "+v"(hw));  // (or the compiler converts each number a second time)
    h[i] = __builtin_bit_cast(f16x2, hw);
    l[i] = f16x2{(f16_t)fmaf((float)h[i].x, minus, x[2 * i]), (f16_t)fmaf((float)h[i].y, minus, x[2 * i + 1])};
  }
  p[0] = make_uint2(__builtin_bit_cast(uint32_t, h[0]), __builtin_bit_cast(uint32_t, h[1]));
  p[1] = make_uint2(__builtin_bit_cast(uint32_t, l[0]), __builtin_bit_cast(uint32_t, l[1]));
}

// The power of two that takes `top`, the largest magnitude of a row, to [2^kPairTop, 2^(kPairTop + 1)); 0 for a row of zeros and
// for one that is not finite.
__device__ __forceinline__ int pair_exponent(float top) {
  const int e = (int)(__float_as_uint(top) >> 23) & 0xff;
  return top == 0.0f || e == 0xff ? 0 : kPairTop + 127 - e;   // (a subnormal number: as if it were normal)
}

// ... of a row of samples, whose corner weights take it: `most` is the largest magnitude of a mask value, and no product
// of the two overflows.  -113 .. 127.
__device__ __forceinline__ int sample_exponent(float top, float most) {
  const int em = (int)(__float_as_uint(most) >> 23) & 0xff;
  return min(pair_exponent(top), min(127, 126 + 127 - em));
}

// weight[Cout][Cin/G][kh][kw] -> wp[G][n_ctiles][nk][2 half steps][3 planes][CT / 32][64 lanes][8 bf16]: A
// operands of the 32x32x16 MFMA in the order the kernel copies and reads them; zero past Cout/G.  Also clears
// the cut-tile counters.
__device__ __forceinline__ void pack_weight_split(const Geom &g, const float *__restrict__ w, void *__restrict__ wp,
                                                  int CT, int n_ctiles, int slabs, long first, long stride,
                                                  uint32_t *__restrict__ zero_ptr, int zero_n) {
  for (long i = first; i < zero_n; i += stride) zero_ptr[i] = 0u;
  const int nk = slabs * g.taps, blocks = CT / 32;
  // 3x3: a lane's eight channels are 288 contiguous, aligned bytes, nine taps at a time.  From 512 -> 512 channels on (whole
  // call, us, one by one / nine: N=1 512 channels 13x13 59.5 / 54.8): with fewer lanes to do it the nine splits of each are the
  // longer chain (128 channels 28x28 29.4 / 31.2, 256 channels 28x28 42.9 / 44.9).
  const long units = (long)g.G * n_ctiles * slabs * 2 * blocks * 64;
  if (g.taps == 9 && (uintptr_t)w % 16 == 0 && units >= 32768) {
    for (long idx = first; idx < units; idx += stride) {
      long r = idx;
      const int lane = (int)(r & 63);
      r >>= 6;
      const int blk = (int)(r % blocks);
      r /= blocks;
      const int half = (int)(r & 1);
      r >>= 1;
      const int slab = (int)(r % slabs);
      r /= slabs;  // (group, tile)
      const int ctile = (int)(r % n_ctiles), grp = (int)(r / n_ctiles);
      const int col = ctile * CT + blk * 32 + (lane & 31);
      const int c0 = slab * 32 + half * 16 + (lane >> 5) * 8;
      float v[72];
      const uint4 *src = (const uint4 *)(w + ((long)(grp * g.cout_g + min(col, g.cout_g - 1)) * g.cin_g + c0) * 9);
#pragma unroll
      for (int i = 0; i < 18; ++i) {
        const uint4 q = src[i];
        __builtin_memcpy(v + 4 * i, &q, 16);
      }
      if (col >= g.cout_g) {
#pragma unroll
        for (int i = 0; i < 72; ++i) v[i] = 0.0f;
      }
#pragma unroll
      for (int i = 0; i < 72; ++i) v[i] *= kSplitScale;
#pragma unroll
      for (int tap = 0; tap < 9; ++tap) {
        uint2 p0[3], p1[3];
        split3({v[tap], v[9 + tap], v[18 + tap], v[27 + tap]}, p0);
        split3({v[36 + tap], v[45 + tap], v[54 + tap], v[63 + tap]}, p1);
        uint4 *dst = (uint4 *)wp + (((r * nk + slab * 9 + tap) * 2 + half) * 3 * blocks + blk) * 64 + lane;
#pragma unroll
        for (int s = 0; s < 3; ++s) dst[(long)s * blocks * 64] = make_uint4(p0[s].x, p0[s].y, p1[s].x, p1[s].y);
      }
    }
    return;
  }
  const long total = (long)g.G * n_ctiles * nk * 2 * blocks * 64;
  for (long idx = first; idx < total; idx += stride) {
    long r = idx;
    const int lane = (int)(r & 63);
    r >>= 6;
    const int blk = (int)(r % blocks);
    r /= blocks;
    const long step = r >> 1;  // (group, tile, K step)
    const int half = (int)(r & 1);
    r = step;
    const int ks = (int)(r % nk);
    r /= nk;
    const int ctile = (int)(r % n_ctiles), grp = (int)(r / n_ctiles);
    const int slab = ks / g.taps, tap = ks - slab * g.taps;
    const int col = ctile * CT + blk * 32 + (lane & 31);
    const int c0 = slab * 32 + half * 16 + (lane >> 5) * 8;
    float v[8];
    const float *src = w + ((long)(grp * g.cout_g + min(col, g.cout_g - 1)) * g.cin_g + c0) * g.taps + tap;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = col < g.cout_g ? src[(long)i * g.taps] * kSplitScale : 0.0f;
    uint2 p0[3], p1[3];
    split3({v[0], v[1], v[2], v[3]}, p0);
    split3({v[4], v[5], v[6], v[7]}, p1);
    uint4 *dst = (uint4 *)wp + ((step * 2 + half) * 3 * blocks + blk) * 64 + lane;
#pragma unroll
    for (int s = 0; s < 3; ++s) dst[(long)s * blocks * 64] = make_uint4(p0[s].x, p0[s].y, p1[s].x, p1[s].y);
  }
}

// The outputs of consumer wave `wave` in the units of its workgroup's schedule that are not finite, from the call's own tensors; units of the last round
// whose bit is set in `skip` were stored by others.
template <int CT, int WC, int MB, int NB, int AHEAD>
__device__ __forceinline__ void remake_not_finite(const FusedArgs &a, uint32_t skip, int nk_tile_pad, int wave, int lane) {
  const Geom &g = a.g;
  const int plane_out = g.Ho * g.Wo;
  PartSchedule us;
  us.init((int)(blockIdx.x & 7), (int)(blockIdx.x >> 3), (int)(gridDim.x >> 3), a.n_ptiles * a.n_ctiles * g.G, nk_tile_pad, AHEAD, 8 / AHEAD,
          a.cut_max, a.cut_even != 0);
#pragma unroll 1
  for (int u = 0; u < us.units(); ++u) {
    if (u >= us.full && (skip >> (u - us.full) & 1)) continue;
    int L = us.unit(u).tile;
    const int ctile = L % a.n_ctiles;
    L /= a.n_ctiles;
    const int grp = L % g.G, ptile = L / g.G;
    const int c0 = ctile * CT + wave % WC * (MB * 32), p0 = ptile * kPT + wave / WC * (NB * 32) + lane;
#pragma unroll 1
    for (int i = 0; i < MB * 32 * (NB / 2); ++i) {
      const int col = c0 + i / (NB / 2), p = p0 + i % (NB / 2) * 64;
      if (col >= g.cout_g || p >= (int)a.total_px) continue;
      const int n = p / plane_out, rem = p - n * plane_out;
      const int co = grp * g.cout_g + col;
      float *o = (float *)a.out + ((long)n * g.Cout + co) * plane_out + rem;
      const float was = __hip_atomic_load(o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (was - was == 0.0f) continue;
      const float v = direct_sum<float, false>(g, (const float *)a.in + (long)n * g.Cin * g.H * g.W, a.in_c, a.in_px, a.om,
                                               (const float *)a.weight, n, co, rem / g.Wo, rem % g.Wo);
      *o = v + (a.bias ? ((const float *)a.bias)[co] : 0.0f);
    }
  }
}

// MULTI_DG, UNBORDERED: as in fused_kernel.  PLANES: bf16 triples or fp16 pairs.
template <int CT, int TMAX, bool MULTI_DG, bool UNBORDERED, int PLANES>
__global__ __launch_bounds__(kThreads, 2) void fused_f32_kernel(FusedArgs a) {
  using E = float;
  using TR = ElemTraits<E>;
  constexpr bool kPairs = PLANES == 2;
  constexpr int AHEAD = kPairs ? kPairAhead : kF32Ahead;
  using TB = ElemTraits<std::conditional_t<kPairs, f16_t, bf16_t>>;
  constexpr int PT = kPT;
  constexpr int KC = TR::KC;
  constexpr int ES = (int)sizeof(E);
  // Consumer waves lie along the channels, so that a weight fragment has one reader: WC of them, MB 32-channel
  // blocks each, over NB 32-pixel blocks.
  constexpr int WC = CT / 32 < 4 ? CT / 32 : 4;
  constexpr int MB = CT / 32 / WC;
  constexpr int NB = WC;   // (4 / (4 / WC))
  constexpr int WBLK = PLANES * CT / 32;    // 1 KiB fragments of a half-step weight tile
  constexpr int TPT = (TMAX + kTapGroups - 1) / kTapGroups;  // table entries per producer lane
  constexpr int XFRAG = PLANES * (PT / 32) * 64;      // 16-byte pieces of a half step of a sample tile
  __shared__ uint4 Xs[kF32Tiles][2 * XFRAG];              // sample tiles
  __shared__ uint32_t tpix[PT * TMAX];                    // (pixel, tap) table, [tap][PT]: corner byte offset
  __shared__ uint4 tws[PT * TMAX];                        // ... and the four weights
  __shared__ uint32_t part_arrived;                       // parts of a cut tile that were there before this one
  __shared__ __align__(16) int row_exp[kPairs ? PT : 4];  // pairs: exponents of the tile's pixels

  const Geom &g = a.g;
  const int taps = g.taps;
  const int nk_tile = a.slabs * taps;
  const int nk_tile_pad = (nk_tile + AHEAD - 1) / AHEAD * AHEAD;
  const int plane_out = g.Ho * g.Wo;
  const int total_px = (int)a.total_px;
  const int spd = g.ch_per_dg / KC;  // slabs per deformable group

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool producer = wave >= 4;

  // XCD-aware persistent schedule: consecutive workgroup ids sit on different
  // XCDs; each XCD walks one contiguous run of tiles so that the halo rows
  // neighbouring tiles share stay in its L2.  Tiles of the run's last round are
  // cut along K (PartSchedule): parts of at least 8 steps.
  PartSchedule us;
  us.init((int)(blockIdx.x & 7), (int)(blockIdx.x >> 3), (int)(gridDim.x >> 3), a.n_ptiles * a.n_ctiles * g.G, nk_tile_pad, AHEAD, 8 / AHEAD,
          a.cut_max, a.cut_even != 0);

  bool bad = false;    // consumer waves: a sum of a stored tile was not finite
  uint32_t skip = 0;   // ... units of the last round that they have not stored: parts of cut tiles
  const int units = us.units();
  for (int u = 0; u < units; ++u) {
    const PartSchedule::Unit un = us.unit(u);
    const bool is_part = un.is_part;
    // K range of the unit: steps kb .. kb + nk - 1 of the tile, padded to nk_pad
    const int kb = un.kb, nk_pad = un.pad;
    const int nk = min(nk_tile - kb, nk_pad);
    int L = un.tile;
    const int ctile = L % a.n_ctiles;
    L /= a.n_ctiles;
    const int grp = L % g.G;
    const int ptile = L / g.G;
    const int p0 = ptile * PT;
    const int ch0 = grp * g.cin_g;  // first input channel of the group
    const int slab0 = ch0 / KC;

    StepCursor cur;  // the next step whose gather is issued
    cur.init(slab0, spd, kb, taps);

    if (producer) {
      // =================== PRODUCER ===================
      const int ptid = tid - 256;
      const int q = ptid & 3;          // this lane handles 16-byte chunks q and q + 4 of a row
      const int pxl = ptid >> 2;       // ... of pixels pxl and pxl + 64 of the tile
      const unsigned char *xt = (const unsigned char *)a.xt;
      // horizontal neighbour: an instruction offset for the copy, a register otherwise
      const uint32_t pxb = UNBORDERED ? a.px_bytes : (uint32_t)kRowB;

      // -- (pixel, tap) table of one deformable group; lane serves pixel ptid%128
      const int tb_pl = ptid & (PT - 1);
      const int tb_p = p0 + tb_pl;
      const bool tb_valid = tb_p < total_px;
      int tb_n = 0, tb_ho = 0, tb_wo = 0, tb_rem = 0;
      if (tb_valid) {
        tb_n = tb_p / plane_out;
        tb_rem = tb_p - tb_n * plane_out;
        tb_ho = tb_rem / g.Wo;
        tb_wo = tb_rem - tb_ho * g.Wo;
      }
      // what takes the lane's pixel to fp16's range (a row of a padded pixel holds zeros)
      float scale = kSplitScale;
      if constexpr (kPairs) {
        const int e = a.row_exp[(long)grp * total_px + min(tb_p, total_px - 1)];
        scale = __uint_as_float((uint32_t)(e + 127) << 23);
        if (ptid < PT) row_exp[tb_pl] = e;
      }
      auto build_table = [&](int dgi) {
        if constexpr (kPairs) {   // made by pair_exponent_kernel; scaled here
          const long at = (long)(dgi * taps) * total_px + min(tb_p, total_px - 1);
          uint32_t pix[TPT];
          float4 w[TPT];
#pragma unroll
          for (int i = 0; i < TPT; ++i) {
            const long e = at + (long)min((ptid >> 7) + kTapGroups * i, taps - 1) * total_px;
            pix[i] = a.tab_pix[e];
            w[i] = a.tab_w[e];
          }
          const float s = tb_valid ? scale : 0.0f;
#pragma unroll
          for (int i = 0; i < TPT; ++i) {
            const int tap = (ptid >> 7) + kTapGroups * i;
            if (tap < taps) {
              tpix[tap * PT + tb_pl] = pix[i];
              tws[tap * PT + tb_pl] = make_uint4(__float_as_uint(w[i].x * s), __float_as_uint(w[i].y * s), __float_as_uint(w[i].z * s),
                                                 __float_as_uint(w[i].w * s));
            }
          }
          return;
        }
        // (an invalid pixel reads the entries of pixel 0 of image 0 and stores zeros)
        const E *off = (const E *)a.om.off + (long)tb_n * a.om.off_n + (long)tb_rem * a.om.off_px +
                       (long)(dgi * 2 * taps) * a.om.off_ch;
        const E *msk = (const E *)a.om.msk + (long)tb_n * a.om.msk_n + (long)tb_rem * a.om.msk_px +
                       (long)(dgi * taps) * a.om.msk_ch;
        // all loads first (unconditional, clamped), then the arithmetic
        E rdy[TPT], rdx[TPT], rm[TPT];
#pragma unroll
        for (int i = 0; i < TPT; ++i) {
          const int tap = min((ptid >> 7) + kTapGroups * i, taps - 1);
          rdy[i] = off[(long)(2 * tap) * a.om.off_ch];
          rdx[i] = off[(long)(2 * tap + 1) * a.om.off_ch];
          rm[i] = msk[(long)tap * a.om.msk_ch];
        }
#pragma unroll
        for (int i = 0; i < TPT; ++i) {
          const int tap = (ptid >> 7) + kTapGroups * i;
          if (tap < taps) {
            const int ti = tap / g.kw, tj = tap - ti * g.kw;
            TapSample sm =
                make_tap_sample(tb_ho * g.sh - g.ph + ti * g.dh, tb_wo * g.sw - g.pw + tj * g.dw,
                                to_f32(rdy[i]), to_f32(rdx[i]), mask_value<E>(rm[i], a.om.logit) * scale, g.H, g.W);
            // byte offset of the upper left corner, slab 0 of image tb_n
            uint32_t pix = (uint32_t)tb_n * a.img_bytes + corner_offset<UNBORDERED>(sm, g, a);
            uint32_t tw[4];
            TR::table_weights(sm, tw);
            if (!tb_valid) {
              pix = 0;
              tw[0] = tw[1] = tw[2] = tw[3] = 0u;
            }
            tpix[tap * PT + tb_pl] = pix;
            tws[tap * PT + tb_pl] = make_uint4(tw[0], tw[1], tw[2], tw[3]);
          }
        }
      };

      // -- gather state: AHEAD register sets, set m % AHEAD holds step m;
      //    [pixel][corner][half of the lane's 32 bytes]
      uint4 gv[AHEAD][kPxPerLane][4][2];
      uint4 gw[AHEAD][kPxPerLane];
      // Gather of the cursor's step (rebuilding the table first when the step
      // opens a new deformable group), then move the cursor on.
      auto issue_gather = [&](uint4 (&v)[kPxPerLane][4][2], uint4 (&w)[kPxPerLane]) {
        if (MULTI_DG && cur.new_dg) {
          // Every producer issued the previous group's last step before the
          // barrier that ended the previous K step, with its weights in registers.
          cur.new_dg = false;
          build_table((ch0 + cur.slab * KC) / g.ch_per_dg);
          MDCN_BARRIER_LDS();  // R: new table visible (the consumers join)
        }
        const uint32_t sbase = (uint32_t)(slab0 + cur.slab) * a.slab_bytes + (uint32_t)q * 16u;
#pragma unroll
        for (int h = 0; h < kPxPerLane; ++h) {
          const int e = cur.tap * PT + pxl + (PT / kPxPerLane) * h;
          const uint32_t o = tpix[e] + sbase;
          w[h] = tws[e];
          const unsigned char *top = xt + o;
          const unsigned char *bot = top + a.row_bytes;
          v[h][0][0] = *(const uint4 *)(top);
          v[h][0][1] = *(const uint4 *)(top + 64);
          v[h][1][0] = *(const uint4 *)(top + pxb);
          v[h][1][1] = *(const uint4 *)(top + pxb + 64);
          v[h][2][0] = *(const uint4 *)(bot);
          v[h][2][1] = *(const uint4 *)(bot + 64);
          v[h][3][0] = *(const uint4 *)(bot + pxb);
          v[h][3][1] = *(const uint4 *)(bot + pxb + 64);
        }
        cur.advance(nk, taps, spd);
      };

      // Blend the set (step s) into sample tile `buf` and refill it with the
      // gather of the cursor's step, 16 bytes x 4 corners at a time: the loads go
      // out between the blends, so the memory pipeline works while the VALU does.
      auto commit_and_refill = [&](int buf, uint4 (&v)[kPxPerLane][4][2], uint4 (&w)[kPxPerLane]) {
        if (MULTI_DG && cur.new_dg) {
          cur.new_dg = false;
          build_table((ch0 + cur.slab * KC) / g.ch_per_dg);
          MDCN_BARRIER_LDS();  // R
        }
        const uint32_t sbase = (uint32_t)(slab0 + cur.slab) * a.slab_bytes + (uint32_t)q * 16u;
        uint32_t o[kPxPerLane];
        uint4 wn[kPxPerLane];
#pragma unroll
        for (int h = 0; h < kPxPerLane; ++h) {
          const int e = cur.tap * PT + pxl + (PT / kPxPerLane) * h;
          o[h] = tpix[e] + sbase;
          wn[h] = tws[e];
        }
#pragma unroll
        for (int h = 0; h < kPxPerLane; ++h) {
          const int row = pxl + (PT / kPxPerLane) * h;
#pragma unroll
          for (int half = 0; half < 2; ++half) {
            uint4 s = TR::blend(v[h][0][half], v[h][1][half], v[h][2][half], v[h][3][half], w[h]);
            // (The set's registers are refilled in place: nothing that reads them may be moved behind the loads, or
            // the loads go elsewhere and the loop ends with copies that wait for all of them.)
            asm volatile("" : "+v"(s.x), "+v"(s.y), "+v"(s.z), "+v"(s.w));
            __builtin_amdgcn_sched_barrier(0);
            const unsigned char *top = xt + o[h] + half * 64;
            const unsigned char *bot = top + a.row_bytes;
            v[h][0][half] = *(const uint4 *)(top);
            v[h][1][half] = *(const uint4 *)(top + pxb);
            v[h][2][half] = *(const uint4 *)(bot);
            v[h][3][half] = *(const uint4 *)(bot + pxb);
            __builtin_amdgcn_sched_barrier(0);
            // channels 4 q .. 4 q + 3 of half step `half`: 8 bytes of the fragments of lane half q >> 1
            uint2 pl[PLANES];
            const float sv[4] = {__uint_as_float(s.x), __uint_as_float(s.y), __uint_as_float(s.z), __uint_as_float(s.w)};
            if constexpr (kPairs) split2(sv, pl);
            else split3(sv, pl);
            uint2 *dst = (uint2 *)&Xs[buf][half * XFRAG + (row >> 5) * 64 + (q >> 1) * 32 + (row & 31)] + (q & 1);
#pragma unroll
            for (int p = 0; p < PLANES; ++p) dst[p * (PT / 32) * 64 * 2] = pl[p];
          }
          w[h] = wn[h];
        }
        cur.advance(nk, taps, spd);
      };

      build_table((ch0 + cur.slab * KC) / g.ch_per_dg);
      MDCN_BARRIER_LDS();  // B0: table visible

#pragma unroll
      for (int j = 0; j < AHEAD; ++j) issue_gather(gv[j], gw[j]);
      commit_and_refill(0, gv[0], gw[0]);
      commit_and_refill(1, gv[AHEAD - 1], gw[AHEAD - 1]);
      MDCN_BARRIER_LDS();  // B1: X[0], X[1] visible

      // (steps past nk repeat the last one and nobody reads what they produce)
      int wt = 2;
      for (int ks = 0; ks < nk_pad; ks += AHEAD) {
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
          commit_and_refill(wt, gv[j], gw[j]);
          wt = wt == kF32Tiles - 1 ? 0 : wt + 1;
          MDCN_BARRIER_LDS();  // end of step ks + j: X[ks+j+2] visible
        }
      }
      // The gathers issued past the last step are never read.  Retire them with a
      // wait the compiler can see: it tracks these loads' destination registers,
      // carries that state round the tile loop into the consumer branch (it cannot
      // know that a wave keeps its role) and would otherwise guard the consumers'
      // registers with vmcnt waits that also wait for their in-flight weight copies.
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), other counters untouched
      MDCN_BARRIER_LDS();   // E0: the K loop is over for everybody
      if (is_part) {        // the consumers' two barriers around the arrival count of a cut tile
        MDCN_BARRIER_LDS();
        MDCN_BARRIER_LDS();
      }
      MDCN_BARRIER_LDS();   // E1: epilogue done, tiles and table may be rewritten
    } else {
      // =================== CONSUMER ===================
      const int wave_p = wave / WC;   // which NB * 32 pixels
      const int wave_c = wave % WC;   // which MB * 32 output channels
      f32x16 acc[NB][MB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[nb][mb][r] = 0.0f;

      const int frow = lane & 31;
      const int fhalf = lane >> 5;
      int wexp[MB];   // pairs: exponents of this lane's output channels
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        wexp[mb] = kPairs ? ((const int *)a.wexp)[(grp * a.n_ctiles + ctile) * CT + (wave_c * MB + mb) * 32 + frow] : 0;
      // bias of this lane's output channels, fetched now so that the epilogue
      // never waits on a load (a wait there would also wait for its own stores)
      float bv[MB];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const int mycol = ctile * CT + (wave_c * MB + mb) * 32 + frow;
        bv[mb] = 0.0f;
        if (a.bias && mycol < g.cout_g) bv[mb] = to_f32(((const E *)a.bias)[grp * g.cout_g + mycol]);
      }
      // mirror of the producers' issue sequence, for the table-rebuild barriers
      auto mirror_issue = [&]() {
        if (MULTI_DG && cur.new_dg) {
          cur.new_dg = false;
          MDCN_BARRIER_LDS();  // R
        }
        cur.advance(nk, taps, spd);
      };
      // Weight fragments come from L2 straight into registers, each half step's a half step ahead: no other wave
      // reads them, so they need neither LDS nor a barrier, and what they cost is one pass through the
      // vector-memory path.
      const uint4 *wp_tile = (const uint4 *)a.wp +
                             ((size_t)(grp * a.n_ctiles + ctile) * nk_tile + kb) * (size_t)(2 * WBLK * 64) +
                             wave_c * MB * 64 + lane;
      uint4 wf[2][PLANES][MB];
      auto load_weights = [&](int hs, uint4 (&w)[PLANES][MB]) {
        const uint4 *src = wp_tile + (size_t)min(hs, 2 * nk - 1) * (WBLK * 64);  // (past the end: never used)
#pragma unroll
        for (int p = 0; p < PLANES; ++p)
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) w[p][mb] = src[(p * (CT / 32) + mb) * 64];
      };
      load_weights(0, wf[0]);
      MDCN_BARRIER_LDS();  // B0
#pragma unroll
      for (int v = 0; v < AHEAD + 2; ++v) mirror_issue();
      MDCN_BARRIER_LDS();  // B1

      // Sample fragments [plane][pixel block], each plane fetched while the products of the one before run -- the
      // first ones of a step during the last products of the step before.
      constexpr bool kEarlyX = CT <= 128;  // two planes that early, where the registers allow
      uint4 xf[PLANES][NB];
      auto load_x = [&](int tile, int half, int p) {
        const uint4 *X = Xs[tile] + half * XFRAG + wave_p * (NB * 64) + lane;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) xf[p][nb] = X[p * (PT / 32) * 64 + nb * 64];
      };
      load_x(0, 0, PLANES - 1);
      if constexpr (kEarlyX && !kPairs) load_x(0, 0, 1);
      int rt = 0;
      for (int ks = 0; ks < nk; ++ks) {
        const int nt = rt == kF32Tiles - 1 ? 0 : rt + 1;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          auto products = [&](int xp, int wpl) {
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
              for (int nb = 0; nb < NB; ++nb) TB::mma(acc[nb][mb], xf[xp][nb], wf[half][wpl][mb]);
            __builtin_amdgcn_sched_barrier(0);
          };
          // (the order is kept: the scheduler, left to itself, reads each fragment right in front of its first use)
          load_weights(2 * ks + half + 1, wf[half ^ 1]);
          if constexpr (!kEarlyX && !kPairs) load_x(rt, half, 1);
          load_x(rt, half, 0);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (!kPairs) {
            products(2, 0);  // smallest terms first
            products(1, 1);
          }
          products(1, 0);
          load_x(half ? nt : rt, half ^ 1, PLANES - 1);
          if constexpr (kEarlyX && !kPairs) load_x(half ? nt : rt, half ^ 1, 1);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (!kPairs) products(0, 2);
          products(0, 1);
          products(0, 0);
        }
        rt = nt;
        mirror_issue();
        MDCN_BARRIER_LDS();  // end of step ks
      }
      for (int ks = nk; ks < nk_pad; ++ks) MDCN_BARRIER_LDS();
      MDCN_BARRIER_LDS();  // E0: the sample tiles become staging

      // ---- a part of a tile: the parts meet in memory.  Every part stores its
      // accumulators (fp32, register order) and counts itself in; the part that
      // arrives last adds them up -- two parts: its own registers plus the other's
      // values, the same in either order; more: all from memory in index order, so
      // the sum does not depend on who was last -- and goes on to the epilogue; the
      // others are done.  Nobody waits for anybody; the last part leaves the counter
      // at zero for the next launch.  Stores and loads are device coherent (sc1):
      // they go past the caches private to a CU or an XCD.  The producers take part in the
      // two barriers.
      bool store_tile = true;
      if (is_part) {
        constexpr int NQ = NB * MB * 4;           // 16-byte quads of accumulators per lane
        constexpr int CQ = 8;                     // quads read back at a time (NQ is a multiple of 8)
        const int tslot = us.counter(un);
        auto part_of = [&](int i) { return (const unsigned char *)a.cut_part + (size_t)us.buffer(un, i) * (size_t)(PT * 256 * 4); };
        const unsigned char *mine = uniform_ptr(part_of(un.idx));
        // quad j of the 256 consumer lanes is one 4 KiB run.  (The offset is opaque to the optimiser,
        // which would otherwise form the addresses below ahead of the unit loop and keep them live.)
        uint32_t voff = (uint32_t)tid * 16u;
        asm volatile("" : "+v"(voff));
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) {
              const f32x16 &c = acc[nb][mb];
              const f32x4 v = {c[4 * qd], c[4 * qd + 1], c[4 * qd + 2], c[4 * qd + 3]};
              const uint32_t vo = voff + (uint32_t)(((nb * MB + mb) * 4 + qd) * 4096);
              // (s_nop: a vector-memory instruction must not read a scalar register within five issue
              // slots of a vector instruction writing it -- a reload of spilled scalars, say -- and the
              // compiler does not look into assembly text to keep that distance)
              asm volatile("s_nop 4\n\tglobal_store_dwordx4 %0, %1, %2 sc1" : : "v"(vo), "v"(v), "s"(mine) : "memory");
            }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        MDCN_BARRIER_LDS();
        if (tid == 0)
          part_arrived = __hip_atomic_fetch_add((uint32_t *)a.cut_cnt + tslot, 1u, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
        MDCN_BARRIER_LDS();
        store_tile = part_arrived == (uint32_t)(un.n - 1);
        if (store_tile) {
          const bool two = un.n == 2;
          for (int i = two ? 1 : 0; i < un.n; ++i) {
            const unsigned char *src = uniform_ptr(part_of(two ? 1 - un.idx : i));
#pragma unroll
            for (int q0 = 0; q0 < NQ; q0 += CQ) {
              f32x4 tmp[CQ];
#pragma unroll
              for (int j = 0; j < CQ; ++j) {
                const uint32_t vo = voff + (uint32_t)((q0 + j) * 4096);
                asm volatile("s_nop 4\n\tglobal_load_dwordx4 %0, %1, %2 sc1" : "=v"(tmp[j]) : "v"(vo), "s"(src));
              }
#pragma unroll
              for (int j = 0; j < CQ; ++j) asm volatile("s_waitcnt vmcnt(0)" : "+v"(tmp[j]));
#pragma unroll
              for (int j = 0; j < CQ; ++j) {
                const int qi = q0 + j, blk = qi >> 2, qd = qi & 3;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                  acc[blk / MB][blk % MB][4 * qd + e] =
                      i == 0 ? tmp[j][e] : acc[blk / MB][blk % MB][4 * qd + e] + tmp[j][e];
              }
            }
          }
          if (tid == 0)
            __hip_atomic_store((uint32_t *)a.cut_cnt + tslot, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }

      // ---- epilogue: bias, round once, transpose through LDS, NCHW store ----
      // Accumulator block (A = samples, B = weights): register r of lane l holds
      //   pixel = (r/4)*8 + (l/32)*4 + r%4,  channel = l%32.
      constexpr int RB = stage_row_bytes<E>();
      constexpr int CHUNK_PX = 16 / ES;           // pixels per 16-byte chunk
      constexpr int CHUNKS = 64 / CHUNK_PX;       // chunks per staged row
      unsigned char *stage = (unsigned char *)&Xs[0][0] + (size_t)wave * 32 * RB;
      E *out = (E *)a.out;
      const bool vec_ok = a.out_vec_ok != 0;      // 16-byte chunks never straddle images, aligned
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        if (!store_tile) break;  // a part that was not the last to arrive has nothing to store
        const int col0 = ctile * CT + (wave_c * MB + mb) * 32;  // channel within the group
#pragma unroll
        for (int np = 0; np < NB / 2; ++np) {   // 64 pixels at a time
        const int pw0 = p0 + (wave_p * NB + np * 2) * 32;
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
#pragma unroll
          for (int r4 = 0; r4 < 4; ++r4) {
            const int px = nb * 32 + r4 * 8 + fhalf * 4;
            const f32x16 &c = acc[np * 2 + nb][mb];
            int pexp[4] = {0, 0, 0, 0};
            if constexpr (kPairs) {
              const int4 pe = *(const int4 *)&row_exp[(wave_p * NB + np * 2) * 32 + px];
              pexp[0] = pe.x, pexp[1] = pe.y, pexp[2] = pe.z, pexp[3] = pe.w;
            }
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
              v[e] = kPairs ? __builtin_amdgcn_ldexpf(c[r4 * 4 + e], -(pexp[e] + wexp[mb])) + bv[mb]
                            : fmaf(c[r4 * 4 + e], kSplitUnscale, bv[mb]);
            TR::store4(stage + frow * RB + px * ES, v[0], v[1], v[2], v[3]);
          }
        }
        // the same wave wrote and now reads: only its own LDS operations matter
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll 1
        for (int it = 0; it < 32 * CHUNKS / 64; ++it) {
          const int idx = it * 64 + lane;
          const int row = idx / CHUNKS;        // channel of the block
          const int chunk_i = idx % CHUNKS;
          const int col = col0 + row;
          const int p = pw0 + chunk_i * CHUNK_PX;
          if (col < g.cout_g && p < total_px) {
            const uint4 val = *(const uint4 *)(stage + row * RB + chunk_i * 16);
            const long cbase = (long)grp * g.cout_g + col;
            if (vec_ok && p + CHUNK_PX <= total_px) {
              const int n = p / plane_out;
              const int rem = p - n * plane_out;
              *(uint4 *)(out + ((long)n * g.Cout + cbase) * plane_out + rem) = val;
            } else {
              // (from where it is staged: an array in registers that is indexed is put into LDS, at an address made from the size of the
              // workgroup, and that stands in the dispatch packet, in the host's memory: 2 048 waves read it there before they
              // do anything else, 15 to 20 us.  fp32 N=1 256 channels 28x28, whole call: 41.7 us, without 31.1)
              const E *ve = (const E *)(stage + row * RB + chunk_i * 16);
#pragma unroll 1
              for (int i = 0; i < CHUNK_PX; ++i) {
                const int pi = p + i;
                if (pi < total_px) {
                  const int ni = pi / plane_out;
                  const int ri = pi - ni * plane_out;
                  out[((long)ni * g.Cout + cbase) * plane_out + ri] = ve[i];
                }
              }
            }
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
      }
      // (sums that are not finite, see split3: looked for in the accumulators, mended behind the last unit)
      float t = 0.0f;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int r = 0; r < 16; ++r) t = fmaf(acc[nb][mb][r], 0.0f, t);
      if (!store_tile) skip |= 1u << (u - us.full);
      bad = bad || (store_tile && __any(t != t));
      MDCN_BARRIER_LDS();  // E1
    }
  }

  // ---- This wave's outputs that are not finite, made again one by one.  Lanes read back what the wave has stored, past the
  // caches.  (The arguments are read again from where the launch put them: kept from the kernel's start for this, they
  // would take the main loop's scalar registers, 3% of a call of N=8, 256 channels, 64x64.) ----
  if (bad) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    auto kernarg = __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(kernarg));
    remake_not_finite<CT, WC, MB, NB, AHEAD>(*(const FusedArgs *)kernarg, skip, nk_tile_pad, wave, lane);
  }
}

}  // namespace mdcn
