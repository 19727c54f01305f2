// fp32 forward as fp16 pairs (mdcn_fused_f32.h): the two launches in front of the main kernel's.
#pragma once

#include "mdcn_prepass.h"

namespace mdcn {

// Exponents of the rows of either operand, and what they are made of.
struct PairArgs {
  Geom g;               // of the launch's images
  const float *w;
  void *wp;
  int *wexp;            // [G][n_ctiles][CT]
  uint16_t *row_max;    // the largest magnitude of each input pixel's channels, slab by slab: [image][unit][pixel][slab of the unit], the upper 16
  int unit;             // bits of a float, rounded up; units of `unit` slabs that one group and one deformable group share
  int *row_exp;         // [G][pixel of the launch]
  uint32_t *tab_pix;    // the main kernel's tables, [deformable group, tap][pixel of the launch]: offset of the upper left corner
  float4 *tab_w;        // in the copy, corner weights
  uint32_t img_bytes, row_bytes;
  OffMaskView om;
  int CT, n_ctiles, slabs, slabs_total;
  uint32_t *zero_ptr;   // cut-tile counters
  int zero_n;
};
constexpr int kPairCols = 8;   // output channels of a workgroup
__host__ __device__ inline int pair_col_groups(const Geom &g, int n_ctiles, int CT) { return g.G * n_ctiles * CT / kPairCols; }

// First launch: the largest weight of each output channel (workgroups of kPairCols channels), conv_offset's weights, the input's copy and
// its row_max.
static __global__ __launch_bounds__(256) void pair_relayout_kernel(PairArgs a, const float *__restrict__ in, float *__restrict__ xt, int n_pchunks,
                                                            int wmax_blocks, OffsetPack op) {
  int b = (int)blockIdx.x;
  if (b < wmax_blocks) {
    const Geom &g = a.g;
    const int tid = threadIdx.x, c = tid >> 5, sub = tid & 31;
    for (int i = b * 256 + tid; i < a.zero_n; i += wmax_blocks * 256) a.zero_ptr[i] = 0u;
    const int idx = b * kPairCols + c, tile = idx / a.CT, grp = tile / a.n_ctiles, col = (tile - grp * a.n_ctiles) * a.CT + idx - tile * a.CT;
    const int K = g.cin_g * g.taps;
    uint32_t top = 0u;
    if (col < g.cout_g) {
      const float *row = a.w + (long)(grp * g.cout_g + col) * K;
      if ((uintptr_t)a.w % 16 == 0) {   // (K is a multiple of 32)
#pragma unroll 4
        for (int k = sub * 4; k < K; k += 128) {
          const uint4 v = *(const uint4 *)(row + k);
          top = max(max(top, v.x & 0x7fffffffu), max(v.y & 0x7fffffffu, max(v.z & 0x7fffffffu, v.w & 0x7fffffffu)));
        }
      } else {
        for (int k = sub; k < K; k += 32) top = max(top, __float_as_uint(row[k]) & 0x7fffffffu);
      }
    }
#pragma unroll
    for (int s = 16; s; s >>= 1) top = max(top, (uint32_t)__shfl_xor((int)top, s));
    if (sub == 0) a.wexp[idx] = pair_exponent(__uint_as_float(top));
    return;
  }
  b -= wmax_blocks;
  if (b < op.blocks) {
    pack_offset_chunks<float>(a.g, op, (long)b * 256 + threadIdx.x, (long)op.blocks * 256);
    return;
  }
  relayout_vec_block<float, true>(a.g, in, xt, n_pchunks, b - op.blocks, ChanMap(), 0, a.row_max, a.unit);
}

// Second launch, last workgroups: weights as fp16 pairs, wp[G][n_ctiles][nk][2 half steps][2 planes][CT / 32][64 lanes][8 fp16], a workgroup
// for kPairCols output channels and a slab.
__device__ __forceinline__ void pack_weight_pairs(const PairArgs &a, int b) {
  constexpr int kRow = 32 * 9 + 1;   // floats of a row in LDS (an odd number of words: eight rows, eight banks)
  __shared__ float rows[kPairCols * kRow];
  const Geom &g = a.g;
  const int tid = threadIdx.x, col_groups = pair_col_groups(g, a.n_ctiles, a.CT);
  const int slab = b / col_groups, idx0 = (b - slab * col_groups) * kPairCols;
  const int tile = idx0 / a.CT, grp = tile / a.n_ctiles, cc = idx0 - tile * a.CT, col0 = (tile - grp * a.n_ctiles) * a.CT + cc;
  const int K = g.cin_g * g.taps, nk = a.slabs * g.taps, len = 32 * g.taps;
  const float *src = a.w + (long)(grp * g.cout_g + col0) * K + slab * len;
  const bool staged = g.taps <= 9;
  if (staged) {
    for (int i = tid; i < kPairCols * len; i += 256) {
      const int c = i / len, k = i - c * len;
      rows[c * kRow + k] = col0 + c < g.cout_g ? src[(long)c * K + k] : 0.0f;
    }
    __syncthreads();
  }
  const int blocks = a.CT / 32;
  for (int i = tid; i < kPairCols * 4 * g.taps; i += 256) {
    const int c = i & 7, lane_half = i >> 3 & 1, half = i >> 4 & 1, tap = i >> 5;
    const int e = a.wexp[idx0 + c], k0 = (half * 16 + lane_half * 8) * g.taps + tap;
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = k0 + j * g.taps;
      v[j] = __builtin_amdgcn_ldexpf(staged ? rows[c * kRow + k] : col0 + c < g.cout_g ? src[(long)c * K + k] : 0.0f, e);
    }
    uint2 p0[2], p1[2];
    split2({v[0], v[1], v[2], v[3]}, p0);
    split2({v[4], v[5], v[6], v[7]}, p1);
    uint4 *dst = (uint4 *)a.wp + ((((long)tile * nk + slab * g.taps + tap) * 2 + half) * 2 * blocks + ((cc + c) >> 5)) * 64 + lane_half * 32 +
                 ((cc + c) & 31);
#pragma unroll
    for (int s = 0; s < 2; ++s) dst[(long)s * blocks * 64] = make_uint4(p0[s].x, p0[s].y, p1[s].x, p1[s].y);
  }
}

// ... the others: exponents of the rows of samples.  The largest magnitude there can be in a row -- of an output pixel and the channels of a
// group -- is that of a tap's corners by the largest number of each corner's channels.  Positions and corner weights, which are made for that, are
// kept for the main kernel's tables: made there they are some 750 instructions of a lane for each tile of channels, 10 of a tile's 240 thousand
// clocks (N=8 256 -> 256 64x64), four times that with four deformable groups.  A workgroup has 64 pixels, a wavefront every fourth
// (deformable group, tap) of theirs.  What bounds it is two trips to memory, one behind the other.
__device__ __forceinline__ void sample_exponents(const PairArgs &a, int b) {
  __shared__ float2 found[4][64];
  constexpr int NB = 3;   // (deformable group, tap) pairs at a time
  const Geom &g = a.g;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int plane = g.Ho * g.Wo, total_px = g.N * plane, px_blocks = (total_px + 63) / 64;
  const int grp = b / px_blocks, p = (b - grp * px_blocks) * 64 + lane;
  const int pc = min(p, total_px - 1), n = pc / plane, rem = pc - n * plane, ho = rem / g.Wo, wo = rem - ho * g.Wo;
  const int slab0 = grp * a.slabs, spd = g.ch_per_dg / 32, taps = g.taps, unit = a.unit;
  const int dg0 = slab0 / spd, entries = ((slab0 + a.slabs - 1) / spd - dg0 + 1) * taps;
  const float *off = (const float *)a.om.off + (long)n * a.om.off_n + (long)rem * a.om.off_px;
  const float *msk = (const float *)a.om.msk + (long)n * a.om.msk_n + (long)rem * a.om.msk_px;
  float bound = 0.0f, most = 0.0f;
  float rdy[NB], rdx[NB], rm[NB];
  auto load = [&](int e0) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int e = dg0 * taps + min(e0 + 4 * i, entries - 1);   // (deformable group, tap)
      rdy[i] = off[(long)(2 * e) * a.om.off_ch];
      rdx[i] = off[(long)(2 * e + 1) * a.om.off_ch];
      rm[i] = msk[(long)e * a.om.msk_ch];
    }
  };
  load(wave);
#pragma unroll 1
  for (int e0 = wave; e0 < entries; e0 += 4 * NB) {
    float wt[NB][4];
    uint32_t at[NB][2];   // the pair of pixels in each row
    int sel[NB];          // bit 0: the left corner is the pair's right pixel, bit 1: the right corner its left one
    int first_unit[NB], units[NB], n_units = 1;   // of the group's part of the entry's deformable group
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int e = min(e0 + 4 * i, entries - 1), dgi = e / taps, tap = e - dgi * taps, ti = tap / g.kw, tj = tap - ti * g.kw;
      first_unit[i] = max(slab0, (dg0 + dgi) * spd) / unit;
      units[i] = min(slab0 + a.slabs, (dg0 + dgi + 1) * spd) / unit - first_unit[i];
      n_units = max(n_units, units[i]);
      const float m = mask_value<float>(rm[i], a.om.logit);
      most = fmaxf(most, fabsf(m));
      const TapSample sm = make_tap_sample(ho * g.sh - g.ph + ti * g.dh, wo * g.sw - g.pw + tj * g.dw, rdy[i], rdx[i], m, g.H, g.W);
      wt[i][0] = fabsf(sm.w00), wt[i][1] = fabsf(sm.w01), wt[i][2] = fabsf(sm.w10), wt[i][3] = fabsf(sm.w11);
      if (p < total_px) {   // (an entry past the last repeats that one; groups that share a deformable group write the same)
        const long to = (long)(dg0 * taps + e) * total_px + p;
        a.tab_pix[to] = (uint32_t)n * a.img_bytes + (sm.inside ? (uint32_t)(sm.y0 + 1) * a.row_bytes + (uint32_t)(sm.x0 + 1) * (uint32_t)kRowB
                                                               : (uint32_t)(g.Wp - 1) * (uint32_t)kRowB);
        a.tab_w[to] = make_float4(sm.w00, sm.w01, sm.w10, sm.w11);
      }
      // (a corner outside the image, which adds nothing, counts as the pixel beside it)
      const int xb = max(min(sm.x0, g.W - 2), 0);
      sel[i] = (sm.x0 > xb ? 1 : 0) | (sm.x0 < xb || g.W == 1 ? 2 : 0);
      at[i][0] = (uint32_t)(max(sm.y0, 0) * g.W + xb);
      at[i][1] = (uint32_t)(min(sm.y0 + 1, g.H - 1) * g.W + xb);
    }
    if (e0 + 4 * NB < entries) load(e0 + 4 * NB);   // while the bounds are on their way
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    auto fold = [](uint32_t x, uint32_t y) {
      return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, x), __builtin_bit_cast(u16x2, y)));
    };
    uint32_t top[NB][2][2];   // [row][pixel of the pair], two 16-bit halves each
#pragma unroll
    for (int i = 0; i < NB; ++i) top[i][0][0] = top[i][0][1] = top[i][1][0] = top[i][1][1] = 0u;
    for (int u = 0; u < n_units; ++u) {
      const uint16_t *base[NB];
#pragma unroll
      for (int i = 0; i < NB; ++i)
        base[i] = a.row_max + ((long)n * (a.slabs_total / unit) + first_unit[i] + min(u, units[i] - 1)) * ((long)g.H * g.W * unit);
      auto pairs_of = [&](auto piece) {   // both pixels of a pair in one load
        using L = decltype(piece);
        L v[NB][2];
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int r = 0; r < 2; ++r) __builtin_memcpy(&v[i][r], base[i] + at[i][r] * (uint32_t)unit, sizeof(L));
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int r = 0; r < 2; ++r) {
            uint32_t w[sizeof(L) / 4];
            __builtin_memcpy(w, &v[i][r], sizeof(L));
            if constexpr (sizeof(L) == 4) {
              top[i][r][0] = fold(top[i][r][0], w[0] & 0xffffu);
              top[i][r][1] = fold(top[i][r][1], w[0] >> 16);
            } else {
              constexpr int H = (int)sizeof(L) / 8;
#pragma unroll
              for (int k = 0; k < H; ++k) {
                top[i][r][0] = fold(top[i][r][0], w[k]);
                top[i][r][1] = fold(top[i][r][1], w[H + k]);
              }
            }
          }
      };
      if (unit == 4) {
        pairs_of(uint4());
      } else if (unit == 2) {
        pairs_of(uint2());
      } else if (unit == 1) {
        pairs_of(uint32_t());
      } else {
        const int step = unit % 8 == 0 ? 8 : 1;
        for (int c = 0; c < unit; c += step) {
          uint4 v[NB][2][2];
#pragma unroll
          for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
              for (int q = 0; q < 2; ++q) {   // (an image one pixel wide has no second one)
                const uint16_t *src = base[i] + (at[i][r] + min(q, g.W - 1)) * (uint32_t)unit + c;
                if (step == 8) v[i][r][q] = *(const uint4 *)src;
                else v[i][r][q] = make_uint4(*src, 0u, 0u, 0u);
              }
#pragma unroll
          for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
              for (int q = 0; q < 2; ++q)
                top[i][r][q] = fold(top[i][r][q], fold(fold(v[i][r][q].x, v[i][r][q].y), fold(v[i][r][q].z, v[i][r][q].w)));
        }
      }
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      float sum = 0.0f;
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const float m0 = __uint_as_float(max(top[i][r][0] << 16, top[i][r][0] & 0xffff0000u));
        const float m1 = __uint_as_float(max(top[i][r][1] << 16, top[i][r][1] & 0xffff0000u));
        sum = fmaf(wt[i][2 * r], sel[i] & 1 ? m1 : m0, sum);
        sum = fmaf(wt[i][2 * r + 1], sel[i] & 2 ? m0 : m1, sum);
      }
      bound = fmaxf(bound, sum);
    }
  }
  found[wave][lane] = make_float2(bound, most);
  __syncthreads();
  if (wave == 0 && p < total_px) {
#pragma unroll
    for (int w = 1; w < 4; ++w) bound = fmaxf(bound, found[w][lane].x), most = fmaxf(most, found[w][lane].y);
    a.row_exp[(long)grp * total_px + p] = sample_exponent(bound, most);
  }
}

// (The samples' workgroups come first: theirs is the longer chain.)
static __global__ __launch_bounds__(256) void pair_exponent_kernel(PairArgs a, int sample_blocks) {
  if ((int)blockIdx.x < sample_blocks)
    sample_exponents(a, (int)blockIdx.x);
  else
    pack_weight_pairs(a, (int)blockIdx.x - sample_blocks);
}

}  // namespace mdcn
