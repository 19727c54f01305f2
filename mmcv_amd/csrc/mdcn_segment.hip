// Segment kernel: implicit GEMM  out[cout, pixel] = W[cout, k] * S[k, pixel]  for
// channel counts that do not fill 128-byte slabs of one deformable group.
//
// The channels of a convolution group fall into segments that belong to one
// deformable group; a segment is padded to whole 16-byte chunks and the input
// copy is chunk-major ([N][chunk][H+2][W+2][16 bytes], zero border).  K runs over
// "pairs" (cq neighbouring chunks of a segment, tap).  A wavefront owns 32
// pixels x up to 256 output channels and keeps everything in registers: its lower
// 32 lanes take the even pairs of the pixels and the upper 32 the odd ones,
// each lane reads its pixel's offsets and mask from the NCHW tensors (32 lanes =
// 32 neighbouring pixels), gathers the four corners of cq chunks and blends them,
// and what comes out is a B operand of the 32x32 MFMA but for its rounding (column =
// lane % 32, K half = lane / 32: K may be walked in any order as long as the
// packed weights follow it).  No LDS tile, no barrier in the K loop; a position
// is computed once per pair and used for cq chunks.  Neighbouring lanes sample
// neighbouring pixels and a 16-byte pixel lets eight of them share a cache line.
// The weights are packed in A-operand order and read from L1/L2.
//
// Few pixels: `kshare` waves of the workgroup split the pairs of a pixel block
// among them and add their accumulators up through LDS, in a fixed order.
//
// Samples are fp32 numbers whatever the tensors are, and the sums those of fp32 products: they run on the bf16 matrix
// pipe, three exact planes per sample.  fp32 weights have three planes too and six of the nine products are summed
// (mdcn_fused_f32.h), fp16 weights fit two (five of six), bf16 weights are one (all three).  Weights are split when they are
// packed, samples behind the blend.  fp32 with one chunk a position (half a fragment) takes the fp32 MFMAs.
// ROUND: small 16-bit calls of shapes that the fused kernels take round samples and corner weights to the type as these do,
// and have nothing to split.
//
// What bounds it: the vector-memory path of the CU (64 bytes of corner data per 16 bytes of S): its address unit is busy in
// 76 % of the cycles of the dg8 case below; VALU (position, blend, split) 26 %, MFMAs 16 % (counters).  Measured against the
// one-thread-per-output kernel that these shapes had before: N=2, 64 -> 64 channels, 8 deformable
// groups, 180x320, fp32 23.9 ms -> 193 us a call with fp32 MFMAs, 173 on the bf16 pipe (error against float64 4.3e-7 -> 1.8e-7);
// N=1 64 -> 64 56x56 22.6 -> 19.1 us; N=4, 96 -> 72 channels, 2 deformable groups, 37x53, bf16 1 733 us -> 21, fp16 21
// (19 and 18 with samples rounded to 16 bits; the dg8 case in bf16 80 and 77, in fp16 88 and 76).
#include "mdcn_segment.h"

#include <algorithm>

#include "../../include/mdcn.h"
#include "mdcn_direct.h"
#include "mdcn_fused_f32.h"

namespace mdcn {

namespace {

// On the bf16 matrix pipe: eight channels, one or two chunks, are a lane's half of the K of one MFMA.
constexpr bool seg_split(int es, int cq, bool rounded) { return !rounded && (es == 2 || cq >= 2); }
// bf16 planes of a weight
template <typename E>
constexpr int kSegPlanes = 3;
template <>
constexpr int kSegPlanes<bf16_t> = 1;
template <>
constexpr int kSegPlanes<f16_t> = 2;
int seg_planes(int dtype, bool rounded) {
  return rounded ? 1 : dtype == MDCN_F32 ? kSegPlanes<float> : dtype == MDCN_F16 ? kSegPlanes<f16_t> : kSegPlanes<bf16_t>;
}
// 16-byte weight fragments of one iteration and 32-channel block
constexpr int seg_frags(int es, int planes, int cq) { return es == 2 ? cq * planes : cq >= 2 ? cq / 2 * planes : cq; }

// Weights to A-operand order and the input to chunk planes, one launch: the first
// pack_blocks workgroups repack, the others copy 256 pixels of the bordered plane
// of one chunk each.
template <typename E>
__global__ __launch_bounds__(256) void seg_prepass_kernel(SegArgs a, const E *__restrict__ in,
                                                          const E *__restrict__ w, int pack_blocks, int px_blocks) {
  constexpr int VC = 16 / (int)sizeof(E);
  const Geom &g = a.g;
  const SegPlan &s = a.s;
  if ((int)blockIdx.x < pack_blocks) {
    const bool split = seg_split((int)sizeof(E), s.cq, s.rounded);
    constexpr int CF = 8 / VC;                  // chunks of a fragment when split
    const int qn = split ? s.cq / CF : s.cq;    // fragments of an iteration, when split as planes
    const long total = (long)g.G * s.n_ctiles * s.iters * qn * s.nb * 64;
    const int grp_per_seg = s.cps / s.cq;
    for (long idx = (long)blockIdx.x * 256 + threadIdx.x; idx < total; idx += (long)pack_blocks * 256) {
      long r = idx;
      const int lane = (int)(r & 63);
      r >>= 6;
      const int nb = (int)(r % s.nb);
      r /= s.nb;
      const long frag = r;  // (group, tile, iteration, fragment)
      const int q = (int)(r % qn);
      r /= qn;
      const int it = (int)(r % s.iters);
      r /= s.iters;
      const int ct = (int)(r % s.n_ctiles);
      const int grp = (int)(r / s.n_ctiles);
      const int p = 2 * it + (lane >> 5);
      const int col = (ct * s.nb + nb) * 32 + (lane & 31);
      const int sg = p / g.taps, tap = p - sg * g.taps;
      const int sl = sg / grp_per_seg;                                   // segment of the group
      // first channel of the fragment in it
      const int c0 = ((sg - sl * grp_per_seg) * s.cq + (split ? CF * q : q)) * VC;
      auto at = [&](int i) {
        const bool ok = p < s.pairs && col < g.cout_g && c0 + i < s.seg;
        const E *src = w + ((long)(grp * g.cout_g + (ok ? col : 0)) * g.cin_g + (ok ? sl * s.seg + c0 + i : 0)) * g.taps +
                       (ok ? tap : 0);
        return ok ? *src : from_f32<E>(0.0f);
      };
      if (split) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = to_f32(at(i)) * kSplitScale;
        uint2 p0[3], p1[3];
        split3({v[0], v[1], v[2], v[3]}, p0);
        split3({v[4], v[5], v[6], v[7]}, p1);
        constexpr int NP = kSegPlanes<E>;  // (the planes that are left out are zero)
#pragma unroll
        for (int k = 0; k < NP; ++k)
          ((uint4 *)a.wp)[((frag * NP + k) * s.nb + nb) * 64 + lane] = make_uint4(p0[k].x, p0[k].y, p1[k].x, p1[k].y);
        continue;
      }
      E v[VC];
#pragma unroll
      for (int i = 0; i < VC; ++i) v[i] = at(i);
      uint4 o;
      __builtin_memcpy(&o, v, 16);
      ((uint4 *)a.wp)[idx] = o;
    }
    return;
  }
  int b = (int)blockIdx.x - pack_blocks;
  const int pb = b % px_blocks;
  b /= px_blocks;
  const int chunks = g.G * s.nseg_g * s.cps;
  const int ch = b % chunks, n = b / chunks;
  const int q = pb * 256 + (int)threadIdx.x;
  if (q >= g.Hp * g.Wp) return;
  const int yp = q / g.Wp, y = yp - 1, x = q - yp * g.Wp - 1;
  const int sl = ch / s.cps, c0 = (ch - sl * s.cps) * VC;
  const bool inside = y >= 0 && y < g.H && x >= 0 && x < g.W;
  const long plane = (long)g.H * g.W;
  const E *src = in + ((long)n * g.Cin + (long)sl * s.seg) * plane + (inside ? (long)y * g.W + x : 0);
  E v[VC];
#pragma unroll
  for (int i = 0; i < VC; ++i) v[i] = src[(long)min(c0 + i, s.seg - 1) * plane];
#pragma unroll
  for (int i = 0; i < VC; ++i)
    if (!inside || c0 + i >= s.seg) v[i] = from_f32<E>(0.0f);
  uint4 o;
  __builtin_memcpy(&o, v, 16);
  *(uint4 *)((unsigned char *)const_cast<void *>(a.xt) + (size_t)n * a.img_bytes + (size_t)ch * a.plane_bytes +
             (size_t)q * 16) = o;
}

// Whether a wave has registers for the weight fragments of a step beside the corners and samples of cq chunks.
constexpr bool seg_fits(int es, int planes, int nb, int cq) {
  return seg_frags(es, planes, cq) * nb <= (cq == 4 ? 16 : 18) && cq * nb <= 12;
}

// Waves per SIMD the register budget is cut for.
constexpr int seg_occupancy(int ES, int NB, int CQ, bool rounded) {
  if (seg_split(ES, CQ, rounded)) return CQ * NB <= 4 && CQ == 2 ? 3 : 2;
  return CQ * NB <= 4 && NB <= 2 ? 4 : (NB <= 4 && CQ * NB <= 8 ? 3 : 2);
}

// 16 bytes of channels of one pixel from the same 16 bytes at its four corners, in fp32.
template <typename E>
__device__ __forceinline__ void blend(const uint4 (&v)[4], const uint32_t (&w)[4], float *o) {
  constexpr int VC = 16 / (int)sizeof(E);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint32_t d[4] = {v[q].x, v[q].y, v[q].z, v[q].w};
    const float wq = __uint_as_float(w[q]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float c[VC / 4];
      if constexpr (VC == 4)
        c[0] = __uint_as_float(d[j]);
      else
        ElemTraits<E>::unpack2(d[j], c[0], c[1]);
#pragma unroll
      for (int k = 0; k < VC / 4; ++k) o[VC / 4 * j + k] = q == 0 ? wq * c[k] : fmaf(wq, c[k], o[VC / 4 * j + k]);
    }
  }
}

template <typename E, int NB, int CQ, bool ROUND>
__global__ __launch_bounds__(256, seg_occupancy((int)sizeof(E), NB, CQ, ROUND)) void segment_kernel(SegArgs a) {
  constexpr int VC = 16 / (int)sizeof(E);
  const Geom &g = a.g;
  const SegPlan &s = a.s;
  extern __shared__ __align__(16) unsigned char smem[];
  // {offset channel of dy, mask channel, ti * dh << 16 | tj * dw, first chunk} of every pair
  uint4 *tab = (uint4 *)smem;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int pxl = lane & 31, half = lane >> 5;

  long L = xcd_work_index(a.n_work);
  if (L < 0) return;
  const int ct = (int)(L % s.n_ctiles);
  L /= s.n_ctiles;
  const int grp = (int)(L % g.G);
  const int ptile = (int)(L / g.G);
  const int wpx = 4 / s.kshare;                 // pixel blocks of the workgroup
  const int ks = wave & (s.kshare - 1);
  const long p0 = ((long)ptile * wpx + wave / s.kshare) * 32;

  const int grp_per_seg = s.cps / s.cq;
  for (int p = tid; p < s.pairs; p += 256) {
    const int sg = p / g.taps, tap = p - sg * g.taps;
    const int sl = sg / grp_per_seg;
    const int ti = tap / g.kw, tj = tap - ti * g.kw;
    const int dgi = ((grp * s.nseg_g + sl) * s.seg) / g.ch_per_dg;
    tab[p] = make_uint4((uint32_t)((dgi * g.taps + tap) * 2), (uint32_t)(dgi * g.taps + tap),
                        ((uint32_t)(ti * g.dh) << 16) | (uint32_t)(tj * g.dw),
                        (uint32_t)((grp * s.nseg_g + sl) * s.cps + (sg - sl * grp_per_seg) * s.cq));
  }
  __syncthreads();

  const int plane_out = g.Ho * g.Wo;
  const long pp = min(p0 + pxl, a.total_px - 1);
  const int n = (int)(pp / plane_out);
  const int rem = (int)(pp - (long)n * plane_out);
  const int ho = rem / g.Wo, wo = rem - ho * g.Wo;
  const int by = ho * g.sh - g.ph, bx = wo * g.sw - g.pw;
  const E *off = (const E *)a.om.off + (long)n * a.om.off_n + (long)rem * a.om.off_px;
  const E *msk = (const E *)a.om.msk + (long)n * a.om.msk_n + (long)rem * a.om.msk_px;
  const unsigned char *xt = (const unsigned char *)a.xt;
  const uint32_t img = (uint32_t)n * a.img_bytes;

  struct Raw {
    E dy, dx, m;
    uint32_t tij, chunk;
  };
  auto load_om = [&](int i, Raw &r) {
    const int p = 2 * i + half;
    const uint4 t = tab[min(p, s.pairs - 1)];
    const E *o = off + (long)t.x * a.om.off_ch;
    r.dy = o[0];
    r.dx = o[a.om.off_ch];
    r.m = msk[(long)t.y * a.om.msk_ch];
    // (the odd pair out: a position outside, i.e. zeros, and not a second copy of the last pair)
    r.tij = p < s.pairs ? t.z : 0x7fff0000u;
    r.chunk = t.w;
  };
  constexpr bool kSplit = seg_split((int)sizeof(E), CQ, ROUND);
  struct Gather {
    uint4 v[CQ][4];
    uint32_t w[4];
  };
  auto gather = [&](const Raw &r, Gather &v) {
    const TapSample sm = make_tap_sample(by + (int)(r.tij >> 16), bx + (int)(r.tij & 0xffffu), to_f32(r.dy), to_f32(r.dx),
                                         mask_value<E>(r.m, a.om.logit) * (kSplit ? kSplitScale : 1.0f), g.H, g.W);
    // (a position outside reads border pixels: see corner_offset())
    const uint32_t pix = sm.inside ? (uint32_t)((sm.y0 + 1) * g.Wp + sm.x0 + 1) : (uint32_t)(g.Wp - 1);
    uint32_t o = img + r.chunk * a.plane_bytes + pix * 16u;
    ElemTraits<typename std::conditional<ROUND, E, float>::type>::table_weights(sm, v.w);
#pragma unroll
    for (int q = 0; q < CQ; ++q) {
      const unsigned char *top = xt + o, *bot = xt + (o + a.row_bytes);
      v.v[q][0] = *(const uint4 *)top;
      v.v[q][1] = *(const uint4 *)(top + 16);
      v.v[q][2] = *(const uint4 *)bot;
      v.v[q][3] = *(const uint4 *)(bot + 16);
      o += a.plane_bytes;
    }
  };
  constexpr int NP = ROUND ? 1 : kSegPlanes<E>;
  constexpr int FR = seg_frags((int)sizeof(E), NP, CQ);
  const uint4 *wp = (const uint4 *)a.wp + (size_t)(grp * s.n_ctiles + ct) * s.iters * (FR * NB * 64) + lane;
  auto load_w = [&](int i, uint4 (&wf)[FR][NB]) {
    const uint4 *src = wp + (size_t)i * (FR * NB * 64);
#pragma unroll
    for (int q = 0; q < FR; ++q)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) wf[q][nb] = src[(q * NB + nb) * 64];
  };

  f32x16 acc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[nb][r] = 0.0f;

  const int i0 = s.iters * ks / s.kshare, i1 = s.iters * (ks + 1) / s.kshare;
  if (i0 < i1) {
    Raw raw;
    Gather gv;
    uint4 wf[FR][NB];
    load_om(i0, raw);
    gather(raw, gv);
    load_w(i0, wf);
    load_om(min(i0 + 1, i1 - 1), raw);
    for (int i = i0; i < i1; ++i) {
      float x[ROUND ? 1 : CQ * VC];
      uint4 xr[ROUND ? CQ : 1];
#pragma unroll
      for (int q = 0; q < CQ; ++q) {
        if constexpr (ROUND)
          xr[q] = ElemTraits<E>::blend(gv.v[q][0], gv.v[q][1], gv.v[q][2], gv.v[q][3],
                                       make_uint4(gv.w[0], gv.w[1], gv.w[2], gv.w[3]));
        else
          blend<E>(gv.v[q], gv.w, x + q * VC);
      }
      uint4 wc[kSplit ? 1 : FR][NB];  // (split samples leave no registers for both: the next fragments are fetched behind the products)
      if constexpr (!kSplit) {
#pragma unroll
        for (int q = 0; q < FR; ++q)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) wc[q][nb] = wf[q][nb];
      }
      // (the last iteration fetches its own data again: nobody reads it)
      gather(raw, gv);
      load_om(min(i + 2, i1 - 1), raw);
      if constexpr (kSplit) {
#pragma unroll
        for (int q = 0; q < CQ * VC / 8; ++q) {
          uint2 lo[3], hi[3];
          const float *f = x + 8 * q;
          split3({f[0], f[1], f[2], f[3]}, lo);
          split3({f[4], f[5], f[6], f[7]}, hi);
          auto products = [&](int xp, int wpl) {
            const uint4 xv = make_uint4(lo[xp].x, lo[xp].y, hi[xp].x, hi[xp].y);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) ElemTraits<bf16_t>::mma(acc[nb], wf[NP * q + wpl][nb], xv);
          };
          products(2, 0);  // smallest terms first
          if constexpr (NP > 2) products(0, 2);
          if constexpr (NP > 1) products(1, 1);
          products(1, 0);
          if constexpr (NP > 1) products(0, 1);
          products(0, 0);
        }
      } else {
#pragma unroll
        for (int q = 0; q < CQ; ++q) {
          if constexpr (!ROUND)
            xr[0] = make_uint4(__float_as_uint(x[4 * q]), __float_as_uint(x[4 * q + 1]), __float_as_uint(x[4 * q + 2]),
                               __float_as_uint(x[4 * q + 3]));
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) ElemTraits<E>::mma(acc[nb], wc[q][nb], xr[ROUND ? q : 0]);
        }
      }
      if constexpr (kSplit) __builtin_amdgcn_sched_barrier(0);
      load_w(min(i + 1, i1 - 1), wf);
    }
  }

  // register r of lane l: output channel (r/4)*8 + (l/32)*4 + r%4 of the block, pixel l%32
  E *out = (E *)a.out;
  const bool px_ok = p0 + pxl < a.total_px;
  E *dst = out + ((long)n * g.Cout + (long)grp * g.cout_g) * plane_out + rem;
  float bad = 0.0f;   // NaN once a sum is not finite
  auto put = [&](int nb, int r, float v) {
    if constexpr (kSplit) {
      bad = fmaf(v, 0.0f, bad);
      v *= kSplitUnscale;
    }
    const int col = (ct * NB + nb) * 32 + (r >> 2) * 8 + half * 4 + (r & 3);
    if (px_ok && col < g.cout_g) {
      if (a.bias) v += to_f32(((const E *)a.bias)[grp * g.cout_g + col]);
      dst[(long)col * plane_out] = from_f32<E>(v);
    }
  };
  if (s.kshare == 1) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int r = 0; r < 16; ++r) put(nb, r, acc[nb][r]);
  } else {
    float *red = (float *)(smem + (size_t)s.pairs * 16);  // [wave][16][64 lanes]
    const int w0 = wave - ks;
    const int per = 16 / s.kshare;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      __syncthreads();
#pragma unroll
      for (int r = 0; r < 16; ++r) red[(wave * 16 + r) * 64 + lane] = acc[nb][r];
      __syncthreads();
      for (int r = ks * per; r < (ks + 1) * per; ++r) {
        float v = 0.0f;
        for (int k = 0; k < s.kshare; ++k) v += red[((w0 + k) * 16 + r) * 64 + lane];
        put(nb, r, v);
      }
    }
  }
  if constexpr (kSplit) {
    // sums that are not finite (split3): this lane's outputs that are not, one by one.  It reads back what it has
    // stored, past the caches.
    if (__any(bad != bad)) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      const int per = 16 / s.kshare;
#pragma unroll 1
      for (int i = 0; i < NB * per; ++i) {
        const int nb = i / per, r = ks * per + i % per;
        const int col = (ct * NB + nb) * 32 + (r >> 2) * 8 + half * 4 + (r & 3);
        if (!px_ok || col >= g.cout_g) continue;
        E *o = dst + (long)col * plane_out;
        using U = typename std::conditional<sizeof(E) == 2, uint16_t, uint32_t>::type;
        const float was = to_f32(__builtin_bit_cast(E, __hip_atomic_load((const U *)o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)));
        if (was - was == 0.0f) continue;
        const int co = grp * g.cout_g + col;
        const float v = direct_sum<E, true>(g, (const E *)a.in + (long)n * g.Cin * g.H * g.W, (long)g.H * g.W, 1, a.om,
                                            (const E *)a.weight, n, co, ho, wo);
        *o = from_f32<E>(v + (a.bias ? to_f32(((const E *)a.bias)[co]) : 0.0f));
      }
    }
  }
}

template <typename E, int NB, int CQ, bool ROUND = false>
hipError_t launch(const SegArgs &a, hipStream_t st) {
  const size_t lds = (size_t)a.s.pairs * 16 + (a.s.kshare > 1 ? 4 * 16 * 64 * 4 : 0);
  hipLaunchKernelGGL((segment_kernel<E, NB, CQ, ROUND>), dim3((unsigned)((a.n_work + 7) / 8 * 8)), dim3(256), lds, st, a);
  return hipGetLastError();
}

template <typename E, int CQ>
hipError_t launch_nb(const SegArgs &a, hipStream_t st) {
  if constexpr (sizeof(E) == 2) {
    if (a.s.rounded) return a.s.nb == 1 ? launch<E, 1, CQ, true>(a, st) : a.s.nb == 2 ? launch<E, 2, CQ, true>(a, st) : hipErrorInvalidValue;
  }
  switch (a.s.nb) {
    case 1: return launch<E, 1, CQ>(a, st);
    case 2: return launch<E, 2, CQ>(a, st);
    default: break;
  }
  if constexpr (seg_fits((int)sizeof(E), kSegPlanes<E>, 3, CQ)) {
    if (a.s.nb == 3) return launch<E, 3, CQ>(a, st);
  }
  if constexpr (seg_fits((int)sizeof(E), kSegPlanes<E>, 4, CQ)) {
    if (a.s.nb == 4) return launch<E, 4, CQ>(a, st);
  }
  if constexpr (seg_fits((int)sizeof(E), kSegPlanes<E>, 6, CQ)) {
    if (a.s.nb == 6) return launch<E, 6, CQ>(a, st);
  }
  if constexpr (CQ == 1) {
    if (a.s.nb == 8) return launch<E, 8, CQ>(a, st);
  }
  return hipErrorInvalidValue;
}

template <typename E>
hipError_t launch_e(const SegArgs &a, hipStream_t st) {
  return a.s.cq == 1 ? launch_nb<E, 1>(a, st) : a.s.cq == 2 ? launch_nb<E, 2>(a, st) : launch_nb<E, 4>(a, st);
}

template <typename E>
hipError_t prepass_e(const SegArgs &a, bool pack, hipStream_t st) {
  const int px_blocks = (a.g.Hp * a.g.Wp + 255) / 256;
  const long blocks = (long)a.g.N * a.g.G * a.s.nseg_g * a.s.cps * px_blocks;
  const long wtotal = (long)a.s.wp_bytes / 16;
  const int pack_blocks = pack ? (int)std::max<long>(1, std::min<long>(wtotal / 256, 512)) : 0;
  hipLaunchKernelGGL(seg_prepass_kernel<E>, dim3((unsigned)(blocks + pack_blocks)), dim3(256), 0, st, a, (const E *)a.in,
                     (const E *)a.weight, pack_blocks, px_blocks);
  return hipGetLastError();
}

}  // namespace

bool seg_plan(const Geom &g, int dtype, bool rounded, int n_images, bool may_share, int cus, SegPlan *s) {
  const int es = dtype == MDCN_F32 ? 4 : 2, VC = 16 / es;
  s->rounded = rounded && es == 2;
  const int planes = seg_planes(dtype, s->rounded);
  int u = g.cin_g, v = g.ch_per_dg;
  while (v) {
    const int t = u % v;
    u = v;
    v = t;
  }
  s->seg = u;
  s->nseg_g = g.cin_g / s->seg;
  const int cps0 = (s->seg + VC - 1) / VC;
  const int blocks = (g.cout_g + 31) / 32;
  s->n_ctiles = (blocks + 7) / 8;
  s->nb = (blocks + s->n_ctiles - 1) / s->n_ctiles;
  if (s->nb == 5) s->nb = 6;
  if (s->nb == 7) s->nb = 8;
  // Chunks per position: as many as share one without padding much.  A chunk costs its gather and
  // blend, a position about one and a half of that.
  double best = 0.0;
  s->cq = 0;
  for (int cq = 4; cq >= 1; cq /= 2) {
    if (!seg_fits(es, planes, s->nb, cq)) continue;
    const int groups = (cps0 + cq - 1) / cq;
    const double cost = groups * 1.5 + groups * cq;
    if (s->cq == 0 || cost < best) best = cost, s->cq = cq;
  }
  s->cps = (cps0 + s->cq - 1) / s->cq * s->cq;
  const long pairs = (long)s->nseg_g * (s->cps / s->cq) * g.taps;
  if (pairs > kSegPairsMax) return false;
  if ((long)(g.kh - 1) * g.dh > 0xffff || (long)(g.kw - 1) * g.dw > 0xffff) return false;
  s->pairs = (int)pairs;
  s->iters = (s->pairs + 1) / 2;
  const uint64_t img = (uint64_t)g.G * s->nseg_g * s->cps * g.Hp * g.Wp * 16;
  if (img * (uint64_t)n_images > 0xF0000000ull) return false;
  s->xt_bytes = (size_t)(img * (uint64_t)n_images);
  s->wp_bytes = (size_t)g.G * s->n_ctiles * s->iters * seg_frags(es, planes, s->cq) * s->nb * 1024;
  // Waves of a workgroup share a pixel block's K range while that leaves the chip's SIMDs short of two waves.
  const long waves = ((long)n_images * g.Ho * g.Wo + 31) / 32 * s->n_ctiles * g.G;
  s->kshare = 1;
  while (may_share && s->kshare < 4 && waves * s->kshare < 8L * cus && s->iters >= 4 * s->kshare) s->kshare *= 2;
  return true;
}

hipError_t seg_prepass(int dtype, const SegArgs &a, bool pack, hipStream_t st) {
  switch (dtype) {
    case MDCN_F32: return prepass_e<float>(a, pack, st);
    case MDCN_F16: return prepass_e<f16_t>(a, pack, st);
    default: return prepass_e<bf16_t>(a, pack, st);
  }
}

hipError_t seg_forward(int dtype, const SegArgs &a, hipStream_t st) {
  switch (dtype) {
    case MDCN_F32: return launch_e<float>(a, st);
    case MDCN_F16: return launch_e<f16_t>(a, st);
    default: return launch_e<bf16_t>(a, st);
  }
}

}  // namespace mdcn
