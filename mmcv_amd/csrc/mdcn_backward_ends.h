// The two launches at the ends of the matrix-core backward: everything its three
// main kernels read that is not an input of the call (pre-pass), and everything
// they leave as fp32 or partial sums turned into the gradients (finish).  Each is
// one launch whose workgroups are dealt out to the jobs by ranges of the block
// index: the jobs are independent, most are small, and a launch of its own costs
// each some four microseconds on the device and as much on the host.
#pragma once

#include "mdcn_backward_fused.h"
#include "mdcn_prepass.h"

namespace mdcn {

constexpr int kPreJobs = 9;
enum { kPreX, kPreG, kPreBiasEarly, kPreRows, kPreZero, kPreColPad, kPreWeight, kPreFar, kPreBias };

struct BwdPreArgs {
  Geom g;
  ChanMap im, om;          // padded orders of the input and output channels
  int cin_p, cout_p;
  int end[kPreJobs];       // job j has the blocks from end[j - 1] on
  const void *in, *gout, *w;
  void *xt, *gT, *wT, *gpad, *col;
  uint16_t *gmax;          // fp32 as fp16 pairs, or null: see ColGradArgs
  int *wexp;
  void *wpair;
  float *gin32;
  long n_in;               // elements of gin32
  int x_chunks, g_chunks;  // pixel chunks of the re-layouts
  long P_pad;
  long col_rows;           // rows of col whose padding is cleared
  int run;                 // WGradArgs::run
  int M_pad;
  int wt_run;              // wT in runs of this many output channels (see there), or 0
  const void *off;
  long n_off, off_step;    // one offset in off_step is looked at
  float far_from;          // ... and counted when it is larger than this
  uint32_t *far;           // one count per block of the job
  float *bpart;            // [Cout][bsplits]
  int bsplits;
};

constexpr int kPrePairRows = 8;              // rows of wT a block writes as fp16 pairs
constexpr int kPreZeroPerBlock = 256 * 32;   // floats a block of the zero job clears
constexpr int kPrePadPerBlock = 256 * 8;     // elements a block of the col-pad job clears

// fp32 as fp16 pairs: wT, and wpair, which is wT with its rows scaled by a power of two that goes by the largest finite number of each, and split.  The 32 values of a slab are four
// times eight, which a lane of the product takes at a time: the first halves of eight in one 16-byte piece, the second ones in the piece two behind
// it.  32 lanes a row, eight output channels each.
__device__ __forceinline__ void pack_weight_row_pairs(const BwdPreArgs &a, int b) {
  const Geom &g = a.g;
  const int lane = threadIdx.x & 31;
  const long row = (long)b * kPrePairRows + ((int)threadIdx.x >> 5);
  if (row >= (long)g.G * a.M_pad) return;
  const int grp = (int)(row / a.M_pad), m = (int)(row - (long)grp * a.M_pad);
  const int tap = m / a.im.cgp;
  int room;
  const int c = chan_source(a.im, m - tap * a.im.cgp, room);  // (of the first group: channel within a group)
  const bool there = tap < g.taps && room > 0;
  const long pitch = (long)g.cin_g * g.taps;
  const float *src = (const float *)a.w + (long)grp * g.cout_g * pitch + (long)c * g.taps + tap;
  const int eights = a.om.cgp / 8;
  // values j of eight number o: of pieces q and q + 2 of their slab
  auto load = [&](int o, float (&v)[8]) {
    const int q = (o >> 1 & 1) * 4 + (o & 1), co0 = (o >> 2) * 32 + q * 4;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int co = co0 + (j & 3) + (j >> 2) * 8;
      v[j] = there && o < eights && co < g.cout_g ? src[co * pitch] : 0.0f;
    }
  };
  float first[8], v[8];
  uint32_t top = 0u;
  auto largest = [&](const float (&x)[8]) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t t = __float_as_uint(x[j]) & 0x7fffffffu;
      top = max(top, t < 0x7f800000u ? t : 0u);
    }
  };
  load(lane, first);
  largest(first);
  for (int o = lane + 32; o < eights; o += 32) {
    load(o, v);
    largest(v);
  }
#pragma unroll
  for (int s = 16; s; s >>= 1) top = max(top, (uint32_t)__shfl_xor((int)top, s));
  const int e = pair_exponent(__uint_as_float(top));
  if (lane == 0) a.wexp[row] = e;
  uint4 *dst = (uint4 *)a.wpair + row * (a.om.cgp / 4);
  float4 *whole = (float4 *)a.wT + row * (a.om.cgp / 4);
  for (int o = lane; o < eights; o += 32) {
    if (o != lane) load(o, v);
    const int at = (o >> 2) * 8 + (o >> 1 & 1) * 4 + (o & 1);
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = o == lane ? first[j] : v[j];
    whole[at] = make_float4(x[0], x[1], x[2], x[3]);
    whole[at + 2] = make_float4(x[4], x[5], x[6], x[7]);
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = __builtin_amdgcn_ldexpf(x[j], e);
    uint2 lo[2], hi[2];
    split2({x[0], x[1], x[2], x[3]}, lo);
    split2({x[4], x[5], x[6], x[7]}, hi);
    uint4 *d = dst + at;
    d[0] = make_uint4(lo[0].x, lo[0].y, hi[0].x, hi[0].y);
    d[2] = make_uint4(lo[1].x, lo[1].y, hi[1].x, hi[1].y);
  }
}

template <typename E>
__global__ __launch_bounds__(256) void bwd_prepass_kernel(BwdPreArgs a) {
  constexpr int EPV = 16 / (int)sizeof(E);
  const Geom &g = a.g;
  const int tid = threadIdx.x;
  const long plane = (long)g.Ho * g.Wo;
  int b = (int)blockIdx.x;
  if (b < a.end[kPreX]) {  // zero-bordered copy of the input in 32-byte records (what the scatter kernel reads per corner)
    relayout_vec_block<E, true, 32, true>(g, (const E *)a.in, (E *)a.xt, a.x_chunks, b, a.im, a.cin_p);
    return;
  }
  if (b < a.end[kPreG]) {  // pixel-major grad_output
    Geom gg = g;
    gg.Cin = g.Cout;
    gg.H = g.Ho;
    gg.W = g.Wo;
    relayout_vec_block<E, false, 128, true>(gg, (const E *)a.gout, (E *)a.gT, a.g_chunks, b - a.end[kPreX], a.om, a.cout_p, a.gmax);
    return;
  }
  __shared__ float red[4];
  if (b >= a.end[kPreFar] || (b >= a.end[kPreG] && b < a.end[kPreBiasEarly])) {
    // sums of grad_output over the pixels, a share of an output channel's runs per block (in one of two places of the launch)
    const int bi = b - (b >= a.end[kPreFar] ? a.end[kPreFar] : a.end[kPreG]);
    const int co = bi / a.bsplits, split = bi - co * a.bsplits;
    const int runs = (int)((plane + kBiasRun - 1) / kBiasRun);
    float s = 0.0f;
    for (int w = split; w < g.N * runs; w += a.bsplits) {
      const int n = w / runs, p0 = (w - n * runs) * kBiasRun;
      const int len = (int)min((long)kBiasRun, plane - p0);
      const E *src = (const E *)a.gout + ((long)n * g.Cout + co) * plane + p0;
      const int nv = len / EPV;
#pragma unroll 4
      for (int v = tid; v < nv; v += 256) {
        uint4 q;
        __builtin_memcpy(&q, src + (long)v * EPV, 16);
        const E *e = (const E *)&q;
#pragma unroll
        for (int i = 0; i < EPV; ++i) s += to_f32(e[i]);
      }
      for (int i = nv * EPV + tid; i < len; i += 256) s += to_f32(src[i]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((tid & 63) == 0) red[tid >> 6] = s;
    __syncthreads();
    if (tid == 0) a.bpart[(long)co * a.bsplits + split] = (red[0] + red[1]) + (red[2] + red[3]);
    return;
  }
  if (b < a.end[kPreRows]) {  // grad_output with rows that start 16-byte aligned, zeros behind the image
    const long per_row = a.P_pad / EPV;
    const long i = (long)(b - a.end[kPreBiasEarly]) * 256 + tid;
    const long r = i / per_row;
    const int p = (int)(i - r * per_row) * EPV;
    if (r >= (long)g.N * g.Cout) return;
    const E *src = (const E *)a.gout + r * plane + p;
    uint4 v;
    if (p + EPV <= plane) {
      __builtin_memcpy(&v, src, 16);
    } else {
      E e[EPV];
#pragma unroll
      for (int k = 0; k < EPV; ++k) e[k] = p + k < plane ? src[k] : from_f32<E>(0.0f);
      __builtin_memcpy(&v, e, 16);
    }
    *(uint4 *)((E *)a.gpad + i * EPV) = v;
    return;
  }
  if (b < a.end[kPreZero]) {  // the fp32 grad_input the scatter kernel adds into
    const long i0 = (long)(b - a.end[kPreRows]) * kPreZeroPerBlock;
    const bool vec = ((uintptr_t)a.gin32 % 16) == 0;
    for (int k = 0; k < kPreZeroPerBlock / 1024; ++k) {
      const long i = i0 + (long)k * 1024 + tid * 4;
      if (vec && i + 4 <= a.n_in) {
        *(float4 *)(a.gin32 + i) = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      } else {
        for (int j = 0; j < 4; ++j)
          if (i + j < a.n_in) a.gin32[i + j] = 0.0f;
      }
    }
    return;
  }
  if (b < a.end[kPreColPad]) {  // padding pixels [P, P_pad) of the columns matrix: of its rows, or of runs of them
    const int run = sizeof(E) == 2 ? a.run : 1;
    const int padn = (int)(a.P_pad - plane) * run;
    const long i0 = (long)(b - a.end[kPreZero]) * kPrePadPerBlock;
    for (int k = 0; k < kPrePadPerBlock / 256; ++k) {
      const long i = i0 + k * 256 + tid, r = i / padn;
      if (r < a.col_rows / run) ((E *)a.col)[(r * a.P_pad + plane) * run + (i - r * padn)] = from_f32<E>(0.0f);
    }
    return;
  }
  if (b < a.end[kPreWeight]) {
    // weight[Cout][cin_g][taps] -> wT[G][M_pad][om.cgp], row m = tap * im.cgp + padded channel, zero where
    // either channel is padding and in the rows up to M_pad.  With wt_run it is [G][run][M_pad][wt_run], the last run what is left: what
    // bwd_fused_kernel copies at a time is one piece of memory for a tap (256 bytes of rows 1 KB apart, as with
    // 512 output channels, are in one of four channels of the L2).
    if constexpr (sizeof(E) == 4) {
      if (a.wexp) {
        pack_weight_row_pairs(a, b - a.end[kPreColPad]);
        return;
      }
    }
    const long total = (long)g.G * a.M_pad * a.om.cgp;
    const long idx = (long)(b - a.end[kPreColPad]) * 256 + tid;
    if (idx >= total) return;
    long r = idx;
    const int co = (int)(r % a.om.cgp);
    r /= a.om.cgp;
    const int m = (int)(r % a.M_pad);
    const int grp = (int)(r / a.M_pad);
    const int tap = m / a.im.cgp;
    int room;
    const int c = chan_source(a.im, m - tap * a.im.cgp, room);  // (of the first group: channel within a group)
    E v = from_f32<E>(0.0f);
    if (tap < g.taps && room > 0 && co < g.cout_g)
      v = ((const E *)a.w)[((long)(grp * g.cout_g + co) * g.cin_g + c) * g.taps + tap];
    long at = idx;
    if (a.wt_run) {
      const int run = co / a.wt_run, len = min(a.wt_run, a.om.cgp - run * a.wt_run);
      at = (long)grp * a.M_pad * a.om.cgp + (long)run * a.wt_run * a.M_pad + (long)m * len + (co - run * a.wt_run);
    }
    ((E *)a.wT)[at] = v;
    return;
  }
  {  // offsets that leave the scatter kernel's window, counted in a sample
    const int nb = a.end[kPreFar] - a.end[kPreWeight], bi = b - a.end[kPreWeight];
    float cnt = 0.0f;  // (64 Ki samples at most: exact)
    for (long i = ((long)bi * 256 + tid) * a.off_step; i < a.n_off; i += (long)nb * 256 * a.off_step)
      cnt += fabsf(to_f32(((const E *)a.off)[i])) > a.far_from ? 1.0f : 0.0f;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o);
    if ((tid & 63) == 0) red[tid >> 6] = cnt;
    __syncthreads();
    if (tid == 0) a.far[bi] = (uint32_t)((red[0] + red[1]) + (red[2] + red[3]));
    return;
  }
}

constexpr int kFinJobs = 5;
enum { kFinInput, kFinOffset, kFinMask, kFinWeight, kFinBias };

struct BwdFinArgs {
  Geom g;
  ChanMap im;
  int end[kFinJobs];
  const float *gin32;   // 16-bit tensors: fp32 grad_input
  void *gin;
  long n_in;
  const float *poff, *pmask;   // [parts][...]
  void *goff, *gmask;
  long off_total, mask_total;
  int parts;
  // fused: cut tiles of each pass of images, `cut` of the first and cut_last of the last
  FusedSchedule sched, sched_last;
  const float *fpart;   // [pass][workgroup][3 taps][256]
  int tw_log, n_chunk, chunks, cut, cut_last;
  const float *wpart;   // [splits][G][cout_g][taps * im.cgp]
  void *gw;
  int splits;
  const float *bpart;   // [Cout][bsplits]
  void *gb;
  int bsplits;
};

// dst[0 .. n) = sum over `parts` of src[part][0 .. n), rounded once; four elements per thread.
template <typename E>
__device__ __forceinline__ void sum_parts_block(const float *__restrict__ src, E *__restrict__ dst, long n, int parts, int b) {
  const long i = ((long)b * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  if (n % 4 == 0 && (uintptr_t)src % 16 == 0) {
    float4 s = *(const float4 *)(src + i);
    for (int p = 1; p < parts; ++p) {
      const float4 t = *(const float4 *)(src + (long)p * n + i);
      s.x += t.x; s.y += t.y; s.z += t.z; s.w += t.w;
    }
    struct Out4 { E v[4]; } o;
    o.v[0] = from_f32<E>(s.x); o.v[1] = from_f32<E>(s.y); o.v[2] = from_f32<E>(s.z); o.v[3] = from_f32<E>(s.w);
    __builtin_memcpy(dst + i, &o, sizeof(o));
    return;
  }
  for (int k = 0; k < 4 && i + k < n; ++k) {
    float s = 0.0f;
    for (int p = 0; p < parts; ++p) s += src[(long)p * n + i + k];
    dst[i + k] = from_f32<E>(s);
  }
}

constexpr int kFinWeightCh = 64;   // padded channels of a row a block of the weight job handles

template <typename E>
__global__ __launch_bounds__(256) void bwd_finish_kernel(BwdFinArgs a) {
  const Geom &g = a.g;
  const int tid = threadIdx.x;
  const int b = (int)blockIdx.x;
  if (b < a.end[kFinInput]) {
    sum_parts_block<E>(a.gin32, (E *)a.gin, a.n_in, 1, b);
    return;
  }
  if (b < a.end[kFinOffset] && a.chunks > 0) {
    const int bi = b - a.end[kFinInput], per = a.cut * 3 * g.taps, c = per ? min(bi / per, a.chunks - 1) : a.chunks - 1;
    fused_sums_block<E>(g, c == a.chunks - 1 ? a.sched_last : a.sched, a.tw_log, c * a.n_chunk,
                        a.fpart + (long)c * FusedSchedule::kGroups * 3 * g.taps * 256, (E *)a.goff, (E *)a.gmask, bi - c * per);
    return;
  }
  if (b < a.end[kFinOffset]) {
    sum_parts_block<E>(a.poff, (E *)a.goff, a.off_total, a.parts, b - a.end[kFinInput]);
    return;
  }
  if (b < a.end[kFinMask]) {
    sum_parts_block<E>(a.pmask, (E *)a.gmask, a.mask_total, a.parts, b - a.end[kFinOffset]);
    return;
  }
  if (b < a.end[kFinWeight]) {
    // A row (group, output channel), kFinWeightCh of its padded channels: the partial sums are read along the
    // channels of a tap, summed in a fixed order and written along the taps of a channel.
    __shared__ float tile[kBwdTapsMax * kFinWeightCh];
    const int cblocks = (a.im.cgp + kFinWeightCh - 1) / kFinWeightCh;
    const int bi = b - a.end[kFinMask];
    const int row = bi / cblocks, c0 = (bi - row * cblocks) * kFinWeightCh;
    const int nc = min(kFinWeightCh, a.im.cgp - c0);
    const long M = (long)g.taps * a.im.cgp;
    const long split_stride = (long)g.Cout * M;
    for (int i = tid; i < g.taps * kFinWeightCh; i += 256) {
      const int tap = i / kFinWeightCh, c = i - tap * kFinWeightCh;
      float s = 0.0f;
      if (c < nc) {
        const float *src = a.wpart + (long)row * M + (long)tap * a.im.cgp + c0 + c;
        int sp = 0;
        for (; sp + 4 <= a.splits; sp += 4) {
          float v[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) v[u] = src[(long)(sp + u) * split_stride];
#pragma unroll
          for (int u = 0; u < 4; ++u) s += v[u];
        }
        for (; sp < a.splits; ++sp) s += src[(long)sp * split_stride];
      }
      tile[i] = s;
    }
    __syncthreads();
    E *dst = (E *)a.gw + (long)row * g.cin_g * g.taps;
    for (int i = tid; i < g.taps * nc; i += 256) {
      const int c = i / g.taps, tap = i - c * g.taps;
      int room;
      const int cs = chan_source(a.im, c0 + c, room);  // (of the first group: channel within a group)
      if (room > 0) dst[(long)cs * g.taps + tap] = from_f32<E>(tile[tap * kFinWeightCh + c]);
    }
    return;
  }
  const int co = (b - a.end[kFinWeight]) * 256 + tid;
  if (co < g.Cout) {
    float s = 0.0f;
    for (int i = 0; i < a.bsplits; ++i) s += a.bpart[(long)co * a.bsplits + i];
    ((E *)a.gb)[co] = from_f32<E>(s);
  }
}

}  // namespace mdcn
