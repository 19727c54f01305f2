// Backward of conv_offset (mdcn_oconv_backward.h).
#include "mdcn_oconv_backward.h"

#include <algorithm>
#include <type_traits>

#include "../../include/mdcn.h"
#include "mdcn_fused.h"
#include "mdcn_host.h"
#include "mdcn_prepass.h"

namespace mdcn {

namespace {

// The gradient of conv_offset's output: that of the offsets as it is, that of the mask through the sigmoid,
// rounded to the element type as the tensor of that gradient would be.  It is written twice, pixel major
// (32 channels of a pixel in a row: the operand of the data kernel) and channel major with rows of whole 32
// pixels (16 bytes of pixels of a channel: the operand of the weight kernel); channels past CO and pixels past
// the row are zero.  A block transposes 64 pixels of a row in LDS.  The other blocks order the weights for
// the data kernel: 16 bytes of output channels of (block of 32 input channels, block of 32 output
// channels, tap, 16-byte pair) per lane, lane l having input channel l % 32 and half l / 32 of the pair.
template <typename E>
__global__ __launch_bounds__(256) void oconv_bwd_prep_kernel(OconvBwdArgs a) {
  constexpr int EPV = 16 / (int)sizeof(E), KQ = 32 / (2 * EPV);
  __shared__ E tile[64 * 34];
  const Geom &g = a.g;
  const int tid = threadIdx.x;
  int b = (int)blockIdx.x;
  if (b < a.g_blocks) {
    const int seg = b % a.segs;
    b /= a.segs;
    const int ho = b % g.Ho, n = b / g.Ho;
    const int wo0 = seg * 64, px = tid & 63, wo = wo0 + px;
    const long plane = (long)g.Ho * g.Wo;
    const int n_off = 2 * g.DG * g.taps, n_msk = a.CO - n_off;
    const long at = (long)ho * g.Wo + min(wo, g.Wo - 1);
    for (int cb = 0; cb < a.cob; ++cb) {
      if (cb) __syncthreads();
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int c = i * 4 + (tid >> 6), co = cb * 32 + c;
        float v = 0.0f;
        if (co < n_off) {
          v = to_f32(((const E *)a.goff)[((long)n * n_off + co) * plane + at]);
        } else if (co < a.CO) {
          const long m = ((long)n * n_msk + co - n_off) * plane + at;
          const float y = to_f32(((const E *)a.mask)[m]);
          v = to_f32(((const E *)a.gmask)[m]) * (1.0f - y) * y;
        }
        tile[px * 34 + c] = from_f32<E>(wo < g.Wo ? v : 0.0f);
      }
      __syncthreads();
      if (a.gcm && wo < a.Wp)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int c = i * 4 + (tid >> 6);
          ((E *)a.gcm)[(((long)n * a.cob * 32 + cb * 32 + c) * g.Ho + ho) * a.Wp + wo] = tile[px * 34 + c];
        }
      if (a.gpm)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int c = tid & 31, p = i * 8 + (tid >> 5);
          if (wo0 + p < g.Wo)
            ((E *)a.gpm)[(((long)n * plane + (long)ho * g.Wo + wo0 + p) * a.cob + cb) * 32 + c] = tile[p * 34 + c];
        }
    }
    return;
  }
  const long total = (long)(g.Cin / 32) * a.cob * g.taps * KQ * 64;
  const long idx = (long)(b - a.g_blocks) * 256 + tid;
  if (idx >= total) return;
  const int lane = (int)(idx & 63);
  long r = idx >> 6;
  const int kq = (int)(r % KQ);
  r /= KQ;
  const int tap = (int)(r % g.taps);
  r /= g.taps;
  const int cb = (int)(r % a.cob), ci = (int)(r / a.cob) * 32 + (lane & 31);
  const int co0 = cb * 32 + (kq * 2 + (lane >> 5)) * EPV;
  E v[EPV];
#pragma unroll
  for (int e = 0; e < EPV; ++e)
    v[e] = co0 + e < a.CO ? ((const E *)a.ow)[((long)(co0 + e) * g.Cin + ci) * g.taps + tap] : from_f32<E>(0.0f);
  uint4 q;
  __builtin_memcpy(&q, v, 16);
  ((uint4 *)a.owf)[idx] = q;
}

__device__ __forceinline__ int floor_div(int v, int d) { return v >= 0 ? v / d : -((-v + d - 1) / d); }

// grad_input += conv_transpose(gradient, weight).  Workgroup = TH rows per wave x 32 columns of the input, and c_per blocks
// of 32 input channels one after the other.  The gradient pixels that the tile meets go to LDS pixel major (a block of 32 output
// channels at a time), each wave multiplies weights (rows: input channels) with them (columns: pixels) tap by tap, so that a
// tap is another LDS address, and a weight fragment serves TH products of each wave -- the waves read it at about the
// same time, three of them from L1.  With a stride only some taps meet a pixel: rows are skipped, lanes whose column a tap
// does not meet read a column of zeros.  The sum is added to grad_input, which the deformable convolution's backward has
// written, and rounded once.  What bounds it: 16-bit types the way to grad_input and back (its 249 MB would take 53 of the 111 us
// of the first call in the header), fp32 the matrix units, whose rounds of waves are not full.  A wave with four rows and channels of
// its own, every wave with its own weights from L2 then: 121 us, 13 and 30 us instead of 10 and 22 for N=2 and 8, 50x84.
// Two pixels a lane on the way to grad_input, traded between neighbours, took longer (137 us).
template <typename E, int TH, bool UNIT, int LDS_BYTES>
__global__ __launch_bounds__(256, 2) void oconv_dgrad_kernel(OconvBwdArgs a) {
  using TR = ElemTraits<E>;
  constexpr int EPV = 16 / (int)sizeof(E), KQ = 32 / (2 * EPV);
  constexpr int RB = 32 * (int)sizeof(E) + 16;  // bytes of a pixel's record: the 32 lanes of a read fall on all banks
  constexpr int AHEAD = 3;
  __shared__ uint4 lds[LDS_BYTES / 16];
  __shared__ int coltab[kOdMaxKw * 32];
  const Geom &g = a.g;
  const int tid = threadIdx.x, nthr = a.waves * 64;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int frow = lane & 31, fhalf = lane >> 5;
  // (neighbouring tiles share cache lines of grad_input and rows of their halo: an XCD has a run of them)
  long b = xcd_work_index(a.d_work);
  if (b < 0) return;
  const int tx = (int)(b % a.tiles_x);
  b /= a.tiles_x;
  const int yt = (int)(b % a.tiles_y) * TH * a.waves, x0 = tx * 32;
  b /= a.tiles_y;
  const int n = (int)(b / a.c_groups), c_first = (int)(b % a.c_groups) * a.c_per, c_end = min(c_first + a.c_per, g.Cin / 32);
  const int y0 = yt + wave * TH;  // this wave's rows
  const int ho0 = floor_div(yt + g.ph - (g.kh - 1) * g.dh, g.sh);
  const int wo0 = floor_div(x0 + g.pw - (g.kw - 1) * g.dw, g.sw);
  const int pitch = (a.gw_cols + 1) * RB;  // a column of zeros behind the last one
  unsigned char *L = (unsigned char *)lds;

  for (int i = tid; i < g.kw * 32; i += nthr) {
    const int v = x0 + (i & 31) + g.pw - (i >> 5) * g.dw, w = floor_div(v, g.sw);
    coltab[i] = (w * g.sw == v ? w - wo0 : a.gw_cols) * RB;
  }

  const int t_end = c_end * a.cob * g.taps;
  uint4 wf[AHEAD][KQ];
  auto load_weights = [&](int t, uint4 (&w)[KQ]) {
    const uint4 *src = (const uint4 *)a.owf + (long)min(t, t_end - 1) * (KQ * 64) + lane;  // (past the end: never used)
#pragma unroll
    for (int q = 0; q < KQ; ++q) w[q] = src[q * 64];
  };
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) load_weights(c_first * a.cob * g.taps + i, wf[i]);

  for (int cblk = c_first; cblk < c_end; ++cblk) {
    // (fp32: two sums of half the products each, whose roundings add up to less than those of one)
    constexpr int NS = sizeof(E) == 4 ? 2 : 1;
    f32x16 acc[TH][NS];
#pragma unroll
    for (int th = 0; th < TH; ++th)
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[th][s][r] = 0.0f;

    // What the sums are added to, on its way while they are formed.  Register r of lane l: input channel (r / 4) * 8 + (l / 32) * 4 +
    // r % 4, column l % 32
    const int x = x0 + frow;
    const long plane_in = (long)g.H * g.W;
    E *out = (E *)a.gin + ((long)n * g.Cin + cblk * 32 + fhalf * 4) * plane_in + (long)y0 * g.W + x;
    auto at = [&](int th, int r) { return out + ((r >> 2) * 8 + (r & 3)) * plane_in + (long)th * g.W; };
    E old[TH][16];
    if (x < g.W) {
#pragma unroll
      for (int th = 0; th < TH; ++th) {
        if (y0 + th >= g.H) break;
#pragma unroll
        for (int r = 0; r < 16; ++r) old[th][r] = *at(th, r);
      }
    }

    constexpr int CPP = 2 * KQ;  // 16-byte chunks of a record
    for (int cb = 0; cb < a.cob; ++cb) {
      if (a.cob > 1 || cblk == c_first) {
        __syncthreads();
        const int cols = a.gw_cols + 1, items = a.gh * cols * CPP;
        for (int i = tid; i < items; i += nthr) {
          const int q = i % CPP, px = i / CPP, r = px / cols, c = px - r * cols;
          const int ho = ho0 + r, wo = wo0 + c;
          uint4 v = make_uint4(0u, 0u, 0u, 0u);
          if (c < a.gw_cols && ho >= 0 && ho < g.Ho && wo >= 0 && wo < g.Wo)
            v = ((const uint4 *)a.gpm)[((((long)n * g.Ho + ho) * g.Wo + wo) * a.cob + cb) * CPP + q];
          *(uint4 *)(L + (long)px * RB + q * 16) = v;
        }
        __syncthreads();
      }
      const int t_base = (cblk * a.cob + cb) * g.taps;
      // Operands are read a step ahead -- a step is 16 bytes of a tap -- and kept there: the compiler would put each read in front
      // of its product, which then waits for it
      auto rows_of = [&](int ti, int (&row)[TH]) {
#pragma unroll
        for (int th = 0; th < TH; ++th) {
          const int v = y0 + th + g.ph - ti * g.dh;
          if constexpr (UNIT) {
            row[th] = v - ho0;
          } else {
            const int h = floor_div(v, g.sh);
            row[th] = h * g.sh == v ? h - ho0 : -1;
          }
        }
      };
      auto read = [&](const int (&row)[TH], int col, int q, uint4 (&gf)[TH]) {
#pragma unroll
        for (int th = 0; th < TH; ++th) gf[th] = *(const uint4 *)(L + (UNIT ? row[th] : max(row[th], 0)) * pitch + col + fhalf * 16 + q * 32);
      };
      int ti = 0, tj = 0, row[TH], row_next[TH];
      int col = coltab[frow];
      uint4 gf[2][TH];
      rows_of(0, row);
      read(row, col, 0, gf[0]);
      for (int g0 = 0; g0 < g.taps; g0 += AHEAD) {
        const int next = t_base + min(g0 + AHEAD, g.taps);
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
          if (g0 + i < g.taps) {
            if (g0 + i + 1 < g.taps && ++tj == g.kw) tj = 0, ++ti;
            const int col_next = coltab[tj * 32 + frow];
            rows_of(ti, row_next);
#pragma unroll
            for (int q = 0; q < KQ; ++q) {
              if (q + 1 < KQ)
                read(row, col, q + 1, gf[(q + 1) & 1]);
              else
                read(row_next, col_next, 0, gf[0]);
              __builtin_amdgcn_sched_barrier(0);
#pragma unroll
              for (int th = 0; th < TH; ++th)
                if (UNIT || row[th] >= 0) TR::mma(acc[th][q % NS], wf[i][q], gf[q & 1][th]);
              __builtin_amdgcn_sched_barrier(0);
            }
            col = col_next;
#pragma unroll
            for (int th = 0; th < TH; ++th) row[th] = row_next[th];
          }
          load_weights(next + i, wf[i]);
        }
      }
    }

    if (x < g.W) {
#pragma unroll
      for (int th = 0; th < TH; ++th) {
        if (y0 + th >= g.H) break;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          *at(th, r) = from_f32<E>(to_f32(old[th][r]) + (NS == 2 ? acc[th][0][r] + acc[th][NS - 1][r] : acc[th][0][r]));
      }
    }
  }
}

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t *lds_s16x4_t;

// Sums over pixels of gradient x input, tap by tap, and of the gradient alone.  Workgroup = 32 output channels (rows)
// x 32 input channels (columns) x three taps per wave, over a share of the tiles of TH x 32 output pixels.  A tile's
// input pixels with their halo and its gradients are copied to LDS directly, the tile's after next while this one's
// products run; the input comes from the zero-bordered copy that the deformable convolution's backward reads, pixel
// major in records of 32 bytes (a pixel outside the image is a border pixel), and serves all taps: a tap
// is another address.  The operand wants 16 bytes of pixels of a channel, beginning at any pixel: 16-bit types read
// them with LDS reads that transpose.  The gradients' copy is channel major, 16 bytes a lane (their chunks swizzled
// against the rows).  A wave has taps of its own and all pixels, so that its sums are its own too; those of the shares meet in the
// finishing launch.  Columns past the end of a row read its last pixel's input: their gradients are zero.
// What bounds it: the copies' latency between two barriers, LDS reads (16-bit types: four of 16 bytes for three products); fp32 the
// matrix units.  Input staged from NCHW by way of registers, transposed with VALU work, took 200 us where this takes 93; reads
// left in front of their products 36 instead of 31 (fp32, N=2, 256 channels, 50x84); six waves, two to three taps, 41.
template <typename E, int LDS_BYTES>
__global__ __launch_bounds__(64 * kOwWaves) void oconv_wgrad_kernel(OconvBwdArgs a, int TH) {
  using TR = ElemTraits<E>;
  constexpr int EPV = 16 / (int)sizeof(E), NG = 16 / (2 * EPV);  // NG: pairs of 16 bytes in a run of 16 pixels
  constexpr int NT = kOwTaps / kOwWaves;
  constexpr int NPL = (int)sizeof(E), CHK = 32 / EPV;  // planes of 32 input channels; chunks of 32 pixels of a gradient
  __shared__ uint4 lds[LDS_BYTES / 16];
  const Geom &g = a.g;
  const int tid = threadIdx.x, waves = blockDim.x >> 6;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int frow = lane & 31, fhalf = lane >> 5;
  // (an XCD has a run of the shares with all their channels: neighbouring tiles share rows of the input, the blocks of
  // channels of a share its gradients)
  const int cblocks = g.Cin / 32;
  const long work = xcd_work_index((long)a.splits * a.tgroups * a.cob * cblocks);
  if (work < 0) return;
  int b = (int)work;
  const int ci0 = b % cblocks * 32;
  b /= cblocks;
  const int cb = b % a.cob;
  b /= a.cob;
  const int t0 = b % a.tgroups * kOwTaps + wave * NT, split = b / a.tgroups;
  const bool sums = ci0 == 0 && t0 == 0;
  const int PC = a.plane_chunks;                     // 16-byte chunks of a plane in LDS
  const int xcopies = (NPL * PC + 63) / 64, copies = xcopies + TH * CHK / 2;
  const int buf_chunks = copies * 64;

  f32x16 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.0f;
  double bsum = 0.0;

  int tapoff[NT];  // (past the last tap: that again, for sums nobody reads)
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int tap = min(t0 + t, g.taps - 1), ti = tap / g.kw, tj = tap - ti * g.kw;
    tapoff[t] = (ti * g.dh * a.lw + tj * g.dw) * 32;
  }
  const int row_bytes = g.sh * a.lw * 32;
  auto tile_at = [&](int tile, int &n, int &ho0, int &wo0) {
    wo0 = tile % a.tiles_x * 32;
    tile /= a.tiles_x;
    ho0 = tile % a.tiles_y * TH;
    n = tile / a.tiles_y;
  };
  // 1 KiB per wave and copy: lane l of copy k fills chunk 64 k + l of the buffer
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lptr_t)(&lds[0]);
  auto issue = [&](int tile, int buf) {
    int n, ho0, wo0;
    tile_at(tile, n, ho0, wo0);
    const int yb = ho0 * g.sh - g.ph + 1, xb = wo0 * g.sw - g.pw + 1;  // in the bordered copy
    const unsigned char *x = (const unsigned char *)a.xt + ((long)n * cblocks + ci0 / 32) * NPL * g.Hp * g.Wp * 32;
    const E *gr = (const E *)a.gcm + ((long)n * a.cob + cb) * 32 * g.Ho * a.Wp + wo0;
    for (int k = wave; k < copies; k += waves) {
      const uint32_t dst = lds0 + (uint32_t)(buf * buf_chunks + k * 64) * 16u;
      const void *src;
      if (k < xcopies) {
        const int i = k * 64 + lane;
        const int j = min((int)(i >= PC) + (int)(i >= 2 * PC) + (int)(i >= 3 * PC), NPL - 1), q = i - j * PC;
        const int r = (int)(((uint32_t)(q >> 1) * a.lw_inv) >> 20), c = (q >> 1) - r * a.lw;  // (padding of a plane: rows past the halo)
        const int y = min(max(yb + r, 0), g.Hp - 1), xx = min(max(xb + c, 0), g.Wp - 1);
        src = x + (((long)j * g.Hp + y) * g.Wp + xx) * 32 + (q & 1) * 16;
      } else {
        const int i = (k - xcopies) * 64 + lane, co = i / CHK % 32, row = i / (32 * CHK);
        const int c = i % CHK ^ (sizeof(E) == 2 ? (co >> 2) & 3 : co & 7);
        src = gr + ((long)co * g.Ho + min(ho0 + row, g.Ho - 1)) * a.Wp + c * EPV;
      }
      copy16_global_to_lds(src, dst);
    }
  };

  issue(split, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  int buf = 0;
  for (int tile = split; tile < a.tiles; tile += a.splits, buf ^= 1) {
    if (tile + a.splits < a.tiles) issue(tile + a.splits, buf ^ 1);
    int n, ho0, wo0;
    tile_at(tile, n, ho0, wo0);
    const int rows = min(TH, g.Ho - ho0);
    const unsigned char *X = (const unsigned char *)lds + (long)buf * buf_chunks * 16;
    const unsigned char *G = X + xcopies * 1024 + frow * (CHK * 16);
    // where this lane's pixels of a run are, output row 0, tap (0, 0)
    constexpr int NA = sizeof(E) == 2 ? 2 : 8;
    const int last = g.Wo - 1 - wo0;
    int colad[2][NA];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int k = 0; k < NA; ++k) {
        if constexpr (sizeof(E) == 2)  // lane's share of a transposing read: 8 bytes of four of the pixels
          colad[ks][k] = min(ks * 16 + fhalf * 8 + k * 4 + ((lane & 15) >> 2), last) * g.sw * 32 + ((lane >> 4) & 1) * PC * 16 + (lane & 3) * 8;
        else
          colad[ks][k] = min(ks * 16 + (k >> 2) * 8 + fhalf * 4 + (k & 3), last) * g.sw * 32 + (frow >> 3) * PC * 16 + (frow & 7) * 4;
      }
    // Operands are read a step ahead -- a step is a pair of 16 bytes of pixels -- and kept there: the compiler would put each read in
    // front of its product, which then waits for it
    auto read = [&](int row, int step, uint4 &gv, uint4 (&xv)[NT]) {
      const int ks = step / NG, s = step % NG, c = (ks * 16) / EPV + 2 * s + fhalf;
      gv = *(const uint4 *)(G + row * (32 * CHK * 16) + (c ^ (sizeof(E) == 2 ? (frow >> 2) & 3 : frow & 7)) * 16);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const unsigned char *p = X + (row * row_bytes + tapoff[t]);
        if constexpr (sizeof(E) == 2) {
          const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)(lptr_t)(void *)(p + colad[ks][0]));
          const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)(lptr_t)(void *)(p + colad[ks][1]));
          const uint2 l2 = __builtin_bit_cast(uint2, lo), h2 = __builtin_bit_cast(uint2, hi);
          xv[t] = make_uint4(l2.x, l2.y, h2.x, h2.y);
        } else {
          xv[t] = make_uint4(*(const uint32_t *)(p + colad[ks][(4 * s) % NA]), *(const uint32_t *)(p + colad[ks][(4 * s + 1) % NA]),
                             *(const uint32_t *)(p + colad[ks][(4 * s + 2) % NA]), *(const uint32_t *)(p + colad[ks][(4 * s + 3) % NA]));
        }
      }
    };
    float tsum = 0.0f;
    uint4 gv[2], xv[2][NT];
    read(0, 0, gv[0], xv[0]);
    for (int row = 0; row < rows; ++row) {
      // (nor sums of these and the row's and the tap's offsets for each of them, carried over the rows)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int k = 0; k < NA; ++k) asm volatile("" : "+v"(colad[ks][k]));
#pragma unroll
      for (int step = 0; step < 2 * NG; ++step) {
        const int cur = step & 1;
        if (step + 1 < 2 * NG)
          read(row, step + 1, gv[cur ^ 1], xv[cur ^ 1]);
        else
          read(min(row + 1, rows - 1), 0, gv[cur ^ 1], xv[cur ^ 1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < NT; ++t) TR::mma(acc[t], gv[cur], xv[cur][t]);
        if (sums) {
          E e[EPV];
          __builtin_memcpy(e, &gv[cur], 16);
          float v = 0.0f;
#pragma unroll
          for (int k = 0; k < EPV; k += 4) v += (to_f32(e[k]) + to_f32(e[k + 1])) + (to_f32(e[k + 2]) + to_f32(e[k + 3]));
          tsum += v;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    bsum += tsum;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }

  // register r of lane l: output channel (r / 4) * 8 + (l / 32) * 4 + r % 4, input channel l % 32
#pragma unroll
  for (int t = 0; t < NT; ++t)
    if (t0 + t < g.taps) {
      float *dst = a.part + (((long)split * g.taps + t0 + t) * (a.cob * 32) + cb * 32 + fhalf * 4) * g.Cin + ci0 + frow;
#pragma unroll
      for (int r = 0; r < 16; ++r) dst[(long)((r >> 2) * 8 + (r & 3)) * g.Cin] = acc[t][r];
    }
  if (sums) {
    bsum += __shfl_xor(bsum, 32);
    if (lane < 32) a.bpart[(long)split * (a.cob * 32) + cb * 32 + lane] = (float)bsum;
  }
}

// The shares' sums added in a fixed order: 64 elements a block, a quarter of the shares per wave.
template <typename E>
__global__ __launch_bounds__(256) void oconv_bwd_finish_kernel(OconvBwdArgs a) {
  __shared__ double quarter[256];
  const Geom &g = a.g;
  const int tid = threadIdx.x;
  const long n_w = a.gw ? (long)g.taps * a.CO * g.Cin : 0;
  const long idx = (long)blockIdx.x * 64 + (tid & 63), ib = idx - n_w;
  const float *src = nullptr;
  long step = 0;
  E *dst = nullptr;
  if (idx < n_w) {
    const int ci = (int)(idx % g.Cin);
    const long r = idx / g.Cin;
    const int co = (int)(r % a.CO), t = (int)(r / a.CO);
    src = a.part + ((long)t * (a.cob * 32) + co) * g.Cin + ci;
    step = (long)g.taps * (a.cob * 32) * g.Cin;
    dst = (E *)a.gw + ((long)co * g.Cin + ci) * g.taps + t;
  } else if (a.gb && ib < a.CO) {
    src = a.bpart + ib;
    step = a.cob * 32;
    dst = (E *)a.gb + ib;
  }
  double s = 0.0;
  if (dst) {
    const int per = (a.splits + 3) / 4, end = min(a.splits, ((tid >> 6) + 1) * per);
    int i = (tid >> 6) * per;
    for (; i + 8 <= end; i += 8) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = src[(long)(i + u) * step];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += v[u];
    }
    for (; i < end; ++i) s += src[(long)i * step];
  }
  quarter[tid] = s;
  __syncthreads();
  if (tid < 64 && dst)
    *dst = from_f32<E>((float)((quarter[tid] + quarter[64 + tid]) + (quarter[128 + tid] + quarter[192 + tid])));
}

template <typename E>
hipError_t run(const OconvBwdPlan &pl, OconvBwdArgs a, hipStream_t st) {
  constexpr int EPV = 16 / (int)sizeof(E), KQ = 32 / (2 * EPV);
  const Geom &g = a.g;
  a.segs = (std::max(g.Wo, pl.weight ? a.Wp : 0) + 63) / 64;
  a.g_blocks = g.N * g.Ho * a.segs;
  const long frags = pl.data ? (long)(g.Cin / 32) * a.cob * g.taps * KQ * 64 : 0;
  hipLaunchKernelGGL(oconv_bwd_prep_kernel<E>, dim3((unsigned)(a.g_blocks + (frags + 255) / 256)), dim3(256), 0, st, a);
  if (pl.data) {
    OconvBwdArgs d = a;
    d.waves = pl.d_waves;
    d.gh = pl.gh;
    d.gw_cols = pl.gw;
    d.c_per = pl.d_cper;
    d.c_groups = (g.Cin / 32 + d.c_per - 1) / d.c_per;
    const int rows = pl.d_th * d.waves;
    d.tiles_y = (g.H + rows - 1) / rows;
    d.tiles_x = (g.W + 31) / 32;
    d.d_work = (long)g.N * d.tiles_y * d.tiles_x * d.c_groups;
    const dim3 grid((unsigned)((d.d_work + 7) / 8 * 8)), block(d.waves * 64);
    auto launch = [&](auto th, auto unit, auto bytes) {
      constexpr int TH = decltype(th)::value, LDS = decltype(bytes)::value;
      hipLaunchKernelGGL((oconv_dgrad_kernel<E, TH, decltype(unit)::value, LDS>), grid, block, 0, st, d);
    };
    auto launch_th = [&](auto th) {
      using Small = std::integral_constant<int, kOdLdsSmall>;
      using Big = std::integral_constant<int, kOdLds>;
      if (g.sh == 1)
        pl.d_lds <= kOdLdsSmall ? launch(th, std::true_type(), Small()) : launch(th, std::true_type(), Big());
      else
        pl.d_lds <= kOdLdsSmall ? launch(th, std::false_type(), Small()) : launch(th, std::false_type(), Big());
    };
    if (pl.d_th == 2)
      launch_th(std::integral_constant<int, 2>());
    else
      launch_th(std::integral_constant<int, 1>());
  }
  if (pl.weight) {
    a.tiles_y = (g.Ho + pl.w_th - 1) / pl.w_th;
    a.tiles_x = (g.Wo + 31) / 32;
    a.tiles = g.N * a.tiles_y * a.tiles_x;
    a.lw = pl.lw;
    a.lw_inv = (1u << 20) / (uint32_t)pl.lw + 1u;
    a.plane_chunks = pl.plane_chunks;
    a.tgroups = pl.tgroups;
    a.splits = pl.splits;
    if (!a.xt) {  // (the backward of the deformable convolution took a path without that copy)
      a.xt = a.own_xt;
      const int n_pchunks = (g.H * g.W + 32 * EPV - 1) / (32 * EPV);
      hipLaunchKernelGGL((relayout_vec_kernel<E, true, 32>), dim3((unsigned)((long)g.N * (g.Cin / (8 * EPV)) * n_pchunks)), dim3(256), 0,
                         st, g, (const E *)a.x, (E *)a.own_xt, n_pchunks);
    }
    const dim3 grid((unsigned)(((long)pl.splits * pl.tgroups * a.cob * (g.Cin / 32) + 7) / 8 * 8));
    const dim3 block(64 * std::min(kOwWaves, (g.taps + kOwTaps / kOwWaves - 1) / (kOwTaps / kOwWaves)));
    if (pl.w_lds <= kOwLds3)
      hipLaunchKernelGGL((oconv_wgrad_kernel<E, kOwLds3>), grid, block, 0, st, a, pl.w_th);
    else if (pl.w_lds <= kOwLds2)
      hipLaunchKernelGGL((oconv_wgrad_kernel<E, kOwLds2>), grid, block, 0, st, a, pl.w_th);
    else
      hipLaunchKernelGGL((oconv_wgrad_kernel<E, kOwLds1>), grid, block, 0, st, a, pl.w_th);
    const long n = (a.gw ? (long)g.taps * a.CO * g.Cin : 0) + (a.gb ? a.CO : 0);
    hipLaunchKernelGGL(oconv_bwd_finish_kernel<E>, dim3((unsigned)((n + 63) / 64)), dim3(256), 0, st, a);
  }
  return hipGetLastError();
}

}  // namespace

bool oconv_bwd_plan(const Geom &g, int dtype, bool unmodulated, bool data, bool weight, bool own_copy, int cus,
                    OconvBwdPlan *pl) {
  const int es = (int)elem_size(dtype), EPV = 16 / es;
  if (dtype == MDCN_F64 || g.Cin % (8 * EPV) || g.kw > kOdMaxKw) return false;
  pl->CO = (unmodulated ? 2 : 3) * g.DG * g.taps;
  pl->cob = (pl->CO + 31) / 32;
  pl->Wp = (g.Wo + 31) / 32 * 32;
  pl->data = data;
  pl->weight = weight;
  const long limit = 1L << 30;  // blocks of a launch, pixels of a plane
  if ((long)g.H * g.W > limit || (long)g.N * g.Ho * ((pl->Wp + 63) / 64) > limit) return false;

  // data: four waves, fewer where their rows' halo does not fit; as many rows a wave (fp32: one) and blocks of channels a
  // workgroup as leave four and eight workgroups per CU
  const int rb = 32 * es + 16;
  auto halo = [](long n, long k, long d, long s) { return (n - 1 + (k - 1) * d) / s + (s > 1 ? 2 : 1); };
  const long gw = halo(32, g.kw, g.dw, g.sw);
  auto d_lds = [&](long rows) { return halo(rows, g.kh, g.dh, g.sh) * (gw + 1) * rb; };
  pl->d_waves = 4;
  while (pl->d_waves > 1 && d_lds(pl->d_waves) > kOdLds) --pl->d_waves;
  const int waves = pl->d_waves, cblocks = g.Cin / 32;
  auto d_tiles = [&](int th) { return (long)g.N * ((g.H + th * waves - 1) / (th * waves)) * ((g.W + 31) / 32); };
  pl->d_th = es == 2 ? 2 : g.sh == 1 ? 1 : 2;  // (of two rows at a stride one meets fewer taps)
  while (pl->d_th > 1 && (d_lds(pl->d_th * waves) > kOdLds || d_tiles(pl->d_th) * cblocks < 4L * cus)) pl->d_th /= 2;
  pl->d_cper = 1;
  while (pl->cob == 1 && pl->d_cper * 2 <= cblocks && d_tiles(pl->d_th) * (cblocks / (pl->d_cper * 2)) >= 8L * cus) pl->d_cper *= 2;
  if (d_lds(pl->d_th * waves) > kOdLds || d_tiles(pl->d_th) * cblocks > limit) return false;
  pl->d_lds = (int)d_lds(pl->d_th * waves);
  pl->gw = (int)gw;
  pl->gh = (int)halo(pl->d_th * waves, g.kh, g.dh, g.sh);

  // weight: the same for the rows of its tiles, whose LDS says how many workgroups share a CU
  const long lw = 31L * g.sw + (long)(g.kw - 1) * g.dw + 1;
  if (lw > 400) return false;  // (what its multiplication by 1 / lw is exact for)
  auto plane_chunks = [&](long th) {  // lanes that read several planes at a time find them on banks of their own
    long c = ((th - 1) * g.sh + (long)(g.kh - 1) * g.dh + 1) * lw * 2;
    while (c % 16 != (es == 2 ? 8 : 2)) ++c;
    return c;
  };
  auto w_lds = [&](int th) { return 2 * ((es * plane_chunks(th) + 63) / 64 * 64 + (long)th * 32 * (32 / EPV)) * 16; };
  pl->tgroups = (g.taps + kOwTaps - 1) / kOwTaps;
  const long per = (long)(g.Cin / 32) * pl->cob * pl->tgroups;
  auto w_tiles = [&](int th) { return (long)g.N * ((g.Ho + th - 1) / th) * (pl->Wp / 32); };
  auto w_slots = [&](int th) { return (w_lds(th) <= kOwLds3 ? 3L : w_lds(th) <= kOwLds2 ? 2L : 1L) * cus; };
  // (a third of the time is the copies of tile and halo; products of one workgroup alone in a CU leave a matrix unit idle)
  auto w_cost = [&](int th) {
    const long rounds = (w_tiles(th) * per + w_slots(th) - 1) / w_slots(th);
    return (double)rounds * std::max(w_slots(th), 2L * cus) * (th + 1.0);
  };
  pl->w_th = 0;
  for (int th : {8, 7, 6, 5, 4, 3, 2, 1})
    if (w_lds(th) <= kOwLds1 && (pl->w_th == 0 || w_cost(th) < w_cost(pl->w_th))) pl->w_th = th;
  if (pl->w_th == 0) return false;
  pl->w_lds = (int)w_lds(pl->w_th);
  pl->lw = (int)lw;
  pl->plane_chunks = (int)plane_chunks(pl->w_th);
  const long tiles = w_tiles(pl->w_th);
  if (tiles > limit) return false;
  pl->splits = (int)std::max<long>(1, std::min<long>(tiles, w_slots(pl->w_th) / per));

  const size_t co_p = (size_t)pl->cob * 32;
  pl->gpm_bytes = data ? align_up((size_t)g.N * g.Ho * g.Wo * co_p * es) : 0;
  pl->gcm_bytes = weight ? align_up((size_t)g.N * co_p * g.Ho * pl->Wp * es) : 0;
  pl->owf_bytes = data ? align_up((size_t)g.Cin * g.taps * co_p * es) : 0;
  pl->part_bytes = weight ? align_up((size_t)pl->splits * g.taps * co_p * g.Cin * 4) : 0;
  pl->bpart_bytes = weight ? align_up((size_t)pl->splits * co_p * 4) : 0;
  pl->xt_bytes = weight && own_copy ? align_up((size_t)g.N * g.Cin * g.Hp * g.Wp * es) : 0;
  return true;
}

// Training calls in us, torch's convolution backward and the operations around it / this one.  What it saves is launches and passes
// over memory, some 50 us of device time and more on the host; what it costs is that both kernels go over padded blocks of 32
// channels of conv_offset, and tap by tap, one after another.
// fp32, whose products are six of bf16 each, at a stride and dilation of 1 (elsewhere torch's own take long) and beyond one block,
// by the work of tiles of 4 x 32 pixels.  Calls with mask: N=4 256 channels 50x84, 2 deformable groups (92 M) 951 / 953, 4 groups (184 M)
// 1 101 / 1 131; N=8 256 25x42, 4 (132 M) 751 / 800; N=8 128 25x42, 4 (66 M) 408 / 406.  Of a long chain of taps and blocks, or without mask:
// N=1 64 30x40, 8 groups (8.2 M) 255 / 241, N=1 256 13x21, 8 (8.3 M) 276 / 314, N=2 64 30x40, 8 (16 M) 238 / 255; 5x5 taps 374 / 416 (9.8 M), 7x7 586 / 741;
// without mask N=1 128 25x42, 4 (6.1 M) 240 / 209, N=2 256 13x21, 4 (7.1 M) 257 / 269, N=8 256 25x42, 2 (66 M) 612 / 640.
// (One block: without mask, N=8 256 25x42, 586 / 595 at worst, with it 611 / 603; N=2 256 50x84 566 / 559 and 595 / 565.)
// 16 bits: only chains as long as those of 7x7 taps where workgroups are few, N=1 64 30x40 (32) 627 / 650 and 606 / 624 without mask; N=4
// (128) 1 902 / 1 800.
bool oconv_bwd_pays(const Geom &g, int dtype, bool unmodulated) {
  const int cob = ((unmodulated ? 2 : 3) * g.DG * g.taps + 31) / 32, chain = cob * g.taps;
  if (dtype != MDCN_F32)
    return chain <= 150 || (long)g.N * ((g.H + 3) / 4) * ((g.W + 31) / 32) * (g.Cin / 32) >= 100;
  if (cob == 1 || g.sh != 1 || g.sw != 1 || g.dh != 1 || g.dw != 1) return true;
  const double work = (double)g.N * ((g.Ho + 3) / 4 * 4) * ((g.Wo + 31) / 32 * 32) * g.Cin * chain;
  return work <= (!unmodulated && chain <= 40 ? 100e6 : 6.2e6);
}

hipError_t oconv_backward(int dtype, const OconvBwdPlan &pl, OconvBwdArgs a, unsigned char *ws, hipStream_t st) {
  auto take = [&](size_t bytes) {
    unsigned char *q = ws;
    ws += bytes;
    return bytes ? q : nullptr;
  };
  a.CO = pl.CO;
  a.cob = pl.cob;
  a.Wp = pl.Wp;
  a.gpm = take(pl.gpm_bytes);
  a.gcm = take(pl.gcm_bytes);
  a.owf = take(pl.owf_bytes);
  a.part = (float *)take(pl.part_bytes);
  a.bpart = (float *)take(pl.bpart_bytes);
  a.own_xt = take(pl.xt_bytes);
  switch (dtype) {
    case MDCN_F32: return run<float>(pl, a, st);
    case MDCN_F16: return run<f16_t>(pl, a, st);
    default: return run<bf16_t>(pl, a, st);
  }
}

}  // namespace mdcn
