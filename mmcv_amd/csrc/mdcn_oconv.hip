// conv_offset on the zero-bordered input copy (mdcn_oconv.h says what for).
#include "mdcn_oconv.h"

#include <algorithm>

#include "../../include/mdcn.h"
#include "mdcn_host.h"

namespace mdcn {

namespace {

// LDS of the tiled kernel's forms, and the workgroups of each that share a CU.
constexpr int kOconvLds3 = 52 * 1024, kOconvLds2 = 80 * 1024, kOconvLds1 = 156 * 1024;
constexpr int oconv_workgroups(int lds) { return lds <= kOconvLds3 ? 3 : (lds <= kOconvLds2 ? 2 : 1); }

// Implicit GEMM raw[pixel][co] = sum_{c, tap} x[pixel + tap][c] * ow[co][c][tap] + ob[co],
// variant without LDS for geometries whose input patch does not fit the tiled
// kernel below (large dilated kernels with stride): the A operand of the MFMA
// (32 pixels x 16 bytes of channels) is loaded from the input copy as it lies,
// the B operand from the packed weights; each wave owns PXF blocks of 32
// consecutive pixels and all COF blocks of 32 output channels.  A tap outside the
// one-pixel zero border (padding > 1) contributes a zero fragment.  Every lane of
// an A load reads another cache line, which makes this the slow variant.
template <typename E, int COF, int PXF>
__global__ __launch_bounds__(256) void oconv_gather_kernel(OconvArgs a) {
  using TR = ElemTraits<E>;
  const Geom &g = a.g;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int frow = lane & 31;
  const int fhalf = lane >> 5;
  const int plane_out = g.Ho * g.Wo;
  const long p_wave = ((long)blockIdx.x * 4 + wave) * (32 * PXF);
  if (p_wave >= a.total_px) return;

  // this lane's pixel of each block: image base and top-left tap position in the copy
  long img_base[PXF];
  int by[PXF], bx[PXF];
#pragma unroll
  for (int pf = 0; pf < PXF; ++pf) {
    long p = p_wave + pf * 32 + frow;
    if (p >= a.total_px) p = a.total_px - 1;  // loads stay in range, nothing is stored
    const int n = (int)(p / plane_out);
    const int rem = (int)(p - (long)n * plane_out);
    const int ho = rem / g.Wo, wo = rem - ho * g.Wo;
    img_base[pf] = (long)n * a.slabs_total * a.plane_px;
    by[pf] = ho * g.sh - g.ph + 1;  // +1: coordinates of the bordered copy
    bx[pf] = wo * g.sw - g.pw + 1;
  }

  f32x16 acc[PXF][COF];
#pragma unroll
  for (int pf = 0; pf < PXF; ++pf)
#pragma unroll
    for (int cf = 0; cf < COF; ++cf)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[pf][cf][r] = 0.0f;

  const uint4 *xt = (const uint4 *)a.xt;
  const uint4 *owp = (const uint4 *)a.owp + lane;
  for (int slab = 0; slab < a.slabs_total; ++slab) {
    for (int ti = 0; ti < g.kh; ++ti) {
      for (int tj = 0; tj < g.kw; ++tj) {
        const int tap = ti * g.kw + tj;
        long pix[PXF];
        bool ok[PXF];
#pragma unroll
        for (int pf = 0; pf < PXF; ++pf) {
          const int y = by[pf] + ti * g.dh, x = bx[pf] + tj * g.dw;
          ok[pf] = (y >= 0) && (y < g.Hp) && (x >= 0) && (x < g.Wp);
          pix[pf] = ok[pf] ? img_base[pf] + (long)slab * a.plane_px + (long)y * g.Wp + x : 0;
        }
        const uint4 *wfrag = owp + (long)((slab * g.taps + tap) * 4) * COF * 64;
#pragma unroll
        for (int ksub = 0; ksub < 4; ++ksub) {
          uint4 af[PXF], bf[COF];
#pragma unroll
          for (int pf = 0; pf < PXF; ++pf) {
            af[pf] = xt[pix[pf] * 8 + ksub * 2 + fhalf];
            if (!ok[pf]) af[pf] = make_uint4(0u, 0u, 0u, 0u);
          }
#pragma unroll
          for (int cf = 0; cf < COF; ++cf) bf[cf] = wfrag[(ksub * COF + cf) * 64];
#pragma unroll
          for (int pf = 0; pf < PXF; ++pf)
#pragma unroll
            for (int cf = 0; cf < COF; ++cf) TR::mma(acc[pf][cf], af[pf], bf[cf]);
        }
      }
    }
  }

  // Accumulator block (A = pixels, B = channels): register r of lane l holds
  //   pixel = (r/4)*8 + (l/32)*4 + r%4,  channel = l%32.
  // Lanes 0..31 of one store cover the 32 consecutive channels of one pixel.
  E *raw = (E *)a.raw;
#pragma unroll
  for (int cf = 0; cf < COF; ++cf) {
    const int co = cf * 32 + frow;
    float b = 0.0f;
    if (a.obias && co < a.CO) b = to_f32(((const E *)a.obias)[co]);
#pragma unroll
    for (int pf = 0; pf < PXF; ++pf) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const long p = p_wave + pf * 32 + (r >> 2) * 8 + fhalf * 4 + (r & 3);
        if (p < a.total_px) raw[p * a.CO_pad + co] = from_f32<E>(acc[pf][cf][r] + b);
      }
    }
  }
}

// Tiled variant, the usual one.  A workgroup of 4 waves computes TH output rows x
// 32 output columns of one image from the input patch those outputs need (PH x PW
// pixels, 128 bytes per channel slab, contiguous runs of PW pixels in the copy).
// The waves share the pixels and split K: wave k takes the 16-byte channel chunks
// 2 k and 2 k + 1 of every slab, so that a weight fragment has one reader, which
// loads it from L2 into registers kOconvAhead fragments ahead, and LDS holds
// nothing but the patch.  At the end the waves' accumulators are added up through
// LDS in the order of the waves.  `stage` slabs of the patch are copied at a time; lane
// (pixel column r, half h) reads chunk 2 k + h of patch pixel
// (row * sh + i * dh, r * sw + j * dw).  Chunk c of patch pixel q sits at c ^ (q & 7),
// which spreads the 32 rows of a fragment read over all banks when sw is odd.
//
// What bounds it: large calls the copies (the input once and its halo), which other workgroups of the CU
// overlap with their MFMAs -- two or three of them fit as the weights are not in LDS; small ones the chain
// copy, MFMAs, sum of one workgroup, hence fewer rows each and all slabs in one stage where they fit.
template <typename E, int COF, int TH, int LDS_BYTES>
__global__ __launch_bounds__(256, oconv_workgroups(LDS_BYTES)) void oconv_tiled_kernel(OconvArgs a) {
  using TR = ElemTraits<E>;
  __shared__ uint4 patch[LDS_BYTES / 16];
  const Geom &g = a.g;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int frow = lane & 31;
  const int fhalf = lane >> 5;

  long L = xcd_work_index(a.tiles);
  if (L < 0) return;
  const int tx = (int)(L % a.tiles_x);
  L /= a.tiles_x;
  const int ty = (int)(L % a.tiles_y);
  const int n = (int)(L / a.tiles_y);
  const int ho0 = ty * TH, wo0 = tx * 32;
  const int py0 = ho0 * g.sh - g.ph + 1;  // patch origin in the bordered copy (may lie outside)
  const int px0 = wo0 * g.sw - g.pw + 1;
  const int patch_chunks = a.PH * a.PW * 8;

  f32x16 acc[TH][COF];
#pragma unroll
  for (int th = 0; th < TH; ++th)
#pragma unroll
    for (int cf = 0; cf < COF; ++cf)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[th][cf][r] = 0.0f;

  // A slab's patch arrives by direct-to-LDS copies, 1 KiB per wave and instruction: lane l of copy j fills
  // chunk i = 256 * j + 64 * wave + l and reads the source chunk that belongs there (the swizzle is applied on
  // the source side).  soff: offset into the slab's plane of the copy, the same for every slab.  What lies outside the
  // copy, or past the patch, reads the copy's corner pixel (0, 0), a stored zero.
  constexpr int NB = LDS_BYTES / 4096;
  const int n_copies = (patch_chunks + 255) / 256;   // at most NB
  int soff[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int idx = tid + 256 * j;
    const int q = idx >> 3;
    const int c = (idx & 7) ^ (q & 7);
    const int r = q / a.PW;
    const int y = py0 + r, x = px0 + (q - r * a.PW);
    const bool in_copy = idx < patch_chunks && y >= 0 && y < g.Hp && x >= 0 && x < g.Wp;
    soff[j] = in_copy ? (y * g.Wp + x) * 8 + c : c;
  }
  const uint32_t lds_wave = (uint32_t)(uintptr_t)(lptr_t)(&patch[0]) + (uint32_t)wave * 1024u;
  auto fetch = [&](int slab, int slot) {
    const uint4 *src = (const uint4 *)a.xt + ((long)n * a.slabs_total + slab) * a.plane_px * 8;
    const uint32_t dst = lds_wave + (uint32_t)(slot * n_copies) * 4096u;
#pragma unroll
    for (int j = 0; j < NB; ++j)
      if (j < n_copies) copy16_global_to_lds(src + soff[j], dst + (uint32_t)j * 4096u);
  };

  // Weight fragments of `AHEAD` taps in registers.  Slot i of the ring holds tap g0 + i of a slab, g0 a multiple of
  // AHEAD, and is refilled behind its use.
  const uint4 *owp = (const uint4 *)a.owp + (size_t)wave * COF * 64 + lane;
  const int t_all = a.slabs_total * g.taps;
  constexpr int AHEAD = COF == 1 ? 9 : 3;
  uint4 wf[AHEAD][COF];
  auto load_weights = [&](int t, uint4 (&w)[COF]) {
    const uint4 *src = owp + (size_t)min(t, t_all - 1) * (4 * COF * 64);  // (past the end: never used)
#pragma unroll
    for (int cf = 0; cf < COF; ++cf) w[cf] = src[cf * 64];
  };
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) load_weights(i, wf[i]);

  const int qcol = frow * g.sw;  // patch pixel of this lane's column, output row 0, tap (0, 0)
  const int row_px = g.sh * a.PW;
  for (int slab0 = 0; slab0 < a.slabs_total; slab0 += a.stage) {
    const int slots = min(a.stage, a.slabs_total - slab0);
    __syncthreads();  // the previous stage's fragment reads are done
    for (int s = 0; s < slots; ++s) fetch(slab0 + s, s);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    for (int s = 0; s < slots; ++s) {
      const uint4 *X = patch + s * n_copies * 256;
      int ti = 0, tj = 0;
      for (int g0 = 0; g0 < g.taps; g0 += AHEAD) {
        const int next = g0 + AHEAD < g.taps ? (slab0 + s) * g.taps + g0 + AHEAD : (slab0 + s + 1) * g.taps;
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
          if (g0 + i < g.taps) {
            const int q0 = qcol + ti * g.dh * a.PW + tj * g.dw;
            uint4 af[TH];
#pragma unroll
            for (int th = 0; th < TH; ++th) {
              const int q = q0 + th * row_px;
              af[th] = X[q * 8 + ((wave * 2 + fhalf) ^ (q & 7))];
            }
#pragma unroll
            for (int th = 0; th < TH; ++th)
#pragma unroll
              for (int cf = 0; cf < COF; ++cf) TR::mma(acc[th][cf], af[th], wf[i][cf]);
            if (++tj == g.kw) tj = 0, ++ti;
          }
          load_weights(next + i, wf[i]);
        }
      }
    }
  }

  // Accumulator block (A = pixels, B = channels): register r of lane l holds
  //   pixel column = (r/4)*8 + (l/32)*4 + r%4,  channel = l%32.
  // The waves' blocks meet in LDS, RB of them at a time; wave w adds up and stores registers 4 w .. 4 w + 3.
  constexpr int RB = LDS_BYTES / 16384;
  f32x4 *red = (f32x4 *)patch;  // [block][wave][quad][64 lanes]
  E *raw = (E *)a.raw;
  const long plane_out = (long)g.Ho * g.Wo;
#pragma unroll
  for (int b0 = 0; b0 < TH * COF; b0 += RB) {
    __syncthreads();
#pragma unroll
    for (int b = b0; b < TH * COF && b < b0 + RB; ++b)
#pragma unroll
      for (int qd = 0; qd < 4; ++qd) {
        const f32x16 &c = acc[b / COF][b % COF];
        red[(((b - b0) * 4 + wave) * 4 + qd) * 64 + lane] = f32x4{c[4 * qd], c[4 * qd + 1], c[4 * qd + 2], c[4 * qd + 3]};
      }
    __syncthreads();
#pragma unroll
    for (int b = b0; b < TH * COF && b < b0 + RB; ++b) {
      f32x4 v = red[((b - b0) * 16 + wave) * 64 + lane];
#pragma unroll
      for (int k = 1; k < 4; ++k) v += red[(((b - b0) * 4 + k) * 4 + wave) * 64 + lane];
      const int ho = ho0 + b / COF, co = b % COF * 32 + frow;
      const float bias = a.obias && co < a.CO ? to_f32(((const E *)a.obias)[co]) : 0.0f;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int wo = wo0 + wave * 8 + fhalf * 4 + r;
        if (ho < g.Ho && wo < g.Wo)
          raw[((long)n * plane_out + (long)ho * g.Wo + wo) * a.CO_pad + co] = from_f32<E>(v[r] + bias);
      }
    }
  }
}

template <typename E, int COF>
hipError_t launch(OconvArgs a, hipStream_t st) {
  const Geom &g = a.g;
  constexpr int BIG = COF == 1 ? 4 : 2;
  a.tiles_x = (g.Wo + 31) / 32;
  a.PW = 31 * g.sw + (g.kw - 1) * g.dw + 1;
  auto tiles = [&](int th) { return (long)g.N * ((g.Ho + th - 1) / th) * a.tiles_x; };
  auto patch_rows = [&](int th) { return (long)(th - 1) * g.sh + (long)(g.kh - 1) * g.dh + 1; };
  // LDS of a slab's patch, whole copies of 4 KiB
  auto patch_bytes = [&](int th) { return (patch_rows(th) * a.PW * kRowB + 4095) / 4096 * 4096; };
  auto go = [&](int th, int lds, auto kernel) {
    a.PH = (int)patch_rows(th);
    a.tiles_y = (g.Ho + th - 1) / th;
    a.tiles = tiles(th);
    a.stage = (int)std::min<long>(a.slabs_total, lds / patch_bytes(th));
    hipLaunchKernelGGL(kernel, dim3((unsigned)((a.tiles + 7) / 8 * 8)), dim3(256), 0, st, a);
    return hipGetLastError();
  };
  // Several rows per workgroup, for the sake of the halo, where that gives every CU two of them
  if (patch_bytes(BIG) <= kOconvLds2 && tiles(BIG) >= 2L * num_cus())
    return patch_bytes(BIG) <= kOconvLds3 ? go(BIG, kOconvLds3, oconv_tiled_kernel<E, COF, BIG, kOconvLds3>)
                                          : go(BIG, kOconvLds2, oconv_tiled_kernel<E, COF, BIG, kOconvLds2>);
  // one row, as many slabs at a time as fit; a CU to itself where there are no more workgroups than CUs
  if (patch_bytes(1) <= kOconvLds2 && tiles(1) > num_cus())
    return go(1, kOconvLds2, oconv_tiled_kernel<E, COF, 1, kOconvLds2>);
  if (patch_bytes(1) <= kOconvLds1) return go(1, kOconvLds1, oconv_tiled_kernel<E, COF, 1, kOconvLds1>);
  constexpr int PXF = COF == 1 ? 4 : (COF == 2 ? 2 : 1);
  const long px_per_block = 4L * 32 * PXF;
  const long blocks = (a.total_px + px_per_block - 1) / px_per_block;
  hipLaunchKernelGGL((oconv_gather_kernel<E, COF, PXF>), dim3((unsigned)blocks), dim3(256), 0, st, a);
  return hipGetLastError();
}

template <typename E>
hipError_t launch_e(const OconvArgs &a, hipStream_t st) {
  switch (a.CO_pad / 32) {
    case 1: return launch<E, 1>(a, st);
    case 2: return launch<E, 2>(a, st);
    case 3: return launch<E, 3>(a, st);
    case 4: return launch<E, 4>(a, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t oconv_forward(int dtype, OconvArgs a, hipStream_t st) {
  switch (dtype) {
    case MDCN_F32: return launch_e<float>(a, st);
    case MDCN_F16: return launch_e<f16_t>(a, st);
    default: return launch_e<bf16_t>(a, st);
  }
}

}  // namespace mdcn
