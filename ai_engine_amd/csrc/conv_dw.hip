// conv_dw.hip -- depthwise KxK conv and the device-side NHWC <-> NHWC-C4 pack.
//
// Depthwise is HBM-bound (2 flops per weight per pixel, no reuse across
// channels). The arithmetic follows the reference depthwise path
// (crates/ai-cpu/src/kernels/dw.rs:40-204, ConvDwSpec
// crates/ai-gpu/src/kernels/conv_dw.rs:21-216): acc = bias, then the taps in
// (ky, kx) order, then act, then + residual.
//
// conv_dw_strip_kernel (k = 3 or 5, stride 1 or 2, dilation 1): a thread owns
// one 16-byte channel vector (4 fp32 or 8 16-bit channels; 8 bytes where a
// 16-bit pixel has no whole ones) of a strip of PX horizontally adjacent
// output pixels. Per kernel row it loads the (PX-1)*S + K input columns the
// strip needs once and reuses each of them for every tap that touches it;
// consecutive threads take consecutive channel vectors of a pixel, so a
// wavefront reads whole pixel rows.
//
// What bounds it: the loads in flight, then HBM (few channels a launch: the
// launch). Columns outside the image get an offset past the buffer and read
// zeros, so no load sits behind a branch that waits for the one before it, and
// indexes are 32-bit multiplications (three 64-bit divisions a thread cost as
// much as a 3x3's taps). SKIP: rows outside the image are branched over and
// the rows' loads follow each other, few registers and 8 wavefronts a SIMD;
// otherwise all rows' loads are out together, and such a row's weights are
// zeroed instead -- better for one-pixel strips, whose rows are short, and for
// fp32, where one row of a strip is enough in flight (measured per strip).
// A pass over buffers in turn: f16 3x3 S = 2 80x144 128 ch b32 42.3 us with a
// branch around each column's load, 26.5 here (118 MB, 4.5 TB/s). On one set of
// buffers again and again, so partly from the 256 MB cache: that call 32.4 ->
// 18.4, 5x5 80x144 96 ch b16 48.1 -> 26.6, 5x5 20x36 96 ch b64 19.0 -> 10.8, 3x3
// 40x72 64 ch b64 18.8 -> 13.2, 10x18 96 ch b1 4.1 -> 3.0; fp32 3x3 S = 2 80x144
// 96 ch b16 19.8 -> 14.5, 5x5 46.4 -> 35.6.
//
// conv_dw_kernel is the general fallback (any k, s, dilation).
#include "aih_device.h"
#include "conv_dw.h"

namespace aih {

template <int DT, int PX>
__global__ __launch_bounds__(256) void conv_dw_kernel(DwArgs a) {
  const uint32_t cg = a.CG;
  const uint64_t gid = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  const uint32_t owb = (a.OW + PX - 1) / PX;  // pixel blocks per output row
  const uint64_t total = (uint64_t)a.N * a.OH * owb * cg;
  if (gid >= total) return;
  const uint32_t g = (uint32_t)(gid % cg);
  uint64_t r = gid / cg;
  const uint32_t xb = (uint32_t)(r % owb);
  r /= owb;
  const uint32_t oy = (uint32_t)(r % a.OH);
  const uint32_t img = (uint32_t)(r / a.OH);
  const uint32_t ox0 = xb * PX;

  const f32x4 b = Vec4IO<DT>::load(a.bias, g);
  f32x4 acc[PX];
#pragma unroll
  for (int p = 0; p < PX; ++p) acc[p] = b;

  const size_t img_base = (size_t)img * a.IH * a.IW;
  for (uint32_t ky = 0; ky < a.K; ++ky) {
    const int32_t iy = (int32_t)(oy * a.S + ky * a.D) - a.PT;
    if ((uint32_t)iy >= a.IH) continue;
    const size_t row = img_base + (size_t)iy * a.IW;
    for (uint32_t kx = 0; kx < a.K; ++kx) {
      const f32x4 w = Vec4IO<DT>::load(a.w, (size_t)(ky * a.K + kx) * cg + g);
#pragma unroll
      for (int p = 0; p < PX; ++p) {
        const int32_t ix = (int32_t)((ox0 + p) * a.S + kx * a.D) - a.PL;
        if ((uint32_t)ix < a.IW && ox0 + p < a.OW) {
          const f32x4 x = Vec4IO<DT>::load(a.x, (row + (uint32_t)ix) * cg + g);
          acc[p] += x * w;
        }
      }
    }
  }
  const size_t orow = ((size_t)img * a.OH + oy) * a.OW;
#pragma unroll
  for (int p = 0; p < PX; ++p) {
    if (ox0 + p >= a.OW) break;
    const size_t vi = (orow + ox0 + p) * cg + g;
    f32x4 v = act4(act_params(a.act), acc[p]);
    if (a.has_res) v += Vec4IO<DT>::load(a.res, vi);
    Vec4IO<DT>::store(a.y, vi, v);
  }
}

// CV consecutive channels as stored: one 16-byte vector, or 8 bytes for
// CV = 4 at 16 bit.
template <int DT, int CV> struct Raw { using T = u32x4; };
template <> struct Raw<DT_F16, 4> { using T = u32x2; };
template <> struct Raw<DT_BF16, 4> { using T = u32x2; };

template <int DT, int CV>
__device__ __forceinline__ void cvt_cv(typename Raw<DT, CV>::T r, float (&out)[CV]) {
  if constexpr (DT == DT_F32) {
    const f32x4 v = __builtin_bit_cast(f32x4, r);
    out[0] = v.x; out[1] = v.y; out[2] = v.z; out[3] = v.w;
  } else if constexpr (CV == 8) {
    const f32x4 lo = unpack4<DT>(u32x2{r.x, r.y}), hi = unpack4<DT>(u32x2{r.z, r.w});
    out[0] = lo.x; out[1] = lo.y; out[2] = lo.z; out[3] = lo.w;
    out[4] = hi.x; out[5] = hi.y; out[6] = hi.z; out[7] = hi.w;
  } else {
    const f32x4 v = unpack4<DT>(r);
    out[0] = v.x; out[1] = v.y; out[2] = v.z; out[3] = v.w;
  }
}

template <int DT, int CV>
__device__ __forceinline__ void st_cv(void *base, size_t idx, const float (&v)[CV]) {
  if constexpr (DT == DT_F32) {
    reinterpret_cast<f32x4 *>(base)[idx] = f32x4{v[0], v[1], v[2], v[3]};
  } else if constexpr (CV == 8) {
    const u32x2 lo = pack4<DT>(f32x4{v[0], v[1], v[2], v[3]});
    const u32x2 hi = pack4<DT>(f32x4{v[4], v[5], v[6], v[7]});
    reinterpret_cast<u32x4 *>(base)[idx] = u32x4{lo.x, lo.y, hi.x, hi.y};
  } else {
    reinterpret_cast<u32x2 *>(base)[idx] = pack4<DT>(f32x4{v[0], v[1], v[2], v[3]});
  }
}

// The strip kernel's thread grid: (image, output row, strip of PX pixels,
// channel vector), channel vectors innermost.
struct DwGrid {
  uint32_t total, cgv, owb;
  FastDiv fd_cgv, fd_owb, fd_oh;
};

// A byte offset past every buffer: a window's valid offsets stay below it,
// and the sum of two of them does not wrap.
constexpr uint32_t kDwOob = 0x40000000u;

template <int DT, int CV, int K, int S, int PX>
__global__ __launch_bounds__(256) void conv_dw_strip_kernel(DwArgs a, DwGrid gr) {
  using V = typename Raw<DT, CV>::T;
  constexpr int NCOL = (PX - 1) * S + K;  // input columns under one strip
  constexpr uint32_t VB = sizeof(V);
  constexpr bool SKIP = DT == DT_F32 ? PX >= 4 && K == 5 : PX >= 2;
  // Workgroups are dealt round-robin to the 8 XCDs; remapping gives each XCD
  // a contiguous run of output rows, so the input rows shared by vertically
  // adjacent outputs are fetched into one L2 instead of one per XCD.
  const uint32_t gid0 = xcd_remap(blockIdx.x, gridDim.x, a.nxcd) * 256;
  // the workgroup's window of the input starts at its first thread's first row
  const uint32_t r0 = fdiv(fdiv(gid0, gr.fd_cgv), gr.fd_owb);
  const uint32_t img0 = fdiv(r0, gr.fd_oh);
  const int32_t top0 = (int32_t)((r0 - img0 * a.OH) * S) - a.PT;
  const uint32_t row0 = img0 * a.IH + (uint32_t)min(max(top0, 0), (int32_t)a.IH - 1);
  const uint32_t row_b = a.IW * gr.cgv * VB;
  const uint64_t left = (uint64_t)(a.N * a.IH - row0) * row_b;
  const __amdgpu_buffer_rsrc_t rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(static_cast<const char *>(a.x)) + (uint64_t)row0 * row_b, 0,
                                        left < kDwOob ? (int)left : (int)kDwOob, 0x00020000);

  const uint32_t gid = gid0 + threadIdx.x;
  if (gid >= gr.total) return;
  const uint32_t q = fdiv(gid, gr.fd_cgv), g = gid - q * gr.cgv;
  const uint32_t r = fdiv(q, gr.fd_owb), ox0 = (q - r * gr.owb) * PX;
  const uint32_t img = fdiv(r, gr.fd_oh), oy = r - img * a.OH;

  const V *wp = static_cast<const V *>(a.w) + g;
  float b[CV];
  cvt_cv<DT, CV>(static_cast<const V *>(a.bias)[g], b);
  float acc[PX][CV];
#pragma unroll
  for (int p = 0; p < PX; ++p)
#pragma unroll
    for (int j = 0; j < CV; ++j) acc[p][j] = b[j];

  uint32_t col[NCOL];
#pragma unroll
  for (int c = 0; c < NCOL; ++c) {
    const uint32_t ix = ox0 * S - (uint32_t)a.PL + c;
    col[c] = ix < a.IW ? (ix * gr.cgv + g) * VB : kDwOob;
  }
#pragma unroll
  for (int ky = 0; ky < K; ++ky) {
    const uint32_t iy = oy * S - (uint32_t)a.PT + ky;
    const bool ok = iy < a.IH;
    if constexpr (SKIP) {
      if (!ok) continue;
    }
    const uint32_t ro = SKIP || ok ? (img * a.IH + iy - row0) * row_b : kDwOob;
    float xv[NCOL][CV];
#pragma unroll
    for (int c = 0; c < NCOL; ++c) {
      if constexpr (VB == 16)
        cvt_cv<DT, CV>(__builtin_amdgcn_raw_buffer_load_b128(rs, (int)(ro + col[c]), 0, 0), xv[c]);
      else
        cvt_cv<DT, CV>(__builtin_amdgcn_raw_buffer_load_b64(rs, (int)(ro + col[c]), 0, 0), xv[c]);
    }
#pragma unroll
    for (int kx = 0; kx < K; ++kx) {
      // a row outside the image adds nothing, whatever its weights hold
      const V wr = wp[(uint32_t)(ky * K + kx) * gr.cgv];
      float w[CV];
      cvt_cv<DT, CV>(SKIP || ok ? wr : V{}, w);
#pragma unroll
      for (int p = 0; p < PX; ++p)
#pragma unroll
        for (int j = 0; j < CV; ++j) acc[p][j] += xv[p * S + kx][j] * w[j];
    }
  }
  const Act actp = act_params(a.act);
  const size_t orow = ((size_t)img * a.OH + oy) * a.OW;
#pragma unroll
  for (int p = 0; p < PX; ++p) {
    if (ox0 + p >= a.OW) break;
    const size_t vi = (orow + ox0 + p) * gr.cgv + g;
    float v[CV];
#pragma unroll
    for (int j = 0; j < CV; ++j) v[j] = acc[p][j];
    act_array<CV>(actp, v);
    if (a.has_res) {
      float rr[CV];
      cvt_cv<DT, CV>(static_cast<const V *>(a.res)[vi], rr);
#pragma unroll
      for (int j = 0; j < CV; ++j) v[j] += rr[j];
    }
    st_cv<DT, CV>(a.y, vi, v);
  }
}

// The thread grid of strips of px outputs; false where 32-bit indexes or a
// workgroup's window of the input do not reach (input rows of 100 MB).
static bool dw_grid(const DwArgs &a, uint32_t cgv, uint32_t vec_bytes, uint32_t px, DwGrid *g) {
  const uint32_t owb = (a.OW + px - 1) / px;
  const uint64_t rows_out = (uint64_t)a.N * a.OH, per = (uint64_t)owb * cgv;
  if (rows_out > 0x7fffffffu || per > 0x7fffffffu || rows_out * per > 0x7fffff00u ||
      (uint64_t)a.N * a.IH > 0x7fffffffu)
    return false;
  // input rows that 256 consecutive threads touch, from the first one's first row on
  const uint64_t nb = 255 / per + 2;
  const int64_t gap = (int64_t)a.IH + a.PT - (int64_t)(a.OH - 1) * a.S;  // last output row to the next image
  const uint64_t rows = nb * a.S + a.K + (nb / a.OH + 1) * (uint64_t)(gap > 0 ? gap : 0);
  if (rows * a.IW * cgv * vec_bytes >= kDwOob) return false;
  *g = DwGrid{(uint32_t)(rows_out * per), cgv, owb, make_fastdiv(cgv), make_fastdiv(owb), make_fastdiv(a.OH)};
  return true;
}

template <int DT, int CV, int K, int S, int PX>
static bool launch_strip_px(const DwArgs &a, hipStream_t st, hipError_t *e) {
  DwGrid g;
  if (!dw_grid(a, a.CG * 4 / CV, sizeof(typename Raw<DT, CV>::T), PX, &g)) return false;
  hipLaunchKernelGGL((conv_dw_strip_kernel<DT, CV, K, S, PX>), dim3((g.total + 255) / 256), dim3(256), 0, st, a, g);
  *e = hipGetLastError();
  return true;
}

// The strip length, by the threads one-pixel strips would make (t1): longer
// strips load each input column once for up to K / S of their pixels, one-pixel
// strips keep a small layer's tap loops short and the chip full. Each line's
// limits are multiples of the CUs; measured on both sides (us per call on one
// set of buffers, f16 unless said, 256 CUs: 256 threads a CU are 64K):
//   K = 3, S = 2: one pixel at every size (80x144 128 ch b32 18.4, strips of 4
//     21.7; fp32 80x144 96 ch b16 14.5 / 16.4). Nothing is shared but a border
//     column.
//   K = 3, S = 1, 8-channel vectors: 4 pixels from 2048 threads a CU (20x36 96
//     ch b64 7.2, 1 pixel 9.0; 10x18 192 ch b64, below it, 5.5 / 2 pixels 5.1),
//     2 from 512 (40x72 128 ch b4 4.2 / 1 pixel 4.4).
//   K = 5, 8-channel vectors: from 256 threads a CU 4 pixels, at S = 2 two
//     (80x144 96 ch b16 26.6 / 1 pixel 56; S = 2 13.9 / 17.8); 1 below (20x36
//     48 ch b1 4.2 / 2 pixels 4.9).
//   4-channel vectors (fp32, or 16 bit with an odd channel group): 4 pixels
//     from 1024 threads a CU, 2 from 256, else 1 (K = 3 S = 1 fp32: 40x72 128
//     ch b4 5.2 / 6.5 at 1 pixel, 80x144 44 ch b1 3.5 / 3.8, 10x18 96 ch b1
//     2.9 / 3.1 at 2); fp32 K = 5 S = 1 8 from 2048 (80x144 96 ch b16 35.6 / 4
//     pixels 42.8), fp32 K = 5 S = 2 at most 2 (21.6 / 4 pixels 28.5).
template <int DT, int CV, int K, int S>
static uint32_t dw_px(const DwArgs &a) {
  const uint64_t t1 = (uint64_t)a.N * a.OH * a.OW * (a.CG * 4 / CV), cus = device_cus();
  constexpr bool F32 = DT == DT_F32;
  if (K == 3 && S == 2 && (F32 || CV == 8)) return 1;
  if (CV == 8) {
    if (K == 5) return t1 >= cus * 256 ? (S == 1 ? 4 : 2) : 1;
    return t1 >= cus * 2048 ? 4 : t1 >= cus * 512 ? 2 : 1;
  }
  if (F32 && K == 5 && S == 1 && t1 >= cus * 2048) return 8;
  if (t1 >= cus * 1024) return F32 && K == 5 && S == 2 ? 2 : 4;
  return t1 >= cus * 256 ? 2 : 1;
}

template <int DT, int CV, int K, int S>
static bool launch_strip(const DwArgs &a, hipStream_t st, hipError_t *e) {
  switch (dw_px<DT, CV, K, S>(a)) {
    case 8:
      if constexpr (DT == DT_F32 && K == 5 && S == 1) return launch_strip_px<DT, CV, K, S, 8>(a, st, e);
      return false;
    case 4: return launch_strip_px<DT, CV, K, S, 4>(a, st, e);
    case 2: return launch_strip_px<DT, CV, K, S, 2>(a, st, e);
    default: return launch_strip_px<DT, CV, K, S, 1>(a, st, e);
  }
}

template <int DT, int CV>
static bool launch_strip_ks(const DwArgs &a, hipStream_t st, hipError_t *e) {
  if (a.K == 3) return a.S == 1 ? launch_strip<DT, CV, 3, 1>(a, st, e) : launch_strip<DT, CV, 3, 2>(a, st, e);
  return a.S == 1 ? launch_strip<DT, CV, 5, 1>(a, st, e) : launch_strip<DT, CV, 5, 2>(a, st, e);
}

hipError_t launch_conv_dw(const DwArgs &a, int dt, hipStream_t st) {
  if (a.D == 1 && (a.K == 3 || a.K == 5) && (a.S == 1 || a.S == 2)) {
    // two 4-channel groups per 16-byte vector where a pixel has whole ones
    const bool cv8 = a.CG % 2 == 0;
    hipError_t e = hipSuccess;
    bool done = false;  // false: past the strip kernel's index range
    switch (dt) {
      case DT_F32: done = launch_strip_ks<DT_F32, 4>(a, st, &e); break;
      case DT_F16: done = cv8 ? launch_strip_ks<DT_F16, 8>(a, st, &e) : launch_strip_ks<DT_F16, 4>(a, st, &e); break;
      case DT_BF16: done = cv8 ? launch_strip_ks<DT_BF16, 8>(a, st, &e) : launch_strip_ks<DT_BF16, 4>(a, st, &e); break;
      default: return hipErrorInvalidValue;
    }
    if (done) return e;
  }
  constexpr int PX = 2;
  const uint64_t total = (uint64_t)a.N * a.OH * ((a.OW + PX - 1) / PX) * a.CG;
  const dim3 grid((unsigned)((total + 255) / 256));
  switch (dt) {
    case DT_F32: hipLaunchKernelGGL((conv_dw_kernel<DT_F32, PX>), grid, dim3(256), 0, st, a); break;
    case DT_F16: hipLaunchKernelGGL((conv_dw_kernel<DT_F16, PX>), grid, dim3(256), 0, st, a); break;
    case DT_BF16: hipLaunchKernelGGL((conv_dw_kernel<DT_BF16, PX>), grid, dim3(256), 0, st, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// Logical NHWC fp32 -> NHWC-C4 in DT (zero-filled channel padding); one
// output vec4 per thread.
template <int DT>
__global__ __launch_bounds__(256) void pack_nhwc_kernel(const float *__restrict__ x, uint64_t px, uint32_t c,
                                                        void *y) {
  const uint32_t cg = (c + 3) / 4;
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= px * cg) return;
  const uint64_t p = i / cg;
  const uint32_t g = (uint32_t)(i - p * cg);
  f32x4 v = {};
#pragma unroll
  for (int l = 0; l < 4; ++l) {
    const uint32_t ch = g * 4 + l;
    if (ch < c) v[l] = x[p * c + ch];
  }
  Vec4IO<DT>::store(y, i, v);
}

hipError_t launch_pack_nhwc(const float *x, uint64_t px, uint32_t c, int dt, void *y, hipStream_t st) {
  const uint64_t n = px * ((c + 3) / 4);
  const dim3 grid((unsigned)((n + 255) / 256));
  switch (dt) {
    case DT_F32: hipLaunchKernelGGL(pack_nhwc_kernel<DT_F32>, grid, dim3(256), 0, st, x, px, c, y); break;
    case DT_F16: hipLaunchKernelGGL(pack_nhwc_kernel<DT_F16>, grid, dim3(256), 0, st, x, px, c, y); break;
    case DT_BF16: hipLaunchKernelGGL(pack_nhwc_kernel<DT_BF16>, grid, dim3(256), 0, st, x, px, c, y); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// Pixels of stride_c storage channels, from channel c_off on -> logical fp32
// NHWC; one value per thread. The way back of a result to the host: with
// the padding gone before the copy (and 16-bit values widened, exactly) the
// copy is the caller's bytes and the host has no pass over them (160x288x2
// fp32 b1: 368 KB instead of 737, and no second buffer).
template <int DT>
__global__ __launch_bounds__(256) void unpack_nhwc_kernel(const typename Storage<DT>::T *__restrict__ x,
                                                          uint32_t stride_c, FastDiv fd_c, uint32_t total,
                                                          float *__restrict__ y) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const uint32_t p = fdiv(i, fd_c);
  const typename Storage<DT>::T v = x[(size_t)p * stride_c + (i - p * fd_c.d)];
  if constexpr (DT == DT_F32) y[i] = v;
  else if constexpr (DT == DT_F16) y[i] = f16_to_f32(v);
  else y[i] = bf16_to_f32(v);
}

hipError_t launch_unpack_nhwc(const void *x, uint32_t px, uint32_t c, uint32_t stride_c, int dt, float *y,
                              hipStream_t st) {
  const uint64_t n = (uint64_t)px * c;
  if (n == 0 || n > 0x7fffff00u) return hipErrorInvalidValue;
  const FastDiv fd = make_fastdiv(c);
  const dim3 grid((unsigned)((n + 255) / 256));
#define AIH_UNPACK(DT)                                                                                      \
  hipLaunchKernelGGL(unpack_nhwc_kernel<DT>, grid, dim3(256), 0, st, static_cast<const Storage<DT>::T *>(x), \
                     stride_c, fd, (uint32_t)n, y)
  switch (dt) {
    case DT_F32: AIH_UNPACK(DT_F32); break;
    case DT_F16: AIH_UNPACK(DT_F16); break;
    case DT_BF16: AIH_UNPACK(DT_BF16); break;
    default: return hipErrorInvalidValue;
  }
#undef AIH_UNPACK
  return hipGetLastError();
}

}  // namespace aih
