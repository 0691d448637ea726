// conv_stream.hip -- conv GEMM with both operands streamed through LDS by
// DMA: pointwise convs and KxK implicit GEMMs (one input, plain or a channel
// view) with 16-bit or fp32 storage, the role of gemm_pw_tiled.wgsl and
// conv_igemm_tiled.wgsl (crates/ai-gpu/src/kernels/{gemm_pw,conv_igemm}.rs),
// with the bias -> act -> +residual epilogue of common/epilogue.rs:13-30.
//
// K is one sequence of 16-byte units (4 fp32 / 8 16-bit channels), tap-major;
// a stage is BKU = 4 or 8 units. A stage's pixel rows and weight rows go from memory to
// LDS without passing through registers, NST - 1 stages ahead of the MFMAs:
// out-of-image taps, missing pixels, missing columns and the K tail get an
// offset past the buffer, which the DMA fills with zeros. The implicit
// im2col costs a lane one tap counter (its unit advances BKU per stage, at most
// one tap further since a tap has at least BKU units) and one add and two mask
// tests per pixel row. One workgroup barrier per stage publishes a landed
// stage and frees the oldest buffer.
//
// LDS layout of a stage: unit u of tile pixel p at slot BKU p + (u ^ swz(p)), so
// the MFMA operand reads (8 pixels, one unit each, per LDS cycle) touch 8
// distinct bank groups while the DMA lanes still read whole 64-byte runs of a
// pixel; weights as kg rows of BN columns (16 bytes a column at fp32, 8 at
// 16 bit), read as one b128 or two b64 of consecutive columns.
//
// MFMA mapping: A = weights (32 channels x K), B = activations (K x 32
// pixels), lane half h takes unit 2q + h of pair q for both operands; a
// wavefront holds TM x TN blocks of 32 pixels x 32 channels, so one operand
// read feeds TM (weights) or TN (activations) MFMAs. Lane l of a result holds
// pixel l%32 and channels 8*(r/4) + 4*(l/32) + r%4 (r = 0..15). The epilogue
// passes 32 pixels x up to 64 channels at a time through the wavefront's own
// LDS rows (the stage buffers, free by then), so stores and residual loads
// move whole runs of a pixel's channels, 16 bytes a lane.
//
// What bounds it: at 16 bit the stages' round trips. A 128 x 128 tile's
// wavefront has 8 MFMAs a stage between two barriers, and of its time 49 %
// waits, while the MFMAs are busy 26 %, the LDS 29 % and the VALU about 30 %
// (counters on 3x3 128 -> 128 f16 at 40x72 b32; 192 -> 768 at 21x37 b64: 43 % and
// 16, 27 and 32 %, 100 MB of HBM traffic at 2.7 TB/s). The LDS rate would come
// next: 2 x 2 blocks read 1 KB per 32-cycle MFMA, 128 bytes a cycle over four
// SIMDs. At fp32 the MFMAs bound it (64 -> 128 3x3 b32: busy 63 %, 222 -> 117
// us of 104 at the rate a large product reaches). Times of a pass over buffers
// in turn: 3x3 128 -> 128 69.5 us on the register-staged tiled GEMM, 39 here
// (700 TFLOP/s), 192 -> 768 64.5 and 39. On one set of buffers again and again
// (38 / 37 us) other shapes of it took: 256 x 128 tiles of 8 wavefronts 55 /
// 41 and 128 x 192 ones 62 / 43 (fewer workgroups to overlap), stages of 8
// units at 128 x 128 49 / 39 (LDS for two workgroups a CU), three stages of 4
// 42 / 36.
#include <hip/hip_runtime.h>

#include "conv_stream.h"

namespace aih {
namespace {

typedef __attribute__((address_space(3))) void cs_lds_void;
constexpr uint32_t kOob = 0x80000000u;  // a byte offset past every buffer

__device__ __forceinline__ __amdgpu_buffer_rsrc_t cs_rsrc(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
}

// The XOR of a pixel's unit index that spreads 8 consecutive pixels' units
// over 8 bank groups: bits 1 and 2 of the pixel (swapped) with 4 units a
// pixel, its low three bits with 8.
template <int BKU>
__device__ __forceinline__ uint32_t cs_swz(uint32_t p) {
  return BKU == 8 ? p & 7 : (((p >> 1) & 1) << 1) | ((p >> 2) & 1);
}

// s_waitcnt vmcnt(N) (expcnt and lgkmcnt not waited for).
template <int N>
__device__ __forceinline__ void cs_wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
}

// vmcnt(n) for a wavefront-uniform n in [0, MAXN].
template <int MAXN>
__device__ __forceinline__ void cs_wait_vm_n(uint32_t n) {
  if constexpr (MAXN > 0) {
    if (n >= (uint32_t)MAXN) {
      cs_wait_vm<MAXN>();
      return;
    }
    cs_wait_vm_n<MAXN - 1>(n);
  } else {
    cs_wait_vm<0>();
  }
}

template <int WM, int WN, int TM, int TN, int BKU, int NST>
struct CsCfg {
  static constexpr int NW = WM * WN, BM = 32 * WM * TM, BN = 32 * WN * TN;
  static constexpr uint32_t A_BYTES = BM * BKU * 16, STAGE = (BM + BN) * BKU * 16;
  static constexpr int CW = TN % 2 == 0 ? 64 : 32;  // channels per staged epilogue chunk
  static constexpr int PITCH = CW + 4;              // floats per staged pixel row
  static constexpr uint32_t LDS =
      NST * STAGE > NW * 32u * PITCH * 4u ? NST * STAGE : NW * 32u * PITCH * 4u;
};

template <int DT, int WM, int WN, int TM, int TN, int BKU, int NST, bool IGEMM>
__global__ __launch_bounds__(64 * WM * WN) void conv_stream_kernel(ConvStreamArgs a) {
  using Cfg = CsCfg<WM, WN, TM, TN, BKU, NST>;
  constexpr bool F32 = DT == DT_F32;
  constexpr int NW = Cfg::NW, BM = Cfg::BM, BN = Cfg::BN;
  constexpr int PPD = 64 / BKU;                     // pixels of a DMA instruction
  constexpr int AI = BM / PPD / NW;                 // pixel-row DMA instructions of a wavefront per stage
  constexpr int W_INS = BN * BKU / 64;                  // weight DMA instructions of a stage
  constexpr int WI = (W_INS + NW - 1) / NW;         // the most of them one wavefront issues
  constexpr int SKG = F32 ? BKU : 2 * BKU;                 // kg rows of a stage
  constexpr int WCOLS = F32 ? BN : BN / 2;          // 16-byte entries of one kg row
  constexpr int CPE = F32 ? 1 : 2;                  // columns of an entry
  constexpr uint32_t KGB = F32 ? 16 : 8;            // bytes of one (kg, column)
  constexpr uint32_t A_BYTES = Cfg::A_BYTES, STAGE = Cfg::STAGE;
  static_assert(BM % (PPD * NW) == 0, "pixel rows split evenly over the wavefronts");
  extern __shared__ __align__(16) char lds[];

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, lh = lane >> 5;
  // wavefront-uniform: every branch on it is a scalar branch
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;

  const uint32_t t = xcd_remap(blockIdx.x, gridDim.x, a.nxcd);
  const uint32_t mt = fdiv(t, a.fd_nt), nt = t - mt * a.ntiles;
  const uint32_t m0 = mt * BM, n0 = nt * BN;
  const uint32_t nst = a.nst;

  const __amdgpu_buffer_rsrc_t rs_x = cs_rsrc(a.x, a.x_bytes);
  const __amdgpu_buffer_rsrc_t rs_w = cs_rsrc(a.w, a.w_bytes);

  // ---- pixel rows: instruction k of this wavefront moves tile pixels
  // PPD i + lane / BKU (i = wave + k NW), LDS slot lane % BKU holding unit
  // (lane % BKU) ^ swz of the pixel (the same unit for every k) ----
  uint32_t xu = (uint32_t)(lane % BKU) ^ cs_swz<BKU>((uint32_t)lane / BKU);  // unit inside the current tap
  uint32_t ky = 0, kx = 0;
  uint32_t x_off[AI];              // byte offset at tap (0, 0), unit 0 (wraps above / left of the image)
  uint32_t x_rows[AI], x_cols[AI]; // bit j: kernel row / column j inside the image
#pragma unroll
  for (int k = 0; k < AI; ++k) {
    const uint32_t m = m0 + PPD * (wave + k * NW) + lane / BKU;
    const bool ok = m < a.M;
    if constexpr (IGEMM) {
      const uint32_t mm = ok ? m : 0;
      const uint32_t img = fdiv(mm, a.fd_ohw);
      const uint32_t rem = mm - img * a.OHW;
      const uint32_t oy = fdiv(rem, a.fd_ow);
      const uint32_t ox = rem - oy * a.OW;
      const int32_t iy0 = (int32_t)(oy * a.S) - a.PT, ix0 = (int32_t)(ox * a.S) - a.PL;
      uint32_t rows = 0, cols = 0;
      for (uint32_t j = 0; j < a.K; ++j) {
        rows |= (uint32_t)((uint32_t)(iy0 + (int32_t)(j * a.D)) < a.IH) << j;
        cols |= (uint32_t)((uint32_t)(ix0 + (int32_t)(j * a.D)) < a.IW) << j;
      }
      x_rows[k] = ok ? rows : 0u;
      x_cols[k] = cols;
      const uint32_t pix = (img * a.IH + (uint32_t)iy0) * a.IW + (uint32_t)ix0;
      x_off[k] = (pix * a.stride_u + a.off_u) * 16u;
    } else {
      x_rows[k] = ok;
      x_cols[k] = 1;
      x_off[k] = (m * a.stride_u + a.off_u) * 16u;
    }
  }
  // ---- weight rows: instruction i (= wave + k NW) moves entries 64 i + lane
  // of the stage's [SKG][WCOLS] rows ----
  uint32_t w_off[WI], w_kg[WI], w_tap[WI];  // byte offset, kg inside the current tap, tap
  bool w_ok[WI];
#pragma unroll
  for (int k = 0; k < WI; ++k) {
    const uint32_t e = 64 * (wave + k * NW) + lane;
    const uint32_t kgl = e / WCOLS, n = n0 + (e - kgl * WCOLS) * CPE;
    w_ok[k] = n < a.N4;
    w_kg[k] = kgl;
    w_tap[k] = 0;
    w_off[k] = (kgl * a.N4 + n) * KGB;
  }
  const uint32_t taps = IGEMM ? a.K * a.K : 1;
  const uint32_t w_step = SKG * a.N4 * KGB, w_wrap = (a.KGP - a.KG) * a.N4 * KGB;

  // requests the next stage (stages are requested in order) into buffer b
  auto issue = [&](uint32_t b) {
    char *base = lds + b * STAGE;
    const uint32_t d_tap = IGEMM ? ((ky * a.D * a.IW + kx * a.D) * a.stride_u + xu) * 16u : xu * 16u;
#pragma unroll
    for (int k = 0; k < AI; ++k) {
      bool ok;
      if constexpr (IGEMM)
        ok = ((x_rows[k] >> ky) & (x_cols[k] >> kx) & 1u) != 0;  // no bits at or past row K: the K tail
      else
        ok = (x_rows[k] != 0) & (xu < a.KU);
      const uint32_t off = ok ? x_off[k] + d_tap : kOob;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_x, (cs_lds_void *)(base + (wave + k * NW) * 1024), 16, off, 0, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < WI; ++k) {
      if (W_INS % NW != 0 && wave + k * NW >= W_INS) break;
      const bool ok = w_ok[k] & (IGEMM ? w_tap[k] < taps : w_kg[k] < a.KG);
      const uint32_t off = ok ? w_off[k] : kOob;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_w, (cs_lds_void *)(base + A_BYTES + (wave + k * NW) * 1024), 16, off,
                                               0, 0, 0);
    }
    // on to the next stage's units: at most one tap further
    xu += BKU;
    if constexpr (IGEMM) {
      const bool wrap = xu >= a.KU;
      xu -= wrap ? a.KU : 0u;
      kx += wrap ? 1u : 0u;
      const bool row = kx == a.K;
      kx = row ? 0u : kx;
      ky += row ? 1u : 0u;
    }
#pragma unroll
    for (int k = 0; k < WI; ++k) {
      w_off[k] += w_step;
      w_kg[k] += SKG;
      if constexpr (IGEMM) {
        const bool wrap = w_kg[k] >= a.KG;
        w_kg[k] -= wrap ? a.KG : 0u;
        w_off[k] += wrap ? w_wrap : 0u;
        w_tap[k] += wrap ? 1u : 0u;
      }
    }
  };

  // LDS byte offsets (inside a stage) of this lane's operands of pair q
  uint32_t a_off[BKU / 2];
  const uint32_t p = 32 * TM * wm + l32;  // tile pixel of this lane in block tm = 0 (the swizzle repeats every 8)
#pragma unroll
  for (int q = 0; q < BKU / 2; ++q) a_off[q] = (BKU * p + ((2 * q + lh) ^ cs_swz<BKU>(p))) * 16;
  const uint32_t wl = A_BYTES + ((F32 ? lh : 2 * lh) * BN + 32 * TN * wn + l32) * KGB;

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x16{};

  auto compute = [&](uint32_t b) {
    const char *base = lds + b * STAGE;
#pragma unroll
    for (int q = 0; q < BKU / 2; ++q) {
      u32x4 xv[TM], wv[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) xv[i] = *reinterpret_cast<const u32x4 *>(base + a_off[q] + i * 32 * BKU * 16);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if constexpr (F32) {
          wv[j] = *reinterpret_cast<const u32x4 *>(base + wl + (2 * q * BN + 32 * j) * KGB);
        } else {
          const u32x2 lo = *reinterpret_cast<const u32x2 *>(base + wl + (4 * q * BN + 32 * j) * KGB);
          const u32x2 hi = *reinterpret_cast<const u32x2 *>(base + wl + ((4 * q + 1) * BN + 32 * j) * KGB);
          wv[j] = u32x4{lo.x, lo.y, hi.x, hi.y};
        }
      }
      if constexpr (F32) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(__builtin_bit_cast(f32x4, wv[j])[c],
                                                               __builtin_bit_cast(f32x4, xv[i])[c], acc[i][j], 0, 0, 0);
      } else {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            if constexpr (DT == DT_F16)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, wv[j]),
                                                                 __builtin_bit_cast(f16x8, xv[i]), acc[i][j], 0, 0, 0);
            else
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, wv[j]),
                                                                  __builtin_bit_cast(bf16x8, xv[i]), acc[i][j], 0, 0, 0);
          }
      }
    }
  };

  // ---- pipeline: stage s + NST - 1 is requested while stage s computes ----
  const uint32_t nmine = AI + (W_INS % NW == 0 ? WI : (uint32_t)((W_INS - wave + NW - 1) / NW));
#pragma unroll
  for (int s = 0; s < NST - 1; ++s)
    if ((uint32_t)s < nst) issue((uint32_t)s);
  uint32_t b_cmp = 0, b_iss = NST - 1;  // buffer of the stage computed / requested
  for (uint32_t s = 0; s < nst; ++s) {
    // this wavefront's copies of stage s have landed once at most those of
    // the stages requested after it are still in flight
    const uint32_t later = nst - 1 - s < (uint32_t)(NST - 2) ? nst - 1 - s : (uint32_t)(NST - 2);
    cs_wait_vm_n<(AI + WI) * (NST - 2)>(later * nmine);
    // every wavefront's copies of stage s are in LDS, and every wavefront is
    // done with stage s - 1, whose buffer the next request reuses: its LDS
    // reads have returned (written out, so that it does not hang on where the
    // compiler puts the MFMAs that wait for them). A bare barrier:
    // __syncthreads()'s workgroup fence would also wait for the copies still
    // in flight.
    __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (s + NST - 1 < nst) issue(b_iss);
    compute(b_cmp);
    b_cmp = b_cmp + 1 == NST ? 0 : b_cmp + 1;
    b_iss = b_iss + 1 == NST ? 0 : b_iss + 1;
  }
  __syncthreads();  // the stage buffers become the wavefronts' staging rows

  // ---- epilogue: act(acc + bias) (+ residual), whole pixel runs ----
  const Act actp = act_params(a.act);
  constexpr int CW = Cfg::CW, PITCH = Cfg::PITCH, CB = CW / 32;
  constexpr int LPR = CW / (F32 ? 4 : 8);  // lanes of one pixel row (16 bytes of storage each)
  constexpr int PPI = 64 / LPR;            // pixels per store instruction
  float *st = reinterpret_cast<float *>(lds) + wave * 32 * PITCH;
  // 16-bit rows start 16-byte aligned only when N4 % 8 == 0
  const bool row16 = F32 || a.N4 % 8 == 0;
  const uint32_t rl = lane / LPR, cl = (lane % LPR) * (F32 ? 4 : 8);
#pragma unroll
  for (int j0 = 0; j0 < TN; j0 += CB) {
    // the lane's channels are the same for every pixel of the chunk
    const uint32_t n = n0 + 32 * (TN * wn + j0) + cl;
    const bool n_ok = n < a.N4, two = n + 8 <= a.N4;
    const f32x4 b0 = n_ok ? Vec4IO<DT>::load(a.bias, n / 4) : f32x4{};
    const f32x4 b1 = !F32 && two ? Vec4IO<DT>::load(a.bias, n / 4 + 1) : f32x4{};
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < CB; ++j)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4)
          *reinterpret_cast<f32x4 *>(st + l32 * PITCH + 32 * j + 8 * r4 + 4 * lh) =
              f32x4{acc[i][j0 + j][4 * r4], acc[i][j0 + j][4 * r4 + 1], acc[i][j0 + j][4 * r4 + 2],
                    acc[i][j0 + j][4 * r4 + 3]};
      __builtin_amdgcn_wave_barrier();
#pragma unroll 2
      for (int g = 0; g < 32 / PPI; ++g) {
        const uint32_t r = g * PPI + rl;
        const uint32_t m = m0 + 32 * (TM * wm + i) + r;
        if (m < a.M && n_ok) {
          const size_t vi = ((size_t)m * a.N4 + n) / 4;
          f32x4 v0 = *reinterpret_cast<const f32x4 *>(st + r * PITCH + cl) + b0;
          if constexpr (F32) {
            v0 = act4(actp, v0);
            if (a.has_res) v0 += reinterpret_cast<const f32x4 *>(a.res)[vi];
            reinterpret_cast<f32x4 *>(a.y)[vi] = v0;
          } else {
            const f32x4 s1 = *reinterpret_cast<const f32x4 *>(st + r * PITCH + cl + 4) + b1;
            float v[8] = {v0.x, v0.y, v0.z, v0.w, s1.x, s1.y, s1.z, s1.w};
            act_array<8>(actp, v);
            v0 = f32x4{v[0], v[1], v[2], v[3]};
            f32x4 v1 = f32x4{v[4], v[5], v[6], v[7]};
            if (a.has_res) {
              if (row16) {
                const u32x4 rv = reinterpret_cast<const u32x4 *>(a.res)[vi / 2];
                v0 += unpack4<DT>(u32x2{rv.x, rv.y});
                v1 += unpack4<DT>(u32x2{rv.z, rv.w});
              } else {
                v0 += Vec4IO<DT>::load(a.res, vi);
                if (two) v1 += Vec4IO<DT>::load(a.res, vi + 1);
              }
            }
            const u32x2 lo = pack4<DT>(v0), hi = pack4<DT>(v1);
            if (row16) {
              reinterpret_cast<u32x4 *>(a.y)[vi / 2] = u32x4{lo.x, lo.y, hi.x, hi.y};
            } else {
              reinterpret_cast<u32x2 *>(a.y)[vi] = lo;
              if (two) reinterpret_cast<u32x2 *>(a.y)[vi + 1] = hi;
            }
          }
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

template <int DT, int WM, int WN, int TM, int TN, int BKU, int NST, bool IGEMM>
hipError_t launch_inst(const ConvStreamArgs &a, hipStream_t st) {
  constexpr uint32_t lds = CsCfg<WM, WN, TM, TN, BKU, NST>::LDS;
  static const hipError_t attr =
      hipFuncSetAttribute(reinterpret_cast<const void *>(conv_stream_kernel<DT, WM, WN, TM, TN, BKU, NST, IGEMM>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL((conv_stream_kernel<DT, WM, WN, TM, TN, BKU, NST, IGEMM>), dim3(a.mtiles * a.ntiles), dim3(64 * WM * WN),
                     lds, st, a);
  return hipGetLastError();
}

template <int DT>
hipError_t launch_dt(const ConvStreamArgs &a, const ConvStreamShape &s, hipStream_t st) {
  // pointwise: output pixel m reads input pixel m (a 1x1 conv with a stride or
  // padding is an implicit GEMM of one tap)
  const bool pw = a.K == 1 && a.S == 1 && a.PT == 0 && a.PL == 0 && a.OW == a.IW && a.OHW == a.IH * a.IW;
#define AIH_CS_CASE(WM, WN, TM, TN, BKU, NST)                                                         \
  if (s.wm == WM && s.wn == WN && s.tm == TM && s.tn == TN && s.bku == BKU && s.nst == NST)            \
    return pw ? launch_inst<DT, WM, WN, TM, TN, BKU, NST, false>(a, st)                               \
              : launch_inst<DT, WM, WN, TM, TN, BKU, NST, true>(a, st);
  AIH_CS_CASE(2, 2, 2, 2, 4, 2)
  AIH_CS_CASE(4, 1, 1, 3, 4, 3)
  AIH_CS_CASE(4, 1, 1, 2, 4, 3)
  AIH_CS_CASE(2, 2, 1, 1, 4, 3)
  AIH_CS_CASE(2, 2, 1, 1, 8, 2)
#undef AIH_CS_CASE
  return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_conv_stream(const ConvStreamArgs &a, int dt, const ConvStreamShape &s, hipStream_t st) {
  const uint32_t bm = conv_stream_bm(s), bn = conv_stream_bn(s);
  if (a.M == 0 || a.KU < s.bku || a.N4 == 0 || a.N4 % 4 || a.K == 0 || a.K > 15 || a.x_bytes >= 0x80000000u ||
      a.w_bytes >= 0x80000000u || a.off_u + a.KU > a.stride_u || a.KG != a.KU * (dt == DT_F32 ? 1u : 2u) ||
      a.KGP < a.KG || a.nst != (a.K * a.K * a.KU + s.bku - 1) / s.bku || a.mtiles != (a.M + bm - 1) / bm ||
      a.ntiles != (a.N4 + bn - 1) / bn || (uint64_t)a.mtiles * a.ntiles > 0x7fffffffu)
    return hipErrorInvalidValue;
  switch (dt) {
    case DT_F32: return launch_dt<DT_F32>(a, s, st);
    case DT_F16: return launch_dt<DT_F16>(a, s, st);
    case DT_BF16: return launch_dt<DT_BF16>(a, s, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace aih
