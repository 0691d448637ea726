// conv_ksplit.hip -- KxK conv for few output pixels, K split over the
// wavefronts of a workgroup: the layers of one frame or a few, whose 32-pixel
// blocks are fewer than the CUs (3x3 72 -> 32 at 40x72: 90 of them), with the
// operands loaded straight from memory into MFMA registers. The reference's
// route for these layers is conv_igemm_direct.wgsl
// (crates/ai-gpu/src/kernels/conv_igemm.rs); the in-workgroup split is its
// gemm_pw_splitk.wgsl:1-57 with the taps in K.
//
// What bounds such a layer is its serial chain: with a whole K a wavefront
// works through 9 taps one after the other, and the weights' copy to LDS comes
// before. Here a workgroup owns 16 pixels x 16 channels and wavefront w the
// (tap, step) pairs [w per, (w + 1) per) -- one tap each at 3x3 -- with a
// batch of operands in flight together; the partials meet in LDS and
// wavefront 0 (bias and residual loaded with its operands) sums them in
// wavefront order and applies act(acc + bias) (+ residual)
// (common/epilogue.rs:13-30). Nothing is staged, so a workgroup re-reads its
// weights from the caches.
//
// A step is 4 units of 16 bytes (4 fp32 / 8 16-bit channels) of one input
// part, lane group q = lane / 16 taking unit 4s + q of both operands (weights
// = A, rows = channels; pixels = B): four v_mfma_f32_16x16x4f32, one per
// component, or one v_mfma_f32_16x16x32. Out-of-image taps, missing pixels,
// missing channels, units past a part and pairs past the range are loaded from
// past the buffer, as zeros. Result lane l holds pixel l%16 and channels
// 4q .. 4q + 3.
#include <hip/hip_runtime.h>

#include "conv_ksplit.h"

namespace aih {
namespace {

constexpr uint32_t kOob = 0x80000000u;  // a byte offset past every buffer
constexpr int W = kConvKsplitWaves;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t ck_rsrc(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
}

// B: (tap, step) pairs whose operands are in flight together.
template <int DT, int B>
__global__ __launch_bounds__(64 * W) void conv_ksplit_kernel(ConvKsplitArgs a) {
  constexpr bool F32 = DT == DT_F32;
  constexpr uint32_t KGB = F32 ? 16 : 8;  // bytes of one (kg, column) of the weights
  constexpr uint32_t KPU = F32 ? 1 : 2;   // kg of a unit
  __shared__ f32x4 part[W][64];
  const int lane = threadIdx.x & 63, l16 = lane & 15;
  const uint32_t q = lane >> 4;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t b = xcd_remap(blockIdx.x, gridDim.x, a.nxcd);
  const uint32_t mb = fdiv(b, a.fd_nblk), nb = b - mb * a.nblk;
  const uint32_t p = mb * 16 + l16;  // this lane's pixel (B column, output pixel)
  const uint32_t n = nb * 16 + l16;  // this lane's output channel (A row)
  const bool pv = p < a.M;

  // the epilogue's operands (wavefront 0) go out with the first K operands
  const uint32_t c0 = nb * 16 + 4 * q;
  const bool ov = pv & (c0 < a.N4);
  const size_t vi = (size_t)p * (a.N4 / 4) + c0 / 4;
  f32x4 bv = {0.0f, 0.0f, 0.0f, 0.0f}, rv = {0.0f, 0.0f, 0.0f, 0.0f};
  if (wave == 0 && ov) {
    bv = Vec4IO<DT>::load(a.bias, c0 / 4);
    if (a.has_res) rv = Vec4IO<DT>::load(a.res, vi);
  }

  const uint32_t pp = pv ? p : 0;
  const uint32_t img = fdiv(pp, a.fd_ohw), rem = pp - img * a.OHW;
  const uint32_t oy = fdiv(rem, a.fd_ow), ox = rem - oy * a.OW;
  const uint32_t iy0 = oy * a.S - (uint32_t)a.PT, ix0 = ox * a.S - (uint32_t)a.PL;
  const __amdgpu_buffer_rsrc_t rs0 = ck_rsrc(a.src[0], a.src_bytes[0]), rs1 = ck_rsrc(a.src[1], a.src_bytes[1]);
  const __amdgpu_buffer_rsrc_t rs_w = ck_rsrc(a.w, a.w_bytes);
  const uint32_t wl = n < a.N4 ? n * KGB : kOob;

  const uint32_t i0 = wave * a.per;
  const uint32_t i1 = i0 + a.per < a.items ? i0 + a.per : a.items;
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  for (uint32_t ib = i0; ib < i1; ib += B) {
    u32x4 wv[B], xv[B];
#pragma unroll
    for (int k = 0; k < B; ++k) {
      const uint32_t i = ib + k;  // uniform, and so are the tap and the step
      const uint32_t tap = fdiv(i, a.fd_st), s = i - tap * a.st;
      const uint32_t ky = fdiv(tap, a.fd_k), kx = tap - ky * a.K;
      const bool p1 = s >= a.st0;
      const uint32_t u = 4 * (s - (p1 ? a.st0 : 0u)) + q;
      const bool uv = (i < i1) & (u < (p1 ? a.nu[1] : a.nu[0]));
      const uint32_t iy = iy0 + ky * a.D, ix = ix0 + kx * a.D;
      const bool xok = uv & pv & (iy < a.IH) & (ix < a.IW);
      const uint32_t pix = (img * a.IH + iy) * a.IW + ix;
      const uint32_t xo = (pix * (p1 ? a.stride_u[1] : a.stride_u[0]) + (p1 ? a.off_u[1] : a.off_u[0]) + u) * 16u;
      xv[k] = __builtin_amdgcn_raw_buffer_load_b128(p1 ? rs1 : rs0, (int)(xok ? xo : kOob), 0, 0);
      const uint32_t kg = (p1 ? a.kg_first[1] : a.kg_first[0]) + u * KPU;
      const uint32_t wo = (tap * a.KGP + kg) * a.N4 * KGB + wl;
      const bool wok = uv & (n < a.N4);
      if constexpr (F32) {
        wv[k] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, (int)(wok ? wo : kOob), 0, 0);
      } else {
        const u32x2 lo = __builtin_amdgcn_raw_buffer_load_b64(rs_w, (int)(wok ? wo : kOob), 0, 0);
        const u32x2 hi = __builtin_amdgcn_raw_buffer_load_b64(rs_w, (int)(wok ? wo + a.N4 * KGB : kOob), 0, 0);
        wv[k] = u32x4{lo.x, lo.y, hi.x, hi.y};
      }
    }
#pragma unroll
    for (int k = 0; k < B; ++k) {
      if constexpr (F32) {
        const f32x4 fw = __builtin_bit_cast(f32x4, wv[k]), fx = __builtin_bit_cast(f32x4, xv[k]);
#pragma unroll
        for (int c = 0; c < 4; ++c) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[c], fx[c], acc, 0, 0, 0);
      } else if constexpr (DT == DT_F16) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, wv[k]), __builtin_bit_cast(f16x8, xv[k]),
                                                     acc, 0, 0, 0);
      } else {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[k]),
                                                      __builtin_bit_cast(bf16x8, xv[k]), acc, 0, 0, 0);
      }
    }
  }

  part[wave][lane] = acc;
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int w = 1; w < W; ++w) acc += part[w][lane];
  if (!ov) return;
  f32x4 o = act4(act_params(a.act), acc + bv);
  if (a.has_res) o += rv;
  Vec4IO<DT>::store(a.y, vi, o);
}

template <int DT>
hipError_t launch_dt(const ConvKsplitArgs &a, hipStream_t st) {
  const dim3 grid((a.M + 15) / 16 * a.nblk), block(64 * W);
  // the fewest batches, then the smallest
  if (a.per <= 2)
    hipLaunchKernelGGL((conv_ksplit_kernel<DT, 2>), grid, block, 0, st, a);
  else if (a.per <= 4)
    hipLaunchKernelGGL((conv_ksplit_kernel<DT, 4>), grid, block, 0, st, a);
  else
    hipLaunchKernelGGL((conv_ksplit_kernel<DT, 6>), grid, block, 0, st, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_conv_ksplit(const ConvKsplitArgs &a, int dt, hipStream_t st) {
  if (a.M == 0 || a.M > 0x0fffffffu || a.N4 == 0 || a.N4 % 4 || a.nblk != (a.N4 + 15) / 16 || a.K == 0 ||
      a.K > kConvKsplitMaxK || a.st == 0 || a.st0 > a.st || a.items != a.K * a.K * a.st || a.per == 0 ||
      (uint64_t)a.per * W < a.items || a.src_bytes[0] >= kOob || a.src_bytes[1] >= kOob || a.w_bytes >= kOob ||
      (uint64_t)((a.M + 15) / 16) * a.nblk > 0x7fffffffu)
    return hipErrorInvalidValue;
  switch (dt) {
    case DT_F32: return launch_dt<DT_F32>(a, st);
    case DT_F16: return launch_dt<DT_F16>(a, st);
    case DT_BF16: return launch_dt<DT_BF16>(a, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace aih
