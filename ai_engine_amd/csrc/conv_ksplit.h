// conv_ksplit.h -- launch interface of the KxK conv for few output pixels
// whose K runs over the wavefronts of a workgroup.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "aih_device.h"

namespace aih {

struct ConvKsplitArgs {
  const void *src[2];     // input parts (one for a plain input)
  uint32_t src_bytes[2];  // bytes of each part's buffer (< 2 GiB)
  uint32_t stride_u[2];   // pixel stride of each part, in 16-byte units
  uint32_t off_u[2];      // first unit of each part inside its pixel
  uint32_t nu[2];         // 16-byte units of each part per pixel
  uint32_t kg_first[2];   // first kg (of the packed weights) of each part
  uint32_t st0, st;       // K steps of 4 units per tap: of part 0, of all parts
  const void *w;          // packed [K*K][KGP][N4][4]
  uint32_t w_bytes;       // bytes of w (< 2 GiB)
  const void *bias;       // [N4]
  const void *res;        // like y, or null
  void *y;                // [M][N4]
  uint32_t KGP, N4;
  uint32_t M, OHW, OW, IH, IW, K, S, D;
  int32_t PT, PL;
  uint32_t items, per;    // (tap, step) pairs: K*K*st, and of one wavefront
  uint32_t nblk;          // 16-channel blocks
  int32_t act, has_res;
  uint32_t nxcd;          // XCDs of the device (workgroup remap)
  FastDiv fd_ohw, fd_ow, fd_nblk, fd_st, fd_k;
};

constexpr uint32_t kConvKsplitWaves = 9;  // a 3x3's taps
constexpr uint32_t kConvKsplitMaxK = 15;

hipError_t launch_conv_ksplit(const ConvKsplitArgs &a, int dt, hipStream_t st);

}  // namespace aih
