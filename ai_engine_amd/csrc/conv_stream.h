// conv_stream.h -- launch interface of the conv GEMM whose operands stream
// through LDS by DMA (buffer loads straight into LDS): pointwise and KxK
// convs over one input (a plain tensor or a channel view).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "aih_device.h"

namespace aih {

struct ConvStreamArgs {
  const void *x;        // [n][IH][IW] pixels of stride_u 16-byte units
  const void *w;        // [K*K][KGP][N4][4] packed weights
  const void *bias;     // [N4]
  const void *res;      // [M][N4], or null
  void *y;              // [M][N4]
  uint32_t x_bytes;     // bytes of x (< 2 GiB)
  uint32_t w_bytes;     // bytes of w (< 2 GiB)
  uint32_t M;           // output pixels over the whole batch
  uint32_t KU;          // 16-byte units (4 fp32 / 8 16-bit channels) of one tap
  uint32_t KG, KGP;     // kg per tap, packed-weight kg per tap
  uint32_t stride_u;    // pixel stride in units
  uint32_t off_u;       // first unit of the input inside a pixel
  uint32_t N4;          // output channels padded to 4
  uint32_t nst;         // K stages of bku units: ceil(K * K * KU / bku)
  uint32_t OHW, OW, IH, IW, K, S, D;
  int32_t PT, PL;
  uint32_t mtiles, ntiles;
  int32_t act, has_res;
  uint32_t nxcd;        // XCDs of the device (workgroup remap)
  FastDiv fd_ohw, fd_ow, fd_nt;
};

// One instantiation: WM x WN wavefronts, each TM x TN blocks of 32 pixels x
// 32 channels; a tile is 32 WM TM pixels x 32 WN TN channels; nst stages of
// bku 16-byte units in flight.
struct ConvStreamShape {
  uint32_t wm, wn, tm, tn, bku, nst;
};

// Tiles for more than 64 outputs in grids of at least two a CU, and for the
// rest (the first for long sums: a KxK tap of 8 units or more, a pointwise K
// of 40).
constexpr ConvStreamShape kConvStreamWide[] = {
    {2, 2, 2, 2, 4, 2},  // 128 x 128
    {4, 1, 1, 2, 4, 3},  // 128 x 64
    {4, 1, 1, 3, 4, 3},  // 128 x 96
};
constexpr ConvStreamShape kConvStreamSmall[] = {
    {2, 2, 1, 1, 8, 2},  // 64 x 64
    {2, 2, 1, 1, 4, 3},  // 64 x 64
};

inline uint32_t conv_stream_bm(const ConvStreamShape &s) { return 32 * s.wm * s.tm; }
inline uint32_t conv_stream_bn(const ConvStreamShape &s) { return 32 * s.wn * s.tn; }

hipError_t launch_conv_stream(const ConvStreamArgs &a, int dt, const ConvStreamShape &shape, hipStream_t st);

}  // namespace aih
