// Launches of flash_attn_kernel at head dims below 128 that are not 64
// (multiples of 8; kernels/splash.py:156-160 accepts every one).
//
// The rows are read and written as they are in memory, with no zero-padded
// copies of q, k and v and no copy of the output, and the MFMAs cover the
// dim rounded up to 16 channels (QK) and 32 (PV) instead of the whole 64 or
// 128.
#include "flash_attn_kernel.h"

namespace dt {

int launch_flash_ragged(const FlashParams& p, const LaunchShape& shape,
                        hipStream_t st) {
  if (p.dim <= 48) return launch_dense<HeadDim<64, 3, true>, false>(p, shape, st);
  if (p.dim < 64) return launch_dense<HeadDim<64, 4, true>, false>(p, shape, st);
  if (p.dim <= 80) return launch_dense<HeadDim<128, 5, true>, false>(p, shape, st);
  if (p.dim <= 96) return launch_dense<HeadDim<128, 6, true>, false>(p, shape, st);
  if (p.dim <= 112) return launch_dense<HeadDim<128, 7, true>, false>(p, shape, st);
  return launch_dense<HeadDim<128, 8, true>, false>(p, shape, st);
}

}  // namespace dt
