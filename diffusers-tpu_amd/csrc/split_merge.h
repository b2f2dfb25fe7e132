// The merge of the tail split's parts (gfx950), shared by the attention
// kernels' launches.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "flash_common.h"

namespace dt {

// Combines the n_split parts of every split query block (the tail split):
// with M the largest m of the parts that saw keys (l > 0), weights
// w = exp2(m - M), l = sum w*l_part and o = sum w*o_part, in LSE space as
// kernels/splash.py:653-662 merges residuals; then writes the normalized
// o and/or the residual (o, M, l) exactly where the unsplit kernel would.
// D/4 lanes per row, 4 channels each; 256 / (D/4) rows per 256-thread block.
// NS bounds n_split (2, 4, 8 or 16): every part's loads are in flight at
// once, and a small bound keeps the register count, and so the occupancy
// that hides HBM latency, where the split is narrow.  A head dim p.dim below D
// has its channels in the first columns of the workspace's rows.
template <int D, int BQ, int NS>
__global__ __launch_bounds__(256) void split_merge_kernel(FlashParams p) {
  constexpr int LPR = D / 4, RPB = 256 / LPR;
  const int g = blockIdx.x * RPB + (threadIdx.x / LPR);
  const int c = 4 * (threadIdx.x % LPR);
  const int tq = g / BQ, r = g - tq * BQ;
  if (tq >= p.n_tail) return;
  const int wg = p.n_main + tq;
  const int qblk = wg % p.n_qblk;
  const int bh = wg / p.n_qblk;
  const int h = bh % p.Hq;
  const int b = bh / p.Hq;
  const int row = qblk * BQ + r;
  if (row >= p.Sq || c >= p.dim) return;
  const int64_t units = (int64_t)p.n_tail * p.n_split;
  const float* wm = p.ws + units * BQ * D;
  const float* wl = wm + units * BQ;
  const int64_t r0 = (int64_t)tq * p.n_split * BQ + r;  // part 0's row
  // Every part's m, l and o slice is requested before any is used (the
  // loop runs to NS under a uniform branch per part), so the merge pays
  // one memory latency instead of one per part.
  const int last = p.n_split - 1;
  float ms[NS], ls[NS];
  f32x4 os[NS];
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    ms[i] = 0.f;
    ls[i] = 0.f;
    os[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (i <= last) {
      const int64_t ri = r0 + (int64_t)i * BQ;
      ms[i] = wm[ri];
      ls[i] = wl[ri];
      os[i] = *(const f32x4*)(p.ws + ri * D + c);
    }
  }
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < NS; ++i)
    if (i <= last && ls[i] > 0.f) mx = fmaxf(mx, ms[i]);
  float lsum = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    const float w = (i <= last && ls[i] > 0.f) ? exp2f(ms[i] - mx) : 0.f;
    lsum += w * ls[i];
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] += w * os[i][e];
  }
  const int64_t bhrow = ((int64_t)b * p.Hq + h) * p.Sq + row;
  if (p.o32 != nullptr) {
    *(f32x4*)(p.o32 + bhrow * p.dim + c) = acc;
    if (c == 0) {
      p.m[bhrow] = lsum > 0.f ? mx : 0.f;
      p.l[bhrow] = lsum;
    }
  }
  if (p.o != nullptr) {
    const float inv = lsum > 0.f ? 1.0f / lsum : 0.f;
    u32x2 w;
    w[0] = pack_bf16x2(acc[0] * inv, acc[1] * inv);
    w[1] = pack_bf16x2(acc[2] * inv, acc[3] * inv);
    *(u32x2*)(p.o + b * p.o_sb + h * p.o_sh + (int64_t)row * p.o_ss + c) = w;
  }
}

template <int D, int BQ>
void launch_split_merge(const FlashParams& p, hipStream_t st) {
  const dim3 mg(p.n_tail * (BQ / (256 / (D / 4))));
  if (p.n_split <= 2)
    hipLaunchKernelGGL((split_merge_kernel<D, BQ, 2>), mg, dim3(256), 0, st, p);
  else if (p.n_split <= 4)
    hipLaunchKernelGGL((split_merge_kernel<D, BQ, 4>), mg, dim3(256), 0, st, p);
  else if (p.n_split <= 8)
    hipLaunchKernelGGL((split_merge_kernel<D, BQ, 8>), mg, dim3(256), 0, st, p);
  else
    hipLaunchKernelGGL((split_merge_kernel<D, BQ, kMaxSplit>), mg, dim3(256), 0,
                       st, p);
}

}  // namespace dt
