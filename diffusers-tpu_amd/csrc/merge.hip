// LSE-space merge of residual (o, m, l) triples from key shards (gfx950): the
// merge an outer ring loop performs on the outputs of residual_attention
// (kernels/splash.py:653-664).
//
//   M = max m_i,  out = sum 2^(m_i - M) o_i / sum 2^(m_i - M) l_i
//
// HBM-bound: every part's o is read once and the result written once, D/4
// lanes per row with 16 bytes of each part each, all parts' loads in flight
// before any is used.  Measured on two parts of 94,500 x 128 (146 MB): 22 to
// 27 us by box, 5.4 to 6.6 TB/s, against about 185 us for the same formula as 19
// torch operations, each a pass over memory.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "../../include/dt_attention.h"
#include "dt_common.h"

namespace dt {
namespace {

constexpr int kThreads = 256;

struct MergeParams {
  const float* o[DT_MERGE_MAX_PARTS];
  const float* m[DT_MERGE_MAX_PARTS];
  const float* l[DT_MERGE_MAX_PARTS];
  float* out;
  int64_t n4;  // rows * D / 4
  int lpr;     // D / 4
  int parts;
};

// NP bounds `parts` (2, 4, 8, 16): the loads of all of them are in flight
// at once, and a small bound keeps the registers, and so the occupancy.
template <int NP>
__global__ __launch_bounds__(kThreads) void merge_kernel(MergeParams p) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= p.n4) return;
  const int64_t row = i / p.lpr;
  float m[NP], l[NP];
  f32x4 o[NP];
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    if (j < p.parts) {
      m[j] = p.m[j][row];
      l[j] = p.l[j][row];
      o[j] = *(const f32x4*)(p.o[j] + 4 * i);
    }
  }
  float mx = m[0];
#pragma unroll
  for (int j = 1; j < NP; ++j)
    if (j < p.parts) mx = fmaxf(mx, m[j]);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  float ls = 0.f;
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    if (j < p.parts) {
      const float w = exp2f(m[j] - mx);  // (a NaN m makes its row NaN)
      ls += w * l[j];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += w * o[j][e];
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = acc[e] / ls;
  __builtin_nontemporal_store(acc, (f32x4*)(p.out + 4 * i));
}

}  // namespace
}  // namespace dt

extern "C" int dt_merge_residuals(const float* const* o, const float* const* m,
                                  const float* const* l, int parts,
                                  int64_t rows, int D, float* out,
                                  void* stream) {
  using namespace dt;
  const char* who = "dt_merge_residuals";
  if (!o || !m || !l || !out) return set_error(DT_ERR_ARG, "%s: null pointer argument", who);
  if (parts < 1 || parts > DT_MERGE_MAX_PARTS)
    return set_error(DT_ERR_ARG, "%s: %d parts (1 to %d)", who, parts,
                     DT_MERGE_MAX_PARTS);
  if (rows <= 0 || D <= 0)
    return set_error(DT_ERR_SHAPE, "%s: rows=%lld D=%d", who, (long long)rows, D);
  if (D % 4)
    return set_error(DT_ERR_UNSUPPORTED, "%s: D %d not a multiple of 4", who, D);
  MergeParams p{};
  for (int i = 0; i < parts; ++i) {
    if (!o[i] || !m[i] || !l[i])
      return set_error(DT_ERR_ARG, "%s: null pointer in part %d", who, i);
    if ((uintptr_t)o[i] & 15u)
      return set_error(DT_ERR_UNSUPPORTED, "%s: misaligned o in part %d", who, i);
    p.o[i] = o[i];
    p.m[i] = m[i];
    p.l[i] = l[i];
  }
  if ((uintptr_t)out & 15u)
    return set_error(DT_ERR_UNSUPPORTED, "%s: misaligned output", who);
  p.out = out;
  p.lpr = D / 4;
  p.n4 = rows * (D / 4);
  p.parts = parts;
  const int64_t blocks = (p.n4 + kThreads - 1) / kThreads;
  if (blocks > 0x7fffffff)
    return set_error(DT_ERR_SHAPE, "%s: too many rows", who);
  const dim3 grid((unsigned)blocks);
  hipStream_t st = (hipStream_t)stream;
  if (parts <= 2)
    hipLaunchKernelGGL(merge_kernel<2>, grid, dim3(kThreads), 0, st, p);
  else if (parts <= 4)
    hipLaunchKernelGGL(merge_kernel<4>, grid, dim3(kThreads), 0, st, p);
  else if (parts <= 8)
    hipLaunchKernelGGL(merge_kernel<8>, grid, dim3(kThreads), 0, st, p);
  else
    hipLaunchKernelGGL(merge_kernel<DT_MERGE_MAX_PARTS>, grid, dim3(kThreads),
                       0, st, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    return set_error(DT_ERR_LAUNCH, "%s: %s", who, hipGetErrorString(e));
  return DT_OK;
}
