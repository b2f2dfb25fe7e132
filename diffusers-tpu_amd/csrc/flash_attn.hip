// Launches of flash_attn_kernel at head dims 128 and 64, the tail-split plan
// and the choice of workgroup shape (kernel: flash_attn_kernel.h; head dims
// in between: flash_dims.hip).
#include "flash_attn_kernel.h"

namespace dt {

SplitPlan split_plan(int64_t n_wg, int ntiles, int n_cu, int D, int bq,
                     size_t max_ws) {
  SplitPlan sp{1, 0, (int)n_wg, 0};
  if (n_cu <= 0 || n_wg <= 0) return sp;
  const int64_t rem = n_wg % n_cu;
  if (rem == 0) return sp;
  // Short sweeps over many rounds: the idle CUs of the last one are a few
  // percent of the call at most, and the split's second launch costs as much.
  // (It decides for E4M3 keys, tile tables and dims above 128: bf16 calls of so
  // few tiles run 128-row workgroups.)  E4M3, H40 Sq 15000, 9.2 rounds, whole
  // against split, us: 8 tiles 164.3, 169.5 in 2; 12 tiles 217.1, 217.0 in 3; 16
  // tiles 265.4, 270.8 in 4; past the line 17 tiles 282.0, 283.2, 24 tiles
  // 367.6, 370.1.  At 4.9 to 29.5 rounds of other fillings nothing would split.
  if (ntiles <= 16 && n_wg >= 8 * (int64_t)n_cu) return sp;
  // The last round's rem query blocks cut into ns parts run as
  // ceil(rem * ns / n_cu) rounds of parts of ntiles / ns tiles; each
  // workgroup also pays a start-up (q load, the first tiles' latency, the
  // epilogue) of about kStartTiles tiles, and the merge reads every part
  // (about kMergeTiles per part).  Pick the ns (at most 16, at least two
  // tiles per part, workspace at most max_ws and 512 MiB) with the shortest
  // tail.
  constexpr int64_t kStartTiles = 8;  // fitted: I1 with 5 parts ran 3.8 % slower than with 2
  constexpr int64_t kMergeTiles = 1;  // fitted: P (16 tiles) 17.4 us at 4 parts, 19.8 at 8
  constexpr size_t kMaxWs = size_t(512) << 20;
  if (max_ws > kMaxWs) max_ws = kMaxWs;
  const size_t unit_bytes = (size_t)bq * (D + 2) * sizeof(float);
  // Above head dim 128 (bq 128) a tile is 32 keys and short, so a split costs
  // more of them: 6 tiles for the merge's launch, 11 for writing and reading
  // 256 parts' outputs, and 15 % a tile when all CUs are busy instead of few.
  // Measured, whole against split (us): D = 256, 128 blocks of 14 tiles 24.6,
  // 32.5 in 2, of 32 tiles 38.7, 42.2, of 64 tiles 63.7, 61.2; 64 blocks of 14
  // tiles 24.1, 25.7, of 32 tiles 37.8, 31.3 in 3; D = 160, 128 blocks of 14
  // tiles 19.1, 25.3, of 64 tiles 53.3, 43.3.
  const bool wide = bq == 128;
  auto cost_of = [&](int64_t ns) -> double {
    const int64_t units = rem * ns, rounds = (units + n_cu - 1) / n_cu;
    const double tiles = (double)((ntiles + ns - 1) / ns);
    if (!wide)
      return (double)rounds * (tiles + kStartTiles) +
             (double)(ns > 1 ? ns * kMergeTiles : 0);
    const double busy = units < n_cu ? (double)units / n_cu : 1.0;
    return (double)rounds * (tiles * (1 + 0.15 * busy) + 2 * kStartTiles) +
           (ns > 1 ? 6 + 11 * (double)units / n_cu : 0.0);
  };
  int64_t best_ns = 1;
  double best_cost = cost_of(1);
  for (int64_t ns = 2; ns <= kMaxSplit && ns <= ntiles / 2; ++ns) {
    if ((size_t)(rem * ns) * unit_bytes > max_ws) break;
    const double cost = cost_of(ns);
    if (cost < best_cost) {
      best_cost = cost;
      best_ns = ns;
    }
  }
  if (best_ns < 2) return sp;
  sp.n_split = (int)best_ns;
  sp.n_tail = (int)rem;
  sp.n_main = (int)(n_wg - rem);
  sp.ws_bytes = (size_t)(rem * best_ns) * unit_bytes;
  return sp;
}

// The CU count of the current device, queried once per device (every
// planned call asks for it).
int device_cu_count(int* n_cu) {
  constexpr int kMaxDev = 64;
  static std::atomic<int> cache[kMaxDev];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess)
    return set_error(DT_ERR_LAUNCH, "dt_flash_fwd: no current device");
  if (dev >= 0 && dev < kMaxDev) {
    const int c = cache[dev].load(std::memory_order_relaxed);
    if (c > 0) {
      *n_cu = c;
      return DT_OK;
    }
  }
  if (hipDeviceGetAttribute(n_cu, hipDeviceAttributeMultiprocessorCount,
                            dev) != hipSuccess)
    return set_error(DT_ERR_LAUNCH, "dt_flash_fwd: CU count query failed");
  if (dev >= 0 && dev < kMaxDev && *n_cu > 0)
    cache[dev].store(*n_cu, std::memory_order_relaxed);
  return DT_OK;
}

// Workgroup shape of a dense bf16 launch: R row wavefronts
// (32 query rows each) times G key groups.  8 x 1 is the shape for long
// sweeps and full grids.  With few query blocks or few key tiles a
// workgroup's start-up, the tail split's second launch and the idle CUs cost
// more than the tile DMA that smaller row blocks repeat:
//   4 x 1  128 rows; one wavefront per SIMD, two workgroups per CU, one
//          computing while the other starts or ends;
//   4 x 2  128 rows, the tiles dealt to two key groups merged in LDS;
//   2 x 4  64 rows, four key groups (head dim 64: four rings fit the LDS).
// The estimate below is microseconds on one MI355X, fitted to N(0,1) calls
// captured in a graph (start-up and gap to the next launch included): `own`
// a lone workgroup per CU, `shared` two per CU, for a sweep of T tiles.
// Measured, D = 128, before (8 x 1 and its split) -> chosen: H8 S512
// 17.0 -> 12.4 us, H24 S512 22.3 -> 12.9, H24 S1024 30.4 -> 21.2, H8 S2048
// 33.6 -> 29.6, H96 S1024 70.1 -> 57.5; kept 8 x 1: H2 S4096 (split 10 ways)
// 33.8 against 49.5, H24 S2048 52.4 against 57.6.  D = 64: H8 S1024
// 16.3 -> 10.6, H16 S2048 29.7 -> 24.6, kept H8 S4096 44.9 against 47.0.
// Dims in between take the constants of their width, D = 64 or 128.  All
// shapes forced at 15 sizes around the lines (2 to 48 heads, 512 to 4096 rows),
// the chosen against the fastest: D = 128 0.2 % slower on average and 2.2 % at
// most, 104 0.2 and 2.1, 72 1.2 and 5.9 (H8 S1024: 17.3 us in 4 x 1, 16.3 in 4
// x 2), 64 0.1 and 0.9, 40 0.3 and 4.8 (B2 H24 S700: 16.1 in 4 x 1, 15.4 in 8 x
// 1).
struct RowShape {
  int r, g;
};
// `sp`: the split that 8 x 1 would take.  `key_groups`: whether the tiles may
// be dealt to key groups.
static RowShape row_shape(int64_t heads, int Sq, int kv_end, int D,
                          const SplitPlan& sp, bool key_groups, int n_cu) {
  const double T = (kv_end + kBKV - 1) / kBKV;
  auto blocks = [&](int rows) { return heads * ((Sq + rows - 1) / rows); };
  const bool d64 = D == 64;
  // 8 x 1: whole rounds, then the last one (split or not)
  const double whole = d64 ? 8 + 0.95 * T : 9 + 1.6 * T;
  const int64_t n8 = blocks(256);
  double best;
  if (sp.n_split > 1) {
    const int64_t tail_rounds =
        ((int64_t)sp.n_tail * sp.n_split + n_cu - 1) / n_cu;
    best = (double)(sp.n_main / n_cu) * whole +
           (double)tail_rounds * ((d64 ? 0.95 : 1.6) * T / sp.n_split) +
           (d64 ? 16 : 20);
  } else {
    best = (double)((n8 + n_cu - 1) / n_cu) * (n8 <= n_cu ? 0.9 : 1.0) * whole;
  }
  RowShape shape{8, 1};
  auto consider = [&](double cost, int r, int g) {
    if (cost < best) {
      best = cost;
      shape = RowShape{r, g};
    }
  };
  const int64_t n4 = blocks(128), per_cu = (n4 + n_cu - 1) / n_cu;
  const double own = d64 ? 4.5 + 0.65 * T : 5.6 + 0.83 * T;
  const double shared = d64 ? 4.5 + 1.07 * T : 5.6 + 1.75 * T;
  consider((double)(per_cu / 2) * shared + (double)(per_cu % 2) * own, 4, 1);
  if (!key_groups) return shape;
  if (n4 <= n_cu) consider(d64 ? 6.0 + 0.46 * T : 7.5 + 0.72 * T, 4, 2);
  if (d64 && blocks(64) <= n_cu) consider(6.5 + 0.26 * T, 2, 4);
  return shape;
}

LaunchShape launch_shape(int B, int Hq, int Sq, int kv_end, int dim,
                         LaunchForm form, size_t ws_bytes, int n_cu) {
  const int D = kernel_dim(dim);
  // (above head dim 128: 4 wavefronts, 32-key tiles)
  const int bq = D == 256 ? 128 : kBQ, bkv = D == 256 ? 32 : kBKV;
  const int64_t heads = (int64_t)B * Hq;
  const int64_t n_wg = heads * ((Sq + bq - 1) / bq);
  const int ntiles = (kv_end + bkv - 1) / bkv;
  if (D == 256) return {4, 1, split_plan(n_wg, ntiles, n_cu, D, bq, ws_bytes)};
  auto shaped = [&](const SplitPlan& sp, bool key_groups) {
    const RowShape w = row_shape(heads, Sq, kv_end, D, sp, key_groups, n_cu);
    if (w.r == 8) return LaunchShape{8, 1, sp};
    const int64_t blocks = heads * ((Sq + 32 * w.r - 1) / (32 * w.r));
    return LaunchShape{w.r, w.g, SplitPlan{1, 0, (int)blocks, w.g > 1 ? kGroupsWs : 0}};
  };
  if (form == LaunchForm::kDense) {
    // (the best of all, where the workspace allows it: a caller who gives what
    // the query says gets it)
    const LaunchShape best =
        shaped(split_plan(n_wg, ntiles, n_cu, D, bq), true);
    if (best.split.ws_bytes <= ws_bytes) return best;
  }
  const SplitPlan sp = split_plan(n_wg, ntiles, n_cu, D, bq, ws_bytes);
  if (form == LaunchForm::kTiles) return {8, 1, sp};
  return shaped(sp, ws_bytes >= kGroupsWs);
}

template <bool QK8, bool SPARSE>
static int launch_d128_v(const FlashParams& p, hipStream_t st) {
  return p.vt != nullptr ? launch_flash<FullDim<128>, QK8, SPARSE, true, 8, 1>(p, st)
                         : launch_flash<FullDim<128>, QK8, SPARSE, false, 8, 1>(p, st);
}

int launch_flash_attn(const FlashParams& p, int D, const LaunchShape& shape,
                      hipStream_t st) {
  if (D == 64) {
    if (p.k8 != nullptr || p.vt != nullptr || p.tile_span != nullptr)
      return set_error(DT_ERR_UNSUPPORTED,
                       "dt_flash_fwd: head dim 64 takes bf16 keys, row-major "
                       "V and no tile table");
    return launch_dense<FullDim<64>, false>(p, shape, st);
  }
  const bool sparse = p.tile_span != nullptr;
  if (p.k8 != nullptr)
    return sparse ? launch_d128_v<true, true>(p, st)
                  : launch_d128_v<true, false>(p, st);
  if (sparse) return launch_d128_v<false, true>(p, st);
  // (packed and row-major V take the same shape: their results are equal
  // bit for bit)
  return p.vt != nullptr ? launch_dense<FullDim<128>, true>(p, shape, st)
                         : launch_dense<FullDim<128>, false>(p, shape, st);
}

}  // namespace dt
