// The fp32 form of a prompt's row-gathered, expert-grouped linears: split products on the bf16 matrix cores
// (kernels/gemm_f32x3.h) with the epilogues of a row linear. Us, exact-f32 MFMA tiles (lr_gemm_kernel) -> here, rows x K x N:
// 16 x 2048 x 8224 91 -> 29; 400 x 5632 x 2048 363 -> 74; 400 x 2048 x 5632 gated 246 -> 136. Relative error against 64 bits,
// 400 x 5632 x 2048: 1.35e-6 -> 1.4e-7 (K split).
#include "../kernels/gemm_f32x3.h"
#include "hy_util.h"
#include "hybrid.h"
#include "row_act.h"

namespace jla {

template <int MT, int GATED, bool SCALED>
__global__ void __launch_bounds__(64 * MT, 2) rows_f32x3_kernel(F3Rows p, RowLinear act, int tiles_n) {
  __shared__ u32x4 lds[f3_lds<MT>()];
  f3_tile<MT, GATED, SCALED>(p, tiles_n, 0, (p.K + F3_BK - 1) / F3_BK, lds, [&](const f32x4 g, const f32x4 u) {
    f32x4 v = g;
    if (act.act != HY_ACT_NONE) {
#pragma unroll
      for (int x = 0; x < 4; ++x) v[x] = lr_act(act, g[x], u[x]);
    }
    return v;
  });
}

// K over gridDim.y workgroups per tile: partial sums of every weight row (gate and up side by side) into their slabs
template <int MT, bool SCALED>
__global__ void __launch_bounds__(64 * MT, 2) rows_f32x3_split_kernel(F3Rows p, int tiles_n, int steps) {
  __shared__ u32x4 lds[f3_lds<MT>()];
  const int t0 = blockIdx.y * steps;
  p.out += (size_t)blockIdx.y * p.R * p.ldo;
  f3_tile<MT, 0, SCALED>(p, tiles_n, t0, min(t0 + steps, (p.K + F3_BK - 1) / F3_BK), lds,
                 [](const f32x4 g, const f32x4) { return g; });
}

// the slabs added in order, and the epilogue; one thread per 4 output columns
__global__ void __launch_bounds__(256) rows_f32_sum_kernel(RowLinear p, const float* slabs, int splits, int gated) {
  const int quads = p.N / 4;
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long long)p.R * quads) return;
  const int r = (int)(i / quads), col = 4 * (int)(i - (long long)r * quads);
  if (p.offs && r >= p.offs[p.E]) return;  // (rows of experts without weights)
  const int nw = gated ? 2 * p.N : p.N;
  const float* at = slabs + (size_t)r * nw + col;
  f32x4 g = *reinterpret_cast<const f32x4*>(at), u = g;
  if (gated) u = *reinterpret_cast<const f32x4*>(at + p.N);
  for (int s = 1; s < splits; ++s) {
    const float* more = at + (size_t)s * p.R * nw;
    g += *reinterpret_cast<const f32x4*>(more);
    if (gated) u += *reinterpret_cast<const f32x4*>(more + p.N);
  }
  f32x4* o = reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.out) + (size_t)(p.dst_idx ? p.dst_idx[r] : r) * p.ldo + col);
  f32x4 v;
#pragma unroll
  for (int x = 0; x < 4; ++x) v[x] = lr_act(p, g[x], u[x]);
  *o = p.add_out ? *o + v : v;
}

// A K of a few steps is over before the pipeline is filled: 64 x 2048 x K 64 6.6 us on lr_gemm_kernel's tiles, 7.2 here; 130 rows of
// K 256 | 384 13.2 | 17.5, 15.0 | 19.7 here (K 512, cut in two: 23.5, 18.6). From 256 rows per expert on those tiles are of 128
// rows and it turns earlier: 300 rows of K 256 20.7, 16.6 here.
constexpr int RF_MIN_K = 512, RF_MIN_K_MANY = 256, RF_MANY_ROWS = 256;

bool hy_rows_f32_takes(const RowLinear& p) {
  auto aligned = [](const void* x) { return ((uintptr_t)x & 15) == 0; };
  return !p.wbf16 && !p.a_bf16 && !p.out_bf16 && !p.a_norm_w && (p.offs || p.E == 1) && p.K % 8 == 0 &&
         p.K >= (p.R / (p.offs ? p.E : 1) >= RF_MANY_ROWS ? RF_MIN_K_MANY : RF_MIN_K) && p.lda % 4 == 0 &&
         p.N % 4 == 0 && p.ldo % 4 == 0 && p.w_stride % 4 == 0 && aligned(p.a) && aligned(p.w) && aligned(p.out);
}

static F3Plan rows_f32_plan(const RowLinear& p) {
  const int E = p.offs ? p.E : 1;
  auto tiles = [&](int bm) {  // (experts: on average, at least one each while there are rows)
    if (E == 1) return (p.R + bm - 1LL) / bm;
    const long long mean = (p.R + bm / 2LL * E) / bm, least = E < p.R ? E : p.R;
    return mean > least ? mean : least;
  };
  return f3_plan(tiles, p.R, (hy_act_gated(p.act) ? 2LL : 1LL) * p.N, p.K, E < p.R ? E : p.R);
}

long long hy_rows_f32_floats(const RowLinear& p) {
  const F3Plan pl = rows_f32_plan(p);
  return pl.splits > 1 ? (long long)pl.splits * p.R * (hy_act_gated(p.act) ? 2 : 1) * p.N : 0;
}

int hy_rows_f32(const RowLinear& p, float* ws, hipStream_t s) {
  const int gated = hy_act_gated(p.act), E = p.offs ? p.E : 1;
  const F3Plan pl = rows_f32_plan(p);
  F3Rows f{reinterpret_cast<const float*>(p.a), p.lda, p.a_idx, p.a_scale, reinterpret_cast<const float*>(p.w),
           p.w_stride, p.N, p.K, reinterpret_cast<float*>(p.out), p.ldo, p.dst_idx, p.add_out, p.offs, p.E, p.R};
  const long long tn = ((gated ? 2LL : 1LL) * p.N + pl.bn - 1) / pl.bn;
  // (experts: every one's last tile may be ragged. One matrix has as many tiles as it has: workgroups without a tile, between the K
  // splits of the others, put two of those on one compute unit: 256 x 2048 x 5632 67 -> 49 us, 128 x 4096 x 4096 51 -> 40)
  const long long row_tiles = p.offs ? p.R / pl.bm + (long long)E : (p.R + pl.bm - 1LL) / pl.bm;
  const long long grid = (row_tiles * tn + 7) / 8 * 8;
  if (grid > 0x7fffffffLL) return -4;
  if (pl.splits > 1) {
    if (!ws || ((uintptr_t)ws & 15)) return -12;
    f.N = f.ldo = gated ? 2 * p.N : p.N;
    f.out = ws;
    f.dst_idx = nullptr;
    f.add = 0;
    const dim3 g((unsigned)grid, pl.splits);
#define RF_SPLIT(MT, SC) rows_f32x3_split_kernel<MT, SC><<<g, 64 * MT, 0, s>>>(f, (int)tn, pl.steps)
    if (pl.bm == 64) {
      if (f.a_scale) RF_SPLIT(4, true);
      else RF_SPLIT(4, false);
    } else {
      if (f.a_scale) RF_SPLIT(8, true);
      else RF_SPLIT(8, false);
    }
#undef RF_SPLIT
    JLA_CHECK_LAUNCH();
    const long long n = (long long)p.R * (p.N / 4);
    rows_f32_sum_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(p, ws, pl.splits, gated);
    JLA_CHECK_LAUNCH();
    return 0;
  }
#define RF_RUN(MT, G)                                                                                     \
  do {                                                                                                    \
    if (f.a_scale) rows_f32x3_kernel<MT, G, true><<<(unsigned)grid, 64 * MT, 0, s>>>(f, p, (int)tn);       \
    else rows_f32x3_kernel<MT, G, false><<<(unsigned)grid, 64 * MT, 0, s>>>(f, p, (int)tn);                \
  } while (0)
  if (pl.bm == 64) {
    if (gated) RF_RUN(4, 1);
    else RF_RUN(4, 0);
  } else {
    if (gated) RF_RUN(8, 1);
    else RF_RUN(8, 0);
  }
#undef RF_RUN
  JLA_CHECK_LAUNCH();
  return 0;
}

}  // namespace jla
