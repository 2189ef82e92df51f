// Some ten to a few hundred rows on row-major bf16 weights: out[dst(r), :] = act(A[src(r), :] @ W[expert(r)]^T), dense or with some
// rows per expert, the rows bf16 or fp32 (rounded as a fragment is read). kernels/mid_tile.h says what bounds it and why the tile is
// as it is; here are its forms, the choice among them, and the epilogue.
// Us, weights in no cache, 16 | 64 | 100 | 200 fp32 rows, the forms before (rows_gemv.hip to 64 rows, lr_gemm_kernel's tiles) -> here, from 65 rows
// on with the rounding of the rows: 2048 x 2048 8.7 | 23.5 | 41 | 39 -> 7.7 | 12.3 | 11.7 | 13.1 (bf16 rows 6.4 | 7.9 | 9.5 | 10.3); 2048 x 5632 19.9 | 55 | 154 |
// 144 -> 13.1 | 16.1 | 19.9 | 24; 4096 x 4096 16.5 | 42 | 107 | 95 -> 13.2 | 17.3 | 21 | 28; 4096 x 14336 50 | 132 | 376 | 354 -> 29 | 33 | 40 | 53. A mixture
// of 8 experts of 2816 x 2048 (7168 x 4096), two per token, both products, 33 | 100 | 256 tokens: 165 | 172 | 133 -> 77 | 80 | 88 (452 | 473 | 425 ->
// 257 | 289 | 297; its weights 237 at 5.95 TB/s).
#include "../kernels/mid_tile.h"
#include "../kernels/row_tiles.h"
#include "hy_util.h"
#include "hybrid.h"
#include "row_act.h"

namespace jla {

JLA_DEV void rm_store(const RowLinear& p, int d, int col, f32x4 v) {
  if (p.out_bf16) {
    *reinterpret_cast<u32x2*>(reinterpret_cast<bf16_t*>(p.out) + (size_t)d * p.ldo + col) = u32x2{pack2bf(v[0], v[1]), pack2bf(v[2], v[3])};
  } else {
    f32x4* o = reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.out) + (size_t)d * p.ldo + col);
    *o = p.add_out ? *o + v : v;
  }
}

// grid: tiles x splits, rounded up to 8; slabs (several splits): [splits][R][weight rows] partial sums instead of the output.
// gated: the 16-column tiles of a wave are gate and up tiles in turn (NT even).
template <int MT, int NT, int WN, int WK, int S, int XB, bool WIDE>
__global__ void __launch_bounds__(64 * WN * WK, (MidShape<MT, NT, WN, WK, S, XB>::PER_SIMD)) rows_mid_kernel(RowLinear p, int gated, int tiles_n, int splits, int steps, float* slabs) {
  using H = MidShape<MT, NT, WN, WK, S, XB>;
  __shared__ u32x4 lds[H::LDS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, q = lane >> 4;
  int e = 0, r0 = 0, rend = 0, tn = 0, split = 0;
  if (!row_tile<H::BM>(p.offs, p.E, p.R, tiles_n, lane, e, r0, rend, tn, splits, split)) return;
  const int K = p.K, N = p.N, t0 = split * steps, t1 = min(K >> 6, t0 + steps);
  const int n0 = tn * (gated ? H::BN / 2 : H::BN);
  const char* const wbase = reinterpret_cast<const char*>(reinterpret_cast<const bf16_t*>(p.w) + (size_t)e * p.w_stride);
  auto xrow = [&](int r) {  // (rows past the end repeat the last one)
    const int row = min(r0 + r, rend - 1);
    return reinterpret_cast<const char*>(p.a) + (size_t)(p.a_idx ? p.a_idx[row] : row) * p.lda * XB;
  };
  auto wrow = [&](int r) {
    const int j = r >> 4, col = min(n0 + (gated ? 16 * (j >> 1) + (r & 15) : r), N - 1);
    return wbase + (size_t)(gated && (j & 1) ? N + col : col) * K * 2;
  };
  f32x4 acc[NT][MT];
  float none[1];
  mid_tile<MT, NT, WN, WK, S, XB, false, false, std::conditional_t<WIDE, f64x4, void>>(lds, xrow, wrow, t0, t1, acc, none, p.offs ? 2 : 4);
  if (wave >= WN) return;
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int row = r0 + 16 * m + c;
    if (row >= rend) continue;
    const int d = slabs ? row : (p.dst_idx ? p.dst_idx[row] : row);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int j = wave * NT + t, col = n0 + 16 * (gated ? j >> 1 : j) + 4 * q;
      if (col >= N) continue;
      if (slabs) {
        const int nw = gated ? 2 * N : N;
        *reinterpret_cast<f32x4*>(slabs + ((size_t)split * p.R + row) * nw + (gated && (t & 1) ? N : 0) + col) = acc[t][m];
      } else if (!gated || !(t & 1)) {
        f32x4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = lr_act(p, acc[t][m][i], gated ? acc[t + 1 < NT ? t + 1 : t][m][i] : 0.f);
        rm_store(p, d, col, v);
      }
    }
  }
}

__global__ void __launch_bounds__(256) rows_mid_sum_kernel(RowLinear p, const float* __restrict__ ws, int splits, int gated) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  const int n4 = p.N / 4;
  const long long r = i / n4;
  if (r >= p.R || (p.offs && r >= p.offs[p.E])) return;  // (rows of experts without weights: nothing wrote their sums)
  const int col = 4 * (int)(i - r * n4), nw = gated ? 2 * p.N : p.N;
  const float* at = ws + r * nw + col;
  auto sum = [&](const float* from) {  // in 64 bits, four loads in flight
    double t[4] = {};
    for (int s0 = 0; s0 < splits; s0 += 4) {
      f32x4 f[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) f[j] = *reinterpret_cast<const f32x4*>(from + (size_t)min(s0 + j, splits - 1) * p.R * nw);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int x = 0; x < 4; ++x) t[x] += s0 + j < splits ? (double)f[j][x] : 0.;
    }
    return f32x4{(float)t[0], (float)t[1], (float)t[2], (float)t[3]};
  };
  const f32x4 g = sum(at), u = gated ? sum(at + p.N) : g;
  f32x4 v;
#pragma unroll
  for (int x = 0; x < 4; ++x) v[x] = lr_act(p, g[x], u[x]);
  rm_store(p, p.dst_idx ? p.dst_idx[r] : (int)r, col, v);
}

struct RmForm {  // (mid_plan)
  int mt, nt, wn, wk, xb;
  float fill, stage, more, sum, mb;
  void (*run)(unsigned, hipStream_t, const RowLinear&, int, int, int, int, float*);
};
// Up to RM_WIDE_SUM_ROWS rows are summed in 64 bits (WIDE), rows by expert every four products as rows_gemv.hip sums them, dense rows, which
// have one fp32 chain per wave there, every eight (every four: up to 3 % slower); more rows had one chain over K on the tiles of before,
// too. Relative errors against 64 bits, one chain | wide: dense, K 2048 2.7e-7 | 8.9e-8, K 14336 3.7e-7 | 9.2e-8; by expert, K 7168 5.3e-7 | 6.5e-8
// (rows_gemv.hip 1.3e-7 dense, 7.0e-8). Us, one chain -> wide, weights in no cache, 16 | 33 | 64 rows: 2048 x 2048 7.6 | 10.2 | 12.3 -> 7.7 | 10.7 | 12.5,
// bf16 rows 6.4 | 7.4 | 7.9 -> 6.5 | 7.5 | 8.0; 4096 x 4096 13.1 | 15.5 | 16.5 -> 13.2 | 16.4 | 17.3; 4096 x 14336 29.1 | 29.8 | 32.5 -> 28.9 | 30.1 | 32.8; 64 rows of
// 8 experts of 4096 x 7168 88 -> 91.
constexpr int RM_WIDE_SUM_ROWS = 64;
template <int MT, int NT, int WN, int WK, int S, int XB>
static void rm_launch(unsigned grid, hipStream_t s, const RowLinear& p, int gated, int tiles_n, int splits, int steps, float* slabs) {
  if constexpr (16 * MT <= RM_WIDE_SUM_ROWS) {
    if (p.R <= RM_WIDE_SUM_ROWS) {
      rows_mid_kernel<MT, NT, WN, WK, S, XB, true><<<grid, 64 * WN * WK, 0, s>>>(p, gated, tiles_n, splits, steps, slabs);
      return;
    }
  }
  rows_mid_kernel<MT, NT, WN, WK, S, XB, false><<<grid, 64 * WN * WK, 0, s>>>(p, gated, tiles_n, splits, steps, slabs);
}
#define RM_FORM(MT, NT, WN, WK, S, XB, ...) {MT, NT, WN, WK, XB, __VA_ARGS__, rm_launch<MT, NT, WN, WK, S, XB>}
static const RmForm RM_FORMS[] = {
    RM_FORM(1, 1, 1, 4, 4, 2, 3.83f, 0.416f, 0.231f, 1.64f, 1.0f), RM_FORM(1, 1, 4, 1, 8, 2, 2.99f, 0.214f, 0.768f, 2.94f, 0.395f),
    RM_FORM(1, 2, 4, 1, 8, 2, 3.36f, 0.352f, 1.03f, 2.77f, 0.753f), RM_FORM(2, 1, 1, 4, 3, 2, 3.92f, 0.73f, 0.1f, 1.23f, 0.926f),
    RM_FORM(2, 1, 4, 1, 6, 2, 3.69f, 0.225f, 0.851f, 2.55f, 0.284f), RM_FORM(2, 2, 4, 1, 6, 2, 4.93f, 0.352f, 1.2f, 1.54f, 0.474f),
    RM_FORM(4, 1, 4, 1, 4, 2, 3.14f, 0.345f, 0.73f, 3.08f, 0.224f), RM_FORM(4, 2, 4, 1, 4, 2, 6.92f, 0.43f, 1.28f, 0.0f, 0.323f),
    RM_FORM(6, 2, 4, 1, 4, 2, 7.82f, 0.472f, 1.32f, 0.0f, 0.282f), RM_FORM(8, 2, 4, 1, 4, 2, 8.0f, 0.672f, 1.25f, 0.233f, 0.222f),
    RM_FORM(1, 1, 1, 4, 4, 4, 4.58f, 0.455f, 1.24f, 1.84f, 1.0f), RM_FORM(1, 1, 4, 1, 8, 4, 4.02f, 0.232f, 0.932f, 1.99f, 1.0f),
    RM_FORM(1, 2, 4, 1, 8, 4, 3.74f, 0.389f, 0.983f, 2.47f, 0.83f), RM_FORM(2, 1, 1, 4, 3, 4, 4.7f, 0.882f, 1.29f, 1.48f, 1.0f),
    RM_FORM(2, 1, 4, 1, 6, 4, 5.62f, 0.312f, 0.963f, 0.618f, 0.779f), RM_FORM(2, 2, 4, 1, 6, 4, 6.8f, 0.434f, 1.06f, 0.0f, 0.595f),
    RM_FORM(4, 1, 4, 1, 4, 4, 6.66f, 0.436f, 1.02f, 0.0f, 0.484f), RM_FORM(4, 2, 4, 1, 4, 4, 7.55f, 0.601f, 1.09f, 0.0f, 0.382f),
};
#undef RM_FORM
// Tiles of rows: with experts, whose counts only the device knows, one and a half standard deviations above the mean each
static long long rm_row_tiles(const RowLinear& p, int bm) {
  if (!p.offs) return (p.R + bm - 1LL) / bm;
  const int E = p.E < p.R ? p.E : p.R;
  const float mean = (float)p.R / (float)E, most = p.even_rows > 0 ? mean : mean + 1.5f * sqrtf(mean);
  return E * (long long)ceilf(most / (float)bm);
}

// The form and split with the least time by the figures above: on average 2.0 % above the best of all that were measured (384 shapes: one
// matrix, 8 and 32 experts, N 64 to 32000, K 512 to 14336, 9 to 3200 rows)
static MidPlan rm_best(const RowLinear& p) {
  const bool gated = hy_act_gated(p.act);
  return mid_plan(RM_FORMS, p.R, gated ? 2LL * p.N : p.N, p.K, p.offs ? (p.E < p.R ? p.E : p.R) : 1, [&](const RmForm& f) {
    return f.xb == (p.a_bf16 ? 2 : 4) && !(gated && f.nt % 2) && !(p.R <= RM_WIDE_SUM_ROWS && 16 * f.mt > RM_WIDE_SUM_ROWS);
  }, [&](int bm) { return rm_row_tiles(p, bm); });
}

// ... of the shapes that this thread has had last (the choice takes 1.1 us of host time, and a product asks for it twice)
static MidPlan rm_plan(const RowLinear& p) {
  struct Kept {
    int R, N, K, E, how;
    MidPlan plan;
  };
  thread_local Kept kept[64];
  const int how = 1 + p.a_bf16 + 2 * hy_act_gated(p.act) + 4 * (p.offs ? 1 : 0) + 8 * (p.even_rows > 0);
  Kept& k = kept[((unsigned)p.R * 31u + (unsigned)p.N / 4 * 7u + (unsigned)p.K / 64 * 5u + (unsigned)p.E + (unsigned)how) % 64];
  if (k.R != p.R || k.N != p.N || k.K != p.K || k.E != p.E || k.how != how) k = Kept{p.R, p.N, p.K, p.E, how, rm_best(p)};
  return k.plan;
}

// The range, and what is faster outside of it:
//  * fp32 rows of one matrix, 9 to 64 (more: the caller rounds them first; their bytes are x's twice). Up to 24 rows of K below 1024
//    rows_gemv.hip: 512 x 512, 16 rows 4.7 us there, 5.5 here; 1024 x 1024 6.1 both.
//  * bf16 rows of one matrix: to 255; from 256 on a prompt's rows have the 256-row tiles (us here | there, weights in no cache: 2048 x 2048,
//    255 | 777 rows 16 | 18, 27 | 25 with its sums; 4096 x 4096, 255 | 300 24.6 | 25.5, 29.9 | 27.7; 8224 x 2048, 300 33.2 | 31.4), and
//    wide outputs from 129 (32000 x 2048, 128 | 200 rows 48.5 | 47.4, 59 | 49; gated 14336 x 4096, 200 92 | 87).
//  * rows by expert: more than 64 up to 104 per expert on average, 64 where rows_gemm.hip's 128-row tiles are enough for every compute unit
//    (us here | there, 8 experts: gated 2816 x 2048, 64 | 80 | 112 rows each 59 | 51, 60 | 51, 67 | 54, gated 7168 x 4096, 80 | 112 213 | 203, 213 |
//    204; too few tiles: 2048 x 2816, 80 | 96 | 112 25 | 35, 25 | 36, 43 | 36, 4096 x 7168 95 | 120, 116 | 122, 175 | 131; 32 experts, 2048 x 2816, 64 | 80
//    90 | 81, 113 | 84), of K below 256 to 64 (16 per-head matrices of 512 x 128, 64 | 80 rows each 7.0 | 8.1, 10.9 | 8.1). Up to 64 rows in all rows_gemv.hip, unless there
//    are five per expert on large matrices (8 experts, 56 rows: gated 7168 x 4096 171 | 213, 4096 x 7168 82 | 106; gated 2816 x 2048 51 | 48, gated 512 x 1024 11 | 8).
constexpr int RM_MIN_ROWS = 9, RM_F32_ROWS = 64, RM_FEW_ROWS = 24, RM_FEW_K = 1024, RM_ROWS = 255;
constexpr int RM_WIDE = 16384, RM_WIDE_ROWS = 128;
constexpr long long RM_SORTED_WORK = 20000000;
constexpr int RM_EXPERT_ROWS = 104, RM_SORTED_ROWS = 64, RM_SHORT_K = 256, RM_SHORT_ROWS = 64;

bool hy_rows_mid_takes(const RowLinear& p) {
  auto aligned = [](const void* x, size_t n) { return ((uintptr_t)x & (n - 1)) == 0; };
  if (!p.wbf16 || p.a_scale || p.a_norm_w || p.tab || p.R < RM_MIN_ROWS || !(p.offs || (p.E == 1 && !p.row_expert)) || p.K % 64 || p.K < 128 ||
      p.lda % (p.a_bf16 ? 8 : 4) || p.N % 4 || p.ldo % 4 || p.w_stride % 8 || (p.add_out && p.out_bf16) || !aligned(p.a, 16) || !aligned(p.w, 16) ||
      !aligned(p.out, p.out_bf16 ? 8 : 16))
    return false;
  const long long nw = hy_act_gated(p.act) ? 2LL * p.N : p.N;
  if (p.offs) {
    if (p.R > RM_SORTED_ROWS) {
      const bool tiles = p.a_bf16 && p.K >= RM_TILES_K && p.E * ((nw + 127) / 128) >= 256;
      return p.R <= (long long)(p.K < RM_SHORT_K || tiles ? RM_SHORT_ROWS : RM_EXPERT_ROWS) * p.E;
    }
    if (p.a_bf16) return p.even_rows >= RM_MIN_ROWS;
    return p.R >= 5LL * p.E && nw >= 4096 && nw * p.K >= RM_SORTED_WORK;
  }
  if (!p.a_bf16) return p.R <= RM_F32_ROWS && !(p.R <= RM_FEW_ROWS && p.K < RM_FEW_K);
  return p.R <= (nw > RM_WIDE ? RM_WIDE_ROWS : RM_ROWS);
}

long long hy_rows_mid_floats(const RowLinear& p) {
  const MidPlan pl = rm_plan(p);
  return pl.splits > 1 ? (long long)pl.splits * p.R * (hy_act_gated(p.act) ? 2 : 1) * p.N : 0;
}

int hy_rows_mid(const RowLinear& p, float* ws, hipStream_t s) {
  const int gated = hy_act_gated(p.act), E = p.offs ? p.E : 1;
  const MidPlan pl = rm_plan(p);
  if (pl.form < 0) return -13;
  const RmForm& f = RM_FORMS[pl.form];
  const int bm = 16 * f.mt, bn = 16 * f.nt * f.wn;
  const long long tn = ((gated ? 2LL : 1LL) * p.N + bn - 1) / bn;
  const long long grid = ((p.offs ? p.R / bm + (long long)E : (p.R + bm - 1LL) / bm) * tn * pl.splits + 7) / 8 * 8;
  if (grid > 0x7fffffffLL) return -4;
  if (pl.splits > 1 && (!ws || ((uintptr_t)ws & 15))) return -12;
  RowLinear q = p;
  q.row_expert = nullptr;
  f.run((unsigned)grid, s, q, gated, (int)tn, pl.splits, pl.steps, pl.splits > 1 ? ws : nullptr);
  JLA_CHECK_LAUNCH();
  if (pl.splits > 1) {
    const long long n = (long long)p.R * (p.N / 4);
    rows_mid_sum_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(q, ws, pl.splits, gated);
    JLA_CHECK_LAUNCH();
  }
  return 0;
}

}  // namespace jla
