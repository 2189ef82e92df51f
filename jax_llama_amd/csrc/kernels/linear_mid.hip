// 17 to 256 rows on packed bf16 weights: y [M, N] = epilogue([inv_rms(x) *] x [M, K] @ W^T), the decode step of a mid-sized
// batch and short prompts (reference ops: the projections of jax_llama/model.py:210, :294, :338 and the head, :736, with the norm
// before them, :384, :395, :662). mid_tile.h says what bounds it and why the tile is as it is; here are its forms and the choice among them.
//
// Without a K split over workgroups the epilogue runs here: a workgroup's sums pass through LDS, so that a store leaves as whole
// rows of the tile and a gate column finds its up column whichever wave had it. With one, the partial sums go to slabs for
// gemm_reduce_kernel. The norm's row statistic comes from the x fragments that the products read anyway.
#include "mid_tile.h"
#include "gemm_out.h"
#include "launchers.h"
#include "row_tiles.h"

namespace jla {

struct LinearMid {
  const bf16_t* x;  // [M, K]
  const bf16_t* w;  // packed fragments [N / 16][K / 32][64][8]
  int M, N, K, mode;
  void* out;
  int accumulate, out_f32;
  bf16_t* mirror;
  float* slabs;  // [splits][M][N], or null: the epilogue here
  float* ssq;    // [splits][M]: partial sums of squares, with slabs
  float rms_eps; // >= 0: norm
  int tiles_n, splits, steps;
  QKVArgs qa;
};

// What was here before, GEMVs that deal K to their waves and tiles that split it over workgroups, has fp32 chains of an eighth to a half of K. One chain
// over a workgroup's steps would be longer, so every LM_RUN steps (eight products) of it are added in 64 bits, or in 32 where a wave's sums would
// not fit its registers twice. Relative errors against 64 bits, before | one chain | now, 64 and 128 rows: 6144 x 4096 1.9e-7 | 1.9e-7 | 9.3e-8, 1.3e-7 |
// 2.7e-7 | 8.9e-8; 28672 x 4096 1.9e-7 | 3.9e-7 | 8.9e-8, 2.7e-7 | 3.9e-7 | 1.2e-7 (32 bits); 4096 x 14336 1.9e-7 | 3.7e-7 | 9.8e-8, 1.9e-7 | 2.6e-7 | 1.2e-7. Us, one
// chain -> now: 19.9 -> 20.8, 23.1 -> 23.5; 49.4 -> 49.3, 51.3 -> 54.2; 29.5 -> 29.9, 33.6 -> 33.9.
constexpr int LM_RUN = 4;
template <int MT, int NT>
using LmSum = std::conditional_t<MT * NT <= 8, f64x4, f32x4>;

// SS: the norm's statistic is wanted
template <int MT, int NT, int WN, int WK, int S, bool SS>
__global__ void __launch_bounds__(64 * WN * WK, (MidShape<MT, NT, WN, WK, S, 2>::PER_SIMD)) linear_mid_kernel(LinearMid p) {
  using H = MidShape<MT, NT, WN, WK, S, 2>;
  constexpr int LD = H::BN + 4;  // floats of a row of the staged sums: the 16 rows of a store on different banks
  static_assert(H::BM * LD / 4 <= H::LDS, "the sums reuse the ring");
  static_assert(H::BN % 32 == 0, "a tile holds both columns of a pair");
  __shared__ u32x4 lds[H::LDS];
  __shared__ float stat[SS ? WK : 1][SS ? H::BM : 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, q = lane >> 4, wn = wave % WN, wk = wave / WN;
  int e = 0, r0 = 0, rend = 0, tn = 0, split = 0;
  if (!row_tile<H::BM>(nullptr, 1, p.M, p.tiles_n, lane, e, r0, rend, tn, p.splits, split)) return;
  const int K = p.K, N = p.N, n0 = tn * H::BN, t0 = split * p.steps, t1 = min(K >> 6, t0 + p.steps);
  auto xrow = [&](int r) { return reinterpret_cast<const char*>(p.x + (size_t)min(r0 + r, rend - 1) * K); };
  auto wrow = [&](int r) { return reinterpret_cast<const char*>(p.w + (size_t)min((n0 + r) >> 4, (N >> 4) - 1) * 16 * K); };
  float ss[SS ? MID_SQ<MT, WN> : 1];
  f32x4 acc[NT][MT];
  mid_tile<MT, NT, WN, WK, S, 2, true, SS, LmSum<MT, NT>>(lds, xrow, wrow, t0, t1, acc, ss, LM_RUN);
  if constexpr (SS) {
#pragma unroll
    for (int m = 0; m < MID_SQ<MT, WN>; ++m) {
      float v = ss[m];
      v += __shfl_xor(v, 16, 64);
      v += __shfl_xor(v, 32, 64);
      const int tile = wn * MID_SQ<MT, WN> + m;
      if (q == 0 && tile < MT) stat[wk][16 * tile + c] = v;
    }
  }
  auto squares = [&](int r) {
    float v = stat[0][r];
#pragma unroll
    for (int w = 1; w < (SS ? WK : 1); ++w) v += stat[w][r];
    return v;
  };
  if (p.slabs) {
    if (wk == 0) {
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int row = r0 + 16 * mid_row_tile<MT, WN, SS>(m, wn) + c;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const int col = n0 + 16 * (wn * NT + t) + 4 * q;
          if (row < rend && col < N) *reinterpret_cast<f32x4*>(p.slabs + ((size_t)split * p.M + row) * N + col) = acc[t][m];
        }
      }
    }
    if (SS && tn == 0) {
      __syncthreads();
      for (int r = tid; r < H::BM; r += 64 * H::WAVES)
        if (r0 + r < rend) p.ssq[(size_t)split * p.M + r0 + r] = squares(r);
    }
    return;
  }
  float* sums = reinterpret_cast<float*>(lds);
  __syncthreads();  // every wave is past the ring
  if (wk == 0) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int t = 0; t < NT; ++t) *reinterpret_cast<f32x4*>(sums + (16 * mid_row_tile<MT, WN, SS>(m, wn) + c) * LD + 16 * (wn * NT + t) + 4 * q) = acc[t][m];
  }
  __syncthreads();
  if constexpr (SS) {  // (a row by one thread: it reads the K groups' shares before it writes over the first)
    for (int r = tid; r < H::BM; r += 64 * H::WAVES) stat[0][r] = 1.f / sqrtf(squares(r) / (float)K + p.rms_eps);
    __syncthreads();
  }
  const bool glu = p.mode == MODE_SWIGLU;
  const int per_row = (glu ? H::BN / 2 : H::BN) / 4, rows = min(H::BM, rend - r0);
  for (int i = tid; i < rows * per_row; i += 64 * H::WAVES) {
    const int r = i / per_row, j = i - r * per_row;
    const int lc = glu ? 32 * (j >> 2) + 4 * (j & 3) : 4 * j, col = n0 + lc;
    if (col >= N) continue;
    const float sc = SS ? stat[0][r] : 1.f;
    const float* at = sums + r * LD + lc;
    const float v[4] = {at[0] * sc, at[1] * sc, at[2] * sc, at[3] * sc};
    switch (p.mode) {  // (uniform)
      case MODE_SWIGLU: {
        const float u[4] = {at[16] * sc, at[17] * sc, at[18] * sc, at[19] * sc};
        gemm_out4<MODE_SWIGLU>(v, u, r0 + r, col, N, p.out, p.accumulate, p.out_f32, p.mirror, p.qa);
        break;
      }
      case MODE_RESIDUAL: gemm_out4<MODE_RESIDUAL>(v, v, r0 + r, col, N, p.out, p.accumulate, 1, p.mirror, p.qa); break;
      case MODE_QKV: gemm_out4<MODE_QKV>(v, v, r0 + r, col, N, nullptr, 0, 0, nullptr, p.qa); break;
      default: gemm_out4<MODE_STORE>(v, v, r0 + r, col, N, p.out, p.accumulate, p.out_f32, nullptr, p.qa);
    }
  }
}

struct LmForm {  // (mid_plan)
  int mt, nt, wn, wk;
  float fill, stage, more, sum, mb;
  void (*run)(unsigned, hipStream_t, const LinearMid&);
};
template <int MT, int NT, int WN, int WK, int S>
static void lm_launch(unsigned grid, hipStream_t s, const LinearMid& p) {
  if (p.rms_eps >= 0.f) linear_mid_kernel<MT, NT, WN, WK, S, true><<<grid, 64 * WN * WK, 0, s>>>(p);
  else linear_mid_kernel<MT, NT, WN, WK, S, false><<<grid, 64 * WN * WK, 0, s>>>(p);
}
#define LM_FORM(MT, NT, WN, WK, S, ...) {MT, NT, WN, WK, __VA_ARGS__, lm_launch<MT, NT, WN, WK, S>}
static const LmForm LM_FORMS[] = {
    LM_FORM(2, 1, 4, 1, 6, 4.14f, 0.242f, 0.876f, 1.81f, 0.322f), LM_FORM(2, 2, 4, 1, 6, 4.6f, 0.383f, 1.16f, 1.41f, 0.4f),
    LM_FORM(4, 1, 4, 1, 4, 4.51f, 0.332f, 0.654f, 1.19f, 0.301f), LM_FORM(4, 1, 4, 2, 4, 5.04f, 0.485f, 1.19f, 1.17f, 0.462f),
    LM_FORM(4, 2, 4, 1, 4, 5.9f, 0.435f, 1.09f, 0.454f, 0.291f), LM_FORM(6, 2, 4, 1, 4, 7.14f, 0.492f, 1.18f, 0.0f, 0.266f),
    LM_FORM(8, 2, 4, 1, 4, 7.85f, 0.586f, 1.28f, 0.0f, 0.225f),
};
#undef LM_FORM
constexpr int LM_N_FORMS = sizeof(LM_FORMS) / sizeof(LM_FORMS[0]);

bool linear_mid_tile(int tile) { return tile >= LINEAR_MID_TILE && tile < LINEAR_MID_TILE + LM_N_FORMS; }

// The form (as a tile config) and K split with the least time by the figures above: on average 1.6 % above the best of all that were
// measured (11 matrices from 256 x 512 to 128256 x 4096, 17 to 256 rows, the epilogues that follow them). Against what ran before, the
// tiles of 128 and 256 rows with their splits and the GEMVs (us here | there, weights in no cache, rows 48 to 128; 17 to 32 within 5 % either
// way, so these stay a measured choice, as do 129 to LINEAR_MID_MAX_M, where narrow outputs gain and wide ones lose):
//   6144 x 4096, 64 | 128 rows 20.8 | 24.8, 23.5 | 26.6;  4096 x 4096 14.7 | 20.8, 18.5 | 23.1;
//   28672 x 4096 49.3 | 62.7, 54.2 | 67.8;  4096 x 14336 29.9 | 34.4, 33.9 | 39.1.
// A head's N from 100 rows on is better off in tiles of more columns: 128256 x 4096, 100 | 128 rows 228 | 217, 238 | 227 (64: 196 | 205).
constexpr int LM_WIDE_M = 96, LM_WIDE_N = 65536;
int linear_mid_plan(int M, int N, int K, int* ksplit) {
  *ksplit = 1;
  if (M < LINEAR_MID_MIN_M || M > LINEAR_MID_MAX_M || (N & 15) || (K & 63) || K < 128 || (M > LM_WIDE_M && N > LM_WIDE_N)) return 0;
  const MidPlan p = mid_plan(LM_FORMS, M, N, K, 1, [](const LmForm&) { return true; }, [&](int bm) { return (M + bm - 1LL) / bm; });
  *ksplit = p.splits;
  return p.form < 0 ? 0 : LINEAR_MID_TILE + p.form;
}

// The product's launch (of splits > 1, or slabs for another reason: the partial sums' one): K in `ksplit` runs, as linear_mid_plan cuts it
int linear_mid(const bf16_t* x, const void* W, void* out, int M, int N, int K, int mode, int accumulate, int out_f32, bf16_t* mirror,
               const QKVArgs* qkv, float* slabs, float* ssq, int ksplit, float rms_eps, int tile, hipStream_t s) {
  if (!linear_mid_tile(tile) || (N & 15) || (K & 63) || K < 64 || M <= 0 || ksplit < 1) return -1;
  const LmForm& f = LM_FORMS[tile - LINEAR_MID_TILE];
  const int T = K >> 6, steps = ((T + ksplit - 1) / ksplit + f.wk - 1) / f.wk * f.wk;
  if (T % f.wk || (T + steps - 1) / steps != ksplit || (ksplit > 1 && !slabs)) return -1;
  LinearMid p{x, reinterpret_cast<const bf16_t*>(W), M, N, K, mode, out, accumulate, out_f32, mirror, slabs, ssq, rms_eps,
              (N + 16 * f.nt * f.wn - 1) / (16 * f.nt * f.wn), ksplit, steps, QKVArgs{}};
  if (qkv) p.qa = *qkv;
  const long long grid = ((M + 16LL * f.mt - 1) / (16LL * f.mt) * p.tiles_n * ksplit + 7) / 8 * 8;
  if (grid > 0x7fffffffLL) return -4;
  f.run((unsigned)grid, s, p);
  JLA_CHECK_LAUNCH();
  return 0;
}

JLA_BOUNDS_ACCESSOR(linear_mid)

}  // namespace jla
