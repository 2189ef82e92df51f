// fp32 GEMM for the precision='highest' lm_head (reference model.py:698-736: only the lm_head honours
// `precision`, jax_test.py:433 runs the parity harness with precision='highest').
//
// y[M, N] = x[M, K] @ W[N, K]^T with fp32 inputs, fp32 accumulation and fp32 output. Rows of whole 16-byte pieces run as
// split products on the bf16 matrix cores (gemm_f32x3.h; us at M x 32000 x 4096, exact-f32 MFMA -> here: 1 555 -> 134, 100 565 -> 200,
// 128 570 -> 204, 600 1785 -> 859, 1500 4182 -> 1918); any other K or N on the exact-f32 MFMA (v_mfma_f32_32x32x2_f32: a
// k-ordered fmaf chain, no xf32 shortcut on gfx950): 128 x 128 output tile per 256-thread workgroup, four waves of 64 x 64
// (2 x 2 MFMA tiles), K staged 32 deep through LDS in k-major images ([k][row]) so a lane's fragment element (row l & 31, k
// l >> 5) is one conflict-free ds_read_b32.
#include "common.h"
#include "gemm_f32x3.h"
#include "launchers.h"

namespace jla {

constexpr int GF_BM = 128, GF_BN = 128, GF_BK = 32, GF_THREADS = 256;

using f32x16 = __attribute__((ext_vector_type(16))) float;

__global__ void __launch_bounds__(GF_THREADS)
    gemm_f32_kernel(const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ y, int M, int N,
                    int K) {
  __shared__ float As[GF_BK][GF_BM];
  __shared__ float Bs[GF_BK][GF_BN];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = blockIdx.y * GF_BM, n0 = blockIdx.x * GF_BN;
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  for (int k0 = 0; k0 < K; k0 += GF_BK) {
    // stage: 128 rows x 32 k of x and of W, one float4 (4 consecutive k) per thread and step
#pragma unroll
    for (int it = 0; it < (GF_BM * GF_BK / 4) / GF_THREADS; ++it) {
      const int e = it * GF_THREADS + tid;  // float4 index in the tile
      const int row = e / (GF_BK / 4), kq = (e % (GF_BK / 4)) * 4;
      const int gk = k0 + kq;
      float av[4] = {0.f, 0.f, 0.f, 0.f}, bv[4] = {0.f, 0.f, 0.f, 0.f};
      const int gm = m0 + row, gn = n0 + row;
      if (gm < M) {
        if (gk + 3 < K && (K & 3) == 0) {
          const float4 v = *reinterpret_cast<const float4*>(x + (size_t)gm * K + gk);
          av[0] = v.x; av[1] = v.y; av[2] = v.z; av[3] = v.w;
        } else {
          for (int q = 0; q < 4; ++q) av[q] = gk + q < K ? x[(size_t)gm * K + gk + q] : 0.f;
        }
      }
      if (gn < N) {
        if (gk + 3 < K && (K & 3) == 0) {
          const float4 v = *reinterpret_cast<const float4*>(w + (size_t)gn * K + gk);
          bv[0] = v.x; bv[1] = v.y; bv[2] = v.z; bv[3] = v.w;
        } else {
          for (int q = 0; q < 4; ++q) bv[q] = gk + q < K ? w[(size_t)gn * K + gk + q] : 0.f;
        }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        As[kq + q][row] = av[q];
        Bs[kq + q][row] = bv[q];
      }
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < GF_BK / 2; ++kk) {
      const int kr = 2 * kk + (lane >> 5);
      float a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) a[i] = As[kr][wm * 64 + i * 32 + (lane & 31)];
#pragma unroll
      for (int j = 0; j < 2; ++j) b[j] = Bs[kr][wn * 64 + j * 32 + (lane & 31)];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  // C/D map of the 32x32 shapes: col = lane & 31, row = (r & 3) + 8 (r >> 2) + 4 (lane >> 5)
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int col = n0 + wn * 64 + j * 32 + (lane & 31);
      if (col >= N) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = m0 + wm * 64 + i * 32 + (r & 3) + 8 * (r >> 2) + 4 * (lane >> 5);
        if (row < M) y[(size_t)row * N + col] = acc[i][j][r];
      }
    }
}

template <int MT>  // (MT waves)
__global__ void __launch_bounds__(64 * MT, 2) gemm_f32x3_kernel(F3Rows p, int tiles_n, int steps) {
  __shared__ u32x4 lds[f3_lds<MT>()];
  const int t0 = blockIdx.y * steps;
  p.out += (size_t)blockIdx.y * p.R * p.ldo;
  f3_tile<MT, 0, false>(p, tiles_n, t0, min(t0 + steps, (p.K + F3_BK - 1) / F3_BK), lds,
                 [](const f32x4 g, const f32x4) { return g; });
}

__global__ void __launch_bounds__(256) gemm_f32_sum_kernel(const f32x4* slabs, f32x4* y, size_t n, int splits) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  f32x4 v = slabs[i];
  for (int s = 1; s < splits; ++s) v += slabs[s * n + i];
  y[i] = v;
}

static bool f32x3_takes(const float* x, const float* w, const float* y, int M, int N, int K) {
  return M > 0 && N > 0 && K > 0 && K % 8 == 0 && N % 4 == 0 && (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15) == 0;
}
static F3Plan f32x3_plan(int M, int N, int K) {
  return f3_plan([&](int bm) { return (long long)(M + bm - 1) / bm; }, M, N, K);
}

long long gemm_f32_workspace(const float* x, const float* w, const float* y, int M, int N, int K) {
  if (!f32x3_takes(x, w, y, M, N, K)) return 0;
  const F3Plan pl = f32x3_plan(M, N, K);
  return pl.splits > 1 ? (long long)pl.splits * M * N : 0;
}

int gemm_f32(const float* x, const float* w, float* y, int M, int N, int K, float* ws, hipStream_t s) {
  if (M <= 0 || N <= 0 || K <= 0) return M < 0 || N < 0 || K < 0 ? -1 : 0;
  if (f32x3_takes(x, w, y, M, N, K)) {
    const F3Plan pl = f32x3_plan(M, N, K);
    if (pl.splits > 1 && (!ws || ((uintptr_t)ws & 15))) return -3;
    const F3Rows p{x, K, nullptr, nullptr, w, (long long)N * K, N, K, pl.splits > 1 ? ws : y, N, nullptr, 0, nullptr, 1, M};
    const long long tn = (N + pl.bn - 1) / pl.bn, tiles = ((M + pl.bm - 1) / pl.bm * tn + 7) / 8 * 8;
    if (tiles > 0x7fffffffLL) return -2;
    const dim3 grid((unsigned)tiles, pl.splits);
    if (pl.bm == 64) gemm_f32x3_kernel<4><<<grid, 256, 0, s>>>(p, (int)tn, pl.steps);
    else gemm_f32x3_kernel<8><<<grid, 512, 0, s>>>(p, (int)tn, pl.steps);
    JLA_CHECK_LAUNCH();
    if (pl.splits > 1) {
      const size_t n = (size_t)M * N / 4;
      gemm_f32_sum_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(reinterpret_cast<const f32x4*>(ws),
                                                                      reinterpret_cast<f32x4*>(y), n, pl.splits);
      JLA_CHECK_LAUNCH();
    }
    return 0;
  }
  dim3 grid((N + GF_BN - 1) / GF_BN, (M + GF_BM - 1) / GF_BM);
  if (grid.y > 65535) return -2;
  gemm_f32_kernel<<<grid, GF_THREADS, 0, s>>>(x, w, y, M, N, K);
  JLA_CHECK_LAUNCH();
  return 0;
}

}  // namespace jla
