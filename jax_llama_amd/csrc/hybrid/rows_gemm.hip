// Row-gathered, expert-grouped linear of a prompt on row-major bf16 weights and a bf16 activation copy:
//   out[dst(r), :] = act(A[src(r), :] @ W[expert(r)]^T),   the large form of linear_rows.hip's lr_gemm_kernel.
//
// What bounds it: the matrix cores. lr_gemm_kernel (64- or 128-row tiles, one LDS stage, VGPR staging) pulls 11 TB/s from
// L2 and stops at 300-450 TFLOP/s. Here one wave per SIMD owns a 128 x 16 NJ output block (NJ x 8 accumulators of
// v_mfma_f32_16x16x32_bf16 in AGPRs), K advances 64 per LDS slot, two slots filled by LDS-DMA, and every fragment read and
// DMA issue sits between MFMAs -- the schedule of the packed GEMM (kernels/gemm4w.h), with both operands row-major: the
// activation rows are gathered by per-lane addresses and the weight rows are read as they lie in the checkpoint, so an
// expert's weights need no second, packed copy. NJ = 8 (256 x 256 tiles) reads 256 B of LDS per MFMA, NJ = 4 (256 x 128)
// 384 B but makes twice the tiles: it is for launches that would leave the last round of workgroups nearly empty.
//
// LDS images of both operands: [rows][8 cells of 16 B] (64 k); cell c of row r holds k-chunk c ^ ((r & 15) >> 1), so the 16
// lanes of a fragment read fall on all 64 banks. A gated activation interleaves 16 gate rows and 16 up rows of W, which
// puts a column's gate and up accumulators into neighbouring tiles of one wave.
// The epilogue passes 64 rows at a time through the wave's own 32 KiB of LDS: the activation is then one small loop and
// rows leave as full lines (fp32: 512 B per row and wave).
#include "../kernels/gemm4w.h"
#include "../kernels/row_tiles.h"
#include "hy_util.h"
#include "hybrid.h"
#include "row_act.h"

namespace jla {

constexpr int RG_BM = 256, RG_BK = 64;
constexpr int RG_SLOT_U4 = 2 * RG_BM * RG_BK * 2 / 16;  // u32x4 of one slot: A 32 KiB + W 32 KiB (NJ = 4: half of it used)

template <int NJ>
__global__ void __launch_bounds__(256, 1) rows_gemm_kernel(RowLinear p, int gated, int tiles_n) {
  static_assert(NJ == 4 || NJ == 8, "16-column tiles per wave");
  constexpr int MPS = NJ / 2;  // MFMAs per slot: 8 NJ in 16 slots
  __shared__ u32x4 lds[2 * RG_SLOT_U4];
  const int lane = threadIdx.x & 63;
  const int wu = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wu >> 1, wc = wu & 1;
  int e = 0, r0 = 0, rend = 0, tn = 0;
  if (!row_tile<RG_BM>(p.offs, p.E, p.R, tiles_n, lane, e, r0, rend, tn)) return;
  const int K = p.K, N = p.N, KT = K / RG_BK;
  const int cols = gated ? 16 * NJ : 32 * NJ;  // output columns of the workgroup
  const int n0 = tn * cols;

  // DMA sources: piece P = wu + 4 j is 8 rows of 128 B; lane -> row 8 P + (lane >> 3), LDS cell lane & 7
  const char* pa[8];
  unsigned ow[NJ];
  const char* const wbase = reinterpret_cast<const char*>(reinterpret_cast<const bf16_t*>(p.w) + (size_t)e * p.w_stride);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int P = wu + 4 * j;
    const int row = min(r0 + 8 * P + (lane >> 3), rend - 1);  // (rows past the expert's end repeat its last one)
    const int chunk = (lane & 7) ^ (4 * (P & 1) + (lane >> 4));
    pa[j] = reinterpret_cast<const char*>(p.a) + ((size_t)(p.a_idx ? p.a_idx[row] : row) * p.lda + 8 * chunk) * 2;
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int P = wu + 4 * j, r = 8 * P + (lane >> 3), jt = r >> 4;
    const int chunk = (lane & 7) ^ (4 * (P & 1) + (lane >> 4));
    const int col = min(n0 + (gated ? 16 * (jt >> 1) + (r & 15) : r), N - 1);
    const int wrow = gated && (jt & 1) ? N + col : col;
    ow[j] = ((unsigned)wrow * (unsigned)K + 8u * (unsigned)chunk) * 2u;
  }
  auto dma = [&](int t, int j) {  // the j-th of this wave's 8 + NJ DMAs of K-tile t
    u32x4* slot = lds + (t & 1) * RG_SLOT_U4;
    if (j < 8) glds16(pa[j] + (size_t)t * 128, slot + (wu + 4 * j) * 64);
    else glds16(wbase + (size_t)t * 128 + ow[j - 8], slot + RG_BM * 8 + (wu + 4 * (j - 8)) * 64);
  };
  const int xrd = (wr * 128 + (lane & 15)) * 8, wrd = RG_BM * 8 + (wc * 16 * NJ + (lane & 15)) * 8;
  const int c0 = (0 + (lane >> 4)) ^ ((lane >> 1) & 7), c1 = (4 + (lane >> 4)) ^ ((lane >> 1) & 7);
  auto rd = [&](u32x4& dst, int slot, int h, int q) {  // q < NJ: W n-tile q; then the 8 m-tiles of A
    const u32x4* s = lds + slot * RG_SLOT_U4 + (h ? c1 : c0);
    dst = q < NJ ? s[wrd + q * 128] : s[xrd + (q - NJ) * 128];
  };

  f32x4 acc[NJ][8];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 w0[NJ], x0[8], w1[NJ], x1[8];

  // 8 NJ MFMAs on (wf, xf) with the 8 + NJ fragment reads of the next half tile and the DMAs of tile td between them
  auto substep = [&](u32x4 (&wf)[NJ], u32x4 (&xf)[8], u32x4 (&wn)[NJ], u32x4 (&xn)[8], bool do_rd, int rslot, int rh,
                     bool do_dma, int td) {
#pragma unroll
    for (int q = 0; q < 16; ++q) {
#pragma unroll
      for (int u = 0; u < MPS; ++u) {
        const int m = MPS * q + u;
        g4_mfma(acc[m >> 3][m & 7], wf[m >> 3], xf[m & 7]);
      }
      if (q < 8 + NJ) {
        if (do_rd) rd(q < NJ ? wn[q < NJ ? q : 0] : xn[q < NJ ? 0 : (q - NJ) & 7], rslot, rh, q);
        if (do_dma) dma(td, q);
      }
    }
  };
  auto mid_barrier = [&]() {  // this wave's DMAs of the next tile have landed; then every wave's have
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

#pragma unroll
  for (int j = 0; j < 8 + NJ; ++j) dma(0, j);
  if (KT > 1) {
#pragma unroll
    for (int j = 0; j < 8 + NJ; ++j) dma(1, j);
    wait_vmcnt<8 + NJ>();
  } else {
    wait_vmcnt<0>();
  }
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int q = 0; q < 8 + NJ; ++q) rd(q < NJ ? w0[q < NJ ? q : 0] : x0[q < NJ ? 0 : (q - NJ) & 7], 0, 0, q);

  int t = 0;
  for (; t + 2 < KT; ++t) {
    substep(w0, x0, w1, x1, true, t & 1, 1, false, 0);
    mid_barrier();
    substep(w1, x1, w0, x0, true, (t + 1) & 1, 0, true, t + 2);
  }
  if (t + 1 < KT) {
    substep(w0, x0, w1, x1, true, t & 1, 1, false, 0);
    mid_barrier();
    substep(w1, x1, w0, x0, true, (t + 1) & 1, 0, false, 0);
    ++t;
  }
  substep(w0, x0, w1, x1, true, t & 1, 1, false, 0);
  substep(w1, x1, w0, x0, false, 0, 0, false, 0);
  g4_acc_fence();
  __syncthreads();  // every wave is past its last fragment read: the slots become the epilogue's staging

  // lane (c = lane & 15, q = lane >> 4) holds row 16 i + c of the wave's 128 at accumulator columns 16 j + 4 q + 0..3
  constexpr int CH = 4 * NJ;  // 16-byte chunks of a staged row; chunk x of row r lies at x ^ (r & 15)
  f32x4* const wl = reinterpret_cast<f32x4*>(lds) + wu * 2048;
  const int c = lane & 15, q4 = lane >> 4;
  const int lanes_per_row = gated ? CH / 2 : CH;
  const int rpi = 64 / lanes_per_row;  // rows per step of the store loop
  const int rr0 = lane / lanes_per_row, oc = lane % lanes_per_row;
  const int gch = gated ? 8 * (oc >> 2) + (oc & 3) : oc;  // the staged chunk of output chunk oc (gate; up is 4 further)
  const int col = n0 + wc * (cols / 2) + 4 * oc;
#pragma unroll
  for (int half = 0; half < 2; ++half) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) wl[(16 * i + c) * CH + ((4 * j + q4) ^ c)] = g4_take(acc[j][4 * half + i]);
    const int rbase = r0 + wr * 128 + 64 * half;
    int drow = rbase + lane;  // lane l: where the half's row l goes (-1: past the expert's rows)
    drow = drow < rend ? (p.dst_idx ? p.dst_idx[drow] : drow) : -1;
#pragma unroll 4
    for (int s = 0; s < 64; s += rpi) {
      const int rr = s + rr0;
      const int d = __shfl(drow, rr, 64);
      const f32x4 g = wl[rr * CH + (gch ^ (rr & 15))];
      f32x4 v = g;
      if (gated) {
        const f32x4 u = wl[rr * CH + ((gch + 4) ^ (rr & 15))];
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = lr_act(p, g[x], u[x]);
      } else if (p.act != HY_ACT_NONE) {
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = lr_act(p, g[x], 0.f);
      }
      if (d >= 0 && col < N) {
        if (p.out_bf16) {
          *reinterpret_cast<u32x2*>(reinterpret_cast<bf16_t*>(p.out) + (size_t)d * p.ldo + col) =
              u32x2{pack2bf(v[0], v[1]), pack2bf(v[2], v[3])};
        } else {
          f32x4* o = reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.out) + (size_t)d * p.ldo + col);
          *o = p.add_out ? *o + v : v;
        }
      }
    }
  }
}

// Where the large tiles win over lr_gemm_kernel's 64-row ones (MI355X, gate / up of 2816 columns and down, us old -> new):
// 24000 rows, 8 experts, K 4096, F 7168: 6182 -> 2553, down 2921 -> 1186; 4096 rows, 8 experts, K 2048: 219 -> 139, 139 ->
// 73; one dense matrix, 777 rows, K 2048, F 5632: 93 -> 69. A tile is padded to 256 rows: with 64 experts of 64 rows the
// padding costs more than the pipeline gives (477 -> 528; of 80 rows 638 -> 609), unless every tile runs in the first
// round of workgroups anyway (8 experts of 32 rows, K 4096: 204 -> 138). Below K = 1024 the pipeline's fill and the
// epilogue outweigh the loop (K 512: 16 -> 21).
constexpr int RG_MIN_ROWS = 80, RG_MIN_ROWS_ONE_ROUND = 32, RG_MIN_K = 1024;

bool hy_rows_gemm_takes(const RowLinear& p) {
  const int E = p.offs ? p.E : 1;
  auto aligned = [](const void* x, size_t n) { return ((uintptr_t)x & (n - 1)) == 0; };
  const long long wrows = hy_act_gated(p.act) ? 2LL * p.N : p.N;
  const int min_rows = E * ((wrows + 255) / 256) <= 256 ? RG_MIN_ROWS_ONE_ROUND : RG_MIN_ROWS;
  return p.wbf16 && p.a_bf16 && !p.a_scale && !p.a_norm_w && (p.offs || p.E == 1) && p.R / E >= min_rows &&
         p.K >= RG_MIN_K && p.K % RG_BK == 0 && p.lda % 8 == 0 && p.N % 4 == 0 && p.ldo % 4 == 0 && p.w_stride % 8 == 0 &&
         aligned(p.a, 16) && aligned(p.w, 16) && aligned(p.out, p.out_bf16 ? 8 : 16) &&
         wrows * p.K * 2 < 0x100000000LL;  // (32-bit offsets into an expert's weights)
}

// For a caller who has yet to round its rows to bf16: a dense gated matrix of a short K whose 64-row tiles of fp32 rows all run at
// once is faster there. Us, 64-row tiles | here with the rounding: K 1024, gated N 1024, 300 | 512 | 700 rows 27.9 | 29.6, 27.7 |
// 30.2, 32.9 | 30.6; N 512, 700 | 1000 rows 28.0 | 31.0, 38.3 | 32.1; N 1376, 256 rows 39.7 | 29.7; K 1152, 512 rows of N 512 |
// 1024 31.1 | 33.0, 31.2 | 32.3; K 1280 even.
constexpr int RG_GATED_K = 1152, RG_GATED_N = 1024, RG_GATED_ROWS = 704, RG_GATED_TILES = 128;

bool hy_rows_gemm_pays(const RowLinear& p) {
  const bool few = hy_act_gated(p.act) && !p.offs && p.K <= RG_GATED_K && p.N <= RG_GATED_N && p.R <= RG_GATED_ROWS &&
                   (p.R + 63) / 64 * ((p.N + 63) / 64) <= RG_GATED_TILES;
  return hy_rows_gemm_takes(p) && !few;
}

int hy_rows_gemm(const RowLinear& p, hipStream_t s) {
  const int gated = hy_act_gated(p.act), E = p.offs ? p.E : 1;
  const long long wrows = gated ? 2LL * p.N : p.N;
  const long long mt_max = p.R / RG_BM + E;          // m-tiles at most (every expert's last one ragged)
  const long long mt = E == 1 ? (p.R + RG_BM - 1) / RG_BM : (p.R + RG_BM / 2LL * E) / RG_BM;  // ... on average
  const long long t8 = (wrows + 255) / 256, t4 = (wrows + 127) / 128;
  // whole rounds of 256 workgroups, a 256 x 128 tile at 0.55 of a 256 x 256 one's time
  const bool narrow = 55 * ((mt * t4 + 255) / 256) < 100 * ((mt * t8 + 255) / 256);
  const long long tn = narrow ? t4 : t8, grid = (mt_max * tn + 7) / 8 * 8;
  if (grid > 0x7fffffffLL) return -4;
  if (narrow) rows_gemm_kernel<4><<<(unsigned)grid, 256, 0, s>>>(p, gated, (int)tn);
  else rows_gemm_kernel<8><<<(unsigned)grid, 256, 0, s>>>(p, gated, (int)tn);
  JLA_CHECK_LAUNCH();
  return 0;
}

}  // namespace jla
