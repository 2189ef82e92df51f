// Row-gathered, expert-grouped linear of a prompt on row-major bf16 weights and a bf16 activation copy:
//   out[dst(r), :] = act(A[src(r), :] @ W[expert(r)]^T),   the large form of linear_rows.hip's lr_gemm_kernel.
//
// What bounds it: the matrix cores, and the rows that whole tiles pad. lr_gemm_kernel (64- or 128-row tiles, one LDS stage, VGPR staging)
// pulls 11 TB/s from L2 and stops at 300-450 TFLOP/s. Here one wave per SIMD owns a 16 MI x 16 NJ output block (NJ x MI accumulators
// of v_mfma_f32_16x16x32_bf16 in AGPRs), K advances 64 per LDS slot, slots filled by LDS-DMA, and every fragment read and
// DMA issue sits between MFMAs -- the schedule of the packed GEMM (kernels/gemm4w.h), with both operands row-major: the
// activation rows are gathered by per-lane addresses and the weight rows are read as they lie in the checkpoint, so an
// expert's weights need no second, packed copy. MI = NJ = 8 (256 x 256 tiles) reads 256 B of LDS per MFMA and is for launches of many
// rounds; 128, 160 or 192 x 128 tiles (NJ = 4) read 384 to 512 B, but two of them share a compute unit, one's products behind
// the other's waits, and they pad less: 8 experts of 2816 x 2048 (7168 x 4096), both products, us with 256-row tiles -> now, 1000 | 2600 | 5000 | 12000
// rows 125 | 188 | 271 | 571 -> 95 | 137 | 211 | 444 (416 | 712 | 1025 | 2265 -> 360 | 533 | 939 | 2056); one gated matrix of 5632 x 2048, 600 | 1500 |
// 3000 rows 65 | 117 | 194 -> 36 | 77 | 136.
//
// Of 256 x 256 tiles a compute unit runs one, and waits are its own: at two slots for both operands a wave stood in them for 18 % of its time
// (the DMAs of K-tile t + 2 could not begin before the second half of t, and spread over it, the last had half a K-tile to land). With a third
// slot for the gathered rows (160 KiB in all) half of the DMAs go out half a K-tile earlier: 8 experts of 7168 x 4096, both products,
// 24000 | 6000 rows 3927 | 1143 -> 3659 | 1111 us. The smaller tiles' DMAs go out within the first half of a half K-tile instead (2600 rows of
// 2816 x 2048 156 -> 151 us).
//
// LDS images of both operands: [rows][8 cells of 16 B] (64 k); cell c of row r holds k-chunk c ^ ((r & 15) >> 1), so the 16
// lanes of a fragment read fall on all 64 banks. A gated activation interleaves 16 gate rows and 16 up rows of W, which
// puts a column's gate and up accumulators into neighbouring tiles of one wave.
// The epilogue passes 64 rows at a time through the wave's own 32 KiB of LDS: the activation is then one small loop (of its own for SwiGLU, the
// clamped gate and for none: 2 to 4 % of a product; in the loop for all activations the clamped gate had lost 2 %) and rows leave as full lines (fp32: 512 B per row and wave).
#include "../kernels/gemm4w.h"
#include "../kernels/row_tiles.h"
#include "hy_util.h"
#include "hybrid.h"
#include "row_act.h"

#include <type_traits>

namespace jla {

constexpr int RG_BK = 64;

template <int NJ, int MI>
constexpr int RG_PER_CU = (32 * MI + 32 * NJ) * RG_BK * 2 * 2 <= 80 * 1024 ? 2 : 1;  // workgroups whose slots fit a compute unit's LDS

// A wave's block: 16 MI rows x 16 NJ columns
template <int NJ, int MI>
__global__ void __launch_bounds__(256, (RG_PER_CU<NJ, MI>)) rows_gemm_kernel(RowLinear p, int gated, int tiles_n) {
  static_assert((NJ == 4 || NJ == 8) && MI >= 4 && MI <= 8, "16-column and 16-row tiles per wave");
  constexpr bool A3 = RG_PER_CU<NJ, MI> == 1;  // three slots of A, two of W
  constexpr int BM = 32 * MI, SA = BM * RG_BK * 2 / 16, SW = 32 * NJ * RG_BK * 2 / 16;  // u32x4 of a slot
  constexpr int W0 = (A3 ? 3 : 2) * SA, CELLS = W0 + 2 * SW;
  constexpr int T = NJ * MI;      // MFMAs of half a K-tile, in 16 groups
  constexpr int EG = MI == 8 ? 4 : (MI % 2 ? 1 : 2);  // row tiles that pass through LDS at a time at the end
  static_assert(CELLS >= 4 * EG * 16 * 4 * NJ && CELLS * 16 <= 160 * 1024, "the epilogue's staging");
  __shared__ u32x4 lds[CELLS];
  const int lane = threadIdx.x & 63;
  const int wu = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wu >> 1, wc = wu & 1;
  int e = 0, r0 = 0, rend = 0, tn = 0;
  if (!row_tile<BM>(p.offs, p.E, p.R, tiles_n, lane, e, r0, rend, tn)) return;
  const int K = p.K, N = p.N, KT = K / RG_BK;
  const int cols = gated ? 16 * NJ : 32 * NJ;  // output columns of the workgroup
  const int n0 = tn * cols;

  // DMA sources: piece P = wu + 4 j is 8 rows of 128 B; lane -> row 8 P + (lane >> 3), LDS cell lane & 7
  const char* pa[MI];
  unsigned ow[NJ];
  const char* const wbase = reinterpret_cast<const char*>(reinterpret_cast<const bf16_t*>(p.w) + (size_t)e * p.w_stride);
#pragma unroll
  for (int j = 0; j < MI; ++j) {
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
  auto a_slot = [&](int t) { return (A3 ? t % 3 : t & 1) * SA; };
  auto dma = [&](int t, int j) {  // the j-th of this wave's MI + NJ DMAs of K-tile t
    if (j < MI) glds16(pa[j < MI ? j : 0] + (size_t)t * 128, lds + a_slot(t) + (wu + 4 * j) * 64);
    else glds16(wbase + (size_t)t * 128 + ow[j < MI ? 0 : j - MI], lds + W0 + (t & 1) * SW + (wu + 4 * (j - MI)) * 64);
  };
  const int xrd = (wr * 16 * MI + (lane & 15)) * 8, wrd = W0 + (wc * 16 * NJ + (lane & 15)) * 8;
  const int c0 = (0 + (lane >> 4)) ^ ((lane >> 1) & 7), c1 = (4 + (lane >> 4)) ^ ((lane >> 1) & 7);
  auto rd = [&](u32x4& dst, int t, int h, int q) {  // of K-tile t: q < NJ: W n-tile q; then the MI m-tiles of A
    const u32x4* s = lds + (h ? c1 : c0);
    dst = q < NJ ? s[wrd + (t & 1) * SW + q * 128] : s[xrd + a_slot(t) + (q - NJ) * 128];
  };

  f32x4 acc[NJ][MI];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 w0[NJ], x0[MI], w1[NJ], x1[MI];

  // MI NJ MFMAs on (wf, xf) with the MI + NJ fragment reads of the next half tile (K-tile tr) and the DMAs [d0, d1) of K-tile td
  // between them
  auto substep = [&](u32x4 (&wf)[NJ], u32x4 (&xf)[MI], u32x4 (&wn)[NJ], u32x4 (&xn)[MI], bool do_rd, int tr, int rh, bool do_dma,
                     int td, int d0, int d1) {
    constexpr int DQ = A3 ? 16 : 8;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
#pragma unroll
      for (int m = q * T / 16; m < (q + 1) * T / 16; ++m) g4_mfma(acc[m / MI][m % MI], wf[m / MI], xf[m % MI]);
      if (do_dma && q < DQ) {
#pragma unroll
        for (int j = d0 + q * (d1 - d0) / DQ; j < d0 + (q + 1) * (d1 - d0) / DQ; ++j) dma(td, j);
      }
      if (q < MI + NJ && do_rd) rd(q < NJ ? wn[q < NJ ? q : 0] : xn[q < NJ ? 0 : (q - NJ) % MI], tr, rh, q);
    }
  };
  // this wave's DMAs of the next tile have landed (the rows of the tile behind it, the last MI issued, may be under way); then every wave's have
  auto mid_barrier = [&](bool rows_under_way) {
    if (rows_under_way) __builtin_amdgcn_s_waitcnt(0x0070 | (MI & 15) | ((MI >> 4) << 14));  // vmcnt(MI) lgkmcnt(0)
    else __builtin_amdgcn_s_waitcnt(0x0070);                                                   // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

#pragma unroll
  for (int j = 0; j < MI + NJ; ++j) dma(0, j);
  if (KT > 1) {
#pragma unroll
    for (int j = 0; j < MI + NJ; ++j) dma(1, j);
    wait_vmcnt<MI + NJ>();
  } else {
    wait_vmcnt<0>();
  }
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int q = 0; q < MI + NJ; ++q) rd(q < NJ ? w0[q < NJ ? q : 0] : x0[q < NJ ? 0 : (q - NJ) % MI], 0, 0, q);

  // (A3: the rows of K-tile t + 2 go into the slot of t - 1 already during the first half of t, the weights into t's own during the second)
  constexpr int DS = A3 ? MI : 0;
  int t = 0;
  for (; t + 2 < KT; ++t) {
    substep(w0, x0, w1, x1, true, t, 1, A3, t + 2, 0, DS);
    mid_barrier(A3);
    substep(w1, x1, w0, x0, true, t + 1, 0, true, t + 2, DS, MI + NJ);
  }
  if (t + 1 < KT) {
    substep(w0, x0, w1, x1, true, t, 1, false, 0, 0, 0);
    mid_barrier(false);
    substep(w1, x1, w0, x0, true, t + 1, 0, false, 0, 0, 0);
    ++t;
  }
  substep(w0, x0, w1, x1, true, t, 1, false, 0, 0, 0);
  substep(w1, x1, w0, x0, false, 0, 0, false, 0, 0, 0);
  g4_acc_fence();
  __syncthreads();  // every wave is past its last fragment read: the slots become the epilogue's staging

  // lane (c = lane & 15, q = lane >> 4) holds row 16 i + c of the wave's 16 MI at accumulator columns 16 j + 4 q + 0..3
  constexpr int CH = 4 * NJ;  // 16-byte chunks of a staged row; chunk x of row r lies at x ^ (r & 15)
  f32x4* const wl = reinterpret_cast<f32x4*>(lds) + wu * (16 * EG * CH);
  const int c = lane & 15, q4 = lane >> 4;
  const int lanes_per_row = gated ? CH / 2 : CH;
  const int rpi = 64 / lanes_per_row;  // rows per step of the store loop
  const int rr0 = lane / lanes_per_row, oc = lane % lanes_per_row;
  const int gch = gated ? 8 * (oc >> 2) + (oc & 3) : oc;  // the staged chunk of output chunk oc (gate; up is 4 further)
  const int col = n0 + wc * (cols / 2) + 4 * oc;
#pragma unroll
  for (int part = 0; part < MI / EG; ++part) {
#pragma unroll
    for (int i = 0; i < EG; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) wl[(16 * i + c) * CH + ((4 * j + q4) ^ c)] = g4_take(acc[j][EG * part + i]);
    const int rbase = r0 + wr * 16 * MI + 16 * EG * part;
    int drow = rbase + (lane & (16 * EG - 1));  // lane l: where the part's row l goes (-1: past the expert's rows)
    drow = drow < rend ? (p.dst_idx ? p.dst_idx[drow] : drow) : -1;
    auto rows_out = [&](auto known) {
      constexpr int ACT = decltype(known)::value;  // -1: whatever p.act says
#pragma unroll 4
      for (int s = 0; s < 16 * EG; s += rpi) {
        const int rr = s + rr0;
        const int d = __shfl(drow, rr, 64);
        f32x4 v = wl[rr * CH + (gch ^ (rr & 15))];
        if constexpr (ACT == HY_ACT_SWIGLU) {
          const f32x4 u = wl[rr * CH + ((gch + 4) ^ (rr & 15))];
#pragma unroll
          for (int x = 0; x < 4; ++x) v[x] = hy_silu(v[x]) * u[x];
        } else if constexpr (ACT == HY_ACT_CLAMP_GLU) {
          const f32x4 u = wl[rr * CH + ((gch + 4) ^ (rr & 15))];
#pragma unroll
          for (int x = 0; x < 4; ++x) v[x] = lr_clamp_glu(p, v[x], u[x]);
        } else if constexpr (ACT != HY_ACT_NONE) {
          const f32x4 u = gated ? wl[rr * CH + ((gch + 4) ^ (rr & 15))] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int x = 0; x < 4; ++x) v[x] = lr_act(p, v[x], u[x]);
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
    };
    // (the switch over activations stays out of the loop)
    if (p.act == HY_ACT_SWIGLU) rows_out(std::integral_constant<int, HY_ACT_SWIGLU>{});
    else if (p.act == HY_ACT_CLAMP_GLU) rows_out(std::integral_constant<int, HY_ACT_CLAMP_GLU>{});
    else if (p.act == HY_ACT_NONE) rows_out(std::integral_constant<int, HY_ACT_NONE>{});
    else rows_out(std::integral_constant<int, -1>{});
  }
}

// Where they win over lr_gemm_kernel's 64-row tiles (gate / up of 2816 columns and down, us there -> 256-row tiles here): 24000 rows, 8
// experts, K 4096, F 7168: 6182 -> 2553, down 2921 -> 1186; 4096 rows, 8 experts, K 2048: 219 -> 139, 139 -> 73; one dense matrix, 777 rows,
// K 2048, F 5632: 93 -> 69. Fewer rows per expert than these minima are rows_mid.hip's, which streams the weights as fast and pads less
// (48 rows each of 8 experts, 4096 x 7168 99 us there, 126 here). Below K = 1024 the pipeline's fill and the epilogue outweigh the loop (K
// 512: 16 -> 21).
constexpr int RG_MIN_ROWS = 65, RG_MIN_ROWS_ONE_ROUND = 32, RG_MIN_K = RM_TILES_K;

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

// A form's measured times, us: launch and fill; a 64-deep step of one workgroup; its rise with every further one of a compute unit, whose
// last round counts as `last` workgroups more; what such a one takes besides (of one workgroup per unit nobody hides its first copies and its stores)
struct RgForm {
  int nj, mi;
  float fill, step, more, last, ends;
};
static const RgForm RG_FORMS[] = {{4, 4, 1.0f, 0.644f, 0.833f, 1.0f, 0.f}, {4, 5, 9.75f, 0.608f, 0.965f, 0.99f, 0.f},
                                  {4, 6, 5.17f, 0.819f, 0.795f, 0.945f, 0.f}, {8, 8, 22.f, 1.3f, 1.2f, 1.0f, 8.f}};

// The form with the least time by the figures above: on average 4.0 % above the best of those measured (375 products, gated and down: 2 to 32
// experts and one matrix, 300 to 24000 rows, K 1024 to 14336, rows dealt unevenly as the rule cannot know). With experts, whose counts only
// the device knows, the row tiles are a mean over four counts around the average. Eight rounds of 256 x 256 tiles and more: these (8 experts of
// gated 7168 x 4096, 6000 | 12000 rows 667 | 1295, 192 x 128 688 | 1336: fewer bytes cost less power).
// The third slot of the 256 x 256 form takes its time off every step, not off a round's ends: of a short K the 192-row tiles stay ahead. Us, 192 rows |
// 256: 8 experts of 4096 x 7168, 9000 rows 590 | 507, gated 7168 x 4096, 6000 rows 740 | 667, 4 of 5120 x 3584, 24000 rows 865 | 760; but 4
// of 1024 x 2048, 24000 rows 98 | 115, 16 of 2048 x 1408, 12000 rows 87 | 93, gated 2048 x 1024, 24000 rows 211 | 236, 8 of 2816 x 2048, 4000
// rows 111 | 115, clamped 119 | 132. (Figures without `ends`: 4.4 % above the best, and those of two slots 4.6 %.)
constexpr long long RG_MANY = 8 * 256;

static const RgForm& rg_form(const RowLinear& p) {
  const int E = p.offs ? p.E : 1;
  const long long wrows = hy_act_gated(p.act) ? 2LL * p.N : p.N;
  const float mean = (float)p.R / (float)E, sd = E > 1 && p.even_rows <= 0 ? sqrtf(mean * (1.f - 1.f / (float)E)) : 0.f;
  const float stream = 3.5f + (float)E * (float)wrows * (float)p.K * 2 / 5.4e6f;  // the weights themselves
  const RgForm* best = nullptr;
  float least = 1e30f;
  for (const RgForm& f : RG_FORMS) {
    float mt = 0.f;
    for (int i = 0; i < 4; ++i) mt += ceilf((mean + (0.8f * (float)i - 1.2f) * sd) / (float)(32 * f.mi));
    const float tiles = mt * .25f * (float)E * (float)((wrows + 32 * f.nj - 1) / (32 * f.nj)), load = tiles / 256.f;
    if (f.mi == 8 && tiles >= (float)RG_MANY) return f;
    const float deep = f.mi == 8 ? ceilf(load - .02f) : (load <= 1.f ? 1.f : (load <= 2.f ? 2.f : load + f.last));
    float us = f.fill + f.ends * (deep - 1.f) + f.step * (float)(p.K / RG_BK) * (1.f + f.more * (deep - 1.f));
    if (us < stream) us = stream;
    if (us < least) {
      least = us;
      best = &f;
    }
  }
  return *best;
}

int hy_rows_gemm(const RowLinear& p, hipStream_t s) {
  const int gated = hy_act_gated(p.act), E = p.offs ? p.E : 1;
  const long long wrows = gated ? 2LL * p.N : p.N;
  const RgForm& f = rg_form(p);
  const long long tn = (wrows + 32 * f.nj - 1) / (32 * f.nj), grid = ((p.R / (32 * f.mi) + (long long)E) * tn + 7) / 8 * 8;
  if (grid > 0x7fffffffLL) return -4;
  const unsigned g = (unsigned)grid;
  if (f.mi == 4) rows_gemm_kernel<4, 4><<<g, 256, 0, s>>>(p, gated, (int)tn);
  else if (f.mi == 5) rows_gemm_kernel<4, 5><<<g, 256, 0, s>>>(p, gated, (int)tn);
  else if (f.mi == 6) rows_gemm_kernel<4, 6><<<g, 256, 0, s>>>(p, gated, (int)tn);
  else rows_gemm_kernel<8, 8><<<g, 256, 0, s>>>(p, gated, (int)tn);
  JLA_CHECK_LAUNCH();
  return 0;
}

}  // namespace jla
