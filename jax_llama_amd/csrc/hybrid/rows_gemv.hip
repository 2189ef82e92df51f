// Few rows on bf16 weights: out[dst(r), :] = act(A[src(r), :] @ W[expert(r)]^T) for a decode step's or a short prompt's rows,
// the weights streamed once per 16 MT rows. The matrix-core form of linear_rows.hip's lr_gemv_kernel.
//
// What bounds it: the weight stream, and for a few MB the number of compute units that pull on it (one streams about 26
// bytes per ns). lr_gemv_kernel multiplies every weight by every row on the vector unit: one row already costs two
// instructions per weight (1.5-3.0 TB/s), eight rows re-read eight fp32 activation rows per column (0.6-1.6 TB/s).
// Here a lane's 16 bytes of a row-major weight row are the A operand of v_mfma_f32_16x16x32_bf16. With up to G = 4 or 8
// rows the instruction's 16 A rows are G output columns times 16 / G neighbouring K ranges and its 16 B columns the G
// activation rows times the same ranges: the diagonal blocks of the product hold the sums, a load covers G rows x 1024 / G
// contiguous bytes, and a workgroup needs only G columns -- enough workgroups for every compute unit from 1024 columns on.
// The waves of a workgroup deal the K steps among themselves, U in flight each, and sum their blocks through LDS.
// Us before -> after, weights in no cache, 1 | 8 | 33 rows: K 2048 x N 5152 11.1 -> 7.7 | 27.4 -> 10.7 | 54 -> 21; 4096 x 10304 42.6 ->
// 19.1 | 62.6 -> 26.6 | 108 -> 59; 2048 x 32000 49.6 -> 24.3 (5.4 TB/s) | 99 -> 29.4 | 67 -> 63; gated 2048 x 5632 17.2 -> 12.4 |
// 44.8 -> 16.0 | 82 -> 34; both products of 2 of 8 experts (4096 x 7168) for 1 | 8 tokens 105 -> 68 | 403 -> 230.
#include "hy_util.h"
#include "hybrid.h"
#include "row_act.h"

namespace jla {

JLA_DEV u32x4 rv_round8(const f32x4 a, const f32x4 b) {
  const float f[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  return pack8(f);
}

// G: output columns of a tile, and rows of a pass per 16 MT / (16 / G); NT: tiles of a workgroup (gated: gate and up tiles
// alternate); MT: 16-row tiles (G = 16); U: K steps in flight per wave. NORM (MT = 1): rows are RMS-normed with a gain
// first, in the order (a * scale) * gain of the norm kernel.
template <int G, int NT, int MT, int WAVES, int U, int NORM>
__global__ void __launch_bounds__(64 * WAVES) rows_gemv_kernel(RowLinear p, int rows_per_group, int gated) {
  static_assert(G == 16 || MT == 1, "several row tiles: whole 16-column tiles");
  constexpr int SEG = 16 / G;                // neighbouring K ranges of one MFMA
  constexpr int H = G == 16 ? 2 : 1;         // MFMAs of a K step (G = 16: the two halves of a 128-byte line)
  constexpr int STEP = 32 * SEG * H;         // K of a step
  constexpr int ROWS = G * MT;               // rows of a pass
  __shared__ f32x4 red[WAVES][NT * MT][64];
  __shared__ float stat[NORM ? WAVES : 1][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, q = lane >> 4;
  // rows of this group: a fixed count, one row with its own expert, or (offs) every row of expert blockIdx.y
  int g0 = blockIdx.y * rows_per_group, g1 = min(g0 + rows_per_group, p.R), e = 0;
  if (p.offs) {
    e = blockIdx.y;
    g0 = p.offs[e];
    g1 = p.offs[e + 1];
  } else if (p.row_expert) {
    e = p.row_expert[g0];
    if (e < 0 || e >= p.E) return;  // (a row of an expert without weights, an identity expert: nothing to compute)
  }
  const int K = p.K, N = p.N, steps = (K + STEP - 1) / STEP;
  const int k0 = 32 * (c / G) + 8 * q;  // this lane's place in a step
  const bf16_t* wbase = reinterpret_cast<const bf16_t*>(p.w) + (size_t)e * p.w_stride;
  const bf16_t* wp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int T = blockIdx.x * NT + t;
    const int col = min(G * (gated ? T >> 1 : T) + c % G, N - 1);
    wp[t] = wbase + (size_t)(gated && (T & 1) ? N + col : col) * K;
  }
  for (int r0 = g0; r0 < g1; r0 += ROWS) {
    const int nr = min(ROWS, g1 - r0);
    const float* xp[MT];
    float xs[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int rr = r0 + min(16 * m + c % G, nr - 1);  // (surplus lanes repeat the last row; their results are dropped)
      xp[m] = reinterpret_cast<const float*>(p.a) + (size_t)(p.a_idx ? p.a_idx[rr] : rr) * p.lda;
      xs[m] = p.a_scale ? p.a_scale[rr] : 1.f;
    }
    // (a lane past the end of a ragged last step reads the row's start; its operands are zeroed before they are used)
    auto at = [&](int s, int h) {
      const int k = STEP * s + 32 * h + k0;
      return k < K ? k : 0;
    };
    if (NORM) {
      float ss = 0.f;
#pragma unroll 4
      for (int s = wave; s < steps; s += WAVES) {
#pragma unroll
        for (int h = 0; h < H; ++h) {
          const int k = at(s, h);
          const f32x4 a = *reinterpret_cast<const f32x4*>(xp[0] + k), b = *reinterpret_cast<const f32x4*>(xp[0] + k + 4);
          float part = 0.f;
#pragma unroll
          for (int i = 0; i < 4; ++i) part = fmaf(b[i], b[i], fmaf(a[i], a[i], part));
          ss += STEP * s + 32 * h + k0 < K ? part : 0.f;
        }
      }
#pragma unroll
      for (int o = G; o < 64; o <<= 1) ss += __shfl_xor(ss, o, 64);
      if (lane < G) stat[wave][lane] = ss;
      __syncthreads();
      ss = 0.f;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) ss += stat[w][c % G];
      xs[0] = 1.f / sqrtf(ss / (float)K + p.a_norm_eps);
    }
    f32x4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int s0 = wave; s0 < steps; s0 += WAVES * U) {
      u32x4 wf[U][H][NT];
      f32x4 xa[U][H][MT], xb[U][H][MT];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int h = 0; h < H; ++h) {
          const int k = at(min(s0 + WAVES * u, steps - 1), h);  // (a step past the last one loads it again, unused)
#pragma unroll
          for (int t = 0; t < NT; ++t) wf[u][h][t] = load_nt(reinterpret_cast<const u32x4*>(wp[t] + k));
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            xa[u][h][m] = *reinterpret_cast<const f32x4*>(xp[m] + k);
            xb[u][h][m] = *reinterpret_cast<const f32x4*>(xp[m] + k + 4);
          }
        }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int s = s0 + WAVES * u;
        if (s >= steps) break;  // (wave-uniform)
#pragma unroll
        for (int h = 0; h < H; ++h) {
          const bool ragged = STEP * s + 32 * (h + 1) * SEG > K;  // (wave-uniform: some lane's range ends before K does)
          const bool in = STEP * s + 32 * h + k0 < K;
          if (ragged) {
#pragma unroll
            for (int t = 0; t < NT; ++t) wf[u][h][t] = in ? wf[u][h][t] : u32x4{0, 0, 0, 0};
          }
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            f32x4 a = xa[u][h][m], b = xb[u][h][m];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              a[i] *= xs[m];
              b[i] *= xs[m];
            }
            if (NORM) {
              const float* gw = p.a_norm_w + at(s, h);
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                a[i] *= gw[i];
                b[i] *= gw[4 + i];
              }
            }
            u32x4 x = rv_round8(a, b);
            if (ragged) x = in ? x : u32x4{0, 0, 0, 0};
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[t][m] = mfma16x16x32(wf[u][h][t], x, acc[t][m]);
          }
        }
      }
    }
    // lane: row (B column) c, columns (A rows) 4 q + 0..3 of tile t
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) red[wave][t * MT + m][lane] = acc[t][m];
    __syncthreads();
    constexpr int QUADS = G / 4, PER = QUADS * G;  // column quads of a tile; (quad, row) pairs per tile
    const int outs = (gated ? NT / 2 : NT) * MT * PER;
    for (int i = tid; i < outs; i += 64 * WAVES) {
      const int x = i % PER, tm = i / PER, to = tm / MT, m = tm - to * MT;  // output tile, row tile
      const int row = 16 * m + x % G, cq = x / G, col = G * (blockIdx.x * (gated ? NT / 2 : NT) + to) + 4 * cq;
      if (row >= nr || col >= N) continue;
      const int slot = (gated ? 2 * to : to) * MT + m;
      f32x4 g = f32x4{0.f, 0.f, 0.f, 0.f}, v = g;
#pragma unroll
      for (int sg = 0; sg < SEG; ++sg) {  // the diagonal block of range sg
        const int l = 16 * (QUADS * sg + cq) + G * sg + x % G;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
          g += red[w][slot][l];
          if (gated) v += red[w][slot + MT][l];
        }
      }
      const int r = r0 + row, drow = p.dst_idx ? p.dst_idx[r] : r;
      float* dst = reinterpret_cast<float*>(p.out) + (size_t)drow * p.ldo + col;
#pragma unroll
      for (int y = 0; y < 4; ++y)
        if (col + y < N) {
          const float val = lr_act(p, g[y], v[y]);
          dst[y] = p.add_out ? dst[y] + val : val;
        }
    }
    __syncthreads();
  }
}

// up to 64 rows, and up to 32 of a wide output, whose tiles fill the chip (64 rows x 32000 columns, K 2048: 70 us on the
// tiles, 82 here); one or two rows of a short K are over before the waves' sum pays (K 64: 3.2 against 3.6 us)
constexpr int RV_MAX_ROWS = 64, RV_MAX_WIDE_ROWS = 32, RV_WIDE = 16384, RV_MAX_NORM_ROWS = 16;

bool hy_rows_gemv_takes(const RowLinear& p) {
  auto aligned = [](const void* x) { return ((uintptr_t)x & 15) == 0; };
  return p.wbf16 && !p.a_bf16 && !p.out_bf16 && p.R <= (p.N >= RV_WIDE ? RV_MAX_WIDE_ROWS : RV_MAX_ROWS) &&
         (p.offs || p.row_expert || p.E == 1) && p.K % 8 == 0 &&
         p.K >= (p.R > 2 ? 64 : 256) && p.lda % 4 == 0 && p.w_stride % 8 == 0 && aligned(p.a) && aligned(p.w) &&
         (!p.a_norm_w || (p.R <= RV_MAX_NORM_ROWS && !p.offs && !p.row_expert && aligned(p.a_norm_w)));
}

int hy_rows_gemv(const RowLinear& p, hipStream_t s) {
  const int gated = hy_act_gated(p.act);
  RowLinear q = p;
  const bool each = !p.offs && p.row_expert;  // one row, one expert per group
  if (p.offs) q.row_expert = nullptr;
  const int groups = p.offs ? p.E : (each ? p.R : 1);
  const int rpg = each ? 1 : p.R;
  if (groups > 65535) return -4;
  // rows of a pass: a dense batch's count rounded up; an expert's share of the sorted rows, twice the mean (at least 4)
  const int even = p.offs && p.even_rows > 0 ? p.even_rows : 0;
  const int rows = each ? 1 : (p.offs ? (even ? even : (p.R < 2 * ((p.R + p.E - 1) / p.E) ? p.R : 2 * ((p.R + p.E - 1) / p.E))) : p.R);
  const int G = rows <= 4 ? 4 : (rows <= 8 ? 8 : 16), mt = rows <= 16 ? 1 : (rows <= 32 ? 2 : 4);
  const long long tiles = (gated ? 2LL : 1LL) * ((p.N + G - 1) / G);
  // one tile per workgroup until there are a few workgroups for every compute unit; then tiles share the workgroup's
  // activation reads, which weigh more the more rows there are (8 rows, K 4096 x N 4096: 1 / 2 / 4 tiles 15.0 / 12.3 / 14.8
  // us; K 2048 x N 32000: 46 / 35 / 29; one row 27.9 / 24.5 / 27.6)
  const long long all = tiles * groups;
  int nt = gated || mt > 1 || all >= (G == 4 ? 1024 : 512) ? 2 : 1;
  if (all >= (G > 4 ? 2048 : (gated ? 2048 : 12288))) nt = 4;
  const long long wgs = (tiles + nt - 1) / nt;
  if (wgs > 0x7fffffffLL) return -4;
  const dim3 grid((unsigned)wgs, groups);
#define RV_RUN(G, NT, MT, U, NORM) rows_gemv_kernel<G, NT, MT, 4, U, NORM><<<grid, 256, 0, s>>>(q, rpg, gated)
#define RV_NT(G, NORM)                  \
  do {                                  \
    if (nt == 1) RV_RUN(G, 1, 1, 4, NORM); \
    else if (nt == 2) RV_RUN(G, 2, 1, 2, NORM); \
    else RV_RUN(G, 4, 1, 2, NORM);      \
  } while (0)
#define RV_G(NORM)                \
  do {                            \
    if (G == 4) RV_NT(4, NORM);   \
    else if (G == 8) RV_NT(8, NORM); \
    else RV_NT(16, NORM);         \
  } while (0)
  if (mt == 4) {
    if (nt == 2) RV_RUN(16, 2, 4, 1, 0);
    else RV_RUN(16, 4, 4, 1, 0);
  } else if (mt == 2) {
    if (nt == 2) RV_RUN(16, 2, 2, 2, 0);
    else RV_RUN(16, 4, 2, 1, 0);
  } else if (p.a_norm_w) {
    RV_G(1);
  } else {
    RV_G(0);
  }
#undef RV_G
#undef RV_NT
#undef RV_RUN
  JLA_CHECK_LAUNCH();
  return 0;
}

}  // namespace jla
