// Few rows on bf16 weights: out[dst(r), :] = act(A[src(r), :] @ W[expert(r)]^T) for a decode step's or a short prompt's rows,
// the weights streamed once per 16 MT rows. The matrix-core form of linear_rows.hip's lr_gemv_kernel.
//
// What bounds it: the weight stream, and for a few MB the number of compute units that pull on it (one streams about 26
// bytes per ns). lr_gemv_kernel multiplies every weight by every row on the vector unit: one row already costs two
// instructions per weight (1.5-3.0 TB/s), eight rows re-read eight fp32 activation rows per column (0.6-1.6 TB/s).
// Here a lane's 16 bytes of a row-major weight row are the A operand of v_mfma_f32_16x16x32_bf16. With up to G = 4 or 8
// rows the instruction's 16 A rows are G output columns times 16 / G neighbouring K ranges and its 16 B columns the G
// activation rows times the same ranges: the diagonals of the product's blocks hold the sums, a load covers G rows x 1024 / G
// contiguous bytes, and a workgroup needs only G columns -- enough workgroups for every compute unit from 1024 columns on.
// Lanes next to each other take the ranges of one row, so that they read 64 (G = 8: 32) bytes in one piece: from a cache a compute unit
// takes 128 bytes per ns in pieces of 64, 75 in pieces of 32 and 38 in pieces of 16, where every lane has another row. Us with a row per lane -> now,
// weights in no cache, 1 | 2 | 8 rows: K 2048 x N 5152 6.8 -> 6.2 | 7.5 -> 6.5 | 9.0 -> 7.7; 4096 x 10304 18.4 -> 16.7 | 20.1 -> 17.1 | 21.0 -> 18.5;
// 5632 x 2048 7.9 -> 7.2 | 9.1 -> 7.4 | 9.9 -> 8.1; gated and normed 2048 x 5632 11.2 -> 10.3 | 12.4 -> 11.3 | 15.2 -> 13.8.
// The waves of a workgroup deal the K steps among themselves, U in flight each, and sum their blocks through LDS. The sums
// of four MFMAs, and then the waves', are added in 64 bits: the matrix instruction cuts the small ones of the 8 products that it adds at a
// time at 24 bits of the largest, and that already is the error of the vector unit's six lane exchanges (against 64 bits, one row
// of K 2048 | 7168: vector unit 7.5e-8 | 9.5e-8; one chain per wave and the waves one by one 9.7e-8 | 13.9e-8; now 6.4e-8 |
// 6.9e-8; 64 rows of 8 experts, K 7168: 9.5e-8, 25.4e-8, 7.0e-8). From nine rows on of one matrix, and from five per expert of several large
// ones, rows_mid.hip takes what it can (hy_rows_mid_takes); the figures of 33 rows are of before that.
// Us before -> after, weights in no cache, 1 | 8 | 33 rows: K 2048 x N 5152 11.1 -> 7.7 | 27.4 -> 10.7 | 54 -> 21; 4096 x 10304 42.6 ->
// 19.1 | 62.6 -> 26.6 | 108 -> 59; 2048 x 32000 49.6 -> 24.3 (5.4 TB/s) | 99 -> 29.4 | 67 -> 63; gated 2048 x 5632 17.2 -> 12.4 |
// 44.8 -> 16.0 | 82 -> 34; both products of 2 of 8 experts (4096 x 7168) for 1 | 8 tokens 105 -> 68 | 403 -> 230. With one output element
// per thread (a third of the epilogue's code to fetch) and the arguments read at once, one row: 2048 x 2048 5.2 -> 4.7, 2048 x 5152
// 7.9 -> 7.2, gated 5632 12.3 -> 11.5, 2048 x 32000 24.3 -> 22.7.
#include "hy_util.h"
#include "hybrid.h"
#include "row_act.h"

namespace jla {

JLA_DEV u32x4 rv_round8(const f32x4 a, const f32x4 b) {
  const float f[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  return pack8(f);
}

// The launch's arguments into registers at once: read where they are used, behind each other's branches, they are a chain of
// scalar loads at the start of a kernel that lasts a few microseconds.
JLA_DEV void rv_arguments(const RowLinear& p) {
  asm volatile("" ::"s"(p.a), "s"(p.lda), "s"(p.a_idx), "s"(p.a_scale), "s"(p.w), "s"(p.w_stride), "s"(p.N), "s"(p.K),
               "s"(p.out), "s"(p.ldo), "s"(p.dst_idx), "s"(p.offs), "s"(p.row_expert), "s"(p.R), "s"(p.a_div), "s"(p.tab));
}

// the expert of linear row r where every row has its own (0: one matrix); -1: none (an identity expert: nothing to compute)
JLA_DEV int rv_expert(const RowLinear& p, int r) {
  if (p.row_expert) {
    const int e = p.row_expert[r];
    return e < 0 || e >= p.E ? -1 : e;
  }
  if (p.tab) {  // choice r % top of token r / top, as the routing kernel reads the table
    int id = p.tab_ids[r / p.tab_top];
    id = id < 0 || id >= p.tab_V ? 0 : id;
    const int e = p.tab[(size_t)id * p.tab_top + r % p.tab_top];
    return e < 0 || e >= p.E ? 0 : e;
  }
  return 0;
}

// the table entry that the gated output column `col` of row r is multiplied by (gelu_gate_rows)
JLA_DEV float rv_table(const RowLinear& p, int r, int col) {
  int id = p.mul_ids[r];
  id = id < 0 || id >= p.mul_V ? 0 : id;
  const size_t at = (size_t)id * p.mul_ld + p.mul_col0 + col;
  return p.mul_bf16 ? bf2f(reinterpret_cast<const bf16_t*>(p.mul_table)[at]) : reinterpret_cast<const float*>(p.mul_table)[at];
}

constexpr int RV_WALK_ROWS = 2, RV_WALK_K = 4096;

// The sum of N partial sums in type T
template <class T, int N>
JLA_DEV float rv_sum(const float (&f)[N]) {
  T s[N];
#pragma unroll
  for (int i = 0; i < N; ++i) s[i] = f[i];
#pragma unroll
  for (int n = N / 2; n > 0; n /= 2)
#pragma unroll
    for (int i = 0; i < n; ++i) s[i] += s[i + n];
  return (float)s[0];
}

// The products of a lane of mfma16x16x32 whose A row SEG i + sg is column i, and whose B column SEG r + sg is row r, on K range sg: lane (c, q) holds
// A rows 4 q + 0..3 of B column c, of which those of range c % SEG count, the j-th of 4 / SEG (column q 4 / SEG + j)
template <int SEG>
JLA_DEV float rv_own(float v0, float v1, float v2, float v3, int c, int j) {
  if constexpr (SEG == 1) return j == 0 ? v0 : j == 1 ? v1 : j == 2 ? v2 : v3;
  const float lo = c & 1 ? v1 : v0, hi = c & 1 ? v3 : v2;
  if constexpr (SEG == 2) return j == 0 ? lo : hi;
  return c & 2 ? hi : lo;
}
// where they lie for column y and row x, range by range, among 4 / SEG planes of 64 lanes
template <int SEG>
JLA_DEV int rv_place(int x, int y) {
  constexpr int EL = 4 / SEG;
  return 64 * (y % EL) + 16 * (y / EL) + SEG * x;
}

// the better of two candidates of a maximum: the larger, ties to the lower index, a NaN never
JLA_DEV void rv_better(float& bv, int& bi, float v, int i) {
  if (v > bv || (v == bv && i < bi)) {
    bv = v;
    bi = i;
  }
}

// FORM of a kernel: -1, any call; else one of plain rows -- in place and order, of one matrix or the table's experts -- whose results go to
// fp32 rows in order through RowAct FORM % 8; RV_RES: with a pending residual add, RV_NORM: a norm, RV_MUL: the gate table, RV_ADD: onto the
// output, RV_ONE: one row per group. The branches that such a call does not take are not in its code: a launch of a few microseconds waits for
// the code on its path, some 0.13 us per KB. One row, weights in no cache, any call's code -> its own: 2048 x 2048 8.4 -> 5.9 KB, 4.1 -> 3.7 us;
// 2048 x 5152 5.5 -> 3.1 KB, 6.2 -> 5.8; walking, normed 2048 x 2048 9.8 -> 3.2 KB, 4.9 -> 4.3, 2048 x 32000 10.6 -> 3.6 KB, 22.8 -> 21.7; 4096 x 4096
// with a residual 10.3 -> 9.5. Over 11 to 13 shapes of K 512 to 4096 and N 1024 to 32000, in parts of the time in any call's code, one row: normed
// 0.92 (no activation, SwiGLU, clamped gate), a pending add 0.94, both 0.97 (up to 3072 columns 0.94, of 5152 and 10304 1.05 to 1.08, of more 0.97); on
// fp32 weights normed 0.97 (soft cap, clamped gate and none), a pending add 0.97 (none, SwiGLU), both 0.98, as it is or onto the output 0.99.
// Only these have one, with the greedy choice behind a norm and the gate table behind a pending add: a token's calls in the families that this was
// measured for. Squared ReLU, GELU gates, the soft cap without its choice on bf16 weights, results in bf16 and two walking rows keep any call's
// (those as a loop over the rows were smaller and slower: the first weights were waited for at its edge).
constexpr int RV_RES = 8, RV_NORM = 16, RV_ONE = 32, RV_MUL = 64, RV_ADD = 128;
constexpr int RV_GATE = HY_ACT_NONE + RV_RES + RV_ONE + RV_MUL;
template <int FORM>
JLA_DEV void rv_form(RowLinear& p) {
  if constexpr (FORM >= 0) {
    p.a_idx = p.dst_idx = p.offs = p.row_expert = nullptr;
    if (!(FORM & RV_MUL)) p.mul_ids = nullptr;
    p.a_scale = nullptr;
    p.out_bf16 = 0;
    p.add_out = (FORM & RV_ADD) != 0;
    p.act = FORM % 8;
    if (!(FORM & RV_RES)) p.res_y = nullptr;
    if (!(FORM & RV_NORM)) p.a_norm_w = nullptr;
  }
}
static int rv_form_of(const RowLinear& p, int rows_per_group) {
  const bool plain = !p.a_idx && !p.dst_idx && !p.offs && !p.row_expert && !p.a_scale && !p.out_bf16;
  return plain ? p.act + (p.res_y ? RV_RES : 0) + (p.a_norm_w ? RV_NORM : 0) + (rows_per_group == 1 || p.R == 1 ? RV_ONE : 0) +
                     (p.mul_ids ? RV_MUL : 0) + (p.add_out ? RV_ADD : 0)
               : -1;
}

// output column col of linear row r from its accumulators
JLA_DEV void rv_store(const RowLinear& p, int r, int col, float g, float v) {
  const size_t at = (size_t)(p.dst_idx ? p.dst_idx[r] : r) * p.ldo + col;
  float val = lr_act(p, g, v);
  if (p.mul_ids) val = hy_gelu_tanh(val) * rv_table(p, r, col);
  if (p.out_bf16) {
    reinterpret_cast<bf16_t*>(p.out)[at] = f2bf(val);
    return;
  }
  float* dst = reinterpret_cast<float*>(p.out) + at;
  *dst = p.add_out ? *dst + val : val;
}

// G: output columns of a tile, and rows of a pass per 16 MT / (16 / G); NT: tiles of a workgroup (gated: gate and up tiles
// alternate); MT: 16-row tiles (G = 16); U: K steps in flight per wave. NORM 1 (MT = 1): rows are RMS-normed with a gain
// first, in the order (a * scale) * gain of the norm kernel. SUM: the type that the MFMAs' sums are added in. XB: bytes of an activation.
// PIPE: a batch of loads goes out before the one ahead of it is waited for.
template <int G, int NT, int MT, int WAVES, int U, int NORM, class SUM, int XB, bool PIPE, int FORM = -1>
__global__ void __launch_bounds__(64 * WAVES) rows_gemv_kernel(RowLinear p, int rows_per_group, int gated) {
  if constexpr (FORM >= 0) gated = hy_act_gated(FORM % 8);
  static_assert(G == 16 || MT == 1, "several row tiles: whole 16-column tiles");
  constexpr int SEG = 16 / G;                // neighbouring K ranges of one MFMA
  constexpr int H = G == 16 ? 2 : 1;         // MFMAs of a K step (G = 16: the two halves of a 128-byte line)
  constexpr int STEP = 32 * SEG * H;         // K of a step
  constexpr bool WIDE = sizeof(SUM) > sizeof(float);
  // steps whose sums share an fp32 accumulator: up to four MFMAs, two of four rows and several tiles; SUM float: all of them
  constexpr int RUN = !WIDE ? U : (G == 4 && NT > 1 ? 2 : 4 / H);
  constexpr int ROWS = G * MT;               // rows of a pass
  using XNum = std::conditional_t<XB == 2, bf16_t, float>;
  constexpr int EL = 4 / SEG;                // products of a lane that count
  __shared__ __align__(16) float red[WAVES][NT * MT][64 * EL];
  __shared__ float stat[NORM ? WAVES : 1][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, q = lane >> 4;
  rv_form<FORM>(p);
  rv_arguments(p);
  // rows of this group: a fixed count, one row with its own expert, or (offs) every row of expert blockIdx.y
  int g0 = blockIdx.y * rows_per_group, g1 = min(g0 + rows_per_group, p.R), e = 0;
  if (p.offs) {
    e = blockIdx.y;
    g0 = p.offs[e];
    g1 = p.offs[e + 1];
  } else {
    e = rv_expert(p, g0);
    if (e < 0) return;
  }
  const int K = p.K, N = p.N, steps = (K + STEP - 1) / STEP;
  const int k0 = 8 * (c % SEG) + 8 * SEG * q;  // this lane's place in a step
  const bf16_t* wbase = reinterpret_cast<const bf16_t*>(p.w) + (size_t)e * p.w_stride;
  const bf16_t* wp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int T = blockIdx.x * NT + t;
    const int col = min(G * (gated ? T >> 1 : T) + c / SEG, N - 1);
    wp[t] = wbase + (size_t)(gated && (T & 1) ? N + col : col) * K;
  }
  for (int r0 = g0; r0 < g1; r0 += ROWS) {
    const int nr = min(ROWS, g1 - r0);
    const XNum* xp[MT];
    float xs[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int rr = r0 + min(16 * m + c / SEG, nr - 1);  // (surplus lanes repeat the last row; their results are dropped)
      xp[m] = reinterpret_cast<const XNum*>(p.a) + (size_t)(p.a_idx ? p.a_idx[rr] : (p.a_div > 1 ? rr / p.a_div : rr)) * p.lda;
      xs[m] = p.a_scale ? p.a_scale[rr] : 1.f;
    }
    // (a lane past the end of a ragged last step reads the row's start; its operands are zeroed before they are used)
    auto at = [&](int s, int h) {
      const int k = STEP * s + 32 * h + k0;
      return k < K ? k : 0;
    };
    if constexpr (NORM != 0) {
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
      for (int o = 1; o < 64; o <<= 1)
        if (o < SEG || o >= 16) ss += __shfl_xor(ss, o, 64);
      if (q == 0 && c % SEG == 0) stat[wave][c / SEG] = ss;
      __syncthreads();
      ss = 0.f;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) ss += stat[w][c / SEG];
      xs[0] = 1.f / sqrtf(ss / (float)K + p.a_norm_eps);
    }
    SUM acc[NT][MT][4];  // (64 bits cost little beside the stream: 8 rows, K 7168 x N 4096: 16.7 -> 17.0 us)
    f32x4 part[NT][MT];  // a run's own sums
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        part[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[t][m][i] = 0;
      }

    if constexpr (XB == 2 || PIPE) {
      struct Batch {
        u32x4 w[U][H][NT], x[U][H][MT][XB / 2];
      };
      auto load = [&](Batch& f, int s0) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int h = 0; h < H; ++h) {
            const int k = at(min(s0 + WAVES * u, steps - 1), h);  // (a step past the last one loads it again, unused)
#pragma unroll
            for (int t = 0; t < NT; ++t) f.w[u][h][t] = load_nt(reinterpret_cast<const u32x4*>(wp[t] + k));
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
              for (int i = 0; i < XB / 2; ++i) f.x[u][h][m][i] = *reinterpret_cast<const u32x4*>(xp[m] + k + 4 * i);
          }
      };
      auto use = [&](Batch& f, int s0) {
#pragma unroll
        for (int u0 = 0; u0 < U; u0 += RUN) {
          if (s0 + WAVES * u0 >= steps) break;  // (wave-uniform)
          if (WIDE) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
              for (int m = 0; m < MT; ++m) part[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
#pragma unroll
          for (int u = u0; u < (u0 + RUN < U ? u0 + RUN : U); ++u) {
            const int s = s0 + WAVES * u;
            if (s >= steps) break;  // (wave-uniform)
#pragma unroll
            for (int h = 0; h < H; ++h) {
              const bool ragged = STEP * s + 32 * (h + 1) * SEG > K;  // (wave-uniform: some lane's range ends before K does)
              const bool in = STEP * s + 32 * h + k0 < K;
              if (ragged) {
#pragma unroll
                for (int t = 0; t < NT; ++t) f.w[u][h][t] = in ? f.w[u][h][t] : u32x4{0, 0, 0, 0};
              }
#pragma unroll
              for (int m = 0; m < MT; ++m) {
                u32x4 x = f.x[u][h][m][0];
                if constexpr (XB == 4) {
                  f32x4 a = __builtin_bit_cast(f32x4, x), b = __builtin_bit_cast(f32x4, f.x[u][h][m][1]);
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
                  x = rv_round8(a, b);
                }
                if (ragged) x = in ? x : u32x4{0, 0, 0, 0};
#pragma unroll
                for (int t = 0; t < NT; ++t) part[t][m] = mfma16x16x32(f.w[u][h][t], x, part[t][m]);
              }
            }
          }
          if (WIDE) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
              for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[t][m][i] += part[t][m][i];
          }
        }
      };
      constexpr int D = WAVES * U;
      if constexpr (PIPE) {  // the next batch's loads go out before this one's are waited for; no branch joins in between
        Batch f, g;
        int s0 = wave;
        if (s0 < steps) {
          load(f, s0);
          for (;;) {
            if (s0 + D >= steps) {
              use(f, s0);
              break;
            }
            load(g, s0 + D);
            use(f, s0);
            s0 += D;
            if (s0 + D >= steps) {
              use(g, s0);
              break;
            }
            load(f, s0 + D);
            use(g, s0);
            s0 += D;
          }
        }
      } else {
        for (int s0 = wave; s0 < steps; s0 += D) {
          Batch f;
          load(f, s0);
          use(f, s0);
        }
      }
    } else {
      // The same loop for fp32 rows without a pipeline, written out: through load() and use() the compiler makes slower code of it (us, here |
      // there: one row of 1024 x 1024 3.5 | 4.0, 10304 x 2048 10.0 | 11.0, gated 2048 x 5632 11.5 | 13.6, 8 rows of 4096 x 14336 34.6 | 45.6; some
      // sorted rows a tenth faster, 64 of 8 experts of 2048 x 2816 30.3 | 28.3)
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
        for (int u0 = 0; u0 < U; u0 += RUN) {
          if (s0 + WAVES * u0 >= steps) break;  // (wave-uniform)
          if (WIDE) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
              for (int m = 0; m < MT; ++m) part[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
#pragma unroll
          for (int u = u0; u < (u0 + RUN < U ? u0 + RUN : U); ++u) {
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
                for (int t = 0; t < NT; ++t) part[t][m] = mfma16x16x32(wf[u][h][t], x, part[t][m]);
              }
            }
          }
          if (WIDE) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
              for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[t][m][i] += part[t][m][i];
          }
        }
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        float own[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) own[i] = WIDE ? (float)acc[t][m][i] : part[t][m][i];
#pragma unroll
        for (int j = 0; j < EL; ++j) red[wave][t * MT + m][64 * j + lane] = rv_own<SEG>(own[0], own[1], own[2], own[3], c, j);
      }
    __syncthreads();
    // one output element per thread: the epilogue's code, which a short launch has to fetch, stays small
    constexpr int PER = G * G;  // (column, row) pairs of a tile
    const int outs = (gated ? NT / 2 : NT) * MT * PER;
    for (int i = tid; i < outs; i += 64 * WAVES) {
      const int y = i % G, x = i / G % G, tm = i / PER, to = tm / MT, m = tm - to * MT;  // column, row; output tile, row tile
      const int row = 16 * m + x, col = G * (blockIdx.x * (gated ? NT / 2 : NT) + to) + y;
      if (row >= nr || col >= N) continue;
      const int slot = (gated ? 2 * to : to) * MT + m;
      auto total = [&](int at) {
        float f[SEG * WAVES];
        const int from = rv_place<SEG>(x, y);
#pragma unroll
        for (int w = 0; w < WAVES; ++w)
#pragma unroll
          for (int sg = 0; sg < SEG; ++sg) f[sg * WAVES + w] = red[w][at][from + sg];
        return rv_sum<SUM>(f);
      };
      const float g = total(slot), v = gated ? total(slot + MT) : 0.f;
      rv_store(p, r0 + row, col, g, v);
    }
    __syncthreads();
  }
}

// v plus that of the lane whose number differs in the bits of a DPP control (quad_perm 0xb1: 1, 0x4e: 2; row_half_mirror 0x141 and row_mirror 0x140
// pair the halves once those hold one sum)
template <int CTRL>
JLA_DEV double rw_add(double v) {
  const u32x2 b = __builtin_bit_cast(u32x2, v);
  const u32x2 o = {(uint32_t)__builtin_amdgcn_update_dpp(0, (int)b[0], CTRL, 0xf, 0xf, true), (uint32_t)__builtin_amdgcn_update_dpp(0, (int)b[1], CTRL, 0xf, 0xf, true)};
  return v + __builtin_bit_cast(double, o);
}

// One or two rows of up to 128 numbers: K is one step, so a wave has whole tiles and nothing passes through LDS. What bounds it: the launch and
// one trip to memory. 0.8 KB of code for the vector GEMV's 9: one | two rows of 2048 x 64 3.1 | 3.7 -> 2.1 | 2.2 us, 4096 x 64 3.4 | 4.1 -> 2.2 |
// 2.3, 512 x 32 2.4 | 2.8 -> 2.0 (a launch that does nothing takes 1.9).
constexpr int RV_SHORT_STEP = 128, RV_SHORT_NT = 2;
__global__ void __launch_bounds__(256) rows_short_kernel(RowLinear p) {
  rv_form<HY_ACT_NONE>(p);
  const int lane = threadIdx.x & 63, c = lane & 15, q = lane >> 4, k0 = 8 * (c % 4) + 32 * q;
  const int T = (blockIdx.x * 4 + (threadIdx.x >> 6)) * RV_SHORT_NT;
  const bool in = k0 < p.K;
  const bf16_t* w = reinterpret_cast<const bf16_t*>(p.w) + (in ? k0 : 0);
  u32x4 wf[RV_SHORT_NT];
#pragma unroll
  for (int t = 0; t < RV_SHORT_NT; ++t) wf[t] = load_nt(reinterpret_cast<const u32x4*>(w + (size_t)min(4 * (T + t) + c / 4, p.N - 1) * p.K));
  const f32x4* x = reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(p.a) + (size_t)min(c / 4, p.R - 1) * p.lda + (in ? k0 : 0));
  const u32x4 xr = in ? rv_round8(x[0], x[1]) : u32x4{0, 0, 0, 0};
#pragma unroll
  for (int t = 0; t < RV_SHORT_NT; ++t) {
    const f32x4 d = mfma16x16x32(in ? wf[t] : u32x4{0, 0, 0, 0}, xr, f32x4{0.f, 0.f, 0.f, 0.f});
    // lane: row c / 4, column q of the tile, K range c % 4
    double v = rv_own<4>(d[0], d[1], d[2], d[3], c, 0);
    v = rw_add<0xb1>(v);
    v = rw_add<0x4e>(v);
    const int col = 4 * (T + t) + q;
    if (c % 4 == 0 && c / 4 < p.R && col < p.N) reinterpret_cast<float*>(p.out)[(size_t)(c / 4) * p.ldo + col] = (float)v;
  }
}

// Linear row r as the product reads it; K <= 1024 V. Every thread of the workgroup (256)
// holds columns 4 tid + 1024 u. load() only issues loads: the weights of the first steps are issued behind
// them, and a wave's loads return in order. With res_y: x + rms(ysc * sum of the row's nsum rows of y) * w, in the
// norm_residual kernel's order, also written to res_out by the launch's first workgroup.
JLA_DEV float rv_block_sum(float v, float (*stat)[16]) {
  v = wave_sum(v);
  __syncthreads();  // (the sum before is read)
  if ((threadIdx.x & 63) == 0) stat[threadIdx.x >> 6][0] = v;
  __syncthreads();
  return stat[0][0] + stat[1][0] + stat[2][0] + stat[3][0];
}
// MIX: the normed row is then blended with the row before it (RowParts), row 0 of the launch's parts also stored as it was.
template <int V, int MIX>
struct RvRow {
  f32x4 x[V], y[V], g[V], w[V], before[MIX ? V : 1], mu[MIX ? V : 1];
  float scale;
  JLA_DEV void load_mix(const RowParts& t, int part, int r, int K, int tid) {
    if constexpr (MIX) {
      const float* m = t.mu + (size_t)max(t.mix[part], 0) * K;
#pragma unroll
      for (int u = 0; u < V; ++u) {
        const int k = 4 * tid + 1024 * u < K ? 4 * tid + 1024 * u : 0;
        before[u] = *reinterpret_cast<const f32x4*>(t.prev + (size_t)r * K + k);
        mu[u] = *reinterpret_cast<const f32x4*>(m + k);
      }
    }
  }
  JLA_DEV f32x4 mixed(const RowParts& t, int part, f32x4 v, int u, int r, int K, int k) const {
    if constexpr (MIX) {
      if (blockIdx.x == 0 && k < K) *reinterpret_cast<f32x4*>(t.row + (size_t)r * K + k) = v;
      if (t.mix[part] >= 0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = fmaf(before[u][j] - v[j], mu[u][j], v[j]);
      }
    }
    return v;
  }
  JLA_DEV void load(const RowLinear& p, int r, int K, int tid) {
    const int src = p.a_idx ? p.a_idx[r] : (p.a_div > 1 ? r / p.a_div : r);
    const float* xp = reinterpret_cast<const float*>(p.a) + (size_t)src * p.lda;
    scale = p.a_scale ? p.a_scale[r] : 1.f;
    int k[V];
#pragma unroll
    for (int u = 0; u < V; ++u) {
      k[u] = 4 * tid + 1024 * u < K ? 4 * tid + 1024 * u : 0;
      x[u] = *reinterpret_cast<const f32x4*>(xp + k[u]);
      y[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if (p.a_norm_w) {
#pragma unroll
      for (int u = 0; u < V; ++u) {
        if (p.a_norm_one) {
          const float w0 = p.a_norm_w[0];
          g[u] = f32x4{w0, w0, w0, w0};
        } else {
          g[u] = *reinterpret_cast<const f32x4*>(p.a_norm_w + k[u]);
        }
      }
    }
    if (p.res_y) {
      const float* yp = p.res_y + (size_t)src * p.res_nsum * K;
#pragma unroll
      for (int u = 0; u < V; ++u) y[u] = *reinterpret_cast<const f32x4*>(yp + k[u]);
      if (p.res_w_vec) {
#pragma unroll
        for (int u = 0; u < V; ++u) w[u] = *reinterpret_cast<const f32x4*>(p.res_w + k[u]);
      } else {
        const float w0 = p.res_w[0];
#pragma unroll
        for (int u = 0; u < V; ++u) w[u] = f32x4{w0, w0, w0, w0};
      }
      for (int n = 1; n < p.res_nsum; ++n) {
#pragma unroll
        for (int u = 0; u < V; ++u) y[u] += *reinterpret_cast<const f32x4*>(yp + (size_t)n * K + k[u]);
      }
    }
  }
  // put(u, k, v): this thread's numbers v at columns k, which may be past K
  template <class Put>
  JLA_DEV void stage(const RowLinear& p, int r, int K, int tid, float (*stat)[16], const RowParts& t, int part, Put put) {
    if (p.res_y) {
      float ss = 0.f;
#pragma unroll
      for (int u = 0; u < V; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          y[u][j] *= p.res_ysc;
          ss = 4 * tid + 1024 * u < K ? fmaf(y[u][j], y[u][j], ss) : ss;
        }
      const float sc = 1.f / sqrtf(rv_block_sum(ss, stat) / (float)K + p.res_eps);
      // (with several linear rows of a source row, its first writes)
      const int src = p.a_idx ? p.a_idx[r] : (p.a_div > 1 ? r / p.a_div : r);
      const bool keep = blockIdx.x == 0 && (p.a_div <= 1 || r % p.a_div == 0);
#pragma unroll
      for (int u = 0; u < V; ++u) {
        const int k = 4 * tid + 1024 * u;
#pragma unroll
        for (int j = 0; j < 4; ++j) x[u][j] += y[u][j] * sc * w[u][j];
        if (keep && k < K) *reinterpret_cast<f32x4*>(p.res_out + (size_t)src * K + k) = x[u];
      }
    }
    if (p.a_norm_w) {
      float ss = 0.f;
#pragma unroll
      for (int u = 0; u < V; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) ss = 4 * tid + 1024 * u < K ? fmaf(x[u][j], x[u][j], ss) : ss;
      scale = 1.f / sqrtf(rv_block_sum(ss, stat) / (float)K + p.a_norm_eps);
    }
#pragma unroll
    for (int u = 0; u < V; ++u) {
      const int k = 4 * tid + 1024 * u;
      f32x4 v = x[u] * scale;
      if (p.a_norm_w) v *= g[u];
      put(u, k, mixed(t, part, v, u, r, K, k));
    }
  }
};

// One or two rows, K <= 128 WAVES U: a wave's share of K is U steps, so the rows' operands stay in its registers, and a
// workgroup walks over groups of NT tiles with the next group's weights issued as this one's are consumed. The rows pass
// through LDS once per workgroup, where a pending residual add (res_y) and the norm are applied behind the first weights.
// grid (workgroups, linear rows with their own expert, else 1). PARTS: several matrices (RowParts) that read the same rows, each with
// a run of the workgroups, the rows blended for it as they are staged.
template <int NT, int U, int V, int PARTS, int BEST = 0, int FORM = -1>
__global__ void __launch_bounds__(256) rows_gemv_walk_kernel(RowLinear p, int rows_per_group, int gated, int tgroups, RowParts parts) {
  constexpr int G = 4, SEG = 4, WAVES = 4, STEP = 128;
  extern __shared__ f32x4 staged[];  // [rows][K]
  __shared__ __align__(16) float red[2][WAVES][NT][64];
  __shared__ float stat[WAVES][16];
  __shared__ float2 cand[BEST ? NT * 4 * RV_WALK_ROWS : 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, q = lane >> 4;
  float bv = -INFINITY;  // BEST: this thread's candidate
  int bi = 0x7fffffff;
  int part = 0, tg = blockIdx.x, walk = gridDim.x;  // this workgroup's first group of tiles, and from one to its next
  if constexpr (PARTS) {
    rv_form<FORM>(p);
    if constexpr (FORM >= 0) {
      gated = 0;
      p.tab = nullptr;
    }
    while (part + 1 < parts.n && tg >= parts.first[part + 1]) ++part;
    tg -= parts.first[part];
    walk = parts.first[part + 1] - parts.first[part];
    tgroups = parts.tgroups[part];
    p.w = parts.w[part];
    p.N = parts.N[part];
    p.out = parts.out[part];
    p.ldo = parts.ldo[part];
    p.act = parts.cap[part] > 0.f ? HY_ACT_SOFTCAP : HY_ACT_NONE;
    p.act_limit = parts.cap[part];
  } else {
    rv_form<FORM>(p);
    if constexpr (FORM >= 0) gated = hy_act_gated(FORM % 8);
    rv_arguments(p);
  }
  const int r0 = blockIdx.y * rows_per_group, nr = FORM >= 0 && (FORM & RV_ONE) ? 1 : min(rows_per_group, p.R - r0);
  const int e = rv_expert(p, r0);
  if (e < 0) return;  // (the whole workgroup)
  const int K = p.K, N = p.N, steps = (K + STEP - 1) / STEP, k0 = 8 * (c % SEG) + 8 * SEG * q;
  const bf16_t* wbase = reinterpret_cast<const bf16_t*>(p.w) + (size_t)e * p.w_stride;
  // this lane's place in step u (a lane past the end of K reads the row's start; its operand is zero)
  auto at = [&](int u) {
    const int k = STEP * (wave + WAVES * u) + k0;
    return k < K ? k : 0;
  };
  u32x4 wf[U][NT];
  auto weight_row = [&](int tg, int t) {
    const int T = tg * NT + t, col = min(G * (gated ? T >> 1 : T) + c / SEG, N - 1);
    return wbase + (size_t)(gated && (T & 1) ? N + col : col) * K;
  };
  RvRow<V, PARTS> row;
  row.load(p, r0, K, tid);
  row.load_mix(parts, part, r0, K, tid);
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const bf16_t* w = weight_row(tg, t);
#pragma unroll
    for (int u = 0; u < U; ++u) wf[u][t] = load_nt(reinterpret_cast<const u32x4*>(w + at(u)));
  }
  auto to_row = [&](int i) {
    return [=](int, int k, f32x4 v) {
      if (k < K) staged[((size_t)i * K + k) / 4] = v;
    };
  };
  row.stage(p, r0, K, tid, stat, parts, part, to_row(0));
  if (nr > 1) {
    row.load(p, r0 + 1, K, tid);
    row.load_mix(parts, part, r0 + 1, K, tid);
    row.stage(p, r0 + 1, K, tid, stat, parts, part, to_row(1));
  }
  __syncthreads();
  u32x4 xr[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {  // (surplus B columns repeat the last row; their results are dropped)
    const f32x4* x = staged + ((size_t)min(c / SEG, nr - 1) * K + at(u)) / 4;
    xr[u] = STEP * (wave + WAVES * u) + k0 < K ? rv_round8(x[0], x[1]) : u32x4{0, 0, 0, 0};
  }
  for (int buf = 0; tg < tgroups; tg += walk, buf ^= 1) {
    const int next = tg + walk;
    const bool more = next < tgroups;  // (workgroup-uniform)
    f32x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const bf16_t* w = more ? weight_row(next, t) : wbase;  // (after the last group: one line, unused)
      acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < U; ++u) {
        // (past the end of K both operands are zero: an infinite weight must not meet a zero)
        const bool in = STEP * (wave + WAVES * u) + k0 < K;
        acc[t] = mfma16x16x32(in ? wf[u][t] : u32x4{0, 0, 0, 0}, xr[u], acc[t]);
        wf[u][t] = load_nt(reinterpret_cast<const u32x4*>(w + (more ? at(u) : 0)));
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) red[buf][wave][t][lane] = rv_own<SEG>(acc[t][0], acc[t][1], acc[t][2], acc[t][3], c, 0);
    __syncthreads();  // (one per group: the other buffer's readers are past the barrier before)
    const int outs = (gated ? NT / 2 : NT) * nr * G;
    if (tid < outs) {
      const int y = tid % G, to = tid / G / nr, x = tid / G - to * nr, slot = gated ? 2 * to : to;
      const int col = G * (tg * (gated ? NT / 2 : NT) + to) + y;
      auto total = [&](int at) {
        float f[4 * WAVES];
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(&red[buf][w][at][rv_place<SEG>(x, y)]);
#pragma unroll
          for (int sg = 0; sg < 4; ++sg) f[sg * WAVES + w] = v[sg];
        }
        return rv_sum<double>(f);
      };
      const float g = total(slot), v = gated ? total(slot + 1) : 0.f;
      if constexpr (BEST) {
        const float val = lr_act(p, g, v);
        if (col < N && val > bv) {  // (a thread's columns ascend; -inf, as a NaN, is never chosen)
          bv = val;
          bi = col;
        }
      } else {
        if (col < N) rv_store(p, r0 + x, col, g, v);
      }
    }
  }
  if constexpr (BEST) {  // (threads below NT nr G hold candidates, row (tid / G) % nr)
    const int outs = NT * nr * G;
    __syncthreads();
    if (tid < outs) cand[tid] = make_float2(bv, __int_as_float(bi));
    __syncthreads();
    if (tid < nr) {
      float2 best = make_float2(-INFINITY, __int_as_float(0x7fffffff));
      for (int i = 0; i < outs; ++i) {
        if (i / G % nr != tid) continue;
        int at = __float_as_int(best.y);
        rv_better(best.x, at, cand[i].x, __float_as_int(cand[i].y));
        best.y = __int_as_float(at);
      }
      p.best[(size_t)(r0 + tid) * gridDim.x + blockIdx.x] = best;
    }
  }
}

// One or two rows on fp32 weights, K <= 1024 V, each number multiplied as it is: a thread's numbers of the rows stay in its registers
// (columns 4 tid + 1024 u, whole lines per wave), a workgroup walks over groups of NT weight rows (gated: gate and up alternate) with the
// next group's loads issued as this one's are consumed, and the first group's go out ahead of the norm. What bounds it: the weight
// stream. lr_gemv_kernel, a wave per column or four, reads a row and its norm before the first weight, every wave again. Us there -> here,
// weights in no cache, one row: 2048 x 2048 6.1 -> 5.4, 2048 x 5632 12.0 -> 10.5, normed 3072 x 2048 8.8 -> 7.2, normed 8224 x 2048 20.9 -> 13.6, gated
// and normed 5632 x 2048 22.3 -> 17.6, normed 32000 x 2048 53.8 -> 42.9 (6.1 TB/s); errors against 64 bits 1.2e-7 to 1.8e-7 -> 0.5e-7 to 1.0e-7 (the 256
// threads' parts added by lane exchanges in 32 bits: 0.8e-7 to 1.2e-7, and 1 to 3 % slower). The same kernel on bf16 weights is as fast as the
// matrix cores' there, not faster (normed 8224 x 2048 9.6 | 8.8, 2048 x 2048 4.2 | 4.4, 2048 x 5632 7.9 | 8.3).
// grid and PARTS as in rows_gemv_walk_kernel; V > 4: rows as they are.
template <int NT, int V, int RW, int PARTS, int FORM = -1>
__global__ void __launch_bounds__(256) rows_walk_f32_kernel(RowLinear p, int rows_per_group, int gated, int tgroups, RowParts parts) {
  static_assert(NT * RW <= 16, "sixteen threads per sum");
  __shared__ float red[2][NT * RW][256];
  __shared__ float stat[4][16];
  const int tid = threadIdx.x;
  int part = 0, tg = blockIdx.x, walk = gridDim.x;
  rv_form<FORM>(p);
  if constexpr (FORM >= 0) gated = !PARTS && hy_act_gated(FORM % 8);
  if constexpr (PARTS) {
    if constexpr (FORM >= 0) p.tab = nullptr;
    while (part + 1 < parts.n && tg >= parts.first[part + 1]) ++part;
    tg -= parts.first[part];
    walk = parts.first[part + 1] - parts.first[part];
    tgroups = parts.tgroups[part];
    p.w = parts.w[part];
    p.N = parts.N[part];
    p.out = parts.out[part];
    p.ldo = parts.ldo[part];
    p.act = parts.cap[part] > 0.f ? HY_ACT_SOFTCAP : HY_ACT_NONE;
    p.act_limit = parts.cap[part];
  } else {
    rv_arguments(p);
  }
  const int r0 = blockIdx.y * rows_per_group, nr = min(rows_per_group, p.R - r0);
  const int e = rv_expert(p, r0);
  if (e < 0) return;  // (the whole workgroup)
  const int K = p.K, N = p.N;
  const float* wbase = reinterpret_cast<const float*>(p.w) + (size_t)e * p.w_stride;
  auto in = [&](int u) { return 4 * tid + 1024 * u < K; };
  auto weight_row = [&](int tg, int t) {  // this thread's first numbers of it (past the end of K: the row's start, which counts as zero)
    const int T = tg * NT + t, col = min(gated ? T >> 1 : T, N - 1);
    return wbase + (size_t)(gated && (T & 1) ? N + col : col) * K;
  };
  auto at = [&](int u) { return in(u) ? 4 * tid + 1024 * u : 0; };
  f32x4 wf[V][NT], x[RW][V];
  auto weights = [&](int tg) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const float* w = weight_row(tg, t);
#pragma unroll
      for (int u = 0; u < V; ++u) wf[u][t] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(w + at(u)));
    }
  };
  if constexpr (V > 4) {
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      const int row = r0 + min(r, nr - 1), src = p.a_idx ? p.a_idx[row] : (p.a_div > 1 ? row / p.a_div : row);
      const float* xp = reinterpret_cast<const float*>(p.a) + (size_t)src * p.lda;
#pragma unroll
      for (int u = 0; u < V; ++u) x[r][u] = *reinterpret_cast<const f32x4*>(xp + at(u));
    }
    weights(tg);
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      const float scale = p.a_scale ? p.a_scale[r0 + min(r, nr - 1)] : 1.f;
#pragma unroll
      for (int u = 0; u < V; ++u) x[r][u] = in(u) ? x[r][u] * scale : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  } else {
    RvRow<V, PARTS> row;
    row.load(p, r0, K, tid);
    row.load_mix(parts, part, r0, K, tid);
    weights(tg);
    row.stage(p, r0, K, tid, stat, parts, part, [&](int u, int k, f32x4 v) { x[0][u] = k < K ? v : f32x4{0.f, 0.f, 0.f, 0.f}; });
    if constexpr (RW > 1) {  // (a single row is there twice; the second result is dropped)
      const int second = r0 + nr - 1;
      row.load(p, second, K, tid);
      row.load_mix(parts, part, second, K, tid);
      row.stage(p, second, K, tid, stat, parts, part, [&](int u, int k, f32x4 v) { x[1][u] = k < K ? v : f32x4{0.f, 0.f, 0.f, 0.f}; });
    }
  }
  for (int buf = 0; tg < tgroups; tg += walk, buf ^= 1) {
    const int next = tg + walk;
    const bool more = next < tgroups;  // (workgroup-uniform)
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const float* w = more ? weight_row(next, t) : wbase;  // (after the last group: one line, unused)
      float a[RW][2];  // even and odd numbers
#pragma unroll
      for (int r = 0; r < RW; ++r) a[r][0] = a[r][1] = 0.f;
#pragma unroll
      for (int u = 0; u < V; ++u) {
        const f32x4 f = in(u) ? wf[u][t] : f32x4{0.f, 0.f, 0.f, 0.f};  // (an infinite weight must not meet a zero)
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
          for (int j = 0; j < 4; ++j) a[r][j & 1] = fmaf(f[j], x[r][u][j], a[r][j & 1]);
        wf[u][t] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(w + (more ? at(u) : 0)));
      }
#pragma unroll
      for (int r = 0; r < RW; ++r) red[buf][t * RW + r][tid] = a[r][0] + a[r][1];
    }
    __syncthreads();  // (one per group: the other buffer's readers are past the barrier before)
    // sixteen threads to a sum, its 256 parts added in 64 bits
    const int i = tid >> 4, sub = tid & 15;
    if (i < NT * RW) {  // (whole rows of 16 lanes; gated: gate and up are rows 16 RW lanes apart, in one wave)
      float f[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) f[j] = red[buf][i][16 * j + sub];
      double d[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) d[j] = f[j];
#pragma unroll
      for (int n = 8; n > 0; n /= 2)
#pragma unroll
        for (int j = 0; j < n; ++j) d[j] += d[j + n];
      d[0] = rw_add<0xb1>(d[0]);
      d[0] = rw_add<0x4e>(d[0]);
      d[0] = rw_add<0x141>(d[0]);
      d[0] = rw_add<0x140>(d[0]);
      const float g = (float)d[0], v = NT > 1 && gated ? __shfl_xor(g, 16 * RW, 64) : 0.f;
      const int r = i % RW, t = i / RW, col = tg * (gated ? NT / 2 : NT) + (gated ? t >> 1 : t);
      if (sub == 0 && !(gated && (t & 1)) && r < nr && col < N) rv_store(p, r0 + r, col, g, v);
    }
  }
}

// up to 64 rows, and up to 32 of a wide output, whose tiles fill the chip (64 rows x 32000 columns, K 2048: 70 us on the
// tiles, 82 here); a short K is over before the waves' sum pays (K 64: one row 3.2 us on the vector unit, 3.6 here, 64 rows
// 4.8 on the tiles, 5.3 here), and with very many columns the tiles stream it as fast (9 | 17 | 32 rows of K 256 x N 32000: weights in
// no cache 9.9 | 14.3 | 16.5 us here, 10.6 | 11.3 | 12.4 on the tiles, in a cache 9.3 | 13.0 | 15.5 and 6.8 | 7.5 | 8.7; N 16384, no
// cache: 6.4 | 8.3 | 9.8 here, 8.7 | 9.5 | 10.4 there; K 512 x N 32000: 10.8 | 15.5 | 17.6, 17.7 | 18.8 | 19.8).
// Rows with an expert of their own and no offsets: as many as the vector unit's form takes.
constexpr int RV_MAX_ROWS = 64, RV_MAX_WIDE_ROWS = 32, RV_WIDE = 16384, RV_MAX_NORM_ROWS = 2;
constexpr int RV_SHORT_K = 512, RV_SHORT_WIDE = 20480;
constexpr int RV_PAIR_K = 1024;

// Rows that are bf16 already (their bytes beside the weights' are what bounds more than two rows: 8 rows of fp32 are twice the bytes of
// the 8 columns that read them): three to eight of one matrix, or that many of each of several.
constexpr int RV_MIN_ROWS16 = 3, RV_MAX_ROWS16 = 8;

static bool rv_takes16(const RowLinear& p) {
  auto aligned = [](const void* x) { return ((uintptr_t)x & 15) == 0; };
  const int rows = p.offs ? p.even_rows : p.R;
  return p.wbf16 && p.a_bf16 && rows >= RV_MIN_ROWS16 && rows <= RV_MAX_ROWS16 && p.R <= RV_MAX_ROWS && (p.offs || p.E == 1) && !p.row_expert &&
         !p.tab && !p.a_scale && !p.a_norm_w && !p.res_y && !p.best && p.a_div <= 1 && p.K % 8 == 0 && p.K >= 64 && p.lda % 8 == 0 &&
         p.w_stride % 8 == 0 && aligned(p.a) && aligned(p.w) && !(p.add_out && p.out_bf16);
}

// fp32 weights: one or two rows of one matrix, or up to eight with an expert each; with a norm or a pending residual add as far as those
// stay in registers. A short K ends before the waves' sum pays (us, vector unit | here: one row, K 256 | 512 x N 2048 3.7 | 3.6, 4.1 | 3.7; two
// rows, K 256 | 512 | 1024 x N 2048 4.3 | 4.4, 4.6 | 4.7, 5.7 | 5.2, K 256 x N 32000 17.0 | 24.1).
constexpr int RV_F32_MIN_K = 512, RV_F32_MIN_K2 = 1024, RV_F32_MAX_K = 8192;
static bool rv_takes32(const RowLinear& p) {
  auto aligned = [](const void* x) { return ((uintptr_t)x & 15) == 0; };
  const bool each = p.tab || p.row_expert;
  return !p.wbf16 && !p.a_bf16 && !p.out_bf16 && !p.offs && !p.best && (each ? p.R <= HY_GEMV_MAX_R : (p.E == 1 && p.R <= RV_WALK_ROWS)) &&
         p.K % 4 == 0 && p.K >= (each || p.R == 1 ? RV_F32_MIN_K : RV_F32_MIN_K2) && p.K <= (p.a_norm_w || p.res_y ? RV_WALK_K : RV_F32_MAX_K) && p.lda % 4 == 0 && p.w_stride % 4 == 0 &&
         aligned(p.a) && aligned(p.w) && (!p.a_norm_w || (!p.a_scale && !each && (p.a_norm_one || aligned(p.a_norm_w))));
}

// rows_short_kernel's calls: few rows as they are, one matrix, more than a few columns (a router stays on the vector unit)
static bool rv_short(const RowLinear& p) {
  auto aligned = [](const void* x) { return ((uintptr_t)x & 15) == 0; };
  return p.wbf16 && !p.a_bf16 && p.R >= 1 && p.R <= RV_WALK_ROWS && p.E == 1 && !p.tab && rv_form_of(p, p.R) >= 0 && (rv_form_of(p, p.R) & ~RV_ONE) == HY_ACT_NONE && !p.best && p.a_div <= 1 &&
         p.K % 8 == 0 && p.K >= 8 && p.K <= RV_SHORT_STEP && p.N >= 64 && p.lda % 4 == 0 && aligned(p.a) && aligned(p.w);
}

bool hy_rows_gemv_takes(const RowLinear& p) {
  if (rv_short(p)) return true;
  if (!p.wbf16) return rv_takes32(p);
  if (p.a_bf16 || p.out_bf16) return rv_takes16(p);
  auto aligned = [](const void* x) { return ((uintptr_t)x & 15) == 0; };
  return p.wbf16 && p.R <= (p.N >= RV_WIDE ? RV_MAX_WIDE_ROWS : RV_MAX_ROWS) &&
         (p.offs || p.tab || (p.row_expert ? p.R <= HY_GEMV_MAX_R : p.E == 1)) && p.K % 8 == 0 &&
         p.K >= (p.R <= 2 ? 256 : (p.R <= 32 ? 64 : 128)) &&
         !(p.R > HY_GEMV_MAX_R && p.E == 1 && !p.offs && p.K < RV_SHORT_K && p.N >= RV_SHORT_WIDE) && p.lda % 4 == 0 && p.w_stride % 8 == 0 && aligned(p.a) && aligned(p.w) &&
         (!p.a_norm_w || (p.R <= RV_MAX_NORM_ROWS && !p.a_scale && !p.offs && !p.row_expert && (p.a_norm_one || aligned(p.a_norm_w))));
}

// One or two normed rows, or with a pending residual add, walk: the plain form would read them twice, the norm ahead of the
// first weight (RMS norm and product, K 2048 x N 2048 | 5152 | 8224 | 32000 | gated 5632: 6.1 | 9.5 | 12.3 | 34.6 | 13.5 us in the
// plain form, 5.3 | 7.5 | 9.7 | 23.0 | 10.8 walking; K 4096 x 10304: 26.1 -> 17.8). Rows as they are gain nothing from it (4.7 | 7.2 |
// 9.3 | 22.7 | 11.5 plain, 5.2 | 7.5 | 9.8 | 22.7 | 11.0 walking). Further rows would not fit the registers.
static bool rv_walks(const RowLinear& p, int rows) {
  return (p.a_norm_w || p.res_y) && !p.offs && rows <= RV_WALK_ROWS && p.K <= RV_WALK_K;
}

// A pending residual add (res_y) exists in the walking form only: the caller asks first.
bool hy_rows_gemv_takes_residual(const RowLinear& p) {
  auto aligned = [](const void* x) { return ((uintptr_t)x & 15) == 0; };
  return hy_rows_gemv_takes(p) && rv_walks(p, p.row_expert || p.tab ? 1 : p.R) && p.R <= RV_WALK_ROWS * (p.a_div > 1 ? p.a_div : 1) &&
         aligned(p.res_y) && aligned(p.res_out) && (!p.res_w_vec || aligned(p.res_w));
}

bool hy_rows_parts_takes(const RowLinear& p, const RowParts& t) {
  auto aligned = [](const void* x) { return ((uintptr_t)x & 15) == 0; };
  bool ok = p.R >= 1 && p.R <= RV_WALK_ROWS && p.a_norm_w && p.K % 8 == 0 && p.K >= 256 && p.K <= RV_WALK_K && p.lda % 4 == 0 && aligned(p.a) &&
            aligned(p.a_norm_w) && aligned(t.prev) && aligned(t.mu) && aligned(t.row) && t.n >= 1 && t.n <= RV_MAX_PARTS;
  for (int i = 0; ok && i < t.n; ++i) ok = t.N[i] >= 1 && aligned(t.w[i]);
  return ok;
}

// What the launch saves: the norm and blend of one row, four products of its blends, a low-rank product of the fifth and a product of
// the row itself (K 2048; N 4 x 2048, 64, 3072) were four launches.
int hy_rows_parts(const RowLinear& p, const RowParts& parts, hipStream_t s) {
  if (!hy_rows_parts_takes(p, parts)) return -1;
  RowParts t = parts;
  const int occ = p.K <= 2048 ? 4 : 2, per = p.wbf16 ? 8 : (p.K <= 2048 ? 4 : 2);  // weight rows of a group
  long long all = 0;
  for (int i = 0; i < t.n; ++i) all += t.tgroups[i] = (t.N[i] + per - 1) / per;
  const int rounds = (int)((all + 256 * occ - 1) / (256 * occ));
  t.first[0] = 0;
  for (int i = 0; i < t.n; ++i) t.first[i + 1] = t.first[i] + (t.tgroups[i] + rounds - 1) / rounds;
  const dim3 grid(t.first[t.n], 1);
  if (!p.wbf16) {
    if (p.K <= 2048) {
      if (p.R == 1) rows_walk_f32_kernel<4, 2, 1, 1, RV_NORM><<<grid, 256, 0, s>>>(p, p.R, 0, 0, t);
      else rows_walk_f32_kernel<4, 2, 2, 1><<<grid, 256, 0, s>>>(p, p.R, 0, 0, t);
    } else if (p.R == 1) {
      rows_walk_f32_kernel<2, 4, 1, 1, RV_NORM><<<grid, 256, 0, s>>>(p, p.R, 0, 0, t);
    } else {
      rows_walk_f32_kernel<2, 4, 2, 1><<<grid, 256, 0, s>>>(p, p.R, 0, 0, t);
    }
    JLA_CHECK_LAUNCH();
    return 0;
  }
  const unsigned lds = (unsigned)(p.R * p.K * sizeof(float));
  // (its rows are in place and order; one row's form without the second's code)
  if (p.R == 1 && p.K <= 2048) rows_gemv_walk_kernel<2, 4, 2, 1, 0, RV_ONE + RV_NORM><<<grid, 256, lds, s>>>(p, 1, 0, 0, t);
  else if (p.R == 1) rows_gemv_walk_kernel<2, 8, 4, 1, 0, RV_ONE + RV_NORM><<<grid, 256, lds, s>>>(p, 1, 0, 0, t);
  else if (p.K <= 2048) rows_gemv_walk_kernel<2, 4, 2, 1><<<grid, 256, lds, s>>>(p, p.R, 0, 0, t);
  else rows_gemv_walk_kernel<2, 8, 4, 1><<<grid, 256, lds, s>>>(p, p.R, 0, 0, t);
  JLA_CHECK_LAUNCH();
  return 0;
}

// workgroups of the walking form over the columns (of one expert), and the groups of tiles they walk
static bool rv_walk_grid(const RowLinear& p, int groups, int& wnt, long long& tg, long long& wgs) {
  // two tiles per step from a few workgroups for every compute unit on; as many workgroups as are resident (four of 88
  // registers per unit, or two of 156, K > 2048), with equally many steps each
  const int gated = hy_act_gated(p.act), occ = p.K <= 2048 ? 4 : 2;
  const long long tiles = (gated ? 2LL : 1LL) * ((p.N + 3) / 4);
  wnt = gated || tiles * groups >= 1024 ? 2 : 1;
  tg = (tiles + wnt - 1) / wnt;
  const long long room = 256LL * occ / groups > 0 ? 256LL * occ / groups : 1, rounds = (tg + room - 1) / room;
  wgs = (tg + rounds - 1) / rounds;
  return tg <= 0x7fffffffLL;
}

int hy_rows_walk_groups(const RowLinear& p) {
  int wnt;
  long long tg, wgs;
  return p.wbf16 && hy_rows_gemv_takes(p) && rv_walks(p, p.R) && !p.row_expert && !p.tab && rv_walk_grid(p, 1, wnt, tg, wgs) && wnt == 2 ? (int)wgs : 0;
}

// bf16 rows. Us, weights in no cache, 8 rows, one | two | four tiles per workgroup: 2048 x 2048 5.4 | 6.3 | 8.0, 3072 x 2048 6.7 | 6.6 | 8.3, 2048 x
// 5632 8.7 | 11.3 | 15.9, 4096 x 4096 10.6 | 10.1 | 13.4, 10304 x 2048 14.3 | 11.9 | 13.0, 10304 x 4096 24.0 | 20.0 | 23.9, 32000 x 2048 33.8 | 26.9 | 25.5
// (fp32 rows 6.3, 8.2, 11.2, 15.1 (10304 x 2048), 29.0 (32000 x 2048)). 4 rows, two | four tiles, of four steps each: 2048 x 2048 4.6 | 5.5, 3072 x
// 2048 5.8 | 5.8, 2048 x 5632 7.9 | 10.3, 4096 x 4096 8.9 | 8.9, 10304 x 2048 13.3 | 11.4, 10304 x 4096 22.0 | 17.7, 32000 x 4096 55 | 41.
static int rv_rows16(const RowLinear& p, int rows, int groups, int gated, hipStream_t s) {
  const int G = rows <= 4 ? 4 : 8;
  const long long tiles = (gated ? 2LL : 1LL) * ((p.N + G - 1) / G), all = tiles * groups;
  const int nt = G == 4 ? (all < 1024 ? 2 : 4) : (all < 512 && !gated ? 1 : (all < 2048 ? 2 : 4));
  const long long wgs = (tiles + nt - 1) / nt;
  if (wgs > 0x7fffffffLL) return -4;
  const dim3 grid((unsigned)wgs, groups);
  const bool plain = rv_form_of(p, p.R) >= 0 && (rv_form_of(p, p.R) & ~RV_ONE) == HY_ACT_NONE;
#define RV_RUN16(G, NT, U, PIPE)                                                                                              \
  do {                                                                                                                        \
    if (plain) rows_gemv_kernel<G, NT, 1, 4, U, 0, double, 2, PIPE, HY_ACT_NONE><<<grid, 256, 0, s>>>(p, p.R, gated);          \
    else rows_gemv_kernel<G, NT, 1, 4, U, 0, double, 2, PIPE><<<grid, 256, 0, s>>>(p, p.R, gated);                             \
  } while (0)
  if (G == 4) {
    if (nt == 2) RV_RUN16(4, 2, 4, true);
    else RV_RUN16(4, 4, 4, false);
  } else {
    if (nt == 1) RV_RUN16(8, 1, 4, true);
    else if (nt == 2) RV_RUN16(8, 2, 2, true);
    else RV_RUN16(8, 4, 2, true);
  }
#undef RV_RUN16
  JLA_CHECK_LAUNCH();
  return 0;
}

// Weight rows per group: one from K 2049 on for a single row, whose groups are longer than a trip to memory anyway, two for two rows; up to K 2048
// four where that leaves whole numbers of groups per compute unit. Us, weights in no cache, one | two | four, one row: 2048 x 2048 5.67 | 6.04 |
// 5.63, 3072 x 2048 normed 7.04 | 7.25 | 7.82, 8224 x 2048 14.5 | 14.6 | 14.1, 2048 x 5632 10.6 | 11.6 | 11.7, 4096 x 7168 20.9 | 22.0 | 31.0, 10304 x
// 4096 normed 29.9 | 31.7 | 31.8; two rows: 10304 x 4096 42.1 | 36.0 | 36.1, 4096 x 7168 24.9 | 24.0 | 32.9.
static int rv_rows32(const RowLinear& p, hipStream_t s) {
  const int gated = hy_act_gated(p.act);
  const bool each = p.row_expert || p.tab;
  const int groups = each ? p.R : 1, rpg = each ? 1 : p.R;
  const long long rows = gated ? 2LL * p.N : p.N, all = rows * groups;  // weight rows
  const int nt = p.K > 2048 ? (rpg == 1 && !gated ? 1 : 2) : (all >= 4096 || (all >= 1024 && all <= 2048) ? 4 : 2);
  const long long tg = (rows + nt - 1) / nt, room = 256LL * 4 / groups, rounds = (tg + room - 1) / room;  // (four workgroups per compute unit)
  if (tg > 0x7fffffffLL) return -4;
  const dim3 grid((unsigned)((tg + rounds - 1) / rounds), groups);
#define RV_RUN32(NT, V, RW) rows_walk_f32_kernel<NT, V, RW, 0><<<grid, 256, 0, s>>>(p, rpg, gated, (int)tg, RowParts{})
// (one row: FORM's comment says which forms have code of their own)
#define RV_FORM32(NT, V, F)                                                                                        \
  if (form == (F)) {                                                                                               \
    rows_walk_f32_kernel<NT, V, 1, 0, F><<<grid, 256, 0, s>>>(p, rpg, gated, (int)tg, RowParts{});                 \
    break;                                                                                                         \
  }
#define RV_ASIS32(NT, V)                 \
  RV_FORM32(NT, V, HY_ACT_NONE)          \
  RV_FORM32(NT, V, HY_ACT_NONE + RV_ADD)
#define RV_ONE32(NT, V)                                          \
  do {                                                           \
    RV_ASIS32(NT, V)                                             \
    RV_FORM32(NT, V, HY_ACT_NONE + RV_RES)                       \
    RV_FORM32(NT, V, HY_ACT_NONE + RV_NORM)                      \
    RV_FORM32(NT, V, HY_ACT_SOFTCAP + RV_NORM)                   \
    RV_FORM32(NT, V, HY_ACT_NONE + RV_RES + RV_NORM)             \
    if constexpr (NT > 1) {                                      \
      RV_FORM32(NT, V, HY_ACT_SWIGLU + RV_RES)                   \
      RV_FORM32(NT, V, HY_ACT_CLAMP_GLU + RV_NORM)               \
    }                                                            \
    RV_RUN32(NT, V, 1);                                          \
  } while (0)
#define RV_LONE32(NT, V)  \
  do {                    \
    RV_ASIS32(NT, V)      \
    RV_RUN32(NT, V, 1);   \
  } while (0)
  const int form = rpg == 1 && rv_form_of(p, 1) >= 0 ? rv_form_of(p, 1) & ~RV_ONE : -1;
#define RV_SHORT32(V)                   \
  do {                                  \
    if (nt == 2) {                      \
      if (rpg == 1) RV_RUN32(2, V, 1);  \
      else RV_RUN32(2, V, 2);           \
    } else if (rpg == 1) {              \
      RV_RUN32(4, V, 1);                \
    } else {                            \
      RV_RUN32(4, V, 2);                \
    }                                   \
  } while (0)
#define RV_LONG32(V)                    \
  do {                                  \
    if (rpg == 1) RV_RUN32(2, V, 1);    \
    else RV_RUN32(2, V, 2);             \
  } while (0)
  if (p.K <= 1024) RV_SHORT32(1);
  else if (p.K <= 2048 && rpg == 1 && nt == 2) RV_ONE32(2, 2);
  else if (p.K <= 2048 && rpg == 1) RV_ONE32(4, 2);
  else if (p.K <= 2048) RV_SHORT32(2);
  else if (p.K <= 4096 && nt == 1) RV_ONE32(1, 4);
  else if (p.K <= 4096 && rpg == 1) RV_ONE32(2, 4);
  else if (p.K <= 4096) RV_RUN32(2, 4, 2);
  else if (p.K <= 6144 && nt == 1) RV_LONE32(1, 6);
  else if (p.K <= 6144) RV_LONG32(6);
  else if (nt == 1) RV_LONE32(1, 8);
  else RV_LONG32(8);
#undef RV_LONE32
#undef RV_ONE32
#undef RV_ASIS32
#undef RV_FORM32
#undef RV_LONG32
#undef RV_SHORT32
#undef RV_RUN32
  JLA_CHECK_LAUNCH();
  return 0;
}

int hy_rows_gemv(const RowLinear& p, hipStream_t s) {
  if (rv_short(p)) {
    constexpr int cols = 4 * 4 * RV_SHORT_NT;
    rows_short_kernel<<<(p.N + cols - 1) / cols, 256, 0, s>>>(p);
    JLA_CHECK_LAUNCH();
    return 0;
  }
  if (!p.wbf16) return rv_rows32(p, s);
  const int gated = hy_act_gated(p.act);
  RowLinear q = p;
  const bool each = !p.offs && (p.row_expert || p.tab);  // one row, one expert per group
  if (p.offs) q.row_expert = nullptr;
  const int groups = p.offs ? p.E : (each ? p.R : 1);
  const int rpg = each ? 1 : p.R;
  if (groups > 65535) return -4;
  // rows of a pass: a dense batch's count rounded up; an expert's share of the sorted rows, twice the mean (at least 4)
  const int even = p.offs && p.even_rows > 0 ? p.even_rows : 0;
  const int rows = each ? 1 : (p.offs ? (even ? even : (p.R < 2 * ((p.R + p.E - 1) / p.E) ? p.R : 2 * ((p.R + p.E - 1) / p.E))) : p.R);
  if ((p.a_norm_one || p.best) && !rv_walks(p, rows)) return -10;
  if (rv_walks(p, rows)) {
    int wnt;
    long long tg, wgs;
    if (!rv_walk_grid(p, groups, wnt, tg, wgs)) return -4;
    const dim3 grid((unsigned)wgs, groups);
    const unsigned lds = (unsigned)(rows * p.K * sizeof(float));
#define RV_WALK_FORM(NT, U, V, F) rows_gemv_walk_kernel<NT, U, V, 0, 0, F><<<grid, 256, lds, s>>>(q, rpg, gated, (int)tg, RowParts{})
#define RV_WALK_ACT(NT, U, V, A)                                                              \
  do {                                                                                        \
    if (form == (A) + RV_ONE + RV_RES) RV_WALK_FORM(NT, U, V, (A) + RV_ONE + RV_RES);         \
    else if (form == (A) + RV_ONE + RV_NORM) RV_WALK_FORM(NT, U, V, (A) + RV_ONE + RV_NORM);  \
    else RV_WALK_FORM(NT, U, V, (A) + RV_ONE + RV_RES + RV_NORM);                             \
  } while (0)
#define RV_WALK(NT, U, V)                                                                     \
  do {                                                                                        \
    const int act = form >= RV_ONE && form < RV_MUL ? form % 8 : -1;                          \
    if (act == HY_ACT_NONE) RV_WALK_ACT(NT, U, V, HY_ACT_NONE);                               \
    else if (NT == 2 && act == HY_ACT_SWIGLU) RV_WALK_ACT(2, U, V, HY_ACT_SWIGLU);            \
    else if (NT == 2 && act == HY_ACT_CLAMP_GLU) RV_WALK_ACT(2, U, V, HY_ACT_CLAMP_GLU);      \
    else if (NT == 1 && form == RV_GATE) RV_WALK_FORM(1, U, V, RV_GATE);                      \
    else RV_WALK_FORM(NT, U, V, -1);                                                          \
  } while (0)
#define RV_BEST_FORM(U, V, F) rows_gemv_walk_kernel<2, U, V, 0, 1, F><<<grid, 256, lds, s>>>(q, rpg, gated, (int)tg, RowParts{})
#define RV_BEST(U, V)                                                                                                  \
  do {                                                                                                                 \
    if (form == HY_ACT_NONE + RV_ONE + RV_NORM) RV_BEST_FORM(U, V, HY_ACT_NONE + RV_ONE + RV_NORM);                    \
    else if (form == HY_ACT_NONE + RV_ONE + RV_NORM + RV_RES) RV_BEST_FORM(U, V, HY_ACT_NONE + RV_ONE + RV_NORM + RV_RES); \
    else if (form == HY_ACT_SOFTCAP + RV_ONE + RV_NORM) RV_BEST_FORM(U, V, HY_ACT_SOFTCAP + RV_ONE + RV_NORM);         \
    else RV_BEST_FORM(U, V, -1);                                                                                       \
  } while (0)
    const int form = rv_form_of(q, rpg);
    if (p.best) {
      if (wnt != 2 || groups != 1 || gated) return -11;
      if (p.K <= 2048) RV_BEST(4, 2);
      else RV_BEST(8, 4);
    } else if (p.K <= 2048) {
      if (wnt == 1) RV_WALK(1, 4, 2);
      else RV_WALK(2, 4, 2);
    } else {
      if (wnt == 1) RV_WALK(1, 8, 4);
      else RV_WALK(2, 8, 4);
    }
#undef RV_BEST
#undef RV_BEST_FORM
#undef RV_WALK
#undef RV_WALK_ACT
#undef RV_WALK_FORM
    JLA_CHECK_LAUNCH();
    return 0;
  }
  if (p.a_bf16) return rv_rows16(q, rows, groups, gated, s);
  const int G = rows <= 4 ? 4 : (rows <= 8 ? 8 : 16), mt = rows <= 16 ? 1 : (rows <= 32 ? 2 : 4);
  const long long tiles = (gated ? 2LL : 1LL) * ((p.N + G - 1) / G);
  // one tile per workgroup until there are a few workgroups for every compute unit; then tiles share the workgroup's
  // activation reads, which weigh more the more rows there are (8 rows, K 4096 x N 4096: 1 / 2 / 4 tiles 15.0 / 12.3 / 14.8
  // us; K 2048 x N 32000: 46 / 35 / 29; one row 27.9 / 24.5 / 27.6). Up to K 1024, where each wave has one batch of loads, two
  // tiles pay from one workgroup per compute unit on: K 1024 x N 2048, weights in no cache, one row 4.1 -> 3.4 us (vector
  // unit 4.6), four rows 5.5 -> 3.6; weights in a cache, one row 4.3 -> 3.3 (3.5); K 4096 5.9 -> 6.8.
  const long long all = tiles * groups;
  int nt = gated || mt > 1 || all >= (G == 4 ? (p.K <= RV_PAIR_K ? 256 : 1024) : 512) ? 2 : 1;
  // Rows by expert, up to four per expert: four tiles from 4096 on where the experts have rows (two per expert on average or as many each; one
  // on average from 512 tiles per expert on), with two per expert and K from 2560 on from 2048; not on weights 4 KiB apart (8 KiB: with two),
  // which share their memory channels. Fewer rows leave too many experts, and workgroups, without work. Us, two | four tiles, 8 experts: 16
  // rows, K 1024 | 2816 | 7168 x N 2048 10.3 | 21.5 | 44, 8.8 | 18.6 | 39, N 1024 6.4 | 12.8 | 24.1, 6.3 | 11.5 | 22.4, K 2048 16.0 | 16.4 and 9.2 | 9.9;
  // 8 rows, K 1024 | 2048 | 2816 | 7168 x N 2048 8.1 | 11.9 | 16.0 | 33.2, 7.3 | 13.2 | 15.2 | 30.5; 16 of 16 experts, K 2816 x N 1024 16.6 | 17.2; one
  // row each, K 128 | 512 x N 2048 5.7 | 8.8, 4.3 | 7.4, N 1024 3.7 | 5.4, 3.7 | 5.5; 3 rows in all, K 2816 | 7168 x N 2048 9.2 | 17.4, 10.1 | 19.8, 4
  // rows x N 1024 7.2 | 12.6, 9.8 | 18.2. 16 rows, K 7168 x N 4096 84 | 75.
  const bool pairs = p.R >= 2LL * p.E, wide = p.K % 2048 != 0 && (even > 0 || (p.R >= p.E && tiles >= 512));
  const bool filled = p.offs && ((all >= 4096 && (wide || (pairs && p.K != 2048))) || (all >= 2048 && pairs && p.K >= 2560));
  if (all >= (G > 4 || gated ? 2048 : 12288) || filled) nt = 4;
  const long long wgs = (tiles + nt - 1) / nt;
  if (wgs > 0x7fffffffLL) return -4;
  const dim3 grid((unsigned)wgs, groups);
#define RV_RUN(G, NT, MT, U, NORM, T) rows_gemv_kernel<G, NT, MT, 4, U, NORM, T, 4, false><<<grid, 256, 0, s>>>(q, rpg, gated)
  // (up to two workgroups per compute unit nobody else hides a wave's wait for its batch: one row of 2048 x 5632 7.9 -> 7.2 us, 2048 x 2048 4.6
  // -> 4.3; three per unit 5.3 -> 6.2)
  const int form = rv_form_of(q, rpg) < 0 ? -1 : rv_form_of(q, rpg) & ~RV_ONE;
  if (G == 4 && nt == 1 && !p.a_norm_w && all <= 512) {
    if (form == HY_ACT_NONE) rows_gemv_kernel<4, 1, 1, 4, 4, 0, double, 4, true, HY_ACT_NONE><<<grid, 256, 0, s>>>(q, rpg, gated);
    else if (form == HY_ACT_NONE + RV_ADD) rows_gemv_kernel<4, 1, 1, 4, 4, 0, double, 4, true, HY_ACT_NONE + RV_ADD><<<grid, 256, 0, s>>>(q, rpg, gated);
    else rows_gemv_kernel<4, 1, 1, 4, 4, 0, double, 4, true><<<grid, 256, 0, s>>>(q, rpg, gated);
    JLA_CHECK_LAUNCH();
    return 0;
  }
#define RV_PLAIN(U, F) rows_gemv_kernel<4, 2, 1, 4, U, 0, double, 4, false, F><<<grid, 256, 0, s>>>(q, rpg, 0)
#define RV_NT(G, NORM, T)                     \
  do {                                        \
    if (nt == 1) RV_RUN(G, 1, 1, 4, NORM, T);  \
    else if (nt == 2) RV_RUN(G, 2, 1, 2, NORM, T); \
    else RV_RUN(G, 4, 1, 2, NORM, T);         \
  } while (0)
#define RV_16(T)                         \
  do {                                   \
    if (mt == 4) {                       \
      if (nt == 2) RV_RUN(16, 2, 4, 1, 0, T); \
      else RV_RUN(16, 4, 4, 1, 0, T);    \
    } else if (mt == 2) {                \
      if (nt == 2) RV_RUN(16, 2, 2, 2, 0, T); \
      else RV_RUN(16, 4, 2, 1, 0, T);    \
    } else {                             \
      RV_NT(16, 0, T);                   \
    }                                    \
  } while (0)
  // (rows that had the vector unit's form are added in 64 bits, to lose no more than it did; more than eight dense rows, those that
  // rows_mid.hip leaves, had the tiles' one fp32 chain over all of K, 2.7e-7 at K 2048, here 1.3e-7 in one chain per wave: 33 rows of 4096 x
  // 10304 60.5 us, 64.5 in 64 bits)
  if (G == 4) {
    // Two tiles: batches of four or three steps where they divide a wave's (a step past the end costs its loads), their sums added in 64 bits
    // every two as in batches of two. Us, weights in no cache, two | three | four steps, one row: 10304 x 2048 10.3 | 13.0 | 9.9, 32000 x 2048 (two
    // tiles) 23.3 | 31.7 | 22.8, 4096 x 4096 9.1 | 9.3 | 8.6, 4096 x 14336 23.0 | 23.2 | 22.6; four rows of 8 experts of 2048 x 2816 12.0 | 10.9 | 13.7.
    const int mine = (p.K + 511) / 512;  // steps of a wave
    if (p.a_norm_w) RV_NT(4, 1, double);  // (at most two rows)
    else if (nt == 2 && mine % 4 == 0 && form == HY_ACT_NONE) RV_PLAIN(4, HY_ACT_NONE);
    else if (nt == 2 && mine % 4 == 0 && form == HY_ACT_NONE + RV_ADD) RV_PLAIN(4, HY_ACT_NONE + RV_ADD);
    else if (nt == 2 && mine % 3 == 0 && form == HY_ACT_NONE) RV_PLAIN(3, HY_ACT_NONE);
    else if (nt == 2 && mine % 3 == 0 && form == HY_ACT_NONE + RV_ADD) RV_PLAIN(3, HY_ACT_NONE + RV_ADD);
    else if (nt == 2 && mine % 4 == 0) RV_RUN(4, 2, 1, 4, 0, double);
    else if (nt == 2 && mine % 3 == 0) RV_RUN(4, 2, 1, 3, 0, double);
    else RV_NT(4, 0, double);
  } else if (G == 8) {
    RV_NT(8, 0, double);
  } else if (p.offs) {
    RV_16(double);
  } else {
    RV_16(float);
  }
#undef RV_16
#undef RV_NT
#undef RV_PLAIN
#undef RV_RUN
  JLA_CHECK_LAUNCH();
  return 0;
}

}  // namespace jla
