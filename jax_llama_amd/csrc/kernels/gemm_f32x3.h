// fp32 products on the bf16 matrix cores: every operand is the sum of three bf16 numbers, each the nearest to what the ones
// before it leave (8 bits each, so the split is exact), and a product is the six largest of the nine partial products, smallest
// first,
//     a w = lo hi + hi lo + mid mid + mid hi + hi mid + hi hi,
// in one fp32 accumulator. |mid| is below 2^-8 and |lo| below 2^-17 of the operand, so what is left out (mid lo, lo mid, lo lo)
// is below 2^-24 of the product, half an fp32 rounding, and of either sign: parts that are cut instead of rounded all have the
// operand's sign, and a sum of products of one sign comes out low (1 x 32000 x 4096, positive numbers, error against 64 bits:
// exact-f32 MFMA 9.9e-7, cut parts 3.2e-6, all of it one-sided, nearest parts 3.2e-7). v_mfma_f32_16x16x32_bf16 adds 8
// products at a time to the accumulator, rounded to nearest: 24 roundings per 32 products here, 5 of 6 of them of a small
// addend, where the fp32 matrix instruction rounds once per product (600 x 4000 x 4096, either sign: 1.14e-6 -> 0.57e-6; 70 x
// 512 x 8: 5.3e-8 -> 3.1e-8). It does 16 times the work of v_mfma_f32_16x16x4_f32 per cycle, so six of them are 2.7 times
// its rate.
//
// One workgroup: BM x 128 outputs, four waves of BM / 2 x 64; K advances 32 per step. The operands are split on their way
// from registers to LDS (6 vector instructions per number, beside the products of the step before), so memory holds plain
// fp32 and nothing is prepared ahead; loads are two steps ahead. LDS: per operand and part [rows][4 cells of
// 16 B], cell c of row r at c ^ ((r >> 2) & 3): the 16 lanes of a fragment read fall on all 64 banks.
// Where the split does not hold, the workgroup computes its tile again on the fp32 matrix instruction (600 x 4000 x 4096 with
// a NaN in every tile: 138 -> 285 us). An infinity or NaN among the operands, or a number that rounds up to an infinity,
// makes its remainder NaN and so every result it enters (a sum past the largest number shows there too); a piece of a row
// whose numbers are all below 2^-95 would have parts that bf16's smallest step of 2^-133 cuts.
#pragma once
#include "common.h"
#include "row_tiles.h"

namespace jla {

struct F3Rows {
  const float* a;  // activation rows, lda apart; a_idx (optional): row of linear row r; a_scale (optional): its factor
  int lda;
  const int32_t* a_idx;
  const float* a_scale;
  const float* w;  // [E][N (gated: gate rows, then up rows)][K]
  long long w_stride;
  int N, K;
  float* out;  // rows ldo apart; dst_idx (optional): row of linear row r; add: out += instead of out =
  int ldo;
  const int32_t* dst_idx;
  int add;
  const int32_t* offs;  // optional [E + 1]
  int E, R;
};

constexpr int F3_BN = 128, F3_BK = 32;
constexpr int F3_RESIDENT = 512;  // workgroups resident at once: two per compute unit

constexpr unsigned F3_EXP = 0x70000000u;  // set in some number of a row piece unless all of them are below 2^-95

struct F3Part {
  u32x4 hi, mid, lo;
};

// 8 numbers -> their three parts, packed; any: the bits that some number so far has
JLA_DEV F3Part f3_split(const f32x4 x, const f32x4 y, unsigned& any) {
  F3Part p;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float v0 = i < 2 ? x[2 * (i & 1)] : y[2 * (i & 1)], v1 = i < 2 ? x[2 * (i & 1) + 1] : y[2 * (i & 1) + 1];
    any |= __float_as_uint(v0) | __float_as_uint(v1);
    p.hi[i] = pack2bf(v0, v1);
    const float r0 = v0 - __uint_as_float(p.hi[i] << 16), r1 = v1 - __uint_as_float(p.hi[i] & 0xffff0000u);
    p.mid[i] = pack2bf(r0, r1);
    p.lo[i] = pack2bf(r0 - __uint_as_float(p.mid[i] << 16), r1 - __uint_as_float(p.mid[i] & 0xffff0000u));
  }
  return p;
}

// K steps [t0, t1). act(gate accumulators, up accumulators) -> outputs of 4 neighbouring columns
template <int BM, int GATED, class Act>
JLA_DEV void f3_tile(const F3Rows& p, int tiles_n, int t0, int t1, u32x4* lds, const Act& act) {
  constexpr int MT = BM / 32;                       // 16-row tiles of a wave
  constexpr int NA = BM * 4 / 256, NW = F3_BN * 4 / 256;  // 8-number pieces per thread and step
  constexpr int AU = BM * 4, WU = F3_BN * 4;        // u32x4 of one part
  constexpr int F3_BUF = 3 * (AU + WU);             // ... of one staged step
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wave >> 1, wc = wave & 1;
  int e = 0, r0 = 0, rend = 0, tn = 0;
  if (!row_tile<BM>(p.offs, p.E, p.R, tiles_n, lane, e, r0, rend, tn)) return;
  const int K = p.K, N = p.N;
  constexpr int COLS = GATED ? F3_BN / 2 : F3_BN;
  const int n0 = tn * COLS;
  const float* const wbase = p.w + (size_t)e * p.w_stride;
  // row x of the weight tile: 16 gate rows and 16 up rows in turn for a gated product
  auto wrow = [&](int x) {
    const int jt = x >> 4, col = min(n0 + (GATED ? 16 * (jt >> 1) + (x & 15) : x), N - 1);
    return wbase + (size_t)(GATED && (jt & 1) ? N + col : col) * K;
  };
  auto arow = [&](int x) {
    const int row = min(r0 + x, rend - 1);  // (rows past the end repeat the last one)
    return p.a + (size_t)(p.a_idx ? p.a_idx[row] : row) * p.lda;
  };
  auto ascale = [&](int x) { return p.a_scale ? p.a_scale[min(r0 + x, rend - 1)] : 1.f; };
  const int sch = tid & 3, srow = tid >> 2;  // staging: piece u is k-chunk sch of row 64 u + srow
  const float* pa[NA];
  float sc[NA];
  const float* pw[NW];
#pragma unroll
  for (int u = 0; u < NA; ++u) {
    pa[u] = arow(64 * u + srow) + 8 * sch;
    sc[u] = ascale(64 * u + srow);
  }
#pragma unroll
  for (int u = 0; u < NW; ++u) pw[u] = wrow(64 * u + srow) + 8 * sch;

  f32x4 acc[4][MT];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4* const la = lds;
  u32x4* const lw = lds + 3 * AU;
  const int cell = sch ^ ((srow >> 2) & 3);  // (64 u does not change it)
  const int rcell = q ^ ((c >> 2) & 3);
  unsigned ta[NA], tw[NW];  // bits of this thread's row pieces
#pragma unroll
  for (int u = 0; u < NA; ++u) ta[u] = 0;
#pragma unroll
  for (int u = 0; u < NW; ++u) tw[u] = 0;
  struct Step {
    f32x4 a[NA][2], w[NW][2];
  };
  auto fetch = [&](Step& f, int t) {  // step t on its way to registers
    const int k0 = F3_BK * t;
    const bool in = k0 + 8 * sch < K;  // (K is a multiple of 8)
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < NA; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) f.a[u][h] = in ? *reinterpret_cast<const f32x4*>(pa[u] + k0 + 4 * h) : z;
#pragma unroll
    for (int u = 0; u < NW; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) f.w[u][h] = in ? *reinterpret_cast<const f32x4*>(pw[u] + k0 + 4 * h) : z;
  };
  auto stage = [&](const Step& f, int buf) {  // split and into LDS
#pragma unroll
    for (int u = 0; u < NA; ++u) {
      const F3Part s = f3_split(f.a[u][0] * sc[u], f.a[u][1] * sc[u], ta[u]);
      u32x4* d = la + buf * F3_BUF + (64 * u + srow) * 4 + cell;
      d[0] = s.hi;
      d[AU] = s.mid;
      d[2 * AU] = s.lo;
    }
#pragma unroll
    for (int u = 0; u < NW; ++u) {
      const F3Part s = f3_split(f.w[u][0], f.w[u][1], tw[u]);
      u32x4* d = lw + buf * F3_BUF + (64 * u + srow) * 4 + cell;
      d[0] = s.hi;
      d[WU] = s.mid;
      d[2 * WU] = s.lo;
    }
  };
  auto products = [&](int buf) {
    u32x4 w[3][4];
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int j = 0; j < 4; ++j) w[x][j] = lw[buf * F3_BUF + x * WU + (64 * wc + 16 * j + c) * 4 + rcell];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      u32x4 a[3];
#pragma unroll
      for (int x = 0; x < 3; ++x) a[x] = la[buf * F3_BUF + x * AU + (wr * (BM / 2) + 16 * i + c) * 4 + rcell];
      constexpr int PW[6] = {2, 0, 1, 1, 0, 0}, PA[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int x = 0; x < 6; ++x)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j][i] = mfma16x16x32(w[PW[x]][j], a[PA[x]], acc[j][i]);
    }
  };
  Step f0, f1;  // two steps on their way
  fetch(f0, t0);
  if (t0 + 1 < t1) fetch(f1, t0 + 1);
  if constexpr (BM == 64) {  // two steps in LDS: one barrier per step, a step's products beside the split of the next
    stage(f0, 0);
    if (t0 + 2 < t1) fetch(f0, t0 + 2);
    __syncthreads();
    for (int t = t0; t < t1; t += 2) {
      products(0);
      if (t + 1 < t1) {
        stage(f1, 1);
        if (t + 3 < t1) fetch(f1, t + 3);
      }
      __syncthreads();
      if (t + 1 < t1) {
        products(1);
        if (t + 2 < t1) {
          stage(f0, 0);
          if (t + 4 < t1) fetch(f0, t + 4);
        }
        __syncthreads();
      }
    }
  } else {  // one step in LDS, so that two workgroups fit a compute unit (two steps and one workgroup: 137 against 157 TFLOP/s)
    for (int t = t0; t < t1; t += 2) {
      __syncthreads();
      stage(f0, 0);
      if (t + 2 < t1) fetch(f0, t + 2);
      __syncthreads();
      products(0);
      if (t + 1 < t1) {
        __syncthreads();
        stage(f1, 0);
        if (t + 3 < t1) fetch(f1, t + 3);
        __syncthreads();
        products(0);
      }
    }
  }
  // lane: rows 16 i + c of the wave's BM / 2, columns (weight tile rows) 16 j + 4 q + 0..3
  bool again = false;
#pragma unroll
  for (int u = 0; u < NA; ++u) again |= (ta[u] & 0x7fffffffu) && !(ta[u] & F3_EXP);
#pragma unroll
  for (int u = 0; u < NW; ++u) again |= (tw[u] & 0x7fffffffu) && !(tw[u] & F3_EXP);
  float none[4] = {0.f, 0.f, 0.f, 0.f};  // (0 x an infinity or NaN)
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) none[r] = fmaf(acc[j][i][r], 0.f, none[r]);
  again |= !((none[0] + none[1]) + (none[2] + none[3]) == 0.f);
  if (__syncthreads_or(again)) {
    const float *ar[MT], *wr_[4];
    float as[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      ar[i] = arow(wr * (BM / 2) + 16 * i + c) + 4 * q;
      as[i] = ascale(wr * (BM / 2) + 16 * i + c);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      wr_[j] = wrow(64 * wc + 16 * j + c) + 4 * q;
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const int k1 = min(K, F3_BK * t1);
#pragma unroll 2
    for (int k = F3_BK * t0; k < k1; k += 16) {  // lane group q: numbers k + 4 q .. + 3 of both operands, one per instruction
      const bool in = k + 4 * q < K;
      const f32x4 z = {0.f, 0.f, 0.f, 0.f};
      f32x4 a[MT], w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = in ? *reinterpret_cast<const f32x4*>(wr_[j] + k) : z;
#pragma unroll
      for (int i = 0; i < MT; ++i) a[i] = in ? *reinterpret_cast<const f32x4*>(ar[i] + k) * as[i] : z;
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j][r], a[i][r], acc[j][i], 0, 0, 0);
    }
  }
  // results leave through the wave's own LDS, 32 rows x 64 accumulator columns at a time: the activation is one small loop
  // and rows leave in whole lines. 16-byte chunk x of row r lies at x ^ (r & 15)
  f32x4* const st = reinterpret_cast<f32x4*>(lds) + wave * 512;
  constexpr int OCH = GATED ? 8 : 16;  // output chunks of a row
  const int rr0 = lane / OCH, oc = lane % OCH;
  const int gch = GATED ? 8 * (oc >> 2) + (oc & 3) : oc;
  const int col = n0 + wc * (COLS / 2) + 4 * oc;
#pragma unroll
  for (int half = 0; half < MT / 2; ++half) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) st[(16 * i + c) * 16 + ((4 * j + q) ^ c)] = acc[j][2 * half + i];
    const int rbase = r0 + wr * (BM / 2) + 32 * half;
    int drow = rbase + (lane & 31);
    drow = drow < rend ? (p.dst_idx ? p.dst_idx[drow] : drow) : -1;
#pragma unroll 2
    for (int s = 0; s < 32; s += 64 / OCH) {
      const int rr = s + rr0;
      const int d = __shfl(drow, rr, 64);
      const f32x4 g = st[rr * 16 + (gch ^ (rr & 15))];
      const f32x4 u = GATED ? st[rr * 16 + ((gch + 4) ^ (rr & 15))] : g;
      if (d >= 0 && col < N) {
        const f32x4 v = act(g, u);
        f32x4* o = reinterpret_cast<f32x4*>(p.out + (size_t)d * p.ldo + col);
        *o = p.add ? *o + v : v;
      }
    }
  }
}

// u32x4 of LDS: two staged steps of 64 rows, one of 128 (and both hold the epilogue's 32 KiB)
template <int BM>
constexpr int f3_lds() {
  return (BM == 64 ? 2 : 1) * 3 * 4 * (BM + F3_BN);
}

// How a launch cuts its work: 64- or 128-row tiles (a step of 512 resident workgroups takes about 1.8 and 2.6 us) and K over
// `splits` workgroups per tile, at least 8 steps each, whose partial sums go through slabs [split][R][N] that the caller's
// second kernel adds in order (about 4 us and the slabs' traffic).
struct F3Plan {
  int bm, splits, steps;  // steps per split
};
inline F3Plan f3_plan(long long mt128, long long mt64, long long tn, int K) {
  const int total = (K + F3_BK - 1) / F3_BK;
  F3Plan best{128, 1, total};
  double least = 1e30;
  for (int bm = 64; bm <= 128; bm += 64) {
    const long long tiles = (bm == 64 ? mt64 : mt128) * tn;
    for (int splits = 1; splits <= 16 && (splits == 1 || total / splits >= 8); ++splits) {
      const int steps = (total + splits - 1) / splits;
      const double slab_us = splits == 1 ? 0. : 4. + (double)tiles * bm * F3_BN * 4 * (splits + 0.5) * 2 / 5e6;
      const double us = (double)((tiles * splits + F3_RESIDENT - 1) / F3_RESIDENT) * steps * (bm == 64 ? 1.8 : 2.6) + slab_us;
      if (us < 0.95 * least) {
        least = us;
        best = {bm, (total + steps - 1) / steps, steps};
      }
    }
  }
  return best;
}

}  // namespace jla
