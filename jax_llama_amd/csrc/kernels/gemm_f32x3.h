// fp32 products on the bf16 matrix cores: every operand is the sum of three bf16 numbers, each the nearest to what the ones
// before it leave (8 bits each, so the split is exact), and a product is the six largest of the nine partial products,
// smallest first,
//     a w = lo hi + hi lo + mid mid + mid hi + hi mid + hi hi,
// in fp32, the sum of a step of 32 from zero and then into the running sum. |mid| is below 2^-8 and |lo| below 2^-17 of the
// operand, so what is left out (mid lo, lo mid, lo lo) is below 2^-24 of the product, half an fp32 rounding, and of either
// sign: parts that are cut instead of rounded all have the operand's sign, and a sum of products of one sign comes out low (1
// x 32000 x 4096, positive numbers, error against 64 bits: exact-f32 MFMA 9.9e-7, cut parts 3.2e-6, all of it one-sided,
// nearest parts 3.2e-7). v_mfma_f32_16x16x32_bf16 adds 8 products at a time to the accumulator, rounded to nearest: 24
// roundings per 32 products, of the step's sum, and one of the running sum, where the fp32 matrix instruction rounds the
// running sum once per product (70 x 512 x 8: 5.3e-8 -> 3.1e-8). It does 16 times the work of v_mfma_f32_16x16x4_f32 per
// cycle, so six of them are 2.7 times its rate.
//
// One workgroup: 128 x 256 outputs in eight waves (two per SIMD) or 64 x 128 in four; a wave has all rows and 32 columns. K
// advances 32 per step. The operands are split on their way (6 vector instructions per number), so memory holds plain fp32 and
// nothing is prepared ahead: the activations through LDS, in two images, a wave's own weights straight into the layout of the
// matrix instruction. LDS: per part [rows][4 cells of 16 B], cell c of row r at c ^ (r & 8 ? 3 : 0): a read of 16 bytes per
// lane takes lanes 0-3, 12-15, 20-23, 24-27 together (then 4-11, 16-19, 28-31, and so above 32), which fall on all 64 banks (c
// ^ ((r >> 2) & 3): half of the reads' cycles were conflicts). What bounds it: the matrix cores at 70 % of their cycles and a
// clock held at 1.95 GHz by power. Each product is followed by the few vector instructions that fit beside it, the one barrier
// of a step lies where the next products' operands are on their way, and a step's six products start from zero, so that the
// running sums are rounded once per step and not 24 times (4 vector additions per tile, 5 % of the time; relative error of
// normal numbers, K 4096 in one chain 1.0e-6 -> 2.2e-7, K 2048 7.0e-7 -> 1.6e-7). Before, 128 x 128 outputs in four waves,
// both operands through LDS, splits and products in turn: us of the product of M x N x K, before -> here, 600 x 32000 x 4096
// 945 -> 859, 1500 2211 -> 1918, 128 224 -> 195, 400 x 14600 x 2048 177 -> 155, 200 x 11264 x 2048 93 -> 82, 64 x 2048 x 2048
// 20 -> 18. Both operands through LDS in this order: 5 % slower.
// Where the split does not hold, the workgroup computes its tile again on the fp32 matrix instruction (600 x 4000 x 4096 with a NaN
// in every tile: 125 -> 338 us). An infinity or NaN among the
// operands, or a number that rounds up to an infinity, makes its remainder NaN and so every result it enters (a sum past the largest
// number shows there too): the results are looked through at the end. A piece of a row whose numbers are all below 2^-95 would have
// parts that bf16's smallest step of 2^-133 cuts: the bits of the exponents are gathered as the pieces are split.
#pragma once
#include <type_traits>
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

constexpr int F3_BK = 32;

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

using F3Global = __attribute__((address_space(1))) f32x4;
// (what a row piece past the tile's last number reads)
__device__ const f32x4 f3_zeros[2] = {};

// K steps [t0, t1). act(gate accumulators, up accumulators) -> outputs of 4 neighbouring columns
template <int MT, int GATED, bool SCALED, class Act>  // MT waves, 16 MT rows
JLA_DEV void f3_tile(const F3Rows& p, int tiles_n, int t0, int t1, u32x4* lds, const Act& act) {
  constexpr int BM = 16 * MT, BN = 32 * MT;  // (so that a thread has a row piece per step)
  static_assert(MT % 4 == 0, "row tiles in fours");
  constexpr int AU = BM * 4;  // u32x4 of one part of the staged rows
  constexpr int BUF = 3 * AU;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int e = 0, r0 = 0, rend = 0, tn = 0;
  if (!row_tile<BM>(p.offs, p.E, p.R, tiles_n, lane, e, r0, rend, tn)) return;
  const int K = p.K, N = p.N;
  constexpr int COLS = GATED ? BN / 2 : BN;
  const int n0 = tn * COLS;
  const float* const wbase = p.w + (size_t)e * p.w_stride;
  // weight row of lane c, column tile j of this wave: 16 gate rows and 16 up rows for a gated product
  auto wrow = [&](int j) {
    const int col = min(GATED ? n0 + 16 * wave + c : n0 + 32 * wave + 16 * j + c, N - 1);
    return wbase + (size_t)(GATED && j ? N + col : col) * K;
  };
  auto arow = [&](int x) {
    const int row = min(r0 + x, rend - 1);  // (rows past the end repeat the last one)
    return p.a + (size_t)(p.a_idx ? p.a_idx[row] : row) * p.lda;
  };
  auto ascale = [&](int x) { return SCALED ? p.a_scale[min(r0 + x, rend - 1)] : 1.f; };
  // pieces of 8 numbers: one of the activations (k-chunk sch of row srow, for all waves), two of this wave's own weights (k-chunk q)
  const int sch = tid & 3, srow = tid >> 2;
  const float* const src[3] = {arow(srow) + 8 * sch, wrow(0) + 8 * q, wrow(1) + 8 * q};
  const float sc = ascale(srow);
  const int kend = min(K, F3_BK * t1);

  f32x4 acc[2][MT];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4* const st = lds + srow * 4 + (sch ^ (srow & 8 ? 3 : 0));
  const u32x4* const ra = lds + c * 4 + (q ^ (c & 8 ? 3 : 0));
  unsigned bits[3] = {0, 0, 0};  // bits of this thread's row pieces
  f32x4 f[3][2];                 // a step on its way
  auto fetch = [&](int t, int n) {
    const int k0 = F3_BK * t;
    const float* from = k0 + 8 * (n ? q : sch) < kend ? src[n] + k0 : reinterpret_cast<const float*>(f3_zeros);  // (K: a multiple of 8)
    const F3Global* at = reinterpret_cast<const F3Global*>(reinterpret_cast<uintptr_t>(from));
    f[n][0] = at[0];
    f[n][1] = at[1];
  };
  auto stage = [&](int buf) {  // the activations split and into LDS
    const F3Part s = SCALED ? f3_split(f[0][0] * sc, f[0][1] * sc, bits[0]) : f3_split(f[0][0], f[0][1], bits[0]);
    u32x4* d = st + buf * BUF;
    d[0] = s.hi;
    d[AU] = s.mid;
    d[2 * AU] = s.lo;
  };
  u32x4 w[2][2][3], a[4][3];  // two steps' weights; four row tiles, two of them on their way
  auto weights = [&](int set, int j) {
    const F3Part s = f3_split(f[1 + j][0], f[1 + j][1], bits[1 + j]);
    w[set][j][0] = s.hi;
    w[set][j][1] = s.mid;
    w[set][j][2] = s.lo;
  };
  auto read = [&](int buf, int i) {
#pragma unroll
    for (int x = 0; x < 3; ++x) a[i & 3][x] = ra[buf * BUF + x * AU + i * 64];
  };
  auto products = [&](int set, int i) {
    constexpr int PW[6] = {2, 0, 1, 1, 0, 0}, PA[6] = {0, 2, 1, 0, 1, 0};
    f32x4 sum[2] = {};  // (of the step: the running sums are rounded once per step)
#pragma unroll
    for (int x = 0; x < 6; ++x)
#pragma unroll
      for (int j = 0; j < 2; ++j) sum[j] = mfma16x16x32(w[set][j][PW[x]], a[i & 3][PA[x]], sum[j]);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[j][i][r] += sum[j][r];
  };
  // Round u of parity P reads step u's image, writes step u + 1's and multiplies the last two row tiles of step u - 1 (not in the
  // first round) and all but the last two of step u: the one barrier at its end finds every read of the image behind it and none of
  // the operands that the next products need.
  auto round = [&](auto first, auto parity, int u) {
    constexpr int P = parity.value;
#pragma unroll
    for (int jj = 0; jj < MT; ++jj) {
      const int i = (MT - 2 + jj) % MT;
      read(P, (i + 2) % MT);
      if (jj == 0) {
        stage(P ^ 1);
        fetch(u + 2, 0);
      }
      if (jj == 2 || jj == (MT > 4 ? 4 : 3)) {
        weights(P ^ 1, jj == 2 ? 0 : 1);
        fetch(u + 2, jj == 2 ? 1 : 2);
      }
      if (!first.value || jj > 1) products(jj < 2 ? P ^ 1 : P, i);
      if (jj % 2) {  // the order of two row tiles' work: a few vector instructions behind every product
#pragma unroll
        for (int m = 0; m < 24; ++m) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                 // MFMA
          if (m % 4 == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
          __builtin_amdgcn_sched_group_barrier(0x002, MT == 4 ? 6 : 3, 0);   // vector
          if (m % 4 == 3) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // LDS write
          if (m > 18) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);     // load
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's reads and writes; loads stay on their way
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
#pragma unroll
  for (int n = 0; n < 3; ++n) fetch(t0, n);
  stage(0);
  weights(0, 0);
  weights(0, 1);
#pragma unroll
  for (int n = 0; n < 3; ++n) fetch(t0 + 1, n);
  __syncthreads();
  using Even = std::integral_constant<int, 0>;
  using Odd = std::integral_constant<int, 1>;
  round(std::true_type{}, Even{}, t0);
  int t = t0 + 1;
#pragma unroll 1
  for (; t + 1 < t1; t += 2) {
    round(std::false_type{}, Odd{}, t);
    round(std::false_type{}, Even{}, t + 1);
  }
  if (t < t1) {
    round(std::false_type{}, Odd{}, t);
    products(1, MT - 2);
    products(1, MT - 1);
  } else {
    products(0, MT - 2);
    products(0, MT - 1);
  }
  // lane: rows 16 i + c, columns (weight tile rows) 16 j + 4 q + 0..3 of the wave's 32
  bool again = false;
#pragma unroll
  for (int n = 0; n < 3; ++n) again |= (bits[n] & 0x7fffffffu) && !(bits[n] & F3_EXP);
  float none[4] = {0.f, 0.f, 0.f, 0.f};  // (0 x an infinity or NaN)
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) none[r] = fmaf(acc[j][i][r], 0.f, none[r]);
  again |= !((none[0] + none[1]) + (none[2] + none[3]) == 0.f);
  if (__syncthreads_or(again)) {
    const float *ar[MT], *wr[2];
    float as[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      ar[i] = arow(16 * i + c) + 4 * q;
      as[i] = ascale(16 * i + c);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      wr[j] = wrow(j) + 4 * q;
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll 2
    for (int k = F3_BK * t0; k < kend; k += 16) {  // lane group q: numbers k + 4 q .. + 3 of both operands, one per instruction
      const bool in = k + 4 * q < K;
      const f32x4 z = {0.f, 0.f, 0.f, 0.f};
      f32x4 x[MT], y[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) y[j] = in ? *reinterpret_cast<const f32x4*>(wr[j] + k) : z;
#pragma unroll
      for (int i = 0; i < MT; ++i) x[i] = in ? *reinterpret_cast<const f32x4*>(ar[i] + k) * as[i] : z;
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(y[j][r], x[i][r], acc[j][i], 0, 0, 0);
    }
  }
  // results leave through the wave's own LDS, 32 rows x 32 accumulator columns at a time: the activation is one small loop
  // and rows leave in whole lines. 16-byte chunk x of row r lies at x ^ (r & 7)
  f32x4* const out = reinterpret_cast<f32x4*>(lds) + wave * 256;
  constexpr int OCH = GATED ? 4 : 8;  // output chunks of a row
  const int rr0 = lane / OCH, oc = lane % OCH;
  const int col = n0 + wave * (COLS / MT) + 4 * oc;
#pragma unroll
  for (int part = 0; part < MT / 2; ++part) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) out[(16 * i + c) * 8 + ((4 * j + q) ^ (c & 7))] = acc[j][2 * part + i];
    const int rbase = r0 + 32 * part;
    int drow = rbase + (lane & 31);
    drow = drow < rend ? (p.dst_idx ? p.dst_idx[drow] : drow) : -1;
#pragma unroll 2
    for (int s = 0; s < 32; s += 64 / OCH) {
      const int rr = s + rr0;
      const int d = __shfl(drow, rr, 64);
      const f32x4 g = out[rr * 8 + (oc ^ (rr & 7))];
      const f32x4 v0 = GATED ? out[rr * 8 + ((oc + 4) ^ (rr & 7))] : g;
      if (d >= 0 && col < N) {
        const f32x4 v = act(g, v0);
        f32x4* o = reinterpret_cast<f32x4*>(p.out + (size_t)d * p.ldo + col);
        *o = p.add ? *o + v : v;
      }
    }
  }
}

// u32x4 of LDS: two staged steps
template <int MT>
constexpr int f3_lds() {
  return 2 * 3 * 4 * 16 * MT;
}

// How a launch cuts its work: the tile and K over `splits` workgroups per tile, at least 8 steps each, whose partial sums go through
// slabs [split][rows][cols] that the caller's second kernel adds in order. The times are fitted to 3000 launches of 8 to 1500 rows, cols x K
// from 64 x 2048 to 32000 x 4096, and choose within 0.2 % of the fastest on average: a step of up to 256 resident 64 x 128 tiles takes 1 us,
// of up to 512 1.45 (1.36 in whole rounds), 3 once; of 256 128 x 256 tiles 2.04 and 5 once; the operands come at 4.6 TB/s at most, 3.2 with one
// workgroup per compute unit; the second kernel 4.5 us and the slabs' traffic at 6.6 TB/s. (With 0.75 and 1.33 for the small tiles and no rate
// of the operands 2.9 %: 777 x 2048 x 2048 61 us, here 52, 8 x 32000 x 4096 158 and 118.)
struct F3Plan {
  int bm, bn, splits, steps;  // steps per split
};
template <class Tiles>  // (int height) -> row tiles; matrices: of cols x K each
inline F3Plan f3_plan(const Tiles& row_tiles, long long rows, long long cols, int K, int matrices = 1) {
  const int total = (K + F3_BK - 1) / F3_BK;
  F3Plan best{128, 256, 1, total};
  double least = 1e30;
  for (int bm = 64; bm <= 128; bm += 64) {
    const bool small = bm == 64;
    // (of the launch: a multiple of 8 per split, and one without work that falls among the others' splits costs as much as one with)
    const long long tiles = (row_tiles(bm) * ((cols + 2 * bm - 1) / (2 * bm)) + 7) / 8 * 8;
    for (int cut = 1; cut <= 16 && (cut == 1 || total / cut >= 8); ++cut) {
      const int steps = (total + cut - 1) / cut, splits = (total + steps - 1) / steps;
      const long long n = tiles * splits, rest = n % 512;
      double us = small ? (double)(n / 512) * (steps * 1.36 + 3.) + (rest ? steps * (rest <= 256 ? 1. : 1.45) + 3. : 0.)
                        : (double)((n + 255) / 256) * (steps * 2.04 + 5.);
      const double rate = small && n <= 256 ? 3.2e6 : 4.6e6, bytes = 4. * K * ((double)cols * matrices + (double)rows);
      if (us < bytes / rate) us = bytes / rate;
      if (splits > 1) us += 4.5 + (double)rows * cols * 4 * (2 * splits + 1) / 6.6e6;
      if (us < 0.99 * least) {
        least = us;
        best = {bm, 2 * bm, splits, steps};
      }
    }
  }
  return best;
}

}  // namespace jla
