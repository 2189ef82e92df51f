// The tile of the products of some ten to a few hundred rows, x [M, K] times W [N, K] with bf16 weights (rows_mid.hip: row-major
// weights; linear_mid.hip: packed ones).
//
// What bounds it: bytes through a compute unit's vector memory path. W comes from HBM once (about 24 bytes per ns and unit with
// every unit pulling), x from L2, and the two do not overlap there: a unit keeps about 32 KB outstanding whatever it asks for,
// so time is the sum of W's and x's bytes at their latencies (64 rows of 4096 x 4096, operands straight to registers: W alone 9.2
// us, x alone 8.7, both 15.8, at any depth of prefetch). So: every weight byte is asked for by as few workgroups as can be, whole
// 128-byte lines of both operands (a fragment that a wave loads from 16 rows at once costs twice the path's time: 26 us instead of
// 15.8 at 64 rows), and x shared by the workgroup's columns through LDS. Both operands come by LDS-DMA, S stages of 64 WK deep in a ring, one
// barrier a stage. WN groups of waves deal the columns (16 NT each), WK groups the K of a stage: WN = 1 keeps a workgroup at 16
// columns, which is what fills the chip with N 2048 without a split of K over workgroups; WN = 4 shares x four times as often.
#pragma once
#include "common.h"

namespace jla {

template <int MT, int NT, int WN, int WK, int S, int XB>  // XB: bytes of an x number (2: bf16, 4: fp32, rounded as it is read)
struct MidShape {
  static constexpr int WAVES = WN * WK, BM = 16 * MT, BN = 16 * NT * WN;
  static constexpr int XP = BM / 8 * (XB / 2), WP = BN / 8, PIECES = (XP + WP) * WK;  // 1 KiB DMA pieces of a K slice of 64; of a stage
  static constexpr int OPS = (PIECES + WAVES - 1) / WAVES;                            // ... of a wave (surplus ones repeat the last piece)
  static constexpr int SLICE = (XP + WP) * 64, SLOT = SLICE * WK;                     // u32x4
  static constexpr int LDS = SLOT * S;
  static_assert(S >= 3 && LDS * 16 <= 160 * 1024, "ring");
  // waves per SIMD that a compute unit's LDS has room for, two at most
  static constexpr int PER_SIMD = WAVES >= 8 || LDS * 16 * 2 <= 160 * 1024 ? 2 : 1;
};
typedef double f64x4 __attribute__((ext_vector_type(4)));

// The form and K split with the least time of a product of `rows` rows and `cols` weight rows (of `matrices` matrices). A form's measured
// times, us: launch and fill; a stage; a stage's rise with every further workgroup of a compute unit (more); a split's second launch (sum), and a
// megabyte through the slabs, write and read (mb). takes(form): whether it runs these operands; row_tiles(height).
struct MidPlan {
  int form = -1, splits = 1, steps = 0;
  float us = 1e30f;
};
constexpr int MID_MAX_SPLITS = 16;

template <class Form, int N, class Takes, class RowTiles>
inline MidPlan mid_plan(const Form (&forms)[N], long long rows, long long cols, int K, int matrices, Takes takes, RowTiles row_tiles) {
  const int T = K >> 6;
  const float stream = (float)matrices * (float)cols * (float)K * 2 / 5.4e6f;  // the weights themselves
  MidPlan best;
  for (int i = 0; i < N; ++i) {
    const Form& f = forms[i];
    if (T % f.wk || !takes(f)) continue;
    const long long tiles = row_tiles(16 * f.mt) * ((cols + 16LL * f.nt * f.wn - 1) / (16LL * f.nt * f.wn));
    int last = 0;
    for (int want = 1; want <= MID_MAX_SPLITS && want <= T; ++want) {
      const int steps = ((T + want - 1) / want + f.wk - 1) / f.wk * f.wk, splits = (T + steps - 1) / steps;
      if (splits == last || (want > 1 && (steps < 2 * f.wk || tiles * splits > 700))) continue;
      last = splits;
      const float load = (float)(tiles * splits) / 256.f, deep = load > 2.f ? load + .3f : (load > 1.f ? 2.f : 1.f);
      float us = f.fill + f.stage * (float)(steps / f.wk) * (1.f + f.more * (deep - 1.f)) + deep - 1.f;
      if (us < 3.5f + stream) us = 3.5f + stream;
      if (splits > 1) us += f.sum + .15f * (float)splits + f.mb * (float)rows * (float)cols * (float)splits * 8e-6f;
      if (f.wn == 1 && load > 2.f) us *= 3.f;  // (16 columns a workgroup: x over and over)
      if (us < best.us) best = MidPlan{i, splits, steps, us};
    }
  }
  return best;
}

// 16-byte cell of chunk x of row r in its 128-byte line of LDS: the 16 lanes that a fragment read serves at a time (rows 0-3 and 12-15
// of one quarter, 4-11 of the next) fall on all 64 banks; fp32 rows, whose quarter is two chunks, need another order for that
JLA_DEV int mid_cell(int x, int r, int xb) {
  const int s = (r >> 1) & 7;
  return x ^ (xb == 4 ? (int)(0x32765410u >> (4 * s)) & 7 : s);
}

// Row tiles whose squares a wave sums (SS below), and the row tile that accumulator m of wave wn of a K group belongs to: with SS each
// wave starts with those that are its own.
template <int MT, int WN>
constexpr int MID_SQ = (MT + WN - 1) / WN;
template <int MT, int WN, bool SS>
JLA_DEV int mid_row_tile(int m, int wn) {
  return SS ? (m + wn * MID_SQ<MT, WN>) % MT : m;
}

// acc[t][m]: lane (c = lane & 15, q = lane >> 4) holds row 16 mid_row_tile(m) + c of the tile at weight columns 4 q .. + 3 of this wave's
// 16-column tile t; after the call in the waves of K group 0 only. Steps [t0, t1) of 64, a positive multiple of WK. xrow(r), wrow(r): the address of row r
// of the tile (BM, BN of them) at K 0; PACKED: wrow(16 j) is where 16-column tile j's fragments start (ops/reference.py
// pack_frag16x32). Tot: the type in which the sums of every `run` steps (a power of two;
// two products each) are added, f64x4 or f32x4, and the K groups' (the squares
// in 64 bits); void: one fp32 chain over all steps. SS (bf16 rows): ss[m] is this lane's share of the squares of row 16 mid_row_tile(m) + c, over quarters q and K groups
// (the row tiles beyond MT, counted from wn MID_SQ on, are another wave's). The waves deal the row tiles, without a branch, which would
// keep a stage's reads and products apart.
template <int MT, int NT, int WN, int WK, int S, int XB, bool PACKED, bool SS, class Tot, class XRow, class WRow>
JLA_DEV void mid_tile(u32x4* lds, XRow xrow, WRow wrow, int t0, int t1, f32x4 (&acc)[NT][MT], float (&ss)[SS ? MID_SQ<MT, WN> : 1],
                      int run = 0) {
  using H = MidShape<MT, NT, WN, WK, S, XB>;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, q = lane >> 4;
  // (a tile's place comes from ballots, in vector registers: without this the stage loop ran under a mask, every address formed per lane)
  t0 = __builtin_amdgcn_readfirstlane(t0);
  t1 = __builtin_amdgcn_readfirstlane(t1);
  const int wn = wave % WN, wk = wave / WN, ns = (t1 - t0) / WK;
  const char* src[H::OPS];
#pragma unroll
  for (int i = 0; i < H::OPS; ++i) {
    const int p = min(wave + H::WAVES * i, H::PIECES - 1) % (H::XP + H::WP);
    if (p < H::XP) {  // 8 rows x 128 bytes; fp32: the first halves of all rows, then the second
      const int row = p % (H::BM / 8) * 8 + (lane >> 3), half = p / (H::BM / 8);
      src[i] = xrow(row) + 128 * half + 16 * mid_cell(lane & 7, row, XB);
    } else {
      const int w = p - H::XP;
      if constexpr (PACKED) {
        src[i] = wrow(16 * (w >> 1)) + 1024 * (w & 1) + 16 * lane;  // fragment w & 1 of tile w >> 1
      } else {
        const int row = w * 8 + (lane >> 3);
        src[i] = wrow(row) + 16 * mid_cell(lane & 7, row, 2);
      }
    }
  }
  auto issue = [&](int st, int slot) {
#pragma unroll
    for (int i = 0; i < H::OPS; ++i) {
      const int p = min(wave + H::WAVES * i, H::PIECES - 1), sl = p / (H::XP + H::WP);
      const bool xs = p % (H::XP + H::WP) < H::XP;
      const int t = min(t0 + st * WK + sl, t1 - 1);  // (past the end: the last step again, unused)
      glds16_asm(src[i] + (size_t)t * (xs ? 64 * XB : (PACKED ? 2048 : 128)), lds + slot * H::SLOT + p * 64);
    }
  };
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int m = 0; m < (SS ? MID_SQ<MT, WN> : 1); ++m) ss[m] = 0.f;
  constexpr bool RUNS = !std::is_void_v<Tot>;
  using Sum = std::conditional_t<RUNS, Tot, f32x4>;
  Sum tot[RUNS ? NT : 1][RUNS ? MT : 1];
  double sq[RUNS && SS ? MID_SQ<MT, WN> : 1];
  auto end_run = [&](bool first) {
#pragma unroll
    for (int t = 0; t < (RUNS ? NT : 0); ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        tot[t][m] = first ? Sum{0, 0, 0, 0} : tot[t][m] + __builtin_convertvector(acc[t][m], Sum);
        acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
    for (int m = 0; m < (RUNS && SS ? MID_SQ<MT, WN> : 0); ++m) {
      sq[m] = first ? 0. : sq[m] + (double)ss[m];
      ss[m] = 0.f;
    }
  };
  end_run(true);
  int xat[MT];  // where accumulator m's rows start in a slice (wave-uniform)
#pragma unroll
  for (int m = 0; m < MT; ++m) xat[m] = 128 * mid_row_tile<MT, WN, SS>(m, wn);
  constexpr int XR = XB / 2;  // 16-byte reads of an x fragment
  auto read_w = [&](u32x4& w, int slot, int h, int t) {
    const u32x4* ws = lds + slot * H::SLOT + wk * H::SLICE + H::XP * 64 + wn * NT * 128;
    w = ws[PACKED ? (2 * t + h) * 64 + lane : (16 * t + c) * 8 + mid_cell(4 * h + q, c, 2)];
  };
  auto read_x = [&](u32x4 (&x)[XR], int slot, int h, int m) {
    const u32x4* xs = lds + slot * H::SLOT + wk * H::SLICE + xat[m] + c * 8;
    if constexpr (XB == 2) {
      x[0] = xs[mid_cell(4 * h + q, c, 2)];
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) x[i] = xs[h * H::BM * 8 + mid_cell(2 * q + i, c, 4)];
    }
  };
  // The products of half a stage, with the reads of the next half (of slot, h) between them, in this order. The products are the
  // compiler's, which waits for their sums wherever it moves or reads them; build.py has their sums in the vector unit's registers, as it
  // copied them out of the matrix unit's own and back at the loop's edge.
  auto half = [&](u32x4 (&w)[NT], u32x4 (&x)[MT][XR], u32x4 (&wnext)[NT], u32x4 (&xnext)[MT][XR], int slot, int h) {
#pragma unroll
    for (int t = 0; t < NT; ++t) read_w(wnext[t], slot, h, t);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      u32x4 f = x[m][0];
      if constexpr (XB == 4) {
        const f32x4 a = __builtin_bit_cast(f32x4, x[m][0]), b = __builtin_bit_cast(f32x4, x[m][1]);
        const float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
        f = pack8(v);
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t][m] = mfma16x16x32(w[t], f, acc[t][m]);
      if constexpr (SS) {
        if (m < MID_SQ<MT, WN>) {  // (plain FMAs: a dot product beside the products costs them more)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float lo = __uint_as_float(f[i] << 16), hi = __uint_as_float(f[i] & 0xffff0000u);
            ss[m] = fmaf(lo, lo, ss[m]);
            ss[m] = fmaf(hi, hi, ss[m]);
          }
        }
      }
      read_x(xnext[m], slot, h, m);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  u32x4 w0[NT], w1[NT], x0[MT][XR], x1[MT][XR];
#pragma unroll
  for (int s = 0; s < S - 1; ++s) issue(s, s);
  wait_vmcnt<(S - 2) * H::OPS>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int t = 0; t < NT; ++t) read_w(w0[t], 0, 0, t);
#pragma unroll
  for (int m = 0; m < MT; ++m) read_x(x0[m], 0, 0, m);
  int slot = 0, fill = S - 1;
  for (int st = 0; st < ns; ++st) {
    half(w0, x0, w1, x1, slot, 1);
    // this wave's pieces of stage st + 1 have landed, then every wave's; and every wave is past the slot that is filled next (its
    // reads of stage st - 1 were behind the products before this barrier)
    wait_vmcnt<(S - 3) * H::OPS>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    issue(st + S - 1, fill);
    slot = slot + 1 == S ? 0 : slot + 1;
    fill = fill + 1 == S ? 0 : fill + 1;
    half(w1, x1, w0, x0, slot, 0);  // (behind the last stage: reads that nothing uses)
    if (RUNS && !((st + 1) & (run - 1))) end_run(false);
  }
  wait_vmcnt<0>();
  end_run(false);
  auto join = [&](Sum (&sum)[NT][MT]) {  // the K groups' sums
    static_assert(WK == 1 || WK * NT * MT * WN / 2 * 64 * (int)sizeof(Sum) <= H::LDS * 16, "they reuse the ring");
    Sum* red = reinterpret_cast<Sum*>(lds);
#pragma unroll
    for (int half = WK / 2; half > 0; half /= 2) {
      __syncthreads();
      if (wk >= half && wk < 2 * half) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int m = 0; m < MT; ++m) red[((((wk - half) * WN + wn) * NT + t) * MT + m) * 64 + lane] = sum[t][m];
      }
      __syncthreads();
      if (wk < half) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int m = 0; m < MT; ++m) sum[t][m] += red[(((wk * WN + wn) * NT + t) * MT + m) * 64 + lane];
      }
    }
  };
  if constexpr (RUNS) {
    join(tot);
#pragma unroll
    for (int m = 0; m < (SS ? MID_SQ<MT, WN> : 0); ++m) ss[m] = (float)sq[m];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[t][m] = __builtin_convertvector(tot[t][m], f32x4);
  } else {
    join(acc);
  }
}

}  // namespace jla
