// 64 keys and values of a decode split in one wave's registers, for caches of heads of 64 or 128 numbers.
//
// What bounds a wave here is its share of the compute unit's memory path. A lane's 16 bytes lie beside its neighbours' in the row, so a load
// takes whole rows (four of 128 bf16 numbers): a lane per key, as the scores fall, touches 64 lines with every load, and values a column or
// two per lane take a load per key (16 + 128 loads of a chunk; here 16 + 16). The lanes of a row then hold parts of a score each, and every
// lane a part of eight columns; both are folded so that half of the numbers change lanes at each step.
// Us, before -> after: eight rows x 32 heads behind 1500 keys 28.4 -> 16.4, one row x 16 heads behind 2048 (attn_step.hip) 11.4 -> 9.3.
#pragma once
#include "hy_util.h"

namespace jla {

// s[0 .. 2 M): the lane keeps the half that its bit L asks for and gets the other lane's part of it, down to s[0 .. STOP)
template <int M, int L, int STOP, int N>
JLA_DEV void kc_fold(float (&s)[N], int lane) {
  const bool up = lane & L;
#pragma unroll
  for (int n = 0; n < M; ++n) {
    const float keep = up ? s[n + M] : s[n], send = up ? s[n] : s[n + M];
    s[n] = keep + __uint_as_float(lane_xor<L>(__float_as_uint(send)));
  }
  if constexpr (M > STOP) kc_fold<M / 2, L / 2, STOP>(s, lane);
}

// dim = 8 DK8, vdim = 64 VREG
template <typename CT, int DK8, int VREG>
struct KeyChunk {
  static constexpr int VK8 = 8 * VREG, RK = 64 / DK8, RV = 64 / VK8;  // lanes of a value row; rows that a load takes
  static constexpr int W = sizeof(CT) / 2;                            // 16-byte loads of eight numbers
  u32x4 k[DK8][W], v[VK8][W];

  // the chunk's key that this lane gets the score of, and the lane that gets key i's
  JLA_DEV static int key(int lane) { return RK * (lane % DK8) + lane / DK8; }
  JLA_DEV static int lane_of(int i) { return i % RK * DK8 + i / RK; }
  // columns VREG vlane + i are this lane's in the end
  JLA_DEV static int vlane(int lane) { return lane % VK8 * RV + lane / VK8; }

  // slot(i): the cache row of key i
  template <class Slot>
  JLA_DEV void load(const CT* kbase, size_t ldk, const CT* vbase, size_t ldv, int lane, Slot slot) {
#pragma unroll
    for (int i = 0; i < DK8; ++i) {
      const u32x4* at = reinterpret_cast<const u32x4*>(kbase + (size_t)slot(RK * i + lane / DK8) * ldk + 8 * (lane % DK8));
#pragma unroll
      for (int w = 0; w < W; ++w) k[i][w] = at[w];
    }
#pragma unroll
    for (int i = 0; i < VK8; ++i) {
      const u32x4* at = reinterpret_cast<const u32x4*>(vbase + (size_t)slot(RV * i + lane / VK8) * ldv + 8 * (lane % VK8));
#pragma unroll
      for (int w = 0; w < W; ++w) v[i][w] = at[w];
    }
  }
  JLA_DEV static void numbers(const u32x4 (&x)[W], float (&f)[8]) {
    if constexpr (W == 1) {
      unpack8(x[0], f);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f[i] = __uint_as_float(x[0][i]);
        f[4 + i] = __uint_as_float(x[W - 1][i]);
      }
    }
  }
  // q . k of key(lane); q: the numbers 8 (lane % DK8) + 0 .. 7 of the query
  JLA_DEV float score(const float (&q)[8], int lane) const {
    float s[DK8];
#pragma unroll
    for (int i = 0; i < DK8; ++i) {
      float f[8], d[2] = {0.f, 0.f};
      numbers(k[i], f);
#pragma unroll
      for (int e = 0; e < 8; ++e) d[e & 1] = fmaf(q[e], f[e], d[e & 1]);
      s[i] = d[0] + d[1];
    }
    kc_fold<DK8 / 2, DK8 / 2, 1>(s, lane);
    return s[0];
  }
  // acc: columns 8 (lane % VK8) + 0 .. 7 over this lane's rows; weight: key(lane)'s
  JLA_DEV void add(float (&acc)[8], float weight, int lane) const {
#pragma unroll
    for (int i = 0; i < VK8; ++i) {
      const float w = __shfl(weight, lane_of(RV * i + lane / VK8), 64);
      float f[8];
      numbers(v[i], f);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = fmaf(w, f[e], acc[e]);
    }
  }
  JLA_DEV static void columns(float (&acc)[8], int lane, float (&out)[VREG]) {
    kc_fold<4, 32, VREG>(acc, lane);
#pragma unroll
    for (int i = 0; i < VREG; ++i) out[i] = acc[i];
  }
};

}  // namespace jla
