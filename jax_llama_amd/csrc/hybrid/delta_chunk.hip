// The gated delta rule of a prompt in chunks of 32 tokens, everything fp32, on v_mfma_f32_16x16x4_f32.
//
// With P(t, i) the product of the decays of tokens i + 1 .. t of a chunk, G_t = P(t, chunk start) and S0 the state the chunk
// starts from, the recurrence of delta_rule.hip (S <- g S; u = beta (v - S^T k); S <- S + k u^T; o = S^T q) unrolls to
//     (I + A) u = beta (v - G S0^T k),   A(t, i) = beta_t P(t, i) k_t . k_i  for i < t      (unit lower triangular)
//     o_t = G_t S0^T q_t + sum_{i <= t} P(t, i) (q_t . k_i) u_i
//     S   = G_last S0 + sum_i P(last, i) k_i u_i^T
// (1) delta_chunk_kernel, one wave per (chunk, head, row): T' = (I + A)^-1 diag(beta) by forward substitution, M(t, i) = P(t,
//     i) q_t . k_i, G and P(last, .); no chunk depends on another. The decays are multiplied up one by one, as the
//     token-by-token form does: no logarithms, no quotients.
// (2) delta_walk_kernel, one wave per (16 value columns, head, row) walks the chunks: five small products per chunk,
//     r = v - G (K S), u = T' r, o = G (Q S) + M u, S = G_last S + K^T (P(last, .) u).
// What bounds it: (2) is a chain of chunks at the fp32 matrix rate of one SIMD (416 + 64 multiply-adds per token and column:
// 216 MFMAs of 32 cycles per chunk at dim 128). The token-by-token kernel spends 0.93 us per token on lane exchanges
// whatever the batch: 2048 tokens of one row, 16 heads of 128 x 128, 1.94 ms -> 0.32; 8 rows of 1500 tokens,
// 32 heads, 3.50 -> 0.58.
// The state stays in the accumulator layout and never leaves its registers: the lane that holds S[16 mb + 4 (l >> 4) + r][l &
// 15] hands it to the next product as the B operand of k-step r, whose A operand is then column 4 (l >> 4) + r of a 16-wide
// block: four k-steps per 16-byte LDS read. Likewise r and u. K, Q, T' and M of a chunk go through LDS once per workgroup (64
// columns); the next chunk's loads are in flight meanwhile.
// A token that is not a number spoils the outputs of its whole chunk (masked products are 0 x NaN), not only later ones.
#include "hy_util.h"
#include "hybrid.h"

namespace jla {

constexpr int DC = 32;                       // tokens of a chunk
constexpr int DC_WS = 2 * DC * DC + 2 * DC;  // floats per (chunk, head, row): T', M, G, P(last, .)

JLA_DEV f32x4 mma_f32(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

JLA_DEV f32x4 dc_load4(const float* p, bool in) {
  return in ? *reinterpret_cast<const f32x4*>(p) : f32x4{0.f, 0.f, 0.f, 0.f};
}

// grid (ceil(chunks / 4), H, B), a wave per chunk. DB = dim / 16.
template <int DB>
__global__ void __launch_bounds__(256) delta_chunk_kernel(DeltaScan p, float* ws, int chunks) {
  __shared__ __attribute__((aligned(16))) float lp[4][DC][DC + 1];  // P(t, i); column DC: G
  __shared__ __attribute__((aligned(16))) float la[4][DC][DC + 4];  // A
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ch = blockIdx.x * 4 + wave, h = blockIdx.y, b = blockIdx.z;
  if (ch >= chunks) return;  // (no barrier below: waves share nothing)
  const int kh = h / (p.H / p.G), t0 = ch * DC, c = lane & 15, q = lane >> 4;
  const size_t m0 = (size_t)b * p.S + t0;
  float* out = ws + (((size_t)b * p.H + h) * chunks + ch) * DC_WS;

  // Gram products: token rows as both operands, 16 x 16 blocks on and below the diagonal
  f32x4 kk[3], qk[3];
#pragma unroll
  for (int x = 0; x < 3; ++x) kk[x] = qk[x] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool in0 = t0 + c < p.S, in1 = t0 + 16 + c < p.S;
  const size_t row0 = ((m0 + c) * p.G + kh) * (16 * DB) + 4 * q, row1 = row0 + (size_t)16 * p.G * (16 * DB);
#pragma unroll
  for (int kb = 0; kb < DB; ++kb) {
    const f32x4 k0 = dc_load4(p.kn + row0 + 16 * kb, in0), k1 = dc_load4(p.kn + row1 + 16 * kb, in1);
    const f32x4 q0 = dc_load4(p.qn + row0 + 16 * kb, in0), q1 = dc_load4(p.qn + row1 + 16 * kb, in1);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      kk[0] = mma_f32(k0[r], k0[r], kk[0]);
      kk[1] = mma_f32(k1[r], k0[r], kk[1]);
      kk[2] = mma_f32(k1[r], k1[r], kk[2]);
      qk[0] = mma_f32(q0[r], k0[r], qk[0]);
      qk[1] = mma_f32(q1[r], k0[r], qk[1]);
      qk[2] = mma_f32(q1[r], k1[r], qk[2]);
    }
  }
  // lane i: the running products from token i on (lane DC: from the chunk's start); tokens past the end keep (decay 1) and
  // write nothing (beta 0)
  const bool mine = lane < DC && t0 + lane < p.S;
  const float g = mine ? p.decay[(m0 + lane) * p.H + h] : 1.f, beta = mine ? p.beta[(m0 + lane) * p.H + h] : 0.f;
  {
    float run = 1.f;
#pragma unroll
    for (int t = 0; t < DC; ++t) {
      const float gt = __shfl(g, t, 64);
      run = (lane < t || lane == DC) ? run * gt : 1.f;
      if (lane <= DC) lp[wave][t][lane] = lane <= t || lane == DC ? run : 0.f;
    }
  }
  __builtin_amdgcn_wave_barrier();  // (LDS is the wave's own and in order)
  // A in LDS, M to the workspace; lane holds row (token) 4 q + r, column (token) c of each block
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    const int rb = x ? 16 : 0, cb = x == 2 ? 16 : 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = rb + 4 * q + r, i = cb + c;
      const float pr = lp[wave][t][i], bt = __shfl(beta, t, 64);  // (every lane takes part in the exchange)
      la[wave][t][i] = i < t ? bt * pr * kk[x][r] : 0.f;
      out[DC * DC + t * DC + i] = pr * qk[x][r];  // (P is 0 above the diagonal)
    }
  }
  __builtin_amdgcn_wave_barrier();
  if (lane < DC) {
    out[2 * DC * DC + lane] = lp[wave][lane][DC];
    out[2 * DC * DC + DC + lane] = lp[wave][DC - 1][lane];
    // column `lane` of the inverse: x_t = [t == lane] - sum_{i < t} A(t, i) x_i
    float x[DC];
#pragma unroll
    for (int t = 0; t < DC; ++t) {
      float s[4] = {lane == t ? 1.f : 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < t; i += 4) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(&la[wave][t][i]);
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (i + u < t) s[u] = fmaf(-a[u], x[i + u], s[u]);
      }
      x[t] = (s[0] + s[1]) + (s[2] + s[3]);
      out[t * DC + lane] = x[t] * beta;
    }
  }
}

// grid (ceil(vdim / 64), H, B), wave w: value columns 64 blockIdx.x + 16 w ..
template <int DB>
__global__ void __launch_bounds__(256, 2) delta_walk_kernel(DeltaScan p, const float* ws, int chunks) {
  constexpr int D = 16 * DB, LK = D + 4, LT = DC + 4;  // LDS row pitches: the 16 rows of a read fall on all banks
  constexpr int NK = DC * D / 4 / 256;                 // 16-byte pieces of K (and of Q) per thread
  __shared__ __attribute__((aligned(16))) float Ks[DC * LK], Qs[DC * LK], Ts[2 * DC * LT], Gs[2 * DC];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, q = lane >> 4;
  const int h = blockIdx.y, b = blockIdx.z, kh = h / (p.H / p.G);
  const int j0 = blockIdx.x * 64 + 16 * wave;
  const bool live = j0 < p.vdim;  // (a wave without columns still stages)
  const int j = live ? j0 + c : 0;
  const float* wsp = ws + ((size_t)b * p.H + h) * chunks * DC_WS;
  float* sp = p.state + ((size_t)b * p.H + h) * D * p.vdim + j;

  f32x4 S[DB];
#pragma unroll
  for (int mb = 0; mb < DB; ++mb)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[mb][r] = sp[(size_t)(16 * mb + 4 * q + r) * p.vdim];

  f32x4 pk[NK], pq[NK], pt[2];
  float pg = 0.f, pv[2][4];
  auto fetch = [&](int ch) {  // chunk ch on its way to registers
    const int t0 = ch * DC;
    const size_t m0 = (size_t)b * p.S + t0;
#pragma unroll
    for (int u = 0; u < NK; ++u) {
      const int e = u * 256 + tid, row = e / (D / 4), c4 = e % (D / 4);
      const bool in = t0 + row < p.S;
      const size_t at = ((m0 + row) * p.G + kh) * D + 4 * c4;
      pk[u] = dc_load4(p.kn + at, in);
      pq[u] = dc_load4(p.qn + at, in);
    }
    const float* w = wsp + (size_t)ch * DC_WS;
#pragma unroll
    for (int u = 0; u < 2; ++u) pt[u] = *reinterpret_cast<const f32x4*>(w + 4 * (u * 256 + tid));
    if (tid < 2 * DC) pg = w[2 * DC * DC + tid];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 16 * mt + 4 * q + r;
        pv[mt][r] = t0 + t < p.S ? p.v[((m0 + t) * p.H + h) * p.vdim + j] : 0.f;
      }
  };
  fetch(0);
  for (int ch = 0; ch < chunks; ++ch) {
    __syncthreads();  // the previous chunk has been read
#pragma unroll
    for (int u = 0; u < NK; ++u) {
      const int e = u * 256 + tid, row = e / (D / 4), c4 = e % (D / 4);
      *reinterpret_cast<f32x4*>(&Ks[row * LK + 4 * c4]) = pk[u];
      *reinterpret_cast<f32x4*>(&Qs[row * LK + 4 * c4]) = pq[u];
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int e = 4 * (u * 256 + tid), row = e / DC, col = e % DC;  // rows 0 .. 31: T', 32 .. 63: M
      *reinterpret_cast<f32x4*>(&Ts[row * LT + col]) = pt[u];
    }
    if (tid < 2 * DC) Gs[tid] = pg;
    float v[2][4];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[mt][r] = pv[mt][r];
    __syncthreads();
    if (ch + 1 < chunks) fetch(ch + 1);
    if (!live) continue;
    f32x4 ks[2], qs[2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) ks[mt] = qs[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < DB; ++kb) {
      f32x4 ka[2], qa[2];
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        ka[mt] = *reinterpret_cast<const f32x4*>(&Ks[(16 * mt + c) * LK + 16 * kb + 4 * q]);
        qa[mt] = *reinterpret_cast<const f32x4*>(&Qs[(16 * mt + c) * LK + 16 * kb + 4 * q]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
          ks[mt] = mma_f32(ka[mt][r], S[kb][r], ks[mt]);
          qs[mt] = mma_f32(qa[mt][r], S[kb][r], qs[mt]);
        }
    }
    f32x4 u[2], r_[2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const f32x4 gt = *reinterpret_cast<const f32x4*>(&Gs[16 * mt + 4 * q]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        r_[mt][r] = fmaf(-gt[r], ks[mt][r], v[mt][r]);
        qs[mt][r] *= gt[r];
      }
      u[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int kb = 0; kb <= mt; ++kb) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(&Ts[(16 * mt + c) * LT + 16 * kb + 4 * q]);
#pragma unroll
        for (int r = 0; r < 4; ++r) u[mt] = mma_f32(a[r], r_[kb][r], u[mt]);
      }
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int kb = 0; kb <= mt; ++kb) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(&Ts[(DC + 16 * mt + c) * LT + 16 * kb + 4 * q]);
#pragma unroll
        for (int r = 0; r < 4; ++r) qs[mt] = mma_f32(a[r], u[kb][r], qs[mt]);
      }
    const int t0 = ch * DC;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = t0 + 16 * mt + 4 * q + r;
        if (t < p.S) p.o[(((size_t)b * p.S + t) * p.H + h) * p.vdim + j] = qs[mt][r];
      }
    const float glast = Gs[DC - 1];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const f32x4 w = *reinterpret_cast<const f32x4*>(&Gs[DC + 16 * mt + 4 * q]);
#pragma unroll
      for (int r = 0; r < 4; ++r) u[mt][r] *= w[r];
    }
#pragma unroll
    for (int mb = 0; mb < DB; ++mb) {
#pragma unroll
      for (int r = 0; r < 4; ++r) S[mb][r] *= glast;
#pragma unroll
      for (int tb = 0; tb < 2; ++tb)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[mb] = mma_f32(Ks[(16 * tb + 4 * q + r) * LK + 16 * mb + c], u[tb][r], S[mb]);
    }
  }
  if (!live) return;
#pragma unroll
  for (int mb = 0; mb < DB; ++mb)
#pragma unroll
    for (int r = 0; r < 4; ++r) sp[(size_t)(16 * mb + 4 * q + r) * p.vdim] = S[mb][r];
}

// Tokens from which the chunks win over the token-by-token kernel (two launches and whole chunks against 0.93 us per token)
constexpr int DC_MIN_TOKENS = 20;  // (16 heads of 128 x 128, one row: 20 tokens 23.6 -> 18.7 us, 64 tokens 55 -> 23)

long long hy_delta_chunk_floats(const DeltaScan& p) {
  if (p.B < 1 || p.S < DC_MIN_TOKENS || p.H < 1 || p.G < 1 || p.H % p.G || (p.dim != 64 && p.dim != 128) || p.vdim < 16 ||
      p.vdim % 16 || p.H > 65535 || p.B > 65535)
    return 0;
  return (long long)p.B * p.H * ((p.S + DC - 1) / DC) * DC_WS;
}

int hy_delta_chunk(const DeltaScan& p, float* ws, hipStream_t s) {
  if (hy_delta_chunk_floats(p) == 0) return -1;
  if (((uintptr_t)p.kn | (uintptr_t)p.qn | (uintptr_t)ws) & 15) return -2;
  const int chunks = (p.S + DC - 1) / DC;
  const dim3 g1((chunks + 3) / 4, p.H, p.B), g2((p.vdim + 63) / 64, p.H, p.B);
  if (p.dim == 128) {
    delta_chunk_kernel<8><<<g1, 256, 0, s>>>(p, ws, chunks);
    delta_walk_kernel<8><<<g2, 256, 0, s>>>(p, ws, chunks);
  } else {
    delta_chunk_kernel<4><<<g1, 256, 0, s>>>(p, ws, chunks);
    delta_walk_kernel<4><<<g2, 256, 0, s>>>(p, ws, chunks);
  }
  JLA_CHECK_LAUNCH();
  return 0;
}

}  // namespace jla
