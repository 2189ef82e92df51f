// The gated delta rule and the scalar-gated memory of a prompt in chunks of 32 tokens, everything fp32, on v_mfma_f32_16x16x4_f32.
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
// whatever the batch: 2048 tokens of one row, 16 heads of 128 x 128, 1.94 ms -> 0.24 (split walk below); 8 rows of 1500
// tokens, 32 heads, 3.50 -> 0.60.
// Error against 64 bits, output | state, token by token -> here: those two 1.05e-7 -> 1.02e-7 | 7.4e-8 -> 6.9e-8 and 1.05e-7 ->
// 1.03e-7 | 7.2e-8 -> 6.9e-8; scalar gates, 777 tokens 1.07e-7 -> 1.02e-7 | 7.1e-8 -> 6.6e-8. It takes short chains: sums over key
// rows in blocks of 16, what a chunk's tokens add to the state in four parts, the diagonal of T' after everything below it, Gram
// products and decays in 64 bits (one chain each, as the products fall, gave 1.32e-7 | 8.2e-8; the walk with scalar gates pays 8 %
// for it, the delta rule's nothing).
// The state stays in the accumulator layout and never leaves its registers: the lane that holds S[16 mb + 4 (l >> 4) + r][l &
// 15] hands it to the next product as the B operand of k-step r, whose A operand is then column 4 (l >> 4) + r of a 16-wide
// block: four k-steps per 16-byte LDS read. Likewise r and u. K, Q, T' and M of a chunk go through LDS once per workgroup (64
// columns); the next chunk's loads are in flight meanwhile.
// A number that is none (in a key, query, value or gate, or by overflow) would spoil every token of its chunk, as masked products
// are 0 x NaN: such a chunk is walked token by token, and only the tokens from that one on see it (the check and the walk's
// registers cost 5 %).
#include "hy_util.h"
#include "hybrid.h"

namespace jla {

constexpr int DC = 32;                       // tokens of a chunk
constexpr int DC_WS = 2 * DC * DC + 3 * DC;  // floats per (chunk, head, row): T' below its diagonal, M, G, P(last, .), beta
constexpr int DC_WS_SCALAR = DC * DC + 2 * DC + 4;  // scalar gates: M, G, P(last, .) write, G_last

JLA_DEV f32x4 mma_f32(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// element r of the sum of eight chains
JLA_DEV double dc_total(const f32x4 (&v)[8], int r) {
  double s[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) s[i] = (double)v[i][r] + v[i + 4][r];
  return (s[0] + s[1]) + (s[2] + s[3]);
}

JLA_DEV f32x4 dc_load4(const float* p, bool in) {
  return in ? *reinterpret_cast<const f32x4*>(p) : f32x4{0.f, 0.f, 0.f, 0.f};
}

// grid (ceil(chunks / 4), H, B), a wave per chunk. DB = dim / 16.
template <int DB>
__global__ void __launch_bounds__(256) delta_chunk_kernel(DeltaScan p, float* ws, int chunks) {
  __shared__ __attribute__((aligned(16))) double lp[4][DC][DC + 1];  // P(t, i); column DC: G
  __shared__ __attribute__((aligned(16))) float la[4][DC][DC + 4];  // A
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ch = blockIdx.x * 4 + wave, h = blockIdx.y, b = blockIdx.z;
  if (ch >= chunks) return;  // (no barrier below: waves share nothing)
  const int kh = h / (p.H / p.G), t0 = ch * DC, c = lane & 15, q = lane >> 4;
  const size_t m0 = (size_t)b * p.S + t0;
  float* out = ws + (((size_t)b * p.H + h) * chunks + ch) * DC_WS;

  // Gram products: token rows as both operands, 16 x 16 blocks on and below the diagonal
  // (eight short chains per block: a long one would lose a bit to the token-by-token form)
  f32x4 kp_[3][8], qp_[3][8];
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int a = 0; a < 8; ++a) kp_[x][a] = qp_[x][a] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool in0 = t0 + c < p.S, in1 = t0 + 16 + c < p.S;
  const size_t row0 = ((m0 + c) * p.G + kh) * (16 * DB) + 4 * q, row1 = row0 + (size_t)16 * p.G * (16 * DB);
#pragma unroll
  for (int kb = 0; kb < DB; ++kb) {
    const f32x4 k0 = dc_load4(p.kn + row0 + 16 * kb, in0), k1 = dc_load4(p.kn + row1 + 16 * kb, in1);
    const f32x4 q0 = dc_load4(p.qn + row0 + 16 * kb, in0), q1 = dc_load4(p.qn + row1 + 16 * kb, in1);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int a = 4 * (kb & 1) + r;
      kp_[0][a] = mma_f32(k0[r], k0[r], kp_[0][a]);
      kp_[1][a] = mma_f32(k1[r], k0[r], kp_[1][a]);
      kp_[2][a] = mma_f32(k1[r], k1[r], kp_[2][a]);
      qp_[0][a] = mma_f32(q0[r], k0[r], qp_[0][a]);
      qp_[1][a] = mma_f32(q1[r], k0[r], qp_[1][a]);
      qp_[2][a] = mma_f32(q1[r], k1[r], qp_[2][a]);
    }
  }
  // lane i: the running products from token i on (lane DC: from the chunk's start); tokens past the end keep (decay 1) and
  // write nothing (beta 0)
  const bool mine = lane < DC && t0 + lane < p.S;
  const float g = mine ? p.decay[(m0 + lane) * p.H + h] : 1.f, beta = mine ? p.beta[(m0 + lane) * p.H + h] : 0.f;
  {
    double run = 1.0;  // (64 bits: an error here would be common to a whole token's part of the state)
#pragma unroll
    for (int t = 0; t < DC; ++t) {
      const float gt = __shfl(g, t, 64);
      run = (lane < t || lane == DC) ? run * gt : 1.0;
      if (lane <= DC) lp[wave][t][lane] = lane <= t || lane == DC ? run : 0.0;
    }
  }
  __builtin_amdgcn_wave_barrier();  // (LDS is the wave's own and in order)
  // A in LDS, M to the workspace; lane holds row (token) 4 q + r, column (token) c of each block
  bool whole = true;  // (a number that is none in a token's key or query shows in its own products)
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    const int rb = x ? 16 : 0, cb = x == 2 ? 16 : 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = rb + 4 * q + r, i = cb + c;
      const double pr = lp[wave][t][i];
      const float bt = __shfl(beta, t, 64);  // (every lane takes part in the exchange)
      const double kk = dc_total(kp_[x], r), qk = dc_total(qp_[x], r);
      whole &= isfinite(kk) && isfinite(qk);
      la[wave][t][i] = i < t ? (float)(pr * bt * kk) : 0.f;
      out[DC * DC + t * DC + i] = (float)(pr * qk);  // (P is 0 above the diagonal)
    }
  }
  whole &= isfinite(g) && isfinite(beta);
  const bool spoiled = __any(!whole);
  __builtin_amdgcn_wave_barrier();
  if (lane < DC) {
    out[2 * DC * DC + lane] = (float)lp[wave][lane][DC];
    out[2 * DC * DC + DC + lane] = (float)lp[wave][DC - 1][lane];
    out[2 * DC * DC + 2 * DC + lane] = spoiled ? NAN : beta;  // (the walk then takes this chunk token by token)
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
      out[t * DC + lane] = lane < t ? x[t] * beta : 0.f;
    }
  }
}

// grid (H, ceil(vdim / 64), B), wave w: value columns 64 blockIdx.y + 16 w ..
template <int DB>
__global__ void __launch_bounds__(256, 2) delta_walk_kernel(DeltaScan p, const float* ws, int chunks) {
  constexpr int D = 16 * DB, LK = D + 4, LT = DC + 4;  // LDS row pitches: the 16 rows of a read fall on all banks
  constexpr int NK = DC * D / 4 / 256;                 // 16-byte pieces of K (and of Q) per thread
  __shared__ __attribute__((aligned(16))) float Ks[DC * LK], Qs[DC * LK], Ts[2 * DC * LT], Gs[3 * DC];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, q = lane >> 4;
  const int h = blockIdx.x, b = blockIdx.z, kh = h / (p.H / p.G);
  const int j0 = blockIdx.y * 64 + 16 * wave;
  const bool live = j0 < p.vdim;  // (a wave without columns still stages)
  const int j = live ? j0 + c : 0;
  const float* wsp = ws + ((size_t)b * p.H + h) * chunks * DC_WS;
  float* const sp = p.state + ((size_t)b * p.H + h) * D * p.vdim;
  const unsigned at_s = (unsigned)(4 * q * p.vdim + j);  // (this lane's place; the rows of a block differ by uniform steps)

  f32x4 S[DB];
#pragma unroll
  for (int mb = 0; mb < DB; ++mb)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[mb][r] = (sp + (size_t)(16 * mb + r) * p.vdim)[at_s];

  // a lane's places behind a chunk's first rows (uniform)
  const int krow = tid / (D / 4);  // piece u of a thread: row krow + 1024 / D u
  const unsigned at_k = (unsigned)(krow * p.G * D + 4 * (tid % (D / 4))), at_v = (unsigned)(4 * q * p.H * p.vdim + j);
  const size_t kstep = (size_t)(1024 / D) * p.G * D, vstep = (size_t)p.H * p.vdim;
  const float* const kbase = p.kn + ((size_t)b * p.S * p.G + kh) * D;
  const float* const qbase = p.qn + ((size_t)b * p.S * p.G + kh) * D;
  const float* const vbase = p.v + ((size_t)b * p.S * p.H + h) * p.vdim;
  float* const obase = p.o + ((size_t)b * p.S * p.H + h) * p.vdim;
  f32x4 pk[NK], pq[NK], pt[2];
  float pg = 0.f, pv[2][4];
  auto fetch = [&](int ch) {  // chunk ch on its way to registers
    const int left = p.S - ch * DC;
#pragma unroll
    for (int u = 0; u < NK; ++u) {
      const size_t up = (size_t)ch * DC * p.G * D + u * kstep;
      pk[u] = dc_load4(kbase + up + at_k, krow + 1024 / D * u < left);
      pq[u] = dc_load4(qbase + up + at_k, krow + 1024 / D * u < left);
    }
    const float* w = wsp + (size_t)ch * DC_WS;
#pragma unroll
    for (int u = 0; u < 2; ++u) pt[u] = *reinterpret_cast<const f32x4*>(w + 4 * (u * 256 + tid));
    if (tid < 3 * DC) pg = w[2 * DC * DC + tid];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        pv[mt][r] = 16 * mt + 4 * q + r < left ? (vbase + ((size_t)ch * DC + 16 * mt + r) * vstep)[at_v] : 0.f;
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
    if (tid < 3 * DC) Gs[tid] = pg;
    float v[2][4];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[mt][r] = pv[mt][r];
    __syncthreads();
    if (ch + 1 < chunks) fetch(ch + 1);
    if (!live) continue;
    // X S of both token tiles, X = K or Q: each block of key rows a chain of its own
    auto times_state = [&](const float* X, f32x4 (&xs)[2]) {
#pragma unroll
      for (int kb = 0; kb < DB; ++kb) {
        f32x4 a[2], blk[2];
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
          a[mt] = *reinterpret_cast<const f32x4*>(&X[(16 * mt + c) * LK + 16 * kb + 4 * q]);
          blk[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int mt = 0; mt < 2; ++mt) blk[mt] = mma_f32(a[mt][r], S[kb][r], blk[mt]);
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) xs[mt] = kb ? xs[mt] + blk[mt] : blk[mt];
      }
    };
    f32x4 u[2], r_[2];
    times_state(Ks, r_);
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const f32x4 g = *reinterpret_cast<const f32x4*>(&Gs[16 * mt + 4 * q]);
#pragma unroll
      for (int r = 0; r < 4; ++r) r_[mt][r] = fmaf(-g[r], r_[mt][r], v[mt][r]);
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
    // (the diagonal of T', beta, last: what the earlier tokens take away is small beside it)
    bool whole = true;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const f32x4 bt = *reinterpret_cast<const f32x4*>(&Gs[2 * DC + 16 * mt + 4 * q]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        u[mt][r] = fmaf(bt[r], r_[mt][r], u[mt][r]);
        whole &= isfinite(u[mt][r]);
      }
    }
    const int t0 = ch * DC;
    if (__any(!whole)) {  // a number that is none spoils the tokens from its own on, not those before it
      const int n = min(p.S - t0, DC);
#pragma unroll 1
      for (int t = 0; t < n; ++t) {
        const size_t m = ((size_t)b * p.S + t0 + t) * p.H + h;
        const float g = p.decay[m];
        float sk = 0.f, oq = 0.f;
#pragma unroll
        for (int mb = 0; mb < DB; ++mb) {
          const f32x4 k = *reinterpret_cast<const f32x4*>(&Ks[t * LK + 16 * mb + 4 * q]);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            S[mb][r] *= g;
            sk = fmaf(S[mb][r], k[r], sk);
          }
        }
        sk += __shfl_xor(sk, 16, 64);
        sk += __shfl_xor(sk, 32, 64);
        const float ut = p.beta[m] * (p.v[m * p.vdim + j] - sk);
#pragma unroll
        for (int mb = 0; mb < DB; ++mb) {
          const f32x4 k = *reinterpret_cast<const f32x4*>(&Ks[t * LK + 16 * mb + 4 * q]);
          const f32x4 x = *reinterpret_cast<const f32x4*>(&Qs[t * LK + 16 * mb + 4 * q]);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            S[mb][r] = fmaf(k[r], ut, S[mb][r]);
            oq = fmaf(S[mb][r], x[r], oq);
          }
        }
        oq += __shfl_xor(oq, 16, 64);
        oq += __shfl_xor(oq, 32, 64);
        if (q == 0) p.o[m * p.vdim + j] = oq;
      }
      continue;
    }
    f32x4 qs[2];
    times_state(Qs, qs);
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const f32x4 g = *reinterpret_cast<const f32x4*>(&Gs[16 * mt + 4 * q]);
      f32x4 in[4];
#pragma unroll
      for (int kb = 0; kb <= mt; ++kb) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(&Ts[(DC + 16 * mt + c) * LT + 16 * kb + 4 * q]);
#pragma unroll
        for (int r = 0; r < 4; ++r) in[r] = mma_f32(a[r], u[kb][r], kb ? in[r] : f32x4{0.f, 0.f, 0.f, 0.f});
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float o = fmaf(qs[mt][r], g[r], (in[0][r] + in[1][r]) + (in[2][r] + in[3][r]));
        if (t0 + 16 * mt + 4 * q + r < p.S) (obase + ((size_t)t0 + 16 * mt + r) * vstep)[at_v] = o;
      }
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
      f32x4 add[4];  // what the tokens add, four short chains: one onto S itself would round S at every token
#pragma unroll
      for (int tb = 0; tb < 2; ++tb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          add[r] = mma_f32(Ks[(16 * tb + 4 * q + r) * LK + 16 * mb + c], u[tb][r], tb ? add[r] : f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int r = 0; r < 4; ++r) S[mb][r] = fmaf(S[mb][r], glast, (add[0][r] + add[1][r]) + (add[2][r] + add[3][r]));
    }
  }
  if (!live) return;
  float* to = sp;
  asm volatile("" : "+s"(to));  // (the addresses are formed again: kept through the walk they would take 64 registers)
#pragma unroll
  for (int mb = 0; mb < DB; ++mb)
#pragma unroll
    for (int r = 0; r < 4; ++r) (to + (size_t)(16 * mb + r) * p.vdim)[at_s] = S[mb][r];
}

// What a walk of chunks reads and writes, for the delta rule and for scalar gates (mlstm): token m, head h at x + m * ldx + hx *
// dim, hx the key head.
struct ChunkWalk {
  const float* q;
  int ldq;
  const float* k;
  int ldk;
  const float* v;  // token m, head h at v + m * ldv + h * vdim; a column vdim (ncols = vdim + 1) is 1
  int ldv;
  const float* ws;
  const float* decay;  // [B * S, H]
  const float* write;  // [B * S, H]: beta, or the scalar gates' write factors
  float* state;  // [B, H, dim, ncols]
  float* o;      // [M, H, ncols]
  int S, H, heads_per_key, vdim, ncols, chunks;
  float o_scale;
};

// The walk where its waves would leave SIMDs idle: the four waves of a workgroup share 16 value columns, each holds a quarter of
// the key rows of their state (DBW 16-row blocks), and the two products that sum over the key rows (K S and Q S) meet in LDS
// once per chunk. Operands come straight from memory, a chunk ahead, their loads between a chunk's first products: 43 of them in one
// run keep the four waves waiting for the memory path. A chunk's chain per wave at dim 128 is 76 MFMAs instead
// of 216; 2048 tokens of one row, 16 heads of 128 x 128: 316 -> 218 us with the delta rule's first launch; loads between the products, an output's
// place formed once and sums in the vector unit's registers (build.py) 233 -> 195 (another day's clock), scalar gates 140 -> 111, 777 tokens 64 -> 53.
// grid (H, ceil(ncols / 16), B): workgroups go round the XCDs by their id, so a head's columns mostly share one L2.
// DELTA 0 (scalar gates): u = v, no K S.
template <int DBW, int DELTA>
__global__ void __launch_bounds__(256) chunk_walk_split_kernel(ChunkWalk p) {
  constexpr int D = 64 * DBW, NP = DELTA ? 4 : 2, WS = DELTA ? DC_WS : DC_WS_SCALAR, OFF_M = DELTA ? DC * DC : 0,
                OFF_G = OFF_M + DC * DC;
  __shared__ f32x4 red[2][4][NP][64];  // [buffer][wave][Q S of both token tiles, K S of both][lane]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, q = lane >> 4;
  const int h = blockIdx.x, b = blockIdx.z, kh = h / p.heads_per_key;
  const int j = 16 * blockIdx.y + c, jv = min(j, p.vdim - 1), js = min(j, p.ncols - 1);
  const int d0 = 16 * DBW * wave;  // this wave's key rows
  float* sp = p.state + ((size_t)b * p.H + h) * D * p.ncols + js;
  f32x4 S[DBW];
#pragma unroll
  for (int mb = 0; mb < DBW; ++mb)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[mb][r] = sp[(size_t)(d0 + 16 * mb + 4 * q + r) * p.ncols];

  // a chunk's first rows and workspace (uniform), and this lane's places behind them: only the uniform part moves
  const float* qp = p.q + (size_t)b * p.S * p.ldq + (size_t)kh * D + d0;
  const float* kp = p.k + (size_t)b * p.S * p.ldk + (size_t)kh * D + d0;
  const float* vp = p.v + (size_t)b * p.S * p.ldv + (size_t)h * p.vdim;
  const float* wp = p.ws + ((size_t)b * p.H + h) * p.chunks * WS;
  const int mt_o = wave & 1;  // the token tile whose output waves 0 and 1 finish
  float* const op = p.o + ((size_t)b * p.S * p.H + h) * p.ncols;
  unsigned oo[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) oo[r] = (unsigned)(16 * mt_o + 4 * q + r) * (unsigned)p.H * (unsigned)p.ncols + (unsigned)j;
  unsigned oq[2], oa[2], ok[2][4], ov[2][4];
  auto places = [&](int left) {  // rows of a chunk with `left` tokens (further ones repeat the last: their u is 0)
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const int m = min(16 * mt + c, left - 1);
      oq[mt] = (unsigned)(m * p.ldq + 4 * q);
      oa[mt] = (unsigned)(m * p.ldk + 4 * q);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = min(16 * mt + 4 * q + r, left - 1);
        ok[mt][r] = (unsigned)(t * p.ldk + c);
        ov[mt][r] = (unsigned)(t * p.ldv + jv);
      }
    }
  };
  struct Operands {
    f32x4 ka[DELTA ? DBW : 1][2], qa[DBW][2], ta[DELTA ? 3 : 1], ma[2], ga[2], wa[2], ba[DELTA ? 2 : 1];
    float kt[DBW][2][4], va[2][4], glast;
  };
  const unsigned row = (unsigned)(c * DC + 4 * q);
  auto fetch = [&](Operands& x, bool last) {  // a chunk on its way to registers; the pointers go to the next one behind it
#pragma unroll
    for (int kb = 0; kb < DBW; ++kb)
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        if (DELTA) x.ka[kb][mt] = *reinterpret_cast<const f32x4*>(kp + oa[mt] + 16 * kb);
        x.qa[kb][mt] = *reinterpret_cast<const f32x4*>(qp + oq[mt] + 16 * kb);
      }
    if (DELTA) {
      x.ta[0] = *reinterpret_cast<const f32x4*>(wp + row);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) x.ta[DELTA ? 1 + kb : 0] = *reinterpret_cast<const f32x4*>(wp + row + 16 * DC + 16 * kb);
    }
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) x.ma[kb] = *reinterpret_cast<const f32x4*>(wp + OFF_M + 16 * mt_o * DC + row + 16 * kb);
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      x.ga[mt] = *reinterpret_cast<const f32x4*>(wp + (unsigned)(4 * q) + OFF_G + 16 * mt);
      x.wa[mt] = *reinterpret_cast<const f32x4*>(wp + (unsigned)(4 * q) + OFF_G + DC + 16 * mt);
      if (DELTA) x.ba[DELTA ? mt : 0] = *reinterpret_cast<const f32x4*>(wp + (unsigned)(4 * q) + OFF_G + 2 * DC + 16 * mt);
    }
    x.glast = DELTA ? wp[OFF_G + DC - 1] : wp[OFF_G + 2 * DC];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x.va[mt][r] = vp[ov[mt][r]];
#pragma unroll
        for (int mb = 0; mb < DBW; ++mb) x.kt[mb][mt][r] = kp[ok[mt][r] + 16 * mb];
      }
    const int on = last ? 0 : DC;  // (no branch, which would keep the loads in front of the products)
    qp += (size_t)(unsigned)on * (unsigned)p.ldq;
    kp += (size_t)(unsigned)on * (unsigned)p.ldk;
    vp += (size_t)(unsigned)on * (unsigned)p.ldv;
    wp += (unsigned)on * (unsigned)(WS / DC) + (on ? (unsigned)(WS % DC) : 0u);
  };
  // chunk ch token by token: a number that is none spoils the tokens from its own on, not those before it. Every wave of the
  // workgroup comes here together.
  auto by_token = [&](int ch) {
    __syncthreads();  // (the chunk's exchange has been read)
    float* const ex = reinterpret_cast<float*>(red);  // [2][4 waves][16 columns] read-outs, then the same of S^T k
    const int end = min(p.S, (ch + 1) * DC);
#pragma unroll 1
    for (int t = ch * DC; t < end; ++t) {
      const size_t m = (size_t)b * p.S + t, mh = m * p.H + h;
      const float* kr = p.k + m * p.ldk + (size_t)kh * D + d0 + 4 * q;
      const float* qr = p.q + m * p.ldq + (size_t)kh * D + d0 + 4 * q;
      const float g = p.decay[mh], v = j < p.vdim ? p.v[m * p.ldv + (size_t)h * p.vdim + j] : 1.f;
      float sk = 0.f, oq = 0.f, u = p.write[mh];
#pragma unroll
      for (int mb = 0; mb < DBW; ++mb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          S[mb][r] *= g;
          if (DELTA) sk = fmaf(S[mb][r], kr[16 * mb + r], sk);
        }
      if (DELTA) {
        sk += __shfl_xor(sk, 16, 64);
        sk += __shfl_xor(sk, 32, 64);
        if (q == 0) ex[128 + 16 * wave + c] = sk;
        __syncthreads();
        sk = (ex[128 + c] + ex[144 + c]) + (ex[160 + c] + ex[176 + c]);
        u *= v - sk;
      } else {
        u *= v;
      }
#pragma unroll
      for (int mb = 0; mb < DBW; ++mb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          S[mb][r] = fmaf(kr[16 * mb + r], u, S[mb][r]);
          oq = fmaf(S[mb][r], qr[16 * mb + r], oq);
        }
      oq += __shfl_xor(oq, 16, 64);
      oq += __shfl_xor(oq, 32, 64);
      float* const eo = ex + 64 * (t & 1);
      if (q == 0) eo[16 * wave + c] = oq;
      __syncthreads();
      if (wave == 0 && q == 0 && j < p.ncols)
        p.o[mh * p.ncols + j] = ((eo[c] + eo[16 + c]) + (eo[32 + c] + eo[48 + c])) * (DELTA ? 1.f : p.o_scale);
    }
    __syncthreads();
  };
  // chunk ch, with the loads of the next one between its first products: in front of them the waves would wait for the memory
  // path to take all of them (behind the last chunk: that one again, unused)
  constexpr int FIRST = (DELTA ? 16 : 8) * DBW, LOADS = DELTA ? 12 * DBW + 19 : 10 * DBW + 14;
  auto step = [&](const Operands& x, Operands& xn, int ch, int buf) {
    const int next = min(ch + 1, p.chunks - 1);
    if ((next + 1) * DC > p.S) places(p.S - next * DC);
    fetch(xn, next + 1 == p.chunks);
    f32x4 qs[2][4], ks[2][4];  // (short chains)
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int a = 0; a < 4; ++a) qs[mt][a] = ks[mt][a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < DBW; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
          if (DELTA) ks[mt][r] = mma_f32(x.ka[kb][mt][r], S[kb][r], ks[mt][r]);
          qs[mt][r] = mma_f32(x.qa[kb][mt][r], S[kb][r], qs[mt][r]);
        }
#pragma unroll
    for (int i = 0; i < FIRST; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // a product, then its share of the loads
      __builtin_amdgcn_sched_group_barrier(0x020, (LOADS + FIRST - 1) / FIRST, 0);
    }
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      red[buf][wave][mt][lane] = (qs[mt][0] + qs[mt][1]) + (qs[mt][2] + qs[mt][3]);
      if (DELTA) red[buf][wave][DELTA ? 2 + mt : 0][lane] = (ks[mt][0] + ks[mt][1]) + (ks[mt][2] + ks[mt][3]);
    }
    __syncthreads();  // (one per chunk: the other buffer's readers are past it)
    f32x4 u[2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) u[mt][r] = ch * DC + 16 * mt + 4 * q + r < p.S ? (j < p.vdim ? x.va[mt][r] : 1.f) : 0.f;
    if (DELTA) {
      f32x4 r_[2];
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        constexpr int K0 = DELTA ? 2 : 0;
        const f32x4 k = (red[buf][0][K0 + mt][lane] + red[buf][1][K0 + mt][lane]) + (red[buf][2][K0 + mt][lane] + red[buf][3][K0 + mt][lane]);
#pragma unroll
        for (int r = 0; r < 4; ++r) r_[mt][r] = fmaf(-x.ga[mt][r], k[r], u[mt][r]);
        u[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        u[0] = mma_f32(x.ta[0][r], r_[0][r], u[0]);
        u[1] = mma_f32(x.ta[DELTA ? 1 : 0][r], r_[0][r], u[1]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) u[1] = mma_f32(x.ta[DELTA ? 2 : 0][r], r_[1][r], u[1]);
      // (the diagonal of T', beta, last: what the earlier tokens take away is small beside it)
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) u[mt][r] = fmaf(x.ba[DELTA ? mt : 0][r], r_[mt][r], u[mt][r]);
    }
    bool whole = DELTA || isfinite(x.wa[0][0]);  // (all waves hold the same u and the same gates)
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) whole &= isfinite(u[mt][r]);
    if (__any(!whole)) return by_token(ch);
    if (wave < 2) {  // o of token tile mt_o
      f32x4 o = (red[buf][0][mt_o][lane] + red[buf][1][mt_o][lane]) + (red[buf][2][mt_o][lane] + red[buf][3][mt_o][lane]);
      const f32x4 g = mt_o ? x.ga[1] : x.ga[0];
      f32x4 in[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) in[r] = mma_f32(x.ma[0][r], u[0][r], f32x4{0.f, 0.f, 0.f, 0.f});
      if (mt_o) {
#pragma unroll
        for (int r = 0; r < 4; ++r) in[r] = mma_f32(x.ma[1][r], u[1][r], in[r]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = fmaf(o[r], g[r], (in[0][r] + in[1][r]) + (in[2][r] + in[3][r]));
      float* const to = op + (size_t)ch * DC * p.H * p.ncols;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (j < p.ncols && ch * DC + 16 * mt_o + 4 * q + r < p.S) to[oo[r]] = DELTA ? o[r] : o[r] * p.o_scale;
    }
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) u[mt][r] *= x.wa[mt][r];
    f32x4 add[DBW][4];  // what the tokens add, four short chains: one onto S itself would round S at every token
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
      for (int mb = 0; mb < DBW; ++mb)
#pragma unroll
        for (int r = 0; r < 4; ++r) add[mb][r] = mma_f32(x.kt[mb][tb][r], u[tb][r], tb ? add[mb][r] : f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int mb = 0; mb < DBW; ++mb)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        S[mb][r] = fmaf(S[mb][r], x.glast, (add[mb][0][r] + add[mb][1][r]) + (add[mb][2][r] + add[mb][3][r]));
  };
  // two sets of operands in turn: moved from one set to another, a chunk's loads would be waited for at the end of each step
  Operands x0, x1;
  places(min(p.S, DC));
  fetch(x0, p.chunks == 1);
  for (int ch = 0; ch < p.chunks; ch += 2) {
    step(x0, x1, ch, 0);
    if (ch + 1 < p.chunks) step(x1, x0, ch + 1, 1);
  }
  if (j < p.ncols) {
#pragma unroll
    for (int mb = 0; mb < DBW; ++mb)
#pragma unroll
      for (int r = 0; r < 4; ++r) sp[(size_t)(d0 + 16 * mb + 4 * q + r) * p.ncols] = S[mb][r];
  }
}

// Scalar gates, step (1): one wave per (chunk, head, row). With keep_t and write_t of a token and P(t, i) the product of the keeps
// of i + 1 .. t:  o_t = (G_t S0^T q_t + sum_{i <= t} P(t, i) write_i (q_t . k_i) v_i) q_scale,  S = G_last S0 + sum_i P(last, i)
// write_i k_i v_i^T.
template <int DB>
__global__ void __launch_bounds__(256, 2) scalar_chunk_kernel(LinScan p, float* ws, int chunks) {
  __shared__ __attribute__((aligned(16))) double lp[4][DC][DC + 1];  // P(t, i) write_i
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ch = blockIdx.x * 4 + wave, h = blockIdx.y, b = blockIdx.z;
  if (ch >= chunks) return;  // (no barrier below: waves share nothing)
  const int t0 = ch * DC, c = lane & 15, q = lane >> 4;
  const size_t m0 = (size_t)b * p.S + t0;
  float* out = ws + (((size_t)b * p.H + h) * chunks + ch) * DC_WS_SCALAR;
  f32x4 part[3][8];  // (eight short chains per block: a long one would lose a bit to the token-by-token form)
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int r = 0; r < 8; ++r) part[x][r] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool in0 = t0 + c < p.S, in1 = t0 + 16 + c < p.S;
  const size_t r0 = m0 + (in0 ? c : 0), r1 = m0 + (in1 ? 16 + c : 0);
  const int at = h * 16 * DB + 4 * q;
#pragma unroll
  for (int kb = 0; kb < DB; ++kb) {
    const f32x4 k0 = dc_load4(p.k + r0 * p.ldk + at + 16 * kb, in0), k1 = dc_load4(p.k + r1 * p.ldk + at + 16 * kb, in1);
    const f32x4 q0 = dc_load4(p.q + r0 * p.ldq + at + 16 * kb, in0), q1 = dc_load4(p.q + r1 * p.ldq + at + 16 * kb, in1);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int a = 4 * (kb & 1) + r;
      part[0][a] = mma_f32(q0[r], k0[r], part[0][a]);
      part[1][a] = mma_f32(q1[r], k0[r], part[1][a]);
      part[2][a] = mma_f32(q1[r], k1[r], part[2][a]);
    }
  }
  // lane i: the running products behind token i (lane DC: from the chunk's start)
  const bool mine = lane < DC && t0 + lane < p.S;
  const size_t mr = m0 + (mine ? lane : 0);
  const float keep = mine ? p.decay[mr * p.H + h] : 1.f, write = mine ? p.write[mr * p.H + h] : 0.f;
  const double first = lane < DC ? write : 1.f;
  double run = first;
#pragma unroll
  for (int t = 0; t < DC; ++t) {
    const float kt = __shfl(keep, t, 64);
    run = (lane < t || lane == DC) ? run * kt : first;
    if (lane < DC) lp[wave][t][lane] = lane <= t ? run : 0.0;
    else if (lane == DC) out[DC * DC + t] = (float)run;
  }
  if (lane == DC) out[DC * DC + 2 * DC] = (float)run;  // G_last
  __builtin_amdgcn_wave_barrier();  // (LDS is the wave's own and in order)
  bool whole = isfinite(keep) && isfinite(write);  // (a number that is none in a token's key or query shows in its own products)
#pragma unroll
  for (int x = 0; x < 4; ++x) {  // (block 3, above the diagonal: zeros)
    const int rb = x == 1 || x == 2 ? 16 : 0, cb = x >= 2 ? 16 : 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = rb + 4 * q + r, i = cb + c;
      const double qk = x < 3 ? dc_total(part[x < 3 ? x : 0], r) : 0.0;
      whole &= isfinite(qk);
      out[t * DC + i] = x < 3 ? (float)(lp[wave][t][i] * qk) : 0.f;
    }
  }
  const bool spoiled = __any(!whole);
  if (lane < DC) out[DC * DC + DC + lane] = spoiled ? NAN : (float)run;  // P(last, i) write_i; the walk takes a spoiled chunk by token
}

// Waves (16 value columns each) from which the walk that keeps a whole column in one wave fills the SIMDs
constexpr long long DC_WHOLE_WAVES = 1024;
static bool dc_splits(int B, int H, int ncols) { return (long long)B * H * ((ncols + 15) / 16) < DC_WHOLE_WAVES; }

// Scalar gates in chunks win over the token-by-token scan from a chunk on (16 heads of 128 x 128, one row, us: 32 tokens 28.4 -> 14.5,
// 777 192 -> 62, 2048 467 -> 139; 8 rows of 2048 2633 -> 746), as long as the scan cannot cut the sequence into many more
// segments side by side than a walk can make up for (4 heads of 64 x 64, 4096 tokens, 64 segments: 102 -> 206; two passes of
// 0.7 us per token against 2.1 us per chunk meet at about 21 segments).
constexpr int DC_SCALAR_MIN_TOKENS = 32, DC_SCALAR_MAX_SEGMENTS = 16;

long long hy_scalar_chunk_floats(const LinScan& p) {
  auto ok = [](const float* x, int ld) { return ((uintptr_t)x & 15) == 0 && ld % 4 == 0; };
  if (p.mode != 0 || p.nseg > DC_SCALAR_MAX_SEGMENTS || p.B < 1 || p.S < DC_SCALAR_MIN_TOKENS || p.H < 1 || (p.dim != 64 && p.dim != 128) || p.vdim < 1 || p.H > 65535 ||
      p.B > 65535 || !p.write || p.ldq < p.H * p.dim || p.ldk < p.H * p.dim || p.ldv < p.H * p.vdim || !ok(p.q, p.ldq) || !ok(p.k, p.ldk))
    return 0;
  return (long long)p.B * p.H * ((p.S + DC - 1) / DC) * DC_WS_SCALAR;
}

int hy_scalar_chunk(const LinScan& p, float* ws, hipStream_t s) {
  if (hy_scalar_chunk_floats(p) == 0) return -1;
  if ((uintptr_t)ws & 15) return -2;
  const int chunks = (p.S + DC - 1) / DC, ncols = p.vdim + 1;
  const ChunkWalk w{p.q, p.ldq, p.k, p.ldk, p.v, p.ldv, ws, p.decay, p.write, p.state, p.o, p.S, p.H, 1, p.vdim, ncols, chunks, p.q_scale};
  const dim3 g1((chunks + 3) / 4, p.H, p.B), g2(p.H, (ncols + 15) / 16, p.B);
  if (p.dim == 128) {
    scalar_chunk_kernel<8><<<g1, 256, 0, s>>>(p, ws, chunks);
    chunk_walk_split_kernel<2, 0><<<g2, 256, 0, s>>>(w);
  } else {
    scalar_chunk_kernel<4><<<g1, 256, 0, s>>>(p, ws, chunks);
    chunk_walk_split_kernel<1, 0><<<g2, 256, 0, s>>>(w);
  }
  JLA_CHECK_LAUNCH();
  return 0;
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
  const dim3 g1((chunks + 3) / 4, p.H, p.B), g2(p.H, (p.vdim + 63) / 64, p.B);
  if (p.dim == 128) delta_chunk_kernel<8><<<g1, 256, 0, s>>>(p, ws, chunks);
  else delta_chunk_kernel<4><<<g1, 256, 0, s>>>(p, ws, chunks);
  if (dc_splits(p.B, p.H, p.vdim)) {
    const ChunkWalk w{p.qn, p.G * p.dim, p.kn, p.G * p.dim, p.v, p.H * p.vdim, ws, p.decay, p.beta, p.state, p.o, p.S, p.H, p.H / p.G, p.vdim, p.vdim, chunks, 1.f};
    const dim3 g3(p.H, p.vdim / 16, p.B);
    if (p.dim == 128) chunk_walk_split_kernel<2, 1><<<g3, 256, 0, s>>>(w);
    else chunk_walk_split_kernel<1, 1><<<g3, 256, 0, s>>>(w);
  } else {
    if (p.dim == 128) delta_walk_kernel<8><<<g2, 256, 0, s>>>(p, ws, chunks);
    else delta_walk_kernel<4><<<g2, 256, 0, s>>>(p, ws, chunks);
  }
  JLA_CHECK_LAUNCH();
  return 0;
}

}  // namespace jla
