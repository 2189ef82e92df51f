// The time-mix memory of a prompt (per-channel decay, bonus for the current token; heads of 64 x 64) in chunks of 16 tokens on the
// fp32 matrix cores, with the gated head norm behind it. Everything fp32.
//
//     o_t = S_(t-1)^T r_t + (sum_i u_i k_t,i r_t,i) v_t,   S_t = diag(d_t) S_(t-1) + k_t v_t^T,   d_t = exp(-exp(pre_t + w0))
// With D(a..b) the product of d_a .. d_b, a chunk that starts from S gives
//     o_t = S^T (r_t D(0..t-1)) + sum_(s<=t) P_ts v_s,   P_ts = sum_i r_t,i k_s,i D(s+1..t-1)_i,   P_tt = sum_i u_i r_t,i k_t,i
//     S' = diag(D(0..15)) S + sum_s (k_s D(s+1..15)) v_s^T
// The products of decays run forward from each key, token by token (a quotient of two running products would be 0 / 0 where a
// channel forgets at once); that and P are the vector unit's work, 16 lanes x 4 channels per key. The three sums are matrix
// products: the state lies in the accumulators of four waves (16 value columns each), row 16 tile + 4 (lane >> 4) + r, which is at
// the same time the B operand of the read-out with the key rows in that order.
// A chunk with a number that is none is taken token by token (the others neutral: r = k = v = 0, d = 1), so that only the tokens
// behind it see it.
// A long sequence is cut into segments that run side by side: every segment's own state and decay product (STATE_ONLY), one walk
// that combines them, and the segments again from the state each starts with.
// What bounds it: the chain of a chunk (stage, decays, products: 3 barriers). The scan that it replaces took 0.8 us per token of a
// segment on its staging and its lane exchanges. Errors against 64 bits, scan | here, output and state: 777 tokens, decays near
// exp(-0.05) 1.12e-7, 9.0e-8 | 9.6e-8, 7.9e-8; 64 tokens near exp(-2.7) 8.2e-8, 3.7e-8 | 7.3e-8, 2.9e-8 (with 32-bit running
// products, one chain per sum and 32-bit joins 1.32e-7, 1.0e-7 and 8.6e-8, 2.9e-8).
// Two workgroups per compute unit: without that bound the form with the norm took 181 registers and as many accumulators as held it to
// one, and 200 rows x 32 heads x 2 tokens took 153 us where the scan had taken 147; with it 101 (1500 tokens of 8 rows 575 -> 465).
#include "hy_util.h"
#include "hybrid.h"

namespace jla {

constexpr int TC_C = 16, TC_D = 64;                // tokens of a chunk, head size
constexpr int TC_P = TC_D + 4, TC_Q = TC_D + 16;  // pitch of a staged token that is read by rows; across four tokens (banks)

using f64x4 = __attribute__((ext_vector_type(4))) double;
JLA_DEV f64x4 tc_wide(const f32x4 x) { return f64x4{x[0], x[1], x[2], x[3]}; }
JLA_DEV f32x4 tc_narrow(const f64x4 x) { return f32x4{(float)x[0], (float)x[1], (float)x[2], (float)x[3]}; }
JLA_DEV float tc_dot(const f32x4 a, const f32x4 b) { return fmaf(a[0], b[0], a[1] * b[1]) + fmaf(a[2], b[2], a[3] * b[3]); }

// grid (segments, H, B); NORM: the gated head norm is applied and p.out written, else the read-out to p.s.o
template <int STATE_ONLY, int NORM>
__global__ void __launch_bounds__(256, 2) timemix_chunk_kernel(TimeMixChunk p, const float* s_init, float* s_final, float* seg_decay) {
  __shared__ __attribute__((aligned(16))) float R[TC_C][TC_P], V[TC_C][TC_Q], W[TC_C][TC_P], RT[TC_C][TC_P], KT[TC_C][TC_Q],
      O[TC_C][TC_P], PM[TC_C][20], all[TC_D];
  const LinScan& q = p.s;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, lg = lane >> 4;
  const int seg = blockIdx.x, h = blockIdx.y, b = blockIdx.z, nseg = gridDim.x;
  const int t_lo = seg * q.seg_len, t_hi = min(q.S, t_lo + q.seg_len);
  const int tt = tid >> 4, g4 = 4 * (tid & 15);  // this thread's token of a chunk and its channels
  const size_t row0 = (size_t)b * q.S;
  f32x4 S[4];
  const int rows = STATE_ONLY ? nseg + 1 : nseg;  // slots of the state array (STATE_ONLY leaves segment s in slot s + 1)
  const size_t at_in = (((size_t)b * nseg + seg) * q.H + h) * TC_D * TC_D;
  const size_t at_out = STATE_ONLY ? (((size_t)b * rows + seg + 1) * q.H + h) * TC_D * TC_D : ((size_t)b * q.H + h) * TC_D * TC_D;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      S[i][r] = STATE_ONLY ? 0.f : s_init[at_in + (size_t)(16 * i + 4 * lg + r) * TC_D + 16 * wave + c];
  const f32x4 w0 = *reinterpret_cast<const f32x4*>(q.w0 + (size_t)h * TC_D + g4);
  const f32x4 u = *reinterpret_cast<const f32x4*>(q.u + (size_t)h * TC_D + g4);
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f}, one = {1.f, 1.f, 1.f, 1.f};
  f32x4 rn, kn, vn, wn, gn = zero;
  auto fetch = [&](int t0) {  // (tokens past the segment: its last one, unused)
    const size_t m = row0 + min(t0 + tt, t_hi - 1);
    if (!STATE_ONLY) rn = *reinterpret_cast<const f32x4*>(q.q + m * q.ldq + (size_t)h * TC_D + g4);
    kn = *reinterpret_cast<const f32x4*>(q.k + m * q.ldk + (size_t)h * TC_D + g4);
    vn = *reinterpret_cast<const f32x4*>(q.v + m * q.ldv + (size_t)h * TC_D + g4);
    wn = *reinterpret_cast<const f32x4*>(q.decay + m * q.ldd + (size_t)h * TC_D + g4);
    if (NORM) gn = *reinterpret_cast<const f32x4*>(p.gate + m * p.ldg + (size_t)h * TC_D + g4);
  };
  f32x4 nw = one;
  if (NORM) nw = *reinterpret_cast<const f32x4*>(p.w + (p.w_heads ? (size_t)h * TC_D : 0) + g4);
  rn = zero;
  double seg_prod = 1.0;
  fetch(t_lo);
  for (int t0 = t_lo; t0 < t_hi; t0 += TC_C) {
    const int nt = min(TC_C, t_hi - t0);
    const f32x4 r4 = rn, k4 = kn, v4 = vn, z4 = gn;
    f32x4 d4;
    bool whole = true;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      d4[i] = expf(-expf(wn[i] + w0[i]));
      whole &= isfinite(r4[i]) && isfinite(k4[i]) && isfinite(v4[i]) && isfinite(d4[i]);
    }
    if (t0 + TC_C < t_hi) fetch(t0 + TC_C);
    const bool single = __syncthreads_or(!whole && tt < nt);  // (workgroup-uniform)
    for (int lo = 0; lo < nt; lo = single ? lo + 1 : nt) {
      const bool live = tt >= lo && tt < (single ? lo + 1 : nt);
      const f32x4 kl = live ? k4 : zero, rl = live ? r4 : zero;
      if (!STATE_ONLY) *reinterpret_cast<f32x4*>(&R[tt][g4]) = rl;
      *reinterpret_cast<f32x4*>(&V[tt][g4]) = live ? v4 : zero;
      *reinterpret_cast<f32x4*>(&W[tt][g4]) = live ? d4 : one;
      __syncthreads();
      // key tt's decays forward to every token behind it, its products with their queries, and the decays before token tt
      // (running products in 64 bits: rounded at every token they would cost the sums more than the scan's running state does)
      f64x4 kd = tc_wide(kl), A = tc_wide(one);
      const f32x4 uk = u * kl;
      float mine = 0.f;
#pragma unroll
      for (int t = 0; t < TC_C; ++t) {
        const f32x4 dt = *reinterpret_cast<const f32x4*>(&W[t][g4]);
        if (!STATE_ONLY) {
          const f32x4 rt = *reinterpret_cast<const f32x4*>(&R[t][g4]);
          const f64x4 pr = tc_wide(rt) * (t > tt ? kd : tc_wide(uk));
          const float pt = row16_sum((float)((pr[0] + pr[1]) + (pr[2] + pr[3])));
          if ((tid & 15) == t) mine = t >= tt ? pt : 0.f;
        }
        kd *= tc_wide(t > tt ? dt : one);
        A *= tc_wide(t < tt ? dt : one);
      }
      *reinterpret_cast<f32x4*>(&KT[tt][g4]) = tc_narrow(kd);
      if (!STATE_ONLY) {
        *reinterpret_cast<f32x4*>(&RT[tt][g4]) = tc_narrow(tc_wide(rl) * A);
        PM[tid & 15][tt] = mine;
      }
      if (tt == TC_C - 1) *reinterpret_cast<f32x4*>(&all[g4]) = tc_narrow(A * tc_wide(live ? d4 : one));
      __syncthreads();
      if (STATE_ONLY && tid < TC_D) seg_prod *= all[tid];
      float vb[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) vb[j] = V[4 * j + lg][16 * wave + c];  // (tokens in order: the last ones, mostly the largest, are added last)
      if (!STATE_ONLY) {
        f32x4 o[10];  // (chains of two, joined in 64 bits)
#pragma unroll
        for (int i = 0; i < 10; ++i) o[i] = zero;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f32x4 a = *reinterpret_cast<const f32x4*>(&RT[c][16 * i + 4 * lg]);
#pragma unroll
          for (int r = 0; r < 4; ++r) o[2 * i + r / 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], S[i][r], o[2 * i + r / 2], 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) o[8 + j / 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(PM[c][4 * j + lg], vb[j], o[8 + j / 2], 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          O[4 * lg + r][16 * wave + c] = (float)(((double)o[0][r] + o[1][r]) + ((double)o[2][r] + o[3][r]) + ((double)o[4][r] + o[5][r]) +
                                                 ((double)o[6][r] + o[7][r]) + ((double)o[8][r] + o[9][r]));
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f32x4 x[2] = {zero, zero};
#pragma unroll
        for (int j = 0; j < 4; ++j)
          x[j / 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(KT[4 * j + lg][16 * i + c], vb[j], x[j / 2], 0, 0, 0);
        const f32x4 dec = *reinterpret_cast<const f32x4*>(&all[16 * i + 4 * lg]);
#pragma unroll
        for (int r = 0; r < 4; ++r) S[i][r] = (float)(fma((double)dec[r], (double)S[i][r], (double)x[0][r]) + x[1][r]);
      }
      __syncthreads();
      if (!STATE_ONLY && live) {
        f32x4 x = *reinterpret_cast<const f32x4*>(&O[tt][g4]);
        const size_t m = row0 + t0 + tt;
        if (NORM) {
          const float ss = row16_sum(tc_dot(x, x));  // (the 16 lanes of a token are live together)
          const float sc = 1.f / sqrtf(ss / (float)TC_D + p.eps);
#pragma unroll
          for (int i = 0; i < 4; ++i) x[i] = x[i] * sc * nw[i] * hy_silu(z4[i]) * p.gain;
          const size_t at = m * p.ldo + (size_t)h * TC_D + g4;
          if (p.out_bf16) *reinterpret_cast<u32x2*>(reinterpret_cast<bf16_t*>(p.out) + at) = u32x2{pack2bf(x[0], x[1]), pack2bf(x[2], x[3])};
          else *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.out) + at) = x;
        } else {
          *reinterpret_cast<f32x4*>(q.o + (m * q.H + h) * TC_D + g4) = x;
        }
      }
    }
  }
  if (STATE_ONLY || seg == nseg - 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) s_final[at_out + (size_t)(16 * i + 4 * lg + r) * TC_D + 16 * wave + c] = S[i][r];
  }
  if (STATE_ONLY && tid < TC_D) seg_decay[(((size_t)b * nseg + seg) * q.H + h) * TC_D + tid] = (float)seg_prod;
}

// seg [B][nseg][H][64][64]: slot 0 <- the carried state, slot s > 0 (segment s - 1's own state) <- the state segment s starts from.
// One thread per four columns; the loads of eight segments in flight, the walk itself in 64 bits.
__global__ void __launch_bounds__(256) timemix_combine_kernel(const f32x4* state, f32x4* seg, const float* seg_decay, int nseg, int H,
                                                              int n) {
  const int e = blockIdx.x * 256 + threadIdx.x, b = blockIdx.y;  // (head, row, four columns) of row b's state
  if (e >= n) return;
  const size_t pitch = (size_t)n, at = (size_t)b * nseg * pitch + e;
  const int hr = e / (TC_D / 4);  // head * 64 + key row
  f64x4 S = tc_wide(state[(size_t)b * pitch + e]);
  seg[at] = tc_narrow(S);
  for (int s0 = 1; s0 < nseg; s0 += 8) {
    f32x4 own[8];
    float d[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int s = min(s0 + u, nseg - 1);
      own[u] = seg[at + s * pitch];
      d[u] = seg_decay[((size_t)b * (nseg - 1) + s - 1) * H * TC_D + hr];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (s0 + u >= nseg) break;
#pragma unroll
      for (int i = 0; i < 4; ++i) S[i] = fma((double)d[u], S[i], (double)own[u][i]);
      seg[at + (s0 + u) * pitch] = tc_narrow(S);
    }
  }
}

// Segments of at least a chunk, up to two workgroups per compute unit (segments of at least 32 tokens: 777 | 400 | 200 | 100 tokens of one row
// x 32 heads 55 | 39 | 31 | 30 us, here 55 | 35 | 25 | 23). Us with the norm behind it, scan | here: 1 x 32 heads, 2 | 16 | 32 | 200 | 777 | 1500 tokens
// 14 | 25 | 36 | 119 | 127 | 181, 8 | 8 | 15 | 25 | 55 | 77; 8 x 32, one segment from 512 workgroups on, 2 | 32 | 1500 tokens 15 | 38 | 1234, 8 | 25 | 465;
// 200 x 32, 2 | 3 | 16 | 32 tokens 147 | 154 | 307 | 490, 101 | 101 | 102 | 181. So every prompt of two tokens and more is taken.
constexpr int TC_TARGET = 512, TC_SEG_MIN = 16;

static void tc_segments(const LinScan& p, int& nseg, int& len) {
  const long long heads = (long long)p.B * p.H;
  long long want = TC_TARGET / heads, most = p.S / TC_SEG_MIN;
  if (want > most) want = most;
  if (want < 2) want = 1;
  len = (int)(((p.S + want - 1) / want + TC_C - 1) / TC_C * TC_C);
  nseg = (p.S + len - 1) / len;
}

bool hy_timemix_chunk_takes(const TimeMixChunk& p) {
  const LinScan& q = p.s;
  auto rows = [](const void* x, int ld) { return ((uintptr_t)x & 15) == 0 && ld % 4 == 0; };
  return q.mode == 1 && q.dim == TC_D && q.vdim == TC_D && q.S > 1 && q.B >= 1 && q.H >= 1 && q.B <= 65535 && q.H <= 65535 && rows(q.q, q.ldq) && rows(q.k, q.ldk) &&
         rows(q.v, q.ldv) && rows(q.decay, q.ldd) && rows(q.w0, 0) && rows(q.u, 0) && rows(q.state, 0) &&
         (p.norm ? rows(p.gate, p.ldg) && rows(p.w, 0) && p.ldo % 4 == 0 && ((uintptr_t)p.out & (p.out_bf16 ? 7 : 15)) == 0 : rows(q.o, 0));
}

long long hy_timemix_chunk_floats(const TimeMixChunk& p) {
  int nseg, len;
  tc_segments(p.s, nseg, len);
  const long long n = (long long)p.s.B * p.s.H * TC_D;
  return nseg > 1 ? n * TC_D * nseg + n * (nseg - 1) : 0;
}

int hy_timemix_chunk(const TimeMixChunk& p0, float* ws, hipStream_t s) {
  TimeMixChunk p = p0;
  LinScan& q = p.s;
  if (q.B < 0 || q.S < 1 || q.H < 1 || !hy_timemix_chunk_takes(p)) return -1;
  if (q.ldq < q.H * q.dim || q.ldk < q.H * q.dim || q.ldv < q.H * q.vdim || q.ldd < q.H * q.dim) return -5;
  if (q.B == 0) return 0;
  int nseg;
  tc_segments(q, nseg, q.seg_len);
  const float* init = q.state;
  if (nseg > 1) {
    if (!ws) return -7;
    float* decay = ws + (long long)q.B * q.H * TC_D * TC_D * nseg;
    timemix_chunk_kernel<1, 0><<<dim3(nseg - 1, q.H, q.B), 256, 0, s>>>(p, nullptr, ws, decay);
    JLA_CHECK_LAUNCH();
    const int n = q.H * TC_D * TC_D / 4;
    timemix_combine_kernel<<<dim3((n + 255) / 256, q.B), 256, 0, s>>>(reinterpret_cast<const f32x4*>(q.state), reinterpret_cast<f32x4*>(ws),
                                                                     decay, nseg, q.H, n);
    JLA_CHECK_LAUNCH();
    init = ws;
  }
  const dim3 grid(nseg, q.H, q.B);
  if (p.norm) timemix_chunk_kernel<0, 1><<<grid, 256, 0, s>>>(p, init, q.state, nullptr);
  else timemix_chunk_kernel<0, 0><<<grid, 256, 0, s>>>(p, init, q.state, nullptr);
  JLA_CHECK_LAUNCH();
  return 0;
}

}  // namespace jla
