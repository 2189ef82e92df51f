// One token of a matrix-state recurrence, from its gates to the gated head norm, in one launch: a decode step's counterpart
// of the scans (recurrent.hip, delta_rule.hip) and of the kernels on both sides of them. Everything fp32.
//
// With the state S [dim, vdim] of a head all four recurrences are   S' = a S + b w^T,   o = c S + e w,
//     exponential gates   a = keep, b = write k, w = v, c = keep q, e = sum write k q   (and the same with w = 1: the normaliser)
//     time mix            a_d = exp(-exp(pre + w0)), b = k, w = v, c = r, e = sum u k r   (read before the write)
//     running memory      b = room sigmoid(-(pre + bias)), a = 1 - b, w = v, c = (1 - b) silu(q), e = sum b silu(q)
//     delta rule          a = g, b = k, w = beta (v - g S^T k), c = g q, e = k . q
// so one pass over the old state gives the read-out (and the delta rule's S^T k), and it is written back from registers.
// What bounds it: the launch and one trip to memory. A scan kernel spends 10-14 us on one token (its staging plan, chunks
// and segments are for many), with its gate kernel and its norm 14-25 us; here a workgroup per (head, row) has the whole
// state in flight at once (16 numbers per thread at 128 x 128) and takes 6.8 us with exponential gates (gates 6.2 + scan
// 14.2 + norm 4.4 before), 6.4 us with the delta rule (scan 9.8 + norm 4.4), one row of 128 x 128 heads. Error of the output
// against 64 bits, scan and norm -> here: delta rule 1.11e-7 -> 1.02e-7, time mix 1.12e-7 -> 1.02e-7, running memory 9.0e-8 ->
// 8.2e-8 (with the slices added in 32 bits 1.20e-7, 1.16e-7, 9.4e-8).
#include "hy_util.h"
#include "hybrid.h"

namespace jla {

constexpr int RS_THREADS = 1024, RS_MAX = 256;
enum { RS_MLSTM = 0, RS_TIMEMIX = 1, RS_RUNNING = 2, RS_DELTA = 3, RS_CONV = 4 };  // (RS_CONV: the delta rule from its projection)
constexpr int RS_TAPS = 4;

// Sums of N numbers per thread over the first `nw` waves of the block; red holds 16 N floats. Every thread gets them.
template <int N>
JLA_DEV void rs_sum(float (&v)[N], int nw, float* red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = wave_sum(v[i]);
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < N; ++i) red[wave * N + i] = v[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = 0.f;
  for (int w = 0; w < nw; ++w) {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] += red[w * N + i];
  }
}

// sum_r w[d, r] x[r] of key row d = t / lanes, over lanes (a power of two up to 64) adjacent threads; every one of them gets it
JLA_DEV float rs_low_rank(const RecStep& p, int b, size_t d, int lane, int lanes) {
  const float* x = p.pre_x + (size_t)b * p.rank;
  float s = 0.f;
  for (int r = 4 * lane; r < p.rank; r += 4 * lanes) {
    const f32x4 xv = *reinterpret_cast<const f32x4*>(x + r);
    if (p.pre_bf16) {
      const u32x2 wv = *reinterpret_cast<const u32x2*>(reinterpret_cast<const bf16_t*>(p.pre_w) + d * p.rank + r);
      s = fmaf(bf2f(f2bf(xv[0])), __uint_as_float(wv[0] << 16), s);
      s = fmaf(bf2f(f2bf(xv[1])), __uint_as_float(wv[0] & 0xffff0000u), s);
      s = fmaf(bf2f(f2bf(xv[2])), __uint_as_float(wv[1] << 16), s);
      s = fmaf(bf2f(f2bf(xv[3])), __uint_as_float(wv[1] & 0xffff0000u), s);
    } else {
      const f32x4 wv = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(p.pre_w) + d * p.rank + r);
#pragma unroll
      for (int i = 0; i < 4; ++i) s = fmaf(xv[i], wv[i], s);
    }
  }
  for (int o = 1; o < lanes; o <<= 1) s += __shfl_xor(s, o, 64);
  return s;
}

// SiLU of the short convolution of channel c at this token; x: its inputs, the carried ones first
JLA_DEV float rs_conv(const RecStep& p, int b, int c, float (&x)[RS_TAPS]) {
  const int C = 2 * p.G * p.dim + p.H * p.vdim;
  const float* tail = p.conv_state + ((size_t)b * C + c) * (RS_TAPS - 1);
#pragma unroll
  for (int i = 0; i < RS_TAPS - 1; ++i) x[i] = tail[i];
  x[RS_TAPS - 1] = p.proj[(size_t)b * p.ldproj + c];
  const f32x4 w = *reinterpret_cast<const f32x4*>(p.conv_w + (size_t)c * RS_TAPS);
  float y = 0.f;
#pragma unroll
  for (int i = 0; i < RS_TAPS; ++i) y = fmaf(w[i], x[i], y);
  return hy_silu(y);
}
JLA_DEV void rs_conv_carry(const RecStep& p, int b, int c, const float (&x)[RS_TAPS]) {
  const int C = 2 * p.G * p.dim + p.H * p.vdim;
  float* tail = p.conv_state + ((size_t)b * C + c) * (RS_TAPS - 1);
#pragma unroll
  for (int i = 0; i < RS_TAPS - 1; ++i) tail[i] = x[i + 1];
}

// grid (H, B). Thread -> value column j = t % cw, key rows [RPT s, RPT s + RPT) of slice s = t / cw (cw: vdim rounded up to
// whole waves).
template <int MODE, int RPT>
__global__ void __launch_bounds__(RS_THREADS) rec_step_kernel(RecStep p, int cw) {
  __shared__ float la[RS_MAX], lb[RS_MAX], lc[RS_MAX], lw[RS_MAX];
  constexpr bool DELTA = MODE == RS_DELTA || MODE == RS_CONV;
  __shared__ float part[(DELTA ? 2 : 1) * RS_THREADS];
  __shared__ float red[4 * 16];
  const int t = threadIdx.x, h = blockIdx.x, b = blockIdx.y;
  const int dim = p.dim, vdim = p.vdim, ncols = MODE == RS_MLSTM ? vdim + 1 : vdim;
  const int sl = t / cw, j = t - sl * cw, d0 = sl * RPT;
  const bool col = j < vdim;
  float* const st = p.state + ((size_t)b * p.H + h) * dim * ncols;
  float S[RPT];
#pragma unroll
  for (int i = 0; i < RPT; ++i) S[i] = st[(size_t)min(d0 + i, dim - 1) * ncols + (col ? j : 0)];
  const bool key = t < dim;
  const int td = key ? t : 0;
  const int kh = DELTA ? h / (p.H / p.G) : h;
  float v = 0.f, q = 0.f, k = 0.f;
  float xq[RS_TAPS], xk[RS_TAPS];  // RS_CONV: the inputs of this thread's query and key channel, which the key head's heads share
  int before = 0;                  // ... and how many of those heads have read the carried ones
  if (MODE == RS_CONV) {
    const int QK = p.G * dim;
    if (t < cw) {
      float xv[RS_TAPS];
      const int c = 2 * QK + h * vdim + (col ? j : 0);
      v = rs_conv(p, b, c, xv);
      if (col) rs_conv_carry(p, b, c, xv);  // (this thread is the channel's only reader)
    }
    if (key) {
      q = rs_conv(p, b, kh * dim + t, xq);
      k = rs_conv(p, b, QK + kh * dim + t, xk);
    }
  } else {
    v = p.v[(size_t)b * p.ldv + (size_t)h * vdim + (col ? j : 0)];
    q = p.q[(size_t)b * p.ldq + (size_t)kh * dim + td];
    k = MODE == RS_RUNNING ? 0.f : p.k[(size_t)b * p.ldk + (size_t)kh * dim + td];
  }
  // the head's vectors over its key rows, and the sums that need them
  float e[2] = {0.f, 0.f};  // e; exponential gates: the normaliser's read-out
  float floor_ = 0.f, m_new = 0.f, g = 0.f, beta = 0.f;
  if (MODE == RS_MLSTM) {
    const float xi = p.gate_i[(size_t)b * p.ldgate + h], xf = p.gate_f[(size_t)b * p.ldgate + h];
    const float zs = st[(size_t)td * ncols + vdim], m = p.mstate[(size_t)b * p.H + h];
    const float a = p.cap * tanhf((xi + p.gate_bias[h]) * (1.f / p.cap));
    const float f = hy_logsigmoid(p.cap * tanhf((xf + p.gate_bias[p.H + h]) * (1.f / p.cap)));
    m_new = fmaxf(f + m, a);
    const float keep = expf(f + m - m_new), write = expf(a - m_new), qs = q * p.q_scale, wk = write * k;
    floor_ = expf(-m_new);
    if (key) {
      la[t] = keep;
      lb[t] = wk;
      lc[t] = keep * qs;
      e[0] = wk * qs;
      e[1] = keep * zs * qs;
      st[(size_t)t * ncols + vdim] = fmaf(keep, zs, wk);  // (no other thread uses what it holds)
    }
  } else if (MODE == RS_TIMEMIX) {
    const float w0 = p.w0[(size_t)h * dim + td], u = p.u[(size_t)h * dim + td];
    float pre;
    if (p.pre_x) {  // (uniform) the decay's low-rank product here, all threads on it; the carried token row beside it
      const int lanes = 1024 / (dim <= 64 ? 64 : (dim <= 128 ? 128 : 256)), d = t / lanes;
      const float s = rs_low_rank(p, b, (size_t)h * dim + min(d, dim - 1), t % lanes, lanes);
      if (t % lanes == 0 && d < dim) lw[d] = s;
      if (p.row) {
        for (int i = h * RS_THREADS + t; i < p.width; i += p.H * RS_THREADS) p.prev[(size_t)b * p.width + i] = p.row[(size_t)b * p.width + i];
      }
      __syncthreads();
      pre = lw[td];
    } else {
      pre = p.pre[(size_t)b * p.ldpre + (size_t)h * dim + td];
    }
    if (key) {
      la[t] = expf(-expf(pre + w0));
      lb[t] = k;
      lc[t] = q;
      e[0] = u * k * q;
    }
  } else if (MODE == RS_RUNNING) {
    const float pre = p.pre[(size_t)b * p.ldpre + (size_t)h * dim + td];
    // one minus the forget gate, taken directly: a gate near 1 keeps the write factor's full accuracy
    const float wr = p.u[(size_t)h * dim + td] * hy_sigmoid(-(pre + p.w0[(size_t)h * dim + td])), qs = hy_silu(q) * p.q_scale;
    if (key) {
      lb[t] = wr;
      lc[t] = (1.f - wr) * qs;
      e[0] = wr * qs;
    }
  } else if (MODE == RS_CONV) {
    const float* row = p.proj + (size_t)b * p.ldproj + 2 * p.G * dim + 2 * p.H * vdim;
    beta = hy_sigmoid(row[h]);
    g = expf(-expf(p.a_log[h]) * hy_softplus(row[p.H + h] + p.dt_bias[h]));
    float n[2] = {q * q, k * k};  // (0 past the key rows)
    rs_sum(n, (dim + 63) / 64, red);
    // a wave has its carried inputs in registers now: it takes its ticket, whose answer is needed at the end only
    if ((t & 63) == 0 && key) before = __hip_atomic_fetch_add(p.tickets + (((size_t)b * p.G + kh) * 4 + t / 64) * 32, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    q *= 1.f / sqrtf(n[0] + 1e-6f) * (1.f / sqrtf((float)dim));
    k *= 1.f / sqrtf(n[1] + 1e-6f);
    if (key) {
      lb[t] = k;
      lc[t] = g * q;
      e[0] = k * q;
    }
    __syncthreads();  // (red is read)
  } else {
    g = p.decay[(size_t)b * p.H + h];
    beta = p.beta[(size_t)b * p.H + h];
    if (key) {
      lb[t] = k;
      lc[t] = g * q;
      e[0] = k * q;
    }
  }
  const int kw = (dim + 63) / 64;
  rs_sum(e, kw, red);  // (its barrier publishes the vectors too)
  if (MODE == RS_MLSTM && t == 0) p.mstate[(size_t)b * p.H + h] = m_new;  // (every thread has read it)
  float o[2] = {0.f, 0.f}, sk[2] = {0.f, 0.f};  // (even and odd rows: half the chain)
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    if (d0 + i < dim) {
      o[i & 1] = fmaf(S[i], lc[d0 + i], o[i & 1]);
      if (DELTA) sk[i & 1] = fmaf(S[i], lb[d0 + i], sk[i & 1]);
    }
  }
  part[t] = o[0] + o[1];
  if (DELTA) part[RS_THREADS + t] = sk[0] + sk[1];
  __syncthreads();
  const int slices = RS_THREADS / cw;
  float out = 0.f;
  if (t < cw) {
    double so = 0.0, ssk = 0.0;  // (one behind the other in 32 bits they would lose more than the scans' lane exchanges do)
    for (int s = 0; s < slices; ++s) {
      so += part[s * cw + t];
      if (DELTA) ssk += part[RS_THREADS + s * cw + t];
    }
    const float w = DELTA ? beta * (float)(v - g * ssk) : v;  // (t < cw: this thread's v is column t's)
    lw[t] = w;
    out = (float)(so + (double)e[0] * w);
    if (MODE == RS_MLSTM) out *= 1.f / (fmaxf(fabsf(e[0] + e[1]), floor_) + 1e-6f);
    if (!col) out = 0.f;
  }
  float ss[1] = {out * out};
  rs_sum(ss, cw / 64, red);  // (publishes lw; the other waves' sums are not counted)
  const float w = lw[j];
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int d = d0 + i;
    if (d < dim && col) {
      const float n = MODE == RS_RUNNING ? fmaf(lb[d], w - S[i], S[i])
                      : fmaf(DELTA ? g : la[d], S[i], lb[d] * w);
      st[(size_t)d * ncols + j] = n;
    }
  }
  if (t < vdim) {
    const float sc = 1.f / sqrtf(ss[0] / (float)vdim + p.eps);
    float gate = 1.f;
    if (p.gate_act != 2) {
      const float z = p.gate[(size_t)b * p.ldg + (size_t)h * vdim + t];
      gate = p.gate_act == 1 ? hy_sigmoid(z) : hy_silu(z);
    }
    const float y = out * sc * p.w[(p.w_heads ? (size_t)h * vdim : 0) + t] * gate * p.gain;
    const size_t at = (size_t)b * p.ldo + (size_t)h * vdim + t;
    if (p.out_bf16) reinterpret_cast<bf16_t*>(p.out)[at] = f2bf(y);
    else reinterpret_cast<float*>(p.out)[at] = y;
  }
  if (MODE == RS_CONV && key) {  // the last of the key head's heads to have read the carried inputs moves them on (nobody waits)
    const int first = __builtin_amdgcn_readfirstlane(before);
    if (first == p.H / p.G - 1) {
      rs_conv_carry(p, b, kh * dim + t, xq);
      rs_conv_carry(p, b, p.G * dim + kh * dim + t, xk);
      if ((t & 63) == 0) __hip_atomic_store(p.tickets + (((size_t)b * p.G + kh) * 4 + t / 64) * 32, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

bool hy_rec_step_takes(int dim, int vdim) {
  if (dim < 1 || vdim < 1 || dim > RS_MAX || vdim > RS_MAX) return false;
  const int cw = (vdim + 63) / 64 * 64;
  return RS_THREADS % cw == 0 && (RS_THREADS / cw) * 16 >= dim;
}

int hy_rec_step(const RecStep& p, hipStream_t s) {
  if (p.mode < 0 || p.mode > 4 || p.B < 0 || p.H < 1 || !hy_rec_step_takes(p.dim, p.vdim)) return -1;
  if (p.mode == RS_DELTA && (p.G < 1 || p.H % p.G)) return -2;
  if (p.gate_act < 0 || p.gate_act > 2 || (p.gate_act != 2 && !p.gate)) return -3;
  if (p.pre_x && (p.mode != RS_TIMEMIX || p.rank < 4 || p.rank % 4 || !p.pre_w)) return -5;
  if (p.mode == RS_CONV && (!p.proj || !p.conv_w || !p.conv_state || !p.a_log || !p.dt_bias || !p.tickets)) return -6;
  if (p.B == 0) return 0;
  if (p.B > 65535) return -4;
  const int cw = (p.vdim + 63) / 64 * 64, slices = RS_THREADS / cw;
  const int rpt = slices * 4 >= p.dim ? 4 : (slices * 8 >= p.dim ? 8 : 16);
  const dim3 grid(p.H, p.B);
#define RS_RUN(M)                                                              \
  do {                                                                         \
    if (rpt == 4) rec_step_kernel<M, 4><<<grid, RS_THREADS, 0, s>>>(p, cw);     \
    else if (rpt == 8) rec_step_kernel<M, 8><<<grid, RS_THREADS, 0, s>>>(p, cw); \
    else rec_step_kernel<M, 16><<<grid, RS_THREADS, 0, s>>>(p, cw);             \
  } while (0)
  if (p.mode == RS_MLSTM) RS_RUN(RS_MLSTM);
  else if (p.mode == RS_TIMEMIX) RS_RUN(RS_TIMEMIX);
  else if (p.mode == RS_RUNNING) RS_RUN(RS_RUNNING);
  else if (p.mode == RS_CONV) RS_RUN(RS_CONV);
  else RS_RUN(RS_DELTA);
#undef RS_RUN
  JLA_CHECK_LAUNCH();
  return 0;
}

}  // namespace jla
