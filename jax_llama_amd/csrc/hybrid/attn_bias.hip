// Attention with per-head RMS-normalised q / k / v, a position-dependent query temperature, a soft cap on the scores
// and a learned bias per key distance, over a per-layer cache of any head size (several layers may read one cache).
//
//   hy_attn_prep : from the fused projection output, per (token, head): divide q and k by their RMS over dim and v by
//                  its RMS over vdim, scale q by 1 + coef * ln(floor((p + 1) / every) + 1), write k / v into the
//                  cache at slot + s (bf16 or fp32), q to a dense fp32 buffer.
//   hy_attn_bias : scores, soft cap, distance bias, causal softmax and PV in fp32. One wave per query (prefill) walks
//                  its keys 64 at a time: a lane scores one key (q broadcast from LDS), the running maximum / sum are
//                  wave reductions, and the lanes then split the value columns. Decode (S = 1) splits the keys of a
//                  (row, head) over several waves whose partials a second kernel merges in split order.
// The bias table is indexed by distance (rows past the last repeat it), so any bucketing is a host-side table fill.
// An optional per-head sink adds exp(sink[h]) to the softmax denominator: the running maximum starts at the sink and
// the running sum at 1 (in decode, for the first key split only), so no kernel needs a branch per key for it.
// Block-local masks (chunk > 0): a query at slot i sees the keys of [floor(i / chunk) * chunk, i]; every kernel starts
// its key walk at that block's first slot, so the keys before it are never read. A per-head factor (head_scale) joins
// the score scale.
// Sliding windows (window > 0): a query at slot i sees the keys of [max(0, i - window + 1), i] and, with keep_first, the
// row's first keep_first slots. Every kernel numbers a query's visible keys 0 .. n - 1 (the kept first ones, then the
// window) and walks that numbering, so hidden keys are never read and the decode splits deal only visible keys; the MFMA
// kernel walks the kept tiles and then the window's tiles. A gate per (token, head) or per output column (sigmoid of
// projection columns) multiplies the normalised output in the kernels that write it; the output may be a column slice of
// a wider row, in fp32 or bf16. Values may be the leading columns of wider rows (ldv): a latent cache whose rows carry a
// rotated key part behind the latent serves as keys (whole row) and values (latent).
// Differential heads (maps = 2): an output head has two query / key maps over the same values; each map is a softmax of its
// own, and the head's output is RMS-normed (a1 - lambda a2) times a constant. A key row holds both maps side by side (ldk =
// 2 dim). Scores are counted per map: query head 2 h + b is map b of head h, and per-head score parameters (sink, factor,
// bias column) are indexed by it. Prefill: one wave runs both maps of its query (plain), or a pair of waves runs one map
// each over the same 32 queries and joins them through LDS (MFMA). Decode: the splits of both maps side by side, joined by
// the merge.
#include "attn_chunk.h"
#include "attn_span.h"

namespace jla {

JLA_DEV float ab_ld(const float* p) { return *p; }
JLA_DEV float ab_ld(const bf16_t* p) { return bf2f(*p); }
JLA_DEV void ab_ld8(const float* p, float* f) {
  const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
  f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w; f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
}
JLA_DEV void ab_ld8(const bf16_t* p, float* f) { unpack8(*reinterpret_cast<const u32x4*>(p), f); }
JLA_DEV void ab_st(float* p, float v) { *p = v; }
JLA_DEV void ab_st(bf16_t* p, float v) { *p = f2bf(v); }

// grid (M, ceil(items / 4)), 4 waves: wave -> item: [0, H) q heads, [H, H + G) k heads, [H + G, H + 2G) v heads
template <typename CT>
__global__ void __launch_bounds__(256) attn_prep_kernel(AttnPrep p) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = blockIdx.x, item = blockIdx.y * 4 + wave;
  const int items = p.H + (p.has_kv ? 2 * p.G : 0);
  if (item >= items) return;
  const float* row = p.proj + (size_t)m * p.ld;
  const int b = m / p.S, sidx = m - b * p.S;
  int kind, head, len, col;
  if (item < p.H) { kind = 0; head = item; len = p.dim; col = head * p.dim; }
  else if (item < p.H + p.G) { kind = 1; head = item - p.H; len = p.dim; col = p.H * p.dim + head * p.dim; }
  else { kind = 2; head = item - p.H - p.G; len = p.vdim; col = (p.H + p.G) * p.dim + head * p.vdim; }
  float sc = 1.f;
  if (kind != 2 || p.norm_v) {
    float ss = 0.f;
    for (int d = lane; d < len; d += 64) {
      const float v = row[col + d];
      ss = fmaf(v, v, ss);
    }
    ss = wave_sum(ss);
    sc = 1.f / sqrtf(ss / (float)len + p.eps);
  }
  const float* gw = kind == 0 ? p.q_w : (kind == 1 ? p.k_w : nullptr);  // gain of the norm, shared by the heads
  if (kind == 0) {
    if (p.temp_coef != 0.f) {
      const int pos = p.positions[m];
      sc *= 1.f + p.temp_coef * logf((float)((pos + 1) / p.temp_every) + 1.f);
    }
    float* q = p.q + ((size_t)m * p.H + head) * p.dim;
    for (int d = lane; d < len; d += 64) q[d] = row[col + d] * sc * (gw ? gw[d] : 1.f);
    return;
  }
  const int t = *p.slot + sidx;
  if (t < 0 || t >= p.T) return;  // cache full: the write is dropped
  CT* dst = (kind == 1 ? reinterpret_cast<CT*>(p.kc) : reinterpret_cast<CT*>(p.vc)) +
            (((size_t)b * p.G + head) * p.T + t) * len;
  for (int d = lane; d < len; d += 64) ab_st(dst + d, row[col + d] * sc * (gw ? gw[d] : 1.f));
}

// The same with 16-byte accesses, 64 / L heads per wave: bound by memory, and one number per lane and load left too little of it on
// its way (12000 tokens, 32 + 8 + 8 heads of 128: 256 -> 106 us, 32 heads without keys 178 -> 73, 2048 tokens, 16 + 4 + 4 17.7 -> 10.5).
template <typename CT, int L>
__global__ void __launch_bounds__(256) attn_prep_vec_kernel(AttnPrep p) {
  const int d = 4 * (threadIdx.x % L);
  const int m = blockIdx.x, item = blockIdx.y * (256 / L) + threadIdx.x / L;
  const int items = p.H + (p.has_kv ? 2 * p.G : 0);
  const int kind = item < p.H ? 0 : (item < p.H + p.G ? 1 : 2);
  const int head = kind == 0 ? item : (kind == 1 ? item - p.H : item - p.H - p.G);
  const int len = kind == 2 ? p.vdim : p.dim;
  const int col = kind == 2 ? (p.H + p.G) * p.dim + head * p.vdim : item * p.dim;
  const bool on = item < items && d < len;
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (on) v = *reinterpret_cast<const f32x4*>(p.proj + (size_t)m * p.ld + col + d);
  const float ss = hy_head_squares<L>(v);
  if (!on) return;
  float sc = kind != 2 || p.norm_v ? 1.f / sqrtf(ss / (float)len + p.eps) : 1.f;
  if (kind == 0 && p.temp_coef != 0.f) sc *= 1.f + p.temp_coef * logf((float)((p.positions[m] + 1) / p.temp_every) + 1.f);
  const float* gw = kind == 0 ? p.q_w : (kind == 1 ? p.k_w : nullptr);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = v[i] * sc * (gw ? gw[d + i] : 1.f);
  if (kind == 0) {
    hy_store4(p.q + ((size_t)m * p.H + head) * p.dim + d, v);
    return;
  }
  const int b = m / p.S, t = *p.slot + m - b * p.S;
  if (t < 0 || t >= p.T) return;  // cache full: the write is dropped
  hy_store4((kind == 1 ? reinterpret_cast<CT*>(p.kc) : reinterpret_cast<CT*>(p.vc)) + (((size_t)b * p.G + head) * p.T + t) * len + d, v);
}

template <typename CT>
static void attn_prep_vec(const AttnPrep& p, int L, int M, int items, hipStream_t s) {
  const dim3 grid(M, (items + 256 / L - 1) / (256 / L));
  if (L == 16) attn_prep_vec_kernel<CT, 16><<<grid, 256, 0, s>>>(p);
  else if (L == 32) attn_prep_vec_kernel<CT, 32><<<grid, 256, 0, s>>>(p);
  else attn_prep_vec_kernel<CT, 64><<<grid, 256, 0, s>>>(p);
}

int hy_attn_prep(const AttnPrep& p, hipStream_t s) {
  if (p.B < 0 || p.S < 1 || p.H < 1 || p.G < 1 || p.H % p.G || p.dim < 1 || p.vdim < 1 || p.T < 1) return -1;
  if (p.temp_coef != 0.f && p.temp_every < 1) return -2;
  const int M = p.B * p.S;
  if (M == 0) return 0;
  const int items = p.H + (p.has_kv ? 2 * p.G : 0);
  if ((items + 3) / 4 > 65535) return -3;
  const int L = p.dim % 4 || p.vdim % 4 || p.ld % 4 ? 0 : hy_head_lanes(max(p.dim, p.has_kv ? p.vdim : 0));
  if (L && !(((uintptr_t)p.proj | (uintptr_t)p.q | (uintptr_t)p.kc | (uintptr_t)p.vc) & 15)) {
    if (p.cbf16) attn_prep_vec<bf16_t>(p, L, M, items, s);
    else attn_prep_vec<float>(p, L, M, items, s);
    JLA_CHECK_LAUNCH();
    return 0;
  }
  dim3 grid(M, (items + 3) / 4);
  if (p.cbf16) attn_prep_kernel<bf16_t><<<grid, 256, 0, s>>>(p);
  else attn_prep_kernel<float><<<grid, 256, 0, s>>>(p);
  JLA_CHECK_LAUNCH();
  return 0;
}

constexpr int AB_MAX_DIM = 1024;  // q head held in LDS per wave (keys may be wider than values: a latent cache row
                                  // with a rotated part behind the latent)
constexpr int AB_MAX_VREG = 8;    // value columns per lane: vdim <= 512

// One wave: visible keys number [j_lo, j_hi) of query (b, query head h) at slot qi (span); returns the running max m, sum l and
// unnormalised acc. with_sink: the wave whose keys start the row also counts the head's sink.
template <typename CT, int VREG>  // VREG: value columns per lane (vdim <= 64 VREG)
JLA_DEV void ab_wave(const AttnBias& p, const float* qs, int b, int h, int qi, const AbSpan& span, int j_lo, int j_hi,
                     bool with_sink, float& m_run, float& l_run, float* acc) {
  constexpr int KB = VREG <= 2 ? 16 : 8;  // keys whose value rows are in flight at a time
  const int lane = threadIdx.x & 63;
  const AbMap mp = ab_map(p, h);
  const CT* kbase = reinterpret_cast<const CT*>(p.kc) + ((size_t)b * p.G + mp.g) * p.T * p.ldk + mp.koff;
  const CT* vbase = reinterpret_cast<const CT*>(p.vc) + ((size_t)b * p.G + mp.g) * p.T * p.ldv;
  const bool fastk = ((p.dim | p.ldk) & 7) == 0 && ((uintptr_t)kbase & 15) == 0;
  const bool sunk = with_sink && p.sink;
  const float hs = p.head_scale ? p.head_scale[h] : 1.f;
  m_run = sunk ? p.sink[h] : -INFINITY;
  l_run = sunk ? 1.f : 0.f;
#pragma unroll
  for (int i = 0; i < VREG; ++i) acc[i] = 0.f;
  for (int j0 = j_lo; j0 < j_hi; j0 += 64) {
    const int j = j0 + lane;
    const int kj = ab_key(span, min(j, j_hi - 1));  // cache slot of this lane's key
    float sc = -INFINITY;
    if (j < j_hi) {
      const CT* kr = kbase + (size_t)kj * p.ldk;
      float d0 = 0.f, d1 = 0.f;
      if (fastk) {  // whole 16-byte groups: branch-free loads the scheduler can batch
#pragma unroll 4
        for (int d = 0; d < p.dim; d += 8) {
          float kf[8];
          ab_ld8(kr + d, kf);
#pragma unroll
          for (int i = 0; i < 8; i += 2) {
            d0 = fmaf(qs[d + i], kf[i], d0);
            d1 = fmaf(qs[d + i + 1], kf[i + 1], d1);
          }
        }
      } else {
        for (int d = 0; d < p.dim; ++d) d0 = fmaf(qs[d], ab_ld(kr + d), d0);
      }
      sc = (d0 + d1) * p.scale * hs;
      if (p.softcap > 0.f) sc = p.softcap * tanhf(sc / p.softcap);
      if (p.bias) sc += p.bias[(size_t)min(qi - kj, p.nbias - 1) * (p.H * p.maps) + h];
    }
    const float m_new = fmaxf(m_run, wave_max(sc));
    const float corr = expf(m_run - m_new);  // first chunk: exp(-inf) = 0
    const float pr = j < j_hi ? expf(sc - m_new) : 0.f;
    l_run = l_run * corr + wave_sum(pr);
    m_run = m_new;
#pragma unroll
    for (int i = 0; i < VREG; ++i) acc[i] *= corr;
    const int nk = min(64, j_hi - j0);
    for (int jj = 0; jj < nk; jj += KB) {
      float vv[KB][VREG];
#pragma unroll
      for (int u = 0; u < KB; ++u) {
        const CT* vr = vbase + (size_t)ab_key(span, min(j0 + jj + u, j_hi - 1)) * p.ldv;
#pragma unroll
        for (int i = 0; i < VREG; ++i) {
          vv[u][i] = ab_ld(vr + min(lane + 64 * i, p.vdim - 1));  // (columns past vdim: never stored)
        }
      }
#pragma unroll
      for (int u = 0; u < KB; ++u) {
        const float pj = __shfl(pr, min(jj + u, 63), 64);  // (keys past nk have pr = 0 or repeat a row times 0)
        const float pw = jj + u < nk ? pj : 0.f;
#pragma unroll
        for (int i = 0; i < VREG; ++i) acc[i] = fmaf(pw, vv[u][i], acc[i]);
      }
    }
  }
}

// prefill of differential heads: grid (ceil(S / 4), H, B), one wave per query, its two maps one after the other
template <typename CT, int VREG>
__global__ void __launch_bounds__(256) attn_diff_prefill_kernel(AttnBias p) {
  __shared__ float qs_all[4][AB_MAX_DIM];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int s = blockIdx.x * 4 + wave, h = blockIdx.y, b = blockIdx.z;
  if (s >= p.S) return;
  float* qs = qs_all[wave];
  const size_t m = (size_t)b * p.S + s;
  const int qi = min(*p.slot + s, p.T - 1);
  const AbSpan span = ab_span(p, qi);
  float o[VREG];
#pragma unroll
  for (int i = 0; i < VREG; ++i) o[i] = 0.f;
  for (int map = 0; map < 2; ++map) {
    const float* q = p.q + (m * p.H * 2 + 2 * h + map) * p.dim;
    __builtin_amdgcn_wave_barrier();
    for (int d = lane; d < p.dim; d += 64) qs[d] = q[d];
    __builtin_amdgcn_wave_barrier();
    float m_run, l_run, acc[VREG];
    ab_wave<CT, VREG>(p, qs, b, 2 * h + map, qi, span, 0, span.n, true, m_run, l_run, acc);
    const float w = (map ? -p.diff_lambda : 1.f) / l_run;
#pragma unroll
    for (int i = 0; i < VREG; ++i) o[i] = fmaf(w, acc[i], o[i]);
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < VREG; ++i)
    if (lane + 64 * i < p.vdim) ss = fmaf(o[i], o[i], ss);
  const float sc = p.diff_gain / sqrtf(wave_sum(ss) / (float)p.vdim + p.diff_eps);
#pragma unroll
  for (int i = 0; i < VREG; ++i) {
    const int c = lane + 64 * i;
    if (c < p.vdim) ab_out(p, m, h, c, o[i] * (sc * ab_gate(p, m, h, c)));
  }
}

// prefill: grid (ceil(S / 4), H, B), one wave per query
template <typename CT, int VREG>
__global__ void __launch_bounds__(256) attn_bias_prefill_kernel(AttnBias p) {
  __shared__ float qs_all[4][AB_MAX_DIM];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int s = blockIdx.x * 4 + wave, h = blockIdx.y, b = blockIdx.z;
  if (s >= p.S) return;
  float* qs = qs_all[wave];
  const float* q = p.q + (((size_t)b * p.S + s) * p.H + h) * p.dim;
  for (int d = lane; d < p.dim; d += 64) qs[d] = q[d];
  __builtin_amdgcn_wave_barrier();
  const int qi = min(*p.slot + s, p.T - 1);
  float m_run, l_run, acc[VREG];
  const AbSpan span = ab_span(p, qi);
  ab_wave<CT, VREG>(p, qs, b, h, qi, span, 0, span.n, true, m_run, l_run, acc);
  const size_t m = (size_t)b * p.S + s;
  const float inv = 1.f / l_run;
#pragma unroll
  for (int i = 0; i < VREG; ++i) {
    const int c = lane + 64 * i;
    if (c < p.vdim) ab_out(p, m, h, c, acc[i] * (inv * ab_gate(p, m, h, c)));
  }
}

// decode: grid (splits, H maps, B), one wave per (row, query head, split); partial = [m, l, acc[vdim]]
template <typename CT, int VREG>
__global__ void __launch_bounds__(64) attn_bias_decode_kernel(AttnBias p) {
  __shared__ float qs[AB_MAX_DIM];
  const int lane = threadIdx.x;
  const int sp = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int heads = p.H * p.maps;
  const float* q = p.q + ((size_t)b * heads + h) * p.dim;
  for (int d = lane; d < p.dim; d += 64) qs[d] = q[d];
  __syncthreads();
  const int qi = min(*p.slot, p.T - 1);
  int j_lo, j_hi;
  const AbSpan span = ab_span(p, qi);
  ab_split_range(p, span, sp, j_lo, j_hi);
  float m_run, l_run, acc[VREG];
  ab_wave<CT, VREG>(p, qs, b, h, qi, span, j_lo, j_hi, sp == 0, m_run, l_run, acc);
  float* w = p.ws + (((size_t)b * heads + h) * p.splits + sp) * (p.vdim + 2);
  if (lane == 0) {
    w[0] = m_run;
    w[1] = l_run;
  }
#pragma unroll
  for (int i = 0; i < VREG; ++i) {
    const int c = lane + 64 * i;
    if (c < p.vdim) w[2 + c] = acc[i];
  }
}

// decode, bf16 caches, dim = 8 DK8 in {64, 128}, vdim = 64 VREG in {64, 128}: the same split as above with every load of
// a 64-key chunk (attn_chunk.h, and the biases) issued before the first use, and q staged into LDS
// behind them: a decode step is a chain of memory round trips, and this form has two.
template <int DK8, int VREG>
__global__ void __launch_bounds__(64) attn_bias_decode_fast_kernel(AttnBias p) {
  constexpr int dim = 8 * DK8, vdim = 64 * VREG;
  using Chunk = KeyChunk<bf16_t, DK8, VREG>;
  __shared__ float qs[dim];
  const int lane = threadIdx.x;
  const int sp = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const AbMap mp = ab_map(p, h);
  const int heads = p.H * p.maps;
  const float* q = p.q + ((size_t)b * heads + h) * dim;
  float qv[dim / 64];
#pragma unroll
  for (int i = 0; i < dim / 64; ++i) qv[i] = q[lane + 64 * i];
  const int qi = min(*p.slot, p.T - 1);
  int j_lo, j_hi;
  const AbSpan span = ab_span(p, qi);
  ab_split_range(p, span, sp, j_lo, j_hi);
  const bf16_t* kbase = reinterpret_cast<const bf16_t*>(p.kc) + ((size_t)b * p.G + mp.g) * p.T * p.ldk + mp.koff;
  const bf16_t* vbase = reinterpret_cast<const bf16_t*>(p.vc) + ((size_t)b * p.G + mp.g) * p.T * p.ldv;
  const bool sunk = p.sink && sp == 0;
  const float hs = p.head_scale ? p.head_scale[h] : 1.f;
  float m_run = sunk ? p.sink[h] : -INFINITY, l_run = sunk ? 1.f : 0.f, q8[8] = {}, acc8[8] = {};
  bool staged = false;
  for (int j0 = j_lo; j0 < j_hi; j0 += 64) {
    auto slot_of = [&](int i) { return ab_key(span, min(j0 + i, j_hi - 1)); };
    Chunk ch;
    ch.load(kbase, p.ldk, vbase, p.ldv, lane, slot_of);
    const int j = j0 + Chunk::key(lane);
    const float bl = p.bias ? p.bias[(size_t)min(qi - slot_of(Chunk::key(lane)), p.nbias - 1) * heads + h] : 0.f;
    if (!staged) {
#pragma unroll
      for (int i = 0; i < dim / 64; ++i) qs[lane + 64 * i] = qv[i];
      __syncthreads();
      staged = true;
#pragma unroll
      for (int e = 0; e < 8; ++e) q8[e] = qs[8 * (lane % DK8) + e];
    }
    float sc = ch.score(q8, lane) * p.scale * hs;
    if (p.softcap > 0.f) sc = p.softcap * tanhf(sc / p.softcap);
    sc += bl;
    if (j >= j_hi) sc = -INFINITY;
    const float m_new = fmaxf(m_run, wave_max(sc));
    const float corr = expf(m_run - m_new);
    const float pr = j < j_hi ? expf(sc - m_new) : 0.f;
    l_run = l_run * corr + wave_sum(pr);
    m_run = m_new;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc8[e] *= corr;
    ch.add(acc8, pr, lane);  // (0 for keys past the split)
  }
  float acc[VREG];
  Chunk::columns(acc8, lane, acc);
  float* w = p.ws + (((size_t)b * heads + h) * p.splits + sp) * (vdim + 2);
  if (lane == 0) {
    w[0] = m_run;
    w[1] = l_run;
  }
#pragma unroll
  for (int i = 0; i < VREG; ++i) w[2 + VREG * Chunk::vlane(lane) + i] = acc[i];
}

// decode over a shared latent: keys = values = ONE bf16 cache head (kc == vc, G == 1), rows of 136 to 512 numbers of
// which the first vdim are the values (all of them, or a latent in front of a rotated key part), no bias / soft cap. The lanes split a row's numbers, 16 bytes each, so one coalesced load per key serves both the score
// (row totals by DPP, the four rows through scalar registers: no LDS round trips) and the value sum; all loads of a
// chunk of keys are issued before the first use. A wave serves HQ heads of one row (HQ = 4 measured slower than 1 at 8
// rows x 16 heads, 94 against 58 us: four times the scalar-register traffic per key on a quarter of the waves; dealing
// the batch rows to XCDs by workgroup id, so that each L2 holds one row's latent, changed nothing: the kernel is bound
// by its own instruction stream, about 50 per key, not by what it reads).
// Grid (splits, H / HQ, B); partial layout as the kernels above.
constexpr int AL_KC = 16;
JLA_DEV float al_lane(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

template <int HQ, int KC>  // heads per wave, keys per chunk
__global__ void __launch_bounds__(64) attn_latent_decode_kernel(AttnBias p) {
  const int lane = threadIdx.x;
  const int sp = blockIdx.x, h0 = blockIdx.y * HQ, b = blockIdx.z;
  const int rank = p.dim;
  const bool on = 8 * lane < rank;
  const int c0 = on ? 8 * lane : 0;  // (surplus lanes re-read the row's start against a zero query)
  float qv[HQ][8];
#pragma unroll
  for (int q = 0; q < HQ; ++q) {
    hy_load8(p.q + ((size_t)b * p.H + h0 + q) * rank + c0, 8, qv[q]);
#pragma unroll
    for (int i = 0; i < 8; ++i) qv[q][i] = on ? qv[q][i] : 0.f;
  }
  const int qi = min(*p.slot, p.T - 1);
  int j_lo, j_hi;
  const AbSpan span = ab_span(p, qi);
  ab_split_range(p, span, sp, j_lo, j_hi);
  const bf16_t* base = reinterpret_cast<const bf16_t*>(p.kc) + (size_t)b * p.T * rank + c0;
  const bool sunk = p.sink && sp == 0;
  float m_run[HQ], l_run[HQ], acc[HQ][8], hs[HQ];
#pragma unroll
  for (int q = 0; q < HQ; ++q) {
    hs[q] = p.head_scale ? p.head_scale[h0 + q] : 1.f;
    m_run[q] = sunk ? p.sink[h0 + q] : -INFINITY;
    l_run[q] = sunk ? 1.f : 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[q][i] = 0.f;
  }
  for (int j0 = j_lo; j0 < j_hi; j0 += KC) {
    u32x4 rows[KC];
#pragma unroll
    for (int u = 0; u < KC; ++u)
      rows[u] = *reinterpret_cast<const u32x4*>(base + (size_t)ab_key(span, min(j0 + u, j_hi - 1)) * rank);
    float sc[HQ][KC], cmax[HQ];
#pragma unroll
    for (int q = 0; q < HQ; ++q) cmax[q] = -INFINITY;
#pragma unroll
    for (int u = 0; u < KC; ++u) {
      float f[8];
      unpack8(rows[u], f);
#pragma unroll
      for (int q = 0; q < HQ; ++q) {
        float d0 = 0.f, d1 = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i += 2) {
          d0 = fmaf(qv[q][i], f[i], d0);
          d1 = fmaf(qv[q][i + 1], f[i + 1], d1);
        }
        const float rt = row16_sum(d0 + d1);
        const float dot = (al_lane(rt, 0) + al_lane(rt, 16) + al_lane(rt, 32) + al_lane(rt, 48)) * p.scale * hs[q];
        sc[q][u] = j0 + u < j_hi ? dot : -INFINITY;
        cmax[q] = fmaxf(cmax[q], sc[q][u]);
      }
    }
    float m_new[HQ];
#pragma unroll
    for (int q = 0; q < HQ; ++q) {
      m_new[q] = fmaxf(m_run[q], cmax[q]);  // (a chunk holds at least one key, so m_new is finite)
      const float corr = expf(m_run[q] - m_new[q]);
      l_run[q] *= corr;
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[q][i] *= corr;
      m_run[q] = m_new[q];
    }
#pragma unroll
    for (int u = 0; u < KC; ++u) {
      float f[8];
      unpack8(rows[u], f);
#pragma unroll
      for (int q = 0; q < HQ; ++q) {
        const float pr = expf(sc[q][u] - m_new[q]);  // (0 past the split's end)
        l_run[q] += pr;
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[q][i] = fmaf(pr, f[i], acc[q][i]);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < HQ; ++q) {
    float* w = p.ws + (((size_t)b * p.H + h0 + q) * p.splits + sp) * (p.vdim + 2);
    if (lane == 0) {
      w[0] = m_run[q];
      w[1] = l_run[q];
    }
    if (on && c0 < p.vdim) {  // (the values are the row's first vdim numbers)
#pragma unroll
      for (int i = 0; i < 8; ++i) w[2 + c0 + i] = acc[q][i];
    }
  }
}

// The splits of head h of row b merged for column c (at most NS: lane sp holds split sp's maximum and sum), gated. Whole waves.
template <int NS>
JLA_DEV float ab_merge_splits(const AttnBias& p, int b, int h, int c) {
  const int lane = threadIdx.x & 63;
  const float* w = p.ws + ((size_t)b * p.H + h) * p.splits * (p.vdim + 2);
  float ms = -INFINITY, ls = 0.f;
  if (lane < p.splits) {
    ms = w[(size_t)lane * (p.vdim + 2)];
    ls = w[(size_t)lane * (p.vdim + 2) + 1];
  }
  float part[NS];
#pragma unroll
  for (int sp = 0; sp < NS; ++sp) part[sp] = w[(size_t)min(sp, p.splits - 1) * (p.vdim + 2) + 2 + c];  // one round trip
  const float gt = ab_gate(p, b, h, c);
  const float m = wave_max(ls > 0.f ? ms : -INFINITY);
  const float wt = ls > 0.f ? expf(ms - m) : 0.f;  // weight of this lane's split
  const float l = wave_sum(ls * wt);
  float a = 0.f;
#pragma unroll
  for (int sp = 0; sp < NS; ++sp) {  // (a split without keys holds zeros and has weight 0)
    const float ws = __shfl(wt, sp, 64);
    a = fmaf(part[sp], sp < p.splits ? ws : 0.f, a);
  }
  return a / l * gt;
}

// (one branch for all of it: one per 16 splits made 64 splits 0.8 us slower, all 64 without one cost few splits 1 us)
JLA_DEV float ab_merge(const AttnBias& p, int b, int h, int c) {
  return p.splits > 32 ? ab_merge_splits<64>(p, b, h, c) : (p.splits > 16 ? ab_merge_splits<32>(p, b, h, c) : ab_merge_splits<16>(p, b, h, c));
}

// grid (H, B, ceil(vdim / 64)), 64 threads: one 64-column slice of the head's output
__global__ void __launch_bounds__(64) attn_bias_merge_kernel(AttnBias p) {
  const int lane = threadIdx.x, h = blockIdx.x, b = blockIdx.y, c0 = blockIdx.z * 64;
  const float v = ab_merge(p, b, h, min(c0 + lane, p.vdim - 1));
  if (c0 + lane < p.vdim) ab_out(p, b, h, c0 + lane, v);
}

// grid (H, B), a wave per 64 value columns: the merged head turned by its query's position (rotate_heads: pairs i, i +
// turn_half), which as a launch of its own costs as much as the merge
__global__ void __launch_bounds__(64 * AB_MAX_VREG) attn_bias_merge_turn_kernel(AttnBias p) {
  __shared__ float row[64 * AB_MAX_VREG];
  const int c = threadIdx.x, h = blockIdx.x, b = blockIdx.y, half = p.turn_half;
  float sn = 0.f, cs = 1.f;
  if (c < 2 * half) {  // sine and cosine of position * frequency, the angle formed and reduced in 64-bit
    const double a = (double)p.turn_pos[b] * p.turn_freq[c < half ? c : c - half];
    sincosf((float)(a - 6.283185307179586476925 * rint(a * 0.159154943091895335769)), &sn, &cs);
    sn *= p.turn_sign;
  }
  const float v = ab_merge(p, b, h, min(c, p.vdim - 1));
  row[c] = v;
  __syncthreads();
  if (c >= p.vdim) return;
  const float o = c < 2 * half ? (c < half ? v * cs - row[c + half] * sn : v * cs + row[c - half] * sn) : v;
  ab_out(p, b, h, c, o * p.turn_gain);
}

// differential heads: grid (H, B), a wave per 64 value columns; both maps' splits merged, then the head's norm over all of
// its columns
__global__ void __launch_bounds__(64 * AB_MAX_VREG) attn_diff_merge_kernel(AttnBias p) {
  __shared__ float red[AB_MAX_VREG];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, h = blockIdx.x, b = blockIdx.y, waves = blockDim.x >> 6;
  const int c = min((int)threadIdx.x, p.vdim - 1);
  const float* w = p.ws + ((size_t)b * p.H + h) * 2 * p.splits * (p.vdim + 2);
  const size_t next = (size_t)p.splits * (p.vdim + 2);  // from a head's first map to its second
  float ms[2] = {-INFINITY, -INFINITY}, ls[2] = {0.f, 0.f}, wt[2], l[2], a[2] = {0.f, 0.f}, part[2][32];
#pragma unroll
  for (int map = 0; map < 2; ++map) {
    if (lane < p.splits) {
      ms[map] = w[map * next + (size_t)lane * (p.vdim + 2)];
      ls[map] = w[map * next + (size_t)lane * (p.vdim + 2) + 1];
    }
  }
  for (int s0 = 0; s0 < p.splits; s0 += 32) {  // 32 splits of both maps per round trip, the first beside the maxima
#pragma unroll
    for (int map = 0; map < 2; ++map)
#pragma unroll
      for (int sp = 0; sp < 32; ++sp)
        part[map][sp] = w[map * next + (size_t)min(s0 + sp, p.splits - 1) * (p.vdim + 2) + 2 + c];
    if (s0 == 0) {
#pragma unroll
      for (int map = 0; map < 2; ++map) {
        const float m = wave_max(ls[map] > 0.f ? ms[map] : -INFINITY);
        wt[map] = ls[map] > 0.f ? expf(ms[map] - m) : 0.f;
        l[map] = wave_sum(ls[map] * wt[map]);
      }
    }
#pragma unroll
    for (int map = 0; map < 2; ++map)
#pragma unroll
      for (int sp = 0; sp < 32; ++sp) {  // (a split without keys holds zeros and has weight 0; lanes past the splits: 0)
        const float ws = __shfl(wt[map], s0 + sp, 64);
        a[map] = fmaf(part[map][sp], ws, a[map]);
      }
  }
  const float o = a[0] / l[0] - p.diff_lambda * (a[1] / l[1]);
  const bool on = (int)threadIdx.x < p.vdim;
  float ss = wave_sum(on ? o * o : 0.f);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  ss = 0.f;
  for (int i = 0; i < waves; ++i) ss += red[i];
  const float sc = p.diff_gain / sqrtf(ss / (float)p.vdim + p.diff_eps);
  if (on) ab_out(p, b, h, c, o * sc * ab_gate(p, b, h, c));
}

// ---- MFMA flash prefill (bf16 caches) ----------------------------------------------------------------------------------
// One wave = 32 queries of one head. Keys go by in tiles of 32:
//   S^T = K Q^T on v_mfma_f32_32x32x16_bf16 with the QUERY on the lane (lane l: query l & 31; its 16 accumulators are 16
//   of the tile's keys, the other half-wave holds the other 16), so scale, soft cap, bias, mask and the online softmax
//   are lane-local plus one exchange with lane ^ 32. The key rows are fed in an order (bits 2 and 3 of the row index
//   swapped) that leaves a lane's accumulators 8c .. 8c + 7 holding keys 16c + 8 (l >> 5) + 0..7: exactly the k-slots
//   of the B operand of O^T += V^T P^T, so P is used in place. V^T comes from a transposed bf16 copy of the values
//   (attn_vt_kernel, zero past the last key), 16-byte loads along the keys.
//   The softmax weights stay 32-bit: P is split into a bf16 high part and a bf16 remainder, two MFMAs per value tile.
//   Scores of the fast path use exp-based tanh and v_exp_f32; fp32 caches: attn_f32.hip or the exact kernel above.
constexpr int AM_Q = 32, AM_K = 32;
using f32x16 = __attribute__((ext_vector_type(16))) float;

// Vt[b][g][c][j] = V[b][g][j][c] for j < n = *slot + S (0 for n <= j < round_up(n, 32)); grid (Tp / 32, vdim / 32, B * G)
__global__ void __launch_bounds__(256) attn_vt_kernel(const bf16_t* __restrict__ vc, bf16_t* __restrict__ vt,
                                                      const int32_t* slot, int S, int T, int Tp, int vdim) {
  __shared__ bf16_t tile[32][34];
  const int n = min(*slot + S, T);
  const int j0 = blockIdx.x * 32, c0 = blockIdx.y * 32;
  if (j0 >= n) return;
  const size_t bg = blockIdx.z;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  for (int r = ty; r < 32; r += 8) {
    const int j = j0 + r;
    tile[r][tx] = j < n ? vc[(bg * T + j) * vdim + c0 + tx] : (bf16_t)0;
  }
  __syncthreads();
  for (int r = ty; r < 32; r += 8) vt[(bg * vdim + c0 + r) * Tp + j0 + tx] = tile[tx][r];
}

JLA_DEV float am_tanh(float x) {  // 1 - 2 / (e^(2x) + 1), saturating cleanly for large |x|
  const float e = __expf(2.f * x);
  return 1.f - 2.f * __builtin_amdgcn_rcpf(e + 1.f);
}

// What a wave keeps of its 32 queries
template <int DK, int VT>
struct AmRow {
  bf16x8_t q[DK];  // the B operand: query lane & 31, k-slots 16 kk + 8 (lane >> 5) + e
  f32x16 o[VT];
  float m, l;      // (l: this half-wave's part of the sum)
  int q0, qi, lo_q, lo_last, kfirst, vh, heads;
  float scale, inv_cap;
};

// The tile of 32 keys from slot j0 on. keys(kk), values(c, v): operand fragments; behind(): what is issued behind the scores' products.
template <int DK, int VT, class Keys, class Values, class Behind>
JLA_DEV void am_tile(const AttnBias& p, AmRow<DK, VT>& w, int j0, Keys keys, Values values, Behind behind) {
  const int lane = threadIdx.x & 63, ql = lane & 31, hi = lane >> 5;
  // scores: rows = keys (fed permuted), columns = queries
  f32x16 sacc;
#pragma unroll
  for (int r = 0; r < 16; ++r) sacc[r] = 0.f;
#pragma unroll
  for (int kk = 0; kk < DK; ++kk)
    sacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, keys(kk)), w.q[kk], sacc, 0, 0, 0);
  // bias of this tile's 63 distances, one per lane: lane t holds distance q0 - j0 - 31 + t
  float bl = 0.f;
  const int dbase = w.q0 - j0 - (AM_K - 1);
  if (p.bias) bl = p.bias[(size_t)min(max(dbase + lane, 0), p.nbias - 1) * w.heads + w.vh];
  behind();
  // key of accumulator r within the tile: 16 (r >> 3) + 8 hi + (r & 7)
#pragma unroll
  for (int r = 0; r < 16; ++r) sacc[r] *= w.scale;
  if (p.softcap > 0.f) {
#pragma unroll
    for (int r = 0; r < 16; ++r) sacc[r] = p.softcap * am_tanh(sacc[r] * w.inv_cap);
  }
  if (p.bias) {
    if (dbase >= p.nbias - 1) {
#pragma unroll
      for (int r = 0; r < 16; ++r) sacc[r] += bl;
    } else {
      float bk[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) bk[r] = __shfl(bl, ql - (16 * (r >> 3) + 8 * hi + (r & 7)) + (AM_K - 1), 64);
#pragma unroll
      for (int r = 0; r < 16; ++r) sacc[r] += bk[r];
    }
  }
  // some (query, key) of the tile is masked
  if (j0 + AM_K - 1 > w.q0 || (j0 < w.lo_last && j0 + AM_K - 1 >= w.kfirst)) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int j = j0 + 16 * (r >> 3) + 8 * hi + (r & 7);
      sacc[r] = j > w.qi || (j < w.lo_q && j >= w.kfirst) ? -INFINITY : sacc[r];
    }
  }
  float tmax = sacc[0];
#pragma unroll
  for (int r = 1; r < 16; ++r) tmax = fmaxf(tmax, sacc[r]);
  tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
  const float m_new = fmaxf(w.m, tmax);
  // (a query without a sink may have no visible key in a tile it shares with its neighbours' earlier blocks)
  const float m_use = m_new == -INFINITY ? 0.f : m_new;
  const float corr = __expf(w.m - m_use);
  w.m = m_new;
  float psum = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    sacc[r] = __expf(sacc[r] - m_use);
    psum += sacc[r];
  }
  w.l = w.l * corr + psum;    // (the halves are added at the end)
  if (__any(corr != 1.f)) {  // (wave-uniform)
#pragma unroll
    for (int v = 0; v < VT; ++v)
#pragma unroll
      for (int r = 0; r < 16; ++r) w.o[v][r] *= corr;
  }
  // O^T += V^T P^T, P = high bf16 part + bf16 remainder
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    float ph[8], pl[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      ph[e] = bf2f(f2bf(sacc[8 * c + e]));
      pl[e] = sacc[8 * c + e] - ph[e];
    }
    const bf16x8_t bh = __builtin_bit_cast(bf16x8_t, pack8(ph)), bo = __builtin_bit_cast(bf16x8_t, pack8(pl));
#pragma unroll
    for (int v = 0; v < VT; ++v) {
      const bf16x8_t vv = __builtin_bit_cast(bf16x8_t, values(c, v));
      w.o[v] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vv, bh, w.o[v], 0, 0, 0);
      w.o[v] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vv, bo, w.o[v], 0, 0, 0);
    }
  }
}

// a lane's columns of its query's output, times inv and the gates per column
template <int VT>
JLA_DEV void am_store(const AttnBias& p, const f32x16 (&o)[VT], size_t m, int h, int hi, float inv) {
  const size_t at = m * p.ldo + (size_t)h * (32 * VT);
  const float* gt = p.gate && p.gate_cols ? p.gate + m * p.ldg + (size_t)h * (32 * VT) : nullptr;
#pragma unroll
  for (int v = 0; v < VT; ++v)
#pragma unroll
    for (int r = 0; r < 16; r += 4) {  // rows (value columns) (r & 3) + 8 (r >> 2) + 4 hi: runs of four
      const int c = 32 * v + 8 * (r >> 2) + 4 * hi;
      float f[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) f[k] = o[v][r + k] * inv * (gt ? hy_sigmoid(gt[c + k]) : 1.f);
      if (p.out_bf16)
        *reinterpret_cast<uint2*>(reinterpret_cast<bf16_t*>(p.out) + at + c) = uint2{pack2bf(f[0], f[1]), pack2bf(f[2], f[3])};
      else
        *reinterpret_cast<float4*>(reinterpret_cast<float*>(p.out) + at + c) = float4{f[0], f[1], f[2], f[3]};
    }
}

// head and block of query tiles of this workgroup (nq blocks per head). Workgroups go round the 8 XCDs by their id: where the heads
// divide evenly, each XCD gets whole runs of neighbouring heads (which share their keys in grouped-query attention), so that a
// head's keys and values pass through one L2. Long rows come first.
JLA_DEV void am_place(const AttnBias& p, int nq, int& hb, int& blk) {
  const int heads = p.H * p.B;
  if (heads % 8 == 0) {
    const int r = blockIdx.x >> 3, hl = r / nq;
    hb = (int)(blockIdx.x & 7) * (heads >> 3) + hl;
    blk = nq - 1 - (r - hl * nq);
  } else {
    hb = blockIdx.x / nq;
    blk = nq - 1 - (blockIdx.x - hb * nq);
  }
}

// the row of query tile s0 before its first key
template <int DK, int VT>
JLA_DEV void am_start(const AttnBias& p, AmRow<DK, VT>& w, int b, int vh, int maps, int s0, int slot, bool sunk) {
  const int lane = threadIdx.x & 63, ql = lane & 31, hi = lane >> 5;
  const int sq = min(s0 + ql, p.S - 1);  // (surplus lanes repeat the last query; never stored)
  const float* q = p.q + (((size_t)b * p.S + sq) * (p.H * maps) + vh) * (16 * DK) + 8 * hi;
#pragma unroll
  for (int kk = 0; kk < DK; ++kk) {
    float f[8];
    hy_load8(q + 16 * kk, 8, f);
    w.q[kk] = __builtin_bit_cast(bf16x8_t, pack8(f));
  }
#pragma unroll
  for (int v = 0; v < VT; ++v)
#pragma unroll
    for (int r = 0; r < 16; ++r) w.o[v][r] = 0.f;
  w.m = sunk ? p.sink[vh] : -INFINITY;
  w.l = sunk && hi == 0 ? 1.f : 0.f;  // (the sink counts once, in the lower half)
  w.q0 = slot + s0;
  w.qi = slot + sq;
  w.vh = vh;
  w.heads = p.H * maps;
  w.scale = p.scale * (p.head_scale ? p.head_scale[vh] : 1.f);
  w.inv_cap = p.softcap > 0.f ? 1.f / p.softcap : 0.f;
  w.lo_q = ab_span(p, w.qi).lo;
  w.lo_last = ab_span(p, min(w.q0 + AM_Q - 1, slot + p.S - 1)).lo;  // (the largest of the wave)
  w.kfirst = p.window > 0 ? p.keep_first : 0;
}

// MAPS = 2 (differential heads): waves 2 t and 2 t + 1 of a workgroup run the two maps of query tile t; the second hands its
// normalised output to the first through LDS, which subtracts, norms and stores.
// KS = 4 (few queries): the four waves of a workgroup take one query tile and every fourth key tile each, joined through LDS; KS = 1: a
// query tile per wave.
// What bounds it: the vector unit, about 2.5 k cycles per tile of 32 x 32 (scores, their exponentials, the split weights) beside 24
// matrix instructions, and the operand loads (below). So the tile has no branch and no wait per score: the options are taken for all
// 16 at once, the accumulators are rescaled only where a maximum grew, and a tile's values are loaded behind its scores' products, the
// next one's keys behind its softmax. Us before -> after, 16 heads of 128: 300 tokens, soft cap and bias, 38.8 -> 16.0; 777 tokens in
// blocks of 1024 54.5 -> 27.9; 64 tokens behind 900 62 -> 21.
template <int DK, int VT, int MAPS, int KS>  // dim = 16 DK, vdim = 32 VT
__global__ void __launch_bounds__(256, DK <= 8 ? 2 : 1) attn_bias_mma_kernel(AttnBias p, const bf16_t* __restrict__ vt, int Tp) {
  static_assert(MAPS == 1 || KS == 1, "differential heads: a map per wave");
  constexpr int TILES = 4 / (MAPS * KS);  // query tiles per workgroup
  constexpr int dim = 16 * DK, vdim = 32 * VT, PITCH = vdim + 4;
  __shared__ float joined[MAPS == 2 ? TILES * VT * 16 * 64 : (KS > 1 ? KS * AM_Q * PITCH : 1)];
  __shared__ float jm[KS > 1 ? KS : 1][AM_Q], jl[KS > 1 ? KS : 1][AM_Q];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int map = wave % MAPS;
  const int ql = lane & 31, hi = lane >> 5;
  const int nq = (p.S + TILES * AM_Q - 1) / (TILES * AM_Q);
  int hb, blk;
  am_place(p, nq, hb, blk);
  const int s0 = (blk * TILES + (KS > 1 ? 0 : wave / MAPS)) * AM_Q;
  const bool live = s0 < p.S;
  if (MAPS == 1 && KS == 1 && !live) return;  // (a pair of waves without queries stays for the workgroup's barrier)
  const int b = hb / p.H, h = hb - b * p.H;
  const int g = h / (p.H / p.G), slot = *p.slot;
  AmRow<DK, VT> w;
  am_start<DK, VT>(p, w, b, h * MAPS + map, MAPS, s0, slot, p.sink && (KS == 1 || wave == 0));
  const bf16_t* kbase = reinterpret_cast<const bf16_t*>(p.kc) + ((size_t)b * p.G + g) * p.T * p.ldk + map * dim + 8 * hi;
  const bf16_t* vbase = vt + (((size_t)b * p.G + g) * vdim + ql) * Tp + 8 * hi;
  const int krow = (ql & 0x13) | ((ql & 4) << 1) | ((ql & 8) >> 1);  // bits 2 and 3 swapped
  const int q_last = live ? min(w.q0 + AM_Q - 1, slot + p.S - 1) : -1;
  const int j_begin = ab_span(p, w.q0).lo / AM_K * AM_K;  // the tile that the walk starts at
  // kept first keys (beside a window): their tiles come first, then the walk jumps to the window's tiles
  const int kf_tiles = min((w.kfirst + AM_K - 1) / AM_K, j_begin / AM_K);
  const int tiles = live ? kf_tiles + (q_last - j_begin) / AM_K + 1 : 0;  // (no tile is walked without queries)
  auto tile_key = [&](int t) { return t < kf_tiles ? t * AM_K : j_begin + (t - kf_tiles) * AM_K; };
  u32x4 kf[DK], vf[2][VT];
  auto fetch_keys = [&](int t) {  // (past the last tile: it again, unused)
    const bf16_t* kr = kbase + (size_t)min(tile_key(min(t, max(tiles, 1) - 1)) + krow, p.T - 1) * p.ldk;
#pragma unroll
    for (int kk = 0; kk < DK; ++kk) kf[kk] = *reinterpret_cast<const u32x4*>(kr + 16 * kk);
  };
  const int t_first = KS > 1 ? wave : 0;
  fetch_keys(t_first);
  for (int t = t_first; t < tiles; t += KS) {
    const int j0 = tile_key(t);
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int v = 0; v < VT; ++v)
        vf[c][v] = *reinterpret_cast<const u32x4*>(vbase + (size_t)(32 * v) * Tp + min(j0, Tp - AM_K) + 16 * c);
    am_tile<DK, VT>(p, w, j0, [&](int kk) { return kf[kk]; }, [&](int c, int v) { return vf[c][v]; }, [&]() { fetch_keys(t + KS); });
  }
  float l_run = w.l;
  const float m_run = w.m;
  auto& o = w.o;
  l_run += __shfl_xor(l_run, 32, 64);
  if constexpr (KS > 1) {  // the waves' parts of the row; then 8 threads per query, 16 columns' worth of steps each
    if (hi == 0) jm[wave][ql] = m_run;
    __syncthreads();
    float m_all = jm[0][ql];
#pragma unroll
    for (int w = 1; w < KS; ++w) m_all = fmaxf(m_all, jm[w][ql]);
    const float wt = m_run == -INFINITY ? 0.f : __expf(m_run - m_all);  // (a wave without keys of this query: zeros)
    if (hi == 0) jl[wave][ql] = l_run * wt;
    float* mine = joined + ((size_t)wave * AM_Q + ql) * PITCH + 4 * hi;
#pragma unroll
    for (int v = 0; v < VT; ++v)
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        *reinterpret_cast<float4*>(mine + 32 * v + 2 * r) =
            float4{o[v][r] * wt, o[v][r + 1] * wt, o[v][r + 2] * wt, o[v][r + 3] * wt};
    __syncthreads();
    const int qt = threadIdx.x >> 3;
    if (s0 + qt >= p.S) return;
    float l = 0.f;
#pragma unroll
    for (int w = 0; w < KS; ++w) l += jl[w][qt];
    const size_t m = (size_t)b * p.S + s0 + qt, at = m * p.ldo + (size_t)h * vdim;
    float inv = 1.f / l;
    if (p.gate && !p.gate_cols) inv *= ab_gate(p, m, h, 0);
#pragma unroll
    for (int c = 4 * (threadIdx.x & 7); c < vdim; c += 32) {
      float f[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < KS; ++w) {
        const float4 x = *reinterpret_cast<const float4*>(joined + ((size_t)w * AM_Q + qt) * PITCH + c);
        f[0] += x.x; f[1] += x.y; f[2] += x.z; f[3] += x.w;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) f[k] *= inv * (p.gate && p.gate_cols ? ab_gate(p, m, h, c + k) : 1.f);
      if (p.out_bf16)
        *reinterpret_cast<uint2*>(reinterpret_cast<bf16_t*>(p.out) + at + c) = uint2{pack2bf(f[0], f[1]), pack2bf(f[2], f[3])};
      else
        *reinterpret_cast<float4*>(reinterpret_cast<float*>(p.out) + at + c) = float4{f[0], f[1], f[2], f[3]};
    }
    return;
  }
  const size_t m = (size_t)b * p.S + s0 + ql;
  float inv = 1.f / l_run;
  if constexpr (MAPS == 2) {
    float* mine = joined + (wave / MAPS) * VT * 16 * 64 + lane;
    if (map == 1) {
#pragma unroll
      for (int v = 0; v < VT; ++v)
#pragma unroll
        for (int r = 0; r < 16; ++r) mine[(v * 16 + r) * 64] = o[v][r] * inv;
    }
    __syncthreads();
    if (map == 1) return;
    float ss = 0.f;  // (a query's columns: this lane's and those of lane ^ 32)
#pragma unroll
    for (int v = 0; v < VT; ++v)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        o[v][r] = o[v][r] * inv - p.diff_lambda * mine[(v * 16 + r) * 64];
        ss = fmaf(o[v][r], o[v][r], ss);
      }
    ss += __shfl_xor(ss, 32, 64);
    inv = p.diff_gain / sqrtf(ss / (float)vdim + p.diff_eps);
  }
  if (s0 + ql >= p.S) return;
  if (p.gate && !p.gate_cols) inv *= ab_gate(p, m, h, 0);
  am_store<VT>(p, o, m, h, hi, inv);
}

// Key widths of 64 and 128, more queries than one tile per head: four waves with neighbouring query tiles of a head share its key tiles, 64 keys at a time, staged by LDS-DMA into one
// of two buffers while the other is used. Straight from the caches (the kernel above) a wave's operand load touches 32 lines for 32
// bytes each, which is what bounds it once every SIMD has waves: 512 line accesses per tile and wave; staged, a line is fetched once
// per workgroup. Images: key rows of 16 DK numbers, chunk c (16 bytes) of row r at c ^ swizzle(r), value rows (64 keys) likewise.
constexpr int AL_KEYS = 64;
template <int DK, int VT, int KS>
__global__ void __launch_bounds__(256 * KS, 2) attn_bias_lds_kernel(AttnBias p, const bf16_t* __restrict__ vt, int Tp) {
  static_assert(DK == 4 || DK == 8, "power-of-two key rows");
  constexpr int dim = 16 * DK, vdim = 32 * VT;
  constexpr int KC = 2 * DK, KU = AL_KEYS * KC, VU = vdim * 8, STAGE = KU + VU;  // 16-byte chunks: of a key row, of the images
  constexpr int PARTS = KS == 2 ? 4 * VT * 16 * 64 / 4 : 0;  // (16-byte units)
  __shared__ u32x4 lds[2 * STAGE > PARTS ? 2 * STAGE : PARTS];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ql = lane & 31, hi = lane >> 5;
  const int nq = (p.S + 4 * AM_Q - 1) / (4 * AM_Q);
  int hb, blk;
  am_place(p, nq, hb, blk);
  const int s_first = blk * 4 * AM_Q, s0 = s_first + (wave & 3) * AM_Q;
  const int b = hb / p.H, h = hb - b * p.H;
  const int g = h / (p.H / p.G), slot = *p.slot;
  AmRow<DK, VT> w;
  am_start<DK, VT>(p, w, b, h, 1, min(s0, p.S - 1), slot, p.sink && wave < 4);  // (a wave without queries walks along)
  const bf16_t* kbase = reinterpret_cast<const bf16_t*>(p.kc) + ((size_t)b * p.G + g) * p.T * p.ldk;
  const bf16_t* vbase = vt + ((size_t)b * p.G + g) * vdim * Tp;
  const int q_last = min(w.q0 + AM_Q - 1, slot + p.S - 1), q_end = min(slot + s_first + 4 * AM_Q, slot + p.S) - 1;
  const int lo_own = ab_span(p, w.q0).lo;
  const int j_begin = ab_span(p, slot + s_first).lo / AL_KEYS * AL_KEYS;
  const int kf_steps = min((w.kfirst + AL_KEYS - 1) / AL_KEYS, j_begin / AL_KEYS);
  const int steps = kf_steps + (q_end - j_begin) / AL_KEYS + 1;
  auto step_key = [&](int t) { return t < kf_steps ? t * AL_KEYS : j_begin + (t - kf_steps) * AL_KEYS; };
  // chunk position of chunk c in row r: the 16 rows of a fragment's half fall on all banks
  auto kpos = [](int r, int c) { return DK == 8 ? c ^ (r & 15) : c ^ ((r >> 1) & 7); };
  auto vpos = [](int r, int c) { return c ^ ((r >> 1) & 7); };
  auto stage = [&](int t) {
    const int j0 = step_key(t);
    u32x4* const buf = lds + (t & 1) * STAGE;
#pragma unroll
    for (int i = 0; i < KU / (256 * KS); ++i) {
      const int first = 64 * (4 * KS * i + wave), at = first + lane, r = at / KC, c = kpos(r, at % KC);  // (the swizzle is its own inverse)
      glds16_asm(kbase + (size_t)min(j0 + r, p.T - 1) * p.ldk + 8 * c, buf + first);
    }
#pragma unroll
    for (int i = 0; i < VU / (256 * KS); ++i) {
      const int first = 64 * (4 * KS * i + wave), at = first + lane, r = at / 8, c = vpos(r, at % 8);
      glds16_asm(vbase + (size_t)r * Tp + min(j0 + 8 * c, Tp - 8), buf + KU + first);
    }
  };
  const int krow = (ql & 0x13) | ((ql & 4) << 1) | ((ql & 8) >> 1);  // bits 2 and 3 swapped
  stage(0);
  for (int t = 0; t < steps; ++t) {
    wait_vmcnt<0>();  // this wave's part of step t has landed; then every wave's has, and step t - 1 is read
    __syncthreads();
    if (t + 1 < steps) stage(t + 1);
    const u32x4* const buf = lds + (t & 1) * STAGE;
#pragma unroll 1
    for (int half = KS == 2 ? wave >> 2 : 0; half < (KS == 2 ? (wave >> 2) + 1 : 2); ++half) {
      const int j0 = step_key(t) + AM_K * half;
      if (s0 >= p.S || j0 > q_last || (j0 + AM_K <= lo_own && j0 >= w.kfirst)) continue;  // (wave-uniform: nothing to see)
      const int kr = AM_K * half + krow;
      am_tile<DK, VT>(
          p, w, j0, [&](int kk) { return buf[kr * KC + kpos(kr, 2 * kk + hi)]; },
          [&](int c, int v) { return buf[KU + (32 * v + ql) * 8 + vpos(32 * v + ql, 4 * half + 2 * c + hi)]; }, []() {});
    }
  }
  float l = w.l + __shfl_xor(w.l, 32, 64);
  if constexpr (KS == 2) {  // the waves of the second halves hand their part over, through the images' memory
    __shared__ float jm[4][AM_Q], jl[4][AM_Q];
    float* const part = reinterpret_cast<float*>(lds) + (size_t)(wave & 3) * VT * 16 * 64 + lane;
    __syncthreads();
    if (wave >= 4) {
      if (hi == 0) jm[wave & 3][ql] = w.m, jl[wave & 3][ql] = l;
#pragma unroll
      for (int v = 0; v < VT; ++v)
#pragma unroll
        for (int r = 0; r < 16; ++r) part[(v * 16 + r) * 64] = w.o[v][r];
    }
    __syncthreads();
    if (wave >= 4) return;
    const float m2 = jm[wave][ql], m_all = fmaxf(w.m, m2);
    const float w1 = w.m == -INFINITY ? 0.f : __expf(w.m - m_all), w2 = m2 == -INFINITY ? 0.f : __expf(m2 - m_all);
    l = l * w1 + jl[wave][ql] * w2;
#pragma unroll
    for (int v = 0; v < VT; ++v)
#pragma unroll
      for (int r = 0; r < 16; ++r) w.o[v][r] = w.o[v][r] * w1 + part[(v * 16 + r) * 64] * w2;
  }
  if (s0 + ql >= p.S) return;
  const size_t m = (size_t)b * p.S + s0 + ql;
  float inv = 1.f / l;
  if (p.gate && !p.gate_cols) inv *= ab_gate(p, m, h, 0);
  am_store<VT>(p, w.o, m, h, hi, inv);
}

// Query tiles up to which they share the chip by their keys: four ways (measured us, four ways / two ways / one: 400 tiles 28 / 33 / 37,
// 768 tiles 38 / 29 / 30, 1024 tiles 105 / 91 / 119), then two ways (2048 tiles 115 / 95 / 92, 4096 tiles 254 / 165 / 165,
// 6032 tiles 305 / 238 / 203). Heads of 64 x 64 have half the bytes to stage and gain nothing from two ways: rows x heads x queries
// behind 0 | 400 | 1500 keys, 9 x 32 x 64 13 | 26 | 59 four ways, 16 | 43 | 105 two ways, 9 x 32 x 128 (1152 tiles) 21 | 39 | 88, 24 | 52 | 115
// and one way 19 | 48 | 116; the kernel before these 14 | 53 | 156 and 23 | 64 | 166; keys of a single staged step one way (9 x 32 x 64 behind
// none 12, four ways 13). Key widths that are not staged (measured on heads of
// 128 without the staging, four ways / one): 105 / 135 at 1024 tiles, 254 / 236 at 4096.
constexpr long long AM_SPLIT4 = 512, AM_SPLIT2 = 1536, AM_SPLIT4_NARROW = 1024, AM_SPLIT4_DIRECT = 1024;
// A head of one query tile has nobody to share staged keys with, three of four waves would walk along: over few keys a wave takes its
// tile directly, over many, or as many as the host does not know, four waves share it by its keys. Us, directly | four ways | two ways (one
// way from 2048 tiles on) | before, soft cap and bias, 2 queries behind 0 | 60 | 400 | 1500 keys: 18 x 32 heads of 128 12, 14, 39, 120 | 15, 17,
// 38, 109 | 27, 29, 71, 193 | 26, 35, 130, 439; 64 x 32 25, 33, 98, 458 | 32, 38, 91, 425 | 38, 46, 135, 507 | 69, 93, 347, 1355; 30 x 32
// heads of 64 10, 13, 37, 107 | 12, 14, 32, 84 | 22, 24, 69, 196 | 12, 16, 53, 167; 9 x 32 heads of 64, 32 queries 9, 11 | 11, 12 | - | 10, 16;
// 20 x 32 of 80 x 64, 32 queries behind none 12 | 14 | - | 12.
constexpr long long AM_ALONE = 256;
constexpr int AM_ALONE_KEYS = 256;

template <int DK, int VT>
static int am_launch(const AttnBias& p, bf16_t* vt, int Tp, hipStream_t s) {
  attn_vt_kernel<<<dim3(Tp / 32, p.vdim / 32, p.B * p.G), 256, 0, s>>>(reinterpret_cast<const bf16_t*>(p.vc), vt, p.slot,
                                                                     p.S, p.T, Tp, p.vdim);
  JLA_CHECK_LAUNCH();
  const long long hb = (long long)p.H * p.B;
  const long long tiles = (p.S + AM_Q - 1) / AM_Q * hb;
  constexpr bool staged = DK == 4 || DK == 8, narrow = DK == 4 && VT == 2;
  const unsigned g4 = (unsigned)((p.S + 4 * AM_Q - 1) / (4 * AM_Q) * hb);
  if (p.maps == 2) attn_bias_mma_kernel<DK, VT, 2, 1><<<(unsigned)((p.S + 63) / 64 * hb), 256, 0, s>>>(p, vt, Tp);
  else if (p.S <= AM_Q && tiles > AM_ALONE && p.t_cap <= AM_ALONE_KEYS)
    attn_bias_mma_kernel<DK, VT, 1, 1><<<g4, 256, 0, s>>>(p, vt, Tp);
  else if (tiles <= (narrow && p.t_cap > AL_KEYS ? AM_SPLIT4_NARROW : (staged ? AM_SPLIT4 : AM_SPLIT4_DIRECT)) || (staged && p.S <= AM_Q))
    attn_bias_mma_kernel<DK, VT, 1, 4><<<(unsigned)tiles, 256, 0, s>>>(p, vt, Tp);
  else if constexpr (!staged) attn_bias_mma_kernel<DK, VT, 1, 1><<<g4, 256, 0, s>>>(p, vt, Tp);
  else if (!narrow && tiles <= AM_SPLIT2) attn_bias_lds_kernel<DK, VT, 2><<<g4, 512, 0, s>>>(p, vt, Tp);
  else attn_bias_lds_kernel<DK, VT, 1><<<g4, 256, 0, s>>>(p, vt, Tp);
  JLA_CHECK_LAUNCH();
  return 0;
}

// key widths the flash kernel is instantiated for (beside 64 and 128: plain numbers plus a rotated part of 16 .. 64)
static bool am_key_width(int dim) {
  return dim == 64 || dim == 80 || dim == 96 || dim == 128 || dim == 160 || dim == 192;
}

// bytes of the transposed-value workspace the MFMA prefill needs, 0 when the shape goes to the plain kernel
long long hy_attn_prefill_ws_bytes(int B, int S, int G, int dim, int vdim, int T, int cbf16) {
  if (!cbf16 || S < 2) return 0;
  if (!am_key_width(dim) || !(vdim == 64 || vdim == 128)) return 0;
  if ((long long)B * G > 65535) return 0;
  return (long long)B * G * vdim * ((T + 31) / 32 * 32) * 2;
}

int hy_attn_decode_splits(int B, int H, int t_cap) {
  // enough waves for the chip (256 CUs x 4 SIMDs x 2), at least one 64-key step per split
  const long long pairs = (long long)B * H;
  long long want = (2048 + pairs - 1) / (pairs > 0 ? pairs : 1);
  const long long by_len = (t_cap + 63) / 64;
  if (want > by_len) want = by_len;
  if (want < 1) want = 1;
  if (want > 64) want = 64;
  return (int)want;
}

// launch KERNEL<cache type, value registers per lane> for p.vdim
#define AB_BY_VREG(KERNEL, GRID, THREADS)                                              \
  do {                                                                                 \
    const int vr = (p.vdim + 63) / 64;                                                 \
    if (p.cbf16) {                                                                     \
      if (vr <= 1) KERNEL<bf16_t, 1><<<GRID, THREADS, 0, s>>>(p);                      \
      else if (vr <= 2) KERNEL<bf16_t, 2><<<GRID, THREADS, 0, s>>>(p);                 \
      else if (vr <= 4) KERNEL<bf16_t, 4><<<GRID, THREADS, 0, s>>>(p);                 \
      else KERNEL<bf16_t, 8><<<GRID, THREADS, 0, s>>>(p);                              \
    } else {                                                                           \
      if (vr <= 1) KERNEL<float, 1><<<GRID, THREADS, 0, s>>>(p);                       \
      else if (vr <= 2) KERNEL<float, 2><<<GRID, THREADS, 0, s>>>(p);                  \
      else if (vr <= 4) KERNEL<float, 4><<<GRID, THREADS, 0, s>>>(p);                  \
      else KERNEL<float, 8><<<GRID, THREADS, 0, s>>>(p);                               \
    }                                                                                  \
  } while (0)

int hy_attn_bias(const AttnBias& p, hipStream_t s) {
  if (p.B < 0 || p.S < 1 || p.H < 1 || p.G < 1 || p.H % p.G || p.T < 1) return -1;
  if (p.dim < 1 || p.dim > AB_MAX_DIM || p.vdim < 1 || p.vdim > 64 * AB_MAX_VREG) return -2;
  if (p.bias && p.nbias < 1) return -3;
  if (p.chunk < 0 || p.window < 0 || p.keep_first < 0 || (p.chunk > 0 && p.window > 0)) return -7;
  if (p.maps != 1 && p.maps != 2) return -10;
  if (p.ldk < p.maps * p.dim) return -8;
  if (p.ldv < p.vdim || (p.gate && p.ldg < (p.gate_cols ? p.H * p.vdim : p.H)) || p.ldo < p.H * p.vdim) return -8;
  if (p.turn_pos && (p.S != 1 || p.maps != 1 || p.turn_half < 0 || 2 * p.turn_half > p.vdim || (p.turn_half && !p.turn_freq))) return -11;
  if (p.B == 0) return 0;
  if ((long long)p.H * p.maps > 65535 || p.B > 65535) return -4;
  if (p.S == 1) {
    if (p.splits < 1 || !p.ws) return -5;
    if (p.splits > 64) return -6;  // (the merge holds one split per lane)
    dim3 grid(p.splits, p.H * p.maps, p.B);
    if (p.cbf16 && (p.dim == 64 || p.dim == 128) && (p.vdim == 64 || p.vdim == 128) && p.ldv == p.vdim && p.ldk % 8 == 0 &&
        (((uintptr_t)p.kc | (uintptr_t)p.vc) & 15) == 0) {
      if (p.dim == 64 && p.vdim == 64) attn_bias_decode_fast_kernel<8, 1><<<grid, 64, 0, s>>>(p);
      else if (p.dim == 64) attn_bias_decode_fast_kernel<8, 2><<<grid, 64, 0, s>>>(p);
      else if (p.vdim == 64) attn_bias_decode_fast_kernel<16, 1><<<grid, 64, 0, s>>>(p);
      else attn_bias_decode_fast_kernel<16, 2><<<grid, 64, 0, s>>>(p);
    } else if (p.cbf16 && p.maps == 1 && p.kc == p.vc && p.G == 1 && p.ldk == p.dim && p.ldv == p.dim && p.vdim <= p.dim && p.vdim % 8 == 0 &&
               p.dim % 8 == 0 && p.dim > 128 && p.dim <= 512 && !p.bias && p.softcap <= 0.f &&
               ((uintptr_t)p.kc & 15) == 0) {
      attn_latent_decode_kernel<1, AL_KC><<<grid, 64, 0, s>>>(p);
    } else {
      AB_BY_VREG(attn_bias_decode_kernel, grid, 64);
    }
    JLA_CHECK_LAUNCH();
    if (p.maps == 2) attn_diff_merge_kernel<<<dim3(p.H, p.B), (p.vdim + 63) / 64 * 64, 0, s>>>(p);
    else if (p.turn_pos) attn_bias_merge_turn_kernel<<<dim3(p.H, p.B), (p.vdim + 63) / 64 * 64, 0, s>>>(p);
    else attn_bias_merge_kernel<<<dim3(p.H, p.B, (p.vdim + 63) / 64), 64, 0, s>>>(p);
    JLA_CHECK_LAUNCH();
    return 0;
  }
  // (the flash kernel stores four columns at a time)
  if (p.vt_ws && (p.S + 63) / 64 * (long long)p.H * p.B <= 0x7fffffffLL && p.ldv == p.vdim && p.ldk % 8 == 0 && p.ldo % 4 == 0 && ((uintptr_t)p.out & (p.out_bf16 ? 7 : 15)) == 0 &&
      hy_attn_prefill_ws_bytes(p.B, p.S, p.G, p.dim, p.vdim, p.T, p.cbf16) > 0) {
    const int Tp = (p.T + 31) / 32 * 32;
    bf16_t* vt = reinterpret_cast<bf16_t*>(p.vt_ws);
#define AM_CASE(DK)                                               \
  case 16 * DK:                                                   \
    return p.vdim == 64 ? am_launch<DK, 2>(p, vt, Tp, s) : am_launch<DK, 4>(p, vt, Tp, s)
    switch (p.dim) {
      AM_CASE(4);
      AM_CASE(5);
      AM_CASE(6);
      AM_CASE(8);
      AM_CASE(10);
      AM_CASE(12);
    }
#undef AM_CASE
    return -9;
  }
  if (hy_attn_f32_takes(p)) return hy_attn_f32(p, s);
  dim3 grid((p.S + 3) / 4, p.H, p.B);
  if (p.maps == 2) AB_BY_VREG(attn_diff_prefill_kernel, grid, 256);
  else AB_BY_VREG(attn_bias_prefill_kernel, grid, 256);
  JLA_CHECK_LAUNCH();
  return 0;
}

}  // namespace jla
