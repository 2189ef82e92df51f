// One decode token of an attention layer in one launch, from the fused q | k | v projection to the head's output: the per-head
// preparation (hy_attn_prep's norms or hy_rope_prep's biases and rotations), the cache write, attention over the cache
// (attn_bias.hip) and the merge of the key splits, which as launches of their own cost 3 to 4 us each on either side of an
// attention of 7.
//
// grid (workgroups of WAVES splits, H, B), a wave per split. Every split prepares its head's query itself, behind its own key and value loads. The
// token's key and value are in no cache yet: the last split of every head prepares them too (rounded as the cache holds them),
// takes them as one more key behind its own, and the first head of a key head writes them; the other splits deal the keys before
// them, so nothing is read that this launch writes. A workgroup publishes its maximum, sum and values past the caches and takes its
// head's ticket; the last one to arrive (nobody waits) merges them in split order and sets the ticket back.
// What bounds it: two trips to memory (slot, then keys and values), the publication and the merge's trip. Tickets lie on lines of their own: counts on one line go one behind
// the other (16 heads x 33 splits on two lines: 4 us).
#include "attn_chunk.h"
#include "attn_span.h"

namespace jla {

JLA_DEV void as_put(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// a number as a cache of that type holds it
JLA_DEV void as_held(bf16_t& d, float v) { d = f2bf(v); }
JLA_DEV void as_held(float& d, float v) { d = v; }
JLA_DEV float as_number(bf16_t v) { return bf2f(v); }
JLA_DEV float as_number(float v) { return v; }
JLA_DEV float as_get(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// LDS that only this wave uses: its accesses stay in program order
JLA_DEV void as_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
// the columns VREG lane + i of a published split
template <int VREG>
JLA_DEV void as_put_row(float* w, const float (&x)[VREG]) {
  if constexpr (VREG == 2) {
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(w), (unsigned long long)__float_as_uint(x[1]) << 32 | __float_as_uint(x[0]),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
    as_put(w, x[0]);
  }
}
template <int VREG>
JLA_DEV void as_get_row(const float* w, float (&x)[VREG]) {
  if constexpr (VREG == 2) {
    const unsigned long long v = __hip_atomic_load(reinterpret_cast<const unsigned long long*>(w), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    x[0] = __uint_as_float((uint32_t)v);
    x[1] = __uint_as_float((uint32_t)(v >> 32));
  } else {
    x[0] = as_get(w);
  }
}

// N numbers of a head's row, lane + 64 i: turned by the angles of the table (pairs i, i + half)
template <int N>
JLA_DEV void as_turn(float (&x)[N], float* row, int half, const float* cs, const float* sn, int lane) {
  as_order();
#pragma unroll
  for (int i = 0; i < N; ++i) row[lane + 64 * i] = x[i];
  as_order();
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int d = lane + 64 * i;
    if (d < 2 * half) {
      const int f = d < half ? d : d - half;
      const float o = row[d < half ? d + half : f];
      x[i] = d < half ? x[i] * cs[f] - o * sn[f] : x[i] * cs[f] + o * sn[f];
    }
  }
}

// 1 / root mean square of the head's numbers
template <int N>
JLA_DEV float as_norm(const float (&x)[N], float eps) {
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) ss = fmaf(x[i], x[i], ss);
  return 1.f / sqrtf(wave_sum(ss) / (float)(64 * N) + eps);
}

// The published splits of a head merged for this lane's columns VREG lane + i (at most NS; lane sp holds split sp's maximum, sum)
template <int NS, int VREG>
JLA_DEV void as_merge(const float* w, int splits, int lane, float (&o)[VREG]) {
  constexpr int pitch = 64 * VREG + 2;
  const int own = min(lane, splits - 1);
  float ms = as_get(w + (size_t)own * pitch), ls = as_get(w + (size_t)own * pitch + 1);
  float part[NS][VREG];
#pragma unroll
  for (int sp = 0; sp < NS; ++sp) as_get_row<VREG>(w + (size_t)min(sp, splits - 1) * pitch + 2 + VREG * lane, part[sp]);  // one round trip
  if (lane >= splits) ls = 0.f;
  const float m = wave_max(ls > 0.f ? ms : -INFINITY);
  const float wt = ls > 0.f ? expf(ms - m) : 0.f;
  const float l = wave_sum(ls * wt);
#pragma unroll
  for (int i = 0; i < VREG; ++i) o[i] = 0.f;
#pragma unroll
  for (int sp = 0; sp < NS; ++sp) {  // (a split without keys holds zeros and has weight 0)
    const float ws = __shfl(wt, sp, 64);
#pragma unroll
    for (int i = 0; i < VREG; ++i) o[i] = fmaf(part[sp][i], sp < splits ? ws : 0.f, o[i]);
  }
#pragma unroll
  for (int i = 0; i < VREG; ++i) o[i] /= l;
}

// dim = 8 DK8, vdim = 64 VREG; ROPE: biases and rotations, else norms and the query temperature
template <typename CT, int DK8, int VREG, int ROPE, int WAVES>
__global__ void __launch_bounds__(64 * WAVES) attn_step_kernel(AttnStep p) {
  constexpr int dim = 8 * DK8, vdim = 64 * VREG, ND = dim / 64;
  __shared__ float qs_[WAVES][dim], row_[WAVES][dim > vdim ? dim : vdim], cs_[WAVES][2][64], sn_[WAVES][2][64];
  __shared__ float join[WAVES > 1 ? WAVES : 1][64 * VREG + 2];
  const AttnBias& a = p.a;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sp = blockIdx.x * WAVES + wave, h = blockIdx.y, b = blockIdx.z;
  float (&qs)[dim] = qs_[wave];
  auto& row = row_[wave];
  auto& cs = cs_[wave];
  auto& sn = sn_[wave];
  const int g = h / (a.H / a.G);
  const bool tail = sp == a.splits - 1;
  const float* pr = p.proj + (size_t)b * p.ld;
  const int slot = *a.slot, pos = p.positions ? p.positions[b] : 0;
  const bool own = p.own && slot >= 0 && slot < a.T;  // (a full cache drops the token's key, as hy_attn_prep does)
  const int kcol = (a.H + g) * dim, vcol = (a.H + a.G) * dim + g * vdim;
  float qv[ND], kx[ND], vx[VREG];
#pragma unroll
  for (int i = 0; i < ND; ++i) qv[i] = pr[h * dim + lane + 64 * i];
#pragma unroll
  for (int i = 0; i < ND; ++i) kx[i] = own && tail ? pr[kcol + lane + 64 * i] : 0.f;
#pragma unroll
  for (int i = 0; i < VREG; ++i) vx[i] = own && tail ? pr[vcol + lane + 64 * i] : 0.f;
  const int qi = min(slot, a.T - 1);
  AbSpan span = ab_span(a, qi);
  if (own) --span.n;  // (the token's own key comes from the projection)
  int j_lo, j_hi;
  ab_split_range(a, span, sp, j_lo, j_hi);
  using Chunk = KeyChunk<CT, DK8, VREG>;
  const int vlane = Chunk::vlane(lane);
  const CT* kbase = reinterpret_cast<const CT*>(a.kc) + ((size_t)b * a.G + g) * a.T * dim;
  const CT* vbase = reinterpret_cast<const CT*>(a.vc) + ((size_t)b * a.G + g) * a.T * vdim;
  Chunk ch;
  float bl = 0.f;
  auto fetch = [&](int j0) {
    auto slot_of = [&](int i) { return ab_key(span, min(j0 + i, j_hi - 1)); };
    ch.load(kbase, dim, vbase, vdim, lane, slot_of);
    bl = a.bias ? a.bias[(size_t)min(qi - slot_of(Chunk::key(lane)), a.nbias - 1) * a.H + h] : 0.f;
  };
  const bool any = j_lo < j_hi;
  if (any) fetch(j_lo);
  // the query, and on the last split the token's key and value
  if (ROPE) {
#pragma unroll 1
    for (int set = 0; set < 2; ++set) {  // angles of q and k, then of v
      const double* freq = set ? p.v_freq : p.qk_freq;
      const int half = set ? p.v_half : p.qk_half;
      if (lane < half) {
        const double t = (double)pos * freq[lane];
        float s_, c_;
        sincosf((float)(t - 6.283185307179586476925 * rint(t * 0.159154943091895335769)), &s_, &c_);
        cs[set][lane] = c_;
        sn[set][lane] = s_;
      }
    }
    if (p.col_bias) {
#pragma unroll
      for (int i = 0; i < ND; ++i) {
        qv[i] += p.col_bias[h * dim + lane + 64 * i];
        kx[i] += p.col_bias[kcol + lane + 64 * i];
      }
#pragma unroll
      for (int i = 0; i < VREG; ++i) vx[i] += p.col_bias[vcol + lane + 64 * i];
    }
    as_turn<ND>(qv, row, p.qk_half, cs[0], sn[0], lane);
    if (own && tail) {
      as_turn<ND>(kx, row, p.qk_half, cs[0], sn[0], lane);
      as_turn<VREG>(vx, row, p.v_half, cs[1], sn[1], lane);
    }
  } else {
    float sc = as_norm<ND>(qv, p.eps);
    if (p.temp_coef != 0.f) sc *= 1.f + p.temp_coef * logf((float)((pos + 1) / p.temp_every) + 1.f);
#pragma unroll
    for (int i = 0; i < ND; ++i) qv[i] *= sc;
    if (own && tail) {
      const float sk = as_norm<ND>(kx, p.eps), sv = as_norm<VREG>(vx, p.eps);
#pragma unroll
      for (int i = 0; i < ND; ++i) kx[i] *= sk;
#pragma unroll
      for (int i = 0; i < VREG; ++i) vx[i] *= sv;
    }
  }
#pragma unroll
  for (int i = 0; i < ND; ++i) qs[lane + 64 * i] = qv[i];
  as_order();
  const bool sunk = a.sink && sp == 0;
  const float hs = a.head_scale ? a.head_scale[h] : 1.f;
  float m_run = sunk ? a.sink[h] : -INFINITY, l_run = sunk ? 1.f : 0.f, acc[VREG];  // acc[i]: column VREG vlane + i
  float q8[8], acc8[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    q8[e] = qs[8 * (lane % DK8) + e];
    acc8[e] = 0.f;
  }
  for (int j0 = j_lo; j0 < j_hi; j0 += 64) {
    if (j0 != j_lo) fetch(j0);
    float sc = ch.score(q8, lane) * a.scale * hs;
    if (a.softcap > 0.f) sc = a.softcap * tanhf(sc / a.softcap);
    sc += bl;
    const bool in = j0 + Chunk::key(lane) < j_hi;
    if (!in) sc = -INFINITY;
    const float m_new = fmaxf(m_run, wave_max(sc));
    const float corr = expf(m_run - m_new);
    const float pw = in ? expf(sc - m_new) : 0.f;  // (0 past the split)
    l_run = l_run * corr + wave_sum(pw);
    m_run = m_new;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc8[e] *= corr;
    ch.add(acc8, pw, lane);
  }
  Chunk::columns(acc8, lane, acc);
  if (own && tail) {  // the token's own key, as the cache holds it
    CT kb[ND], vb[VREG];
    float dot = 0.f;
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      as_held(kb[i], kx[i]);
      dot = fmaf(qv[i], as_number(kb[i]), dot);
    }
    as_order();  // (row: the rotations are done)
#pragma unroll
    for (int i = 0; i < VREG; ++i) {
      as_held(vb[i], vx[i]);
      row[lane + 64 * i] = as_number(vb[i]);
    }
    if (h % (a.H / a.G) == 0) {
      CT* kd = const_cast<CT*>(reinterpret_cast<const CT*>(a.kc)) + (((size_t)b * a.G + g) * a.T + slot) * dim;
      CT* vd = const_cast<CT*>(reinterpret_cast<const CT*>(a.vc)) + (((size_t)b * a.G + g) * a.T + slot) * vdim;
#pragma unroll
      for (int i = 0; i < ND; ++i) kd[lane + 64 * i] = kb[i];
#pragma unroll
      for (int i = 0; i < VREG; ++i) vd[lane + 64 * i] = vb[i];
    }
    float sc = wave_sum(dot) * a.scale * hs;
    if (a.softcap > 0.f) sc = a.softcap * tanhf(sc / a.softcap);
    if (a.bias) sc += a.bias[h];
    const bool none = sc == -INFINITY;  // (alone in its split it must not turn the split's empty sums into NaN)
    const float m_new = fmaxf(m_run, sc), corr = none ? 1.f : expf(m_run - m_new), pw = none ? 0.f : expf(sc - m_new);
    l_run = l_run * corr + pw;
    m_run = m_new;
    as_order();
#pragma unroll
    for (int i = 0; i < VREG; ++i) acc[i] = fmaf(pw, row[VREG * vlane + i], acc[i] * corr);
  }
  float o[VREG];
  if (WAVES > 1) {  // the workgroup's splits, joined by its first wave
    if (lane == 0) {
      join[wave][0] = m_run;
      join[wave][1] = l_run;
    }
#pragma unroll
    for (int i = 0; i < VREG; ++i) join[wave][2 + VREG * vlane + i] = acc[i];
    __syncthreads();
    if (wave) return;
    float m = m_run;
#pragma unroll
    for (int w = 1; w < WAVES; ++w) m = join[w][1] > 0.f ? fmaxf(m, join[w][0]) : m;
    const float mine = l_run > 0.f ? expf(m_run - m) : 0.f;
    l_run *= mine;
#pragma unroll
    for (int i = 0; i < VREG; ++i) acc[i] *= mine;
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
      const float wt = join[w][1] > 0.f ? expf(join[w][0] - m) : 0.f;
      l_run = fmaf(join[w][1], wt, l_run);
#pragma unroll
      for (int i = 0; i < VREG; ++i) acc[i] = fmaf(join[w][2 + VREG * vlane + i], wt, acc[i]);
    }
    m_run = m;
  }
  const int groups = (a.splits + WAVES - 1) / WAVES;
  const int at_o = groups > 1 ? lane : vlane;  // o[i]: column VREG at_o + i
  if (groups > 1) {
    constexpr int pitch = vdim + 2;
    float* head = a.ws + ((size_t)b * a.H + h) * a.splits * pitch;
    float* w = head + (size_t)blockIdx.x * pitch;
    if (lane == 0) {
      as_put(w, m_run);
      as_put(w + 1, l_run);
    }
    as_put_row<VREG>(w + 2 + VREG * vlane, acc);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the split's numbers are out before its ticket is
    int32_t* ticket = p.tickets + ((size_t)b * a.H + h) * AS_TICKET;
    int before = 0;
    if (lane == 0) before = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane(before) != groups - 1) return;
    asm volatile("" ::: "memory");
    if (lane == 0) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // (one branch for all of it, as in ab_merge; one wave per workgroup: at most 16 splits, two: 64)
    if (WAVES > 1 && groups > 16) as_merge<32, VREG>(head, groups, lane, o);
    else as_merge<16, VREG>(head, groups, lane, o);
  } else {
#pragma unroll
    for (int i = 0; i < VREG; ++i) o[i] = acc[i] / l_run;
  }
  if (ROPE && p.turn) {  // the summed values turned back by the query's position
    as_order();
#pragma unroll
    for (int i = 0; i < VREG; ++i) row[VREG * at_o + i] = o[i];
    as_order();
#pragma unroll
    for (int i = 0; i < VREG; ++i) {
      const int c = VREG * at_o + i, half = p.v_half, f = c < half ? c : c - half;
      if (c < 2 * half) {
        const float s_ = p.turn_sign * sn[1][f], other = row[c < half ? c + half : f];
        o[i] = c < half ? o[i] * cs[1][f] - other * s_ : o[i] * cs[1][f] + other * s_;
      }
      o[i] *= p.turn_gain;
    }
  }
#pragma unroll
  for (int i = 0; i < VREG; ++i) {
    const size_t at = (size_t)b * a.ldo + (size_t)h * vdim + VREG * at_o + i;
    if (a.out_bf16) reinterpret_cast<bf16_t*>(a.out)[at] = f2bf(o[i]);
    else reinterpret_cast<float*>(a.out)[at] = o[i];
  }
}

// Heads of 64 or 128 numbers, up to 2560 splits in all. hy_attn_decode_splits cuts rows x heads = P of long caches in 2048 / P, rounded up: that
// is within it for P up to 640 and most beyond (683 to 853, 1024 to 1280, 2048 to 2560), while P of 641 to 682, 854 to 1023 and 1281 to 2047,
// which round up past it, keep the separate launches that they had (not measured here). A decode step with two of these launches in the place of
// three or four each, us, separate | here, heads of 128, rows x heads x splits: norms, 2 x 16 x 47 317 | 312, 3 x 16 x 33 384 | 378, 8 x 16 x 16 442 |
// 435, 8 x 32 x 5 1164 | 1146, 32 x 16 x 4 663 | 662; rotations, 8 x 16 x 16 274 | 268, 13 x 32 x 5 708 | 695, 32 x 16 x 4 447 | 435, 128 x 16 x 1 721 | 707.
constexpr long long AS_MAX_WAVES = 2560;
constexpr int AS_PAIR_SPLITS = 16;  // more of them: two per workgroup (hy_attn_step)

bool hy_attn_step_takes(const AttnStep& p) {
  const AttnBias& a = p.a;
  return a.S == 1 && a.maps == 1 && (a.dim == 64 || a.dim == 128) && (a.vdim == 64 || a.vdim == 128) &&
         a.ldk == a.dim && a.ldv == a.vdim && ((uintptr_t)a.kc & 15) == 0 && ((uintptr_t)a.vc & 15) == 0 && a.splits >= 1 &&
         a.splits <= 64 && (long long)a.B * a.H * a.splits <= AS_MAX_WAVES;
}

int hy_attn_step(const AttnStep& p, hipStream_t s) {
  const AttnBias& a = p.a;
  if (a.B < 0 || a.H < 1 || a.G < 1 || a.H % a.G || a.T < 1 || !hy_attn_step_takes(p)) return -1;
  if (a.bias && a.nbias < 1) return -3;
  if (a.chunk < 0 || a.window < 0 || a.keep_first < 0 || (a.chunk > 0 && a.window > 0)) return -7;
  if (a.gate || a.ldo < a.H * a.vdim) return -8;
  if (p.rope && (p.qk_half < 0 || 2 * p.qk_half > a.dim || p.v_half < 0 || 2 * p.v_half > a.vdim || !p.positions)) return -2;
  if (!p.rope && p.temp_coef != 0.f && (p.temp_every < 1 || !p.positions)) return -2;
  if (p.ld < a.H * a.dim + (p.own ? a.G * (a.dim + a.vdim) : 0)) return -4;
  if (a.splits > 1 && (!a.ws || !p.tickets)) return -5;
  if (a.B == 0) return 0;
  // Two splits per workgroup halve what a head publishes, from 17 splits on (33 splits, keys in no cache: a decode step with two of
  // these launches 241.8 -> 236.2 us; 2 splits alone 7.2 -> 8.7).
  const int waves = a.splits > AS_PAIR_SPLITS ? 2 : 1;
  const dim3 grid((a.splits + waves - 1) / waves, a.H, a.B);
#define AS_ONE(DK8, VREG, ROPE)                                                                      \
  do {                                                                                               \
    if (!a.cbf16 && waves == 2) attn_step_kernel<float, DK8, VREG, ROPE, 2><<<grid, 128, 0, s>>>(p); \
    else if (!a.cbf16) attn_step_kernel<float, DK8, VREG, ROPE, 1><<<grid, 64, 0, s>>>(p);           \
    else if (waves == 2) attn_step_kernel<bf16_t, DK8, VREG, ROPE, 2><<<grid, 128, 0, s>>>(p);       \
    else attn_step_kernel<bf16_t, DK8, VREG, ROPE, 1><<<grid, 64, 0, s>>>(p);                        \
  } while (0)
#define AS_RUN(DK8, VREG)              \
  do {                                 \
    if (p.rope) AS_ONE(DK8, VREG, 1);  \
    else AS_ONE(DK8, VREG, 0);         \
  } while (0)
  if (a.dim == 64 && a.vdim == 64) AS_RUN(8, 1);
  else if (a.dim == 64) AS_RUN(8, 2);
  else if (a.vdim == 64) AS_RUN(16, 1);
  else AS_RUN(16, 2);
#undef AS_RUN
#undef AS_ONE
  JLA_CHECK_LAUNCH();
  return 0;
}

}  // namespace jla
