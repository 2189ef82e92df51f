// Prompt attention over fp32 caches on the fp32 matrix instruction (heads of 64 or 128 numbers): the exact form of attn_bias.hip's
// flash kernel.
//
// A workgroup takes 16 queries of a head and deals the key tiles of 16 to its four waves, whose maxima, sums and values are joined
// through LDS. S^T = K Q^T: a lane holds key (row) or query (column) lane & 15 and four consecutive numbers per 16, so rows come in
// 16-byte loads and step r of v_mfma_f32_16x16x4_f32 takes the numbers 16 i + 4 (lane >> 4) + r of both. Its result, keys
// 4 (lane >> 4) + r of query lane & 15, is in place the B operand of O^T += V^T P^T with the keys in that order; value tile
// (jj, e) holds the columns 64 jj + 4 row + e, so that values too come and go in 16-byte pieces.
// Masked keys have weight 0; where a masked tile holds a value that is not finite, the value takes no part in the product, and only
// the queries that see its key get in its column what the product would give them: an infinity, or NaN.
// What bounds it: the chain of a tile (32 + 32 matrix instructions, the softmax between them) over the keys / 64 tiles of a wave.
// One wave per query that read every key for itself took 138 us for 400 tokens and 173 us for 200 tokens behind 400 (16 heads of 128).
// Two workgroups share a compute unit (three at 64 x 64), with their accumulators among the vector unit's registers, which rescale
// them (231 at 128 x 128): a column that counts in a masked tile keeps two sums and not one per kind. With three sums the kernel took
// 254 and half of its accumulators, one workgroup: 13 rows x 32 heads x 64 tokens behind 400 129 us, 101 without bounds on the
// registers; over 2 to 400 tokens behind 0 to 1500 of one row x 16 heads of 128 9 % and 6 % more time than here, 32 x 32 36 % and 1 %.
#include "attn_span.h"

namespace jla {

constexpr int AF_Q = 16, AF_K = 16;

template <int DK, int VT>  // dim = 16 DK, vdim = 64 VT
__global__ void __launch_bounds__(256, DK == 4 && VT == 1 ? 3 : 2) attn_f32_kernel(AttnBias p) {
  constexpr int dim = 16 * DK, vdim = 64 * VT, PITCH = vdim + 4;
  __shared__ __attribute__((aligned(16))) float os[4][AF_Q][PITCH];
  __shared__ float ms[4][AF_Q], ls[4][AF_Q];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, lg = lane >> 4;
  const int nq = (p.S + AF_Q - 1) / AF_Q;
  const int s0 = (nq - 1 - (int)blockIdx.x) * AF_Q, h = blockIdx.y, b = blockIdx.z;  // long rows first
  const int g = h / (p.H / p.G), slot = *p.slot;
  const int sq = min(s0 + c, p.S - 1);  // (surplus lanes repeat the last query; never stored)
  const int qi = min(slot + sq, p.T - 1), q0 = min(slot + s0, p.T - 1), q_last = min(slot + min(s0 + AF_Q, p.S) - 1, p.T - 1);
  f32x4 qf[DK];
  {
    const float* q = p.q + (((size_t)b * p.S + sq) * p.H + h) * dim + 4 * lg;
#pragma unroll
    for (int i = 0; i < DK; ++i) qf[i] = *reinterpret_cast<const f32x4*>(q + 16 * i);
  }
  const float* kbase = reinterpret_cast<const float*>(p.kc) + ((size_t)b * p.G + g) * p.T * dim;
  const float* vbase = reinterpret_cast<const float*>(p.vc) + ((size_t)b * p.G + g) * p.T * vdim;
  f32x4 o[VT][4];
#pragma unroll
  for (int j = 0; j < VT; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[j][e] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool sunk = p.sink && wave == 0;  // (l_run holds this quarter's part of the sum: the sink counts once)
  float m_run = sunk ? p.sink[h] : -INFINITY, l_run = sunk && lg == 0 ? 1.f : 0.f;
  const float hs = p.head_scale ? p.head_scale[h] : 1.f;
  const int lo_q = ab_span(p, qi).lo, lo_last = ab_span(p, q_last).lo;
  const int j_begin = ab_span(p, q0).lo / AF_K * AF_K;
  const int kfirst = p.window > 0 ? p.keep_first : 0;
  const int kf_tiles = min((kfirst + AF_K - 1) / AF_K, j_begin / AF_K);  // kept first keys' tiles, then the walk from j_begin on
  const int tiles = kf_tiles + (q_last - j_begin) / AF_K + 1;
  auto tile_key = [&](int t) { return t < kf_tiles ? t * AF_K : j_begin + (t - kf_tiles) * AF_K; };
  f32x4 kn[DK], vn[VT][4];
  auto fetch = [&](int t) {
    const int j0 = tile_key(min(t, tiles - 1));
    const float* kr = kbase + (size_t)min(j0 + c, p.T - 1) * dim + 4 * lg;
#pragma unroll
    for (int i = 0; i < DK; ++i) kn[i] = *reinterpret_cast<const f32x4*>(kr + 16 * i);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < VT; ++j)
        vn[j][r] = *reinterpret_cast<const f32x4*>(vbase + (size_t)min(j0 + 4 * lg + r, p.T - 1) * vdim + 64 * j + 4 * c);
  };
  fetch(wave);
  for (int t = wave; t < tiles; t += 4) {
    const int j0 = tile_key(t);
    f32x4 kc[DK], vc[VT][4];
#pragma unroll
    for (int i = 0; i < DK; ++i) kc[i] = kn[i];
#pragma unroll
    for (int j = 0; j < VT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) vc[j][r] = vn[j][r];
    fetch(t + 4);  // (past the last tile: it again, unused)
    f32x4 sa[4];  // (four chains: none longer than the plain kernel's)
#pragma unroll
    for (int r = 0; r < 4; ++r) sa[r] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < DK; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) sa[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(kc[i][r], qf[i][r], sa[r], 0, 0, 0);
    f32x4 sc = (sa[0] + sa[1]) + (sa[2] + sa[3]);
    // some (query, key) of the tile is masked
    const bool diag = j0 + AF_K - 1 > q0 || (j0 < lo_last && j0 + AF_K - 1 >= kfirst);
    bool seen[4];
    float tmax = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = j0 + 4 * lg + r;
      float x = sc[r] * p.scale * hs;
      if (p.softcap > 0.f) x = p.softcap * tanhf(x / p.softcap);
      if (p.bias) x += p.bias[(size_t)min(max(qi - j, 0), p.nbias - 1) * p.H + h];
      seen[r] = j <= qi && (j >= lo_q || j < kfirst);
      sc[r] = seen[r] ? x : -INFINITY;
      tmax = fmaxf(tmax, sc[r]);
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    const float m_new = fmaxf(m_run, tmax);
    // (a query may have no visible key in a tile that it shares with its neighbours)
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float corr = expf(m_run - m_use);
    m_run = m_new;
    float psum = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      sc[r] = seen[r] ? expf(sc[r] - m_use) : 0.f;
      psum += sc[r];
    }
    l_run = fmaf(l_run, corr, psum);
#pragma unroll
    for (int j = 0; j < VT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) o[j][e] *= corr;
    bool whole = true;
    if (diag) {
#pragma unroll
      for (int j = 0; j < VT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e) whole &= isfinite(vc[j][r][e]);
    }
    if (__any(!whole)) {  // (wave-uniform)
#pragma unroll
      for (int j = 0; j < VT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // of this column the query sees: infinities (those below in units of 32, a tile has 16 keys), and products that are none
          f32x4 ends = {0.f, 0.f, 0.f, 0.f}, none = ends;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float v = vc[j][r][e], end = isinf(v) ? (v > 0.f ? 1.f : 32.f) : 0.f;
            const bool weighed = sc[r] > 0.f;
            ends = __builtin_amdgcn_mfma_f32_16x16x4f32(end, weighed ? 1.f : 0.f, ends, 0, 0, 0);
            none = __builtin_amdgcn_mfma_f32_16x16x4f32(isnan(v) ? 1.f : 0.f, seen[r] ? 1.f : 0.f, none, 0, 0, 0);
            none = __builtin_amdgcn_mfma_f32_16x16x4f32(end, seen[r] && !weighed ? 1.f : 0.f, none, 0, 0, 0);  // (0 x an infinity)
            if (!isfinite(v)) vc[j][r][e] = 0.f;
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int n = (int)ends[r];
            if (n & 31) o[j][e][r] += INFINITY;
            if (n >> 5) o[j][e][r] -= INFINITY;
            if (none[r] > 0.f) o[j][e][r] = NAN;
          }
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < VT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[j][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vc[j][r][e], sc[r], o[j][e], 0, 0, 0);
  }
  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);
  if (lg == 0) ms[wave][c] = m_run;
  __syncthreads();
  const float m_all = fmaxf(fmaxf(ms[0][c], ms[1][c]), fmaxf(ms[2][c], ms[3][c]));
  const float wt = m_run == -INFINITY ? 0.f : expf(m_run - m_all);  // (a wave without keys of this query: zeros)
  if (lg == 0) ls[wave][c] = l_run * wt;
#pragma unroll
  for (int j = 0; j < VT; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r)  // rows 4 lg + r of the tiles e: columns 64 j + 16 lg + 4 r + e
      *reinterpret_cast<f32x4*>(&os[wave][c][64 * j + 16 * lg + 4 * r]) = f32x4{o[j][0][r], o[j][1][r], o[j][2][r], o[j][3][r]} * wt;
  __syncthreads();
  const int t = threadIdx.x >> 4, k4 = 4 * (threadIdx.x & 15);
  if (s0 + t >= p.S) return;
  const float l = (ls[0][t] + ls[1][t]) + (ls[2][t] + ls[3][t]);
  const size_t m = (size_t)b * p.S + s0 + t;
#pragma unroll
  for (int j = 0; j < VT; ++j) {
    const int col = 64 * j + k4;
    auto at = [&](int w) { return *reinterpret_cast<const f32x4*>(&os[w][t][col]); };
    const f32x4 x = (at(0) + at(1)) + (at(2) + at(3));
#pragma unroll
    for (int e = 0; e < 4; ++e) ab_out(p, m, h, col + e, x[e] / l * ab_gate(p, m, h, col + e));
  }
}

// Two to four queries per row over a few keys leave most of a 16 x 16 tile idle; where the workgroups take more than a round (two per
// compute unit, three at 64 x 64) they stay with a wave per query. Us, that | here, heads of 128, soft cap and bias (without), rows x heads:
// 13 x 32, 2 queries over 2 keys 6.5 | 6.8 (6.4 | 6.3); 64 x 32, 2 queries over 2 | 32 | 62 | 122 keys 9.4 | 18 | 30 | 56, here 24 | 31 | 41 |
// 67 (9.3 | 18 | 29 | 55, 22 | 26 | 33 | 49); 4 over 4 | 34 | 64 15 | 32 | 46, 25 | 36 | 41; 6 over 6 28 | 26, 8 over 8 30 | 27. Heads of
// 64: 24 x 32, 4 over 4 6.3 | 5.9; 64 x 32, 2 over 2 | 62 6.8 | 17, 13 | 24. How many keys there are is known where the host knows the
// slot.
static bool af_few(const AttnBias& p) {
  const long long most = (long long)p.S * p.t_cap, round = p.dim == 64 && p.vdim == 64 ? 768 : 512;
  return p.S <= 4 && (long long)p.B * p.H > round && p.t_cap > 0 && most <= (p.bias && p.S == 2 ? 250 : 128);
}

bool hy_attn_f32_takes(const AttnBias& p) {
  auto aligned = [](const void* x) { return ((uintptr_t)x & 15) == 0; };
  return !p.cbf16 && p.S > 1 && !af_few(p) && p.maps == 1 && (p.dim == 64 || p.dim == 128) && (p.vdim == 64 || p.vdim == 128) && p.ldk == p.dim &&
         p.ldv == p.vdim && aligned(p.q) && aligned(p.kc) && aligned(p.vc);
}

int hy_attn_f32(const AttnBias& p, hipStream_t s) {
  const dim3 grid((p.S + AF_Q - 1) / AF_Q, p.H, p.B);
  if (p.dim == 64 && p.vdim == 64) attn_f32_kernel<4, 1><<<grid, 256, 0, s>>>(p);
  else if (p.dim == 64) attn_f32_kernel<4, 2><<<grid, 256, 0, s>>>(p);
  else if (p.vdim == 64) attn_f32_kernel<8, 1><<<grid, 256, 0, s>>>(p);
  else attn_f32_kernel<8, 2><<<grid, 256, 0, s>>>(p);
  JLA_CHECK_LAUNCH();
  return 0;
}

}  // namespace jla
