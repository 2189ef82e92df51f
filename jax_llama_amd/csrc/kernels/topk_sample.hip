// On-device top-k / top-p sampler (replaces HF FlaxTemperatureLogitsWarper ->
// FlaxTopKLogitsWarper -> FlaxTopPLogitsWarper -> categorical that the reference inherits through
// generation.py:28-41 with do_sample = temperature != 0, top_k = 50).
//
// Two kernels, no host sync, hipGraph-capturable:
//   topk_chunk:  grid (ceil(V/8192), B). A 256-thread workgroup holds a chunk of 8192 logits in registers, 32 per thread, in whole lines
//                per load. A bound that at least K of them reach comes from the threads' maxima, wave by wave (16 ballots); the survivors, about
//                1.5 K, rank themselves by counting the better ones, a fourth of the list per wave. It emits exactly K candidates, sorted.
//   topk_merge:  one workgroup per row ranks the C = chunks*K candidates the same way, and either writes
//                them (vocab-parallel TP: each rank's top-K is all-gathered, 400 B per rank per row,
//                then merged again -- exact, since the global top-K is inside the union) or samples:
//                temperature, top-p over the sorted survivors (HF keep rule: a token survives if the
//                probability mass strictly before it is < top_p; the first always survives), then
//                Gumbel-max with counter-based Philox4x32-10 keyed by (seed, step, row, rank) -- every
//                TP rank draws the same token from the same candidates without communicating.
// More survivors than threads (flat, tied or clustered keys, mostly -inf), and always a last chunk of fewer than K + 3 columns: the exact select
// (four radix passes over keys as order-preserving uint32) on all keys of the chunk, read again for every pass.
// Ties: lower vocabulary index first (lax.top_k order).
// What bounds it: of few rows the dependent steps and the code on their path (some 0.13 us per KB in a launch of a few us), of many the vector unit's
// issue and the logits' bytes. Warm, both launches, top 50, us: chunks of 16384 with two radix selects and a sort | of 4096, bound by a radix select
// | here: 128256 columns, 1 row 17.5 | 13.8 | 11.8, 7 17.8 | 15.0 | 12.5, 64 20.9 | 19.7 | 17.2, 300 42.1 | 42.8 | 36.2, 1400 188 | 181 | 145; 32000,
// 1 row 19.4 | 12.3 | 10.0, 1000 45.1 | 50.5 | 30.9, 2048 73.6 | 92.3 | 52.0; top 64 of 300 x 128256 41.9 | 62.1 | 37.1. Chunks of 4096 in the present
// form: 1 x 16032 9.1 for 10.4, 300 x 128256 39.1, 1400 x 32000 43.9 for 38.7.
#include "common.h"
#include "launchers.h"

namespace jla {

constexpr int TK_THREADS = 256, TK_E = 32, TK_CHUNK = TK_THREADS * TK_E, TK_MAX_E = TOPK_MAX_CANDIDATES / TK_THREADS;

JLA_DEV uint32_t fkey(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
JLA_DEV float kfloat(uint32_t k) { return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k); }

struct TkShared {
  uint32_t hist[256];
  uint32_t wsum[TK_THREADS / 64], bound[TK_THREADS / 64];
  uint32_t sel[2];
  uint64_t c[TK_THREADS];   // survivors: key, then the index from its end (the better of two is the larger)
  uint64_t best[64];        // merge: the best K
};

// Block-wide radix select over E keys per thread, key(j) the j-th: T = the K-th largest key; need_eq = how many
// keys equal to T are part of the top K (all keys > T are). Requires K <= number of keys.
template <class Key>
JLA_DEV void radix_select(int E, Key key, int K, TkShared& sh, uint32_t& T, int& need_eq) {
  uint32_t prefix = 0, mask = 0;
  int kr = K;
  for (int shift = 24; shift >= 0; shift -= 8) {
    for (int i = threadIdx.x; i < 256; i += TK_THREADS) sh.hist[i] = 0;
    __syncthreads();
#pragma unroll 1
    for (int j = 0; j < E; ++j) {
      const uint32_t k = key(j);
      if ((k & mask) == prefix) atomicAdd(&sh.hist[(k >> shift) & 255u], 1u);
    }
    __syncthreads();
    if (threadIdx.x < 64) {
      const int l = threadIdx.x;
      uint32_t c[4], s = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {  // lane l owns bins 255-4l .. 252-4l (descending)
        c[q] = sh.hist[255 - 4 * l - q];
        s += c[q];
      }
      const uint32_t incl = wave_scan(s);
      uint32_t above = incl - s;
      if (above < (uint32_t)kr && (uint32_t)kr <= incl) {  // exactly one lane
        for (int q = 0; q < 4; ++q) {
          if ((uint32_t)kr <= above + c[q]) {
            sh.sel[0] = 255 - 4 * l - q;
            sh.sel[1] = above;
            break;
          }
          above += c[q];
        }
      }
    }
    __syncthreads();
    prefix |= sh.sel[0] << shift;
    mask |= 255u << shift;
    kr -= (int)sh.sel[1];
    __syncthreads();
  }
  T = prefix;
  need_eq = kr;
}

// exclusive block scan of one uint32 per thread (256 threads)
JLA_DEV uint32_t block_excl_scan(uint32_t v, TkShared& sh) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint32_t incl = wave_scan(v);
  if (lane == 63) sh.wsum[w] = incl;
  __syncthreads();
  uint32_t base = 0;
  for (int i = 0; i < w; ++i) base += sh.wsum[i];
  __syncthreads();
  return base + incl - v;
}

JLA_DEV uint64_t tk_word(uint32_t key, int idx) { return (uint64_t)key << 32 | (uint32_t)(0x7fffffff - idx); }

// the largest number of 16 bits (of a key: sign, exponent, 7 mantissa bits), zeros behind it, that at least k lanes of the wave reach
JLA_DEV uint32_t wave_bound(uint32_t key, int k) {
  uint32_t t = 0;
#pragma unroll
  for (int bit = 31; bit >= 16; --bit) {
    const uint32_t c = t | 1u << bit;
    if (__popcll(__ballot(key >= c)) >= k) t = c;
  }
  return t;
}

// Survivors sh.c[0 .. S), S <= threads, in any order, sh.hist cleared: calls put(rank, word) for the best K. Every wave counts for all of them the
// better ones in its fourth. TIED: words may be equal (then the first is the better one).
template <bool TIED, class F>
JLA_DEV void rank_few(int S, int K, TkShared& sh, F put) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, part = (S + 15) / 16 * 4;
  if ((int)threadIdx.x >= S && (int)threadIdx.x < 4 * part) sh.c[threadIdx.x] = 0;  // (better than none)
  __syncthreads();
  for (int g = 0; g < S; g += 64) {
    const uint64_t own = sh.c[g + lane];
    uint32_t better = 0;
    for (int i = wave * part; i < (wave + 1) * part; i += 4) {
      uint64_t o[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) o[u] = sh.c[i + u];
#pragma unroll
      for (int u = 0; u < 4; ++u) better += o[u] > own || (TIED && o[u] == own && i + u < g + lane);
    }
    if (g + lane < S) atomicAdd(&sh.hist[g + lane], better);
  }
  __syncthreads();
  if ((int)threadIdx.x < S) {
    const int rank = sh.hist[threadIdx.x];
    if (rank < K) put(rank, sh.c[threadIdx.x]);
  }
}

// A bound that at least K keys of the block reach, and of logits about 1.5 K: a fourth of K of every wave's threads hold a key that reaches their
// wave's, `most` a thread's largest. Clears sh.hist.
JLA_DEV uint32_t block_bound(uint32_t most, int K, TkShared& sh) {
  constexpr int WAVES = TK_THREADS / 64;
  const uint32_t own = wave_bound(most, (K + WAVES - 1) / WAVES);
  if ((threadIdx.x & 63) == 0) sh.bound[threadIdx.x >> 6] = own;
  sh.hist[threadIdx.x] = 0;
  __syncthreads();
  uint32_t t = sh.bound[0];
#pragma unroll
  for (int w = 1; w < WAVES; ++w) t = min(t, sh.bound[w]);
  return __builtin_amdgcn_readfirstlane(t);
}

// The top K of the block's keys, sorted, where few enough reach the bound: calls put(slot, word) once per slot 0..K-1. reaches(j): whether this
// thread's j-th of E does; word(j): the key and its index (0 .. 0x7fffffff). False: more than threads.
template <int E, bool TIED, class Reaches, class Word, class F>
JLA_DEV bool select_few(Reaches reaches, int K, TkShared& sh, Word word, F put) {
  const int wave = threadIdx.x >> 6;
  uint32_t ns = 0;
#pragma unroll
  for (int j = 0; j < E; ++j) ns += reaches(j);
  const uint32_t incl = wave_scan(ns);
  if ((threadIdx.x & 63) == 63) sh.wsum[wave] = incl;
  __syncthreads();
  uint32_t at = incl - ns;
  int S = 0;
#pragma unroll
  for (int w = 0; w < TK_THREADS / 64; ++w) {
    if (w < wave) at += sh.wsum[w];
    S += sh.wsum[w];
  }
  if (S > TK_THREADS) return false;
#pragma unroll
  for (int j = 0; j < E; ++j)
    if (reaches(j)) sh.c[at++] = word(j);
  rank_few<TIED>(S, K, sh, put);
  return true;
}

// ... of any keys, E neighbouring ones per thread, key(j) this thread's j-th: put(slot, key, j), slots above the threshold in element order, then
// the lowest elements at it. (The keys are read again for every pass: the rare case takes no registers from the other.)
template <class Key, class F>
JLA_DEV void select_all(int E, Key key, int K, TkShared& sh, F put) {
  uint32_t T, ngt = 0, neq = 0;
  int need_eq;
  radix_select(E, key, K, sh, T, need_eq);
#pragma unroll 1
  for (int j = 0; j < E; ++j) {
    const uint32_t k = key(j);
    ngt += k > T;
    neq += k == T;
  }
  const uint32_t ex = block_excl_scan((ngt << 16) | neq, sh);
  int gpos = ex >> 16, epos = ex & 0xffff;
#pragma unroll 1
  for (int j = 0; j < E; ++j) {
    const uint32_t k = key(j);
    if (k > T) put(gpos++, k, j);
    else if (k == T && epos++ < need_eq) put(K - need_eq + epos - 1, k, j);
  }
}

__global__ void __launch_bounds__(TK_THREADS, 8)
    topk_chunk_kernel(const float* __restrict__ logits, int V, int K, int idx_offset, float* __restrict__ cv,
                      int32_t* __restrict__ ci) {
  __shared__ TkShared sh;
  const int b = blockIdx.y, c = blockIdx.x, nch = gridDim.x, base = c * TK_CHUNK;
  const float* x = logits + (size_t)b * V;
  // four numbers per access; else one, and of the last few columns neighbours are dealt to the waves in turn (the bound needs K / 4 in each)
  const bool last = V - base < 4 * TK_THREADS, vec = (V & 3) == 0 && !last;
  const int place = last ? 4 * ((int)threadIdx.x & 63) + ((int)threadIdx.x >> 6) : (int)threadIdx.x;
  auto element = [&](int j) { return base + (vec ? 4 * TK_THREADS * (j / 4) + 4 * (int)threadIdx.x + j % 4 : TK_THREADS * j + place); };
  float v[TK_E];
  if (vec && base + TK_CHUNK <= V) {
#pragma unroll
    for (int q = 0; q < TK_E / 4; ++q) {
      const float4 f = *reinterpret_cast<const float4*>(x + element(4 * q));
      v[4 * q] = f.x, v[4 * q + 1] = f.y, v[4 * q + 2] = f.z, v[4 * q + 3] = f.w;
    }
  } else if (vec) {
#pragma unroll
    for (int q = 0; q < TK_E / 4; ++q) {
      const bool in = element(4 * q) < V;
      const float4 f = in ? *reinterpret_cast<const float4*>(x + element(4 * q)) : float4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
      v[4 * q] = f.x, v[4 * q + 1] = f.y, v[4 * q + 2] = f.z, v[4 * q + 3] = f.w;
    }
  } else {
#pragma unroll
    for (int j = 0; j < TK_E; ++j) v[j] = element(j) < V ? x[element(j)] : -INFINITY;
  }
  float* ov = cv + ((size_t)b * nch + c) * K;
  int32_t* oi = ci + ((size_t)b * nch + c) * K;
  auto put = [&](int slot, uint32_t k, int e) {
    ov[slot] = e < V ? kfloat(k) : -INFINITY;
    oi[slot] = e < V ? idx_offset + e : 0x7fffffff;
  };
  float most = -INFINITY;
#pragma unroll
  for (int j = 0; j < TK_E; ++j) most = fmaxf(most, v[j]);
  const float bound = kfloat(block_bound(fkey(most), K, sh));
  // (not below the bound: a NaN, which comes first, is kept; where the bound is that of -inf everything is)
  if (select_few<TK_E, false>([&](int j) { return !(v[j] < bound); }, K, sh, [&](int j) { return element(j) < V ? tk_word(fkey(v[j]), element(j)) : 0; },
                              [&](int slot, uint64_t w) { put(slot, (uint32_t)(w >> 32), 0x7fffffff - (int)(uint32_t)w); }))
    return;
  const int first = base + TK_E * (int)threadIdx.x;  // (in element order now)
  __syncthreads();
  select_all(TK_E, [&](int j) { return first + j < V ? fkey(x[first + j]) : 0u; }, K, sh, [&](int slot, uint32_t k, int j) { put(slot, k, first + j); });
}

JLA_DEV uint4 philox4x32_10(uint4 ctr, uint2 k) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint32_t lo0 = 0xD2511F53u * ctr.x, hi0 = __umulhi(0xD2511F53u, ctr.x);
    const uint32_t lo1 = 0xCD9E8D57u * ctr.z, hi1 = __umulhi(0xCD9E8D57u, ctr.z);
    ctr = make_uint4(hi1 ^ ctr.y ^ k.x, lo1, hi0 ^ ctr.w ^ k.y, lo0);
    k.x += 0x9E3779B9u;
    k.y += 0xBB67AE85u;
  }
  return ctr;
}

// mode 0: write the sorted top-K (out_v/out_i [B, K]); mode 1: sample one token per row into nxt[B].
// E candidates per thread: the smallest that covers C, so that the candidates spread over most threads and the bound from their maxima is close.
template <int E>
__global__ void __launch_bounds__(TK_THREADS)
    topk_merge_kernel(const float* __restrict__ cv, const int32_t* __restrict__ ci, int C, int K, int mode,
                      float* __restrict__ out_v, int32_t* __restrict__ out_i, int32_t* __restrict__ nxt,
                      float inv_temp, float top_p, uint32_t seed_lo, uint32_t seed_hi,
                      const int32_t* __restrict__ step) {
  __shared__ TkShared sh;
  const int b = blockIdx.x;
  const float* bv = cv + (size_t)b * C;
  const int32_t* bi = ci + (size_t)b * C;
  auto put = [&](int slot, uint64_t w) { sh.best[slot] = w; };
  bool few = true;
  if constexpr (E == 1) {  // every candidate is ranked
    if ((int)threadIdx.x < C) sh.c[threadIdx.x] = tk_word(fkey(bv[threadIdx.x]), bi[threadIdx.x]);
    sh.hist[threadIdx.x] = 0;
    rank_few<true>(C, K, sh, put);
  } else {
    // (the candidates of a chunk are sorted: dealt to the waves in turn and, turned by 37 threads from one 256 to the next, to threads of
    // their own, whatever K divides, so that the bound is close: K 64 without the turn: 16 threads in 64 held the best of every chunk, and
    // from 20 chunks on more candidates than threads reached it)
    auto from = [&](int j) { return (4 * ((int)threadIdx.x & 63) + ((int)threadIdx.x >> 6) + 37 * j) % TK_THREADS + TK_THREADS * j; };
    constexpr int AT = E <= 16 ? E : 1;  // indices held; of more candidates they are read where needed (registers)
    uint32_t key[E], most = 0;
    int32_t at[AT];
#pragma unroll
    for (int j = 0; j < E; ++j) {
      const int e = from(j);
      key[j] = e < C ? fkey(bv[e]) : 0u;
      if constexpr (AT == E) at[j] = e < C ? bi[e] : 0x7fffffff;
      most = max(most, key[j]);
    }
    const uint32_t bound = block_bound(most, K, sh);
    few = select_few<E, true>([&](int j) { return key[j] >= bound; }, K, sh,
                              [&](int j) { return tk_word(key[j], AT == E ? at[j % AT] : (from(j) < C ? bi[from(j)] : 0x7fffffff)); }, put);
  }
  if (!few) {
    const int base = threadIdx.x * E;
    __syncthreads();
    select_all(E, [&](int j) { return base + j < C ? fkey(bv[base + j]) : 0u; }, K, sh,
               [&](int slot, uint32_t k, int j) { sh.best[slot] = tk_word(k, base + j < C ? bi[base + j] : 0x7fffffff); });
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x;
  // value descending, then index ascending
  uint64_t v = lane < K ? sh.best[lane] : 0ull;
  if (!few) {
#pragma unroll
    for (int k = 2; k <= 64; k <<= 1) {
      lane_halves([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        if (j >= k) return;
        const uint32_t lo = lane_xor<j>((uint32_t)v), hi = lane_xor<j>((uint32_t)(v >> 32));
        const uint64_t o = ((uint64_t)hi << 32) | lo;
        const bool desc = (lane & k) == 0;  // final k = 64: whole wave descending
        const bool lower = (lane & j) == 0;
        const bool take_max = desc == lower;
        v = take_max ? (o > v ? o : v) : (o < v ? o : v);
      });
    }
  }
  const float val = lane < K ? kfloat((uint32_t)(v >> 32)) : -INFINITY;
  const int32_t idx = lane < K ? 0x7fffffff - (int32_t)(uint32_t)v : 0x7fffffff;
  if (mode == 0) {
    if (lane < K) {
      out_v[(size_t)b * K + lane] = val;
      out_i[(size_t)b * K + lane] = idx;
    }
    return;
  }
  // temperature -> softmax over the survivors -> top-p keep mask
  const float l = lane < K ? val * inv_temp : -INFINITY;
  const float mx = __shfl(l, 0, 64);  // sorted: lane 0 holds the max
  float p = lane < K ? __expf(l - mx) : 0.f;
  p /= wave_sum(p);
  float incl = p;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float t = __shfl_up(incl, o, 64);
    if (lane >= o) incl += t;
  }
  const bool keep = lane < K && (lane == 0 || (incl - p) < top_p);
  // Gumbel-max with Philox(seed; counter = (lane, row, step, 0))
  const uint4 r = philox4x32_10(make_uint4((uint32_t)lane, (uint32_t)b, (uint32_t)step[0], 0u),
                                make_uint2(seed_lo, seed_hi));
  const float u = ((float)(r.x >> 8) + 0.5f) * (1.0f / 16777216.0f);
  const float g = -__logf(-__logf(u));
  float score = keep ? l + g : -INFINITY;
  int best = lane;
  lane_halves([&](auto j) {
    constexpr int J = decltype(j)::value;
    const float os = __uint_as_float(lane_xor<J>(__float_as_uint(score)));
    const int ob = (int)lane_xor<J>((uint32_t)best);
    if (os > score || (os == score && ob < best)) {
      score = os;
      best = ob;
    }
  });
  const int32_t tok = __shfl(idx, best, 64);
  if (lane == 0) nxt[b] = tok;
}

int topk_chunks(int V) { return (V + TK_CHUNK - 1) / TK_CHUNK; }

int topk_chunk(const float* logits, int B, int V, int K, int idx_offset, float* cv, int32_t* ci, hipStream_t s) {
  if (B <= 0) return 0;
  if (K < 1 || K > 64 || K > V) return -1;
  dim3 grid(topk_chunks(V), B);
  topk_chunk_kernel<<<grid, TK_THREADS, 0, s>>>(logits, V, K, idx_offset, cv, ci);
  JLA_CHECK_LAUNCH();
  return 0;
}

int topk_merge(const float* cv, const int32_t* ci, int B, int C, int K, int mode, float* out_v, int32_t* out_i,
               int32_t* nxt, float temperature, float top_p, uint64_t seed, const int32_t* step, hipStream_t s) {
  if (B <= 0) return 0;
  if (K < 1 || K > 64 || K > C || C > TOPK_MAX_CANDIDATES) return -1;
  if (mode == 1 && (!nxt || !step || !(temperature > 0.f))) return -2;
#define JLA_TKM(E)                                                                                          \
  topk_merge_kernel<E><<<B, TK_THREADS, 0, s>>>(cv, ci, C, K, mode, out_v, out_i, nxt, 1.0f / temperature, top_p, \
                                                (uint32_t)seed, (uint32_t)(seed >> 32), step)
  if (C <= TK_THREADS / 2)
    JLA_TKM(1);
  else if (C <= 4 * TK_THREADS)
    JLA_TKM(4);
  else if (C <= 8 * TK_THREADS)
    JLA_TKM(8);
  else if (C <= 16 * TK_THREADS)
    JLA_TKM(16);
  else
    JLA_TKM(TK_MAX_E);
#undef JLA_TKM
  JLA_CHECK_LAUNCH();
  return 0;
}

}  // namespace jla
