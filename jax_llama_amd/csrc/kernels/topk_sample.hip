// On-device top-k / top-p sampler (replaces HF FlaxTemperatureLogitsWarper ->
// FlaxTopKLogitsWarper -> FlaxTopPLogitsWarper -> categorical that the reference inherits through
// generation.py:28-41 with do_sample = temperature != 0, top_k = 50).
//
// Two kernels, no host sync, hipGraph-capturable:
//   topk_chunk:  grid (ceil(V/4096), B). A 256-thread workgroup holds a 4096-logit chunk in registers (16 keys per thread,
//                order-preserving uint32 of the fp32 logit, whole lines per load). A bound that at least K keys reach comes from the
//                threads' maxima (LDS radix select, 8 bits per pass, one wave scans the 256-bin histogram with lane moves, two passes);
//                the survivors, about K, rank themselves by counting the better ones. It emits exactly K candidates, sorted.
//   topk_merge:  one workgroup per row ranks the C = chunks*K candidates the same way, and either writes
//                them (vocab-parallel TP: each rank's top-K is all-gathered, 400 B per rank per row,
//                then merged again -- exact, since the global top-K is inside the union) or samples:
//                temperature, top-p over the sorted survivors (HF keep rule: a token survives if the
//                probability mass strictly before it is < top_p; the first always survives), then
//                Gumbel-max with counter-based Philox4x32-10 keyed by (seed, step, row, rank) -- every
//                TP rank draws the same token from the same candidates without communicating.
// More survivors than threads (flat, tied or clustered keys): the exact select on all keys of the chunk.
// Ties: lower vocabulary index first (lax.top_k order).
// What bounds it: dependent steps within a wave and code on its path (some 0.13 us per KB in a launch of a few us). Seven rows x 128256 columns, the
// two kernels: 64 keys per thread in 8 chunks, read 256 bytes apart, exact select and sort of the survivors in six radix passes and 21 exchanges
// 10.9 + 8.9 us; here 6.2 + 9.4. Warm, both, before -> now: 1 row 17.7 -> 14.7, 7 18.0 -> 15.1, 64 20.9 -> 20.7, 300 42.0 -> 44.5, 1400 186 -> 184;
// 200 x 32000 22.8 -> 19.5. (32 keys per thread: 7 rows 16.0, 1400 302; the rare case's keys in registers: 1400 203.)
#include "common.h"
#include "launchers.h"

namespace jla {

constexpr int TK_THREADS = 256, TK_E = 16, TK_CHUNK = TK_THREADS * TK_E, TK_MAX_E = TOPK_MAX_CANDIDATES / TK_THREADS;

JLA_DEV uint32_t fkey(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
JLA_DEV float kfloat(uint32_t k) { return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k); }

struct TkShared {
  uint32_t hist[256];
  uint32_t wsum[TK_THREADS / 64];
  uint32_t sel[2];
  uint64_t c[TK_THREADS];   // survivors: key, then the index from its end (the better of two is the larger)
  uint32_t total;
};

// Block-wide radix select over E keys per thread, key(j) the j-th: T = the K-th largest key; need_eq = how many
// keys equal to T are part of the top K (all keys > T are). Requires K <= number of keys.
// last_shift 16: two passes only, T = the K-th largest key with its low 16 bits cleared (a lower bound with at least K
// keys >= T; need_eq is then meaningless).
template <class Key>
JLA_DEV void radix_select(int E, Key key, int K, TkShared& sh, uint32_t& T, int& need_eq, int last_shift = 0) {
  uint32_t prefix = 0, mask = 0;
  int kr = K;
  for (int shift = 24; shift >= last_shift; shift -= 8) {
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

// The top K of the block's keys, sorted, where few enough reach the bound: calls put(slot, word) once per slot 0..K-1. word(j): key j's and its index
// (0 .. 0x7fffffff). The bound: the top 16 bits (sign, exponent, 7 mantissa bits) of the K-th largest of the 256 per-thread maxima; at least K keys
// reach it, and about that many of logits. False: more than threads.
template <int E, class Word, class F>
JLA_DEV bool select_few(const uint32_t (&key)[E], int K, TkShared& sh, Word word, F put, bool over = false) {
  uint32_t most = 0, T0, ns = 0;
  int none;
#pragma unroll
  for (int j = 0; j < E; ++j) most = max(most, key[j]);
  radix_select(1, [&](int) { return most; }, K, sh, T0, none, 16);
#pragma unroll
  for (int j = 0; j < E; ++j) ns += key[j] >= T0;
  uint32_t at = block_excl_scan(ns, sh);
  if (threadIdx.x == TK_THREADS - 1) sh.total = at + ns;
  __syncthreads();
  const int S = sh.total;
  if (S > TK_THREADS) return false;
#pragma unroll
  for (int j = 0; j < E; ++j)
    if (key[j] >= T0) sh.c[at++] = word(j);
  if ((int)threadIdx.x >= S && threadIdx.x < ((S + 3) & ~3)) sh.c[threadIdx.x] = 0;  // (better than none)
  __syncthreads();
  int rank = K;
  uint64_t own = 0;
  if ((int)threadIdx.x < S) {
    own = sh.c[threadIdx.x];
    rank = 0;
    for (int i = 0; i < S; i += 4) {
      uint64_t o[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) o[u] = sh.c[i + u];
#pragma unroll
      for (int u = 0; u < 4; ++u) rank += o[u] > own || (o[u] == own && i + u < (int)threadIdx.x);
    }
  }
  if (over) __syncthreads();  // (put writes where others read)
  if (rank < K) put(rank, own);
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
  uint32_t key[TK_E];
  auto element = [&](int j) { return base + 4 * TK_THREADS * (j / 4) + 4 * (int)threadIdx.x + j % 4; };
  if ((V & 3) == 0 && base + TK_CHUNK <= V) {
#pragma unroll
    for (int q = 0; q < TK_E / 4; ++q) {
      const float4 v = *reinterpret_cast<const float4*>(x + element(4 * q));
      key[4 * q] = fkey(v.x);
      key[4 * q + 1] = fkey(v.y);
      key[4 * q + 2] = fkey(v.z);
      key[4 * q + 3] = fkey(v.w);
    }
  } else {
#pragma unroll
    for (int j = 0; j < TK_E; ++j) key[j] = element(j) < V ? fkey(x[element(j)]) : 0u;  // 0 < key(-inf)
  }
  float* ov = cv + ((size_t)b * nch + c) * K;
  int32_t* oi = ci + ((size_t)b * nch + c) * K;
  auto put = [&](int slot, uint32_t k, int e) {
    ov[slot] = e < V ? kfloat(k) : -INFINITY;
    oi[slot] = e < V ? idx_offset + e : 0x7fffffff;
  };
  if (select_few(key, K, sh, [&](int j) { return tk_word(key[j], element(j)); },
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
// E candidates per thread: the smallest that covers C, so the candidates spread over most threads and the
// per-thread-maximum prefilter of select_topk compacts them (with TK_E per thread, 16 chunks x 50 candidates sat
// in 25 threads and every merge fell back to the full select)
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
  uint32_t key[E];
  int32_t at[E];
#pragma unroll
  for (int j = 0; j < E; ++j) {  // (a chunk's candidates are sorted: dealt out, so that the threads' maxima are the row's best)
    const int e = threadIdx.x + TK_THREADS * j;
    key[j] = e < C ? fkey(bv[e]) : 0u;
    at[j] = e < C ? bi[e] : 0x7fffffff;
  }
  const bool few = select_few(key, K, sh, [&](int j) { return tk_word(key[j], at[j]); }, [&](int slot, uint64_t w) { sh.c[slot] = w; }, true);
  if (!few) {
    const int base = threadIdx.x * E;
    __syncthreads();
    select_all(E, [&](int j) { return base + j < C ? fkey(bv[base + j]) : 0u; }, K, sh,
               [&](int slot, uint32_t k, int j) { sh.c[slot] = tk_word(k, base + j < C ? bi[base + j] : 0x7fffffff); });
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x;
  // value descending, then index ascending
  uint64_t v = lane < K ? sh.c[lane] : 0ull;
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
  if (C <= 4 * TK_THREADS)
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
