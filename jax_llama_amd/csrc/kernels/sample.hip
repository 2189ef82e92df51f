// Token selection and decode-loop bookkeeping (replaces HF FlaxGenerationMixin's loop body that the
// reference inherits: generation.py:28-41 -> _greedy_search / _sample).
//
// argmax: first index of the row maximum (jnp.argmax semantics), also returns the max value so a
//   vocab-parallel (TP) caller can pick the global winner from one (value, index) pair per rank.
// decode_update: finished rows emit pad, is_sent_finished |= (token == eos), sequences[:, cur_len]
//   = token, positions += 1, cache slot += 1, cur_len += 1 -- all on the device so the whole decode
//   step (model + sampler + state) replays from one hipGraph without host round trips.
#include "common.h"
#include "launchers.h"

namespace jla {

// Greedy choice over logits in memory: the largest, ties to the lowest index, a NaN never chosen; all -inf (or NaN) gives
// index 0. What bounds it: one compute unit pulls about 26 bytes per ns, so a row goes to several workgroups until every
// unit has a few (whose results a second launch of one wave per row reduces), 16 bytes per load, four in flight. One
// workgroup of 1024 threads per row took 8.1 us for 1 x 32000, 23.4 for 1 x 128256 and 45.9 for 200 x 128256 (replayed
// back to back); now 4.4, 4.4 and 19.0.
JLA_DEV void am_better(float& bv, int& bi, float ov, int oi) {
  if (ov > bv || (ov == bv && oi < bi)) {
    bv = ov;
    bi = oi;
  }
}
JLA_DEV void am_wave(float& bv, int& bi) {
  lane_halves([&](auto j) {
    constexpr int J = decltype(j)::value;
    const float ov = __uint_as_float(lane_xor<J>(__float_as_uint(bv)));
    am_better(bv, bi, ov, (int)lane_xor<J>((uint32_t)bi));
  });
}

// grid (splits, rows): columns [c0, c0 + chunk) of row blockIdx.y; VEC: 16-byte aligned rows. part: [rows][splits] (value,
// index bits), or null: the row's result.
template <int VEC>
__global__ void __launch_bounds__(256) argmax_kernel(const float* __restrict__ logits, int V, int chunk, int row0,
                                                     float2* __restrict__ part, int32_t* __restrict__ idx,
                                                     float* __restrict__ val) {
  __shared__ float sv[4];
  __shared__ int si[4];
  const int row = row0 + blockIdx.y, c0 = blockIdx.x * chunk, c1 = min(c0 + chunk, V);
  const float* x = logits + (size_t)row * V;
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  constexpr int W = VEC ? 4 : 1, U = 4;
  for (int i = c0 + (int)threadIdx.x * W; i < c1; i += 256 * W * U) {
    float f[U][W];
#pragma unroll
    for (int u = 0; u < U; ++u) {  // (a group past the end loads the thread's first one again: nothing new)
      const int at = i + 256 * W * u < c1 ? i + 256 * W * u : i;
      if (VEC) {
        const float4 t = *reinterpret_cast<const float4*>(x + at);
        f[u][0] = t.x; f[u][W > 1 ? 1 : 0] = t.y; f[u][W > 2 ? 2 : 0] = t.z; f[u][W > 3 ? 3 : 0] = t.w;
      } else {
        f[u][0] = x[at];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < W; ++e)
        if (f[u][e] > bv) {  // ascending columns, strictly greater: the first index within a thread's columns
          bv = f[u][e];
          bi = i + 256 * W * u + e;
        }
  }
  am_wave(bv, bi);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) {
    sv[wid] = bv;
    si[wid] = bi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) am_better(bv, bi, sv[w], si[w]);
    if (part) {
      part[(size_t)row * gridDim.x + blockIdx.x] = make_float2(bv, __int_as_float(bi));
    } else {
      idx[row] = bi == 0x7fffffff ? 0 : bi;
      val[row] = bv;
    }
  }
}

// one wave per row over its splits (at most 64)
__global__ void __launch_bounds__(256) argmax_splits_kernel(const float2* __restrict__ part, int splits, int B,
                                                            int32_t* __restrict__ idx, float* __restrict__ val) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= B) return;
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  if (lane < splits) {
    const float2 t = part[(size_t)row * splits + lane];
    bv = t.x;
    bi = __float_as_int(t.y);
  }
  am_wave(bv, bi);
  if (lane == 0) {
    idx[row] = bi == 0x7fffffff ? 0 : bi;
    val[row] = bv;
  }
}

// workgroups per row: about 1024 in all, at most 64 and at least 2048 columns each; a row that one workgroup reads in three
// rounds does not pay for the second launch (1 | 500 rows of 5000 columns: two workgroups 5.5 | 6.8 us, one 3.6 | 4.4; 200 rows of
// 12001 columns: 6.2, 5.5)
static int argmax_splits(int B, int V) {
  if (B <= 0 || V < 12288) return 1;
  const int want = (1024 + B - 1) / B, most = V / 2048;
  return max(1, min(min(want, most), 64));
}

long long argmax_workspace(int B, int V) {
  const int splits = argmax_splits(B, V);
  return splits > 1 ? 2LL * B * splits : 0;
}

int argmax(const float* logits, int B, int V, int32_t* idx, float* val, float* ws, hipStream_t s) {
  if (B <= 0) return 0;
  const int splits = argmax_splits(B, V);
  if (splits > 1 && !ws) return -1;
  const int chunk = ((V + splits - 1) / splits + 3) / 4 * 4;
  float2* part = splits > 1 ? reinterpret_cast<float2*>(ws) : nullptr;
  const bool vec = V % 4 == 0 && ((uintptr_t)logits & 15) == 0;
  for (int r0 = 0; r0 < B; r0 += 65535) {  // (the grid's second axis)
    const dim3 grid(splits, min(B - r0, 65535));
    if (vec) argmax_kernel<1><<<grid, 256, 0, s>>>(logits, V, chunk, r0, part, idx, val);
    else argmax_kernel<0><<<grid, 256, 0, s>>>(logits, V, chunk, r0, part, idx, val);
    JLA_CHECK_LAUNCH();
  }
  if (part) {
    argmax_splits_kernel<<<(B + 3) / 4, 256, 0, s>>>(part, splits, B, idx, val);
    JLA_CHECK_LAUNCH();
  }
  return 0;
}

__global__ void decode_update_kernel(const int32_t* __restrict__ nxt, int32_t* __restrict__ finished,
                                     int32_t* __restrict__ sequences, int32_t* __restrict__ cur_len,
                                     int32_t* __restrict__ tokens, int32_t* __restrict__ positions,
                                     int32_t* __restrict__ slot, int B, int L, int pad, int eos) {
  const int cl = cur_len[0];
  for (int b = threadIdx.x; b < B; b += blockDim.x) {  // one workgroup: any batch size
    int t = nxt[b];
    const int fin = finished[b];
    if (fin) t = pad;
    finished[b] = (fin || t == eos) ? 1 : 0;
    if (cl < L)
      sequences[(size_t)b * L + cl] = t;
    else
      JLA_FLAG(JLA_BOUNDS_SEQ);
    tokens[b] = t;
    positions[b] += 1;
  }
  __syncthreads();  // every thread has read cur_len before it advances
  if (threadIdx.x == 0) {
    cur_len[0] = cl + 1;
    slot[0] += 1;
  }
}

// The greedy choice over partials [B][n] (value, index bits; argmax_kernel's, or a product's that took its maximum itself) and the
// loop's bookkeeping in one launch of one workgroup: decode_update behind a launch that reduces cost 3 us more per token. Up to 64
// partials a wave takes a row, else the workgroup does.
constexpr int AN_ROWS = 256;
__global__ void __launch_bounds__(1024) argmax_next_kernel(const float2* __restrict__ part, int n, int32_t* __restrict__ finished,
                                                           int32_t* __restrict__ sequences, int32_t* __restrict__ cur_len,
                                                           int32_t* __restrict__ tokens, int32_t* __restrict__ positions,
                                                           int32_t* __restrict__ slot, int B, int L, int pad, int eos) {
  __shared__ int nxt[AN_ROWS];
  __shared__ float sv[16];
  __shared__ int si[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int cl = cur_len[0];
  if (n <= 64) {
    for (int r0 = wave; r0 < B; r0 += 64) {
      float2 t[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int row = r0 + 16 * u;
        t[u] = row < B && lane < n ? part[(size_t)row * n + lane] : make_float2(-INFINITY, __int_as_float(0x7fffffff));
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        int bi = __float_as_int(t[u].y);
        am_wave(t[u].x, bi);
        if (lane == 0 && r0 + 16 * u < B) nxt[r0 + 16 * u] = bi == 0x7fffffff ? 0 : bi;
      }
    }
  } else {
    for (int row = 0; row < B; ++row) {
      float bv = -INFINITY;
      int bi = 0x7fffffff;
      for (int i = tid; i < n; i += 4096) {
        float2 t[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          t[u] = i + 1024 * u < n ? part[(size_t)row * n + i + 1024 * u] : make_float2(-INFINITY, __int_as_float(0x7fffffff));
#pragma unroll
        for (int u = 0; u < 4; ++u) am_better(bv, bi, t[u].x, __float_as_int(t[u].y));
      }
      am_wave(bv, bi);
      if (lane == 0) {
        sv[wave] = bv;
        si[wave] = bi;
      }
      __syncthreads();
      if (wave == 0) {
        bv = lane < 16 ? sv[lane] : -INFINITY;
        bi = lane < 16 ? si[lane] : 0x7fffffff;
        am_wave(bv, bi);
        if (lane == 0) nxt[row] = bi == 0x7fffffff ? 0 : bi;
      }
      __syncthreads();
    }
  }
  __syncthreads();
  if (tid < B) {
    int t = nxt[tid];
    const int fin = finished[tid];
    if (fin) t = pad;
    finished[tid] = (fin || t == eos) ? 1 : 0;
    if (cl < L)
      sequences[(size_t)tid * L + cl] = t;
    else
      JLA_FLAG(JLA_BOUNDS_SEQ);
    tokens[tid] = t;
    positions[tid] += 1;
  }
  if (tid == 0) {  // (every thread has read cur_len before the barriers)
    cur_len[0] = cl + 1;
    slot[0] += 1;
  }
}

int argmax_part_count(int B, int V) { return argmax_splits(B, V); }

int argmax_parts(const float* logits, int B, int V, float* part, hipStream_t s) {
  if (B <= 0 || B > AN_ROWS || !part) return -1;
  const int splits = argmax_splits(B, V), chunk = ((V + splits - 1) / splits + 3) / 4 * 4;
  const dim3 grid(splits, B);
  if (V % 4 == 0 && ((uintptr_t)logits & 15) == 0) argmax_kernel<1><<<grid, 256, 0, s>>>(logits, V, chunk, 0, reinterpret_cast<float2*>(part), nullptr, nullptr);
  else argmax_kernel<0><<<grid, 256, 0, s>>>(logits, V, chunk, 0, reinterpret_cast<float2*>(part), nullptr, nullptr);
  JLA_CHECK_LAUNCH();
  return 0;
}

int argmax_next(const float* part, int n, int32_t* finished, int32_t* sequences, int32_t* cur_len, int32_t* tokens, int32_t* positions,
                int32_t* slot, int B, int L, int pad, int eos, hipStream_t s) {
  if (B <= 0 || B > AN_ROWS || n < 1) return -1;
  argmax_next_kernel<<<1, 1024, 0, s>>>(reinterpret_cast<const float2*>(part), n, finished, sequences, cur_len, tokens, positions, slot, B,
                                        L, pad, eos);
  JLA_CHECK_LAUNCH();
  return 0;
}

int decode_update(const int32_t* nxt, int32_t* finished, int32_t* sequences, int32_t* cur_len, int32_t* tokens,
                  int32_t* positions, int32_t* slot, int B, int L, int pad, int eos, hipStream_t s) {
  if (B <= 0) return -1;
  decode_update_kernel<<<1, min(1024, ((B + 63) / 64) * 64), 0, s>>>(nxt, finished, sequences, cur_len, tokens, positions, slot,
                                                          B, L, pad, eos);
  JLA_CHECK_LAUNCH();
  return 0;
}

JLA_BOUNDS_ACCESSOR(sample)

}  // namespace jla
