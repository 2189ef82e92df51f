// The epilogues of a tiled product, for four consecutive columns of one row.
#pragma once
#include "common.h"
#include "launchers.h"

namespace jla {

// v: columns col .. col + 3 of row m, the norm's row scale applied (two RoPE pairs; a 16-column tile never straddles them).
// SwiGLU: v is of a gate tile, the even one of a pair of 16-column tiles, u the same columns of the up tile behind it.
template <int MODE>
JLA_DEV void gemm_out4(const float (&v)[4], const float (&u)[4], int m, int col, int N, void* out, int accumulate, int out_f32,
                       bf16_t* mirror, const QKVArgs& qa) {
  const size_t idx = (size_t)m * N + col;
  if constexpr (MODE == MODE_SWIGLU) {
    const int tile = col >> 4, c0 = col & 15;
    bf16_t* o = static_cast<bf16_t*>(out) + (size_t)m * (N >> 1) + (tile >> 1) * 16 + c0;
    const uint2 pk = make_uint2(pack2bf(silu(v[0]) * u[0], silu(v[1]) * u[1]), pack2bf(silu(v[2]) * u[2], silu(v[3]) * u[3]));
    *reinterpret_cast<uint2*>(o) = pk;
    // decode M: also the packed copy (common.h pack_off) the next projection's packed-x GEMV reads
    if (qa.pack) *reinterpret_cast<uint2*>(qa.pack + pack_off(m, (tile >> 1) * 16 + c0, N >> 1)) = pk;
  } else if constexpr (MODE == MODE_RESIDUAL) {
    float4* o = reinterpret_cast<float4*>(static_cast<float*>(out) + idx);
    float4 r = make_float4(v[0], v[1], v[2], v[3]);
    if (accumulate) {
      const float4 h = *o;
      r = make_float4(h.x + v[0], h.y + v[1], h.z + v[2], h.w + v[3]);
    }
    *o = r;
    if (mirror) {
      const uint2 pk = make_uint2(pack2bf(r.x, r.y), pack2bf(r.z, r.w));
      *reinterpret_cast<uint2*>(mirror + idx) = pk;
      if (qa.pack) *reinterpret_cast<uint2*>(qa.pack + pack_off(m, col, N)) = pk;  // packed copy of the mirror
    }
  } else if constexpr (MODE == MODE_QKV) {
    const int head = col / qa.Dh, d0 = col - head * qa.Dh;
    const int b = m / qa.S, sq = m - b * qa.S;
    float r[4] = {v[0], v[1], v[2], v[3]};
    if (head < qa.H + qa.Hkv) {
      int pos = qa.positions[m];
      if (pos < 0 || pos >= qa.table_len) JLA_FLAG(JLA_BOUNDS_ROPE_POS);
      pos = pos < 0 ? 0 : (pos >= qa.table_len ? qa.table_len - 1 : pos);
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const float2 cs = qa.table[(size_t)pos * (qa.Dh >> 1) + (d0 >> 1) + p];
        const float xr = v[2 * p], xi = v[2 * p + 1];
        r[2 * p] = xr * cs.x - xi * cs.y;
        r[2 * p + 1] = xr * cs.y + xi * cs.x;
      }
    }
    const uint2 packed = make_uint2(pack2bf(r[0], r[1]), pack2bf(r[2], r[3]));
    if (head < qa.H) {
      *reinterpret_cast<uint2*>(qa.q + ((size_t)m * qa.H + head) * qa.Dh + d0) = packed;
    } else {
      const int slot = qa.slot[0] + sq;
      if (slot < qa.T) {
        const bool is_k = head < qa.H + qa.Hkv;
        const int kh = is_k ? head - qa.H : head - qa.H - qa.Hkv;
        bf16_t* cache = is_k ? qa.kc : qa.vc;
        *reinterpret_cast<uint2*>(cache + (((size_t)b * qa.Hkv + kh) * qa.T + slot) * qa.Dh + d0) = packed;
      } else {
        JLA_FLAG(JLA_BOUNDS_KV_SLOT);
      }
    }
  } else {
    if (out_f32)
      *reinterpret_cast<float4*>(static_cast<float*>(out) + idx) = make_float4(v[0], v[1], v[2], v[3]);
    else
      *reinterpret_cast<uint2*>(static_cast<bf16_t*>(out) + idx) = make_uint2(pack2bf(v[0], v[1]), pack2bf(v[2], v[3]));
  }
}

}  // namespace jla
