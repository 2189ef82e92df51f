// Small device helpers shared by the hybrid-mixer kernels.
#pragma once
#include "../kernels/common.h"

namespace jla {

// 8 consecutive elements of a row (zero beyond the `n` valid ones) as floats; 16-byte loads where aligned
JLA_DEV void hy_load8(const float* p, int n, float* f) {
  if (n >= 8 && ((uintptr_t)p & 15) == 0) {
    const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
    f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w; f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = i < n ? p[i] : 0.f;
  }
}
JLA_DEV void hy_load8(const bf16_t* p, int n, float* f) {
  if (n >= 8 && ((uintptr_t)p & 15) == 0) {
    unpack8(*reinterpret_cast<const u32x4*>(p), f);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = i < n ? bf2f(p[i]) : 0.f;
  }
}

JLA_DEV float hy_silu(float x) { return x / (1.f + expf(-x)); }
JLA_DEV float hy_sigmoid(float x) { return 1.f / (1.f + expf(-x)); }
JLA_DEV float hy_gelu_tanh(float z) {
  return 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}
JLA_DEV float hy_logsigmoid(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }
JLA_DEV float hy_softplus(float x) { return x > 20.f ? x : log1pf(expf(x)); }

// Heads of up to 4 L numbers in groups of L lanes, four neighbouring numbers per lane: the sum of squares of the group's head
template <int L>
JLA_DEV float hy_head_squares(const f32x4 v) {
  float ss = fmaf(v[0], v[0], v[1] * v[1]) + fmaf(v[2], v[2], v[3] * v[3]);
#pragma unroll
  for (int o = L / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
  return ss;
}
// ... whether heads of n numbers run in such groups, and L (0: they do not)
inline int hy_head_lanes(int n) { return n % 4 || n > 256 ? 0 : (n <= 64 ? 16 : (n <= 128 ? 32 : 64)); }
JLA_DEV void hy_store1(float* p, float v) { *p = v; }
JLA_DEV void hy_store1(bf16_t* p, float v) { *p = f2bf(v); }
JLA_DEV void hy_store4(float* p, const f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }
JLA_DEV void hy_store4(bf16_t* p, const f32x4 v) { *reinterpret_cast<u32x2*>(p) = u32x2{pack2bf(v[0], v[1]), pack2bf(v[2], v[3])}; }

}  // namespace jla
