// The epilogue of a row linear (RowAct), shared by its kernels.
#pragma once
#include "hy_util.h"
#include "hybrid.h"

namespace jla {

JLA_DEV void lr_out(float* p, float v) { *p = v; }
JLA_DEV void lr_out(bf16_t* p, float v) { *p = f2bf(v); }

JLA_DEV float lr_clamp_glu(const RowLinear& p, float g, float u) {
  const float gc = fminf(g, p.act_limit), uc = fminf(fmaxf(u, -p.act_limit), p.act_limit);
  return gc * hy_sigmoid(p.act_alpha * gc) * (uc + 1.f);
}
// the epilogue of one output element: g the (gate) accumulator, u the up accumulator of the gated forms
JLA_DEV float lr_act(const RowLinear& p, float g, float u) {
  switch (p.act) {
    case HY_ACT_RELU2: {
      const float r = fmaxf(g, 0.f);
      return r * r;
    }
    case HY_ACT_SWIGLU:
      return hy_silu(g) * u;
    case HY_ACT_CLAMP_GLU:
      return lr_clamp_glu(p, g, u);
    case HY_ACT_SOFTCAP:
      return p.act_limit * tanhf(g / p.act_limit);
    case HY_ACT_GELU_GLU:
      return hy_gelu_tanh(g) * u;
    default:
      return g;
  }
}
JLA_DEV float lr_in(const float* p) { return *p; }
JLA_DEV float lr_in(const bf16_t* p) { return bf2f(*p); }

}  // namespace jla
