// What the attention kernels over a per-layer cache share: which keys a query sees, how a decode step deals them to its splits,
// and how an output column is gated and stored.
#pragma once
#include "hy_util.h"
#include "hybrid.h"

namespace jla {

// The keys a query at slot qi sees: slots [0, kf) (kept first keys, only beside a window) and [lo, qi], numbered
// 0 .. n - 1 in that order.
struct AbSpan {
  int kf, lo, n;
};
JLA_DEV AbSpan ab_span(const AttnBias& p, int qi) {
  AbSpan sp;
  sp.lo = p.chunk > 0 ? qi / p.chunk * p.chunk : (p.window > 0 ? max(0, qi - p.window + 1) : 0);
  sp.kf = p.window > 0 ? min(p.keep_first, sp.lo) : 0;
  sp.n = sp.kf + qi + 1 - sp.lo;
  return sp;
}
// query head vh = map vh % maps of output head vh / maps: its key / value head, and its keys' offset within a key row
struct AbMap {
  int g, koff;
};
JLA_DEV AbMap ab_map(const AttnBias& p, int vh) {
  const int h = vh / p.maps;
  return {h / (p.H / p.G), (vh - h * p.maps) * p.dim};
}
JLA_DEV int ab_key(const AbSpan& sp, int v) { return v < sp.kf ? v : sp.lo + (v - sp.kf); }
// gate of column c of head h: one per head, or one per column
JLA_DEV float ab_gate(const AttnBias& p, size_t m, int h, int c) {
  return p.gate ? hy_sigmoid(p.gate[m * p.ldg + (p.gate_cols ? h * p.vdim + c : h)]) : 1.f;
}
JLA_DEV void ab_out(const AttnBias& p, size_t m, int h, int c, float v) {
  const size_t at = m * p.ldo + (size_t)h * p.vdim + c;
  if (p.out_bf16) reinterpret_cast<bf16_t*>(p.out)[at] = f2bf(v);
  else reinterpret_cast<float*>(p.out)[at] = v;
}

// visible keys number [j_lo, j_hi) of decode split sp: the query's n visible keys dealt to the splits in runs of 64
JLA_DEV void ab_split_range(const AttnBias& p, const AbSpan& span, int sp, int& j_lo, int& j_hi) {
  const int n = span.n;
  const int per = ((n + p.splits - 1) / p.splits + 63) / 64 * 64;
  j_lo = min(n, sp * per);
  j_hi = min(n, j_lo + per);
}

}  // namespace jla
