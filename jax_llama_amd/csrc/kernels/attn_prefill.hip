// Prefill (multi-query) attention over the KV cache: flash-style online softmax on MFMA.
//
// Reference semantics: model.py:236-291 (causal mask sliced at cache_index, AND padding mask,
// additive finfo.min bias, softmax in fp32, P.V), without ever materialising the (S x T) score
// matrix or the (L x L) causal mask (model.py:154). Query s of row b sits at cache slot slot0 + s
// and attends keys j with kv_start[b] <= j <= slot0 + s (and key_mask[b, j] if given). A query
// with no valid key (a left-pad position) outputs 0, never NaN.
//
// Workgroup = (64-query block, q head, batch row), 4 waves x 16 query rows. Per 32-key tile:
//   K tile [32 x 128] and V^T tile [128 x 32] are staged in LDS (V transposed on the way in so the
//   P.V B operand is a contiguous ds_read_b128); padded rows make every fragment read
//   bank-conflict free;
//   S = Q K^T: 2 key sub-tiles x 4 d-steps of v_mfma_f32_16x16x32_bf16 (Q fragments live in VGPRs);
//   online softmax on the accumulator layout (row stats reduced over 16 lanes);
//   P goes through a small per-wave LDS tile to become the A operand; O += P V: 8 MFMAs.
#include <type_traits>

#include "common.h"
#include "launchers.h"

namespace jla {

constexpr int AP_DH = 128;
constexpr int AP_QB = 64;             // queries per workgroup
constexpr int AP_KT = 32;             // keys per tile
constexpr int AP_KROW = AP_DH + 8;    // K tile row (bf16 elements): 272 B
constexpr int AP_VROW = AP_KT + 8;    // V^T tile row: 80 B
constexpr int AP_PROW = AP_KT + 8;    // P tile row: 80 B

__global__ void __launch_bounds__(256)
    attn_prefill_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc, const bf16_t* __restrict__ vc,
                        const int32_t* __restrict__ slot_ptr, const int32_t* __restrict__ kv_start,
                        const uint8_t* __restrict__ key_mask, int mask_len, bf16_t* __restrict__ out, int S, int H,
                        int Hkv, int T, float scale) {
  __shared__ __attribute__((aligned(16))) bf16_t Kt[AP_KT * AP_KROW];
  __shared__ __attribute__((aligned(16))) bf16_t Vt[AP_DH * AP_VROW];
  __shared__ __attribute__((aligned(16))) bf16_t Pt[4][16 * AP_PROW];

  const int qb = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int g = lane >> 4, li = lane & 15;
  const int rep = H / Hkv, kvh = h / rep;
  const int slot0 = slot_ptr[0];
  if (slot0 + S > T && threadIdx.x == 0) JLA_FLAG(JLA_BOUNDS_ATTN_T);
  const int lo = kv_start[b];
  const uint8_t* mrow = key_mask ? key_mask + (size_t)b * mask_len : nullptr;

  // Q fragments (A operand): row li of this wave's 16 queries, d = 32*kk + 8*g
  const int qrow_a = min(qb * AP_QB + w * 16 + li, S - 1);
  u32x4 qa[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk)
    qa[kk] = *reinterpret_cast<const u32x4*>(q + (((size_t)b * S + qrow_a) * H + h) * AP_DH + 32 * kk + 8 * g);

  // this lane's 4 accumulator rows
  int qslot[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) qslot[i] = slot0 + qb * AP_QB + w * 16 + 4 * g + i;

  f32x4 o[8];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float mrun[4], lrun[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    mrun[i] = -INFINITY;
    lrun[i] = 0.f;
  }

  const int last_key = min(slot0 + min(S, (qb + 1) * AP_QB) - 1, T - 1);
  const int t_begin = (lo / AP_KT) * AP_KT;
  const bf16_t* kb = kc + ((size_t)b * Hkv + kvh) * T * AP_DH;
  const bf16_t* vb = vc + ((size_t)b * Hkv + kvh) * T * AP_DH;

  for (int t0 = t_begin; t0 <= last_key; t0 += AP_KT) {
    // ---- stage K (row-major) and V (transposed); 512 x 16 B per tile each, 2 per thread
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int idx = tid + r * 256;  // 0..511
      const int key = idx >> 4, d0 = (idx & 15) * 8;
      const int j = min(t0 + key, T - 1);
      const u32x4 kv = *reinterpret_cast<const u32x4*>(kb + (size_t)j * AP_DH + d0);
      const u32x4 vv = *reinterpret_cast<const u32x4*>(vb + (size_t)j * AP_DH + d0);
      *reinterpret_cast<u32x4*>(&Kt[key * AP_KROW + d0]) = kv;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        Vt[(d0 + 2 * e) * AP_VROW + key] = (bf16_t)(vv[e] & 0xffffu);
        Vt[(d0 + 2 * e + 1) * AP_VROW + key] = (bf16_t)(vv[e] >> 16);
      }
    }
    __syncthreads();

    // ---- S = Q K^T for two 16-key sub-tiles
    f32x4 s[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      s[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const u32x4 kf = *reinterpret_cast<const u32x4*>(&Kt[(n * 16 + li) * AP_KROW + 32 * kk + 8 * g]);
        s[n] = mfma16x16x32(qa[kk], kf, s[n]);
      }
    }
    // ---- mask + online softmax (row i of this lane = query 4g+i; column = key n*16+li)
    float p[2][4];
    float alpha[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float mt = -INFINITY;
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        const int j = t0 + n * 16 + li;
        bool valid = j <= qslot[i] && j >= lo && j < T;
        if (mrow && j < mask_len) valid = valid && mrow[j] != 0;
        const float v = valid ? s[n][i] * scale : -INFINITY;
        p[n][i] = v;
        mt = fmaxf(mt, v);
      }
      mt = fmaxf(mt, __shfl_xor(mt, 1, 64));
      mt = fmaxf(mt, __shfl_xor(mt, 2, 64));
      mt = fmaxf(mt, __shfl_xor(mt, 4, 64));
      mt = fmaxf(mt, __shfl_xor(mt, 8, 64));
      const float mn = fmaxf(mrun[i], mt);
      float rs = 0.f;
      if (mn == -INFINITY) {
        alpha[i] = 1.f;
        p[0][i] = 0.f;
        p[1][i] = 0.f;
      } else {
        alpha[i] = __expf(mrun[i] - mn);
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          p[n][i] = (p[n][i] == -INFINITY) ? 0.f : __expf(p[n][i] - mn);
          rs += p[n][i];
        }
      }
      rs += __shfl_xor(rs, 1, 64);
      rs += __shfl_xor(rs, 2, 64);
      rs += __shfl_xor(rs, 4, 64);
      rs += __shfl_xor(rs, 8, 64);
      lrun[i] = lrun[i] * alpha[i] + rs;
      mrun[i] = mn;
    }
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[dt][i] *= alpha[i];

    // ---- P (C layout) -> LDS -> A operand
    bf16_t* pw = Pt[w];
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int i = 0; i < 4; ++i) pw[(4 * g + i) * AP_PROW + n * 16 + li] = f2bf(p[n][i]);
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's P writes landed
    __builtin_amdgcn_wave_barrier();
    const u32x4 pa = *reinterpret_cast<const u32x4*>(&pw[li * AP_PROW + 8 * g]);
    // ---- O += P V
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      const u32x4 vf = *reinterpret_cast<const u32x4*>(&Vt[(dt * 16 + li) * AP_VROW + 8 * g]);
      o[dt] = mfma16x16x32(pa, vf, o[dt]);
    }
  }

  // ---- epilogue: out[b*S + q][h*Dh + d]
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int qr = qb * AP_QB + w * 16 + 4 * g + i;
    if (qr >= S) continue;
    const float inv = lrun[i] > 0.f ? 1.f / lrun[i] : 0.f;
    bf16_t* dst = out + ((size_t)b * S + qr) * H * AP_DH + (size_t)h * AP_DH;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) dst[dt * 16 + li] = f2bf(o[dt][i] * inv);
  }
}

// ================================================================================================
// v2: GQA-shared flash prefill on v_mfma_f32_32x32x16_bf16.
//
// Workgroup = NW waves = (batch row b, kv head, group of q heads, block of query positions); every wave
// owns 32 query rows of ONE q head, and all NW waves read the SAME K/V tiles from LDS, so a (b, kv head)
// K/V tile is fetched once per rep/hpw workgroups instead of once per q head (rep = H / Hkv).
// Per 64-key tile and wave:
//   S^T = K Q^T   (A = K fragment by ds_read_b128 from an XOR-swizzled image, B = Q^T fragments held in
//                  VGPRs for the whole kernel): 2 key blocks x 8 dk-steps = 16 MFMAs. The C layout puts the
//                  wave's query on the LANE (col = lane & 31) and 32 of the 64 keys in its registers, so the
//                  online softmax is lane-local plus one exchange with lane ^ 32;
//   O^T += V^T P^T (A = V^T by ds_read_b64_tr_b16 transposed reads of the row-major V image, B = the bf16 P
//                  registers used in place with the permuted k order of the accumulator layout): 4 d tiles x
//                  4 key steps = 16 MFMAs. O^T again has the query on the lane, so the rescale by
//                  exp2(m_old - m_new) is lane-local too.
// K/V tiles come by LDS-DMA into two slots each (64 KiB per workgroup): K(i+1) and V(i) are there during tile i while
// K(i+2) and V(i+1) go into the slots that tile i-1 was done with, so a tile ends with ONE wait and barrier. The DMA is
// inline asm: with the builtin, hipcc waits for the DMA of the next tiles before the first V read of a tile.
// Causal: the workgroup stops at its last query's slot; a wave whose queries all precede a tile skips its MFMAs; only
// tiles that cross the diagonal, kv_start or T are masked element-wise. Each workgroup runs a heavy and a light query
// block (causal balance).
constexpr int FA_KT = 64;  // keys per tile

// byte offset of 16-byte chunk ch (0..15) of row `row` in a [rows][128 bf16] image whose XOR swizzle
// serves both ds_read_b128 row reads and ds_read_b64_tr_b16 transposed reads without bank conflicts
JLA_DEV int fa_off(int row, int ch) { return 256 * row + 16 * (ch ^ (((row & 3) << 2) | ((row >> 2) & 3))); }

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

JLA_DEV f32x16 mfma32(const u32x4 a, const u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                 0, 0, 0);
}
JLA_DEV u32x2 ld_tr(const char* lds, int off) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                       (__attribute__((address_space(3))) s16x4*)(lds + off)));
}

// One query block of 32 per wave (a 64-query "QB = 2" form halved the LDS bytes per MFMA but needed ~340 registers,
// one workgroup per CU, and ran 1.4-2x slower: profiles/r2_attn_prefill_qb2_ab.jsonl -- removed).
//
// What bounds it: the matrix pipe (1024 cycles a tile and wave) and the VALU (about 900: 32 exp at a quarter of the
// rate, fma, sum, pack, max) of a wave take turns unless the code puts independent work of both next to each other: two
// waves per SIMD in step with each other don't. So all of a tile is in the fixed order of `tile`: an MFMA, then one
// element's exp of the NEXT key step, then an LDS read, ten times a key step (sched_group_barrier); the scores of tile
// i+1 are spread over key steps 0..2 of tile i, its max stands beside the PV MFMAs of key step 3, and only the P of its
// first key step has no MFMA beside it. The max exchange of the two lane halves is a permlane32 swap, the halves of the
// sum meet once at the end, two tiles are unrolled (constant LDS slots, no scores moved), and the masks take a lane's
// two limits instead of 32 key indexes held in registers.
// Measured (32 heads, 8 kv heads of 128, causal): S = 8192 604 -> 496 us (1.1 PFLOP/s), 16 x 2048 735 -> 649 us,
// S = 2048 62.5 -> 50.7, S = 600 with 32 kv heads 26.3 -> 20.0, 2048 x 128 1411 -> 1325 us.
// Lazy rescale (every launch): the running max (and with it the O / l rescale) moves only when a lane's tile max
// exceeds it by more than 8 (log2 units): exp2 of the rest stays <= 256, exact in fp32 and bf16-representable for P;
// the 64 O multiplies per tile run only in a wave-uniform branch when some lane needs them (mostly the first tiles).
template <int NW>
__global__ void __launch_bounds__(NW * 64, 2)
    attn_prefill_v2_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc, const bf16_t* __restrict__ vc,
                           const int32_t* __restrict__ slot_ptr, const int32_t* __restrict__ kv_start,
                           const uint8_t* __restrict__ key_mask, int mask_len, bf16_t* __restrict__ out, int S, int H,
                           int Hkv, int T, float scale_log2, int npb, int hgroups, int n_qb, int split) {
  constexpr int TILE_BYTES = FA_KT * AP_DH * 2;            // 16 KiB
  constexpr int QW = 32;                                    // queries per wave
  __shared__ __attribute__((aligned(16))) char lds[4 * TILE_BYTES];

  // split = 1 (small grids): the heavy and the light block of a pair are two workgroups of a 1-D grid, all heavy
  // ones first -- ids g and g + items are the same pair, so when the second round of dispatch lands on the CUs in
  // the order of the first, every CU again holds one (heavy, light) pair, now as two resident workgroups
  int bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z, pass_lo = 0, pass_hi = 2;
  if (split) {
    const int P = (n_qb + 1) / 2, Y = Hkv * hgroups;  // 1-D grid of 2 x P x Y x B workgroups
    const int items = (int)gridDim.x / 2;
    int g = blockIdx.x;
    const bool light = g >= items;
    if (light) g -= items;
    bx = g % P;
    by = (g / P) % Y;
    bz = g / (P * Y);
    pass_lo = light ? 1 : 0;
    pass_hi = light ? 2 : 1;
  }
  const int kvh = by / hgroups, hg = by - kvh * hgroups;
  const int b = bz;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hi = lane >> 5, col = lane & 31;
  const int rep = H / Hkv, hpw = NW / npb;
  const int r = w / npb, pb = w - r * npb;
  const int h = kvh * rep + hg * hpw + r;
  // causal balance: workgroup x runs query block n_qb-1-x (heavy) and then block x (light), so every
  // workgroup streams ~the same number of K/V tiles (with one block per workgroup, S = 2048 at B = 1 ran
  // the heaviest workgroup ~2x longer than the average one)
  for (int pass = pass_lo; pass < pass_hi; ++pass) {
  const int qb = pass == 0 ? n_qb - 1 - bx : bx;
  if (pass == 1 && qb >= n_qb - 1 - bx) break;  // odd n_qb: the middle block runs once
  if (pass == 1) __syncthreads();  // every wave is done with the LDS images of the first block
  const int p0 = qb * QW * npb + QW * pb;   // first query position of this wave
  const int slot0 = slot_ptr[0];
  if (slot0 + S > T && threadIdx.x == 0) JLA_FLAG(JLA_BOUNDS_ATTN_T);
  const int lo = kv_start[b];
  const uint8_t* mrow = key_mask ? key_mask + (size_t)b * mask_len : nullptr;

  // Q^T fragments (B operand): lane holds Q[p0 + col][16 ks + 8 hi .. +7]
  u32x4 qf[8];
  const bf16_t* qrow = q + (((size_t)b * S + min(p0 + col, S - 1)) * H + h) * AP_DH + 8 * hi;
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) qf[ks] = *reinterpret_cast<const u32x4*>(qrow + 16 * ks);
  f32x16 o[4];
  float m_run = -INFINITY, l_run = 0.f;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;

  const int wg_last_pos = min(S, (qb + 1) * QW * npb) - 1;
  const int last_key = min(slot0 + wg_last_pos, T - 1);
  const int t_begin = (lo / FA_KT) * FA_KT;
  // (a wave behind the last query only helps to stage: 1000 rows of 33 queries, 32 kv heads, 404 -> 364 us)
  const int wave_last_slot = p0 < S ? slot0 + min(p0 + QW - 1, S - 1) : -1;
  const bf16_t* kb = kc + ((size_t)b * Hkv + kvh) * T * AP_DH;
  const bf16_t* vb = vc + ((size_t)b * Hkv + kvh) * T * AP_DH;

  // per-lane LDS read offsets: K row reads (key block kb, dk step ks -> chunk 2 ks + hi)
  // V transposed reads: 16-lane group G = lane >> 4 covers d columns 16 (G & 1) .. +15 of a 32-wide d tile,
  // lane 4q + p of the group addresses row q of the 4-key block, columns 4p .. 4p + 3.
  const int gq = (lane & 15) >> 2, gp = lane & 3, G = lane >> 4;
  // LDS-DMA staging (no VGPRs held across the tile): wave w fills 1-KiB blocks w, w + NW, ... of a tile
  // image; lane L of block bi writes row 4 bi + L / 16, slot L % 16, so it fetches the source chunk that
  // fa_off's swizzle puts in that slot
  auto Kr = [&](int i) { return lds + i * TILE_BYTES; };
  auto Vr = [&](int i) { return lds + (2 + i) * TILE_BYTES; };
  auto dma = [&](const bf16_t* src, int t0, char* dst) {
#pragma unroll
    for (int i = 0; i < 16 / NW; ++i) {
      const int bi = w + NW * i, row = 4 * bi + (lane >> 4);
      const int ch = (lane & 15) ^ (((row & 3) << 2) | ((row >> 2) & 3));
      // (ch is the same for every i: 4 NW i rows leave the swizzle as it is)
      glds16_asm(src + (size_t)t0 * AP_DH, 256 * min(row, T - 1 - t0) + 16 * ch, dst + 1024 * bi);
    }
  };
  auto scores = [&](const char* Kt, f32x16 (&s)[2]) {
#pragma unroll
    for (int kbk = 0; kbk < 2; ++kbk) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[kbk][i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < 8; ++ks)
        s[kbk] = mfma32(*reinterpret_cast<const u32x4*>(Kt + fa_off(32 * kbk + col, 2 * ks + hi)), qf[ks], s[kbk]);
    }
  };
  const int n_t = t_begin <= last_key ? (last_key - t_begin) / FA_KT + 1 : 0;
  const int qfirst = slot0 + p0, qslot = qfirst + col;
  f32x16 st[2];
  if (n_t > 0) {
    dma(kb, t_begin, Kr(0));
    dma(vb, t_begin, Vr(0));
  }
  if (n_t > 1) dma(kb, t_begin + FA_KT, Kr(1));
  wait_vmcnt<0>();
  __syncthreads();
  if (n_t > 0 && t_begin <= wave_last_slot) scores(Kr(0), st);
  // the first iteration's DMA of K(2) lands in K(0)'s slot: every wave must be done reading it
  if (n_t > 2) __syncthreads();
  // a lane's LDS offsets, of which the rest of fa_off is constants: K row read (dk step ks: ^ 32 ks; key block: + 8192),
  // V transposed read (d tile dt: ^ 64 dt; keys + 8: ^ 32, + 2048; key step s: + 4096 s)
  const int k_off = fa_off(col, hi), v_off = fa_off(4 * (G >> 1) + gq, 2 * (G & 1) + (gp >> 1)) + 8 * (gp & 1);
  f32x16 st2[2];
  float m_use = 0.f, rs = 0.f;
  u32x4 pf = {0, 0, 0, 0};
  // P of key step s: 8 of a lane's 32 scores
  auto probs = [&](const f32x16 (&s2)[2], int s) {
    float e[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      e[j] = __builtin_amdgcn_exp2f(fmaf(s2[s >> 1][8 * (s & 1) + j], scale_log2, -m_use));
      rs += e[j];
    }
    return pack8(e);
  };
  auto largest = [&](const f32x16 (&s2)[2]) {
    float m = -INFINITY;
#pragma unroll
    for (int kbk = 0; kbk < 2; ++kbk)
#pragma unroll
      for (int i = 0; i < 16; ++i) m = fmaxf(m, s2[kbk][i]);
    return m;
  };
  // what a tile needs before its PV: masks (wave-uniform branch: only tiles crossing kv_start, the diagonal, T, or a
  // key mask), the running max, P of its first key step; raw: the lane's largest score before masks
  auto enter = [&](int t0, f32x16 (&s2)[2], float raw) {
    const bool full = !mrow && t0 >= lo && t0 + FA_KT - 1 <= qfirst && t0 + FA_KT - 1 < T;
    if (!full) {
      int first = t0 + 4 * hi;  // (opaque: or the keys of a lane's 32 scores are kept in registers over the loop)
      asm volatile("" : "+v"(first));
      const int from = lo - first, upto = min(min(qslot, T - 1), mrow ? mask_len - 1 : T) - first;
#pragma unroll
      for (int kbk = 0; kbk < 2; ++kbk)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int j = 32 * kbk + (i & 3) + 8 * (i >> 2);
          s2[kbk][i] = j >= from && j <= upto ? s2[kbk][i] : -INFINITY;
        }
      if (mrow && mask_len > 0) {
#pragma unroll
        for (int kbk = 0; kbk < 2; ++kbk)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int j = 32 * kbk + (i & 3) + 8 * (i >> 2);
            s2[kbk][i] = mrow[min(first + j, mask_len - 1)] ? s2[kbk][i] : -INFINITY;
          }
      }
      raw = largest(s2);
    }
    const float tmax = lane_max32(raw) * scale_log2;  // scale > 0: max of the scaled scores
    if (__ballot(tmax > m_run + 8.f)) {
      const float m_new = fmaxf(m_run, tmax);
      const float alpha = __builtin_amdgcn_exp2f(m_run - (m_new == -INFINITY ? 0.f : m_new));
      l_run *= alpha;
      m_run = m_new;
      m_use = m_new == -INFINITY ? 0.f : m_new;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
    }
    rs = 0.f;
    pf = probs(s2, 0);
  };
  // tile it of parity cur (a constant: an LDS address is a lane's own and an immediate, and no scores move): key
  // step s has the PV MFMAs of P(s), a share of the next tile's scores and, on the VALU beside them, P(s + 1)
  auto tile = [&](int it, auto parity, f32x16 (&s2)[2], f32x16 (&sn)[2]) {
    constexpr int cur = decltype(parity)::value;
    const int t0 = t_begin + it * FA_KT;
    const bool has1 = it + 1 < n_t, has2 = it + 2 < n_t;
    // K(i+2) into K(i)'s slot and V(i+1) into V(i-1)'s: both last read before the previous barrier
    if (has2) dma(kb, t0 + 2 * FA_KT, Kr(cur));
    if (has1) dma(vb, t0 + FA_KT, Vr(cur ^ 1));
    if (t0 <= wave_last_slot) {  // wave-uniform; every later tile is inactive too
      auto score = [&](int f) {
        sn[f & 1] = mfma32(*reinterpret_cast<const u32x4*>(Kr(cur ^ 1) + (k_off ^ (32 * (f >> 1))) + 8192 * (f & 1)),
                           qf[f >> 1], sn[f & 1]);
      };
      auto pv = [&](int s, int dt) {
        const u32x2 lo4 = ld_tr(Vr(cur), (v_off ^ (64 * dt)) + 4096 * s);
        const u32x2 hi4 = ld_tr(Vr(cur), (v_off ^ (64 * dt) ^ 32) + 2048 + 4096 * s);
        const u32x4 vf = {lo4[0], lo4[1], hi4[0], hi4[1]};
        o[dt] = mfma32(vf, pf, o[dt]);
      };
#pragma unroll
      for (int i = 0; i < 16; ++i) sn[0][i] = sn[1][i] = 0.f;
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int f = 6 * s; f < (s < 2 ? 6 * s + 6 : 16); ++f) score(f);
        const u32x4 next = probs(s2, s + 1);
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) pv(s, dt);
        pf = next;
        __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
        for (int i = 0; i < (s < 2 ? 10 : 8); ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
          __builtin_amdgcn_sched_group_barrier(0x400, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }

      }
      __builtin_amdgcn_sched_barrier(0);
      l_run += rs;  // (this half's keys; the halves meet at the end)
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) pv(3, dt);
      const float raw = largest(sn);
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }

      __builtin_amdgcn_sched_barrier(0);
      if (has1 && t0 + FA_KT <= wave_last_slot) enter(t0 + FA_KT, sn, raw);
    }
    wait_vmcnt<0>();
    __syncthreads();
  };
  if (n_t > 0 && t_begin <= wave_last_slot) enter(t_begin, st, largest(st));
  for (int it = 0; it < n_t; it += 2) {
    tile(it, std::integral_constant<int, 0>{}, st, st2);
    if (it + 1 < n_t) tile(it + 1, std::integral_constant<int, 1>{}, st2, st);
  }
  l_run = lane_sum32(l_run);

  // ---- epilogue: lane (query pos, half hi) holds d = 32 dt + 8 g + 4 hi + (0..3) in o[dt][4 g .. 4 g + 3]
  const int pos = p0 + col;
  if (pos < S) {
    const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
    bf16_t* dst = out + ((size_t)b * S + pos) * H * AP_DH + (size_t)h * AP_DH + 4 * hi;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        u32x2 pk;
        pk[0] = pack2bf(o[dt][4 * g] * inv, o[dt][4 * g + 1] * inv);
        pk[1] = pack2bf(o[dt][4 * g + 2] * inv, o[dt][4 * g + 3] * inv);
        *reinterpret_cast<u32x2*>(dst + 32 * dt + 8 * g) = pk;
      }
  }
  }  // pass
}

// v2 launch with NW waves per workgroup: NW / rep position blocks (rep < NW) or NW of the rep q heads (rep >= NW) share
// each K/V tile the workgroup stages
template <int NW>
static void launch_prefill_v2(const bf16_t* q, const bf16_t* kc, const bf16_t* vc, const int32_t* slot,
                              const int32_t* kv_start, const uint8_t* key_mask, int mask_len, bf16_t* out, int B, int S,
                              int H, int Hkv, int T, int rep, hipStream_t s) {
  const int npb = rep >= NW ? 1 : NW / rep;    // position blocks per workgroup
  const int hpw = NW / npb;                    // q heads per workgroup
  const int hgroups = rep / hpw;
  const float sl2 = 1.4426950408889634f / sqrtf((float)AP_DH);
  const int n_qb = (S + 32 * npb - 1) / (32 * npb);
  const int pairs = (n_qb + 1) / 2 * Hkv * hgroups * B;
  // fewer pairs than two workgroups per CU (B = 1 prefill): each half of a pair is its own workgroup, so a CU
  // holds two resident workgroups instead of one (of 4 waves: of 8, a CU holds one)
  const bool split = NW == 4 && pairs < 2 * 256;
  if (split) {
    attn_prefill_v2_kernel<NW><<<dim3(2 * pairs, 1, 1), NW * 64, 0, s>>>(
        q, kc, vc, slot, kv_start, key_mask, mask_len, out, S, H, Hkv, T, sl2, npb, hgroups, n_qb, 1);
  } else {
    dim3 grid2((n_qb + 1) / 2, Hkv * hgroups, B);  // a (heavy, light) pair of query blocks per workgroup
    attn_prefill_v2_kernel<NW><<<grid2, NW * 64, 0, s>>>(q, kc, vc, slot, kv_start, key_mask, mask_len, out, S,
                                                                H, Hkv, T, sl2, npb, hgroups, n_qb, 0);
  }
}

// impl (attn_prefill_set_impl, A/B): 2 = default dispatch; 7 = 4 waves per workgroup, 13 = 8 waves; 1 = the v1 kernel (also the
// fallback for a non-power-of-two GQA ratio)
static int g_attn_prefill_impl = 2;
void attn_prefill_set_impl(int impl) { g_attn_prefill_impl = impl; }

int attn_prefill(const bf16_t* q, const bf16_t* kc, const bf16_t* vc, const int32_t* slot, const int32_t* kv_start,
                 const uint8_t* key_mask, int mask_len, bf16_t* out, int B, int S, int H, int Hkv, int Dh, int T,
                 hipStream_t s) {
  if (B <= 0 || S <= 0) return 0;
  if (Dh != AP_DH || H % Hkv) return -1;
  const int rep = H / Hkv;
  const bool pow2rep = rep == 1 || rep == 2 || rep == 4 || rep == 8;
  int impl = g_attn_prefill_impl;
  // default (impl 2): 8 waves per workgroup (twice the queries per staged K / V tile, one workgroup resident per CU)
  // where the prompt is long, the paired grid's rounds over the 256 CUs are nearly full (a last round of >= 90 %; with
  // one round, >= 75 %) and so are the workgroups' query rows (>= 73 % of what the rounds have room for: an odd number of query blocks leaves
  // half a pair, the last block may be nearly empty), else 4 waves. Measured, 4 -> 8 waves, us: S = 4096 143 -> 133 (one full round), 2 x 4096
  // 279 -> 265 (two), S = 3000 103 -> 89 (192 workgroups), 124 -> 107 (240); but S = 4096 226 -> 250 (320), 4 x 1500 101 -> 111 (384),
  // S = 1500 39 -> 53 (96); of 32 kv heads 2 x 1025 39 -> 54 (192, rows 50 %), 2 x 1300 57 -> 60 (192, 63 %), 16 x 1100 293 -> 326 (1536, 72 %),
  // of 40 4 x 1200 118 -> 110 (480, 73 %), of 32 2 x 1531 67 -> 63 (192, 75 %); at S <= 1024 4 waves are ahead nearly everywhere (16 x 512 76 -> 79, 64 x 128 60 -> 83): a query
  // block is then twice as many rows for the same few tiles.
  if (impl == 2 && pow2rep) {
    const int npb8 = rep >= 8 ? 1 : 8 / rep;
    const int n_qb8 = (S + 32 * npb8 - 1) / (32 * npb8);
    const long long wg8 = (long long)((n_qb8 + 1) / 2) * Hkv * (rep / (8 / npb8)) * B;
    const long long rounds = (wg8 + 255) / 256;
    const long long rows = (long long)S * Hkv * (rep / (8 / npb8)) * B;  // a workgroup takes 64 npb8
    impl = S > 1024 && (10 * wg8 >= 9 * 256 * rounds || (rounds == 1 && wg8 >= 192)) && 100 * rows >= 73LL * 256 * rounds * 64 * npb8 ? 13 : 7;
  }
  const int nw = impl == 7 ? 4 : impl == 13 ? 8 : 0;
  if (nw && (rep % nw == 0 || nw % rep == 0)) {
    if (nw == 4)
      launch_prefill_v2<4>(q, kc, vc, slot, kv_start, key_mask, mask_len, out, B, S, H, Hkv, T, rep, s);
    else
      launch_prefill_v2<8>(q, kc, vc, slot, kv_start, key_mask, mask_len, out, B, S, H, Hkv, T, rep, s);
    JLA_CHECK_LAUNCH();
    return 0;
  }
  dim3 grid((S + AP_QB - 1) / AP_QB, H, B);
  attn_prefill_kernel<<<grid, 256, 0, s>>>(q, kc, vc, slot, kv_start, key_mask, mask_len, out, S, H, Hkv, T,
                                           1.f / sqrtf((float)Dh));
  JLA_CHECK_LAUNCH();
  return 0;
}

JLA_BOUNDS_ACCESSOR(attn_prefill)

}  // namespace jla
