// What the quantized matvec (gemv.hip) and matrix product (gemm.hip) kernels
// share: launch arguments, code unpacking, the epilogues, and the product
// kernel's launcher.
#pragma once

#include "common.h"
#include "paged_common.h"

namespace mkq {

constexpr int EPI_NONE = 0;
constexpr int EPI_RESIDUAL = 1;
constexpr int EPI_GATE_UP = 2;
constexpr int EPI_ROPE_KV = 3;  // qkv rows -> split + interleaved RoPE + paged K/V write

template <int BITS>
struct QFmt {
  static constexpr int KL = BITS == 4 ? 64 : 32;     // k per lane chunk (32 code bytes)
  static constexpr int KC = 4 * KL;                  // k per wave chunk
  static constexpr int STEPS = BITS == 4 ? 8 : 4;    // MFMA k32 steps per chunk
  static constexpr int ROW_BYTES_NUM = BITS;         // row bytes = K * BITS / 8
};

// --------------------------------------------------------------------------
// activation operand: 8 halves of x for one MFMA step, in the k order the
// weight unpack produces.
// --------------------------------------------------------------------------
template <int BITS, bool MAGIC>
__device__ __forceinline__ u32x4 xperm(u32x4 X) {
  if constexpr (!MAGIC) {
    return X;  // natural order
  } else if constexpr (BITS == 4) {
    // weight order [0,4,1,5,2,6,3,7]
    u32x4 r;
    r[0] = pack_lo16(X[0], X[2]);
    r[1] = pack_hi16(X[0], X[2]);
    r[2] = pack_lo16(X[1], X[3]);
    r[3] = pack_hi16(X[1], X[3]);
    return r;
  } else {
    // weight order [0,2,1,3,4,6,5,7]
    u32x4 r;
    r[0] = pack_lo16(X[0], X[1]);
    r[1] = pack_hi16(X[0], X[1]);
    r[2] = pack_lo16(X[2], X[3]);
    r[3] = pack_hi16(X[2], X[3]);
    return r;
  }
}

// Per-group dequant parameters.  The integer part zi of the zero point is
// subtracted exactly from the magic-biased codes: (1024 + c) - (1024 + zi)
// for codes at mantissa bits 0..3 (q8: 0..7) of 1024.0h, (64 + c) - (64 + zi)
// for q4 codes left in place at bits 4..7 under 64.0h (ulp 1/16) -- c - zi
// exactly in fp16 for |zi| < 1024 -- so w = fma(c - zi, s, corr) with
// corr = -(z - zi) s rounds once, to the fp16 of (c - z) s whenever z is an
// integer (the rounding of the reference's fp32 dequant, for any fp16 scale),
// and keeps a fractional z exact to ulp(corr).  (Zero points past 1024 lose bits
// of 1024 + zi; the layouts of gemv_generic_kernel never come here.)
struct GpMagic {
  f16x2 s;     // (s, s)
  f16x2 kz;    // (1024 + zi)
  f16x2 kz64;  // (64 + zi)
  f16x2 corr;  // -(z - zi) * s
};
struct GpExact {
  float s;
  float z;
};

__device__ __forceinline__ f16x2 h2(f16 v) { return (f16x2){v, v}; }

__device__ __forceinline__ GpMagic make_gp_magic(f16 s, f16 z) {
  GpMagic g;
  const float zf = (float)z;
  const float zi = rintf(zf);
  g.s = h2(s);
  g.kz = h2((f16)(1024.0f + zi));
  g.kz64 = h2((f16)(64.0f + zi));
  g.corr = h2((f16)(-(zf - zi) * (float)s));
  return g;
}

// q4 word (8 codes) -> 8 fp16 weights in order [0,4,1,5,2,6,3,7].
// `magic` = 0x64006400 (1024.0h pair) and `magic_hi` = 0x54005400 (64.0h
// pair) held in VGPRs so each unpack is one v_and_or_b32.
__device__ __forceinline__ u32x4 dq4_magic(uint32_t u, const GpMagic& g, uint32_t magic, uint32_t magic_hi) {
  const uint32_t v = u >> 8;
  f16x2 a = bitcast<f16x2>((u & 0x000F000Fu) | magic) - g.kz;       // c0 - zi, c4 - zi
  f16x2 b = bitcast<f16x2>((u & 0x00F000F0u) | magic_hi) - g.kz64;  // c1 - zi, c5 - zi
  f16x2 c = bitcast<f16x2>((v & 0x000F000Fu) | magic) - g.kz;       // c2, c6
  f16x2 d = bitcast<f16x2>((v & 0x00F000F0u) | magic_hi) - g.kz64;  // c3, c7
  a = __builtin_elementwise_fma(a, g.s, g.corr);
  b = __builtin_elementwise_fma(b, g.s, g.corr);
  c = __builtin_elementwise_fma(c, g.s, g.corr);
  d = __builtin_elementwise_fma(d, g.s, g.corr);
  u32x4 r;
  r[0] = bitcast<uint32_t>(a);
  r[1] = bitcast<uint32_t>(b);
  r[2] = bitcast<uint32_t>(c);
  r[3] = bitcast<uint32_t>(d);
  return r;
}

// byte-pair unpack of q8 codes with v_perm_b32: bytes (b0, 0x64, b2, 0x64)
// and (b1, 0x64, b3, 0x64) of {magic8 = 0x64646464, u} are 1024+b0 / 1024+b2
// and 1024+b1 / 1024+b3 as fp16 pairs.
__device__ __forceinline__ uint32_t q8_lo_pair(uint32_t u, uint32_t magic8) {
  return perm_b32(magic8, u, 0x04020400u);
}
__device__ __forceinline__ uint32_t q8_hi_pair(uint32_t u, uint32_t magic8) {
  return perm_b32(magic8, u, 0x04030401u);
}

// two q8 words (8 codes) -> 8 fp16 weights in order [0,2,1,3,4,6,5,7].
__device__ __forceinline__ u32x4 dq8_magic(uint32_t u0, uint32_t u1, const GpMagic& g,
                                           uint32_t magic8) {
  f16x2 a0 = bitcast<f16x2>(q8_lo_pair(u0, magic8)) - g.kz;
  f16x2 b0 = bitcast<f16x2>(q8_hi_pair(u0, magic8)) - g.kz;
  f16x2 a1 = bitcast<f16x2>(q8_lo_pair(u1, magic8)) - g.kz;
  f16x2 b1 = bitcast<f16x2>(q8_hi_pair(u1, magic8)) - g.kz;
  a0 = __builtin_elementwise_fma(a0, g.s, g.corr);
  b0 = __builtin_elementwise_fma(b0, g.s, g.corr);
  a1 = __builtin_elementwise_fma(a1, g.s, g.corr);
  b1 = __builtin_elementwise_fma(b1, g.s, g.corr);
  u32x4 r;
  r[0] = bitcast<uint32_t>(a0);
  r[1] = bitcast<uint32_t>(b0);
  r[2] = bitcast<uint32_t>(a1);
  r[3] = bitcast<uint32_t>(b1);
  return r;
}

// Exact path: w = AT((q - z) * s) computed in fp32, natural k order.
template <typename AT>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  AT a = from_f32<AT>(lo), b = from_f32<AT>(hi);
  return (uint32_t)bitcast<uint16_t>(a) | ((uint32_t)bitcast<uint16_t>(b) << 16);
}

template <typename AT>
__device__ __forceinline__ u32x4 dq4_exact(uint32_t u, const GpExact& g) {
  float w[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) w[e] = ((float)((u >> (4 * e)) & 15u) - g.z) * g.s;
  u32x4 r;
#pragma unroll
  for (int p = 0; p < 4; ++p) r[p] = pack2<AT>(w[2 * p], w[2 * p + 1]);
  return r;
}

template <typename AT>
__device__ __forceinline__ u32x4 dq8_exact(uint32_t u0, uint32_t u1, const GpExact& g) {
  float w[8];
#pragma unroll
  for (int e = 0; e < 4; ++e) w[e] = ((float)((u0 >> (8 * e)) & 255u) - g.z) * g.s;
#pragma unroll
  for (int e = 0; e < 4; ++e) w[4 + e] = ((float)((u1 >> (8 * e)) & 255u) - g.z) * g.s;
  u32x4 r;
#pragma unroll
  for (int p = 0; p < 4; ++p) r[p] = pack2<AT>(w[2 * p], w[2 * p + 1]);
  return r;
}

template <typename AT>
__device__ __forceinline__ f32x4 mfma_k32(u32x4 a, u32x4 b, f32x4 c);

template <>
__device__ __forceinline__ f32x4 mfma_k32<f16>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(bitcast<f16x8>(a), bitcast<f16x8>(b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4 mfma_k32<bf16>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(bitcast<bf16x8>(a), bitcast<bf16x8>(b), c, 0, 0,
                                                 0);
}

// The decode token's cache write fused into the qkv projection's epilogue
// (EPI_ROPE_KV): the operands of qkv_rope_update_kernel.
struct RopeKV {
  const float* cos_t;   // [cos_rows, D/2]
  const float* sin_t;
  const int32_t* pos;   // [M]
  const int32_t* bt;    // [M, max_blocks]
  void* kp;             // [num_pages, P, Hkv, D] f16
  void* vp;
  void* q_out;          // [M, Hq, D] f16
  int Hq, Hkv, D, P, max_blocks, num_pages, cos_rows;
};

struct GemvArgs {
  const void* x;         // [M, K]
  const uint8_t* w[2];   // [N, row_bytes]
  const void* s[2];      // [N, G]
  const void* z[2];      // [N, G] or null, each by itself
  const void* residual;  // [M, N] or null
  void* y0;              // EPI_NONE: y; EPI_RESIDUAL: y_mm (nullable); GATE_UP: gate (nullable)
  void* y1;              // EPI_RESIDUAL: out;  GATE_UP: up (nullable)
  void* y2;              // GATE_UP: mlp (nullable)
  int M, N, K;
  int row_bytes;
  int G;
  int lg;                // log2(group size)
  int kw;                // waves per row group (K split)
  int rg;                // dot kernel: row groups per workgroup
  // residual + RMSNorm prologue (NORM dot kernels, M = 1): the product is
  // taken against n = fp16(z * rsqrt(mean(z^2) + eps) * nw), z = fp16(x +
  // nres) (z = x when nres is null); workgroup 0 writes z and n when zout /
  // nout are given
  const void* nres;      // [K] or null
  const void* nw;        // [K] fp16
  void* zout;            // [K]
  void* nout;            // [K] or null
  float eps;
  RopeKV rk;             // EPI_ROPE_KV only
};

// Both matrices of a pair have zero points, or neither: what every kernel but
// gemv_mfma_kernel and gemv_generic_kernel takes for granted (they test z[0]
// and read both).
template <int NMAT>
inline bool zeros_alike(const GemvArgs& a) {
  return NMAT == 1 || (a.z[0] == nullptr) == (a.z[1] == nullptr);
}

// --------------------------------------------------------------------------
// shared epilogue: value(s) of output row n for activation row m
// --------------------------------------------------------------------------
template <typename AT, int EPI>
__device__ __forceinline__ void store_out(const GemvArgs& args, size_t o, float v0, float v1) {
  if constexpr (EPI == EPI_NONE) {
    reinterpret_cast<AT*>(args.y0)[o] = saturate_cast<AT>(v0);
  } else if constexpr (EPI == EPI_RESIDUAL) {
    const AT d = saturate_cast<AT>(v0);
    if (args.y0) reinterpret_cast<AT*>(args.y0)[o] = d;
    const float r = to_f32(reinterpret_cast<const AT*>(args.residual)[o]);
    reinterpret_cast<AT*>(args.y1)[o] = from_f32<AT>(r + to_f32(d));
  } else {
    const AT g = saturate_cast<AT>(v0);
    const AT u = saturate_cast<AT>(v1);
    if (args.y0) reinterpret_cast<AT*>(args.y0)[o] = g;
    if (args.y1) reinterpret_cast<AT*>(args.y1)[o] = u;
    if (args.y2) {
      const float gf = to_f32(g);
      const float sil = gf / (1.0f + expf(-gf));
      reinterpret_cast<AT*>(args.y2)[o] = from_f32<AT>(sil * to_f32(u));
    }
  }
}

// EPI_ROPE_KV: the launch's rows' cache slots (page * P + offset, -1 when
// skipped), looked up once per workgroup before its reduction barrier, so the
// later-row-wins rule reads LDS in the epilogue (rows <= 32 per launch).
constexpr int kRopeRows = 32;
__device__ __forceinline__ void rope_fill_slots(const GemvArgs& a, int* slots) {
  const int t = threadIdx.x;
  if (t < a.M && t < kRopeRows) {
    const RopeKV& r = a.rk;
    int off;
    const int pg = slot_page(r.bt, r.pos, t, r.max_blocks, r.P, r.num_pages, &off);
    slots[t] = pg < 0 ? -1 : pg * r.P + off;
  }
}
// this row's slot, or -1 when skipped or taken by a later row of the launch
__device__ __forceinline__ int rope_slot(const GemvArgs& a, const int* slots, int m) {
  const int sl = slots[m];
  if (sl < 0) return -1;
  for (int b2 = m + 1; b2 < a.M; ++b2)
    if (slots[b2] == sl) return -1;
  return sl;
}

// EPI_ROPE_KV: qkv output n of row m, rounded as the projection stores it,
// then the arithmetic of qkv_rope_update_kernel -- q and k pairs (n, n ^ 1)
// rotated in fp32 and rounded, v copied; q to q_out, k and v to the token's
// cache slot unless its position is out of range or a later row takes the
// slot.  Called by every lane of the pair (the partner value comes by
// shuffle), whether or not (m, n) is in range.
__device__ __forceinline__ void rope_kv_store(const GemvArgs& a, const int* slots, int m, int n, float v) {
  const f16 hv = saturate_cast<f16>(v);
  const float xv = to_f32(hv);
  const float xo = __shfl_xor(xv, 1, 64);
  if (n >= a.N || m >= a.M) return;
  const RopeKV& r = a.rk;
  const int p = r.pos[m];
  if (p < 0 || p >= r.cos_rows) return;
  const int D = r.D, QD = r.Hq * D, KD = r.Hkv * D;
  const int d = n % D;
  f16 out = hv;
  f16* dst = reinterpret_cast<f16*>(r.vp);
  int h;
  if (n < QD + KD) {
    const bool even = (d & 1) == 0;
    const size_t ci = (size_t)p * (D / 2) + (d >> 1);
    float ye, yo;
    rope_pair(even ? xv : xo, even ? xo : xv, r.cos_t[ci], r.sin_t[ci], &ye, &yo);
    out = from_f32<f16>(even ? ye : yo);
    if (n < QD) {
      reinterpret_cast<f16*>(r.q_out)[(size_t)m * QD + n] = out;
      return;
    }
    dst = reinterpret_cast<f16*>(r.kp);
    h = (n - QD) / D;
  } else {
    h = (n - QD - KD) / D;
  }
  const int sl = rope_slot(a, slots, m);
  if (sl < 0) return;
  dst[(size_t)sl * KD + (size_t)h * D + d] = out;
}

// EPI_ROPE_KV with both values of an (even n, n + 1) pair in one lane (the
// MFMA kernels' output layout): the same arithmetic as rope_kv_store.  RES:
// slots[m] already holds the row's final slot (-1 when skipped or taken by a
// later row) and pos_l[m] its position, both in LDS.
template <bool RES = false>
__device__ __forceinline__ void rope_kv_pair(const GemvArgs& a, const int* slots, int m, int n, float v0,
                                             float v1, const int* pos_l = nullptr) {
  if (n >= a.N || m >= a.M) return;
  const RopeKV& r = a.rk;
  const int p = RES ? pos_l[m] : r.pos[m];
  if (p < 0 || p >= r.cos_rows) return;
  const int D = r.D, QD = r.Hq * D, KD = r.Hkv * D;
  const int d = n % D;
  const f16 h0 = saturate_cast<f16>(v0), h1 = saturate_cast<f16>(v1);
  f16 o0 = h0, o1 = h1;
  f16* dst = reinterpret_cast<f16*>(r.vp);
  int h;
  if (n < QD + KD) {
    const size_t ci = (size_t)p * (D / 2) + (d >> 1);
    float ye, yo;
    rope_pair(to_f32(h0), to_f32(h1), r.cos_t[ci], r.sin_t[ci], &ye, &yo);
    o0 = from_f32<f16>(ye);
    o1 = from_f32<f16>(yo);
    if (n < QD) {
      f16* q = reinterpret_cast<f16*>(r.q_out) + (size_t)m * QD + n;
      q[0] = o0;
      q[1] = o1;
      return;
    }
    dst = reinterpret_cast<f16*>(r.kp);
    h = (n - QD) / D;
  } else {
    h = (n - QD - KD) / D;
  }
  const int sl = RES ? slots[m] : rope_slot(a, slots, m);
  if (sl < 0) return;
  f16* o = dst + (size_t)sl * KD + (size_t)h * D + d;
  o[0] = o0;
  o[1] = o1;
}

// The rows' final slots (the later-row-wins rule applied) and positions into
// LDS: call after rope_fill_slots(a, raw) and a barrier; the values are
// visible after the next barrier.
__device__ __forceinline__ void rope_resolve_slots(const GemvArgs& a, const int* raw, int* res, int* pos_l) {
  const int t = threadIdx.x;
  if (t < a.M && t < kRopeRows) {
    int sl = raw[t];
    for (int b2 = t + 1; b2 < a.M; ++b2)
      if (raw[b2] == sl) sl = -1;
    res[t] = sl;
    pos_l[t] = a.rk.pos[t];
  }
}

// (q - z) * s of 8 codes rounded to AT, in natural k order.  fp16 scales and
// zero points: z * s is exact in fp32, so fma(q, s, -(z * s)) is the product
// of the exact difference rounded once; fp32 ones subtract first.  The fp16
// form has no conversion: a code's bits are the fp16 subnormal q 2^-24 (a
// nibble at bit 4, q 2^-20), which v_fma_mix_f32 reads as they lie, against
// s 2^24 (s 2^20): 17 instructions for 8 q4 codes where conversions of bytes
// take 23 (q8: 16 and 20).  bf16 activations, us: MLP block of 4096 and 14336 at
// 4 rows 50.2 -> 44.7, 28672 x 4096 at 32 rows 33.8 -> 29.7, 14336 x 4096 at 512
// rows 114 -> 105 (q8 113 -> 107).
template <typename ST>
struct ExactGp {
  float s, z;  // fp16: s 2^24 and -(z s); fp32: s and z
};
template <typename ST>
__device__ __forceinline__ ExactGp<ST> make_exact_gp(ST s, ST z) {
  if constexpr (sizeof(ST) == 2) return {(float)s * 0x1p24f, -((float)z * (float)s)};
  else return {s, z};
}
template <int BITS, typename AT, typename ST>
__device__ __forceinline__ u32x4 dq_exact8(uint32_t u0, uint32_t u1, const ExactGp<ST>& g) {
  float c[8];
  if constexpr (sizeof(ST) == 2) {
    const float s4 = g.s * 0x1p-4f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      // q4: codes e and e + 4; q8: codes 2 e and 2 e + 1
      const uint32_t h = BITS == 4   ? (e & 2 ? u0 >> 8 : u0) & (e & 1 ? 0x00F000F0u : 0x000F000Fu)
                         : e & 1 ? perm_b32(0u, e & 2 ? u1 : u0, 0x0C030C02u)
                                 : perm_b32(0u, e & 2 ? u1 : u0, 0x0C010C00u);
      const f16x2 v = bitcast<f16x2>(h);
      const float sc = BITS == 4 && (e & 1) ? s4 : g.s;
      c[BITS == 4 ? e : 2 * e] = fmaf((float)v[0], sc, g.z);
      c[BITS == 4 ? e + 4 : 2 * e + 1] = fmaf((float)v[1], sc, g.z);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t q = BITS == 4 ? (u0 >> (4 * e)) & 15u : ((e & 4 ? u1 : u0) >> (8 * (e & 3))) & 255u;
      c[e] = ((float)q - g.z) * g.s;
    }
  }
  u32x4 r;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    // (as a vector: v_fma_mixlo and v_fma_mixhi write the pair, 13 instructions)
    if constexpr (__is_same(AT, f16)) r[p] = bitcast<uint32_t>((f16x2){(f16)c[2 * p], (f16)c[2 * p + 1]});
    else r[p] = pack2<AT>(c[2 * p], c[2 * p + 1]);
  }
  return r;
}

// Epilogue of output rows nb .. nb + 3 (nb a multiple of 4) for activation
// row m; `vec`: whole 8-byte stores apply.  One kernel serves the plain and
// the residual product (EPI_RESIDUAL; the tests are uniform).
template <typename AT, int EPI>
__device__ __forceinline__ void store_out4(const GemvArgs& args, bool vec, int m, int nb, f32x4 v0, f32x4 v1) {
  const size_t o = (size_t)m * args.N + nb;
  if (!vec) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (nb + i >= args.N) continue;
      if (EPI == EPI_RESIDUAL && !args.residual) store_out<AT, EPI_NONE>(args, o + i, v0[i], v1[i]);
      else store_out<AT, EPI>(args, o + i, v0[i], v1[i]);
    }
    return;
  }
  if (nb >= args.N) return;
  typedef AT at4 __attribute__((ext_vector_type(4)));
  at4 a, b, c;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a[i] = saturate_cast<AT>(v0[i]);
    b[i] = saturate_cast<AT>(v1[i]);
  }
  if constexpr (EPI == EPI_RESIDUAL) {
    if (args.y0) *reinterpret_cast<at4*>(reinterpret_cast<AT*>(args.y0) + o) = a;
    if (!args.residual) return;
    const at4 r = *reinterpret_cast<const at4*>(reinterpret_cast<const AT*>(args.residual) + o);
#pragma unroll
    for (int i = 0; i < 4; ++i) c[i] = from_f32<AT>(to_f32((AT)r[i]) + to_f32((AT)a[i]));
    *reinterpret_cast<at4*>(reinterpret_cast<AT*>(args.y1) + o) = c;
  } else {
    if (args.y0) *reinterpret_cast<at4*>(reinterpret_cast<AT*>(args.y0) + o) = a;
    if (args.y1) *reinterpret_cast<at4*>(reinterpret_cast<AT*>(args.y1) + o) = b;
    if (args.y2) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float gf = to_f32((AT)a[i]);
        c[i] = from_f32<AT>(gf / (1.0f + expf(-gf)) * to_f32((AT)b[i]));
      }
      *reinterpret_cast<at4*>(reinterpret_cast<AT*>(args.y2) + o) = c;
    }
  }
}

// CUs of the current device, cached per device.
inline int device_cu_count() {
  static int cache[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cache[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cache[dev] = n;
  }
  return cache[dev];
}

// The product of many activation rows (gemm.hip), one launch for all a.M rows
// of what gemm_rows_ok accepts (EPI_RESIDUAL without a residual: the plain
// product into y0).
template <int BITS, int NMAT>
bool gemm_rows_ok(const GemvArgs& a, int64_t M, int64_t gs);
float gemm_rows_us(int bits, int nmat, int M, int N, int K);  // estimated time of that launch
template <int BITS, int NMAT, int EPI>
int launch_gemm_rows(const GemvArgs& a, int act_dt, int sc_dt, hipStream_t st);

// The few-row matvec (gemv_few.hip), a.M <= 32 rows (8-bit codes: 16) of what
// few_ok accepts, with few_workspace_bytes of workspace (0 unless K > 4096 is cut
// into slices; EPI_ROPE_KV and EPI_GATE_UP need it 0, so their K ends at 4096).
size_t few_workspace_bytes(int64_t M, int64_t N, int64_t K);
template <int BITS, int NMAT>
bool few_ok(const GemvArgs& a, int64_t M, int64_t gs, int sc_dt, size_t ws_bytes);
template <int BITS, int NMAT, int EPI>
int launch_few(const GemvArgs& a, int act_dt, float* ws, hipStream_t st);

}  // namespace mkq
