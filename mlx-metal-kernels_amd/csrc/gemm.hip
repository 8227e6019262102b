// Quantized matrix product for many activation rows (a prompt's rows through
// an MLP block, the rows of a speculative verify pass):
//   y[m,n] = clip(sum_k x[m,k] * W[n,k], +-max(act)),  W = (q - z) * s rounded
//   to the activation type (ops/quant_ops.py:509-526, 574-588, 634-738),
// with the epilogues of the matvec kernels (SwiGLU of gate and up, residual).
//
// The decode kernels walk the weights once per 32 rows; from there on a
// product is bound by the matrix cores, and the question is what feeds them.
// A wave owns 64 weight rows (32 of each matrix for gate/up) against MT * 16
// activation rows, so an unpacked weight operand serves MT products (16 VALU
// instructions for 8 codes against MT * 16 matrix cycles: 64 of 128 at MT =
// 8) and never passes LDS; with 64 weight rows per wave the activation
// operands, read from LDS, take 64 bytes per cycle and CU, half of what it
// delivers.  Unpacked weights in LDS would take twice that.
//
// Codes, activations and scales come to LDS by global_load_lds, 64 k per
// stage in a ring of two or three: no registers hold data in flight (loads
// through registers left either one stage in flight, 2.7 us a turn instead
// of 1.8, or spilled), and the only waits are one vmcnt and one barrier per
// stage.  A turn's unpacking and operand reads are interleaved with its
// products in chunks of two column tiles (152 -> 149 us below).
//
// A workgroup is WN groups of weight rows by WK slices of K, whose
// accumulators are added in LDS at the end: where few output rows meet a long
// K (the down projection: 64 waves' worth of weight rows by 4 of activation
// rows, for 256 CUs), the K slices fill the chip.
//
// Measured, q4 g64 fp16, us (passes of 32 rows before -> now): 509 rows
// 2 x 14336 x 4096 + SwiGLU 428 -> 131 (915 TFLOP/s; as first built 141, 125
// without the copies, 115 without the unpacking) and 4096 x 14336 537 -> 95 (630;
// as first built 100, 67 without the copies); 128 rows 109 -> 52 and 135 -> 67; 64
// rows 57 -> 35.  bf16 128 x 6144 x 4096 120 -> 26; q8 bf16 g32 300 x 32000 x 4096
// 1225 -> 162.
#include "common.h"
#include "gemv_common.h"

using namespace mkq;

namespace {

constexpr int GK = 64;   // k per stage
constexpr int GNT = 4;   // 16-row weight tiles per wave

// Global memory to LDS without passing registers: lane l of the wave writes
// SIZE bytes at l * max(SIZE, 4) past the (wave-uniform) LDS address.  The
// compiler neither counts nor waits for these copies: stage_wait does.
template <int SIZE>
__device__ __forceinline__ void lds_copy(const void* g, void* l) {
  static_assert(SIZE == 2 || SIZE == 4 || SIZE == 16, "sizes the copy instruction has");
  const auto* gp = (const __attribute__((address_space(1))) void*)g;
  auto* lp = (__attribute__((address_space(3))) void*)l;
  if constexpr (SIZE == 16) __builtin_amdgcn_global_load_lds(gp, lp, 16, 0, 0);
  else if constexpr (SIZE == 4) __builtin_amdgcn_global_load_lds(gp, lp, 4, 0, 0);
  else __builtin_amdgcn_global_load_lds(gp, lp, 2, 0, 0);
}

// This wave's copies but the N youngest have landed and its LDS reads are
// done; then the workgroup's barrier.
template <int N>
__device__ __forceinline__ void stage_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt holds 6 bits");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// q4 word (8 codes) -> 8 fp16 weights in natural k order, so that the
// activations go to LDS as they are: byte p of the word twice (v_perm), its
// low nibble under 1024.0h in the low half (1024 + c), its high nibble in
// place under 64.0h in the high half (64 + c); then the subtraction and fma of
// dq4_magic.  `magic` = 0x54006400 in a VGPR.
struct GpNat {
  f16x2 kz;    // (1024 + zi, 64 + zi); q8: (1024 + zi) twice
  f16x2 s;
  f16x2 corr;  // -(z - zi) * s
};
template <int BITS>
__device__ __forceinline__ GpNat make_gp_nat(f16 s, f16 z) {
  const float zf = (float)z;
  const float zi = rintf(zf);
  GpNat g;
  g.kz = (f16x2){(f16)(1024.0f + zi), (f16)((BITS == 4 ? 64.0f : 1024.0f) + zi)};
  g.s = h2(s);
  g.corr = h2((f16)(-(zf - zi) * (float)s));
  return g;
}
template <int BITS>
__device__ __forceinline__ u32x4 dq_nat8(uint32_t u0, uint32_t u1, const GpNat& g, uint32_t magic) {
  u32x4 r;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    uint32_t t;
    if constexpr (BITS == 4) {
      // bytes (p, 0, p, 0): selector 0x0C is the constant 0
      t = (perm_b32(0u, u0, 0x0C000C00u + 0x00010001u * p) & 0x00F0000Fu) | magic;
    } else {
      const uint32_t u = p < 2 ? u0 : u1;
      t = perm_b32(magic, u, (p & 1) ? 0x04030402u : 0x04010400u);  // (b, 0x64, b + 1, 0x64)
    }
    const f16x2 d = bitcast<f16x2>(t) - g.kz;
    r[p] = bitcast<uint32_t>(__builtin_elementwise_fma(d, g.s, g.corr));
  }
  return r;
}

// LDS: the ring's stages -- a K slice's activations, a wave's codes and, with
// SZ8 off, its scales and zero points as a dword each per row and half stage --
// then, with SZ8 on, every wave's two buffers of 8 groups' scales and zero
// points
constexpr int gemm_x_bytes(int mt) { return mt * 16 * GK * 2; }
constexpr int gemm_code_bytes(int bits) { return 16 * GNT * GK * bits / 8; }
constexpr int gemm_sz_bytes(bool sz8) { return sz8 ? 0 : 4 * 16 * GNT * 4; }
constexpr int gemm_slot_bytes(int bits, int mt, int wn, int wk, bool sz8) {
  return wk * gemm_x_bytes(mt) + wk * wn * (gemm_code_bytes(bits) + gemm_sz_bytes(sz8));
}
// the whole is reused for the K slices' accumulators at the end
constexpr size_t gemm_lds_bytes(int bits, int mt, int wn, int wk, bool sz8, int ring) {
  const size_t stages = (size_t)ring * gemm_slot_bytes(bits, mt, wn, wk, sz8) + (sz8 ? wn * wk * 4096 : 0);
  const size_t sums = (size_t)wn * mt * (wk - 1) * GNT * 64 * sizeof(f32x4);
  return stages > sums ? stages : sums;
}

// SZ8: fp16 scales and zero points in rows of whole 16-byte vectors (G % 8 ==
// 0) are copied 8 groups at a time.  Otherwise each stage copies every row's
// two (a group of 32 spans half a stage) by themselves: 64 separate lines per
// copy instruction where the codes touch 32 and the activations 8.
//
// MAGIC: fp16 weights by the exponent trick, which holds a fractional zero
// point's part in fp16; otherwise (q - z) * s in fp32, rounded once.
template <int BITS, typename AT, typename ST, int NMAT, int EPI, bool SZ8, bool MAGIC, int MT, int WN, int WK, int RING>
__global__ __launch_bounds__(64 * WN * WK) __attribute__((amdgpu_waves_per_eu(2))) void gemm_rows_kernel(
    const GemvArgs args) {
  static_assert(!SZ8 || sizeof(ST) == 2, "SZ8 copies 8 fp16 values");
  static_assert(!MAGIC || (sizeof(ST) == 2 && __is_same(AT, f16)), "MAGIC unpacks to fp16 with fp16 scales");
  constexpr int XC = MT * 16 * (GK / 8) / (64 * WN);    // 16-byte activation chunks copied per thread and stage
  constexpr int WC = gemm_code_bytes(BITS) / (64 * 16); // 16-byte code copies per thread and stage
  constexpr int COPIES = XC + WC + (SZ8 ? 0 : 4);       // copies per wave and stage (SZ8: 2 more now and then)
  constexpr int CB = GK * BITS / 8;                     // code bytes per row and stage
  typedef uint32_t codes_t __attribute__((ext_vector_type(BITS == 4 ? 2 : 4)));  // a lane's 16 k

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % WN, kg = wave / WN;
  const int M = args.M, N = args.N, K = args.K, G = args.G;
  const int r = lane & 15, kb = lane >> 4;

  // tiles of activation rows are the inner index of one XCD's sequence
  // (workgroups are dealt out to the 8 XCDs in turn), so the workgroups that
  // read the same codes run on one XCD, close together
  const int mtiles = args.rg;
  const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
  const int tm = seq % mtiles;
  const int tn = (seq / mtiles) * 8 + xcd;
  constexpr int ROWS = 16 * GNT / NMAT;  // output rows of a wave
  if (tn * WN * ROWS >= N) return;       // the whole workgroup: past the last tile
  const int n0 = (tn * WN + wn) * ROWS;
  const int m0 = tm * 16 * MT;

  extern __shared__ __align__(16) uint8_t gemm_lds[];
  constexpr int SLOT = gemm_slot_bytes(BITS, MT, WN, WK, SZ8);
  uint8_t* const xlds = gemm_lds + kg * gemm_x_bytes(MT);
  uint8_t* const wlds = gemm_lds + WK * gemm_x_bytes(MT) + wave * (gemm_code_bytes(BITS) + gemm_sz_bytes(SZ8));
  uint8_t* const szlds = gemm_lds + RING * SLOT + wave * 4096;  // SZ8: [chunk & 1][s|z][row][8 groups]

  // this wave's K slice, in stages of 64 k: every slice takes `per` turns
  // (the barriers), `mine` of them with work
  const int stages = (K + GK - 1) / GK;
  const int per = (stages + WK - 1) / WK;
  const int st0 = kg * per;
  const int mine = min(per, stages - st0);

  // A wave's 64 weight rows in LDS: row i is row i % 16 of tile i / 16, tile t
  // being 16-row block t / NMAT of matrix t % NMAT.  Rows past N read row
  // N - 1 and are not stored.  Byte offsets fit 32 bits (dispatcher).
  auto weight_row = [&](int i, int* q) {
    const int t = i >> 4;
    *q = t % NMAT;
    return (uint32_t)min(n0 + (t / NMAT) * 16 + (i & 15), N - 1);
  };
  constexpr int LPR = CB / 16;  // lanes per row in a code copy
  const uint8_t* wsrc[WC];
#pragma unroll
  for (int j = 0; j < WC; ++j) {
    int q;
    const uint32_t n = weight_row((64 * j + lane) / LPR, &q);
    wsrc[j] = (q ? args.w[NMAT - 1] : args.w[0]) + (size_t)(n * (uint32_t)args.row_bytes);
  }
  const int wk16 = lane % LPR;  // which 16 code bytes of the row's CB
  const bool has_z = args.z[0] != nullptr;
  const ST *ssrc, *zsrc;
  {
    int q;
    const uint32_t n = weight_row(lane, &q);
    ssrc = reinterpret_cast<const ST*>(q ? args.s[NMAT - 1] : args.s[0]) + (size_t)(n * (uint32_t)G);
    zsrc = has_z ? reinterpret_cast<const ST*>(q ? args.z[NMAT - 1] : args.z[0]) + (size_t)(n * (uint32_t)G) : ssrc;
  }
  // activation chunks: LDS position p = 64 * WN * i + tl holds chunk
  // (p % 8) ^ (row & 7) of row p / 8 (16-byte chunks rotated by the row, so
  // that the 16 rows of an operand read fall into different banks); a
  // thread's rows are 8 * WN apart and share one rotation.  Rows past M read
  // row M - 1 and are not stored.
  const int tl = tid - kg * 64 * WN;
  const int xk = 8 * ((tl & 7) ^ ((tl >> 3) & 7));  // k of its chunks within a stage
  const AT* xsrc[XC];
#pragma unroll
  for (int i = 0; i < XC; ++i)
    xsrc[i] = reinterpret_cast<const AT*>(args.x) + (size_t)((uint32_t)min(m0 + (tl >> 3) + i * 8 * WN, M - 1) * (uint32_t)K);

  // request the stage of turn it into its ring slot; scales first, so that
  // the waits, which count COPIES, only ever wait for more than they need
  const int szperiod = max(1, (8 << args.lg) / GK);  // SZ8: stages per chunk of 8 groups
  auto request = [&](int it) {
    const int k0 = (st0 + it) * GK;
    const int slot = (it % RING) * SLOT;
    uint8_t* const xd = xlds + slot + (wn * 64) * 16;
    if constexpr (SZ8) {
      if (it == 0 || (st0 + it) % szperiod == 0) {
        const int chunk = (k0 >> args.lg) >> 3;
        lds_copy<16>(ssrc + 8 * chunk, szlds + (chunk & 1) * 2048);
        lds_copy<16>(zsrc + 8 * chunk, szlds + (chunk & 1) * 2048 + 1024);
      }
    } else {
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const int grp = min((k0 + g * (GK / 2)) >> args.lg, G - 1);
        lds_copy<sizeof(ST)>(ssrc + grp, wlds + slot + gemm_code_bytes(BITS) + (2 * g) * 256);
        lds_copy<sizeof(ST)>(zsrc + grp, wlds + slot + gemm_code_bytes(BITS) + (2 * g + 1) * 256);
      }
    }
    if (k0 + GK <= K) {
#pragma unroll
      for (int i = 0; i < XC; ++i) lds_copy<16>(xsrc[i] + k0 + xk, xd + i * 64 * WN * 16);
#pragma unroll
      for (int j = 0; j < WC; ++j) lds_copy<16>(wsrc[j] + (k0 * BITS / 8 + 16 * wk16), wlds + slot + j * 1024);
    } else {
      // the last, partial stage: chunks past K are zero, and the codes they
      // meet (the row's first, re-read) are unpacked with a zero scale, so that
      // they add nothing
#pragma unroll
      for (int i = 0; i < XC; ++i) {
        uint8_t* const d = xd + i * 64 * WN * 16;
        if (k0 + xk < K) lds_copy<16>(xsrc[i] + k0 + xk, d);
        else *reinterpret_cast<u32x4*>(d + lane * 16) = (u32x4){0u, 0u, 0u, 0u};
      }
#pragma unroll
      for (int j = 0; j < WC; ++j) {
        const int k = k0 + wk16 * (128 / BITS);
        // K % (128 / BITS) == 0: these 16 code bytes exist or not
        lds_copy<16>(wsrc[j] + (k < K ? k * BITS / 8 : 0), wlds + slot + j * 1024);
      }
    }
  };

  f32x4 acc[GNT][MT];
#pragma unroll
  for (int t = 0; t < GNT; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = (f32x4){0.f, 0.f, 0.f, 0.f};

  const uint32_t magic = in_vgpr(BITS == 4 ? 0x54006400u : 0x64646464u);
  const int xpos[2] = {r * 128 + (((2 * kb) ^ (r & 7)) << 4), r * 128 + (((2 * kb + 1) ^ (r & 7)) << 4)};
  const int wpos = r * CB + kb * (CB / 4);
  const int spos = gemm_code_bytes(BITS) + (kb >> 1) * 512 + r * 4;

#pragma unroll
  for (int j = 0; j < RING - 1; ++j)
    if (j < mine) request(j);
  for (int it = 0; it < per; ++it) {
    // this turn's stage has landed when at most the later stages' copies are
    // outstanding; the barrier then also frees the slot of the turn before,
    // which takes the stage RING - 1 turns on
    const int later = min(RING - 2, mine - 1 - it);
    if (later >= 2) stage_wait<2 * COPIES>();
    else if (later == 1) stage_wait<COPIES>();
    else stage_wait<0>();
    if (it + RING - 1 < mine) request(it + RING - 1);
    if (it >= mine) continue;
    const int slot = (it % RING) * SLOT;
    const uint8_t* const xb = xlds + slot;
    const uint8_t* const wb = wlds + slot;
    // SZ8: the group of this lane's 16 k (past K: the row's last one)
    const int grp = min(((st0 + it) * GK + 16 * kb) >> args.lg, G - 1);
    codes_t c[GNT];
    ST sv[GNT], zv[GNT];
#pragma unroll
    for (int t = 0; t < GNT; ++t) {
      c[t] = *reinterpret_cast<const codes_t*>(wb + wpos + t * 16 * CB);
      zv[t] = (ST)0.0f;
      if constexpr (SZ8) {
        const uint8_t* const p = szlds + ((grp >> 3) & 1) * 2048 + (16 * t + r) * 16 + (grp & 7) * 2;
        sv[t] = *reinterpret_cast<const ST*>(p);
        if (has_z) zv[t] = *reinterpret_cast<const ST*>(p + 1024);
      } else {
        sv[t] = *reinterpret_cast<const ST*>(wb + spos + t * 64);
        if (has_z) zv[t] = *reinterpret_cast<const ST*>(wb + spos + 256 + t * 64);
      }
    }
    if ((st0 + it + 1) * GK > K) {
      // The last, partial stage: lanes past K.  A weight that is none may be
      // infinite once rounded, and infinity times the zero activation is NaN.
      // (The asm keeps this a branch: as selects, every turn pays 2 % for it.)
      const bool past = (st0 + it) * GK + 16 * kb >= K;
      asm volatile("");
#pragma unroll
      for (int t = 0; t < GNT; ++t) {
        sv[t] = past ? (ST)0.0f : sv[t];
        zv[t] = past ? (ST)0.0f : zv[t];
      }
    }
    ExactGp<ST> ge[GNT];
    GpNat gp[GNT];
#pragma unroll
    for (int t = 0; t < GNT; ++t) {
      if constexpr (MAGIC) {
        gp[t] = make_gp_nat<BITS>((f16)sv[t], (f16)zv[t]);
      } else {
        ge[t] = make_exact_gp<ST>(sv[t], zv[t]);
      }
    }
    auto dequant = [&](int t, int h) {
      const uint32_t u0 = c[t][BITS == 4 ? h : 2 * h], u1 = c[t][BITS == 4 ? h : 2 * h + 1];
      if constexpr (MAGIC) return dq_nat8<BITS>(u0, u1, gp[t], magic);
      else return dq_exact8<BITS, AT, ST>(u0, u1, ge[t]);
    };
    // Chunks of two column tiles: a chunk requests the next one's activation
    // operands and unpacks a part of the second half's weights beside its
    // own products.
    constexpr int PER = MT / 2;  // chunks per half
    u32x4 xf[2][2], a[2][GNT];
    auto read_x = [&](int ch) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
        xf[ch & 1][j] = *reinterpret_cast<const u32x4*>(xb + (2 * (ch % PER) + j) * 16 * 128 + xpos[ch / PER]);
    };
    read_x(0);
#pragma unroll
    for (int t = 0; t < GNT; ++t) a[0][t] = dequant(t, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ch = 0; ch < 2 * PER; ++ch) {
      if (ch + 1 < 2 * PER) read_x(ch + 1);
      if (ch < PER) {
#pragma unroll
        for (int t = ch * GNT / PER; t < (ch + 1) * GNT / PER; ++t) a[1][t] = dequant(t, 1);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int t = 0; t < GNT; ++t) {
          const int mt = 2 * (ch % PER) + j;
          acc[t][mt] = mfma_k32<AT>(a[ch / PER][t], xf[ch & 1][j], acc[t][mt]);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  const bool vec = (N & 3) == 0 && ((reinterpret_cast<uintptr_t>(args.y0) | reinterpret_cast<uintptr_t>(args.y1) |
                                     reinterpret_cast<uintptr_t>(args.y2) |
                                     reinterpret_cast<uintptr_t>(args.residual)) & 7) == 0;
  if constexpr (WK == 1) {
#pragma unroll
    for (int t = 0; t < GNT; t += NMAT)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int m = m0 + 16 * mt + r;
        if (m < M)
          store_out4<AT, EPI>(args, vec, m, n0 + (t / NMAT) * 16 + 4 * kb, acc[t][mt], acc[t + NMAT - 1][mt]);
      }
  } else {
    // the K slices' accumulators meet in LDS: slice kg finishes the column
    // tiles mt with mt % WK == kg, the others leave theirs for it there
    // ([wn][mt][slice but the finishing one][t][lane])
    stage_wait<0>();  // every wave is done with the ring
    f32x4* red = reinterpret_cast<f32x4*>(gemm_lds);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int own = mt % WK;
      if (kg != own) {
        f32x4* d = red + (size_t)((wn * MT + mt) * (WK - 1) + (kg > own ? kg - 1 : kg)) * GNT * 64 + lane;
#pragma unroll
        for (int t = 0; t < GNT; ++t) d[t * 64] = acc[t][mt];
      }
    }
    lds_barrier();
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if (kg != mt % WK) continue;
      const int m = m0 + 16 * mt + r;
#pragma unroll
      for (int t = 0; t < GNT; ++t)
#pragma unroll
        for (int k2 = 0; k2 < WK - 1; ++k2)
          acc[t][mt] += red[(size_t)((wn * MT + mt) * (WK - 1) + k2) * GNT * 64 + t * 64 + lane];
#pragma unroll
      for (int t = 0; t < GNT; t += NMAT)
        if (m < M)
          store_out4<AT, EPI>(args, vec, m, n0 + (t / NMAT) * 16 + 4 * kb, acc[t][mt], acc[t + NMAT - 1][mt]);
    }
  }
}

// Workgroup shapes: MT column tiles, WN groups of 64 weight rows by WK slices
// of K, all of them one workgroup per CU (LDS).  `turn_us`: a turn of 64 k of
// such a workgroup with every CU busy, measured (q4, fp16, groups of 64):
// 2 x 14336 x 4096 at 509 rows 141 us as 8x8x1 (64 turns), 4096 x 14336 100 us
// as 8x1x4 and 101 as 4x2x4 (56 turns), 2 x 14336 x 4096 at 128 rows 55 us as
// 8x2x2 (32 turns), 4096 x 14336 at 64 rows 67 us as 4x1x4 (56 turns).  The times
// of this one type decide for all: bf16 takes 3-10 % longer, 8-bit codes 10-15 %
// less where a turn is short and up to as much more where scales come one by one,
// which may choose the second best shape, by as much.
struct GemmShape {
  int mt, wn, wk;
  float turn_us;
};
constexpr GemmShape kGemmShapes[] = {
    {8, 8, 1, 2.2f}, {8, 1, 4, 1.8f}, {4, 2, 4, 1.8f}, {8, 2, 2, 1.65f}, {4, 1, 4, 1.25f}};
constexpr int kGemmShapes4 = 5;
constexpr float kGemmFixedUs = 6.0f;  // launch, first stages and the slices' sum

// the shape with the least estimated time: rounds of workgroups over the CUs
// by turns.  (8 x 1 x 4 fits LDS with 4-bit codes only.)
inline int gemm_plan(int bits, int M, int N, int K, int nmat, int cus, float* us_out = nullptr) {
  int best = 0;
  float best_us = 0.0f;
  for (int i = 0; i < kGemmShapes4; ++i) {
    const GemmShape& g = kGemmShapes[i];
    if (bits == 8 && g.mt * g.wk == 32) continue;
    const int64_t rows = g.wn * 64 / nmat;
    const int64_t wgs = (int64_t)((M + 16 * g.mt - 1) / (16 * g.mt)) * ((N + rows - 1) / rows);
    const int64_t turns = ((K + GK - 1) / GK + g.wk - 1) / g.wk;
    const float us = kGemmFixedUs + (float)((wgs + cus - 1) / cus) * (float)turns * g.turn_us;
    if (i == 0 || us < best_us) {
      best = i;
      best_us = us;
    }
  }
  if (us_out) *us_out = best_us;
  return best;
}

template <int BITS, typename AT, typename ST, int NMAT, int EPI, bool SZ8, bool MAGIC, int MT, int WN, int WK, int RING>
int launch_plan(GemvArgs a, hipStream_t st) {
  const int rows = WN * 16 * GNT / NMAT;
  a.rg = (a.M + 16 * MT - 1) / (16 * MT);
  const int64_t tn8 = ((int64_t)((a.N + rows - 1) / rows) + 7) / 8 * 8;
  const int64_t grid = tn8 * a.rg;
  if (grid >= (1LL << 31)) return MK_ERR_UNSUPPORTED;
  constexpr size_t lds = gemm_lds_bytes(BITS, MT, WN, WK, SZ8, RING);
  static_assert(lds <= 160 * 1024, "the ring fits a CU's LDS");
  gemm_rows_kernel<BITS, AT, ST, NMAT, EPI, SZ8, MAGIC, MT, WN, WK, RING>
      <<<dim3((unsigned)grid), dim3(64 * WN * WK), lds, st>>>(a);
  MK_CHECK_LAUNCH();
  return MK_OK;
}

template <int BITS, typename AT, typename ST, int NMAT, int EPI, bool SZ8, bool MAGIC>
int launch_types(const GemvArgs& a, hipStream_t st) {
#define MK_PLAN(I, RING4, RING8)                                                                      \
  return launch_plan<BITS, AT, ST, NMAT, EPI, SZ8, MAGIC, kGemmShapes[I].mt, kGemmShapes[I].wn, kGemmShapes[I].wk, \
                     BITS == 4 ? RING4 : RING8>(a, st)
  // ring depths: as many stages as fit
  switch (gemm_plan(BITS, a.M, a.N, a.K, NMAT, device_cu_count())) {
    case 0: MK_PLAN(0, 2, 2);
    case 1:
      if constexpr (BITS == 4) MK_PLAN(1, 2, 2);
    case 2: MK_PLAN(2, 2, 2);
    case 3: MK_PLAN(3, 3, 2);
    default: MK_PLAN(4, 3, 2);
  }
#undef MK_PLAN
}

template <int BITS, typename AT, typename ST, int NMAT, int EPI>
int launch_scales(const GemvArgs& a, hipStream_t st) {
  // fp16 weights by the exponent trick where gemv_mfma_kernel would take it too;
  // exact for the layouts that were gemv_generic_kernel's alone, so that no
  // weight is held in fewer bits than there.  (Exact everywhere: 2 x 14336 x 4096
  // at 64 rows 35.4 -> 36.4 us, q8 4096 x 14336 at 300 rows 97 -> 105.)
  constexpr bool F16 = sizeof(ST) == 2 && __is_same(AT, f16);
  const bool exact = a.K % QFmt<BITS>::KL != 0;
  if constexpr (sizeof(ST) == 2) {
    bool sz8 = (a.G % 8) == 0;
    for (int t = 0; t < NMAT; ++t)
      sz8 = sz8 && mk_aligned(a.s[t], 16) && (a.z[0] == nullptr || mk_aligned(a.z[t], 16));
    if (sz8) {
      if constexpr (F16)
        if (exact) return launch_types<BITS, AT, ST, NMAT, EPI, true, false>(a, st);
      return launch_types<BITS, AT, ST, NMAT, EPI, true, F16>(a, st);
    }
  }
  if constexpr (F16)
    if (exact) return launch_types<BITS, AT, ST, NMAT, EPI, false, false>(a, st);
  return launch_types<BITS, AT, ST, NMAT, EPI, false, F16>(a, st);
}

}  // namespace

namespace mkq {

// rows of whole 16-byte code vectors, groups of a power of two >= 32, 16-byte
// activation chunks, 32-bit offsets into every operand
template <int BITS, int NMAT>
bool gemm_rows_ok(const GemvArgs& a, int64_t M, int64_t gs) {
  bool ok = a.lg >= 5 && (int64_t)1 << a.lg == gs && (a.K % (128 / BITS)) == 0 && mk_aligned(a.x, 16) &&
            (int64_t)a.N * a.row_bytes < (1LL << 31) && (int64_t)a.N * a.G < (1LL << 30) &&
            M * a.K < (1LL << 31) && zeros_alike<NMAT>(a);
  for (int t = 0; t < NMAT; ++t) ok = ok && mk_aligned(a.w[t], 16);
  return ok;
}

float gemm_rows_us(int bits, int nmat, int M, int N, int K) {
  float us;
  gemm_plan(bits, M, N, K, nmat, device_cu_count(), &us);
  return us;
}

template <int BITS, int NMAT, int EPI>
int launch_gemm_rows(const GemvArgs& a, int act_dt, int sc_dt, hipStream_t st) {
  if (act_dt == MK_DT_F16)
    return sc_dt == MK_DT_F16 ? launch_scales<BITS, f16, f16, NMAT, EPI>(a, st)
                              : launch_scales<BITS, f16, float, NMAT, EPI>(a, st);
  return sc_dt == MK_DT_F16 ? launch_scales<BITS, bf16, f16, NMAT, EPI>(a, st)
                            : launch_scales<BITS, bf16, float, NMAT, EPI>(a, st);
}

#define MK_INST(B)                                                                          \
  template bool gemm_rows_ok<B, 1>(const GemvArgs&, int64_t, int64_t);                               \
  template bool gemm_rows_ok<B, 2>(const GemvArgs&, int64_t, int64_t);                               \
  template int launch_gemm_rows<B, 1, EPI_RESIDUAL>(const GemvArgs&, int, int, hipStream_t); \
  template int launch_gemm_rows<B, 2, EPI_GATE_UP>(const GemvArgs&, int, int, hipStream_t);
MK_INST(4)
MK_INST(8)
#undef MK_INST

}  // namespace mkq
