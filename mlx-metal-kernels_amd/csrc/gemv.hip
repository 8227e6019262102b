// Groupwise-affine q4/q8 decode matvec family for gfx950.
//
// Semantics (ops/quant_ops.py:509-526, 574-588, 634-738):
//   y[m,n] = clip(sum_k x[m,k] * W[n,k], +-max(act)) rounded to the activation
//   type, W[n,k] = (q[n,k] - z[n,k/g]) * s[n,k/g].
// q4 codes are packed two per byte (low nibble = even k), so on little-endian
// hardware a 32-bit word holds 8 consecutive codes, nibble i at bits 4i.
//
// Who takes a launch (gemv_dispatch; each kernel's own conditions stand at its
// *_eligible or *_ok function):
//   1-4 rows (q8: 2), fp16 with fp16 scales, also those that passes of 32 leave
//     over: the v_dot2 kernel below;
//   up to 32 rows (q8: 16), fp16 scales, any activation type: the few-row kernel
//     (gemv_few.hip), in two passes up to twice that; without a workspace rows of
//     up to 4096 k only;
//   33 and more rows (q8 pairs and fp16: 17): the product kernel (gemm.hip), or
//     two passes where that is faster;
//   fp16 with fp16 scales, where they are faster or the few-row kernel does not
//     apply: the K-split kernel (one q4 matrix) and the tile kernel (17-32 rows);
//   what is left, fp32 scales above all: the MFMA kernel of 16 rows a launch, and
//     the generic kernel for odd layouts.
// The MFMA kernel (M <= 16 per launch, K % 64 == 0 for q4 / % 32 for q8, power-of-two
// group size >= 16 (q4) / >= 8 (q8)):
//   * one workgroup owns a 16-row output tile; its KW waves split K;
//   * lane (n = l%16, kb = l/16) streams 32 contiguous code bytes of row n per
//     chunk with two 128-bit loads, dequantizes them in registers and feeds
//     v_mfma_f32_16x16x32_{f16,bf16} with A = W tile (16 n x 32 k) and
//     B = x^T tile (32 k x 16 m); decode batches M < 16 pad B with zeros;
//   * the waves' partial 16x16 tiles are summed through LDS; the epilogue
//     saturates, and optionally fuses SwiGLU (gate/up) or a residual add.
// fp16 activations with fp16 scales use an exponent-magic dequant: a code c
// OR'ed into the mantissa of 1024.0h gives 1024+c exactly, so with zi the
// rounded zero point
//   w = fma((1024 + c) - (1024 + zi), s, -(z - zi) s)  (two packed-f16 ops
// per pair of weights; one rounding for integer zero points).
// The MFMA contraction is order-free in k, so the activation operand is built
// in the same permuted k order the magic unpack produces.
#include "common.h"
#include "gemv_common.h"
#include "norm_chunks.h"
#include "paged_common.h"

using namespace mkq;

namespace {

// --------------------------------------------------------------------------
// fast MFMA kernel (any M <= 16)
// --------------------------------------------------------------------------
template <int BITS, typename ST, int NMAT, int GPC>
struct WFrag {
  u32x4 w[NMAT][2];
  ST s[NMAT][GPC];
  ST z[NMAT][GPC];
};

template <int BITS, typename AT, typename ST, bool MAGIC, int GPC, int NMAT, int EPI>
__global__ __launch_bounds__(512) void gemv_mfma_kernel(const GemvArgs args) {
  using F = QFmt<BITS>;
  constexpr int STEPS = F::STEPS;
  constexpr int SPG = STEPS / GPC;  // MFMA steps per quantization group

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int kw = args.kw;
  const int M = args.M, N = args.N, K = args.K;

  const int n0 = blockIdx.x * 16;
  const int nl = lane & 15;
  const int kb = lane >> 4;
  const int n = n0 + nl;
  const int n_ld = n < N ? n : N - 1;  // rows past N load a valid row; results discarded
  const int m = lane & 15;
  const bool x_active = m < M;
  const uint32_t magic = in_vgpr(BITS == 4 ? 0x64006400u : 0x64646464u);
  const uint32_t magic_hi = in_vgpr(0x54005400u);  // q4 odd nibbles under 64.0h

  // this wave's chunk range
  const int chunks = (K + F::KC - 1) / F::KC;
  const int c_begin = (chunks * wave) / kw;
  const int c_end = (chunks * (wave + 1)) / kw;

  const uint8_t* wrow[NMAT];
  const ST* srow[NMAT];
  const ST* zrow[NMAT];
#pragma unroll
  for (int t = 0; t < NMAT; ++t) {
    wrow[t] = args.w[t] + (size_t)n_ld * args.row_bytes + kb * 32;
    srow[t] = reinterpret_cast<const ST*>(args.s[t]) + (size_t)n_ld * args.G;
    zrow[t] = args.z[t] ? reinterpret_cast<const ST*>(args.z[t]) + (size_t)n_ld * args.G : nullptr;
  }
  const AT* xrow = reinterpret_cast<const AT*>(args.x) + (size_t)(x_active ? m : 0) * K + kb * F::KL;

  // weights and scales of chunk c (the HBM streams); zero past K
  auto load_w = [&](int c, WFrag<BITS, ST, NMAT, GPC>& f) {
    const int k0 = c * F::KC + kb * F::KL;
    if (c < c_end && k0 < K) {
      const size_t boff = (size_t)c * (F::KC * BITS / 8);
      const int g0 = k0 >> args.lg;
#pragma unroll
      for (int t = 0; t < NMAT; ++t) {
        f.w[t][0] = ldg128_stream(wrow[t] + boff);
        f.w[t][1] = ldg128_stream(wrow[t] + boff + 16);
#pragma unroll
        for (int j = 0; j < GPC; ++j) {
          f.s[t][j] = srow[t][g0 + j];
          f.z[t][j] = zrow[t] ? zrow[t][g0 + j] : (ST)0.0f;
        }
      }
    } else {
#pragma unroll
      for (int t = 0; t < NMAT; ++t) {
        f.w[t][0] = (u32x4){0u, 0u, 0u, 0u};
        f.w[t][1] = (u32x4){0u, 0u, 0u, 0u};
#pragma unroll
        for (int j = 0; j < GPC; ++j) {
          f.s[t][j] = (ST)0.0f;
          f.z[t][j] = (ST)0.0f;
        }
      }
    }
  };

  f32x4 acc[NMAT];
#pragma unroll
  for (int t = 0; t < NMAT; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};

  WFrag<BITS, ST, NMAT, GPC> cur, nxt;
  load_w(c_begin, cur);
  for (int c = c_begin; c < c_end; ++c) {
    load_w(c + 1, nxt);  // prefetch: next chunk's weights are in flight while this one computes
    const int k0 = c * F::KC + kb * F::KL;
    u32x4 xv[STEPS];
    if (x_active && k0 < K) {
#pragma unroll
      for (int s = 0; s < STEPS; ++s) xv[s] = ldg128(xrow + (size_t)c * F::KC + 8 * s);
    } else {
#pragma unroll
      for (int s = 0; s < STEPS; ++s) xv[s] = (u32x4){0u, 0u, 0u, 0u};
    }

#pragma unroll
    for (int t = 0; t < NMAT; ++t) {
#pragma unroll
      for (int j = 0; j < GPC; ++j) {
        if constexpr (MAGIC) {
          const GpMagic gp = make_gp_magic((f16)cur.s[t][j], (f16)cur.z[t][j]);
#pragma unroll
          for (int s = j * SPG; s < (j + 1) * SPG; ++s) {
            u32x4 a;
            if constexpr (BITS == 4) a = dq4_magic(cur.w[t][s >> 2][s & 3], gp, magic, magic_hi);
            else a = dq8_magic(cur.w[t][s >> 1][(2 * s) & 3], cur.w[t][s >> 1][(2 * s + 1) & 3], gp, magic);
            acc[t] = mfma_k32<AT>(a, xperm<BITS, MAGIC>(xv[s]), acc[t]);
          }
        } else {
          GpExact gp;
          gp.s = to_f32(cur.s[t][j]);
          gp.z = to_f32(cur.z[t][j]);
#pragma unroll
          for (int s = j * SPG; s < (j + 1) * SPG; ++s) {
            u32x4 a;
            if constexpr (BITS == 4) a = dq4_exact<AT>(cur.w[t][s >> 2][s & 3], gp);
            else a = dq8_exact<AT>(cur.w[t][s >> 1][(2 * s) & 3], cur.w[t][s >> 1][(2 * s + 1) & 3], gp);
            acc[t] = mfma_k32<AT>(a, xv[s], acc[t]);
          }
        }
      }
    }
    cur = nxt;
  }

  // ---- cross-wave reduction through LDS
  __shared__ f32x4 red[NMAT][8][64];
  __shared__ int rk_slots[EPI == EPI_ROPE_KV ? kRopeRows : 1];
  if constexpr (EPI == EPI_ROPE_KV) rope_fill_slots(args, rk_slots);
#pragma unroll
  for (int t = 0; t < NMAT; ++t) red[t][wave][lane] = acc[t];
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int t = 0; t < NMAT; ++t) {
    f32x4 v = red[t][0][lane];
    for (int w = 1; w < kw; ++w) v += red[t][w][lane];
    acc[t] = v;
  }

  // ---- epilogue: lane holds D[n = nb + i][m], i = 0..3
  if (!x_active) return;
  const int nb = n0 + 4 * kb;
  if constexpr (EPI == EPI_ROPE_KV) {  // fp16 rows; nb is even, the pairs are (nb, nb+1), (nb+2, nb+3)
    rope_kv_pair(args, rk_slots, m, nb, acc[0][0], acc[0][1]);
    rope_kv_pair(args, rk_slots, m, nb + 2, acc[0][2], acc[0][3]);
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int nn = nb + i;
    if (nn >= N) break;
    store_out<AT, EPI>(args, (size_t)m * N + nn, acc[0][i], acc[NMAT - 1][i]);
  }
}

// --------------------------------------------------------------------------
// Batched decode tile kernel: fp16 activations and fp16 scales, M <= 16 * MT
// rows per launch, power-of-two group size >= 32, K % 128 == 0.  Used with
// MT = 2 for 17-32 rows that the few-row and product kernels do not take or take
// longer for (tile_rows_us): one pass over the weights instead of two 16-row
// MFMA passes.
//
// A workgroup owns 16 output rows of NMAT matrices; its kw waves split K
// into 128-k chunks.  Per chunk, lane (r = l % 16, kb = l / 16) takes the 32
// consecutive k at 32 * kb: 16 code bytes (q4) or 32 (q8) of row r, the
// (s, z) of the one group they lie in, and x over the same k for column r of
// each of the MT activation tiles -- four v_mfma_f32_16x16x32_f16 steps, the
// dequantized weight operand shared by the MT column tiles.
// The loads run NB chunks ahead in a ring of register buffers refilled in
// place (the loop is unrolled by NB, so no buffer is copied and every buffer
// keeps its registers): a chunk's x, codes and scales were issued NB - 1
// chunks before it is computed, and vmcnt retires in issue order, so computing
// a chunk waits for its own loads only.  Columns past M read row M - 1 (their
// results are dropped); the chunks past a wave's range in its last ring
// re-read its first chunk and are computed with x and s zeroed.
// --------------------------------------------------------------------------
template <int BITS, int NMAT, int MT>
struct TileBuf {
  u32x4 x[MT][4];                     // 4 steps x 8 halves per column tile
  u32x4 w[NMAT][BITS == 4 ? 1 : 2];   // 16 / 32 code bytes
  f16 s[NMAT];
  f16 z[NMAT];
  bool live;
};

template <int BITS, int NMAT, int MT, int NB, int EPI>
__global__ __launch_bounds__(NMAT == 1 && BITS == 4 ? 1024 : 512) void gemv_tile_kernel(const GemvArgs args) {
  constexpr int WB = BITS == 4 ? 1 : 2;  // 16-byte code vectors per lane per chunk
  constexpr int CB = 16 * WB;            // code bytes per lane per chunk
  using Buf = TileBuf<BITS, NMAT, MT>;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: scalar loop control
  const int kw = args.kw;
  const int M = args.M, N = args.N, K = args.K;
  const int n0 = blockIdx.x * 16;
  const int r = lane & 15;
  const int kb = lane >> 4;
  const int n_ld = n0 + r < N ? n0 + r : N - 1;  // rows past N load a valid row; results dropped
  const uint32_t magic = in_vgpr(BITS == 4 ? 0x64006400u : 0x64646464u);
  const uint32_t magic_hi = in_vgpr(0x54005400u);  // q4 odd nibbles under 64.0h
  const bool has_z = args.z[0] != nullptr;

  const int chunks = K >> 7;
  const int c_begin = (chunks * wave) / kw;
  const int c_end = (chunks * (wave + 1)) / kw;

  const uint8_t* wrow[NMAT];
  const f16* srow[NMAT];
  const f16* zrow[NMAT];
#pragma unroll
  for (int t = 0; t < NMAT; ++t) {
    wrow[t] = args.w[t] + (size_t)n_ld * args.row_bytes + kb * CB;
    srow[t] = reinterpret_cast<const f16*>(args.s[t]) + (size_t)n_ld * args.G;
    zrow[t] = has_z ? reinterpret_cast<const f16*>(args.z[t]) + (size_t)n_ld * args.G : srow[t];
  }
  const f16* xrow[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = 16 * mt + r;
    xrow[mt] = reinterpret_cast<const f16*>(args.x) + (size_t)(m < M ? m : M - 1) * K + 32 * kb;
  }

  // x first, then the codes and scales: the order the chunk is consumed in
  auto issue = [&](int c, Buf& b) {
    b.live = c < c_end;
    const int cc = b.live ? c : c_begin;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int s = 0; s < 4; ++s) b.x[mt][s] = ldg128(xrow[mt] + cc * 128 + 8 * s);
    const int g = (cc * 128 + 32 * kb) >> args.lg;
#pragma unroll
    for (int t = 0; t < NMAT; ++t) {
      const uint8_t* p = wrow[t] + (size_t)cc * (4 * CB);
#pragma unroll
      for (int v = 0; v < WB; ++v) b.w[t][v] = ldg128_stream(p + 16 * v);
      b.s[t] = srow[t][g];
      b.z[t] = zrow[t][g];
    }
  };

  f32x4 acc[NMAT][MT];
#pragma unroll
  for (int t = 0; t < NMAT; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = (f32x4){0.f, 0.f, 0.f, 0.f};

  auto compute = [&](const Buf& b, auto masked) {
    constexpr bool MASKED = decltype(masked)::value;
    u32x4 xp[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        xp[mt][s] = xperm<BITS, true>(b.x[mt][s]);
        if constexpr (MASKED)
          if (!b.live) xp[mt][s] = (u32x4){0u, 0u, 0u, 0u};
      }
#pragma unroll
    for (int t = 0; t < NMAT; ++t) {
      f16 sc = b.s[t];
      if constexpr (MASKED)
        if (!b.live) sc = (f16)0.0f;
      const GpMagic gp = make_gp_magic(sc, has_z ? b.z[t] : (f16)0.0f);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        u32x4 a;
        if constexpr (BITS == 4) a = dq4_magic(b.w[t][0][s], gp, magic, magic_hi);
        else a = dq8_magic(b.w[t][s >> 1][(2 * s) & 3], b.w[t][s >> 1][(2 * s + 1) & 3], gp, magic);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[t][mt] = mfma_k32<f16>(a, xp[mt][s], acc[t][mt]);
      }
    }
  };

  // scheduling barriers keep each buffer's loads together and in ring order,
  // so the wait before a chunk's compute leaves NB - 1 buffers in flight
  Buf b[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    issue(c_begin + i, b[i]);
    __builtin_amdgcn_sched_barrier(0);
  }
  int c = c_begin;
  for (; c + NB < c_end; c += NB) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      compute(b[i], std::false_type{});
      __builtin_amdgcn_sched_barrier(0);
      issue(c + NB + i, b[i]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) compute(b[i], std::true_type{});

  // ---- cross-wave reduction through LDS: [kw][NMAT * MT][64] partial tiles
  extern __shared__ __align__(16) uint8_t tile_red_raw[];
  f32x4* red = reinterpret_cast<f32x4*>(tile_red_raw);
  __shared__ int rk_slots[EPI == EPI_ROPE_KV ? kRopeRows : 1];
  if constexpr (EPI == EPI_ROPE_KV) rope_fill_slots(args, rk_slots);
#pragma unroll
  for (int t = 0; t < NMAT; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) red[(wave * NMAT * MT + t * MT + mt) * 64 + lane] = acc[t][mt];
  __syncthreads();
  // wave j finishes column tile j (j < MT): lane holds D[n = 4 kb + i][m = 16 j + r]
  if (wave >= MT) return;
  const int mt = wave;
  const int m = 16 * mt + r;
  f32x4 v[NMAT];
#pragma unroll
  for (int t = 0; t < NMAT; ++t) {
    v[t] = red[(t * MT + mt) * 64 + lane];
    for (int w = 1; w < kw; ++w) v[t] += red[(w * NMAT * MT + t * MT + mt) * 64 + lane];
  }
  if (m >= M) return;
  const int nb = n0 + 4 * kb;
  if constexpr (EPI == EPI_ROPE_KV) {
    rope_kv_pair(args, rk_slots, m, nb, v[0][0], v[0][1]);
    rope_kv_pair(args, rk_slots, m, nb + 2, v[0][2], v[0][3]);
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int nn = nb + i;
    if (nn >= N) break;
    store_out<f16, EPI>(args, (size_t)m * N + nn, v[0][i], v[NMAT - 1][i]);
  }
}

// --------------------------------------------------------------------------
// K-split batched kernel (q4, fp16 activations and scales, 5..32 rows, one
// matrix, K % 128 == 0 with 2048 <= K <= 16384, N % 16 == 0): long rows, in one
// launch where the few-row kernel cuts them into slices and sums those through a
// workspace -- of calls that give none, and of the batch sizes that one round of
// it takes sooner (gemv_dispatch).  One 16-row tile per workgroup of 16 waves;
// wave w takes an equal run of the row's 128-k halves (7 at K = 14336) and
// requests all of its
// codes up front (one 16-byte load per half: lane (r, kb) reads k in
// [128 h + 32 kb, +32) of row r, so each instruction reads the 16 rows'
// aligned 64-byte half lines), then walks its halves with the activations of
// the next two in flight -- four v_mfma_f32_16x16x32_f16 steps per half and
// column tile.  The tile's scales and zero points are staged in LDS once; the
// 16 partial tiles meet in LDS at the end.  The earlier MFMA kernel loaded a
// chunk's activations behind the next chunk's codes (so each chunk waited for
// the whole prefetch) and gathered (s, z) per lane.
// --------------------------------------------------------------------------
constexpr int XK_WAVES = 16;
constexpr int XK_MAX_HALVES = 8;  // 128-k halves per wave: K <= 16 x 8 x 128

inline size_t xk_lds_bytes(int mt, int G) {
  return (size_t)XK_WAVES * mt * 64 * sizeof(f32x4) + (size_t)2 * 16 * (G + 2) * 2;
}

template <int MT, int EPI>
__global__ __launch_bounds__(1024) void gemv_xk_kernel(const GemvArgs args) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int M = args.M, N = args.N, K = args.K, G = args.G;
  const int r = lane & 15, kb = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int H = K >> 7;
  const int h0 = (H * wave) / XK_WAVES;
  const int nh = (H * (wave + 1)) / XK_WAVES - h0;  // 1..XK_MAX_HALVES (checked by the dispatcher)
  const uint32_t magic = in_vgpr(0x64006400u);
  const uint32_t magic_hi = in_vgpr(0x54005400u);  // odd nibbles under 64.0h
  const bool has_z = args.z[0] != nullptr;

  // LDS: [16][MT][64] f32x4 partial tiles, then [2][16][G + 2] fp16 (s, z)
  extern __shared__ __align__(16) uint8_t xk_lds[];
  f32x4* red = reinterpret_cast<f32x4*>(xk_lds);
  const int gp = G + 2;
  f16* szs = reinterpret_cast<f16*>(xk_lds + (size_t)XK_WAVES * MT * 64 * sizeof(f32x4));
  __shared__ int rk_slots[EPI == EPI_ROPE_KV ? kRopeRows : 1];

  // (s, z) of the tile: 16-byte vectors v = tid and tid + 1024 (piece, row,
  // 8 groups), requested first so staging them waits for nothing else
  const int vpp = 2 * G;  // vectors per piece: 16 rows x G / 8
  u32x4 szv[2];
  int szo[2];
  bool szl[2], szz[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int v = tid + 1024 * j;
    szl[j] = v < 2 * vpp;
    const int vv = szl[j] ? v : 0;
    const int p = vv / vpp, e = vv - p * vpp;
    const int row = e / (G >> 3), c8 = e - row * (G >> 3);
    szz[j] = p == 1 && !has_z;
    const f16* base = reinterpret_cast<const f16*>(p == 1 && has_z ? args.z[0] : args.s[0]);
    szv[j] = ldg128(base + (size_t)(n0 + row) * G + 8 * c8);
    szo[j] = (p * 16 + row) * gp + 8 * c8;
  }
  __builtin_amdgcn_sched_barrier(0);

  // activations of half i in slot i % XR (the first XR requested before the
  // codes, the rest as slots free up; a ring of four measured no faster):
  // column 16 mt + r, k = 128 h + 32 kb + 8 s.  With one column tile the
  // columns past M are zero and not loaded (half the activation traffic at
  // 5..8 rows); results past M are dropped.
  constexpr int XR = 2;
  const f16* xr[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    xr[mt] = reinterpret_cast<const f16*>(args.x) + (size_t)min(16 * mt + r, M - 1) * K + 32 * kb;
  u32x4 xs[XR][MT][4];
  auto load_x = [&](int i, int slot) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if (MT == 2 || r < M) {  // two column tiles: rows past M repeat row M - 1 (no branch)
#pragma unroll
        for (int st = 0; st < 4; ++st) xs[slot][mt][st] = ldg128(xr[mt] + 128 * (h0 + i) + 8 * st);
      } else {
#pragma unroll
        for (int st = 0; st < 4; ++st) xs[slot][mt][st] = (u32x4){0u, 0u, 0u, 0u};
      }
    }
  };
#pragma unroll
  for (int i = 0; i < XR; ++i)
    if (i < nh) load_x(i, i);
  __builtin_amdgcn_sched_barrier(0);

  // all of this wave's codes
  const uint8_t* wr = args.w[0] + (size_t)(n0 + r) * args.row_bytes + 16 * kb;
  u32x4 w[XK_MAX_HALVES];
#pragma unroll
  for (int i = 0; i < XK_MAX_HALVES; ++i)
    if (i < nh) w[i] = ldg128_stream(wr + 64 * (h0 + i));
  __builtin_amdgcn_sched_barrier(0);

#pragma unroll
  for (int j = 0; j < 2; ++j)
    if (szl[j]) {
      uint32_t* d = reinterpret_cast<uint32_t*>(szs + szo[j]);
#pragma unroll
      for (int e = 0; e < 4; ++e) d[e] = szz[j] ? 0u : szv[j][e];
    }
  __syncthreads();

  f32x4 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const f16* sl = szs + r * gp;
#pragma unroll
  for (int i = 0; i < XK_MAX_HALVES; ++i) {
    if (i < nh) {
      const int g = (128 * (h0 + i) + 32 * kb) >> args.lg;
      const GpMagic gpm = make_gp_magic(sl[g], sl[16 * gp + g]);
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const u32x4 a = dq4_magic(w[i][st], gpm, magic, magic_hi);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt] = mfma_k32<f16>(a, xperm<4, true>(xs[i % XR][mt][st]), acc[mt]);
      }
      if (i + XR < nh) load_x(i + XR, i % XR);
    }
  }

  // the 16 partial tiles; wave j finishes column tile j (lane holds
  // D[n = 4 kb + i][m = 16 j + r])
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) red[(wave * MT + mt) * 64 + lane] = acc[mt];
  if constexpr (EPI == EPI_ROPE_KV) rope_fill_slots(args, rk_slots);
  __syncthreads();
  if (wave >= MT) return;
  const int mt = wave;
  const int m = 16 * mt + r;
  f32x4 v = red[mt * 64 + lane];
  for (int ww = 1; ww < XK_WAVES; ++ww) v += red[(ww * MT + mt) * 64 + lane];
  if (m >= M) return;
  const int nb = n0 + 4 * kb;
  if constexpr (EPI == EPI_ROPE_KV) {
    rope_kv_pair(args, rk_slots, m, nb, v[0], v[1]);
    rope_kv_pair(args, rk_slots, m, nb + 2, v[2], v[3]);
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) store_out<f16, EPI>(args, (size_t)m * N + nb + i, v[i], v[i]);
}

// --------------------------------------------------------------------------
// M <= 4 kernel: v_dot2_f32_f16 on (nearly) raw codes.
//
// A lane handles 32-k "units" (16 code bytes for q4, 32 for q8) of R output
// rows (x NMAT matrices); the R rows share the lane's x registers, and with
// several activation rows (a small decode batch) every row's dot products
// reuse the same unpacked codes -- 4 v_dot2 per 8 codes and row against a
// 5-instruction unpack, where the MFMA path spends 13 instructions per 8
// codes on dequantization and at M <= 4 uses at most a quarter of each
// 16-column product.  The codes
// are never scaled: the exponent-magic trick turns each code pair into an
// fp16 pair, v_dot2 accumulates x . code in fp32, and the group's affine map
// is applied once per unit in fp32:
//   sum_k x_k (c_k - z) s = s * (t - B - z * X),   X = sum of x.
// q4 low nibbles become exact codes c (1024 + c, minus 1024); high nibbles
// stay 1024 + 16c against x/16, i.e. c + 64 per unit of x, so B = 64 * X_hi
// (X_hi = sum of the x's met by high nibbles).  q8 bytes are 1024 + c with
// B = 1024 * X.  Keeping the offset small next to (c - z) keeps the fp32
// cancellation in (t - B) harmless.  Scales and zero points of the
// workgroup's rows are staged in LDS.  Needs fp16 activations, fp16 scales,
// power-of-two group size >= 32, K % 32 == 0.
// --------------------------------------------------------------------------
// rows per workgroup (per matrix): 4 for gate/up (twice the workgroups of 8
// rows keep more waves queued behind the resident ones, which shortens the
// drain at the end of the launch), 8 for a single matrix (whose K-split over
// up to 8 waves already gives each workgroup enough waves).  A small q4
// single-matrix launch at M = 1 -- under 2048 waves at 8 rows, i.e. fewer
// than two per SIMD, such as 4096 x 4096 -- takes 4 rows instead (launch_dot;
// measured 4096 x 4096 4.74 -> 4.35 us per call; the 4096 x 14336 down at 4
// rows, 7168 waves, measured 9.8 against 8.8 us).
template <int BITS, int NMAT>
constexpr int dot_rows() {
  return NMAT == 2 ? 4 : 8;
}
constexpr int kDotSmallRows = 4;
constexpr int kDotSmallWaves = 2048;
constexpr int DOT_SZ_VEC = 2;  // 16-byte (s|z) vectors staged per lane
constexpr int SEG_STRIDE = 64; // fp16 entries per staged (s|z) run

__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2(bitcast<f16x2>(a), bitcast<f16x2>(b), c, false);
}

// Partner exchange at lane distance D for the reductions below.  D = 32 and
// 16 use the gfx950 permlane swaps: permlane32_swap(a, b) leaves a = (a.lo,
// b.lo) and b = (a.hi, b.hi) by 32-lane halves, permlane16_swap does the same
// for the odd/even 16-lane rows, so a + b holds, in lanes with bit D clear,
// the pair sum of a and, in lanes with bit D set, the pair sum of b.  Smaller
// distances pair lanes inside a 16-lane row with DPP (row_partner below).
template <int D>
__device__ __forceinline__ float swap_sum(float a, float b) {
  static_assert(D == 32 || D == 16, "permlane swaps cover D = 32, 16");
  const auto r = D == 32 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false)
                         : __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The value of a partner lane that differs from this one in bit D (D = 8, 4,
// 2, 1), read with a DPP modifier (folded into the add that consumes it, no
// LDS round trip): D = 8 row_mirror (lane i <-> 15 - i, i.e. xor 15), D = 4
// row_half_mirror (xor 7), D = 2 / 1 quad_perm [2,3,0,1] / [1,0,3,2].  The
// masks 32, 16 (permlane swaps), 15, 7, 2, 1 are independent over GF(2), so
// the butterflies below still sum every lane of a group exactly once, and
// each pairing flips bit D, which is all the halving step's keep/send choice
// reads.  (Measured against ds_swizzle xor partners: the M = 1 down
// projection 8.8 -> 8.5 us.)
template <int D>
__device__ __forceinline__ float row_partner(float v) {
  static_assert(D == 8 || D == 4 || D == 2 || D == 1, "DPP row partners cover D < 16");
  constexpr int ctrl = D == 8 ? 0x140 : D == 4 ? 0x141 : D == 2 ? 0x4E : 0xB1;
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, 0xF, 0xF, false));
}

// Butterfly that halves the live values per step: at distance d a lane keeps
// the half selected by (lane & d) and adds the partner's copy of it.  After
// log2(CNT) steps every lane holds one value, then plain butterflies finish
// the 64-lane sum.  Lane l ends with the total of value index idx(l), where
// idx adds CNT/2, CNT/4, ... for each set bit 32, 16, ... of l.
template <int CNT, int D>
__device__ __forceinline__ void reduce_scatter(float* v, int lane) {
  if constexpr (D >= 1) {
    if constexpr (CNT > 1) {
      constexpr int H = CNT / 2;
      if constexpr (D >= 16) {
#pragma unroll
        for (int j = 0; j < H; ++j) v[j] = swap_sum<D>(v[j], v[j + H]);
      } else {
        const bool upper = (lane & D) != 0;
#pragma unroll
        for (int j = 0; j < H; ++j) {
          const float keep = upper ? v[j + H] : v[j];
          const float send = upper ? v[j] : v[j + H];
          v[j] = keep + row_partner<D>(send);
        }
      }
      reduce_scatter<H, D / 2>(v, lane);
    } else {
      if constexpr (D >= 16) v[0] = swap_sum<D>(v[0], v[0]);
      else v[0] += row_partner<D>(v[0]);
      reduce_scatter<1, D / 2>(v, lane);
    }
  }
}

template <int BITS, int NMAT, int R, int MR>
struct DotFrag {
  u32x4 w[NMAT][R][BITS == 4 ? 1 : 2];
  u32x4 x[MR][4];
};

// Full 64-lane sum, in every lane.
__device__ __forceinline__ float wave_total(float v) {
  v = swap_sum<32>(v, v);
  v = swap_sum<16>(v, v);
  v += row_partner<8>(v);
  v += row_partner<4>(v);
  v += row_partner<2>(v);
  return v + row_partner<1>(v);
}

// Workgroup layout: rg row groups of R rows (per matrix) x kw waves, one
// 2048-k slice per wave.  The plain kernel has one row group and each wave
// reads its slice of x straight from memory.  With the norm prologue (NORM)
// the workgroup loads x, the residual and the norm weight once, 16 bytes per
// thread, normalises the row into LDS, and every wave reads its slice from
// there: two row groups share that work, and the activation traffic per
// code byte is what keeps the prologue cheap.
// MR activation rows (1, 2 or 4; rows past M repeat row M - 1 and are not
// stored) share each lane's code unpack: a batched decode step costs 4 MR
// v_dot2 per 8 codes on top of the 5-instruction unpack.
template <int BITS, int NMAT, int EPI, bool NORM, int MR, int R = dot_rows<BITS, NMAT>()>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void gemv_dot_kernel(
    const GemvArgs args) {
  static_assert(!NORM || MR == 1, "the norm prologue takes one activation row");
  constexpr int V = NMAT * R;  // values per activation row reduced per lane
  constexpr int VT = V * MR;   // values reduced per lane
  constexpr int NSEG = V * 2;  // (matrix, row, s|z) runs staged per wave
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int kw = args.kw;
  const int grp = wave / kw;     // row group of this wave
  const int ks = wave - grp * kw;  // k slice of this wave
  const int N = args.N, K = args.K, G = args.G;
  const int n0 = ((int)blockIdx.x * args.rg + grp) * R;
  const uint32_t magic = in_vgpr(BITS == 4 ? 0x64006400u : 0x64646464u);
  const f16* x = reinterpret_cast<const f16*>(args.x);

  const uint8_t* wrow[NMAT][R];
#pragma unroll
  for (int t = 0; t < NMAT; ++t)
#pragma unroll
    for (int r = 0; r < R; ++r) wrow[t][r] = args.w[t] + (size_t)min(n0 + r, N - 1) * args.row_bytes;

  // unit u = ks * 64 + lane: one 128-bit code load per row (two for q8) and
  // four 16-byte x vectors; a wave's 64 units are contiguous in k
  const int U = K / 32;
  const int ubase = ks * 64;

  // dynamic LDS: [normalised row, K fp16 | NORM][(s, z) stage per wave]
  extern __shared__ __align__(16) uint8_t dot_lds[];
  f16* xrow = reinterpret_cast<f16*>(dot_lds);
  uint8_t* stage = dot_lds + (NORM ? (size_t)K * 2 : 0) + wave * (NSEG * 2 * SEG_STRIDE);

  // Scales and zero points: each wave stages, in its own LDS region, the
  // (s, z) of its rows for the groups its 64 units cover -- NSEG runs of gpw
  // fp16 values (gpw <= 64), fetched with 128-bit loads and stored at a fixed
  // stride of 64 entries so a row's run sits at a compile-time offset.  They
  // are requested first, then the activations, then the codes (vmcnt retires
  // in issue order, so each later wait leaves the code loads in flight).  With
  // the norm prologue the activations go first: the prologue then waits for
  // its L2-resident operands only, not for the (s, z) vectors from HBM
  // (measured 15.3 -> 14.8 us at 2 x 14336 x 4096; the plain kernel keeps the
  // (s, z) vectors first, 12.7 against 12.9 us).
  const int lsv = 8 - args.lg;      // log2(16-byte vectors per run), gpw = 8 << lsv
  const int nvec = NSEG << lsv;     // <= 64 * DOT_SZ_VEC (checked by the dispatcher)
  u32x4 szv[DOT_SZ_VEC];
  uint32_t sz_zero[DOT_SZ_VEC];
  auto issue_sz = [&]() {
    // branch-free: lanes without a run (or a missing zero tensor) read a valid
    // vector of the same row and drop it, so every load counts in order for
    // vmcnt.  A partial last slice clamps its vectors to the row's last 8
    // groups: the units past K that would use them are dropped.
    const int g0 = (ubase * 32) >> args.lg;
    const f16* s0 = reinterpret_cast<const f16*>(args.s[0]);
    const f16* s1 = reinterpret_cast<const f16*>(args.s[NMAT - 1]);
    const f16* z0 = args.z[0] ? reinterpret_cast<const f16*>(args.z[0]) : s0;
    const f16* z1 = args.z[NMAT - 1] ? reinterpret_cast<const f16*>(args.z[NMAT - 1]) : s1;
    const uint32_t has_z = args.z[0] != nullptr ? 1u : 0u;
#pragma unroll
    for (int j = 0; j < DOT_SZ_VEC; ++j) {
      const int v = lane + 64 * j;
      const int vv = v < nvec ? v : 0;
      const int seg = vv >> lsv;
      const int e = vv & ((1 << lsv) - 1);
      const int t = seg / (2 * R), r = (seg >> 1) % R, isz = seg & 1;
      const f16* base = t == 0 ? (isz ? z0 : s0) : (isz ? z1 : s1);
      const int nr = min(n0 + r, N - 1);
      szv[j] = ldg128(base + (size_t)nr * G + min(g0 + 8 * e, G - 8));
      sz_zero[j] = (uint32_t)isz & (has_z ^ 1u);  // zero tensor absent: z = 0
    }
  };
  auto stage_sz = [&]() {
#pragma unroll
    for (int j = 0; j < DOT_SZ_VEC; ++j) {
      const int v = lane + 64 * j;
      if (v < nvec) {
        const int seg = v >> lsv, e = v & ((1 << lsv) - 1);
        *reinterpret_cast<u32x4*>(stage + seg * (2 * SEG_STRIDE) + e * 16) =
            sz_zero[j] ? (u32x4){0u, 0u, 0u, 0u} : szv[j];
      }
    }
  };
  if constexpr (!NORM) {
    issue_sz();
    __builtin_amdgcn_sched_barrier(0);  // keep the small loads ahead of the rest
  }
  // residual epilogue: the lane that stores output (m, n0 + rr) requests its
  // residual value now, with the operands, not after the reduction (which
  // would add a memory trip to the last workgroup's tail); every lane loads
  // (an in-range element where it stores nothing) so the load counts in order
  f16 res_pre = (f16)0.0f;
  if constexpr (EPI == EPI_RESIDUAL) {
    const int m = lane / R, rr = lane - (lane / R) * R;
    const bool st = lane < R * MR && n0 + rr < N && m < args.M;
    res_pre = reinterpret_cast<const f16*>(args.residual)[st ? (size_t)m * N + n0 + rr : 0];
  }

  // activations: NORM -- 16-byte chunks c = threadIdx.x (+ blockDim.x) of x,
  // the residual and the norm weight, at most two per thread (the dispatcher
  // keeps K / 8 <= 2 * blockDim.x), clamped so every load issues; otherwise
  // -- this lane's four vectors of its unit of x.
  const int nthr = blockDim.x;
  u32x4 ax[NORM ? 2 : 1], ar[NORM ? 2 : 1], aw[NORM ? 2 : 1];
  DotFrag<BITS, NMAT, R, MR> f;
  const int u = ubase + lane;
  const int k0 = (u < U ? u : 0) * 32;
  if constexpr (NORM) {
    // chunks past the row (threads beyond K / 8, which the norm below
    // leaves out) re-read a chunk inside it, so every load stays in the row
    const NormChunks nc = norm_prologue_chunks(threadIdx.x, nthr, K);
    const int c0c = nc.c0, c1c = nc.c1;
    // no residual: the loads read x again and are dropped, so every load
    // still issues in order
    const f16* rp = reinterpret_cast<const f16*>(args.nres ? args.nres : args.x);
    const f16* wp = reinterpret_cast<const f16*>(args.nw);
    ax[0] = ldg128(x + 8 * c0c);
    ax[1] = ldg128(x + 8 * c1c);
    ar[0] = ldg128(rp + 8 * c0c);
    ar[1] = ldg128(rp + 8 * c1c);
    aw[0] = ldg128(wp + 8 * c0c);
    aw[1] = ldg128(wp + 8 * c1c);
    __builtin_amdgcn_sched_barrier(0);
    issue_sz();
  } else {
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      const f16* xm = x + (size_t)(m < args.M ? m : args.M - 1) * K;
#pragma unroll
      for (int j = 0; j < 4; ++j) f.x[m][j] = ldg128(xm + k0 + 8 * j);
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // the activation loads stay ahead of the codes
#pragma unroll
  for (int t = 0; t < NMAT; ++t)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint8_t* p = wrow[t][r] + (uint32_t)(k0 * BITS / 8);
      f.w[t][r][0] = ldg128_stream(p);
      if constexpr (BITS == 8) f.w[t][r][BITS == 4 ? 0 : 1] = ldg128_stream(p + 16);
    }
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (!NORM) stage_sz();

  if constexpr (NORM) {
    const int c0 = threadIdx.x, c1 = threadIdx.x + nthr;
    const NormChunks nc = norm_prologue_chunks(threadIdx.x, nthr, K);
    const bool has0 = nc.has0, has1 = nc.has1;
    {
      // z = fp16(x + r) and the row's sum of z^2 (the packed fp16 add rounds
      // the exact sum once, as the norm kernel's fp32 add-then-round does for
      // fp16 inputs), then n = fp16((z * inv) * w) in fp32 -- the arithmetic
      // of rms_norm_vec_kernel; workgroup 0 writes z and n out.  (No
      // residual: the loads above read x again; they are dropped here, after
      // the code requests, since selecting them waits for them.)
      if (!args.nres) ar[0] = ar[1] = (u32x4){0u, 0u, 0u, 0u};
      u32x4 zz[2];
      float ss = 0.0f;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          zz[i][e] = bitcast<uint32_t>(bitcast<f16x2>(ax[i][e]) + bitcast<f16x2>(ar[i][e]));
          const float sq = dot2(zz[i][e], zz[i][e], 0.0f);
          ss += (i == 0 ? has0 : has1) ? sq : 0.0f;
        }
      ss = wave_total(ss);
      __shared__ float norm_part[8];
      if (lane == 0) norm_part[wave] = ss;
      __syncthreads();
      float tot = 0.0f;
      for (int w = 0; w < (int)(nthr >> 6); ++w) tot += norm_part[w];
      const float inv = rsqrtf(tot / (float)K + args.eps);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (!(i == 0 ? has0 : has1)) continue;
        const int c = i == 0 ? c0 : c1;
        u32x4 nv;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const f16x2 zh = bitcast<f16x2>(zz[i][e]);
          const f16x2 wh = bitcast<f16x2>(aw[i][e]);
          const f16x2 nh = {(f16)(((float)zh[0] * inv) * (float)wh[0]),
                            (f16)(((float)zh[1] * inv) * (float)wh[1])};
          nv[e] = bitcast<uint32_t>(nh);
        }
        *reinterpret_cast<u32x4*>(xrow + 8 * c) = nv;
        if (blockIdx.x == 0) {
          if (args.zout) *reinterpret_cast<u32x4*>(reinterpret_cast<f16*>(args.zout) + 8 * c) = zz[i];
          if (args.nout) *reinterpret_cast<u32x4*>(reinterpret_cast<f16*>(args.nout) + 8 * c) = nv;
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) f.x[0][j] = *reinterpret_cast<const u32x4*>(xrow + k0 + 8 * j);
    stage_sz();
  } else {
    __builtin_amdgcn_wave_barrier();
  }

  float acc[VT];  // index m * V + t * R + r
#pragma unroll
  for (int i = 0; i < VT; ++i) acc[i] = 0.0f;

  {  // one 64-unit slice per wave (the dispatcher guarantees U <= 64 * kw)
    // a lane past the last unit computes on x = 0: its codes, offsets and
    // zero-point terms all vanish, so its sums add nothing
    if (u >= U) {
#pragma unroll
      for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int j = 0; j < 4; ++j) f.x[m][j] = (u32x4){0u, 0u, 0u, 0u};
    }

    // activation operands in the unpack order, and their sums, per row m
    uint32_t xp[MR][16];
    float xsm[MR], nboff[MR];
    const uint32_t one2 = 0x3C003C00u;  // (1.0h, 1.0h)
#pragma unroll
    for (int m = 0; m < MR; ++m) {
    float xs = 0.0f;  // X, the sum of the slice's x
    float boff;       // what the exponent-magic offsets add to the code sums
    if constexpr (BITS == 4) {
      // low nibbles decode to 1024 + c, high nibbles (in place) to
      // 1024 + 16 c against x / 16: the offsets sum to 1024 X_lo + 64 X_hi
      float xs_hi = 0.0f, xs_lo = 0.0f;
      const f16x2 sixteenth = {(f16)0.0625f, (f16)0.0625f};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        // word j covers x[8j .. 8j+8): pairs (0,4) (1,5)/16 (2,6) (3,7)/16
        const uint32_t p0 = pack_lo16(f.x[m][j][0], f.x[m][j][2]);
        const uint32_t p1 = pack_hi16(f.x[m][j][0], f.x[m][j][2]);
        const uint32_t p2 = pack_lo16(f.x[m][j][1], f.x[m][j][3]);
        const uint32_t p3 = pack_hi16(f.x[m][j][1], f.x[m][j][3]);
        xs_hi = dot2(p1, one2, dot2(p3, one2, xs_hi));
        xs_lo = dot2(p0, one2, dot2(p2, one2, xs_lo));
        xp[m][4 * j + 0] = p0;
        xp[m][4 * j + 1] = bitcast<uint32_t>(bitcast<f16x2>(p1) * sixteenth);
        xp[m][4 * j + 2] = p2;
        xp[m][4 * j + 3] = bitcast<uint32_t>(bitcast<f16x2>(p3) * sixteenth);
      }
      xs = xs_lo + xs_hi;
      boff = 1024.0f * xs_lo + 64.0f * xs_hi;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        // two words per 8 x's: pairs (0,2) (1,3) (4,6) (5,7)
        xp[m][4 * j + 0] = pack_lo16(f.x[m][j][0], f.x[m][j][1]);
        xp[m][4 * j + 1] = pack_hi16(f.x[m][j][0], f.x[m][j][1]);
        xp[m][4 * j + 2] = pack_lo16(f.x[m][j][2], f.x[m][j][3]);
        xp[m][4 * j + 3] = pack_hi16(f.x[m][j][2], f.x[m][j][3]);
        xs = dot2(xp[m][4 * j + 0], one2, dot2(xp[m][4 * j + 1], one2,
                  dot2(xp[m][4 * j + 2], one2, dot2(xp[m][4 * j + 3], one2, xs))));
      }
      boff = 1024.0f * xs;
    }
    xsm[m] = xs;
    nboff[m] = -boff;
    }
    // this lane's group within the wave's slice; run seg is at seg * 64
    const f16* szl = reinterpret_cast<const f16*>(stage) + ((lane * 32) >> args.lg);

#pragma unroll
    for (int t = 0; t < NMAT; ++t)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float tsum[MR];
#pragma unroll
        for (int m = 0; m < MR; ++m) tsum[m] = nboff[m];
        if constexpr (BITS == 4) {
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            const uint32_t q = f.w[t][r][0][w];
            const uint32_t v = q >> 8;
            const uint32_t c0 = (q & 0x000F000Fu) | magic, c1 = (q & 0x00F000F0u) | magic;
            const uint32_t c2 = (v & 0x000F000Fu) | magic, c3 = (v & 0x00F000F0u) | magic;
#pragma unroll
            for (int m = 0; m < MR; ++m) {
              tsum[m] = dot2(c0, xp[m][4 * w + 0], tsum[m]);
              tsum[m] = dot2(c1, xp[m][4 * w + 1], tsum[m]);
              tsum[m] = dot2(c2, xp[m][4 * w + 2], tsum[m]);
              tsum[m] = dot2(c3, xp[m][4 * w + 3], tsum[m]);
            }
          }
        } else {
#pragma unroll
          for (int w = 0; w < 8; ++w) {
            const uint32_t q = f.w[t][r][w >> 2][w & 3];
            const uint32_t lo = q8_lo_pair(q, magic), hi = q8_hi_pair(q, magic);
#pragma unroll
            for (int m = 0; m < MR; ++m) {
              tsum[m] = dot2(lo, xp[m][2 * w + 0], tsum[m]);
              tsum[m] = dot2(hi, xp[m][2 * w + 1], tsum[m]);
            }
          }
        }
        const int seg = (t * R + r) * 2;
        const float sv = (float)szl[seg * SEG_STRIDE];
        const float zv = (float)szl[(seg + 1) * SEG_STRIDE];
#pragma unroll
        for (int m = 0; m < MR; ++m)
          acc[m * V + t * R + r] = fmaf(sv, fmaf(-zv, xsm[m], tsum[m]), acc[m * V + t * R + r]);
      }
  }

  // ---- 64-lane reduction (halving butterfly), then across the row group's
  // waves in LDS
  static_assert(VT <= 64 && (VT & (VT - 1)) == 0, "lane reduction shape");
  reduce_scatter<VT, 32>(acc, lane);
  const float tot = acc[0];
  int idx = 0;
#pragma unroll
  for (int d = 32, h = VT / 2; h >= 1; d >>= 1, h >>= 1)
    if (lane & d) idx += h;
  __shared__ float red[8][VT];
  __shared__ int rk_slots[EPI == EPI_ROPE_KV ? kRopeRows : 1];
  if constexpr (EPI == EPI_ROPE_KV) rope_fill_slots(args, rk_slots);
  constexpr int QUAD = 64 / VT;  // lanes holding the same index
  if ((lane & (QUAD - 1)) == 0) red[wave][idx] = tot;
  __syncthreads();
  if (ks != 0 || lane >= R * MR) return;
  const int m = lane / R, rr = lane - m * R;
  float v0 = 0.0f, v1 = 0.0f;
  for (int w = 0; w < kw; ++w) {
    v0 += red[wave + w][m * V + rr];
    if constexpr (NMAT == 2) v1 += red[wave + w][m * V + R + rr];
  }
  const int nn = n0 + rr;
  if constexpr (EPI == EPI_ROPE_KV) {
    rope_kv_store(args, rk_slots, m, nn, v0);  // lane pairs (rr even, rr + 1) never straddle a head: R and D even
    return;
  }
  if (nn < N && m < args.M) {
    if constexpr (EPI == EPI_RESIDUAL) {  // store_out's arithmetic with the prefetched residual
      const f16 d = saturate_cast<f16>(v0);
      if (args.y0) reinterpret_cast<f16*>(args.y0)[(size_t)m * N + nn] = d;
      reinterpret_cast<f16*>(args.y1)[(size_t)m * N + nn] = from_f32<f16>(to_f32(res_pre) + to_f32(d));
    } else {
      store_out<f16, EPI>(args, (size_t)m * N + nn, v0, v1);
    }
  }
}

// --------------------------------------------------------------------------
// generic kernel: any K (odd K uses ceil(K/2) packed columns), any group size,
// any M.  One wave per output row; fp32 math with the dequantized weight
// rounded to the activation type first, as the reference path does
// (ops/quant_ops.py:523-526).
// --------------------------------------------------------------------------
template <int BITS, typename AT, typename ST, int NMAT, int EPI>
__global__ __launch_bounds__(256) void gemv_generic_kernel(const GemvArgs args, int gs) {
  const int lane = threadIdx.x & 63;
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n >= args.N) return;
  const int K = args.K, M = args.M, N = args.N;
  const AT* x = reinterpret_cast<const AT*>(args.x);
  for (int m = 0; m < M; ++m) {
    float dot[NMAT];
#pragma unroll
    for (int t = 0; t < NMAT; ++t) {
      const uint8_t* wr = args.w[t] + (size_t)n * args.row_bytes;
      const ST* sr = reinterpret_cast<const ST*>(args.s[t]) + (size_t)n * args.G;
      const ST* zr = args.z[t] ? reinterpret_cast<const ST*>(args.z[t]) + (size_t)n * args.G : nullptr;
      float a = 0.f;
      for (int k = lane; k < K; k += 64) {
        uint32_t q;
        if constexpr (BITS == 4) {
          const uint8_t b = wr[k >> 1];
          q = (k & 1) ? (b >> 4) : (b & 15u);
        } else {
          q = wr[k];
        }
        const int g = k / gs;
        const float s = to_f32(sr[g]);
        const float z = zr ? to_f32(zr[g]) : 0.0f;
        const float w = to_f32(from_f32<AT>(((float)q - z) * s));
        a += to_f32(x[(size_t)m * K + k]) * w;
      }
      dot[t] = wave_sum(a);
    }
    if (lane != 0) continue;
    const size_t o = (size_t)m * N + n;
    if constexpr (EPI == EPI_NONE) {
      reinterpret_cast<AT*>(args.y0)[o] = saturate_cast<AT>(dot[0]);
    } else if constexpr (EPI == EPI_RESIDUAL) {
      const AT d = saturate_cast<AT>(dot[0]);
      if (args.y0) reinterpret_cast<AT*>(args.y0)[o] = d;
      const float r = to_f32(reinterpret_cast<const AT*>(args.residual)[o]);
      reinterpret_cast<AT*>(args.y1)[o] = from_f32<AT>(r + to_f32(d));
    } else {
      const AT g = saturate_cast<AT>(dot[0]);
      const AT u = saturate_cast<AT>(dot[NMAT - 1]);
      if (args.y0) reinterpret_cast<AT*>(args.y0)[o] = g;
      if (args.y1) reinterpret_cast<AT*>(args.y1)[o] = u;
      if (args.y2) {
        const float gf = to_f32(g);
        const float sil = gf / (1.0f + expf(-gf));
        reinterpret_cast<AT*>(args.y2)[o] = from_f32<AT>(sil * to_f32(u));
      }
    }
  }
}

// --------------------------------------------------------------------------
// host dispatch
// --------------------------------------------------------------------------
inline int ilog2_exact(int64_t v) {
  if (v <= 0 || (v & (v - 1))) return -1;
  int l = 0;
  while ((1LL << l) < v) ++l;
  return l;
}

template <int BITS, typename AT, typename ST, bool MAGIC, int NMAT, int EPI>
int launch_fast(const GemvArgs& a, int gpc, hipStream_t st) {
  const dim3 grid((a.N + 15) / 16);
  const dim3 block(64 * a.kw);
  switch (gpc) {
    case 1: gemv_mfma_kernel<BITS, AT, ST, MAGIC, 1, NMAT, EPI><<<grid, block, 0, st>>>(a); break;
    case 2: gemv_mfma_kernel<BITS, AT, ST, MAGIC, 2, NMAT, EPI><<<grid, block, 0, st>>>(a); break;
    case 4: gemv_mfma_kernel<BITS, AT, ST, MAGIC, 4, NMAT, EPI><<<grid, block, 0, st>>>(a); break;
    default: return MK_ERR_UNSUPPORTED;
  }
  MK_CHECK_LAUNCH();
  return MK_OK;
}

// Tile kernel plan: rings of two chunks (the registers that two column tiles'
// activations leave) and kw waves per 16-row tile, kw <= 16 for a single q4
// matrix, else 8 (1024 / 512 threads), preferring a split that gives every wave a
// whole number of rings and at least one.
constexpr int kTileRing = 2;

template <int BITS, int NMAT>
inline int tile_choose_kw(int64_t K, int nb) {
  const int64_t chunks = K / 128;
  const int kmax = NMAT == 1 && BITS == 4 ? 16 : 8;
  for (int kw = kmax; kw >= 1; --kw)
    if (chunks % kw == 0 && (chunks / kw) % nb == 0) return kw;
  int64_t kw = (chunks + nb - 1) / nb;  // every wave at least one ring
  return (int)(kw < 1 ? 1 : (kw > kmax ? kmax : kw));
}

template <int BITS, int NMAT, int MT, int EPI>
int launch_tile(GemvArgs a, hipStream_t st) {
  constexpr int NB = kTileRing;
  a.kw = tile_choose_kw<BITS, NMAT>(a.K, NB);
  if (a.kw < MT) a.kw = MT;  // wave j finishes column tile j
  const dim3 grid((unsigned)((a.N + 15) / 16));
  const dim3 block((unsigned)(64 * a.kw));
  const size_t lds = (size_t)a.kw * NMAT * MT * 64 * sizeof(f32x4);
  gemv_tile_kernel<BITS, NMAT, MT, NB, EPI><<<grid, block, lds, st>>>(a);
  MK_CHECK_LAUNCH();
  return MK_OK;
}

constexpr int kXkMinRows = 5;  // fewer: the v_dot2 and MFMA kernels
constexpr size_t kXkMaxLds = 160 * 1024;

// K-split launch: one 16-row tile per workgroup of 16 waves
template <int MT, int EPI>
int launch_xk(GemvArgs a, hipStream_t st) {
  const dim3 grid((unsigned)(a.N / 16));
  const dim3 block(64 * XK_WAVES);
  gemv_xk_kernel<MT, EPI><<<grid, block, xk_lds_bytes(MT, a.G), st>>>(a);
  MK_CHECK_LAUNCH();
  return MK_OK;
}

// q4, one matrix, fp16 activations and scales, power-of-two group >= 32,
// K % 128 == 0 with 16 <= K / 128 <= 16 x 8, N % 16 == 0, the tile's (s, z)
// within two 16-byte vectors per thread, 16-byte aligned operands
template <int BITS, int NMAT>
bool xk_eligible(const GemvArgs& a, int mt, int act_dt, int sc_dt) {
  const int H = a.K / 128;
  bool ok = BITS == 4 && NMAT == 1 && act_dt == MK_DT_F16 && sc_dt == MK_DT_F16 && a.lg >= 5 &&
            (a.K % 128) == 0 && H >= XK_WAVES && H <= XK_WAVES * XK_MAX_HALVES && (a.N % 16) == 0 &&
            (a.G % 8) == 0 && 4 * a.G <= 2 * 64 * XK_WAVES && xk_lds_bytes(mt, a.G) <= kXkMaxLds &&
            mk_aligned(a.x, 16) && (size_t)a.row_bytes % 16 == 0 && mk_aligned(a.w[0], 16) &&
            mk_aligned(a.s[0], 16) && (a.z[0] == nullptr || mk_aligned(a.z[0], 16));
  return ok;
}

// fp16 activations and scales, power-of-two group >= 32, K % 128 == 0, 16-byte
// aligned x and codes
template <int NMAT>
bool tile_eligible(const GemvArgs& a, int act_dt, int sc_dt) {
  bool ok = act_dt == MK_DT_F16 && sc_dt == MK_DT_F16 && a.lg >= 5 && (a.K % 128) == 0 &&
            mk_aligned(a.x, 16) && (size_t)a.row_bytes % 16 == 0 && zeros_alike<NMAT>(a);
  for (int t = 0; t < NMAT; ++t) ok = ok && mk_aligned(a.w[t], 16);
  return ok;
}

// Row groups per dot workgroup: one for the plain kernel (measured: sharing
// x through LDS costs a barrier that outweighs its L2 savings); two for the
// norm prologue (four at K <= 2048), which keeps K / 8 <= 2 * blockDim.x for
// K <= 8192 and halves the activation reads per code byte.
template <bool NORM>
inline int dot_row_groups(int kw) { return NORM ? (kw >= 2 ? 2 : 4) : 1; }

template <int BITS, int NMAT, int EPI, bool NORM, int R>
int launch_dot_rows(GemvArgs a, hipStream_t st) {
  a.rg = dot_row_groups<NORM>(a.kw);
  const int rows = R * a.rg;
  const dim3 grid((unsigned)((a.N + rows - 1) / rows));
  const dim3 block((unsigned)(64 * a.kw * a.rg));
  const size_t stage_bytes = (size_t)a.kw * a.rg * NMAT * R * 2 * (2 * SEG_STRIDE);
  const size_t lds = (NORM ? (size_t)a.K * 2 : 0) + stage_bytes;
  if constexpr (NORM) {
    MK_REQUIRE(a.K / 8 <= 2 * (int)block.x);  // the prologue's two 16-byte chunks per thread cover the row
    gemv_dot_kernel<BITS, NMAT, EPI, true, 1, R><<<grid, block, lds, st>>>(a);
  } else {
    if (a.M <= 1) gemv_dot_kernel<BITS, NMAT, EPI, false, 1, R><<<grid, block, lds, st>>>(a);
    else if constexpr (R != dot_rows<BITS, NMAT>()) return MK_ERR_UNSUPPORTED;  // small-launch rows: M = 1 only
    else if (a.M == 2) gemv_dot_kernel<BITS, NMAT, EPI, false, 2, R><<<grid, block, lds, st>>>(a);
    else if constexpr (BITS == 4) gemv_dot_kernel<BITS, NMAT, EPI, false, 4, R><<<grid, block, lds, st>>>(a);
    else return MK_ERR_UNSUPPORTED;  // q8: at most two rows (four would spill)
  }
  MK_CHECK_LAUNCH();
  return MK_OK;
}

template <int BITS, int NMAT, int EPI, bool NORM = false>
int launch_dot(GemvArgs a, hipStream_t st) {
  constexpr int R = dot_rows<BITS, NMAT>();
  if constexpr (BITS == 4 && NMAT == 1 && R > kDotSmallRows) {
    // a q4 single matrix at M = 1 that would run under kDotSmallWaves waves
    const int rg = dot_row_groups<NORM>(a.kw);
    const int64_t waves = (int64_t)((a.N + R * rg - 1) / (R * rg)) * rg * a.kw;
    if (a.M <= 1 && waves < kDotSmallWaves) return launch_dot_rows<BITS, NMAT, EPI, NORM, kDotSmallRows>(a, st);
  }
  return launch_dot_rows<BITS, NMAT, EPI, NORM, R>(a, st);
}

template <int BITS, typename AT, typename ST, int NMAT, int EPI>
int launch_generic(const GemvArgs& a, int gs, hipStream_t st) {
  const dim3 grid((a.N + 3) / 4);
  gemv_generic_kernel<BITS, AT, ST, NMAT, EPI><<<grid, dim3(256), 0, st>>>(a, gs);
  MK_CHECK_LAUNCH();
  return MK_OK;
}

// Waves per workgroup: enough K-parallelism to keep >= ~4 waves per SIMD
// in flight on 256 CUs, without giving a wave less than one chunk.
inline int choose_kw(int64_t N, int64_t K, int kc) {
  const int64_t tiles = (N + 15) / 16;
  const int64_t chunks = (K + kc - 1) / kc;
  int kw = tiles >= 1024 ? 4 : 8;
  if (kw > chunks) kw = (int)chunks;
  if (kw < 1) kw = 1;
  return kw;
}

// Shape facts every launch needs: fills N, K, G, row_bytes and lg of a;
// returns the groups per 32-code lane chunk of the MFMA path (0: none) and
// whether the aligned fast layouts apply.
template <int BITS, int NMAT>
int gemv_prepare(GemvArgs& a, int64_t N, int64_t K, int64_t gs, bool* fast) {
  using F = QFmt<BITS>;
  a.N = (int)N;
  a.K = (int)K;
  a.G = (int)((K + gs - 1) / gs);
  a.row_bytes = BITS == 4 ? (int)((K + 1) / 2) : (int)K;
  const int lg = ilog2_exact(gs);
  int gpc = 0;
  if (lg >= 0) {
    if (gs >= F::KL) gpc = 1;
    else if (gs >= 8 && F::KL / gs <= 4) gpc = (int)(F::KL / gs);
  }
  bool f = gpc > 0 && (K % F::KL) == 0 && mk_aligned(a.x, 16);
  for (int t = 0; t < NMAT; ++t) f = f && mk_aligned(a.w[t], 16);
  a.lg = lg;
  *fast = f;
  return gpc;
}

// The dot kernel (M <= 4): one 64-unit (2048-k) slice per wave, <= 8 waves;
// the (s, z) runs of a slice must be whole 16-byte vectors and fit the stage.
template <int BITS, int NMAT>
bool dot_eligible(const GemvArgs& a, bool fast, int64_t mrows, int act_dt, int sc_dt) {
  const int lg = a.lg;
  const int64_t K = a.K;
  const int64_t gpw = lg >= 0 ? (2048 >> lg) : 0;
  return fast && mrows >= 1 && mrows <= (BITS == 4 ? 4 : 2) && act_dt == MK_DT_F16 && sc_dt == MK_DT_F16 &&
         lg >= 5 && lg <= 8 &&
         (K % 32) == 0 && K <= 8 * 2048 && (a.G % 8) == 0 && (gpw % 8) == 0 &&
         (int64_t)NMAT * dot_rows<BITS, NMAT>() * 2 * (gpw / 8) <= 64 * DOT_SZ_VEC &&
         mk_aligned(a.s[0], 16) && mk_aligned(a.s[NMAT - 1], 16) &&
         zeros_alike<NMAT>(a) &&
         (a.z[0] == nullptr || (mk_aligned(a.z[0], 16) && mk_aligned(a.z[NMAT - 1], 16)));
}

// waves per dot-kernel workgroup: one per 64-unit slice
inline int dot_waves(int64_t K) {
  int64_t kwd = (K / 32 + 63) / 64;
  return (int)(kwd < 1 ? 1 : (kwd > 8 ? 8 : kwd));
}

// rows from which the matrix-product kernel takes a launch (below: passes of
// up to 32 rows through the kernels here)
constexpr int64_t kGemmMinRows = 33;

// Estimated us of the tile kernel's 17-32 rows: rounds of workgroups over the
// CUs, each as long as a row.  Measured at 32 rows (17 rows), this in brackets,
// q8: 4096 x 4096 13.8 (11.3) [13.9 (10.5)], 6144 x 4096 24.6 (19.2) [24.8
// (18.0)], 4096 x 14336 41.4 (32.1) [41.1 (29.6)], 33000 x 1024 27.7 [27.5], 2 x
// 4096 x 4096 18.9 (16.4) [18.6 (16.4)], 2 x 14336 x 4096 65.4 (55.0) [65.4
// (56.7)]; q4: 2 x 8192 x 8192 55.2 [55.2].
template <int BITS, int NMAT>
inline float tile_rows_us(int64_t M, int64_t N, int64_t K) {
  const int cus = device_cu_count();
  const float rounds = (float)(((N + 15) / 16 + cus - 1) / cus);
  const float us = BITS == 4 ? 3.26f : NMAT == 2 ? 3.9f : 2.72f;  // per 1024 k
  const float rows = NMAT == 2 ? 0.7f + 0.0094f * (float)M : 0.53f + 0.0147f * (float)M;
  return 3.0f + rounds * us * rows * (float)K / 1024.0f;
}

// Rows of a whole pass.  The 1-4 rows (q8: 1-2) that a batch leaves past its last
// one take the v_dot2 kernel, which does not round W: other kernels would hold
// their weights in fp16 only because of the rows beside them (error of such a row
// against 64 bits 2.1e-4, 3.0e-4 with rounded weights).  32 rows, or 16: where the
// tile kernel does not apply, and for pairs of 128 groups of 32.
template <int BITS, int NMAT>
inline int64_t pass_rows(int64_t N, int64_t K, int64_t gs) {
  const bool pair32 = BITS == 4 && NMAT == 2 && K == 4096 && gs == 32 && N % 16 == 0 && N >= 4096;
  return K % 128 != 0 || pair32 ? 16 : 32;
}

template <int BITS, int NMAT, int EPI>
int gemv_dispatch(GemvArgs a, int64_t M, int64_t N, int64_t K, int64_t gs, int act_dt, int sc_dt,
                  hipStream_t st, float* ws = nullptr, size_t ws_bytes = 0, int64_t product_rows = kGemmMinRows) {
  using F = QFmt<BITS>;
  MK_REQUIRE(M >= 0 && N > 0 && K > 0 && gs > 0);
  MK_REQUIRE(act_dt == MK_DT_F16 || act_dt == MK_DT_BF16);
  MK_REQUIRE(sc_dt == MK_DT_F16 || sc_dt == MK_DT_F32);
  MK_REQUIRE(N < (1LL << 31) && K < (1LL << 31));
  if (M == 0) return MK_OK;
  for (int t = 0; t < NMAT; ++t) MK_REQUIRE(a.w[t] && a.s[t]);
  MK_REQUIRE(a.x);

  bool fast;
  const int gpc = gemv_prepare<BITS, NMAT>(a, N, K, gs, &fast);

  const size_t xe = 2;  // activation element size
  int rc = MK_OK;
  // rows m0.. of every row-indexed operand
  auto rows_from = [&](GemvArgs& b, int64_t m0) {
    b.x = (const char*)a.x + (size_t)m0 * K * xe;
    if (a.residual) b.residual = (const char*)a.residual + (size_t)m0 * N * xe;
    if (a.y0) b.y0 = (char*)a.y0 + (size_t)m0 * N * xe;
    if (a.y1) b.y1 = (char*)a.y1 + (size_t)m0 * N * xe;
    if (a.y2) b.y2 = (char*)a.y2 + (size_t)m0 * N * xe;
    if constexpr (EPI == EPI_ROPE_KV) {
      // rows of a later pass write after this one: the later row of a
      // colliding pair still wins
      b.rk.pos = a.rk.pos + m0;
      b.rk.bt = a.rk.bt + (size_t)m0 * a.rk.max_blocks;
      b.rk.q_out = (char*)a.rk.q_out + (size_t)m0 * a.rk.Hq * a.rk.D * xe;
    }
  };
  if constexpr (EPI == EPI_ROPE_KV) {
    // fp16 projections on the fast layouts only (the caller falls back)
    if (act_dt != MK_DT_F16 || sc_dt != MK_DT_F16 || !fast) return MK_ERR_UNSUPPORTED;
  }
  {
    const int64_t pass = pass_rows<BITS, NMAT>(N, K, gs), tail = M % pass;
    if (M > pass && dot_eligible<BITS, NMAT>(a, fast, tail, act_dt, sc_dt)) {
      // us at 33 / 36 / 65 rows, all rows in one form -> this, q4 g64:
      // 2 x 14336 x 4096 36 / 35 / 53 -> 35 / 42 / 47, 6144 x 4096 18 / 18 / 22
      // -> 16 / 18 / 26, 4096 x 14336 35 / 36 / 67 -> 24 / 28 / 41
      rc = gemv_dispatch<BITS, NMAT, EPI>(a, M - tail, N, K, gs, act_dt, sc_dt, st, ws, ws_bytes,
                                          BITS == 4 && NMAT == 2 ? 32 : kGemmMinRows);
      if (rc != MK_OK) return rc;
      GemvArgs b = a;
      b.M = (int)tail;
      rows_from(b, M - tail);
      b.kw = dot_waves(K);
      return launch_dot<BITS, NMAT, EPI>(b, st);
    }
  }
  // The few-row kernel takes up to 32 rows a pass (8-bit codes: 16) of what
  // the v_dot2 kernel does not.  From kGemmMinRows rows one product of all
  // rows, unless two passes take less: few output rows over a long K leave the
  // product 64 workgroups (4096 x 14336 at 40 rows 66 us against 34; a pass of
  // 17-32 rows takes 6.5 us + 0.14 ns per 1000 weights for q4 fp16, 6.3 + 0.175
  // for bf16, and 3.3 for the sum of K slices).  17-32 rows over 8-bit codes, fp16:
  // the product or the tile kernel below, whichever is estimated to take less (2
  // x 14336 x 4096 at 32 rows 40 us and 65, 2 x 4096 x 4096 23.3 and 18.9, 33000 x
  // 1024 23.2 and 27.7), and two passes where neither applies (4096 x 4064 19.0,
  // the MFMA kernel 23.2; not with K slices: 4096 x 4128 25.6 against 24.4).  bf16:
  // the product for pairs (two passes 66), two passes for one matrix (4096 x
  // 14336 44 against 78).
  {
    constexpr int64_t kPass = BITS == 4 ? 32 : 16;
    const int64_t tiles = (N + 15) / 16, cus = device_cu_count();
    // a few of the batch sizes on one round of the K-split kernel, which has no sum
    // of slices (4096 x 6144 at 8 rows 9.2 against 10.5, at 16 10.6 against 10.9; 4096
    // x 8192 at 6 10.6 against 11.5, at 12 11.8 against 11.9; 2560 x 6912, not in
    // whole 512s, at 17 12.9 against 14.4; 4096 x 14336 at 6 15.2 against 15.1; two
    // rounds 5120 x 8192 at 6 18.2 against 13.0)
    const int64_t most = K > 12288 ? 0 : K % 512 != 0 ? 20 : K <= 6144 ? 16 : K <= 11264 ? 12 : 8;
    const bool ksplit = NMAT == 1 && K > 4096 && M >= kXkMinRows && M <= most &&
                        tiles <= cus && 2 * tiles > cus && xk_eligible<BITS, NMAT>(a, 1, act_dt, sc_dt);
    // rows of more than 4096 k, not in whole 512s (the few-row kernel's slices are
    // uneven there and its scales come one by one): up to 8 rows by the MFMA kernel,
    // which has no sum of slices (q4 fp16 at 5 rows 4096 x 11008 13.6 against 16.3,
    // 4096 x 5056 9.5 against 11.2, 3072 x 9984 12.1 against 13.7, but 1024 x 11008
    // 12.5 against 9.4; q8 4096 x 11008 18.1 against 20.1, 4096 x 8256 17.3 against
    // 16.9; bf16 q4 16.5 against 16.1)
    const bool uneven = NMAT == 1 && fast && K > 4096 && K % 512 != 0 && M <= 8 && 2 * tiles > cus &&
                        (BITS == 4 ? act_dt == MK_DT_F16 : K > 10240);
    // short rows of few outputs: the few-row kernel's waves have 512 k each, the
    // kernels below share a row among more (2048 x 512, us: q4 fp16 at 17 rows 3.2
    // against 4.6, q8 fp16 at 8 rows 3.3 against 4.0, q8 bf16 at 32 rows 6.6 against
    // 8.6; 2 x 2048 x 512 q4 fp16 at 17 rows 4.3 against 6.3; 2 x 8192 x 512 bf16 6.9
    // against 6.0; 2 x 4864 x 896 at 17 rows 7.2 against 8.9)
    const int64_t few_rows = BITS == 8 || act_dt == MK_DT_F16 ? 32 : 16;
    const bool brief = fast && ((K <= 512 && tiles <= 128 && M <= few_rows) ||
                                (NMAT == 2 && K < 1024 && K % 512 != 0 && M >= 17 && M <= 32 &&
                                 tile_eligible<NMAT>(a, act_dt, sc_dt)));
    const bool few = M <= 2 * kPass && !ksplit && !uneven && !brief && !dot_eligible<BITS, NMAT>(a, fast, M, act_dt, sc_dt) &&
                     (EPI != EPI_ROPE_KV || act_dt == MK_DT_F16) &&
                     few_ok<BITS, NMAT>(a, M < kPass ? M : kPass, gs, sc_dt, ws_bytes);
    const bool wide8 = BITS == 8 && M > kPass;
    const bool few_rest = M > 32 && M <= 48 && few_ok<BITS, NMAT>(a, M - 32, gs, sc_dt, ws_bytes);
    if constexpr (EPI != EPI_ROPE_KV) {
      const bool tile = tile_eligible<NMAT>(a, act_dt, sc_dt);
      bool product = (M >= product_rows || (wide8 && (NMAT == 2 || tile))) && M < (1LL << 24) &&
                     gemm_rows_ok<BITS, NMAT>(a, M, gs);
      if (product && M < kGemmMinRows && tile && !(BITS == 4 && few)) {
        // (short rows: the estimate leaves out what a second round of workgroups
        // takes to start.  Product and tile kernel, us at 32 rows: 2 x 20480 x 1024
        // 24.1 and 22.8, 2 x 10400 x 1024 12.7 and 15.0, 2 x 5632 x 1024 9.6 and
        // 10.9, 2 x 14336 x 512 9.5 and 10.0, at 17 rows 9.5 and 8.7)
        const bool rounds = NMAT * N > 128 * cus;
        const float by = K > 1024 ? 0.9f : rounds ? 1.2f : K <= 512 ? 1.05f : 0.95f;
        const float us = by * gemm_rows_us(BITS, NMAT, (int)M, a.N, a.K);
        product = us < tile_rows_us<BITS, NMAT>(M, N, K);
      } else if (product && few && M <= kPass) {
        product = false;  // one pass
      } else if (product && few && M >= kGemmMinRows && BITS == 4 && NMAT == 1) {
        const float weights = (float)N * (float)K, sum = K > 4096 ? 3.3f : 0.0f;
        const float pass = act_dt == MK_DT_F16 ? 6.5f + 1.4e-7f * weights + sum : 6.3f + 1.75e-7f * weights + sum;
        product = gemm_rows_us(BITS, NMAT, (int)M, a.N, a.K) < 2.0f * pass;
      }
      if (BITS == 8 && NMAT == 1 && product && few_rest && tile) {
        // 33-48 rows: the tile kernel and a few-row pass (5-6 us + 0.24 ns per
        // 1000 weights, 3.3 for the sum of K slices) where the product's
        // workgroups are few: 4096 x 14336 at 40 rows 63 us against 70, 4096 x
        // 11008 50 against 67, but 2048 x 2048 13.4 against 12.1
        const float pass = 4.9f + 0.07f * (float)(M - 32) + 2.4e-7f * (float)N * (float)K + (K > 4096 ? 3.3f : 0.0f);
        if (tile_rows_us<BITS, NMAT>(32, N, K) + pass < 0.9f * gemm_rows_us(BITS, NMAT, (int)M, a.N, a.K)) {
          rc = gemv_dispatch<BITS, NMAT, EPI>(a, 32, N, K, gs, act_dt, sc_dt, st, ws, ws_bytes);
          GemvArgs b = a;
          rows_from(b, 32);
          return rc != MK_OK ? rc : gemv_dispatch<BITS, NMAT, EPI>(b, M - 32, N, K, gs, act_dt, sc_dt, st, ws, ws_bytes);
        }
      }
      if (product) {
        GemvArgs b = a;
        b.M = (int)M;
        return launch_gemm_rows<BITS, NMAT, NMAT == 1 ? EPI_RESIDUAL : EPI>(b, act_dt, sc_dt, st);
      }
    }
    if (few && !(wide8 && act_dt == MK_DT_F16 && (tile_eligible<NMAT>(a, act_dt, sc_dt) || K > 4096))) {
      for (int64_t m0 = 0; m0 < M && rc == MK_OK; m0 += kPass) {
        GemvArgs b = a;
        b.M = (int)(M - m0 < kPass ? M - m0 : kPass);
        rows_from(b, m0);
        rc = launch_few<BITS, NMAT, EPI == EPI_NONE ? EPI_RESIDUAL : EPI>(b, act_dt, ws, st);
      }
      return rc;
    }
  }
  int64_t m_done = 0;
  // up to 32 rows at a time through the K-split kernel (ksplit, and long rows
  // without a workspace)
  if constexpr (NMAT == 1) {
    if (M - m_done >= kXkMinRows && xk_eligible<BITS, NMAT>(a, 1, act_dt, sc_dt)) {
      while (M - m_done >= kXkMinRows && rc == MK_OK) {
        GemvArgs b = a;
        int64_t mrows = (M - m_done) < 32 ? (M - m_done) : 32;
        if (mrows > 16 && !xk_eligible<BITS, NMAT>(a, 2, act_dt, sc_dt)) mrows = 16;
        b.M = (int)mrows;
        rows_from(b, m_done);
        rc = mrows > 16 ? launch_xk<2, EPI>(b, st) : launch_xk<1, EPI>(b, st);
        m_done += mrows;
      }
    }
  }
  // 17-32 rows at a time through the two-column-tile kernel, the rest below
  if (tile_eligible<NMAT>(a, act_dt, sc_dt)) {
    while (M - m_done >= 17 && rc == MK_OK) {
      GemvArgs b = a;
      const int64_t mrows = (M - m_done) < 32 ? (M - m_done) : 32;
      b.M = (int)mrows;
      rows_from(b, m_done);
      rc = launch_tile<BITS, NMAT, 2, EPI>(b, st);
      m_done += mrows;
    }
  }
  const int64_t mblocks = (M - m_done + 15) / 16;
  for (int64_t mb = 0; mb < mblocks && rc == MK_OK; ++mb) {
    GemvArgs b = a;
    const int64_t m0 = m_done + mb * 16;
    const int64_t mrows = (M - m0) < 16 ? (M - m0) : 16;
    b.M = (int)mrows;
    rows_from(b, m0);
    if (dot_eligible<BITS, NMAT>(b, fast && mk_aligned(b.x, 16), mrows, act_dt, sc_dt)) {
      b.kw = dot_waves(K);
      rc = launch_dot<BITS, NMAT, EPI>(b, st);
    } else if constexpr (EPI == EPI_ROPE_KV) {
      b.kw = choose_kw(N, K, F::KC);
      rc = launch_fast<BITS, f16, f16, true, NMAT, EPI>(b, gpc, st);
    } else if (fast) {
      b.kw = choose_kw(N, K, F::KC);
      if (act_dt == MK_DT_F16 && sc_dt == MK_DT_F16)
        rc = launch_fast<BITS, f16, f16, true, NMAT, EPI>(b, gpc, st);
      else if (act_dt == MK_DT_F16)
        rc = launch_fast<BITS, f16, float, false, NMAT, EPI>(b, gpc, st);
      else if (sc_dt == MK_DT_F16)
        rc = launch_fast<BITS, bf16, f16, false, NMAT, EPI>(b, gpc, st);
      else
        rc = launch_fast<BITS, bf16, float, false, NMAT, EPI>(b, gpc, st);
    } else {
      b.M = (int)mrows;
      if (act_dt == MK_DT_F16 && sc_dt == MK_DT_F16)
        rc = launch_generic<BITS, f16, f16, NMAT, EPI>(b, (int)gs, st);
      else if (act_dt == MK_DT_F16)
        rc = launch_generic<BITS, f16, float, NMAT, EPI>(b, (int)gs, st);
      else if (sc_dt == MK_DT_F16)
        rc = launch_generic<BITS, bf16, f16, NMAT, EPI>(b, (int)gs, st);
      else
        rc = launch_generic<BITS, bf16, float, NMAT, EPI>(b, (int)gs, st);
    }
  }
  return rc;
}

template <int BITS>
int matvec_entry(const void* x, const uint8_t* w, const void* s, const void* z, const void* residual,
                 void* y_mm, void* y_out, int64_t M, int64_t N, int64_t K, int64_t gs, int act_dt,
                 int sc_dt, void* stream, void* ws = nullptr, size_t ws_bytes = 0) {
  GemvArgs a = {};
  a.x = x;
  a.w[0] = a.w[1] = w;
  a.s[0] = a.s[1] = s;
  a.z[0] = a.z[1] = z;
  a.residual = residual;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (residual) {
    MK_REQUIRE(y_out);
    a.y0 = y_mm;
    a.y1 = y_out;
    return gemv_dispatch<BITS, 1, EPI_RESIDUAL>(a, M, N, K, gs, act_dt, sc_dt, st, (float*)ws, ws_bytes);
  }
  void* y = y_out ? y_out : y_mm;
  MK_REQUIRE(y);
  a.y0 = y;
  int rc = gemv_dispatch<BITS, 1, EPI_NONE>(a, M, N, K, gs, act_dt, sc_dt, st, (float*)ws, ws_bytes);
  if (rc == MK_OK && y_mm && y_out && y_mm != y_out) {
    hipError_t e = hipMemcpyAsync(y_mm, y_out, (size_t)M * N * 2, hipMemcpyDeviceToDevice, st);
    if (e != hipSuccess) return -(int)e - 1000;
  }
  return rc;
}

template <int BITS>
int gate_up_entry(const void* x, const uint8_t* wg, const uint8_t* wu, const void* sg,
                  const void* su, const void* zg, const void* zu, void* gate_out, void* up_out,
                  void* mlp_out, int64_t M, int64_t N, int64_t K, int64_t gs, int act_dt,
                  int sc_dt, void* stream) {
  MK_REQUIRE(gate_out || up_out || mlp_out);
  GemvArgs a = {};
  a.x = x;
  a.w[0] = wg;
  a.w[1] = wu;
  a.s[0] = sg;
  a.s[1] = su;
  a.z[0] = zg;
  a.z[1] = zu;
  a.y0 = gate_out;
  a.y1 = up_out;
  a.y2 = mlp_out;
  return gemv_dispatch<BITS, 2, EPI_GATE_UP>(a, M, N, K, gs, act_dt, sc_dt,
                                             reinterpret_cast<hipStream_t>(stream));
}

// Residual add + RMSNorm + gate/up (+ SwiGLU) of one MLP block: one launch
// (the norm as the dot kernel's prologue) for an M = 1 fp16 q4 decode row the
// dot kernel takes, else the norm kernel and then the gate/up launch (q8's
// doubled code registers leave no room for the prologue's operands).
template <int BITS>
int norm_gate_up_entry(const void* x, const void* residual, const void* norm_w, float eps, const uint8_t* wg,
                       const uint8_t* wu, const void* sg, const void* su, const void* zg, const void* zu,
                       void* z_out, void* normed_out, void* gate_out, void* up_out, void* mlp_out, int64_t M,
                       int64_t N, int64_t K, int64_t gs, int act_dt, int sc_dt, int nw_dt, void* stream) {
  MK_REQUIRE(x && residual && norm_w && z_out && wg && wu && sg && su);
  MK_REQUIRE(gate_out || up_out || mlp_out);
  MK_REQUIRE(M >= 0 && N > 0 && K > 0 && gs > 0 && N < (1LL << 31) && K < (1LL << 31));
  MK_REQUIRE(act_dt == MK_DT_F16 || act_dt == MK_DT_BF16);
  MK_REQUIRE(sc_dt == MK_DT_F16 || sc_dt == MK_DT_F32);
  MK_REQUIRE(nw_dt == MK_DT_F16 || nw_dt == MK_DT_BF16 || nw_dt == MK_DT_F32);
  if (M == 0) return MK_OK;
  GemvArgs a = {};
  a.x = x;
  a.w[0] = wg;
  a.w[1] = wu;
  a.s[0] = sg;
  a.s[1] = su;
  a.z[0] = zg;
  a.z[1] = zu;
  a.y0 = gate_out;
  a.y1 = up_out;
  a.y2 = mlp_out;
  bool fast;
  gemv_prepare<BITS, 2>(a, N, K, gs, &fast);
  {
    // K <= 8192: the row fits two 16-byte chunks per thread of the workgroup
    if (nw_dt == MK_DT_F16 && K <= 4 * 2048 && M == 1 && dot_eligible<BITS, 2>(a, fast, M, act_dt, sc_dt) &&
        mk_aligned(residual, 16) &&
        mk_aligned(norm_w, 16) && mk_aligned(z_out, 16) && (!normed_out || mk_aligned(normed_out, 16))) {
      a.M = 1;
      a.kw = dot_waves(K);
      a.nres = residual;
      a.nw = norm_w;
      a.zout = z_out;
      a.nout = normed_out;
      a.eps = eps;
      return launch_dot<BITS, 2, EPI_GATE_UP, true>(a, reinterpret_cast<hipStream_t>(stream));
    }
  }
  MK_REQUIRE(normed_out);  // the two-launch path passes the normalised rows through it
  const int rc = mk_residual_rms_norm(x, residual, norm_w, z_out, normed_out, M, K, eps, act_dt, nw_dt, stream);
  if (rc != MK_OK) return rc;
  return gate_up_entry<BITS>(normed_out, wg, wu, sg, su, zg, zu, gate_out, up_out, mlp_out, M, N, K, gs, act_dt,
                             sc_dt, stream);
}

// The whole MLP block: the front above, then down + residual z.
template <int BITS>
int mlp_block_entry(const void* x, const void* residual, const void* norm_w, float eps, const uint8_t* wg,
                    const uint8_t* wu, const uint8_t* wd, const void* sg, const void* su, const void* sd,
                    const void* zg, const void* zu, const void* zd, void* z_out, void* normed_out, void* mlp_out,
                    void* out, int64_t M, int64_t I, int64_t K, int64_t gs, int act_dt, int sc_dt, int down_sc_dt,
                    int nw_dt, void* ws, size_t ws_bytes, void* stream) {
  MK_REQUIRE(wd && sd && mlp_out && out);
  MK_REQUIRE(down_sc_dt == MK_DT_F16 || down_sc_dt == MK_DT_F32);
  MK_REQUIRE(ws_bytes == 0 || (ws && mk_aligned(ws, 16)));
  const int rc = norm_gate_up_entry<BITS>(x, residual, norm_w, eps, wg, wu, sg, su, zg, zu, z_out, normed_out, nullptr,
                                          nullptr, mlp_out, M, I, K, gs, act_dt, sc_dt, nw_dt, stream);
  if (rc != MK_OK) return rc;
  return matvec_entry<BITS>(mlp_out, wd, sd, zd, z_out, nullptr, out, M, K, I, gs, act_dt, down_sc_dt, stream, ws,
                            ws_bytes);
}

// RMSNorm + matvec: y = fp16(x * rsqrt(mean(x^2) + eps) * norm_w) . W^T.
// One launch (the norm as the dot kernel's prologue, no residual) for an
// M = 1 fp16 q4 row the dot kernel takes, else the norm kernel into
// normed_out and then the matvec.
template <int BITS>
int norm_matvec_entry(const void* x, const void* norm_w, float eps, const uint8_t* w, const void* s,
                      const void* z, void* normed_out, void* y, int64_t M, int64_t N, int64_t K, int64_t gs,
                      int act_dt, int sc_dt, int nw_dt, void* stream) {
  MK_REQUIRE(x && norm_w && w && s && y);
  MK_REQUIRE(M >= 0 && N > 0 && K > 0 && gs > 0 && N < (1LL << 31) && K < (1LL << 31));
  MK_REQUIRE(act_dt == MK_DT_F16 || act_dt == MK_DT_BF16);
  MK_REQUIRE(sc_dt == MK_DT_F16 || sc_dt == MK_DT_F32);
  MK_REQUIRE(nw_dt == MK_DT_F16 || nw_dt == MK_DT_BF16 || nw_dt == MK_DT_F32);
  if (M == 0) return MK_OK;
  GemvArgs a = {};
  a.x = x;
  a.w[0] = a.w[1] = w;
  a.s[0] = a.s[1] = s;
  a.z[0] = a.z[1] = z;
  a.y0 = y;
  bool fast;
  gemv_prepare<BITS, 1>(a, N, K, gs, &fast);
  if constexpr (BITS == 4) {
    // K <= 8192: the row fits two 16-byte chunks per thread of the workgroup
    if (nw_dt == MK_DT_F16 && K <= 4 * 2048 && M == 1 &&
        dot_eligible<BITS, 1>(a, fast && mk_aligned(x, 16), M, act_dt, sc_dt) &&
        mk_aligned(norm_w, 16) && (!normed_out || mk_aligned(normed_out, 16))) {
      a.M = 1;
      a.kw = dot_waves(K);
      a.nres = nullptr;
      a.nw = norm_w;
      a.zout = nullptr;
      a.nout = normed_out;
      a.eps = eps;
      return launch_dot<BITS, 1, EPI_NONE, true>(a, reinterpret_cast<hipStream_t>(stream));
    }
  }
  MK_REQUIRE(normed_out);  // the two-launch path passes the normalised rows through it
  const int rc = mk_rms_norm(x, norm_w, normed_out, M, K, eps, act_dt, nw_dt, stream);
  if (rc != MK_OK) return rc;
  return matvec_entry<BITS>(normed_out, w, s, z, nullptr, nullptr, y, M, N, K, gs, act_dt, sc_dt, stream);
}

// RMSNorm + qkv projection + split + RoPE + paged K/V write.  One launch
// (the NORM dot kernel with the EPI_ROPE_KV epilogue) for a q4 fp16 row with
// K <= 8192; otherwise the projection into qkv_scratch, then
// mk_qkv_rope_paged_update.
template <int BITS>
int norm_qkv_rope_entry(const void* x, const void* norm_w, float eps, const uint8_t* w, const void* s,
                        const void* z, void* qkv_scratch, void* normed_out, const float* cos_t,
                        const float* sin_t, const int32_t* positions, const int32_t* block_table, void* K_pages,
                        void* V_pages, void* q_out, int64_t M, int64_t Hq, int64_t Hkv, int64_t D, int64_t P,
                        int64_t max_blocks, int64_t num_pages, int64_t cos_rows, int64_t K, int64_t gs,
                        int act_dt, int sc_dt, int nw_dt, void* stream) {
  MK_REQUIRE(x && norm_w && w && s && qkv_scratch && cos_t && sin_t && positions && block_table && K_pages &&
             V_pages && q_out);
  MK_REQUIRE(M >= 0 && M < 65536 && Hq > 0 && Hkv > 0 && D > 0 && (D % 2) == 0 && P > 0 && max_blocks > 0 &&
             num_pages > 0 && cos_rows > 0 && K > 0 && gs > 0);
  MK_REQUIRE((Hq + 2 * Hkv) * D < (1LL << 31) && num_pages * P < (1LL << 31) && max_blocks * P < (1LL << 31));
  MK_REQUIRE(act_dt == MK_DT_F16 || act_dt == MK_DT_BF16);
  if (M == 0) return MK_OK;
  const int64_t N = (Hq + 2 * Hkv) * D;
  if constexpr (BITS == 4) {
    GemvArgs a = {};
    a.x = x;
    a.w[0] = a.w[1] = w;
    a.s[0] = a.s[1] = s;
    a.z[0] = a.z[1] = z;
    bool fast;
    gemv_prepare<BITS, 1>(a, N, K, gs, &fast);
    if (act_dt == MK_DT_F16 && sc_dt == MK_DT_F16 && nw_dt == MK_DT_F16 && K <= 4 * 2048 && M == 1 &&
        dot_eligible<BITS, 1>(a, fast && mk_aligned(x, 16), M, act_dt, sc_dt) && mk_aligned(norm_w, 16) &&
        (!normed_out || mk_aligned(normed_out, 16))) {
      a.M = 1;
      a.kw = dot_waves(K);
      a.nres = nullptr;
      a.nw = norm_w;
      a.zout = nullptr;
      a.nout = normed_out;
      a.eps = eps;
      a.rk = RopeKV{cos_t, sin_t, positions, block_table, K_pages, V_pages, q_out, (int)Hq, (int)Hkv, (int)D,
                    (int)P, (int)max_blocks, (int)num_pages, (int)cos_rows};
      return launch_dot<BITS, 1, EPI_ROPE_KV, true>(a, reinterpret_cast<hipStream_t>(stream));
    }
  }
  MK_REQUIRE(normed_out);  // the multi-launch paths pass the normalised rows through it
  if (act_dt == MK_DT_F16 && sc_dt == MK_DT_F16 && max_blocks * P < (1LL << 31)) {
    // the norm kernel, then the projection whose epilogue rotates and writes
    GemvArgs a = {};
    a.x = normed_out;
    a.w[0] = a.w[1] = w;
    a.s[0] = a.s[1] = s;
    a.z[0] = a.z[1] = z;
    a.rk = RopeKV{cos_t, sin_t, positions, block_table, K_pages, V_pages, q_out, (int)Hq, (int)Hkv, (int)D,
                  (int)P, (int)max_blocks, (int)num_pages, (int)cos_rows};
    GemvArgs probe = a;
    bool fast;
    gemv_prepare<BITS, 1>(probe, N, K, gs, &fast);
    // from kGemmMinRows rows on, one product of all rows and the update kernel
    // beat passes of 32 rows with the update in their epilogue (the same arithmetic,
    // fp32 sums in another order)
    const bool product = M >= kGemmMinRows && gemm_rows_ok<BITS, 1>(probe, M, gs);
    if (fast && !product) {
      int rc = mk_rms_norm(x, norm_w, normed_out, M, K, eps, act_dt, nw_dt, stream);
      if (rc != MK_OK) return rc;
      return gemv_dispatch<BITS, 1, EPI_ROPE_KV>(a, M, N, K, gs, act_dt, sc_dt, reinterpret_cast<hipStream_t>(stream));
    }
  }
  const int rc = norm_matvec_entry<BITS>(x, norm_w, eps, w, s, z, normed_out, qkv_scratch, M, N, K, gs, act_dt,
                                         sc_dt, nw_dt, stream);
  if (rc != MK_OK) return rc;
  return mk_qkv_rope_paged_update(qkv_scratch, cos_t, sin_t, positions, block_table, K_pages, V_pages, q_out, M, Hq,
                                  Hkv, D, P, max_blocks, num_pages, cos_rows, act_dt, stream);
}

}  // namespace

extern "C" {

int mk_q4_rmsnorm_qkv_rope_paged(const void* x, const void* norm_w, float eps, const uint8_t* w, const void* scales,
                                 const void* zeros, void* qkv_scratch, void* normed_out, const float* cos_t,
                                 const float* sin_t, const int32_t* positions, const int32_t* block_table,
                                 void* K_pages, void* V_pages, void* q_out, int64_t M, int64_t Hq, int64_t Hkv,
                                 int64_t D, int64_t page_size, int64_t max_blocks, int64_t num_pages,
                                 int64_t cos_rows, int64_t K, int64_t group_size, int act_dtype, int scale_dtype,
                                 int norm_w_dtype, void* stream) {
  return norm_qkv_rope_entry<4>(x, norm_w, eps, w, scales, zeros, qkv_scratch, normed_out, cos_t, sin_t, positions,
                                block_table, K_pages, V_pages, q_out, M, Hq, Hkv, D, page_size, max_blocks,
                                num_pages, cos_rows, K, group_size, act_dtype, scale_dtype, norm_w_dtype, stream);
}

int mk_q8_rmsnorm_qkv_rope_paged(const void* x, const void* norm_w, float eps, const uint8_t* w, const void* scales,
                                 const void* zeros, void* qkv_scratch, void* normed_out, const float* cos_t,
                                 const float* sin_t, const int32_t* positions, const int32_t* block_table,
                                 void* K_pages, void* V_pages, void* q_out, int64_t M, int64_t Hq, int64_t Hkv,
                                 int64_t D, int64_t page_size, int64_t max_blocks, int64_t num_pages,
                                 int64_t cos_rows, int64_t K, int64_t group_size, int act_dtype, int scale_dtype,
                                 int norm_w_dtype, void* stream) {
  return norm_qkv_rope_entry<8>(x, norm_w, eps, w, scales, zeros, qkv_scratch, normed_out, cos_t, sin_t, positions,
                                block_table, K_pages, V_pages, q_out, M, Hq, Hkv, D, page_size, max_blocks,
                                num_pages, cos_rows, K, group_size, act_dtype, scale_dtype, norm_w_dtype, stream);
}

int mk_q4_rmsnorm_matvec(const void* x, const void* norm_w, float eps, const uint8_t* w, const void* scales,
                         const void* zeros, void* normed_out, void* y, int64_t M, int64_t N, int64_t K,
                         int64_t group_size, int act_dtype, int scale_dtype, int norm_w_dtype, void* stream) {
  return norm_matvec_entry<4>(x, norm_w, eps, w, scales, zeros, normed_out, y, M, N, K, group_size, act_dtype,
                              scale_dtype, norm_w_dtype, stream);
}

int mk_q8_rmsnorm_matvec(const void* x, const void* norm_w, float eps, const uint8_t* w, const void* scales,
                         const void* zeros, void* normed_out, void* y, int64_t M, int64_t N, int64_t K,
                         int64_t group_size, int act_dtype, int scale_dtype, int norm_w_dtype, void* stream) {
  return norm_matvec_entry<8>(x, norm_w, eps, w, scales, zeros, normed_out, y, M, N, K, group_size, act_dtype,
                              scale_dtype, norm_w_dtype, stream);
}


int mk_q4_matvec(const void* x, const uint8_t* w, const void* scales, const void* zeros,
                 const void* residual, void* y_mm, void* y_out, int64_t M, int64_t N, int64_t K,
                 int64_t group_size, int act_dtype, int scale_dtype, void* stream) {
  return matvec_entry<4>(x, w, scales, zeros, residual, y_mm, y_out, M, N, K, group_size, act_dtype,
                         scale_dtype, stream);
}

int mk_q8_matvec(const void* x, const uint8_t* w, const void* scales, const void* zeros,
                 const void* residual, void* y_mm, void* y_out, int64_t M, int64_t N, int64_t K,
                 int64_t group_size, int act_dtype, int scale_dtype, void* stream) {
  return matvec_entry<8>(x, w, scales, zeros, residual, y_mm, y_out, M, N, K, group_size, act_dtype,
                         scale_dtype, stream);
}

size_t mk_matvec_workspace_bytes(int64_t M, int64_t N, int64_t K) { return few_workspace_bytes(M, N, K); }

int mk_q4_matvec_ws(const void* x, const uint8_t* w, const void* scales, const void* zeros, const void* residual,
                    void* y_mm, void* y_out, int64_t M, int64_t N, int64_t K, int64_t group_size, int act_dtype,
                    int scale_dtype, void* workspace, size_t workspace_bytes, void* stream) {
  MK_REQUIRE(workspace_bytes == 0 || (workspace && mk_aligned(workspace, 16)));
  return matvec_entry<4>(x, w, scales, zeros, residual, y_mm, y_out, M, N, K, group_size, act_dtype, scale_dtype,
                         stream, workspace, workspace_bytes);
}

int mk_q8_matvec_ws(const void* x, const uint8_t* w, const void* scales, const void* zeros, const void* residual,
                    void* y_mm, void* y_out, int64_t M, int64_t N, int64_t K, int64_t group_size, int act_dtype,
                    int scale_dtype, void* workspace, size_t workspace_bytes, void* stream) {
  MK_REQUIRE(workspace_bytes == 0 || (workspace && mk_aligned(workspace, 16)));
  return matvec_entry<8>(x, w, scales, zeros, residual, y_mm, y_out, M, N, K, group_size, act_dtype, scale_dtype,
                         stream, workspace, workspace_bytes);
}

int mk_q4_gate_up(const void* x, const uint8_t* w_gate, const uint8_t* w_up, const void* s_gate,
                  const void* s_up, const void* z_gate, const void* z_up, void* gate_out,
                  void* up_out, void* mlp_out, int64_t M, int64_t N, int64_t K,
                  int64_t group_size, int act_dtype, int scale_dtype, void* stream) {
  return gate_up_entry<4>(x, w_gate, w_up, s_gate, s_up, z_gate, z_up, gate_out, up_out, mlp_out,
                          M, N, K, group_size, act_dtype, scale_dtype, stream);
}

int mk_q8_gate_up(const void* x, const uint8_t* w_gate, const uint8_t* w_up, const void* s_gate,
                  const void* s_up, const void* z_gate, const void* z_up, void* gate_out,
                  void* up_out, void* mlp_out, int64_t M, int64_t N, int64_t K,
                  int64_t group_size, int act_dtype, int scale_dtype, void* stream) {
  return gate_up_entry<8>(x, w_gate, w_up, s_gate, s_up, z_gate, z_up, gate_out, up_out, mlp_out,
                          M, N, K, group_size, act_dtype, scale_dtype, stream);
}

int mk_q4_rmsnorm_gate_up(const void* x, const void* residual, const void* norm_w, float eps,
                          const uint8_t* w_gate, const uint8_t* w_up, const void* s_gate, const void* s_up,
                          const void* z_gate, const void* z_up, void* z_out, void* normed_out, void* gate_out,
                          void* up_out, void* mlp_out, int64_t M, int64_t N, int64_t K, int64_t group_size,
                          int act_dtype, int scale_dtype, int norm_w_dtype, void* stream) {
  return norm_gate_up_entry<4>(x, residual, norm_w, eps, w_gate, w_up, s_gate, s_up, z_gate, z_up, z_out,
                               normed_out, gate_out, up_out, mlp_out, M, N, K, group_size, act_dtype, scale_dtype,
                               norm_w_dtype, stream);
}

int mk_q8_rmsnorm_gate_up(const void* x, const void* residual, const void* norm_w, float eps,
                          const uint8_t* w_gate, const uint8_t* w_up, const void* s_gate, const void* s_up,
                          const void* z_gate, const void* z_up, void* z_out, void* normed_out, void* gate_out,
                          void* up_out, void* mlp_out, int64_t M, int64_t N, int64_t K, int64_t group_size,
                          int act_dtype, int scale_dtype, int norm_w_dtype, void* stream) {
  return norm_gate_up_entry<8>(x, residual, norm_w, eps, w_gate, w_up, s_gate, s_up, z_gate, z_up, z_out,
                               normed_out, gate_out, up_out, mlp_out, M, N, K, group_size, act_dtype, scale_dtype,
                               norm_w_dtype, stream);
}

int mk_q4_mlp_block(const void* x, const void* residual, const void* norm_w, float eps, const uint8_t* w_gate,
                    const uint8_t* w_up, const uint8_t* w_down, const void* s_gate, const void* s_up,
                    const void* s_down, const void* z_gate, const void* z_up, const void* z_down, void* z_out,
                    void* normed_out, void* mlp_out, void* out, int64_t M, int64_t I, int64_t K, int64_t group_size,
                    int act_dtype, int scale_dtype, int down_scale_dtype, int norm_w_dtype, void* workspace,
                    size_t workspace_bytes, void* stream) {
  return mlp_block_entry<4>(x, residual, norm_w, eps, w_gate, w_up, w_down, s_gate, s_up, s_down, z_gate, z_up, z_down,
                            z_out, normed_out, mlp_out, out, M, I, K, group_size, act_dtype, scale_dtype,
                            down_scale_dtype, norm_w_dtype, workspace, workspace_bytes, stream);
}

int mk_q8_mlp_block(const void* x, const void* residual, const void* norm_w, float eps, const uint8_t* w_gate,
                    const uint8_t* w_up, const uint8_t* w_down, const void* s_gate, const void* s_up,
                    const void* s_down, const void* z_gate, const void* z_up, const void* z_down, void* z_out,
                    void* normed_out, void* mlp_out, void* out, int64_t M, int64_t I, int64_t K, int64_t group_size,
                    int act_dtype, int scale_dtype, int down_scale_dtype, int norm_w_dtype, void* workspace,
                    size_t workspace_bytes, void* stream) {
  return mlp_block_entry<8>(x, residual, norm_w, eps, w_gate, w_up, w_down, s_gate, s_up, s_down, z_gate, z_up, z_down,
                            z_out, normed_out, mlp_out, out, M, I, K, group_size, act_dtype, scale_dtype,
                            down_scale_dtype, norm_w_dtype, workspace, workspace_bytes, stream);
}

}  // extern "C"
