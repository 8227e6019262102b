// Quantized matvecs of a few activation rows (a decode batch, M <= 32): the
// activation-stationary form of the matrix product.
//
// At these sizes the work is the stream of codes, and what costs is anything
// that keeps a CU from having many of them in flight.  A workgroup of up to 8
// waves covers up to 4096 k; wave w keeps the activations of its 512 k in
// registers as MFMA operands (64 per 16 columns) and walks the workgroup's
// run of 16-row weight tiles.  Per tile and matrix (a "unit") a lane loads 16
// bytes of codes for each 128 k (32 k of row r; 32 bytes for 8 bits) and the
// groups of its row and k, and the units run in a ring of DU register buffers
// -- 40 KB in flight per CU and unit -- without a barrier: the waves meet once
// per ring turn, when their partial tiles are added through LDS.
// Longer rows are cut into K slices of at most 4096 k whose fp32 sums go to a
// workspace, added (with the residual) by a second kernel.
//
// The activations come to LDS as whole 1 KB runs (global_load_lds) and from
// there to the operand layout; read straight into it, every load instruction
// touches 64 separate 64-byte pieces.
//
// Measured, us in a graph over weights that no cache holds, the kernels before
// -> this (gate/up + SwiGLU 2 x 14336 x 4096 | 4096 x 14336 | 6144 x 4096 | 4096 x
// 4096, g64):
//   q4 fp16  8 rows  19.3 -> 19.7 | 16.2 -> 14.9 |  9.1 ->  8.2 |  7.0 -> 5.5
//   q4 fp16 32 rows  26.6 -> 23.4 | 33.2 -> 17.9 | 14.8 -> 11.1 | 12.7 -> 8.5
//   q4 bf16  4 rows  34.9 -> 24.7 | 20.0 -> 17.5 | 11.9 ->  9.2 |  8.1 -> 6.6
//   q4 bf16 32 rows  77.9 -> 28.9 | 50.1 -> 20.4 | 30.4 -> 12.3 | 18.2 -> 8.6
//   q8 fp16  8 rows  46.0 -> 31.9 | 26.6 -> 22.1 | 15.6 -> 11.2 |  9.3 -> 8.4
// What is left is the stream: 128256 x 4096 at 8 rows takes 68 us (78 before),
// 60 without the unpacking and products, 65 without the turns' barriers.
#include "common.h"
#include "gemv_common.h"

using namespace mkq;

namespace {

constexpr int FKW = 512;        // k per wave
constexpr int FB = FKW / 128;   // 128-k blocks per wave
constexpr int FMAXW = 8;        // waves per workgroup

// LDS: 16 activation rows of FKW halves per wave, then reused for the partial
// tiles, [2 turns][DU units][MT][waves][64] f32x4
// (XL rows of activations: one turn behind them)
constexpr size_t few_lds_bytes(int nw, int mt, int du, int xl) {
  if (xl) return (size_t)nw * xl * FKW * 2 + (size_t)du * nw * 64 * sizeof(f32x4);
  const size_t x = (size_t)nw * 16 * FKW * 2, red = (size_t)2 * du * mt * nw * 64 * sizeof(f32x4);
  return x > red ? x : red;
}

// k of lane column kb in block j (32 consecutive ones), from the wave's first:
// q4 lanes hold 64 consecutive k of each pair of blocks, q8 lanes 32 of each
// block, so that either way a load instruction touches whole 128-byte lines
// of its 16 rows (q4 half lines, as 32 k of each block: 79 us where this takes
// 72, 128256 x 4096 at 8 rows)
template <int BITS>
__device__ __forceinline__ int lane_k(int j, int kb) {
  return BITS == 4 ? 256 * (j >> 1) + 64 * kb + 32 * (j & 1) : 128 * j + 32 * kb;
}

// Scales and zero points of a lane's row over the wave's 512 k.  LG 5, 6, 7
// (groups of 32, 64, 128): the row's run of 16, 8, 4 fp16 in whole vectors,
// the scales by the lanes below 32 and the zero points by the others -- half
// the load instructions -- brought to where they are used by permlane32_swap.
// LG 0: any power-of-two group >= 32, one value per block and lane.
template <int LG>
struct SzRun {
  static constexpr int DW = LG == 5 ? 8 : LG == 6 ? 4 : LG == 7 ? 2 : 2 * FB;
  static constexpr int LOADS = LG == 5 ? 2 : LG == 0 ? 2 * FB : 1;
  uint32_t d[DW];
};

// row pointers of the scales and zero points; vector runs start at group g0
template <int LG>
__device__ __forceinline__ void load_sz(SzRun<LG>& v, const f16* srow, const f16* zrow, int g0, const int* gb,
                                        bool upper) {
  if constexpr (LG == 0) {
#pragma unroll
    for (int j = 0; j < FB; ++j) {
      v.d[j] = *reinterpret_cast<const uint16_t*>(srow + gb[j]);
      v.d[FB + j] = *reinterpret_cast<const uint16_t*>(zrow + gb[j]);
    }
  } else {
    const f16* row = (upper ? zrow : srow) + g0;
    if constexpr (LG == 7) {
      const u32x2 t = ldg64(row);
      v.d[0] = t[0];
      v.d[1] = t[1];
    } else {
#pragma unroll
      for (int i = 0; i < SzRun<LG>::LOADS; ++i) {
        const u32x4 t = ldg128(row + 8 * i);
#pragma unroll
        for (int e = 0; e < 4; ++e) v.d[4 * i + e] = t[e];
      }
    }
  }
}

// lanes below 32: (scale dword lo, zero-point dword lo); the others: of hi
__device__ __forceinline__ u32x2 sz_swap(uint32_t lo, uint32_t hi) {
  const auto r = __builtin_amdgcn_permlane32_swap(lo, hi, false, false);
  return (u32x2){r[0], r[1]};
}

// (scale, zero point) of block j for lane column kb: entry lane_k >> LG of the
// run, found in dwords that differ by the upper bit of kb only (sz_swap's
// halves), then by the lower one
template <int BITS, int LG>
__device__ __forceinline__ void sz_at(const SzRun<LG>& v, int j, int kb, f16* s, f16* z) {
  if constexpr (LG == 0) {
    *s = bitcast<f16>((uint16_t)v.d[j]);
    *z = bitcast<f16>((uint16_t)v.d[FB + j]);
  } else {
    const int base = (lane_k<BITS>(j, 0) >> LG) / 2;  // first dword of the block's entries
    u32x2 u;
    int sh;
    if constexpr (BITS == 4 && LG == 5) {  // entries 2 kb + (j & 1): a dword per kb
      const u32x2 a = sz_swap(v.d[base], v.d[base + 2]), b = sz_swap(v.d[base + 1], v.d[base + 3]);
      u = kb & 1 ? b : a;
      sh = 16 * (j & 1);
    } else if constexpr ((BITS == 4 && LG == 6) || (BITS == 8 && LG == 5)) {  // entries kb
      u = sz_swap(v.d[base], v.d[base + 1]);
      sh = 16 * (kb & 1);
    } else {  // entries kb / 2, or one for all kb: in one dword
      u = sz_swap(v.d[base], v.d[base]);
      sh = (BITS == 4 && LG == 7) || (BITS == 8 && LG == 6) ? 16 * (kb >> 1) : 16 * ((lane_k<BITS>(j, 0) >> LG) & 1);
    }
    *s = bitcast<f16>((uint16_t)(u[0] >> sh));
    *z = bitcast<f16>((uint16_t)(u[1] >> sh));
  }
}

struct FewArgs {
  GemvArgs g;
  float* ws;       // K slices' sums [slices][M][N], or null: one slice, epilogue here
  int slices, nw;  // K slices, waves per workgroup
  int runs;        // workgroups (runs of tiles) per slice
  int tiles;       // 16-row tiles
};

// XL: one tile per workgroup, activations read from LDS as they are used (at
// most XL rows of them), so that two workgroups of 128 registers share a CU
// MAGIC: fp16 weights by the exponent trick, which holds a fractional zero
// point's part in fp16; otherwise (q - z) * s in fp32, rounded once
template <int BITS, typename AT, int NMAT, int MT, int DU, int LG, bool MAGIC, int EPI, int XL>
__global__ __launch_bounds__(64 * FMAXW) __attribute__((amdgpu_waves_per_eu(XL ? 4 : 2))) void gemv_few_kernel(
    const FewArgs fa) {
  static_assert(DU % NMAT == 0, "a ring turn holds whole tiles");
  static_assert(!XL || (MT == 1 && DU == NMAT), "XL: one tile");
  constexpr int XROWS = XL ? XL : 16;
  static_assert(!MAGIC || __is_same(AT, f16), "MAGIC unpacks to fp16");
  constexpr int WV = BITS == 4 ? 1 : 2;  // 16-byte code vectors per lane and block
  constexpr int RT = DU / NMAT;          // tiles per ring turn
  const GemvArgs& args = fa.g;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = fa.nw;
  const int M = args.M, N = args.N, K = args.K, G = args.G;
  const int r = lane & 15, kb = lane >> 4;
  const int slice = blockIdx.x / fa.runs, run = blockIdx.x - slice * fa.runs;
  // balanced runs: the first `rem` take one tile more
  const int per = fa.tiles / fa.runs, rem = fa.tiles - per * fa.runs;
  const int t_begin = run * per + min(run, rem);
  const int t_end = t_begin + per + (run < rem ? 1 : 0);
  const int k0 = (slice * nw + wave) * FKW;  // this wave's k (may start past K: zero activations)

  extern __shared__ __align__(16) uint8_t few_lds[];
  __shared__ int rk_slots[EPI == EPI_ROPE_KV ? kRopeRows : 1];
  __shared__ int rk_res[EPI == EPI_ROPE_KV ? kRopeRows : 1];
  __shared__ int rk_pos[EPI == EPI_ROPE_KV ? kRopeRows : 1];
  uint8_t* const xl = few_lds + wave * XROWS * FKW * 2;

  // Activation rows to LDS: lane l copies 16-byte chunk l ^ row of the row's 1
  // KB run to position l, so that an operand read's 16 rows fall into
  // different banks.  Chunks past K are not copied (and read as zero).
  auto copy_x = [&](int mt) {
    const int rows = min(XROWS, M - 16 * mt);
    for (int i = 0; i < rows; ++i) {
      const int k = k0 + 8 * (lane ^ i);
      if (k < K)
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void*)(reinterpret_cast<const AT*>(args.x) +
                                                            (size_t)(16 * mt + i) * K + k),
            (__attribute__((address_space(3))) void*)(xl + i * FKW * 2), 16, 0, 0);
    }
  };
  u32x4 xp[MT][XL ? 4 : 4 * FB];
  const int xr = r & (XROWS - 1);  // columns past XL repeat its rows (not stored)
  auto read_block = [&](int j, u32x4* x) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const u32x4 v =
          *reinterpret_cast<const u32x4*>(xl + xr * FKW * 2 + (((lane_k<BITS>(j, kb) / 8 + s) ^ xr) << 4));
      x[s] = k0 + lane_k<BITS>(j, kb) < K ? xperm<BITS, MAGIC>(v) : (u32x4){0u, 0u, 0u, 0u};
    }
  };
  auto read_x = [&](int mt) {
    if constexpr (!XL) {
#pragma unroll
      for (int j = 0; j < FB; ++j) read_block(j, &xp[mt][4 * j]);
    }
  };

  // lane offsets within a weight row: its code bytes of block j and its groups
  // there; blocks past K re-read the row's first (they meet zero activations)
  int cofs[FB], gb[FB];
#pragma unroll
  for (int j = 0; j < FB; ++j) {
    const int k = k0 + lane_k<BITS>(j, kb);
    const int kc = k < K ? k : 0;
    cofs[j] = kc * BITS / 8;
    gb[j] = kc >> args.lg;
  }
  const int g0 = k0 < K ? k0 >> args.lg : 0;  // LG > 0: K % FKW == 0, the wave's groups lie in the row
  const bool idle = LG > 0 && k0 >= K;        // LG > 0: nor is a wave partly past K; its sums are zero (LG 0: see block)
  const bool has_z = args.z[0] != nullptr;

  u32x4 w[DU][FB][WV];
  SzRun<LG> sz[DU];
  // unit u of the run: tile t_begin + u / NMAT, matrix u % NMAT; units past
  // the run re-read its last tile (their partial tiles are not used)
  auto issue = [&](int u, int slot, int q) {
    const int t = min(t_begin + u / NMAT, t_end - 1);
    const int n = min(16 * t + r, N - 1);
    const uint8_t* p = args.w[q] + (size_t)n * args.row_bytes;
#pragma unroll
    for (int j = 0; j < FB; ++j)
#pragma unroll
      for (int v = 0; v < WV; ++v) w[slot][j][v] = ldg128(p + cofs[j] + 16 * v);
    load_sz<LG>(sz[slot], reinterpret_cast<const f16*>(args.s[q]) + (size_t)n * G,
                reinterpret_cast<const f16*>(has_z ? args.z[q] : args.s[q]) + (size_t)n * G, g0, gb, lane >= 32);
  };
  constexpr int LOADS = FB * WV + SzRun<LG>::LOADS;  // vector loads per unit

  const uint32_t magic = in_vgpr(BITS == 4 ? 0x64006400u : 0x64646464u);
  const uint32_t magic_hi = in_vgpr(0x54005400u);

  copy_x(0);
  if constexpr (MT == 2) {
    // the second 16 columns pass through the same LDS
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    read_x(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    copy_x(1);
  }
  if constexpr (EPI == EPI_ROPE_KV) rope_fill_slots(args, rk_slots);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < DU; ++u) issue(u, u, u % NMAT);
  __builtin_amdgcn_sched_barrier(0);
  // the copies have landed when only the units' loads (all issued after
  // them, vmcnt retires in order; at most 63 can be told apart) are left
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(DU * LOADS < 63 ? DU * LOADS : 63) : "memory");
  read_x(MT - 1);
  if constexpr (!XL || EPI == EPI_ROPE_KV) lds_barrier();  // every wave has read its activations: LDS is free
  if constexpr (EPI == EPI_ROPE_KV) rope_resolve_slots(args, rk_slots, rk_res, rk_pos);

  // XL: the partial tiles lie past the activations, which others still read
  f32x4* const red = reinterpret_cast<f32x4*>(few_lds + (XL ? (size_t)nw * XL * FKW * 2 : 0));
  const int slab = DU * MT * nw * 64;
  const bool vec = (N & 3) == 0 && ((reinterpret_cast<uintptr_t>(args.y0) | reinterpret_cast<uintptr_t>(args.y1) |
                                     reinterpret_cast<uintptr_t>(args.y2) |
                                     reinterpret_cast<uintptr_t>(args.residual)) & 7) == 0;
  // block j of unit u against the activations at xp[.][x0]
  auto block = [&](int u, int j, f32x4* acc, int x0) {
    f16 sv, zv;
    sz_at<BITS, LG>(sz[u], j, kb, &sv, &zv);
    if (!has_z) zv = (f16)0.0f;
    if constexpr (LG == 0) {
      // blocks past K re-read real weights, which may be infinite once rounded:
      // times the zero activations that would be NaN
      const bool past = k0 + lane_k<BITS>(j, kb) >= K;
      sv = past ? (f16)0.0f : sv;
      zv = past ? (f16)0.0f : zv;
    }
    GpMagic gp;
    ExactGp<f16> ge;
    if constexpr (MAGIC) {
      gp = make_gp_magic(sv, zv);
    } else {
      ge = make_exact_gp<f16>(sv, zv);
    }
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      u32x4 a;
      if constexpr (BITS == 4) {
        if constexpr (MAGIC) a = dq4_magic(w[u][j][0][st], gp, magic, magic_hi);
        else a = dq_exact8<4, AT, f16>(w[u][j][0][st], 0u, ge);
      } else {
        const uint32_t u0 = w[u][j][st >> 1][(2 * st) & 3], u1 = w[u][j][st >> 1][(2 * st + 1) & 3];
        if constexpr (MAGIC) a = dq8_magic(u0, u1, gp, magic);
        else a = dq_exact8<8, AT, f16>(u0, u1, ge);
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt] = mfma_k32<AT>(a, xp[mt][x0 + st], acc[mt]);
    }
  };
  int turn = 0;
  for (int t0 = t_begin; t0 < t_end; t0 += RT, ++turn) {
    f32x4* const rb = red + (turn & 1) * slab;
    if constexpr (XL) {
      f32x4 acc[DU];
#pragma unroll
      for (int u = 0; u < DU; ++u) acc[u] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < FB; ++j) {
        read_block(j, xp[0]);
#pragma unroll
        for (int u = 0; u < DU; ++u) {
          // one block's operands at a time: its codes are not unpacked earlier
          // (registers), and are waited for here
#pragma unroll
          for (int v = 0; v < WV; ++v) asm volatile("" : "+v"(w[u][j][v]));
          block(u, j, &acc[u], 0);
          asm volatile("" : "+v"(acc[u]));
          __builtin_amdgcn_sched_barrier(0);
        }
      }
#pragma unroll
      for (int u = 0; u < DU; ++u) rb[(u * nw + wave) * 64 + lane] = idle ? (f32x4){0.f, 0.f, 0.f, 0.f} : acc[u];
    } else {
      // every buffer takes its next unit once it is used (unconditional loads:
      // the wait counts stay exact; past the run they re-read its last tile)
#pragma unroll
      for (int u = 0; u < DU; ++u) {
        f32x4 acc[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < FB; ++j) block(u, j, acc, 4 * j);
        __builtin_amdgcn_sched_barrier(0);
        issue((t0 - t_begin) * NMAT + u + DU, u, u % NMAT);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          rb[((u * MT + mt) * nw + wave) * 64 + lane] = idle ? (f32x4){0.f, 0.f, 0.f, 0.f} : acc[mt];
      }
    }
    lds_barrier();
    // wave i adds the partial tiles of every nw-th (tile, column tile) of the
    // turn; lane holds D[n = 4 kb + i][m = 16 mt + r].  The other buffer takes
    // the next turn's, and the barrier after it frees this one.
    for (int it = wave; it < RT * MT; it += nw) {
      const int tt = it / MT, mt = it - tt * MT;
      const int t = t0 + tt;
      if (t >= t_end) break;
      f32x4 v[NMAT];
#pragma unroll
      for (int q = 0; q < NMAT; ++q) {
        const f32x4* p = rb + ((tt * NMAT + q) * MT + mt) * nw * 64 + lane;
        v[q] = p[0];
        for (int i = 1; i < nw; ++i) v[q] += p[i * 64];
      }
      const int m = 16 * mt + r, nb = 16 * t + 4 * kb;
      if (m >= M) continue;
      if constexpr (EPI == EPI_ROPE_KV) {
        rope_kv_pair<true>(args, rk_res, m, nb, v[0][0], v[0][1], rk_pos);
        rope_kv_pair<true>(args, rk_res, m, nb + 2, v[0][2], v[0][3], rk_pos);
      } else if (EPI == EPI_RESIDUAL && fa.ws) {
        float* o = fa.ws + ((size_t)slice * M + m) * N + nb;
        if ((N & 3) == 0) {
          if (nb < N) *reinterpret_cast<f32x4*>(o) = v[0];
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (nb + i < N) o[i] = v[0][i];
        }
      } else {
        store_out4<AT, EPI>(args, vec, m, nb, v[0], v[NMAT - 1]);
      }
    }
  }
}

// sums of the K slices, in slice order, and the epilogue: 4 outputs a thread
template <typename AT>
__global__ __launch_bounds__(256) void gemv_slices_kernel(const GemvArgs args, const float* ws, int slices) {
  const int64_t total = (int64_t)args.M * args.N;
  const int64_t i0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i0 >= total) return;
  const int cnt = total - i0 < 4 ? (int)(total - i0) : 4;
  float v[4];
  if (cnt == 4 && (total & 3) == 0) {
    f32x4 a = *reinterpret_cast<const f32x4*>(ws + i0);
    for (int s = 1; s < slices; ++s) a += *reinterpret_cast<const f32x4*>(ws + s * total + i0);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = a[e];
  } else {
    for (int e = 0; e < cnt; ++e) {
      v[e] = ws[i0 + e];
      for (int s = 1; s < slices; ++s) v[e] += ws[s * total + i0 + e];
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (e >= cnt) break;
    if (args.residual) store_out<AT, EPI_RESIDUAL>(args, i0 + e, v[e], v[e]);
    else store_out<AT, EPI_NONE>(args, i0 + e, v[e], v[e]);
  }
}

struct FewPlan {
  int slices, nw, runs, tiles;
};
// K slices of at most FMAXW waves, and the workgroups of a slice: a CU's eight
// waves are one workgroup or, where rows are short, several.  (One a CU, then
// this, us at 8 rows of 33000 x 1024: q4 fp16 13.2 -> 7.9, bf16 18.0 -> 9.4, q8
// fp16 15.3 -> 10.6.  Pairs of 8-bit codes keep half of the waves idle rather
// than double them: 2 x 8192 x 2048 11.9, 12.4 with two workgroups.)
template <int BITS, int NMAT>
inline FewPlan few_plan(int N, int K, int cus) {
  FewPlan p;
  const int waves = (K + FKW - 1) / FKW;
  p.slices = (waves + FMAXW - 1) / FMAXW;
  p.nw = (waves + p.slices - 1) / p.slices;
  p.tiles = (N + 15) / 16;
  const int groups = cus * (BITS == 8 && NMAT == 2 && p.nw > 2 ? 1 : FMAXW / p.nw);
  const int runs = groups / p.slices > 0 ? groups / p.slices : 1;
  p.runs = p.tiles < runs ? p.tiles : runs;
  return p;
}

template <int BITS, typename AT, int NMAT, int MT, int DU, int LG, bool MAGIC, int EPI, int XL>
int few_launch(const GemvArgs& a, float* ws, hipStream_t st) {
  FewPlan p = few_plan<BITS, NMAT>(a.N, a.K, device_cu_count());
  if (XL) p.runs = p.tiles;
  FewArgs f;
  f.g = a;
  f.ws = p.slices > 1 ? ws : nullptr;
  f.slices = p.slices;
  f.nw = p.nw;
  f.runs = p.runs;
  f.tiles = p.tiles;
  gemv_few_kernel<BITS, AT, NMAT, MT, DU, LG, MAGIC, EPI, XL>
      <<<dim3((unsigned)(p.runs * p.slices)), dim3(64 * p.nw), few_lds_bytes(p.nw, MT, DU, XL), st>>>(f);
  MK_CHECK_LAUNCH();
  if (p.slices > 1) {
    const int64_t total = (int64_t)a.M * a.N;
    gemv_slices_kernel<AT><<<dim3((unsigned)((total + 1023) / 1024)), dim3(256), 0, st>>>(a, ws, p.slices);
    MK_CHECK_LAUNCH();
  }
  return MK_OK;
}

template <int BITS, typename AT, int NMAT, int EPI, int LG, bool MAGIC = __is_same(AT, f16)>
int few_columns(const GemvArgs& a, float* ws, hipStream_t st) {
  const FewPlan p = few_plan<BITS, NMAT>(a.N, a.K, device_cu_count());
  // tiles of a run: the longest, unless few are that long (4096 x 11008: 85 runs
  // of three slices, one of them 4 tiles, the others 3)
  const int run = p.tiles / p.runs + (4 * (p.tiles % p.runs) >= p.runs ? 1 : 0);
  // Up to 8 rows of the forms whose unpacking weighs most, while tiles are
  // few: one tile per workgroup (XL), two workgroups a CU.  Against the ring,
  // us: q8 fp16 at 8 rows 6144 x 4096 11.2 / 13.0, 14336 x 4096 19.5 / 19.7; bf16
  // q4 at 4 rows 8192 x 4096 9.3 / 9.8, 16384 x 4096 14.7 / 14.9, 2 x 8192 x 2048
  // 10.1 / 10.2.  The ring is ahead for fp16 q4 and q8 pairs, where tiles are
  // many, and for bf16 q4 at 5-8 rows of more than 20 waves a CU (12288 x 4096
  // 12.2 / 13.2, 4096 x 14336 17.9 / 19.4; 5120 x 5120 14.0 / 12.0) unless scales
  // come one by one (4096 x 11008 16.6 / 18.6).
  constexpr bool ONE = NMAT == 2 ? BITS == 4 && !__is_same(AT, f16) : BITS == 8 || !__is_same(AT, f16);
  if constexpr (ONE) {
    const int64_t ones = (int64_t)p.tiles * p.slices, cus = device_cu_count();
    const bool few_waves = BITS == 8 || NMAT == 2 || a.M <= 4 || LG == 0 || ones * p.nw <= 20 * cus;
    if (a.M <= 8 && ones <= 4 * cus && few_waves) {
      if (a.M <= 4) return few_launch<BITS, AT, NMAT, 1, NMAT, LG, MAGIC, EPI, 4>(a, ws, st);
      return few_launch<BITS, AT, NMAT, 1, NMAT, LG, MAGIC, EPI, 8>(a, ws, st);
    }
  }
  // The ring: a turn of one tile for pairs and for short odd runs, of two for
  // other runs.  What a turn holds past the run's end is fetched and multiplied
  // for nothing.  us at 5 rows of q4 fp16, turns of 1 / 2 / 4 tiles: 12288 x 4096
  // (runs of 3) 10.5 / 12.1 / 13.5, 20480 x 4096 (5) 15.1 / 15.7 / 19.7, 4096 x
  // 14336 (4 a slice) 14.9 / 14.8 / 16.6, 128256 x 4096 72 / 68 / 69; the pair 2 x
  // 11008 x 4096 with one tile 15.8, with two 19.4.
  const bool odd = (run & 1) && run <= 5;
  if (a.M <= 16) {
    if constexpr (NMAT == 1)
      if (odd) return few_launch<BITS, AT, NMAT, 1, 1, LG, MAGIC, EPI, 0>(a, ws, st);
    return few_launch<BITS, AT, NMAT, 1, 2, LG, MAGIC, EPI, 0>(a, ws, st);
  }
  if constexpr (BITS == 4) {
    if constexpr (NMAT == 1)
      if (odd) return few_launch<BITS, AT, NMAT, 2, 1, LG, MAGIC, EPI, 0>(a, ws, st);
    return few_launch<BITS, AT, NMAT, 2, 2, LG, MAGIC, EPI, 0>(a, ws, st);
  }
  return MK_ERR_UNSUPPORTED;
}

template <int BITS, typename AT, int NMAT, int EPI>
int few_groups(const GemvArgs& a, float* ws, hipStream_t st) {
  if constexpr (BITS == 4 && __is_same(AT, f16) && EPI != EPI_ROPE_KV) {
    // the layouts that were gemv_generic_kernel's alone: no weight in fewer bits
    // than there (2 x 14336 x 4064 at 32 rows 30.1 us, 28.4 by the exponent trick;
    // exact everywhere would cost 21.0 -> 23.4 at 8 rows of 2 x 14336 x 4096)
    if (a.K % QFmt<BITS>::KL) return few_columns<BITS, AT, NMAT, EPI, 0, false>(a, ws, st);
  }
  bool v16 = (a.G % 8) == 0 && (a.K % FKW) == 0, v8 = (a.G % 4) == 0 && (a.K % FKW) == 0;
  for (int t = 0; t < NMAT; ++t) {
    v16 = v16 && mk_aligned(a.s[t], 16) && mk_aligned(a.z[t], 16);
    v8 = v8 && mk_aligned(a.s[t], 8) && mk_aligned(a.z[t], 8);
  }
  if (a.lg == 5 && v16) return few_columns<BITS, AT, NMAT, EPI, 5>(a, ws, st);
  if (a.lg == 6 && v16) return few_columns<BITS, AT, NMAT, EPI, 6>(a, ws, st);
  if (a.lg == 7 && v8) return few_columns<BITS, AT, NMAT, EPI, 7>(a, ws, st);
  return few_columns<BITS, AT, NMAT, EPI, 0>(a, ws, st);
}

}  // namespace

namespace mkq {

size_t few_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M > 32 && M <= 68) M = 32;  // two passes (and up to 4 rows past them)
  if (M < 1 || M > 32 || N < 1 || K < 1 || N >= (1LL << 26) || K >= (1LL << 26)) return 0;
  const FewPlan p = few_plan<4, 1>((int)N, (int)K, device_cu_count());  // (slices do not depend on the form)
  return p.slices > 1 ? (size_t)p.slices * M * N * sizeof(float) : 0;
}

template <int BITS, int NMAT>
bool few_ok(const GemvArgs& a, int64_t M, int64_t gs, int sc_dt, size_t ws_bytes) {
  bool ok = sc_dt == MK_DT_F16 && a.lg >= 5 && (int64_t)1 << a.lg == gs && (a.K % 32) == 0 && M >= 1 &&
            M <= (BITS == 4 ? 32 : 16) && a.N < (1 << 26) && a.K < (1 << 26) && mk_aligned(a.x, 16) &&
            zeros_alike<NMAT>(a);
  for (int t = 0; t < NMAT; ++t) ok = ok && mk_aligned(a.w[t], 16);
  return ok && few_workspace_bytes(M, a.N, a.K) <= ws_bytes;
}

template <int BITS, int NMAT, int EPI>
int launch_few(const GemvArgs& a, int act_dt, float* ws, hipStream_t st) {
  if (act_dt == MK_DT_F16) return few_groups<BITS, f16, NMAT, EPI>(a, ws, st);
  if constexpr (EPI == EPI_ROPE_KV) return MK_ERR_UNSUPPORTED;  // fp16 caches only
  else return few_groups<BITS, bf16, NMAT, EPI>(a, ws, st);
}

#define MK_INST(B)                                                                                    \
  template bool few_ok<B, 1>(const GemvArgs&, int64_t, int64_t, int, size_t);                         \
  template bool few_ok<B, 2>(const GemvArgs&, int64_t, int64_t, int, size_t);                         \
  template int launch_few<B, 1, EPI_RESIDUAL>(const GemvArgs&, int, float*, hipStream_t);             \
  template int launch_few<B, 1, EPI_ROPE_KV>(const GemvArgs&, int, float*, hipStream_t);              \
  template int launch_few<B, 2, EPI_GATE_UP>(const GemvArgs&, int, float*, hipStream_t);
MK_INST(4)
MK_INST(8)
#undef MK_INST

}  // namespace mkq
