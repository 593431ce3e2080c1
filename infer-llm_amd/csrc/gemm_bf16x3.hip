// gemm_bf16x3.hip — out[m][n] = sum_k x[m][k] w[n][k] (+ residual[m][n]) in
// F32 on the bf16 matrix cores (v_mfma_f32_32x32x16_bf16): the products
// gemm_plan (gemm.hip) gives it instead of the F32 MFMA kernel.
//
// Why: the F32 matrix pipe ends at 157 TFLOP/s and the F32 kernel was at
// 92-97% of it. The bf16 pipe does 16 times as many flops, so an F32 product
// taken apart into bf16 ones still has 2.67 times the room.
//
// The split is exact: a float x is h + m + l, each the bf16 nearest to what
// is left (8 + 8 + 8 bits of significand, the residues exact in F32). Of the
// nine products of two such sums six are formed, all into one F32
// accumulator: h h, h m, m h, m m, h l, l h. The three left out are below
// 2^-26 of the product (2^-33 on average), under the rounding of an F32
// product. A 16-column MFMA rounds its sum once, so an output sees 6 roundings
// per 16 columns against 4 (16 x 16 x 4) of the F32 kernel's, most of them of
// small terms; the distance to a 64-bit sum, 2-norm relative, measured at
// normal data (x unit, w 0.02): k = 1024 4.9e-7 against 5.7e-7, k = 4096
// 1.0e-6 against 1.15e-6, k = 12288 1.8e-6 against 2.0e-6, less with K
// groups or splits (their partial sums are smaller); gemm_plan takes it only
// where the F32 kernel's plan has no more K ranges than this one's.
//
// Inputs that the split does not carry are found as they are split, or by the
// sums they leave, and the tile is formed again on F32 MFMAs. Looking at every
// split costs 0.6% of 4096-token products and 1-3% of those that the VALU
// bounds (4096 x 4096 at 509 tokens 99.5 -> 101.7 us); one look at the largest
// sum of a wave cost nothing, and missed a small row among ordinary ones and
// small floats against large ones. With every tile formed again 4096 x 4096 at
// 777 tokens takes 663 us against 159 (two MFMA tiles at a time 503, but 0.5%
// on every small product).
//
// Layout:
//   * A workgroup owns BW weight rows x BT tokens: WM wavefronts (per K
//     group), each TM x TN MFMA tiles of 32 x 32, K in steps of 32 columns.
//     Weights are the A operand and go from memory straight to the registers
//     of the one wave that multiplies them (no other wave has the same rows),
//     where they are split; tokens are the B operand of every wave, so they
//     are split once per workgroup and staged in LDS as three bf16 planes.
//     That halves the LDS traffic of staging both (a product reads 12 bytes
//     of pieces per 8 of F32).
//   * 32 x 32 x 16 rather than 16 x 16 x 32: a wave issues the 48 VALU
//     instructions of 8 floats' split between MFMAs, and four of them behind
//     one 32-cycle MFMA cost half a cycle (probe: 16.5 cycles per half MFMA),
//     while two behind a 16-cycle one cost 4.5.
//   * Step s multiplies while step s + 1 is split (weights in registers,
//     tokens to the other LDS buffer) and step s + 2 is loaded. The splits
//     are spread over the step's token tiles; the barrier stands before the
//     last one, so that its MFMAs cover the LDS reads of the next step.
//   * A staged token row is 64 bytes per plane, its four 16-byte pieces
//     XOR-ed with (row / 4) % 4: 16 lanes that read one piece of 16 rows, or
//     write four pieces of 4 rows, meet 64 different banks.
//   * KG = 2: two K groups of waves take alternate halves of a split's
//     columns with buffers of their own and add up through LDS. For few
//     tiles: a second wave per SIMD without a second launch's worth of
//     partials.
//   * Tile order and split K as in gemm.hip.
//
// Measured (us, F32 kernel -> this one, graph of calls, one box): 8B gate/up
// at 4096 tokens 2760 -> 1650 (250 TFLOP/s; the chip is then power-bound: the
// same loop on a quarter of the CUs runs 1.4 times as fast per CU), 8B q/o
// 930 -> 560, at 777 tokens 230 -> 141, at 128 tokens 39 -> 34; 0.6B q at
// 2048 tokens 74 -> 48, down at 2048 91 -> 75. Tried and not kept: the
// residues by v_dot2_f32_bf16 (28 VALU instructions instead of 44, but 15%
// slower: it shares the matrix pipe), load instructions over 16 rows x 64
// bytes with lane swaps (4-7% slower when power-bound, equal otherwise), two
// steps of loads in flight (equal).
#include "bf16x3.hpp"
#include "coherent.hpp"
#include "gemm.hpp"
#include "ikv_common.hpp"

#include <climits>

namespace {

using namespace ikv::pieces;

constexpr int BK = 32;      // columns per step: one MFMA's contraction
constexpr int kXcds = 8;
constexpr int kGroupT = 8;   // token tiles per group of the tile order
template <int TM, int TN, int WM, int KG, int MINW>
__global__ __launch_bounds__(WM * KG * 64, MINW) void gemm_bf16x3_kernel(
    const float *__restrict__ w, const float *__restrict__ x, float *out, const float *residual,
    int n_out, int k, int m, int tiles_t, int n_tiles, int n_split, float *part, int *counters) {
  constexpr int NT = WM * 64;       // threads of one K group
  constexpr int BW = 32 * TM * WM;  // weight rows per tile
  constexpr int BT = 32 * TN;       // tokens per tile
  constexpr int XI = BT * 4;        // staged items (8 columns of a token) per step
  static_assert(XI % NT == 0, "whole items per thread");
  constexpr int NX = XI / NT;
  static_assert(TN >= 2, "the step's barrier stands before its last token tile");
  constexpr int PLANE = BT * BK;    // bf16 of one piece of the token tile
  constexpr int LDS_HALFS = KG * 2 * 3 * PLANE;
  constexpr int XCH_HALFS = (KG - 1) * TM * TN * WM * 64 * 16 * 2;
  __shared__ int s_last;
  __shared__ int s_lost;
  __shared__ __attribute__((aligned(16))) unsigned short s_x[LDS_HALFS > XCH_HALFS ? LDS_HALFS : XCH_HALFS];

  const int b = static_cast<int>(blockIdx.x);
  const int per = (n_tiles + kXcds - 1) / kXcds;
  const int jb = b / kXcds;
  const int t = (b % kXcds) * per + jb % per;
  const int sp = jb / per;
  if (t >= n_tiles) return;
  const int tiles_w = n_tiles / tiles_t;
  // groups of kGroupT token tiles walked weight tile by weight tile
  const int grp = t / (kGroupT * tiles_w);
  const int first = grp * kGroupT;
  const int gsize = min(kGroupT, tiles_t - first);
  const int in_grp = t - grp * kGroupT * tiles_w;
  const int tt = first + in_grp % gsize, tw = in_grp / gsize;
  const int t0 = tt * BT, w0 = tw * BW;

  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wv / WM, wave = wv % WM;
  const int tid = threadIdx.x % NT;
  const int lane = threadIdx.x & 63;
  const int r32 = lane & 31;
  const int c2 = lane >> 5;

  const int all_steps = k / BK / KG;  // steps of a group, unsplit
  const int s_lo = static_cast<int>(static_cast<int64_t>(sp) * all_steps / n_split);
  const int s_hi = static_cast<int>(static_cast<int64_t>(sp + 1) * all_steps / n_split);
  const int n_steps = s_hi - s_lo;
  const int k_lo = (s_lo * KG + kg * n_steps) * BK;

  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(w + static_cast<size_t>(w0) * k), 0, min(BW, n_out - w0) * k * 4,
      ikv::kBufWord3);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(x + static_cast<size_t>(t0) * k), 0, min(BT, m - t0) * k * 4,
      ikv::kBufWord3);
  // MFMA half h (16 columns) of a step: lane (row r32, c2) holds columns
  // 16 h + 8 c2 .. + 7 of its row
  unsigned wof[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
    wof[i] = static_cast<unsigned>((((wave * TM + i) * 32 + r32) * k + 8 * c2) * 4);
  unsigned xof[NX];
  int xdst[NX];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int q = tid + NT * i;
    const int r = q >> 2, c = q & 3;  // piece c = 2 h + c2
    xof[i] = static_cast<unsigned>((r * k + 8 * c) * 4);
    xdst[i] = r * BK + 8 * (c ^ ((r >> 2) & 3));
  }
  int xsrc[2];  // + 32 * BK per token tile
#pragma unroll
  for (int h = 0; h < 2; ++h) xsrc[h] = r32 * BK + 8 * ((2 * h + c2) ^ ((r32 >> 2) & 3));

  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = floatx16{};

  floatx4 wr[2 * TM][2], xr[NX][2];  // step s + 1's floats, then step s + 2's
  Pieces a[2][TM][2];
  bf16x8 bc[2][3];
  unsigned lost = 0;  // what this thread's splits dropped
  if (threadIdx.x == 0) s_lost = 0;

  auto load_w = [&](int u, int st) {
    const int off = (k_lo + min(st, n_steps - 1) * BK) * 4;
    wr[u][0] = __builtin_amdgcn_raw_buffer_load_b128(rw, wof[u / 2] + 64 * (u & 1), off, 0);
    wr[u][1] = __builtin_amdgcn_raw_buffer_load_b128(rw, wof[u / 2] + 64 * (u & 1) + 16, off, 0);
  };
  auto load_x = [&](int i, int st) {
    const int off = (k_lo + min(st, n_steps - 1) * BK) * 4;
    xr[i][0] = __builtin_amdgcn_raw_buffer_load_b128(rx, xof[i], off, 0);
    xr[i][1] = __builtin_amdgcn_raw_buffer_load_b128(rx, xof[i] + 16, off, 0);
  };
  unsigned short *const sx = s_x + kg * (2 * 3 * PLANE);
  auto put_x = [&](int i, unsigned short *buf) {
    const Pieces s = split8<true>(xr[i][0], xr[i][1], lost);
#pragma unroll
    for (int p = 0; p < 3; ++p)
      *reinterpret_cast<bf16x8 *>(buf + p * PLANE + xdst[i]) = s.p[p];
  };
  auto read_x = [&](const unsigned short *buf, int j, bf16x8 (*d)[3]) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int p = 0; p < 3; ++p)
        d[h][p] = *reinterpret_cast<const bf16x8 *>(buf + p * PLANE + xsrc[h] + 32 * BK * j);
  };

  constexpr int U = NX + 2 * TM;  // conversion units of a step: token items, then weight halves
  auto step = [&](int s, auto par) {
    constexpr int P = decltype(par)::value;
    const unsigned short *cur = sx + P * (3 * PLANE);
    unsigned short *nbuf = sx + (P ^ 1) * (3 * PLANE);
    static_for<TN>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      constexpr bool more = j + 1 < TN;
      constexpr int lo = j * U / TN, hi = (j + 1) * U / TN;
      static_assert(more || lo >= NX, "token items are staged before the barrier");
      __builtin_amdgcn_sched_barrier(0);
      bf16x8 bn[2][3];
      if constexpr (more)
        read_x(cur, j + 1, bn);
      else
        read_x(nbuf, 0, bn);
#pragma unroll
      for (int u = lo; u < hi; ++u) {
        if (u < NX) {
          put_x(u, nbuf);
          load_x(u, s + 2);
        } else {
          const int v = u - NX;
          a[P ^ 1][v / 2][v & 1] = split8<true>(wr[v][0], wr[v][1], lost);
          load_w(v, s + 2);
        }
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int p = 0; p < 6; ++p)
#pragma unroll
          for (int i = 0; i < TM; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[P][i][h].p[kPieceA[p]], bc[h][kPieceB[p]],
                                                                 acc[i][j], 0, 0, 0);
      if constexpr (hi > lo) {
        constexpr int NM = 12 * TM;
        constexpr int per_mfma = ((hi - lo) * kSplitOps + NM - 1) / NM;
#pragma unroll
        for (int q = 0; q < NM; ++q) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);         // MFMA
          __builtin_amdgcn_sched_group_barrier(0x002, per_mfma, 0);  // VALU
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (j == TN - 2) __syncthreads();
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int p = 0; p < 3; ++p) bc[h][p] = bn[h][p];
    });
  };

#pragma unroll
  for (int i = 0; i < NX; ++i) load_x(i, 0);
#pragma unroll
  for (int i = 0; i < 2 * TM; ++i) load_w(i, 0);
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    put_x(i, sx);
    load_x(i, 1);
  }
#pragma unroll
  for (int i = 0; i < 2 * TM; ++i) {
    a[0][i / 2][i & 1] = split8<true>(wr[i][0], wr[i][1], lost);
    load_w(i, 1);
  }
  __syncthreads();
  read_x(sx, 0, bc);
  // Pairs of steps, so that nothing leaves the loop between a step's splits
  // and their use (the compiler would sink the splits behind the branch). The
  // last step splits and stages its own columns once more, unused.
  using P0 = std::integral_constant<int, 0>;
  using P1 = std::integral_constant<int, 1>;
  int s = 0;
  for (; s + 2 <= n_steps; s += 2) {
    step(s, P0{});
    step(s + 1, P1{});
  }
  if (s < n_steps) step(s, P0{});

  // (a token's pieces serve every wave: if any split dropped bits, all start
  // over)
  if (any_lost(lost) && lane == 0) s_lost = 1;
  __syncthreads();
  const bool redo = s_lost != 0;

  auto quad = [&](int i, int j, int q) {
    return floatx4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                   acc[i][j][4 * q + 3]};
  };
  const bool mine = KG == 1 || kg == 0;  // group 0 ends with the tile's sums
  if constexpr (KG > 1) {
    floatx4 *const xch = reinterpret_cast<floatx4 *>(s_x);  // (its readers are past the barrier above)
    if (!mine) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            xch[((((kg - 1) * TM + i) * TN + j) * 4 + q) * NT + tid] = quad(i, j, q);
    }
    __syncthreads();
    if (mine) {
#pragma unroll
      for (int g = 1; g < KG; ++g)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const floatx4 v = xch[((((g - 1) * TM + i) * TN + j) * 4 + q) * NT + tid];
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[i][j][4 * q + r] += v[r];
            }
    }
  }

  // Inputs the split does not carry: an infinite or NaN input (or one that
  // rounds to an infinite bf16) leaves NaNs in the wave's sums, and splits of
  // floats below 2^-109 may have dropped bits. The sums are then formed again
  // with F32 MFMAs from memory, 128 columns at a time.
  if (mine) {
    bool odd = redo;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) odd |= !(fabsf(acc[i][j][r]) < INFINITY);
    if (__builtin_amdgcn_ballot_w64(odd) != 0) {
      // (an MFMA tile at a time: this path is to cost the main loop no registers)
      const int kb1 = s_hi * KG * BK;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const unsigned wo = static_cast<unsigned>((((wave * TM + i) * 32 + r32) * k + 4 * c2) * 4);
          const unsigned xo = static_cast<unsigned>(((32 * j + r32) * k + 4 * c2) * 4);
          acc[i][j] = floatx16{};
#pragma unroll 1
          for (int kb0 = s_lo * KG * BK; kb0 < kb1; kb0 += 128) {
            floatx16 sum{};
            // MFMA e of 8 columns from kb contracts columns kb + e and kb + 4 + e
#pragma unroll 1
            for (int kb = kb0; kb < min(kb0 + 128, kb1); kb += 8) {
              const floatx4 av = __builtin_amdgcn_raw_buffer_load_b128(rw, wo, kb * 4, 0);
              const floatx4 bv = __builtin_amdgcn_raw_buffer_load_b128(rx, xo, kb * 4, 0);
#pragma unroll
              for (int e = 0; e < 4; ++e)
                sum = __builtin_amdgcn_mfma_f32_32x32x2f32(av[e], bv[e], sum, 0, 0, 0);
            }
            acc[i][j] += sum;
          }
        }
    }
  }

  if (n_split > 1) {
    // partial float4 (i, j, q) of thread tid of split sp of tile t at float4
    // index (((t * n_split + sp) * TM * TN + i * TN + j) * 4 + q) * NT + tid
    const auto rs = ikv::partial_rsrc(
        part, static_cast<size_t>(n_tiles) * n_split * TM * TN * 4 * NT * sizeof(floatx4));
    auto at = [&](int z, int i, int j, int q) {
      return static_cast<unsigned>(
          ((((static_cast<size_t>(t) * n_split + z) * TM * TN + i * TN + j) * 4 + q) * NT + tid) *
          sizeof(floatx4));
    };
    if (mine) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const floatx4 v = quad(i, j, q);
            ikv::store4_agent(rs, at(sp, i, j, q), make_float4(v[0], v[1], v[2], v[3]));
          }
    }
    __builtin_amdgcn_s_waitcnt(0);  // this wave's stores performed
    __syncthreads();                // ... and every other wave's
    if (threadIdx.x == 0)
      s_last = __hip_atomic_fetch_add(counters + t, 1, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT) == n_split - 1;
    __syncthreads();
    if (!s_last || !mine) return;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          floatx4 sum{};
          for (int z = 0; z < n_split; ++z) {
            floatx4 v = quad(i, j, q);
            if (z != sp) {
              const float4 l = ikv::load4_agent(rs, at(z, i, j, q));
              v = floatx4{l.x, l.y, l.z, l.w};
            }
            sum = z == 0 ? v : sum + v;
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[i][j][4 * q + r] = sum[r];
        }
    if (threadIdx.x == 0)
      __hip_atomic_store(counters + t, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (!mine) return;

  // acc[i][j] register 4 q + r of lane l: weight row (wave * TM + i) * 32 +
  // 8 q + 4 (l / 32) + r, token 32 j + l % 32 of the tile.
  const bool vec =
      ((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(residual)) & 15) == 0;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int tok = t0 + 32 * j + r32;
    if (tok < m) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = w0 + (wave * TM + i) * 32 + 8 * q + 4 * c2;
          if (n < n_out) {
            const size_t o = static_cast<size_t>(tok) * n_out + n;
            floatx4 v = quad(i, j, q);
            if (vec) {
              if (residual) v += *reinterpret_cast<const floatx4 *>(residual + o);
              *reinterpret_cast<floatx4 *>(out + o) = v;
            } else {
#pragma unroll
              for (int r = 0; r < 4; ++r) out[o + r] = residual ? v[r] + residual[o + r] : v[r];
            }
          }
        }
    }
  }
}

template <int TM, int TN, int WM, int KG, int MINW>
int launch(const float *w, const float *x, float *out, const float *residual, int n_out, int k,
           int m, int n_split, float *part, int *counters, hipStream_t s) {
  constexpr int BW = 32 * TM * WM, BT = 32 * TN;
  static_assert(BW <= ikv::kBf16x3MaxRows && BT <= ikv::kBf16x3MaxRows, "a panel is one buffer range");
  const int64_t tiles_t = (m + BT - 1) / BT;
  const int64_t n_tiles = tiles_t * ((n_out + BW - 1) / BW);
  const int64_t per = (n_tiles + kXcds - 1) / kXcds;
  if (n_tiles > INT_MAX / 2 || per * n_split * kXcds > INT_MAX / 2) return -EOVERFLOW;
  gemm_bf16x3_kernel<TM, TN, WM, KG, MINW>
      <<<static_cast<unsigned>(per * n_split * kXcds), WM * KG * 64, 0, s>>>(
          w, x, out, residual, n_out, k, m, static_cast<int>(tiles_t), static_cast<int>(n_tiles),
          n_split, part, counters);
  return ikv::launch_status();
}

}  // namespace

namespace ikv {

int gemm_bf16x3_tile(int code, int n_split, const float *w, const float *x, float *out,
                     const float *residual, int n, int kk, int mm, float *part, int *counters,
                     hipStream_t s) {
  if (!gemm_bf16x3_supported(n, kk, mm)) return -ENOTSUP;
  if (n_split < 1 || n_split > kk / 64) return -EINVAL;
  switch (code) {
    case 0: return launch<2, 4, 4, 1, 1>(w, x, out, residual, n, kk, mm, n_split, part, counters, s);
    case 1: return launch<1, 4, 4, 1, 2>(w, x, out, residual, n, kk, mm, n_split, part, counters, s);
    case 2: return launch<1, 2, 4, 1, 2>(w, x, out, residual, n, kk, mm, n_split, part, counters, s);
    case 3: return launch<1, 2, 2, 2, 2>(w, x, out, residual, n, kk, mm, n_split, part, counters, s);
    default: return -EINVAL;
  }
}

}  // namespace ikv
