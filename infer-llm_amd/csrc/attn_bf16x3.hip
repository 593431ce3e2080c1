// attn_bf16x3.hip — causal GQA flash attention in F32 on the bf16 matrix cores
// (v_mfma_f32_32x32x16_bf16): prompts behind ikv_attn_prefill_f32 and its
// paged form, for any head_dim up to 128 that is a multiple of 4 and any
// grouping, where the contexts are long enough (the rules are at the callers,
// attn_prefill.hip and attn_generic.hip). Semantics as there: key j is visible
// to query t iff j <= n_past + t; query head h reads KV head h / G
// (src/backends/cpu_backend.cpp:525-634).
//
// Every float is three bf16 pieces (bf16x3.hpp), so Q K^T and P V are F32
// products on a pipe with 2.67 times the F32 one's room after the six piece
// products; the scores, the softmax and the sums stay F32. Distance to 64
// bits, 2-norm relative, against the F32 kernels': 2048 tokens of 16 heads of
// 128 2.4e-7 (3.9e-7), 777 tokens behind 3319 5.9e-7 (1.2e-6), heads of 64,
// 1500 behind 500, 4.0e-7 (6.7e-7).
//
// Layout:
//   * A workgroup owns BR = 32 RW rows (row = token * G + query head) of one
//     KV head: RW wavefronts of 32 rows in each of KG key groups, which take
//     key tiles (32 keys) kg, kg + KG, ... and meet through LDS at the end.
//     blockIdx % n_head_kv is the KV head (with 8, one per XCD); the longest
//     blocks start first.
//   * S^T = K Q^T and O^T += V^T P^T, so a lane (and lane ^ 32) holds one
//     query row in both: P goes from the softmax into the second product's B
//     operand in place. The key order of an MFMA is the one in which S^T
//     leaves them in a lane (16 t + 4 c2 + 0..3, + 8), and V is staged in it.
//   * K and V tiles go through registers, are split once per workgroup and
//     staged as three bf16 planes: K rows of D halfs, their 16-byte pieces
//     XOR-ed with the key; V transposed, 64 bytes (32 keys) a dim, the order
//     of dims and pieces chosen so that the 16 lanes of a read or write meet
//     all banks (v_at). One K buffer, two V buffers.
//   * One wave per SIMD with up to 512 registers (heads of 64: two of 256),
//     and the overlap inside the wave: while tile i + 1's Q K^T runs, tile
//     i's softmax and the split of its P are issued between the MFMAs; while
//     P V runs, the splits of K (i + 2) and V (i + 1). A share of four VALU
//     instructions fits behind a 32-cycle MFMA; the shares are laid out by
//     hand, a scheduling region per six MFMAs, and two LDS fragments ahead.
//   * The row maximum moves only when a score exceeds it by 2^8; h h products
//     of S are summed apart from the small ones.
//   * What bounds it: the matrix pipe is busy about half the time; the rest
//     is the VALU work that does not fit behind the MFMAs, the 48 LDS reads
//     per tile and the two barriers. Measured (us, the
//     kernels before -> this one, graphs): Qwen3-8B heads, 4096 tokens 999 ->
//     746, 777 behind 3319 487 -> 338; 0.6B heads, 2048 tokens 164 -> 137; 12
//     heads of 64 over 4, 1500 behind 500 235 -> 63; 32 of 64 over 8, 900
//     tokens 134 -> 36; 12 of 128 over 4, 512 tokens 58 -> 32.
//   * What the pieces do not carry: a wave starts over on F32 where its sums
//     are not finite, or where a split of V or Q dropped bits (floats below
//     2^-109; V's are looked at one by one, as a dim of small values has only
//     small sums) or Q is so large that bits dropped from K would count;
//     probabilities are split times 2^17. That costs 1-3% (0.6B heads, 2048
//     tokens 112.7 -> 115.7 us cold); one look at a wave's largest output cost
//     nothing, and missed a small dim among ordinary ones and small keys
//     against large queries. 2048 tokens with every wave starting over: 790.
//   * Tried and not kept: two waves per SIMD with Q's last pieces in LDS (0.6B
//     2048 125, 8B 4096 824: 256 registers leave no room to schedule in); K
//     and V two tiles ahead (equal); blocks in pairs of a long and a short one
//     (0.6B 3000 286 against 241 with the longest first).
#include "attn_bf16x3.hpp"
#include "bf16x3.hpp"
#include "coherent.hpp"
#include "ikv_common.hpp"

#include <algorithm>
#include <climits>

namespace {

using namespace ikv::pieces;

constexpr int kCUs = 256;         // MI355X compute units
constexpr int BN = 32;            // keys per tile
constexpr float kRescale = 8.0f;  // log2 headroom before the running max is moved
// Probabilities go into their pieces (and the row sums) times 2^17, so that all
// down to the smallest normal float, which is as small as exp2 gives them, keep
// their bits. The factor leaves with the division by the row's sum.
constexpr float kProbScale = 0x1p17f;

__device__ __forceinline__ float pair_max(float x) {  // lanes l and l ^ 32
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
__device__ __forceinline__ float pair_sum(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}

template <int N>
__device__ __forceinline__ void load_dims(__amdgpu_buffer_rsrc_t r, unsigned off, float *d) {
  if constexpr (N == 1) {
    d[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
  } else if constexpr (N == 2) {
    const auto t = __builtin_bit_cast(floatx2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
    d[0] = t[0], d[1] = t[1];
  } else {
    const auto t = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
    d[0] = t[0], d[1] = t[1], d[2] = t[2], d[3] = t[3];
  }
}

template <int DT, int RW, int KG, int MINW, bool PAGED>
__global__ __launch_bounds__(RW * KG * 64, MINW) void attn_bf16x3_kernel(
    const float *__restrict__ q, const float *__restrict__ k, const float *__restrict__ v,
    float *__restrict__ out, int n_head_kv, int G, int dim, int n_rows, int n_kv, int n_past,
    int n_blocks, float scale_log2, ikv::Pages pages) {
  constexpr int D = 32 * DT;
  constexpr int KS = D / 16;       // MFMA steps of Q K^T
  constexpr int NT = RW * 64;      // threads of a key group
  constexpr int BR = 32 * RW;      // rows of a block
  constexpr int VD = 2 * DT / RW;  // dims of a thread's V item, K items of a thread
  constexpr int PLANE = BN * D;    // bf16 of one piece of a K or V tile
  __shared__ __attribute__((aligned(16))) unsigned short s_k[KG][3 * PLANE];
  __shared__ __attribute__((aligned(16))) unsigned short s_v[KG][2][3 * PLANE];
  constexpr bool BLOCKED = KG == 1;
  __shared__ floatx4 s_o[BLOCKED ? RW * 64 * 4 * DT : 1];

  const int g = blockIdx.x % n_head_kv;
  const int item = blockIdx.x / n_head_kv;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wv / RW, slot = wv % RW;
  const int tid = threadIdx.x % NT;
  const int r32 = lane & 31, c2 = lane >> 5;
  const int n_head = n_head_kv * G;
  const int stride = n_head_kv * dim;  // floats of a token row

  // staging: a thread's K items (a key's 8 dims) and V item (VD dims of 8 keys)
  unsigned kof[VD][2];
  int kdst[VD];
#pragma unroll
  for (int i = 0; i < VD; ++i) {
    const int it = tid + NT * i;
    const int key = it / (D / 8), c = it % (D / 8);
#pragma unroll
    for (int u = 0; u < 2; ++u)
      kof[i][u] = 8 * c + 4 * u < dim ? static_cast<unsigned>((key * stride + 8 * c + 4 * u) * 4) : 0x80000000u;
    kdst[i] = key * D + 8 * (D == 128 ? c ^ (key & 15) : c ^ ((key >> 1) & 7));
  }
  const int vd0 = tid % (D / VD) * VD, vc = tid / (D / VD);  // vc = 2 t + c2: keys 16 t + 4 c2 .. + 3, + 8
  const unsigned vof =
      vd0 < dim ? static_cast<unsigned>(((16 * (vc >> 1) + 4 * (vc & 1)) * stride + vd0) * 4) : 0x80000000u;
  auto v_at = [](int d, int c) {  // halfs: piece c of dim d
    return (d >> 2) * 128 + ((((d & 3) ^ ((d >> 4) & 3)) << 2) + (c ^ ((d >> 2) & 3))) * 8;
  };
  unsigned short *const sk = s_k[kg];
  floatx4 kraw[VD][2];
  float vraw[8][VD];
  unsigned lost = 0;  // what this thread's splits of Q and V dropped
  __shared__ int s_lost;
  if (threadIdx.x == 0) s_lost = 0;
  // (first: the tile's row of the cache or the pool)
  auto tile_rsrc = [&](const float *base, int tile, int first) {
    const int rows = min(BN, n_kv - tile * BN);
    return __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(base + static_cast<size_t>(first) * stride + g * dim), 0,
        ((rows - 1) * stride + dim) * 4, ikv::kBufWord3);
  };
  auto load_k = [&](int tile, int first) {
    const auto r = tile_rsrc(k, tile, first);
#pragma unroll
    for (int i = 0; i < VD; ++i)
#pragma unroll
      for (int u = 0; u < 2; ++u) kraw[i][u] = __builtin_amdgcn_raw_buffer_load_b128(r, kof[i][u], 0, 0);
  };
  auto load_v = [&](int tile, int first) {
    const auto r = tile_rsrc(v, tile, first);
#pragma unroll
    for (int e = 0; e < 8; ++e)
      load_dims<VD>(r, vof + static_cast<unsigned>(((e & 3) + 8 * (e >> 2)) * stride * 4), vraw[e]);
  };
  auto put_k = [&]() {
#pragma unroll
    for (int i = 0; i < VD; ++i) {
      unsigned none = 0;
      const Pieces p = split8<false>(kraw[i][0], kraw[i][1], none);
#pragma unroll
      for (int z = 0; z < 3; ++z) *reinterpret_cast<bf16x8 *>(sk + z * PLANE + kdst[i]) = p.p[z];
    }
  };
  auto put_v = [&](unsigned short *sv) {
#pragma unroll
    for (int i = 0; i < VD; ++i) {
      const Pieces p = split8<false>(floatx4{vraw[0][i], vraw[1][i], vraw[2][i], vraw[3][i]},
                              floatx4{vraw[4][i], vraw[5][i], vraw[6][i], vraw[7][i]}, lost);
#pragma unroll
      for (int z = 0; z < 3; ++z) *reinterpret_cast<bf16x8 *>(sv + z * PLANE + v_at(vd0 + i, vc)) = p.p[z];
    }
  };
  auto read_k = [&](int s, bf16x8 *d) {
    const int at = r32 * D + 8 * (D == 128 ? (2 * s + c2) ^ (r32 & 15) : (2 * s + c2) ^ ((r32 >> 1) & 7));
#pragma unroll
    for (int z = 0; z < 3; ++z) d[z] = *reinterpret_cast<const bf16x8 *>(sk + z * PLANE + at);
  };
  auto read_v = [&](const unsigned short *sv, int j, bf16x8 *d) {  // of MFMA group j = t * DT + dt
    const int at = v_at(32 * (j % DT) + r32, 2 * (j / DT) + c2);
#pragma unroll
    for (int z = 0; z < 3; ++z) d[z] = *reinterpret_cast<const bf16x8 *>(sv + z * PLANE + at);
  };

  const int blk = n_blocks - 1 - item;  // the longest blocks first
  const int row0 = blk * BR + slot * 32;
  const int row = row0 + r32;
  const bool row_ok = row < n_rows;
  const int tok = min(row, n_rows - 1) / G;
  const int head = g * G + min(row, n_rows - 1) % G;
  const int first_tok = min(row0, n_rows - 1) / G;
  const int n_tiles =
      (min(n_kv, n_past + (min((blk + 1) * BR, n_rows) - 1) / G + 1) + BN - 1) / BN;
  const int n_it = (n_tiles + KG - 1) / KG;  // tiles kg, kg + KG, ... of each group
  // (a tile past the end is masked whole; what is staged for it is the last one)
  auto staged = [&](int i) { return min(kg + KG * i, n_tiles - 1); };
  // The staged tiles' rows, one after the other. A paged cache's next 64 block
  // table entries are held one per lane, checked as they are read, and tiles
  // and blocks are counted along: a look into the table, its check and a
  // division at every load cost 8 % (777 tokens behind 3319 of 32 heads over 8:
  // 319 us, here 298, contiguous 293).
  int next = kg, blk_of = 0, in_blk = 0, last_blk = 0, last_in = 0, ent = 0, ent0 = 0;
  const int per_blk = PAGED ? pages.bt / BN : 1;  // at least 2
  auto entries = [&](int b) {
    ent0 = b;
    ent = pages.table[min(b + lane, last_blk)];
    if (static_cast<unsigned>(ent) >= static_cast<unsigned>(pages.n_blocks)) {
      ikv::raise_status(pages.status, IKV_STATUS_BLOCK);
      ent = 0;
    }
  };
  if constexpr (PAGED) {
    blk_of = kg / per_blk, in_blk = kg % per_blk;
    last_blk = (n_tiles - 1) / per_blk, last_in = (n_tiles - 1) % per_blk;
    entries(min(blk_of, last_blk));
  }
  auto next_row = [&]() -> int {
    const int tile = min(next, n_tiles - 1);
    const bool last = next >= n_tiles - 1;
    next += KG;
    if constexpr (PAGED) {
      const int b = last ? last_blk : blk_of, at = last ? last_in : in_blk;
      in_blk += KG;
#pragma unroll
      for (int z = 0; z < (KG + 1) / 2; ++z)
        if (in_blk >= per_blk) in_blk -= per_blk, ++blk_of;
      if (b - ent0 >= 64) entries(b);
      return __builtin_amdgcn_readlane(ent, b - ent0) * pages.bt + at * BN;
    }
    return tile * BN;
  };

  // Q: lane (row r32, c2) holds dims 16 s + 8 c2 .. + 7 of step s
  bf16x8 qp[KS][3];
  {
    const float *qr = q + (static_cast<size_t>(tok) * n_head + head) * dim;
    float top = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int d = 16 * s + 8 * c2;
      floatx4 u{}, w{};
      if (row_ok && d < dim) u = *reinterpret_cast<const floatx4 *>(qr + d);
      if (row_ok && d + 4 < dim) w = *reinterpret_cast<const floatx4 *>(qr + d + 4);
      const Pieces p = split8<false>(u, w, lost);
#pragma unroll
      for (int z = 0; z < 3; ++z) qp[s][z] = p.p[z];
#pragma unroll
      for (int e = 0; e < 4; ++e) top = fmaxf(fmaxf(top, fabsf(u[e])), fabsf(w[e]));
    }
    // Bits dropped from K (below 2^-133) move a score by less than 2^-60 times
    // this bound on Q: K's splits are not looked at.
    if (top * fmaxf(scale_log2, 1.f) >= 0x1p64f) lost = ~0u;
  }
  floatx16 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = floatx16{};
  float m_row = -INFINITY, l_part = 0.f;
  floatx16 s0{}, s1{};  // S of the next tile: h h products, and the others
  bf16x8 fr[3][3];      // K or V pieces of this and the next two MFMA groups
  auto qk = [&](int s) {
    const bf16x8 *c = fr[s % 3];
    s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[2], qp[s][0], s == 0 ? floatx16{} : s1, 0, 0, 0);
    s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[0], qp[s][2], s1, 0, 0, 0);
    s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[1], qp[s][1], s1, 0, 0, 0);
    s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[1], qp[s][0], s1, 0, 0, 0);
    s0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[0], qp[s][0], s == 0 ? floatx16{} : s0, 0, 0, 0);
    s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[0], qp[s][1], s1, 0, 0, 0);
  };

  const int row_0 = next_row();
  int row_1 = next_row(), row_2 = next_row(), row_3 = next_row();  // of tiles i + 1, i + 2, i + 3
  load_k(staged(0), row_0);
  load_v(staged(0), row_0);
  put_k();
  put_v(s_v[kg][0]);
  load_k(staged(1), row_1);
  __syncthreads();
  read_k(0, fr[0]);
  read_k(1, fr[1]);
  static_for<KS>([&](auto sc) {
    constexpr int s = decltype(sc)::value;
    if constexpr (s + 2 < KS) read_k(s + 2, fr[(s + 2) % 3]);
    qk(s);
  });
  __syncthreads();
  put_k();
  load_k(staged(2), row_2);
  __syncthreads();
  read_k(0, fr[0]);
  read_k(1, fr[1]);

  using P0 = std::integral_constant<int, 0>;
  using P1 = std::integral_constant<int, 1>;
  auto step = [&](int i, auto par) {
    constexpr int P = decltype(par)::value;  // i & 1: the V buffers
    // S of tile i is in s0 + s1, K of tile i + 1 and V of tile i are staged,
    // K of tile i + 2 is on its way
    const int kbase = (kg + KG * i) * BN;
    float p[16];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 16; ++e) p[e] = s0[e] + s1[e];
    if (kbase + BN - 1 > n_past + first_tok || kbase + BN > n_kv) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int kk = kbase + 8 * (e >> 2) + 4 * c2 + (e & 3);
        if (kk > n_past + tok || kk >= n_kv) p[e] = -INFINITY;
      }
    }
    // Q K^T of the next tile, the softmax of this one between its MFMAs, a
    // share per MFMA step: first the maximum, then (exp of 8, two halves
    // of their split) twice
    float ref = 0.f;
    uintx4 pw[2][3];
    static_for<KS>([&](auto sc) {
      constexpr int s = decltype(sc)::value;
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (s + 2 < KS)
        read_k(s + 2, fr[(s + 2) % 3]);
      else
        read_v(s_v[kg][P], s + 2 - KS, fr[(s + 2) % 3]);
      float mt = p[0];
      constexpr int lo = s == 0 ? 0 : (s - 1) * 6 / (KS - 1), hi = s == 0 ? 0 : s * 6 / (KS - 1);
      if constexpr (s == 0) {
#pragma unroll
        for (int e = 1; e < 16; ++e) mt = fmaxf(mt, p[e]);
      }
      static_for<hi - lo>([&](auto wc) {
        constexpr int w = lo + decltype(wc)::value, t = w / 3;
        if constexpr (w % 3 == 0) {
#pragma unroll
          for (int e = 8 * t; e < 8 * t + 8; ++e) {
            p[e] = ikv::fast_exp2(fmaf(p[e], scale_log2, -ref)) * kProbScale;
            l_part += p[e];
          }
        } else {
          constexpr int h = w % 3 - 1;
#pragma unroll
          for (int e = 2 * h; e < 2 * h + 2; ++e) {
            unsigned x, y, z, none = 0;
            split2(p[8 * t + 2 * e], p[8 * t + 2 * e + 1], x, y, z, none);
            asm volatile("" : "+v"(x), "+v"(y), "+v"(z));
            pw[t][0][e] = x, pw[t][1][e] = y, pw[t][2][e] = z;
          }
        }
      });
      if constexpr (s == 1) load_v(staged(i + 1), row_1);
      qk(s);
      constexpr int kShare = s == 0 ? 3 : 4 * (hi - lo) + 2 * ((hi + 2) / 3 - (lo + 2) / 3);  // 8 of exp are 32
#pragma unroll
      for (int z = 0; z < 6; ++z) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (s == 1 && z > 0) __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
        if (z % 2 == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, kShare, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (s == 0) {
        if (__builtin_amdgcn_ballot_w64(mt * scale_log2 > m_row + kRescale) != 0) {
          const float m_new = fmaxf(m_row, pair_max(mt) * scale_log2);
          const float alpha = m_new == -INFINITY ? 1.f : ikv::fast_exp2(m_row - m_new);
          m_row = m_new;
          l_part *= alpha;
#pragma unroll
          for (int t = 0; t < DT; ++t) o[t] *= alpha;
        }
        ref = m_row == -INFINITY ? 0.f : m_row;
      }
    });
    __syncthreads();  // every wave's K reads are done
    // P V of this tile, the splits of the next ones between its MFMAs: half
    // a split8 at a time (the reads of a region come before its writes: the
    // compiler cannot tell the buffers apart)
    uintx4 cw[3];
    static_for<2 * DT>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      constexpr int lo = j * 4 * VD / (2 * DT), hi = (j + 1) * 4 * VD / (2 * DT);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (j + 2 < 2 * DT) read_v(s_v[kg][P], j + 2, fr[(KS + j + 2) % 3]);
      if constexpr (j == DT) load_k(staged(i + 3), row_3);
      static_for<hi - lo>([&](auto wc) {
        constexpr int w = lo + decltype(wc)::value, u = w / 2, h = w & 1;
        float x[4];
        unsigned none = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          x[e] = u < VD ? kraw[u % VD][h][e] : vraw[4 * h + e][u % VD];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          unsigned y0, y1, y2;
          split2(x[2 * e], x[2 * e + 1], y0, y1, y2, u < VD ? none : lost);
          // (pinned to this region: the first half has no use in it)
          asm volatile("" : "+v"(y0), "+v"(y1), "+v"(y2));
          cw[0][2 * h + e] = y0, cw[1][2 * h + e] = y1, cw[2][2 * h + e] = y2;
        }
        if constexpr (u >= VD) asm volatile("" : "+v"(lost));
        if constexpr (h == 1) {
          unsigned short *dst = u < VD ? sk + kdst[u % VD] : s_v[kg][P ^ 1] + v_at(vd0 + u % VD, vc);
#pragma unroll
          for (int z = 0; z < 3; ++z) *reinterpret_cast<uintx4 *>(dst + z * PLANE) = cw[z];
        }
      });
#pragma unroll
      for (int z = 0; z < 6; ++z)
        o[j % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            fr[(KS + j) % 3][kPieceA[z]], __builtin_bit_cast(bf16x8, pw[j / DT][kPieceB[z]]), o[j % DT], 0, 0, 0);
#pragma unroll
      for (int z = 0; z < 6; ++z) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (j == DT && z > 0) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        if (j + 2 < 2 * DT && z % 2 == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        // (one more where V's splits also collect what they drop: 2% of the
        // forms of two groups)
        __builtin_amdgcn_sched_group_barrier(0x002, 4 * (hi - lo) + (j >= DT ? 1 : 0), 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    __syncthreads();  // every wave's V reads are done, the next tiles are staged
    row_1 = row_2, row_2 = row_3, row_3 = next_row();
    read_k(0, fr[0]);
    read_k(1, fr[1]);
  };
  // With one key group, O is set aside in LDS every 16 tiles and starts again
  // from zero, so that a long context's sum does not round at its full size
  // at every tile. m_aside: the reference maximum of what was set aside.
  float m_aside = -INFINITY;
  bool aside = false;
  auto set_aside = [&]() {
    floatx4 *const mine = s_o + slot * (64 * 4 * DT) + lane;
    const float f = m_aside == -INFINITY ? 0.f : ikv::fast_exp2(m_aside - m_row);
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int z = 0; z < 4; ++z) {
        floatx4 x = {o[t][4 * z], o[t][4 * z + 1], o[t][4 * z + 2], o[t][4 * z + 3]};
        if (aside) x += mine[(4 * t + z) * 64] * f;
        mine[(4 * t + z) * 64] = x;
      }
    m_aside = m_row;
    aside = true;
  };
  int i = 0;
  for (; i + 2 <= n_it; i += 2) {
    step(i, P0{});
    step(i + 1, P1{});
    if constexpr (BLOCKED) {
      if ((i & 14) == 14) {
        set_aside();
#pragma unroll
        for (int t = 0; t < DT; ++t) o[t] = floatx16{};
      }
    }
  }
  if (i < n_it) step(i, P0{});
  if constexpr (BLOCKED) {
    if (aside) {
      set_aside();
      const floatx4 *const mine = s_o + slot * (64 * 4 * DT) + lane;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int z = 0; z < 4; ++z) {
          const floatx4 x = mine[(4 * t + z) * 64];
#pragma unroll
          for (int e = 0; e < 4; ++e) o[t][4 * z + e] = x[e];
        }
    }
  }

  if (any_lost(lost) && lane == 0) s_lost = 1;  // (V's pieces serve every wave)
  if constexpr (KG == 1) __syncthreads();
  if constexpr (KG > 1) {
    // the groups' states meet in LDS: groups 1 .. hand theirs to group 0
    constexpr int XW = 16 * DT + 2;
    static_assert(sizeof(float) * (KG - 1) * RW * 64 * XW <= sizeof(s_v), "the states fit the V buffers");
    float *const xch = reinterpret_cast<float *>(s_v);
    if (kg > 0) {
      float *x = xch + ((kg - 1) * RW + slot) * XW * 64 + lane;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) x[(16 * t + e) * 64] = o[t][e];
      x[16 * DT * 64] = m_row;
      x[(16 * DT + 1) * 64] = l_part;
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
      for (int src = 1; src < KG; ++src) {
        const float *x = xch + ((src - 1) * RW + slot) * XW * 64 + lane;
        const float mb = x[16 * DT * 64];
        const float M = fmaxf(m_row, mb);
        const float ea = m_row == -INFINITY ? 0.f : ikv::fast_exp2(m_row - M);
        const float eb = mb == -INFINITY ? 0.f : ikv::fast_exp2(mb - M);
        l_part = l_part * ea + x[(16 * DT + 1) * 64] * eb;
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int e = 0; e < 16; ++e) o[t][e] = o[t][e] * ea + x[(16 * t + e) * 64] * eb;
        m_row = M;
      }
    }
  }
  if (kg != 0) return;
  float inv = 1.0f / pair_sum(l_part);
  // Inputs the pieces do not carry (bf16x3.hpp) dropped bits in a split or leave
  // a result that is not finite: the wave then starts over, on F32 MFMAs over
  // the tiles that all its rows see whole and key by key over the rest, where
  // a row takes only the keys it sees (a masked key weighs 0, but 0 times an
  // infinite value is NaN)
  bool odd = s_lost != 0 || !(fabsf(inv) < INFINITY);
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int e = 0; e < 16; ++e) odd |= !(fabsf(o[t][e] * inv) < INFINITY);
  if (__builtin_amdgcn_ballot_w64(odd) != 0) {
#pragma unroll
    for (int t = 0; t < DT; ++t) o[t] = floatx16{};
    m_row = -INFINITY;
    l_part = 0.f;
    const float *qr = q + (static_cast<size_t>(tok) * n_head + head) * dim;
    const int last_tok = min(row0 + 31, n_rows - 1) / G;
    const int my_end = min(n_kv, n_past + last_tok + 1);
    const int full = min(n_kv, n_past + first_tok + 1) / BN;  // tiles that every row sees whole
    for (int tile = 0; tile < full; ++tile) {
      int first = tile * BN;
      if constexpr (PAGED) first += static_cast<int>(ikv::page_shift(pages, first));
      const auto rk = tile_rsrc(k, tile, first);
      const auto rv = tile_rsrc(v, tile, first);
      floatx16 s{};
      for (int d = 4 * c2; d < D; d += 8) {  // dims 8 j + 4 c2 .. + 3
        const floatx4 a = __builtin_amdgcn_raw_buffer_load_b128(
            rk, d < dim ? static_cast<unsigned>((r32 * stride + d) * 4) : 0x80000000u, 0, 0);
        floatx4 b{};
        if (row_ok && d < dim) b = *reinterpret_cast<const floatx4 *>(qr + d);
#pragma unroll
        for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], s, 0, 0, 0);
      }
      float p[16], mt = -INFINITY;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        p[e] = s[e] * scale_log2;
        mt = fmaxf(mt, p[e]);
      }
      const float m_new = fmaxf(m_row, pair_max(mt));
      const float ref = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = m_new == -INFINITY ? 1.f : ikv::fast_exp2(m_row - m_new);
      m_row = m_new;
      l_part *= alpha;
      floatx16 ot[DT] = {};  // this tile's sums
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float x = ikv::fast_exp2(p[e] - ref);
        l_part += x;
        const int key = 8 * (e >> 2) + 4 * c2 + (e & 3);
#pragma unroll
        for (int t = 0; t < DT; ++t) {
          const unsigned at = 32 * t + r32 < dim ? static_cast<unsigned>((key * stride + 32 * t + r32) * 4)
                                                 : 0x80000000u;
          ot[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(
              __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rv, at, 0, 0)), x, ot[t], 0, 0, 0);
        }
      }
#pragma unroll
      for (int t = 0; t < DT; ++t) o[t] = o[t] * alpha + ot[t];
    }
    for (int key = full * BN; key < my_end; ++key) {
      const bool sees = key <= n_past + tok;
      int at = key;
      if constexpr (PAGED) at += static_cast<int>(ikv::page_shift(pages, key));
      const float *kr = k + static_cast<size_t>(at) * stride + g * dim;
      const float *vr = v + static_cast<size_t>(at) * stride + g * dim;
      float dot = 0.f;  // a lane's half of the dims
      for (int d = 4 * c2; d < dim; d += 8) {
        const floatx4 a = *reinterpret_cast<const floatx4 *>(kr + d);
        const floatx4 b = *reinterpret_cast<const floatx4 *>(qr + d);
#pragma unroll
        for (int e = 0; e < 4; ++e) dot = fmaf(a[e], b[e], dot);
      }
      const float sc = pair_sum(dot) * scale_log2;
      if (sees) {
        const float m_new = fmaxf(m_row, sc);
        const float ref = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = m_new == -INFINITY ? 1.f : ikv::fast_exp2(m_row - m_new);
        const float x = ikv::fast_exp2(sc - ref);
        m_row = m_new;
        l_part = fmaf(l_part, alpha, c2 == 0 ? x : 0.f);
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int z = 0; z < 4; ++z) {
            const int d = 32 * t + 8 * z + 4 * c2;
            if (d < dim) {
              const floatx4 y = *reinterpret_cast<const floatx4 *>(vr + d);
#pragma unroll
              for (int e = 0; e < 4; ++e) o[t][4 * z + e] = fmaf(x, y[e], o[t][4 * z + e] * alpha);
            }
          }
      }
    }
    inv = 1.0f / pair_sum(l_part);
  }
  if (row_ok) {
    float *orow = out + (static_cast<size_t>(tok) * n_head + head) * dim;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int z = 0; z < 4; ++z) {
        const int d = 32 * t + 8 * z + 4 * c2;
        if (d < dim)
          *reinterpret_cast<floatx4 *>(orow + d) =
              floatx4{o[t][4 * z], o[t][4 * z + 1], o[t][4 * z + 2], o[t][4 * z + 3]} * inv;
      }
  }
}

template <int DT, int RW, int KG, int MINW>
void launch(const float *q, const float *k, const float *v, float *out, int n_head_kv, int G,
            int dim, int n_rows, int n_kv, int n_past, float sl2, const ikv::Pages *pg, hipStream_t s) {
  constexpr int BR = 32 * RW;
  const int n_blocks = (n_rows + BR - 1) / BR;
  const unsigned grid = static_cast<unsigned>(n_blocks) * n_head_kv;
  if (pg)
    attn_bf16x3_kernel<DT, RW, KG, MINW, true><<<grid, RW * KG * 64, 0, s>>>(
        q, k, v, out, n_head_kv, G, dim, n_rows, n_kv, n_past, n_blocks, sl2, *pg);
  else
    attn_bf16x3_kernel<DT, RW, KG, MINW, false><<<grid, RW * KG * 64, 0, s>>>(
        q, k, v, out, n_head_kv, G, dim, n_rows, n_kv, n_past, n_blocks, sl2, ikv::Pages{});
}

}  // namespace

namespace {

// A form of the kernel and its estimated time: blocks of `rows` rows, `groups`
// key groups, `slots` workgroups on the card at once. us = fixed + the larger
// of alone * (the longest block's steps) and busy * (the busiest slot's: the
// average per slot, plus a shortest block where they do not divide evenly; the
// longest blocks start first), a step being a tile of each group and a block's
// start and end counting as `ends` steps more. Fitted to 1110 prompts (3 to
// 128 heads of 32 to 128 over 1 to 128, 65-4096 tokens behind 0-4000): 3-6%
// rms, and the first form up to 64 dims 15% where it is not the better one; on
// average 0.1% from the better form of two. Without the blocks' ends a card
// full of short ones took the wrong one: 128 heads of 64, 140 tokens 27.8 us
// against 12.3, 64 heads, 400 tokens 43.7 against 20.0.
struct Form {
  int rows, groups, slots;
  double fixed, alone, busy, ends;
};

double time_of(const Form &f, int64_t rows, int G, int64_t n_kv, int64_t n_past, int heads) {
  auto steps = [&](int64_t row) {  // of a block that ends with this row
    const int64_t tiles = (std::min(n_kv, n_past + row / G + 1) + BN - 1) / BN;
    return static_cast<double>((tiles + f.groups - 1) / f.groups) + f.ends;
  };
  const double first = steps(std::min<int64_t>(f.rows, rows) - 1), last = steps(rows - 1);
  const double per_slot = double((rows + f.rows - 1) / f.rows) * heads / f.slots;
  const double load = per_slot * (first + last) / 2 + (std::ceil(per_slot) - per_slot) * first;
  return f.fixed + std::max(f.alone * last, f.busy * load);
}

// heads of 128: 128 rows and one key group, or 64 and two; heads of 64: 64 rows
// and two groups, two workgroups on a CU, or 32 rows and four groups
constexpr Form kForms128[2] = {{128, 1, kCUs, 0.0, 2.37, 2.37, 3.3}, {64, 2, kCUs, 0.0, 2.8, 2.8, 3.4}};
constexpr Form kForms64[2] = {{64, 2, 2 * kCUs, 0.0, 1.74, 1.91, 3.5}, {32, 4, kCUs, 1.6, 2.37, 2.37, 2.5}};

}  // namespace

namespace ikv {

bool attn_bf16x3_supported(const void *q, const void *k, const void *v, const void *out, int n_head,
                           int n_head_kv, int head_dim, int64_t n_q, int64_t n_kv, int64_t n_past) {
  if (head_dim % 4 != 0 || head_dim < 4 || head_dim > 128) return false;
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out)) return false;
  const int G = n_head / n_head_kv;
  // rows, keys and the workgroup count in int; a tile's rows one buffer range
  return n_q <= INT_MAX / 4 / G && n_kv <= INT_MAX / 4 && n_past <= INT_MAX / 4 &&
         n_q * G / 32 + 1 <= INT_MAX / n_head_kv &&
         static_cast<int64_t>(n_head_kv) * head_dim <= INT_MAX / (BN * 4);
}

int attn_bf16x3(const float *q, const float *k, const float *v, const Pages *pages, float *out,
                int n_head, int n_head_kv, int head_dim, int64_t n_q, int64_t n_kv, int64_t n_past,
                float scale, hipStream_t s) {
  if (!attn_bf16x3_supported(q, k, v, out, n_head, n_head_kv, head_dim, n_q, n_kv, n_past)) return -ENOTSUP;
  const int G = n_head / n_head_kv;
  if (!(scale > 0.0f)) scale = 1.0f / sqrtf(static_cast<float>(head_dim));
  const float sl2 = scale * kLog2e;
  const int64_t rows = n_q * G;
  // cache rows behind the prompt (a longer cache, its rows not yet written)
  // are not read: a masked key's weight of 0 would not silence a NaN there
  n_kv = std::min(n_kv, n_past + n_q);
  auto us = [&](const Form &f) { return time_of(f, rows, G, n_kv, n_past, n_head_kv); };
#define IKV_A3(...)                                                                                \
  launch<__VA_ARGS__>(q, k, v, out, n_head_kv, G, head_dim, static_cast<int>(rows),                \
                      static_cast<int>(n_kv), static_cast<int>(n_past), sl2, pages, s)
  if (head_dim > 64) {
    if (us(kForms128[0]) <= us(kForms128[1]))
      IKV_A3(4, 4, 1, 1);
    else
      IKV_A3(4, 2, 2, 1);
  } else {
    if (us(kForms64[0]) <= us(kForms64[1]))
      IKV_A3(2, 2, 2, 2);
    else
      IKV_A3(2, 1, 4, 1);
  }
#undef IKV_A3
  return launch_status();
}

}  // namespace ikv
