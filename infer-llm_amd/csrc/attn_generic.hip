// attn_generic.hip — causal GQA attention for the shapes the tuned kernels
// (attn_decode.hip, attn_prefill.hip: head_dim 128, query groups of 1, 2, 4
// or 8) do not take: any head_dim up to kGenericMaxDim and any ratio of query
// to KV heads, contiguous or paged caches. The semantics are
// CPUBackend::compute_flash_attn's (src/backends/cpu_backend.cpp:525-634):
// key j is visible to query t iff j <= n_past + t and j < n_kv; q head h
// reads KV head h / (n_head / n_head_kv).
//
// Prompts with long rows and head_dim a multiple of 4 up to 128 go to
// attn_bf16x3.hip. Others (and any n_q): a workgroup of 4 wavefronts owns 16 query rows of
// one KV head g (row r = token * G + query head in the group, so a block of
// rows covers every query head of its tokens and each K / V tile serves all
// of them). Key tiles of KT rows (64 keys for head_dim <= 128, fewer for
// wider heads so a tile stays about 34 KB) are staged in LDS (16-byte loads
// when rows are 16-byte aligned) with rows padded by 4 floats (16-byte reads
// from 16 rows hit distinct banks). A wave
// holds 4 rows: for the scores each lane takes a key (and, with KT < 64, a
// part of its dims, the parts summed by lane swaps) and forms its dot with
// the 4 query rows, broadcast from LDS; online softmax in base 2 per row
// over the wave; the weights go through LDS and every lane then adds the
// tile's V rows for its output dims (lane, lane + 64, ...), once per key for
// all 4 rows.
//
// One query token (a decode step): the split form below.
#include "attn_bf16x3.hpp"
#include "attn_generic.hpp"
#include "ikv_common.hpp"

#include <algorithm>
#include <climits>
#include <initializer_list>

namespace {

// Pool row of logical key j (per lane): table[j / bt] * bt + j % bt; an entry
// outside the pool reads block 0 and raises IKV_STATUS_BLOCK.
__device__ __forceinline__ int64_t key_row(const ikv::Pages &pg, bool paged, int j) {
  if (!paged) return j;
  const int b = j / pg.bt;
  int blk = pg.table[b];
  if (static_cast<unsigned>(blk) >= static_cast<unsigned>(pg.n_blocks)) {
    ikv::raise_status(pg.status, IKV_STATUS_BLOCK);
    blk = 0;
  }
  return static_cast<int64_t>(blk) * pg.bt + (j - b * pg.bt);
}

// Keys of the longest row from which attn_bf16x3 takes a prompt: 12 heads of
// 64 over 4, 64 tokens 7.4 us here against 8.3 there, 128 tokens 11.0 against
// 10.5, 37 tokens behind 1000 65 against 28; heads of 80, 100 tokens 16.6
// against 14.5. From here on it was ahead at every shape measured (3 to 128
// heads of 32 to 96 over 1 to 128, up to 3500 tokens).
constexpr int64_t kPiecesMinKeys = 96;

constexpr int kTileRowsPerWave = 4;  // 8 measured slower (fewer workgroups, more registers)
constexpr int kTileRows = 4 * kTileRowsPerWave;  // query rows per workgroup

template <int DL>  // dims per lane: head_dim <= 64 * DL
__global__ __launch_bounds__(256) void generic_tile_kernel(
    const float *__restrict__ q, const float *__restrict__ k, const float *__restrict__ v,
    float *__restrict__ out, int n_head, int n_head_kv, int dim, int n_q, int n_kv, int n_past,
    float scale_log2, bool paged, ikv::Pages pg, bool vec4) {
  constexpr int KT = DL <= 2 ? 64 : 128 / DL;  // keys per tile: 64, 64, 32, 16
  constexpr int LPK = 64 / KT;                 // lanes per key in the score phase
  constexpr int DA = 64 * DL;                  // dims held (zeros past head_dim)
  constexpr int DP = DA + 4;                   // padded LDS row
  constexpr int DPART = DA / LPK;              // dims of a lane's score part
  constexpr int RW = kTileRowsPerWave;
  __shared__ __attribute__((aligned(16))) float s_k[KT * DP];
  __shared__ __attribute__((aligned(16))) float s_v[KT * DP];
  __shared__ __attribute__((aligned(16))) float s_q[kTileRows * DP];
  __shared__ __attribute__((aligned(16))) float s_p[4][RW][KT];
  const int G = n_head / n_head_kv;
  const int g = static_cast<int>(blockIdx.x) % n_head_kv;
  const int blk = static_cast<int>(blockIdx.x) / n_head_kv;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n_rows = n_q * G;
  const int r0 = blk * kTileRows;
  const size_t tok_stride = static_cast<size_t>(n_head_kv) * dim;
  const size_t head_off = static_cast<size_t>(g) * dim;

  // the block's query rows, pre-scaled, zero past head_dim and past the rows
  for (int i = tid; i < kTileRows * DA; i += 256) {
    const int rr = i / DA, d = i - rr * DA;
    const int r = r0 + rr;
    float x = 0.f;
    if (r < n_rows && d < dim) {
      const int t = r / G, hh = r - t * G;
      x = q[(static_cast<size_t>(t) * n_head + g * G + hh) * dim + d] * scale_log2;
    }
    s_q[rr * DP + d] = x;
  }
  const int r_last = min(r0 + kTileRows, n_rows) - 1;
  const int kv_end = min(n_kv, n_past + r_last / G + 1);  // keys any row of the block sees

  int tok[RW];
  bool rok[RW];
  float m[RW], l[RW], o[RW][DL];
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const int r = r0 + wave * RW + i;
    rok[i] = r < n_rows;
    tok[i] = rok[i] ? r / G : 0;
    m[i] = -INFINITY;
    l[i] = 0.f;
#pragma unroll
    for (int t = 0; t < DL; ++t) o[i][t] = 0.f;
  }
  const int jl = lane % KT;    // this lane's key in the score phase
  const int part = lane / KT;  // and its part of the dims
  for (int kb = 0; kb < kv_end; kb += KT) {
    __syncthreads();  // the previous tile's readers are done (and q is staged)
    if (vec4) {
      // 16-byte pieces: thread tid takes piece c = tid + 256 i of the tile
      constexpr int P4 = DA / 4;  // pieces per padded row
#pragma unroll
      for (int i = 0; i < KT * P4 / 256; ++i) {
        const int c = tid + 256 * i;
        const int jj = c / P4, d = 4 * (c - jj * P4);
        const int j = kb + jj;
        float4 kx = make_float4(0.f, 0.f, 0.f, 0.f), vx = kx;
        if (j < kv_end && d < dim) {
          const int64_t row = key_row(pg, paged, j);
          kx = *reinterpret_cast<const float4 *>(k + row * tok_stride + head_off + d);
          vx = *reinterpret_cast<const float4 *>(v + row * tok_stride + head_off + d);
        }
        *reinterpret_cast<float4 *>(s_k + jj * DP + d) = kx;
        *reinterpret_cast<float4 *>(s_v + jj * DP + d) = vx;
      }
    } else {
      for (int i = tid; i < KT * DA; i += 256) {
        const int jj = i / DA, d = i - jj * DA;
        const int j = kb + jj;
        float kx = 0.f, vx = 0.f;
        if (j < kv_end && d < dim) {
          const int64_t row = key_row(pg, paged, j);
          kx = k[row * tok_stride + head_off + d];
          vx = v[row * tok_stride + head_off + d];
        }
        s_k[jj * DP + d] = kx;
        s_v[jj * DP + d] = vx;
      }
    }
    __syncthreads();
    // scores of key kb + jl with the wave's 4 rows, over this lane's part
    float sc[RW];
#pragma unroll
    for (int i = 0; i < RW; ++i) sc[i] = 0.f;
    const float *kp = s_k + jl * DP + part * DPART;
    const float *qp = s_q + (wave * RW) * DP + part * DPART;
#pragma unroll 4
    for (int d4 = 0; d4 < DPART; d4 += 4) {
      const float4 kx = *reinterpret_cast<const float4 *>(kp + d4);
#pragma unroll
      for (int i = 0; i < RW; ++i) {
        const float4 qx = *reinterpret_cast<const float4 *>(qp + i * DP + d4);
        sc[i] = fmaf(qx.x, kx.x, sc[i]);
        sc[i] = fmaf(qx.y, kx.y, sc[i]);
        sc[i] = fmaf(qx.z, kx.z, sc[i]);
        sc[i] = fmaf(qx.w, kx.w, sc[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      if constexpr (LPK >= 2) {  // parts at lanes l, l ^ 32 (and l ^ 16)
        auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(sc[i]), __float_as_uint(sc[i]),
                                                  false, false);
        sc[i] = __uint_as_float(a[0]) + __uint_as_float(a[1]);
      }
      if constexpr (LPK >= 4) {
        auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(sc[i]), __float_as_uint(sc[i]),
                                                  false, false);
        sc[i] = __uint_as_float(b[0]) + __uint_as_float(b[1]);
      }
    }
    const int j = kb + jl;
    float alpha[RW];
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const bool vis = rok[i] && j < kv_end && j <= n_past + tok[i];
      const float s = vis ? sc[i] : -INFINITY;
      const float m_new = fmaxf(m[i], ikv::wave_max(s));
      // a row that has seen no key yet keeps a zero state (reference 0)
      const float ref = (m_new == -INFINITY) ? 0.f : m_new;
      alpha[i] = ikv::fast_exp2(m[i] - ref);
      const float p = ikv::fast_exp2(s - ref);
      l[i] = fmaf(l[i], alpha[i], ikv::wave_sum(part == 0 ? p : 0.f));
      if (part == 0) s_p[wave][i][jl] = p;
      m[i] = m_new;
    }
    // the wave's weights are in LDS (its own writes, in order): add V
#pragma unroll
    for (int i = 0; i < RW; ++i)
#pragma unroll
      for (int t = 0; t < DL; ++t) o[i][t] *= alpha[i];
    for (int j4 = 0; j4 < KT; j4 += 4) {  // 4 keys: the rows' weights as one 16-byte read
      float vd[4][DL];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int t = 0; t < DL; ++t) vd[u][t] = s_v[(j4 + u) * DP + lane + 64 * t];
#pragma unroll
      for (int i = 0; i < RW; ++i) {
        const float4 pj = *reinterpret_cast<const float4 *>(&s_p[wave][i][j4]);
#pragma unroll
        for (int t = 0; t < DL; ++t) {
          o[i][t] = fmaf(pj.x, vd[0][t], o[i][t]);
          o[i][t] = fmaf(pj.y, vd[1][t], o[i][t]);
          o[i][t] = fmaf(pj.z, vd[2][t], o[i][t]);
          o[i][t] = fmaf(pj.w, vd[3][t], o[i][t]);
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    if (!rok[i]) continue;
    const int r = r0 + wave * RW + i;
    const int hh = r - tok[i] * G;
    float *orow = out + (static_cast<size_t>(tok[i]) * n_head + g * G + hh) * dim;
    const float inv = 1.0f / l[i];
#pragma unroll
    for (int t = 0; t < DL; ++t) {
      const int d = lane + 64 * t;
      if (d < dim) orow[d] = o[i][t] * inv;
    }
  }
}

// ---------------------------------------------------------------------------
// One query token (a decode step), split over the context: workgroup
// (KV head g, split) serves all G query heads of g over keys [t_begin,
// t_end), so every K and V row is read once. Its 4 wavefronts take keys
// t_begin + wave, + 4, ...; a key's row is spread over the lanes (dims lane,
// lane + 64, ...: DL per lane, head_dim <= 64 DL), loaded 4 keys ahead, and
// each query head's score is a wave sum. Online softmax in base 2 per head;
// the waves meet in LDS and the split's (max, sum, unnormalised output) per
// head goes to the workspace; a second launch merges the splits in split
// order. Registers hold G x DL query and output values per lane: G * DL <=
// kSplitHeadDims.
constexpr int kSplitHeadDims = 32;
constexpr int kSplitWaves = 4;
// keys per wave in flight: 16 dims' worth of registers per lane for K and V
constexpr int split_ahead(int dl) { return dl >= 8 ? 2 : 16 / dl; }
constexpr int kSplitMinKeys = 64;
constexpr int kSplitTargetWgs = 256;  // one per MI355X compute unit

template <int DL>
__global__ __launch_bounds__(kSplitWaves * 64) void generic_split_kernel(
    const float *__restrict__ q, const float *__restrict__ k, const float *__restrict__ v,
    float *__restrict__ part_ml, float *__restrict__ part_o, int n_head_kv, int G, int dim,
    int n_kv, int keys_per_split, int n_splits, float scale_log2, bool paged, ikv::Pages pg) {
  constexpr int GM = kSplitHeadDims / DL;  // most query heads per KV head
  constexpr int kSplitAhead = split_ahead(DL);
  __shared__ float s_m[kSplitWaves][GM], s_l[kSplitWaves][GM];
  __shared__ float s_o[kSplitWaves][GM][64 * DL];
  const int g = static_cast<int>(blockIdx.x) % n_head_kv;
  const int split = static_cast<int>(blockIdx.x) / n_head_kv;
  const int t_begin = split * keys_per_split;
  const int t_end = min(n_kv, t_begin + keys_per_split);
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const size_t tok_stride = static_cast<size_t>(n_head_kv) * dim;
  const size_t head_off = static_cast<size_t>(g) * dim;

  float qv[GM][DL], o[GM][DL], m[GM], l[GM];
#pragma unroll
  for (int h = 0; h < GM; ++h) {
    m[h] = -INFINITY;
    l[h] = 0.f;
#pragma unroll
    for (int t = 0; t < DL; ++t) {
      const int d = lane + 64 * t;
      qv[h][t] = (h < G && d < dim)
                     ? q[(static_cast<size_t>(g) * G + h) * dim + d] * scale_log2
                     : 0.f;
      o[h][t] = 0.f;
    }
  }
  for (int j0 = t_begin + wave; j0 < t_end; j0 += kSplitWaves * kSplitAhead) {
    float kr[kSplitAhead][DL], vr[kSplitAhead][DL];
#pragma unroll
    for (int u = 0; u < kSplitAhead; ++u) {
      const int j = j0 + kSplitWaves * u;
      const bool ok = j < t_end;
      const int64_t row = key_row(pg, paged, ok ? j : t_begin);
      const float *kp = k + row * tok_stride + head_off;
      const float *vp = v + row * tok_stride + head_off;
#pragma unroll
      for (int t = 0; t < DL; ++t) {
        const int d = lane + 64 * t;
        kr[u][t] = (ok && d < dim) ? kp[d] : 0.f;
        vr[u][t] = (ok && d < dim) ? vp[d] : 0.f;
      }
    }
    // per query head: the chunk's scores (independent wave sums), then one
    // online-softmax step over them (the chunk's first key is always valid)
#pragma unroll
    for (int h = 0; h < GM; ++h) {
      if (h < G) {  // (guards, not breaks: the register arrays stay unrolled)
        float sc[kSplitAhead];
#pragma unroll
        for (int u = 0; u < kSplitAhead; ++u) {
          float part = 0.f;
#pragma unroll
          for (int t = 0; t < DL; ++t) part = fmaf(qv[h][t], kr[u][t], part);
          const float w = ikv::wave_sum(part);
          sc[u] = (j0 + kSplitWaves * u < t_end) ? w : -INFINITY;
        }
        float mx = m[h];
#pragma unroll
        for (int u = 0; u < kSplitAhead; ++u) mx = fmaxf(mx, sc[u]);
        const float alpha = ikv::fast_exp2(m[h] - mx);  // 0 on the first chunk
        float psum = 0.f;
#pragma unroll
        for (int t = 0; t < DL; ++t) o[h][t] *= alpha;
#pragma unroll
        for (int u = 0; u < kSplitAhead; ++u) {
          const float pu = ikv::fast_exp2(sc[u] - mx);  // 0 for a key past the split
          psum += pu;
#pragma unroll
          for (int t = 0; t < DL; ++t) o[h][t] = fmaf(pu, vr[u][t], o[h][t]);
        }
        l[h] = fmaf(l[h], alpha, psum);
        m[h] = mx;
      }
    }
  }
  // the waves meet in LDS (a wave with no key holds m = -inf, l = 0, o = 0)
#pragma unroll
  for (int h = 0; h < GM; ++h) {
    if (h < G) {
      if (lane == 0) {
        s_m[wave][h] = m[h];
        s_l[wave][h] = l[h];
      }
#pragma unroll
      for (int t = 0; t < DL; ++t) s_o[wave][h][lane + 64 * t] = o[h][t];
    }
  }
  __syncthreads();
  const size_t rec0 = static_cast<size_t>(g) * G * n_splits + split;  // record of head 0
  for (int idx = threadIdx.x; idx < G * dim; idx += kSplitWaves * 64) {
    const int h = idx / dim, d = idx - h * dim;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < kSplitWaves; ++w) M = fmaxf(M, s_m[w][h]);
    float L = 0.f, O = 0.f;
#pragma unroll
    for (int w = 0; w < kSplitWaves; ++w) {
      const float mw = s_m[w][h];
      const float e = (mw == -INFINITY) ? 0.f : ikv::fast_exp2(mw - M);
      L = fmaf(e, s_l[w][h], L);
      O = fmaf(e, s_o[w][h][d], O);
    }
    const size_t rec = rec0 + static_cast<size_t>(h) * n_splits;
    part_o[rec * dim + d] = O;
    if (d == 0) {
      part_ml[2 * rec] = M;
      part_ml[2 * rec + 1] = L;
    }
  }
}

// out[head][d] = sum_s e_s O_s[d] / sum_s e_s L_s, e_s = 2^(M_s - max_s M_s):
// one workgroup per query head. Wave 0 forms the weights (lanes over splits)
// and the sum; the threads take output dims, and where a head has at most
// 128 of them several threads share a dim, each taking a run of the splits,
// the runs added in order. All latency: a thread's first AHEAD partials load
// while wave 0 forms the weights (40 splits of 64 dims 4.1 -> 3.7 us), and no
// branch stands between the loads or between the weights (with one per split, a
// decode step of 6 heads of 300 over 2 at 9000 keys took 45 us, 35 without).
constexpr int kMergeThreads = 256;
constexpr int kMaxAhead = 16;
constexpr int merge_runs(int dim) { return dim <= 64 ? 4 : dim <= 128 ? 2 : 1; }
template <int AHEAD>
__global__ __launch_bounds__(kMergeThreads) void generic_merge_kernel(
    const float *__restrict__ part_ml, const float *__restrict__ part_o, float *__restrict__ out,
    int dim, int n_splits) {
  constexpr int kPerLane = kSplitTargetWgs / 64;
  __shared__ float s_e[kSplitTargetWgs + kMaxAhead];
  __shared__ float s_L;
  __shared__ float s_part[kMergeThreads];
  const int head = blockIdx.x;
  const size_t rec0 = static_cast<size_t>(head) * n_splits;
  const int runs = merge_runs(dim);
  const int per = kMergeThreads / runs, r = threadIdx.x / per;
  const int lo = r * n_splits / runs, hi = (r + 1) * n_splits / runs;
  float a[AHEAD];
  // no branch between the loads (past the run: the last split's, as 0)
  auto load = [&](int d, int sp0) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
      a[u] = part_o[(rec0 + min(sp0 + u, n_splits - 1)) * dim + min(d, dim - 1)];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
      if (sp0 + u >= hi) a[u] = 0.f;
  };
  load(threadIdx.x % per, lo);
  if (threadIdx.x >= kMergeThreads - kMaxAhead)
    s_e[kSplitTargetWgs + kMergeThreads - 1 - threadIdx.x] = 0.f;
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    float2 ml[kPerLane];
    float M = -INFINITY, L = 0.f;
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
      const int sp = lane + 64 * i;
      ml[i] = make_float2(-INFINITY, 0.f);
      if (sp < n_splits) ml[i] = reinterpret_cast<const float2 *>(part_ml)[rec0 + sp];
    }
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) M = fmaxf(M, ml[i].x);
    M = ikv::wave_max(M);
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
      const float e = ml[i].x == -INFINITY ? 0.f : ikv::fast_exp2(ml[i].x - M);
      s_e[lane + 64 * i] = e;
      L = fmaf(e, ml[i].y, L);
    }
    L = ikv::wave_sum(L);
    if (lane == 0) s_L = L;
  }
  __syncthreads();
  const float inv = 1.0f / s_L;
  auto run = [&](int d) {
    float O = 0.f;
    for (int sp = lo; sp < hi; sp += AHEAD) {
      if (sp != lo) load(d, sp);
      // (a branch per split made each wait for its weight alone)
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) O = fmaf(s_e[sp + u], a[u], O);
    }
    return O;
  };
  if (runs > 1) {
    const int d = threadIdx.x % per;
    s_part[threadIdx.x] = run(d);
    __syncthreads();
    if (r == 0 && d < dim) {
      float O = s_part[d];
      for (int i = 1; i < runs; ++i) O += s_part[i * per + d];
      out[static_cast<size_t>(head) * dim + d] = O * inv;
    }
    return;
  }
  for (int d = threadIdx.x; d < dim; d += kMergeThreads) {
    if (d != static_cast<int>(threadIdx.x)) load(d, lo);
    out[static_cast<size_t>(head) * dim + d] = run(d) * inv;
  }
}

void merge(const float *part_ml, const float *part_o, float *out, int n_head, int dim, int n_splits,
           hipStream_t s) {
  // (few splits: a short batch, whose loads past the run cost less)
  const auto kernel = n_splits <= 4 * merge_runs(dim) ? generic_merge_kernel<4> : generic_merge_kernel<kMaxAhead>;
  kernel<<<static_cast<unsigned>(n_head), kMergeThreads, 0, s>>>(part_ml, part_o, out, dim, n_splits);
}

// The split decode for rows of 16-byte pieces: head_dim a multiple of 4 up to
// 256, at most 8 query heads per KV head. LPK lanes (a power of two >= dim / 4)
// hold a key's row, a float4 each, so a wave scores 64 / LPK keys at once and a
// score's sum takes log2(LPK) lane steps for all of them (generic_split_kernel
// spends a 64-lane sum per key and head: its sums were most of its time). Each
// lane group keeps its own softmax state; the states of the workgroup's 4
// waves meet in LDS. The new token is folded in: with k_new, the split that
// holds key n_kv - 1 takes its rows from there and writes them to the caches,
// and with PRO every split first forms its rotated q rows (and that one the k
// row), with the operations of head_rope_kernel, while its first keys are in
// flight. Latency-bound at these sizes, hence one launch for what took five:
// 12 heads of 64 over 4 at 2500 keys, with qk-norm + RoPE, 21.1 us in five
// launches before, 6.4 here.
template <int LPK, int GM, bool PRO>
__global__ __launch_bounds__(256) void decode_rows_kernel(
    const float *__restrict__ q, float *__restrict__ k, float *__restrict__ v,
    const float *__restrict__ k_new, const float *__restrict__ v_new, float *__restrict__ part_ml,
    float *__restrict__ part_o, int n_head_kv, int G, int dim, int n_kv, int keys_per_split,
    int n_splits, float scale_log2, bool paged, ikv::Pages pg, ikv::DecodeNew pro) {
  constexpr int KPW = 64 / LPK;            // keys a wave scores at once
  constexpr int U = LPK == 16 ? 4 : 8;     // of them in flight
  constexpr int STATES = 4 * KPW;
  __shared__ __attribute__((aligned(16))) float s_q[GM * 4 * LPK], s_kn[4 * LPK], s_vn[4 * LPK];
  __shared__ float s_m[STATES][GM], s_l[STATES][GM];
  __shared__ __attribute__((aligned(16))) float s_o[STATES][GM][4 * LPK];
  const int g = static_cast<int>(blockIdx.x) % n_head_kv;
  const int split = static_cast<int>(blockIdx.x) / n_head_kv;
  const int t_begin = split * keys_per_split;
  const int t_end = min(n_kv, t_begin + keys_per_split);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane % LPK, state = wave * KPW + lane / LPK;
  const bool on = 4 * c < dim;
  const size_t tok_stride = static_cast<size_t>(n_head_kv) * dim;
  const size_t at = static_cast<size_t>(g) * dim + 4 * c;
  const bool newest = k_new && t_end == n_kv;  // this split holds the new token
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);

  float4 kr[U], vr[U];
  auto load = [&](int j0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = j0 + STATES * u;
      const int64_t row = key_row(pg, paged, j < t_end ? j : t_begin);
      kr[u] = vr[u] = zero;
      if (on && j < t_end) {
        kr[u] = *reinterpret_cast<const float4 *>(k + row * tok_stride + at);
        vr[u] = *reinterpret_cast<const float4 *>(v + row * tok_stride + at);
      }
    }
  };
  load(t_begin + state);

  if constexpr (PRO) {
#pragma clang fp contract(off)
    constexpr int HD = 2 * LPK;  // dim == 4 LPK; lane c holds the pairs (2c, 2c + 1) of both halves
    const int32_t p = pro.pos[0];
    const bool in = p >= 0 && p < pro.n_ctx;
    const size_t ang = static_cast<size_t>(in ? p : 0) * HD;
    const float2 cs = reinterpret_cast<const float2 *>(pro.cos_tab + ang)[c];
    const float2 sn = reinterpret_cast<const float2 *>(pro.sin_tab + ang)[c];
    const int rows = G + (newest ? 1 : 0);  // row G: the key
    for (int r0 = 0; r0 < rows; r0 += STATES) {
      const int r = min(r0 + state, rows - 1);
      const float *x = r < G ? q + (static_cast<size_t>(g) * G + r) * dim : k_new + static_cast<size_t>(g) * dim;
      const float *w = r < G ? pro.q_norm_w : pro.k_norm_w;
      float2 lo = reinterpret_cast<const float2 *>(x)[c], hi = reinterpret_cast<const float2 *>(x)[LPK + c];
      const float2 wl = reinterpret_cast<const float2 *>(w)[c], wh = reinterpret_cast<const float2 *>(w)[LPK + c];
      const double sq = ikv::add_squares(0.0, make_float4(lo.x, lo.y, hi.x, hi.y));
      const double sum = LPK == 16   ? ikv::row16_sum_f64(sq)
                         : LPK == 32 ? ikv::half_wave_sum_f64(sq)
                                     : ikv::wave_sum_f64(sq);
      float sc = -1.f;
      if (!ikv::certified_rms_scale(sum, 4 * LPK, pro.eps, (4 * LPK - 1) + 4 + 6, sc)) sc = -1.f;
      for (unsigned long long todo = __builtin_amdgcn_ballot_w64(sc < 0.f); todo != 0;) {
        const int src = __builtin_ctzll(todo);
        const int rr = __builtin_amdgcn_readlane(r, src);
        const float *xr = rr < G ? q + (static_cast<size_t>(g) * G + rr) * dim : k_new + static_cast<size_t>(g) * dim;
        const float sx = ikv::ordered_rms_scale_wave(xr, 4 * LPK, pro.eps, lane);
        if (lane / LPK == src / LPK) sc = sx;
        todo &= ~((LPK == 64 ? ~0ull : (1ull << (LPK % 64)) - 1) << (src / LPK * LPK));
      }
      const float a0 = lo.x * sc, a1 = lo.y * sc, b0 = hi.x * sc, b1 = hi.y * sc;
      const float x0 = a0 * wl.x, x1 = a1 * wl.y, y0 = b0 * wh.x, y1 = b1 * wh.y;
      const float m0 = x0 * cs.x, n0 = y0 * sn.x, m1 = x1 * cs.y, n1 = y1 * sn.y;
      const float e0 = x0 * sn.x, f0 = y0 * cs.x, e1 = x1 * sn.y, f1 = y1 * cs.y;
      float *dst = r < G ? s_q + r * 4 * LPK : s_kn;
      reinterpret_cast<float2 *>(dst)[c] = in ? make_float2(m0 - n0, m1 - n1) : make_float2(0.f, 0.f);
      reinterpret_cast<float2 *>(dst)[LPK + c] = in ? make_float2(e0 + f0, e1 + f1) : make_float2(0.f, 0.f);
    }
    if (!in && newest && threadIdx.x == 0) ikv::raise_status(pro.status, IKV_STATUS_POSITION);
  } else {
    for (int i = threadIdx.x; i < G * dim; i += 256)
      s_q[i / dim * 4 * LPK + i % dim] = q[static_cast<size_t>(g) * G * dim + i];
    if (newest)
      for (int i = threadIdx.x; i < dim; i += 256) s_kn[i] = k_new[static_cast<size_t>(g) * dim + i];
  }
  if (newest)
    for (int i = threadIdx.x; i < dim; i += 256) s_vn[i] = v_new[static_cast<size_t>(g) * dim + i];
  __syncthreads();
  if (newest && threadIdx.x < LPK && on) {  // the append
    const int64_t row = key_row(pg, paged, n_kv - 1);
    if (!paged || ikv::page_ok(pg, n_kv - 1)) {
      *reinterpret_cast<float4 *>(k + row * tok_stride + at) = *reinterpret_cast<const float4 *>(s_kn + 4 * c);
      *reinterpret_cast<float4 *>(v + row * tok_stride + at) = *reinterpret_cast<const float4 *>(s_vn + 4 * c);
    }
  }

  float4 qv[GM], o[GM];
  float m[GM], l[GM];
#pragma unroll
  for (int h = 0; h < GM; ++h) {
    qv[h] = h < G && on ? ikv::scale4(scale_log2, *reinterpret_cast<const float4 *>(s_q + h * 4 * LPK + 4 * c)) : zero;
    o[h] = zero;
    m[h] = -INFINITY;
    l[h] = 0.f;
  }
  for (int j0 = t_begin + state; j0 - state < t_end; j0 += STATES * U) {
    if (j0 - state != t_begin) load(j0);
    if (newest) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (j0 + STATES * u == n_kv - 1 && on) {
          kr[u] = *reinterpret_cast<const float4 *>(s_kn + 4 * c);
          vr[u] = *reinterpret_cast<const float4 *>(s_vn + 4 * c);
        }
    }
#pragma unroll
    for (int h = 0; h < GM; ++h) {
      if (h < G) {
        float sc[U], mx = m[h];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const float d = ikv::dot4(qv[h], kr[u]);
          const float w = LPK == 16   ? ikv::row16_sum(d)
                          : LPK == 32 ? ikv::half_wave_sum_valu(d)
                                      : ikv::wave_sum(d);
          sc[u] = j0 + STATES * u < t_end ? w : -INFINITY;
          mx = fmaxf(mx, sc[u]);
        }
        // a lane group without a key yet keeps a zero state (reference 0)
        const float ref = mx == -INFINITY ? 0.f : mx;
        const float alpha = ikv::fast_exp2(m[h] - ref);
        float psum = 0.f;
        o[h] = ikv::scale4(alpha, o[h]);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const float pu = ikv::fast_exp2(sc[u] - ref);
          psum += pu;
          o[h] = ikv::fma4(pu, vr[u], o[h]);
        }
        l[h] = fmaf(l[h], alpha, psum);
        m[h] = mx;
      }
    }
  }
#pragma unroll
  for (int h = 0; h < GM; ++h) {
    if (h < G) {
      if (c == 0) {
        s_m[state][h] = m[h];
        s_l[state][h] = l[h];
      }
      *reinterpret_cast<float4 *>(&s_o[state][h][4 * c]) = o[h];
    }
  }
  __syncthreads();
  const size_t rec0 = static_cast<size_t>(g) * G * n_splits + split;  // record of head 0
  for (int idx = threadIdx.x; idx < G * dim; idx += 256) {
    const int h = idx / dim, d = idx - h * dim;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < STATES; ++w) M = fmaxf(M, s_m[w][h]);
    float L = 0.f, O = 0.f;
#pragma unroll
    for (int w = 0; w < STATES; ++w) {
      const float mw = s_m[w][h];
      const float e = mw == -INFINITY ? 0.f : ikv::fast_exp2(mw - M);
      L = fmaf(e, s_l[w][h], L);
      O = fmaf(e, s_o[w][h][d], O);
    }
    const size_t rec = rec0 + static_cast<size_t>(h) * n_splits;
    part_o[rec * dim + d] = O;
    if (d == 0) {
      part_ml[2 * rec] = M;
      part_ml[2 * rec + 1] = L;
    }
  }
}

struct SplitPlan {
  int dl = 0;  // dims per lane; 0: the shape does not fit the split kernel
  int n_splits = 0, keys_per_split = 0;
};

SplitPlan split_plan(int n_head, int n_head_kv, int head_dim, int64_t n_kv) {
  SplitPlan p;
  const int G = n_head / n_head_kv;
  const int dl = head_dim <= 64 ? 1 : head_dim <= 128 ? 2 : head_dim <= 256 ? 4 : 8;
  if (G * dl > kSplitHeadDims || n_kv < 1 || n_kv > INT_MAX / 2) return p;
  const int64_t target = std::max<int64_t>(1, (kSplitTargetWgs + n_head_kv - 1) / n_head_kv);
  int64_t per = (n_kv + target - 1) / target;
  if (per < kSplitMinKeys) per = kSplitMinKeys;
  p.dl = dl;
  p.keys_per_split = static_cast<int>(per);
  p.n_splits = static_cast<int>((n_kv + per - 1) / per);
  return p;
}

size_t split_ws_bytes(int n_head, int head_dim, int n_splits) {
  const size_t ml = (sizeof(float) * 2 * static_cast<size_t>(n_head) * n_splits + 255) & ~size_t(255);
  return ml + sizeof(float) * static_cast<size_t>(n_head) * n_splits * head_dim;
}

}  // namespace

namespace ikv {

bool generic_attn_shape(int n_head, int n_head_kv, int head_dim) {
  return n_head > 0 && n_head_kv > 0 && n_head % n_head_kv == 0 && head_dim >= 1 &&
         head_dim <= kGenericMaxDim;
}

int attn_generic(const float *q, const float *k, const float *v, const Pages *pages, float *out,
                 int n_head, int n_head_kv, int head_dim, int64_t n_q, int64_t n_kv,
                 int64_t n_past, float scale, hipStream_t s) {
  if (n_q == 0) return 0;
  if (!generic_attn_shape(n_head, n_head_kv, head_dim)) return -ENOTSUP;
  if (n_q < 0 || n_kv <= 0 || n_past < 0) return -EINVAL;
  if (n_q > INT_MAX / n_head || n_kv > INT_MAX / 2 || n_past > INT_MAX / 2) return -EOVERFLOW;
  if (std::min(n_kv, n_past + n_q) >= kPiecesMinKeys &&
      attn_bf16x3_supported(q, k, v, out, n_head, n_head_kv, head_dim, n_q, n_kv, n_past))
    return attn_bf16x3(q, k, v, pages, out, n_head, n_head_kv, head_dim, n_q, n_kv, n_past, scale, s);
  if (!(scale > 0.0f)) scale = 1.0f / sqrtf(static_cast<float>(head_dim));
  const int dl = head_dim <= 64 ? 1 : head_dim <= 128 ? 2 : head_dim <= 256 ? 4 : 8;
  const int64_t rows = n_q * (n_head / n_head_kv);
  const int64_t blocks = (rows + kTileRows - 1) / kTileRows;
  if (blocks * n_head_kv > INT_MAX) return -EOVERFLOW;
  const unsigned grid = static_cast<unsigned>(blocks * n_head_kv);
  const float sl2 = scale * kLog2e;
  const Pages pgv = pages ? *pages : Pages{};
  // K and V rows staged 16 bytes at a time when every row starts 16-byte
  // aligned
  const bool vec4 = head_dim % 4 == 0 && aligned16(k) && aligned16(v);
#define IKV_GENERIC_TILE(DD)                                                                  \
  generic_tile_kernel<DD><<<grid, 256, 0, s>>>(q, k, v, out, n_head, n_head_kv, head_dim,     \
                                               static_cast<int>(n_q), static_cast<int>(n_kv), \
                                               static_cast<int>(n_past), sl2, pages != nullptr, pgv, \
                                               vec4)
  switch (dl) {
    case 1: IKV_GENERIC_TILE(1); break;
    case 2: IKV_GENERIC_TILE(2); break;
    case 4: IKV_GENERIC_TILE(4); break;
    default: IKV_GENERIC_TILE(8); break;
  }
#undef IKV_GENERIC_TILE
  return launch_status();
}

}  // namespace ikv

namespace ikv {

size_t generic_decode_ws_bytes(int n_head, int n_head_kv, int head_dim, int64_t n_kv) {
  if (!generic_attn_shape(n_head, n_head_kv, head_dim)) return 0;
  const SplitPlan p = split_plan(n_head, n_head_kv, head_dim, n_kv);
  return p.dl ? split_ws_bytes(n_head, head_dim, p.n_splits) : 0;
}

bool generic_decode_folds(const float *q, const float *k, const float *v, const float *k_new,
                          const float *v_new, const Pages *pages, int n_head, int n_head_kv,
                          int head_dim, int64_t n_kv, const void *workspace,
                          size_t workspace_bytes, const DecodeNew *pro) {
  if (head_dim % 4 != 0 || head_dim > 256 || n_head / n_head_kv > 8 || n_kv <= 0) return false;
  if (!aligned16(k) || !aligned16(v) || !workspace || !aligned16(workspace)) return false;
  const SplitPlan p = split_plan(n_head, n_head_kv, head_dim, n_kv);
  if (!p.dl || workspace_bytes < split_ws_bytes(n_head, head_dim, p.n_splits)) return false;
  if (pages && k_new && (!aligned16(v_new) || (!pro && !aligned16(k_new)))) return false;
  if (!pro) return true;
  // head_rope_kernel's head sizes and alignment: the same rows, bit for bit
  if (head_dim != 64 && head_dim != 128 && head_dim != 256) return false;
  for (const void *x : {static_cast<const void *>(q), static_cast<const void *>(k_new),
                        static_cast<const void *>(pro->q_norm_w), static_cast<const void *>(pro->k_norm_w),
                        static_cast<const void *>(pro->sin_tab), static_cast<const void *>(pro->cos_tab)})
    if (reinterpret_cast<uintptr_t>(x) & 7) return false;
  return true;
}

int attn_generic_decode_folded(const float *q, float *k, float *v, const float *k_new,
                               const float *v_new, const Pages *pages, float *out, int n_head,
                               int n_head_kv, int head_dim, int64_t n_kv, float scale,
                               void *workspace, const DecodeNew *pro, hipStream_t s) {
  const SplitPlan p = split_plan(n_head, n_head_kv, head_dim, n_kv);
  if (!(scale > 0.0f)) scale = 1.0f / sqrtf(static_cast<float>(head_dim));
  float *part_ml = static_cast<float *>(workspace);
  float *part_o = part_ml + ((sizeof(float) * 2 * static_cast<size_t>(n_head) * p.n_splits + 255) & ~size_t(255)) / sizeof(float);
  const unsigned grid = static_cast<unsigned>(n_head_kv) * static_cast<unsigned>(p.n_splits);
  const int G = n_head / n_head_kv;
  const Pages pg = pages ? *pages : Pages{};
  const DecodeNew nw = pro ? *pro : DecodeNew{};
#define IKV_ROWS(LPK, GM, PRO)                                                                        \
  decode_rows_kernel<LPK, GM, PRO><<<grid, 256, 0, s>>>(                                              \
      q, k, v, k_new, v_new, part_ml, part_o, n_head_kv, G, head_dim, static_cast<int>(n_kv),         \
      p.keys_per_split, p.n_splits, scale * kLog2e, pages != nullptr, pg, nw)
#define IKV_ROWS_G(LPK)                                                            \
  do {                                                                             \
    if (pro) {                                                                     \
      if (G <= 4) IKV_ROWS(LPK, 4, true); else IKV_ROWS(LPK, 8, true);             \
    } else {                                                                       \
      if (G <= 4) IKV_ROWS(LPK, 4, false); else IKV_ROWS(LPK, 8, false);           \
    }                                                                              \
  } while (0)
  if (head_dim <= 64)
    IKV_ROWS_G(16);
  else if (head_dim <= 128)
    IKV_ROWS_G(32);
  else
    IKV_ROWS_G(64);
#undef IKV_ROWS_G
#undef IKV_ROWS
  merge(part_ml, part_o, out, n_head, head_dim, p.n_splits, s);
  return launch_status();
}

int attn_generic_decode(const float *q, const float *k, const float *v, const Pages *pages,
                        float *out, int n_head, int n_head_kv, int head_dim, int64_t n_kv,
                        float scale, void *workspace, size_t workspace_bytes, hipStream_t s) {
  if (!generic_attn_shape(n_head, n_head_kv, head_dim)) return -ENOTSUP;
  if (n_kv <= 0) return -EINVAL;
  const SplitPlan p = split_plan(n_head, n_head_kv, head_dim, n_kv);
  if (!p.dl || !workspace || !aligned16(workspace) ||
      workspace_bytes < split_ws_bytes(n_head, head_dim, p.n_splits))
    return attn_generic(q, k, v, pages, out, n_head, n_head_kv, head_dim, 1, n_kv, n_kv - 1,
                        scale, s);
  if (!(scale > 0.0f)) scale = 1.0f / sqrtf(static_cast<float>(head_dim));
  float *part_ml = static_cast<float *>(workspace);
  float *part_o = reinterpret_cast<float *>(
      static_cast<char *>(workspace) +
      ((sizeof(float) * 2 * static_cast<size_t>(n_head) * p.n_splits + 255) & ~size_t(255)));
  const unsigned grid = static_cast<unsigned>(n_head_kv) * static_cast<unsigned>(p.n_splits);
  const int G = n_head / n_head_kv;
  const float sl2 = scale * kLog2e;
  const Pages pg = pages ? *pages : Pages{};
#define IKV_GENERIC_SPLIT(DD)                                                                \
  generic_split_kernel<DD><<<grid, kSplitWaves * 64, 0, s>>>(                                \
      q, k, v, part_ml, part_o, n_head_kv, G, head_dim, static_cast<int>(n_kv),              \
      p.keys_per_split, p.n_splits, sl2, pages != nullptr, pg)
  switch (p.dl) {
    case 1: IKV_GENERIC_SPLIT(1); break;
    case 2: IKV_GENERIC_SPLIT(2); break;
    case 4: IKV_GENERIC_SPLIT(4); break;
    default: IKV_GENERIC_SPLIT(8); break;
  }
#undef IKV_GENERIC_SPLIT
  merge(part_ml, part_o, out, n_head, head_dim, p.n_splits, s);
  return launch_status();
}

}  // namespace ikv
