// rope_norm.hip — RMSNorm, NeoX RoPE and the fused qk-RMSNorm + RoPE that
// feed the KV append.
//
// Arithmetic of the reference CPU backend:
//   RMSNorm  (reference src/backends/cpu_backend.cpp:335-382): float squares
//            accumulated in double, scale = float(1.0 / sqrt(sum/dim + eps))
//            in double, out = (x*scale)*w; the order of the double sum is
//            below.
//   RoPE     (src/backends/cpu_backend.cpp:443-523): o_j = x0*c - x1*s,
//            o_{j+h} = x0*s + x1*c with c, s the glibc cosf/sinf of the angle
//            table entry; here they come from sin/cos tables built once on the
//            host (ikv_rope_sincos_table_f32) and kept resident in HBM.
// Contraction into FMA is disabled in this file so every product and sum
// rounds exactly as the reference's separate float operations do.
//
// Sums of squares: the reference adds a row's float squares in index order in
// double, a chain of dim dependent double adds (about 1.1 us for 128 on
// MI355X). The kernels add them in parallel instead and certify the float
// scale against the index-order sum (ikv::certified_rms_scale): the two sums
// differ by a bounded amount, and when the double scale is farther than that
// from a float rounding midpoint, both round to the same float. When it is
// not (about 2^-19 of rows of 1024 floats), the sum is redone in index order. Every
// scale is therefore the reference's bit for bit.
//  * rows shorter than kLongRow: half-wave per row, lane c adds elements c,
//    c + 32, ..., then a xor butterfly; the head rows of qk-norm: each lane
//    adds its four;
//  * rows of kLongRow or more floats, a multiple of 256 (the model-width
//    rows of attn_norm / ffn_norm / output_norm): one wavefront per row; lane
//    l adds the squares of elements 256*j + 4*l + c (j ascending, the four c
//    apart), then the lane sums combine. The GEMV kernels that fold this norm
//    into their input (ikv_model.h) certify the same scale.
//
// Head rows of 64, 128 or 256 floats with RoPE: head_rope_kernel below. Other
// short rows: each workgroup is 4 wavefronts owning up to 16 rows. It issues
// all of its row loads at once (coalesced, float4 when aligned) together with
// the positions, norm weights and sin/cos rows of its first RoPE pairs, then
// stages the rows in LDS (row stride dim+1 floats, so the per-lane row walks
// are bank-conflict free); half-wave r sums row r while the RoPE inputs land; then
// every thread takes elements (or RoPE pairs) of the block in turn, so
// weights, sin/cos and outputs move coalesced. A block stages all its rows
// before writing any output, so x == out (in place) is safe.
#pragma clang fp contract(off)

#include "ikv_common.hpp"
#include "../../include/ikv.h"

#include <climits>
#include <initializer_list>
#include <vector>

namespace {

constexpr int kLdsFloats = 64 * 129;  // 33 KB: the largest short-row block staged in LDS
constexpr int kLongRow = 512;
constexpr int kRowThreads = 256;     // 4 wavefronts per short-row block
constexpr int kMaxRows = 16;         // rows per short-row block
// Staging registers per thread: every float (or float4) of the largest block.
constexpr int kStage = (kLdsFloats + kRowThreads - 1) / kRowThreads;
constexpr int kStage4 = (kLdsFloats / 4 + kRowThreads - 1) / kRowThreads;
// RoPE pairs per thread whose position, sin/cos and weights are loaded before
// the sums (all of them for head_dim 128); further pairs load afterwards.
constexpr int kPairPF = 4;

int rows_per_block(int dim) {
  int r = kLdsFloats / (dim + 1);
  if (r > kMaxRows) r = kMaxRows;
  if (r < 1) r = 1;
  return r;
}

bool long_row(int64_t dim) { return dim >= kLongRow && dim % 256 == 0; }

// Short rows (head_dim rows of qk-norm and RoPE, rows shorter than kLongRow).
// A block of 4 wavefronts owns up to kMaxRows rows. Every load the block needs
// before its sums is issued at once: the rows (float4 when `vec`), and for
// this thread's first kPairPF RoPE pairs the position, the norm weights and,
// once the position is back, the sin/cos row; those land while lanes
// 0..rows-1 of wavefront 0 run the ordered double sums. All of a block's rows
// are staged in LDS before any output is written, so x == out is safe.
template <bool NORM, bool ROPE>
__global__ __launch_bounds__(kRowThreads) void row_kernel(const float *__restrict__ x,
                                                          const float *__restrict__ w, float *out,
                                                          const int32_t *__restrict__ pos, int64_t rows,
                                                          int dim, int rpb, float eps, int n_heads,
                                                          const float *__restrict__ sin_tab,
                                                          const float *__restrict__ cos_tab,
                                                          int64_t n_ctx, int *status, int vec) {
  extern __shared__ float lds[];
  __shared__ float s_scale[kMaxRows];
  const int tid = threadIdx.x;
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * rpb;
  const int64_t left = rows - row0;
  const int nr = static_cast<int>(left < rpb ? left : rpb);
  const int stride = dim + 1;
  const int total = nr * dim;
  const int hd = dim / 2;
  const int n_pairs = ROPE ? nr * hd : 0;
  const float *xb = x + row0 * dim;

  // Stage the rows: all loads first, then the LDS stores.
  if (vec) {
    const float4 *xb4 = reinterpret_cast<const float4 *>(xb);
    const int total4 = total >> 2;
    float4 v[kStage4];
#pragma unroll
    for (int k = 0; k < kStage4; ++k) {
      const int i = tid + k * kRowThreads;
      if (i < total4) v[k] = xb4[i];
    }
#pragma unroll
    for (int k = 0; k < kStage4; ++k) {
      const int i = tid + k * kRowThreads;
      if (i < total4) {
        const int e = 4 * i;  // dim % 4 == 0: the four floats share a row
        const int r = e / dim;
        float *d = &lds[r * stride + (e - r * dim)];
        d[0] = v[k].x;
        d[1] = v[k].y;
        d[2] = v[k].z;
        d[3] = v[k].w;
      }
    }
  } else {
    float v[kStage];
#pragma unroll
    for (int k = 0; k < kStage; ++k) {
      const int i = tid + k * kRowThreads;
      if (i < total) v[k] = xb[i];
    }
#pragma unroll
    for (int k = 0; k < kStage; ++k) {
      const int i = tid + k * kRowThreads;
      if (i < total) {
        const int r = i / dim;
        lds[r * stride + (i - r * dim)] = v[k];
      }
    }
  }

  // RoPE inputs of this thread's first pairs, in flight during the sums.
  int32_t pp[kPairPF];
  float w0[kPairPF], w1[kPairPF], cs[kPairPF], sn[kPairPF];
  if constexpr (ROPE) {
#pragma unroll
    for (int k = 0; k < kPairPF; ++k) {
      const int i = tid + k * kRowThreads;
      pp[k] = -1;
      if (i < n_pairs) {
        const int r = i / hd;
        const int j = i - r * hd;
        pp[k] = pos[(row0 + r) / n_heads];
        if (NORM) {
          w0[k] = w[j];
          w1[k] = w[j + hd];
        }
      }
    }
#pragma unroll
    for (int k = 0; k < kPairPF; ++k) {
      const int i = tid + k * kRowThreads;
      cs[k] = 0.0f;
      sn[k] = 0.0f;
      if (i < n_pairs && pp[k] >= 0 && pp[k] < n_ctx) {
        const int j = i - (i / hd) * hd;
        cs[k] = cos_tab[static_cast<int64_t>(pp[k]) * hd + j];
        sn[k] = sin_tab[static_cast<int64_t>(pp[k]) * hd + j];
      }
    }
  }
  __syncthreads();

  if (NORM) {
    // Row r's sum by half-wave r % 8 (rows r and r + 8 for 16 rows): lane c
    // adds the squares of elements c, c + 32, ... in double, a xor butterfly
    // adds the lanes, and the scale is certified against the reference's
    // index-order sum; lane 0 sums in index order when it is not certain.
    // The index-order sum alone is a chain of dim dependent double adds
    // (about 1.1 us for 128).
    const int hw = tid >> 5;
    const int c = tid & 31;
    for (int r = hw; r < nr; r += kRowThreads / 32) {
      const float *rp = &lds[r * stride];
      double part = 0.0;
      for (int i = c; i < dim; i += 32) {
        const float xv = rp[i];
        const float sq = xv * xv;
        part += static_cast<double>(sq);
      }
      part = ikv::half_wave_sum_f64(part);
      float sc = 0.f;
      const bool certain =
          ikv::certified_rms_scale(part, dim, eps, (dim - 1) + (dim + 31) / 32 + 4, sc);
      if (c == 0) s_scale[r] = certain ? sc : ikv::ordered_rms_scale(rp, dim, eps);
    }
  }
  __syncthreads();

  float *ob = out + row0 * dim;
  if (!ROPE) {
    for (int i = tid; i < total; i += kRowThreads) {
      const int r = i / dim;
      const int c = i - r * dim;
      const float t = lds[r * stride + c] * s_scale[r];
      ob[i] = t * w[c];
    }
    return;
  }
  // One pair: x0 = x[j], x1 = x[j + hd] (normed first when NORM), rotated by
  // the angle of its token's position; a position outside the table gives a
  // zero pair and raises *status.
  auto rotate = [&](int i, int32_t p, float wa, float wb, float c, float s) {
    const int r = i / hd;
    const int j = i - r * hd;
    float x0 = lds[r * stride + j];
    float x1 = lds[r * stride + j + hd];
    if (NORM) {
      const float sc = s_scale[r];
      const float t0 = x0 * sc;
      const float t1 = x1 * sc;
      x0 = t0 * wa;
      x1 = t1 * wb;
    }
    float o0 = 0.0f, o1 = 0.0f;
    if (p < 0 || p >= n_ctx) {
      ikv::raise_status(status, IKV_STATUS_POSITION);
    } else {
      const float a = x0 * c;
      const float b = x1 * s;
      const float e = x0 * s;
      const float f = x1 * c;
      o0 = a - b;
      o1 = e + f;
    }
    ob[static_cast<int64_t>(r) * dim + j] = o0;
    ob[static_cast<int64_t>(r) * dim + j + hd] = o1;
  };
#pragma unroll
  for (int k = 0; k < kPairPF; ++k) {
    const int i = tid + k * kRowThreads;
    if (i < n_pairs) rotate(i, pp[k], NORM ? w0[k] : 0.0f, NORM ? w1[k] : 0.0f, cs[k], sn[k]);
  }
  for (int i = tid + kPairPF * kRowThreads; i < n_pairs; i += kRowThreads) {
    const int r = i / hd;
    const int j = i - r * hd;
    const int32_t p = pos[(row0 + r) / n_heads];
    const bool ok = p >= 0 && p < n_ctx;
    const float c = ok ? cos_tab[static_cast<int64_t>(p) * hd + j] : 0.0f;
    const float s = ok ? sin_tab[static_cast<int64_t>(p) * hd + j] : 0.0f;
    rotate(i, p, NORM ? w[j] : 0.0f, NORM ? w[j + hd] : 0.0f, c, s);
  }
}

// Model-width rows: one wavefront per row, lane-strided double sum (the
// order described above), float4 loads and stores. Bound by memory with many
// rows and by the latency of one row's loads with few, so rows of up to
// 256 * NV floats are loaded once, all loads in flight together, and stay in
// registers (NV = 0: longer rows, read twice). Graphs of 20 launches: 4096 rows
// of 4096 floats 292 us (mostly one wave's index-order sum) -> 22.5 (5.9 TB/s),
// 1024 rows 9.7 -> 7.3, one row 5.0 -> 3.5; 2048 rows of 1024 4.5 -> 4.2. Five
// sizes of NV, since the pieces past a row cost: 2048 rows of 1280 5.85 us with
// 16 of them, 4.44 with 6 (4.7 read twice); 4096 of 2560 15.7 and, with 12, 13.8.
template <int NV>
__global__ __launch_bounds__(256) void long_row_norm_kernel(const float *__restrict__ x,
                                                            const float *__restrict__ w, float *out,
                                                            int64_t rows, int dim, float eps) {
  const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  const int nj = dim / 256;
  const float4 *xr = reinterpret_cast<const float4 *>(x + row * dim);
  const float4 *w4 = reinterpret_cast<const float4 *>(w);
  float4 *o4 = reinterpret_cast<float4 *>(out + row * dim);
  auto scaled = [](float4 v, float4 g, float s) {
    const float a = v.x * s, b = v.y * s, c = v.z * s, d = v.w * s;
    return make_float4(a * g.x, b * g.y, c * g.z, d * g.w);
  };
  if constexpr (NV > 0) {
    // pieces past the row load its last one and count as zeros, so that no
    // branch stands between the loads
    float4 v[NV], g[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] = xr[64 * min(j, nj - 1) + lane];
#pragma unroll
    for (int j = 0; j < NV; ++j) g[j] = w4[64 * min(j, nj - 1) + lane];
    double s[4] = {0.0, 0.0, 0.0, 0.0};  // four chains of adds instead of one
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const float a = v[j].x * v[j].x, b = v[j].y * v[j].y, c = v[j].z * v[j].z, d = v[j].w * v[j].w;
      const bool on = j < nj;
      s[0] += on ? static_cast<double>(a) : 0.0;
      s[1] += on ? static_cast<double>(b) : 0.0;
      s[2] += on ? static_cast<double>(c) : 0.0;
      s[3] += on ? static_cast<double>(d) : 0.0;
    }
    const float scale = ikv::rms_scale_of_lane_sums((s[0] + s[1]) + (s[2] + s[3]),
                                                    reinterpret_cast<const float *>(xr), dim, eps, lane);
#pragma unroll
    for (int j = 0; j < NV; ++j)
      if (j < nj) o4[64 * j + lane] = scaled(v[j], g[j], scale);
  } else {
    const float scale = ikv::rms_scale_strided(xr, dim, eps, lane);
    for (int j = lane; j < dim / 4; j += 64) o4[j] = scaled(xr[j], w4[j], scale);
  }
}

// Head rows of 64, 128 or 256 floats with RoPE (and qk-norm): LPR = dim / 4
// lanes per row, lane c holding the pairs (2c, 2c + 1) of both halves, so a
// row's rotation is lane-local and nothing goes through LDS or a barrier. A
// wave owns R sets of 64 / LPR rows, all their loads in flight together.
// Bound by memory with many rows (4096 tokens x 32 heads of 128: 134 MB) and
// by the chain position -> angles -> rotation with few. With R = 4 the four
// sums of a lane's rows are certified by the four lanes of a quad at once
// (the double square root and divisions of every row in every lane cost as
// much as the memory). Measured against row_kernel in graphs of 20 launches:
// 4096 tokens x 32 heads of 128 50.1 -> 23.3 us (5.8 TB/s), 2048 x 16 17.1 ->
// 7.9, 37 x 16 5.9 -> 2.5, one token 5.5 -> 2.2; 1500 x 12 of 64 8.0 -> 3.7.
template <int LPR, int R, bool NORM>
__global__ __launch_bounds__(256) void head_rope_kernel(
    const float *__restrict__ x, const float *__restrict__ w, float *out,
    const int32_t *__restrict__ pos, unsigned rows, float eps, unsigned n_heads,
    const float *__restrict__ sin_tab, const float *__restrict__ cos_tab, int64_t n_ctx,
    int *status) {
  constexpr int DIM = 4 * LPR, HD = 2 * LPR;
  constexpr unsigned SETS = 64 / LPR;  // rows per set
  const int lane = threadIdx.x & 63;
  const int c = lane % LPR;
  const unsigned row0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * (SETS * R) + lane / LPR;
  float2 lo[R], hi[R], cs[R], sn[R];
  int32_t p[R];
  unsigned row[R];
#pragma unroll
  for (int r = 0; r < R; ++r) row[r] = min(row0 + SETS * r, rows - 1);  // past the end: not stored
#pragma unroll
  for (int r = 0; r < R; ++r) p[r] = pos[row[r] / n_heads];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float2 *xr = reinterpret_cast<const float2 *>(x + static_cast<size_t>(row[r]) * DIM);
    lo[r] = xr[c];
    hi[r] = xr[LPR + c];
  }
  float2 wl = make_float2(0.f, 0.f), wh = wl;
  if constexpr (NORM) {
    wl = reinterpret_cast<const float2 *>(w)[c];
    wh = reinterpret_cast<const float2 *>(w)[LPR + c];
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const bool in = p[r] >= 0 && p[r] < n_ctx;
    const size_t at = static_cast<size_t>(in ? p[r] : 0) * HD;
    cs[r] = reinterpret_cast<const float2 *>(cos_tab + at)[c];
    sn[r] = reinterpret_cast<const float2 *>(sin_tab + at)[c];
  }
  if constexpr (NORM) {
    double sum[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const double s = ikv::add_squares(0.0, make_float4(lo[r].x, lo[r].y, hi[r].x, hi[r].y));
      sum[r] = LPR == 16   ? ikv::row16_sum_f64(s)
               : LPR == 32 ? ikv::half_wave_sum_f64(s)
                           : ikv::wave_sum_f64(s);
    }
    // lane of quad position k certifies row set k (R == 1: every lane its own)
    double mine = sum[0];
    if constexpr (R == 4) {
      const int k = lane & 3;
      mine = k == 0 ? sum[0] : k == 1 ? sum[1] : k == 2 ? sum[2] : sum[3];
    }
    float scale = -1.f;  // (a certified scale is positive)
    if (!ikv::certified_rms_scale(mine, DIM, eps, (DIM - 1) + 4 + 6, scale)) scale = -1.f;
    float sc[R];
    if constexpr (R == 4) {
      sc[0] = ikv::dpp<0x00>(scale);  // quad_perm [k, k, k, k]
      sc[1] = ikv::dpp<0x55>(scale);
      sc[2] = ikv::dpp<0xAA>(scale);
      sc[3] = ikv::dpp<0xFF>(scale);
    } else {
      sc[0] = scale;
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      // rows in doubt: the wave sums each in index order
      for (unsigned long long todo = __builtin_amdgcn_ballot_w64(sc[r] < 0.f); todo != 0;) {
        const int src = __builtin_ctzll(todo);
        const unsigned rr = __builtin_amdgcn_readlane(row[r], src);
        const float s = ikv::ordered_rms_scale_wave(x + static_cast<size_t>(rr) * DIM, DIM, eps, lane);
        if (lane / LPR == src / LPR) sc[r] = s;
        todo &= ~((LPR == 64 ? ~0ull : (1ull << (LPR % 64)) - 1) << (src / LPR * LPR));
      }
      const float a = lo[r].x * sc[r], b = lo[r].y * sc[r], d = hi[r].x * sc[r], e = hi[r].y * sc[r];
      lo[r] = make_float2(a * wl.x, b * wl.y);
      hi[r] = make_float2(d * wh.x, e * wh.y);
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (row0 + SETS * r >= rows) continue;
    float2 o0 = make_float2(0.f, 0.f), o1 = o0;
    if (p[r] < 0 || p[r] >= n_ctx) {
      ikv::raise_status(status, IKV_STATUS_POSITION);
    } else {
      const float a0 = lo[r].x * cs[r].x, b0 = hi[r].x * sn[r].x;
      const float a1 = lo[r].y * cs[r].y, b1 = hi[r].y * sn[r].y;
      const float e0 = lo[r].x * sn[r].x, f0 = hi[r].x * cs[r].x;
      const float e1 = lo[r].y * sn[r].y, f1 = hi[r].y * cs[r].y;
      o0 = make_float2(a0 - b0, a1 - b1);
      o1 = make_float2(e0 + f0, e1 + f1);
    }
    float2 *orow = reinterpret_cast<float2 *>(out + static_cast<size_t>(row[r]) * DIM);
    orow[c] = o0;
    orow[LPR + c] = o1;
  }
}

bool aligned8(std::initializer_list<const void *> ptrs) {
  for (const void *q : ptrs)
    if (reinterpret_cast<uintptr_t>(q) & 7) return false;
  return true;
}

// R = 4 row sets per wave once that still gives every SIMD two waves.
constexpr int64_t kManyRows = 8 * 2048;

template <bool NORM>
int launch_heads(const float *x, const float *w, float *out, const int32_t *pos, int64_t rows,
                 int dim, float eps, int n_heads, const float *sin_tab, const float *cos_tab,
                 int64_t n_ctx, int *status, void *stream) {
  const int sets = 256 / dim;  // rows of one set of a wave
  const int r = rows * dim >= kManyRows * 128 ? 4 : 1;
  const unsigned per_block = 4u * static_cast<unsigned>(sets * r);
  const unsigned blocks = (static_cast<unsigned>(rows) + per_block - 1) / per_block;
  hipStream_t s = static_cast<hipStream_t>(stream);
#define IKV_HEADS(LPR, RR)                                                                       \
  head_rope_kernel<LPR, RR, NORM><<<blocks, 256, 0, s>>>(x, w, out, pos,                         \
                                                         static_cast<unsigned>(rows), eps,       \
                                                         static_cast<unsigned>(n_heads), sin_tab, \
                                                         cos_tab, n_ctx, status)
  if (dim == 64) {
    if (r == 4) IKV_HEADS(16, 4); else IKV_HEADS(16, 1);
  } else if (dim == 128) {
    if (r == 4) IKV_HEADS(32, 4); else IKV_HEADS(32, 1);
  } else {
    if (r == 4) IKV_HEADS(64, 4); else IKV_HEADS(64, 1);
  }
#undef IKV_HEADS
  return ikv::launch_status();
}

template <bool NORM, bool ROPE>
int launch_rows(const float *x, const float *w, float *out, const int32_t *pos, int64_t rows,
                int dim, float eps, int n_heads, const float *sin_tab, const float *cos_tab,
                int64_t n_ctx, int *status, void *stream) {
  if constexpr (ROPE) {
    if ((dim == 64 || dim == 128 || dim == 256) && rows <= INT_MAX &&
        aligned8({x, w, out, sin_tab, cos_tab}))
      return launch_heads<NORM>(x, w, out, pos, rows, dim, eps, n_heads, sin_tab, cos_tab, n_ctx,
                                status, stream);
  }
  const int rpb = rows_per_block(dim);
  const int64_t blocks = (rows + rpb - 1) / rpb;
  if (blocks > INT_MAX) return -EOVERFLOW;
  const size_t shmem = sizeof(float) * static_cast<size_t>(rpb) * (dim + 1);
  // float4 staging needs 16-byte rows: dim % 4 == 0 and x 16-byte aligned.
  const int vec = (dim % 4 == 0 && ikv::aligned16(x)) ? 1 : 0;
  row_kernel<NORM, ROPE><<<static_cast<unsigned>(blocks), kRowThreads, shmem,
                           static_cast<hipStream_t>(stream)>>>(
      x, w, out, pos, rows, dim, rpb, eps, n_heads, sin_tab, cos_tab, n_ctx, status, vec);
  return ikv::launch_status();
}

}  // namespace

extern "C" int ikv_rms_norm_f32(const float *x, const float *w, float *out, int64_t rows,
                                int64_t dim, float eps, void *stream) {
  if (rows == 0) return 0;
  if (!x || !w || !out || rows < 0 || dim <= 0) return -EINVAL;
  if (rows > INT64_MAX / dim) return -EOVERFLOW;
  if (long_row(dim) && dim <= INT_MAX && ikv::aligned16(x) && ikv::aligned16(w) &&
      ikv::aligned16(out)) {
    const int64_t blocks = (rows + 3) / 4;
    if (blocks > INT_MAX) return -EOVERFLOW;
    const auto kernel = dim <= 1024   ? long_row_norm_kernel<4>
                        : dim <= 1536 ? long_row_norm_kernel<6>
                        : dim <= 2048 ? long_row_norm_kernel<8>
                        : dim <= 3072 ? long_row_norm_kernel<12>
                        : dim <= 4096 ? long_row_norm_kernel<16>
                                      : long_row_norm_kernel<0>;
    kernel<<<static_cast<unsigned>(blocks), 256, 0, static_cast<hipStream_t>(stream)>>>(
        x, w, out, rows, static_cast<int>(dim), eps);
    return ikv::launch_status();
  }
  if (dim > kLdsFloats - 1) return -ENOTSUP;
  return launch_rows<true, false>(x, w, out, nullptr, rows, static_cast<int>(dim), eps, 1, nullptr,
                                  nullptr, 0, nullptr, stream);
}

extern "C" int ikv_rope_theta_table_f32(float theta_base, int head_dim, int64_t n_ctx,
                                        float *theta_host) {
  if (head_dim <= 0 || (head_dim & 1) || n_ctx < 0) return -EINVAL;
  if (n_ctx == 0) return 0;
  if (!theta_host) return -EINVAL;
  const int half = head_dim / 2;
  // the exponent 2i/d and the reciprocal power are float operations (the
  // reference's float arguments to std::pow select powf); the angle is the
  // position times the widened frequency, rounded once to float
  std::vector<double> freq(static_cast<size_t>(half));
  for (int i = 0; i < half; ++i) {
    const float e = (2.0f * static_cast<float>(i)) / static_cast<float>(head_dim);
    freq[static_cast<size_t>(i)] = static_cast<double>(1.0f / powf(theta_base, e));
  }
  for (int64_t pos = 0; pos < n_ctx; ++pos) {
    float *row = theta_host + pos * half;
    for (int i = 0; i < half; ++i)
      row[i] = static_cast<float>(static_cast<double>(pos) * freq[static_cast<size_t>(i)]);
  }
  return 0;
}

extern "C" int ikv_rope_sincos_table_f32(const float *theta_host, size_t count, float *sin_host,
                                         float *cos_host) {
  if (count == 0) return 0;
  if (!theta_host || !sin_host || !cos_host) return -EINVAL;
  for (size_t i = 0; i < count; ++i) {
    sin_host[i] = sinf(theta_host[i]);
    cos_host[i] = cosf(theta_host[i]);
  }
  return 0;
}

static int check_rope_args(const float *x, float *out, const int32_t *pos, int64_t n_tokens,
                           int n_heads, int head_dim, const float *sin_tab, const float *cos_tab,
                           int64_t n_ctx) {
  if (!x || !out || !pos || !sin_tab || !cos_tab) return -EINVAL;
  if (n_tokens < 0 || n_heads <= 0 || head_dim <= 0 || (head_dim & 1) || n_ctx <= 0) return -EINVAL;
  if (head_dim > kLdsFloats - 1) return -ENOTSUP;
  if (n_tokens > INT64_MAX / n_heads / head_dim) return -EOVERFLOW;
  return 0;
}

extern "C" int ikv_rope_neox_f32(const float *x, float *out, const int32_t *pos, int64_t n_tokens,
                                 int n_heads, int head_dim, const float *sin_tab,
                                 const float *cos_tab, int64_t n_ctx, int *status, void *stream) {
  if (n_tokens == 0) return 0;
  const int rc = check_rope_args(x, out, pos, n_tokens, n_heads, head_dim, sin_tab, cos_tab, n_ctx);
  if (rc) return rc;
  return launch_rows<false, true>(x, nullptr, out, pos, n_tokens * n_heads, head_dim, 0.0f,
                                  n_heads, sin_tab, cos_tab, n_ctx, status, stream);
}

extern "C" int ikv_qk_norm_rope_f32(const float *x, const float *w, float *out, const int32_t *pos,
                                    int64_t n_tokens, int n_heads, int head_dim, float eps,
                                    const float *sin_tab, const float *cos_tab, int64_t n_ctx,
                                    int *status, void *stream) {
  if (n_tokens == 0) return 0;
  if (!w) return -EINVAL;
  const int rc = check_rope_args(x, out, pos, n_tokens, n_heads, head_dim, sin_tab, cos_tab, n_ctx);
  if (rc) return rc;
  return launch_rows<true, true>(x, w, out, pos, n_tokens * n_heads, head_dim, eps, n_heads,
                                 sin_tab, cos_tab, n_ctx, status, stream);
}
