// Masked softmax cross-entropy and argmax accuracy over the logit rows of a
// partition, fp32, in one pass over the logits, which also writes the train
// rows' loss gradient before its scalar scale; gr_xent_backward scales it and
// fills in the other rows' zeros.
//
// Row r carries a mask byte: bit 0 = train (contributes to the loss),
// bit 1 = val, bit 2 = test (contribute to the accuracy counts).  For a row,
//   m = max_c x_c,  lse = m + log(sum_c exp(x_c - m)),  nll = lse - x_y,
//   pred = the first c with x_c == m,
// the arithmetic of torch's log_softmax + NLL and argmax.  Sums and counts
// are reduced in a fixed order (per-workgroup partials in double, then a
// fixed tree), so results do not depend on scheduling.  Labels of train /
// val / test rows outside [0, C) are counted and reported, not read.
// Gradient rows: g[r, c] = exp(x_c - m) / sum - [c == y] on train rows (0 if
// the label is out of range), i.e. d(sum of train nll)/dx, the backward of
// log_softmax + NLL; other rows are 0, or, where the train rows' bits are kept
// for xent_backward to tell them apart, not written.
//
// 1M rows of 47 classes, 60% train: forward 136 us (and 8 for the statistics'
// last sum), backward 62 and four small launches when every row's gradient was
// written, with a second exponential per element, and scaled by torch; now 92
// (and 8) and 58 us, the backward in one launch.
#include <algorithm>

#include "gr_internal.h"
#include "wave.h"

namespace gr_loss {

constexpr int kStats = 7;  // nll_sum, train_n, val_ok, val_n, test_ok, test_n, bad_labels

using gr_wave::group_max;
using gr_wave::group_min_int;
using gr_wave::group_sum;

// Accumulates one row's contribution to the seven statistics.
__device__ __forceinline__ void add_row_stats(double (&acc)[kStats], uint8_t mk, bool ok_label,
                                              float lse, float xy, bool hit) {
  if (mk != 0 && !ok_label) {
    acc[6] += 1.0;
    return;
  }
  if (mk & 1) {
    acc[0] += (double)(lse - xy);
    acc[1] += 1.0;
  }
  if (mk & 2) {
    acc[2] += hit ? 1.0 : 0.0;
    acc[3] += 1.0;
  }
  if (mk & 4) {
    acc[4] += hit ? 1.0 : 0.0;
    acc[5] += 1.0;
  }
}

// Ordered sum of the workgroup's 256 per-thread statistics into part[blockIdx]:
// a butterfly inside each wavefront, then the 4 wavefront sums in order.
__device__ __forceinline__ void block_stats(double (&acc)[kStats], double* __restrict__ part) {
  __shared__ double red[4][kStats];
#pragma unroll
  for (int k = 0; k < kStats; ++k) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) acc[k] += __shfl_xor(acc[k], off, 64);
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int k = 0; k < kStats; ++k) red[wave][k] = acc[k];
  }
  __syncthreads();
  if (threadIdx.x < kStats) {
    const int k = threadIdx.x;
    part[(int64_t)blockIdx.x * kStats + k] = ((red[0][k] + red[1][k]) + red[2][k]) + red[3][k];
  }
}

constexpr int kRowsPerBlock = 256;
constexpr int kSmallC = 64;

// Row and column of element e of a block of C-wide rows, C <= 64, e < 2^14: the
// product with ceil(2^20 / C) is exact over that range.
struct RowOf {
  uint32_t inv;
  int C;
  __device__ __forceinline__ explicit RowOf(int c) : inv(((1u << 20) + c - 1) / c), C(c) {}
  __device__ __forceinline__ uint32_t operator()(uint32_t e) const {
    return (uint32_t)(((uint64_t)e * inv) >> 20);
  }
};

// Four floats at any 4-byte boundary, moved as one 16-byte access.
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));

// Which of the workgroup's rows are train rows, one bit each, for
// xent_backward: the caller may change its mask bytes in between.
__device__ __forceinline__ void keep_train_bits(const uint8_t* __restrict__ mask, int64_t row0,
                                                int64_t rows, uint64_t* __restrict__ bits) {
  if (bits == nullptr) return;
  const int64_t r = row0 + (threadIdx.x & 63);
  const uint64_t b = __ballot(r < rows && (mask[r < rows ? r : rows - 1] & 1));
  if ((threadIdx.x & 63) == 0) bits[row0 / 64] = b;
}

// C <= G * R * V <= 64: G lanes a row, R pieces of V neighbouring columns a
// lane (piece l, l + G, ...), 64 / G rows a wavefront and step, U steps' loads
// in flight; 64 rows a wavefront, 256 a workgroup.  Pieces of 4 columns (C >= 4)
// are 16-byte accesses at any boundary; one that would end past the row starts
// at its last 4 columns instead, and the columns it shares with the piece
// before are left out of the sum.  Everything stays in registers: occupancy
// hides the loads, and few lanes with many columns each leave little of the
// cross-lane and per-row work to a column.  1M rows of 47 classes, 60% train: a
// row a thread with the rows staged in LDS (48 KB, three workgroups a CU)
// 123 us, 16 lanes of 3 single columns 102 us, 4 lanes of 3 pieces 93 us.
//
// U is 4 while that keeps at most 48 loaded columns a lane, else 2.  Repeated
// forward calls on 1M rows, 60% train, with 1, 2 and 4 steps (us): 10 columns
// 31.0 / 30.6 / 30.4, 20 columns 39.8 / 39.5 / 38.9, 47 columns 78.9 / 74.5 / 72.8,
// 60 columns 111.7 / 107.5 / 104.7, 64 columns 90.9 / 90.7 / 92.7.
template <int G, int R, int V>
__global__ __launch_bounds__(256) void xent_rows_narrow(const float* __restrict__ x, int64_t ld,
                                                        int64_t rows, int C,
                                                        const int64_t* __restrict__ labels,
                                                        const uint8_t* __restrict__ mask,
                                                        float* __restrict__ lse_out,
                                                        float* __restrict__ grad, int64_t ldg,
                                                        double* __restrict__ part,
                                                        uint64_t* __restrict__ bits) {
  constexpr int RPW = 64 / G, U = R * V * 4 <= 48 ? 4 : 2;
  static_assert(G % U == 0, "64 rows in steps of U * RPW");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l = lane % G, sub = lane / G;
  const int64_t row0 = (int64_t)blockIdx.x * kRowsPerBlock + wave * 64;
  double nll = 0.0;
  int count[6] = {0, 0, 0, 0, 0, 0};
  int start[R];  // first column of piece k
#pragma unroll
  for (int k = 0; k < R; ++k) start[k] = max(0, min((l + k * G) * V, C - V));
  // Column start[k] + i belongs to piece k (only the last one can reach back).
  auto own = [&](int k, int i) {
    return k + 1 < R || start[k] + i >= (l + k * G) * V;
  };
  for (int it = 0; it < G; it += U) {
    if (row0 + it * RPW >= rows) break;  // the same for the whole wavefront
    float v[U][R][V];
    uint8_t mk[U];
    int64_t y[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t r = row0 + (it + u) * RPW + sub;
      const int64_t rr = r < rows ? r : rows - 1;
      mk[u] = mask[rr];
      y[u] = labels[rr];
      const float* row = x + rr * ld;
#pragma unroll
      for (int k = 0; k < R; ++k) {
        if constexpr (V == 4) {
          const float4u q = *reinterpret_cast<const float4u*>(row + start[k]);
#pragma unroll
          for (int i = 0; i < V; ++i) v[u][k][i] = q[i];
        } else {
          v[u][k][0] = row[start[k]];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t r = row0 + (it + u) * RPW + sub;
      const bool in = r < rows;
      const bool ok = in && y[u] >= 0 && y[u] < C;
      const int yc = ok ? (int)y[u] : -1;
      float m = -INFINITY;
#pragma unroll
      for (int k = 0; k < R; ++k)
#pragma unroll
        for (int i = 0; i < V; ++i) m = fmaxf(m, v[u][k][i]);
      m = group_max<G>(m);
      // The first column holding the maximum; a NaN in column 0 counts as one.
      int first = C;
      float sum = 0.f, xy = 0.f;
      const bool nan0 = l == 0 && v[u][0][0] != v[u][0][0];
#pragma unroll
      for (int k = R - 1; k >= 0; --k)
#pragma unroll
        for (int i = V - 1; i >= 0; --i) {
          const float e = v[u][k][i];
          first = e == m ? start[k] + i : first;
          xy = start[k] + i == yc ? e : xy;
          v[u][k][i] = expf(e - m);
          sum += own(k, i) ? v[u][k][i] : 0.f;
        }
      if (nan0) first = 0;
      sum = group_sum<G>(sum);
      first = group_min_int<G>(first);
      const float lse = m + logf(sum);
      const bool lead = l == 0 && in;
      if (lse_out != nullptr && lead) lse_out[r] = lse;
      const bool hit = first == yc;
      // The label's column lies in one piece, held by lane (yc / V) % G.
      if (ok && (mk[u] & 1) && (yc / V) % G == l) nll += (double)(lse - xy);
      count[0] += __popcll(__ballot(lead && ok && (mk[u] & 1)));
      count[1] += __popcll(__ballot(lead && ok && (mk[u] & 2) && hit));
      count[2] += __popcll(__ballot(lead && ok && (mk[u] & 2)));
      count[3] += __popcll(__ballot(lead && ok && (mk[u] & 4) && hit));
      count[4] += __popcll(__ballot(lead && ok && (mk[u] & 4)));
      count[5] += __popcll(__ballot(lead && mk[u] != 0 && !ok));
      const bool train = mk[u] & 1;
      if (grad != nullptr && in && (train || bits == nullptr)) {
        const float inv = 1.f / sum;
        float* g = grad + r * ldg;
#pragma unroll
        for (int k = 0; k < R; ++k) {
          float q[V];
#pragma unroll
          for (int i = 0; i < V; ++i)
            q[i] = ok && train ? v[u][k][i] * inv - (start[k] + i == yc ? 1.f : 0.f) : 0.f;
          if (k + 1 == R && (l + k * G) * V >= C) continue;  // nothing of its own
          if constexpr (V == 4) {
            *reinterpret_cast<float4u*>(g + start[k]) = float4u{q[0], q[1], q[2], q[3]};
          } else {
            g[start[k]] = q[0];
          }
        }
      }
    }
  }
  __shared__ double red[4][kStats];
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) nll += __shfl_xor(nll, off, 64);
  if (lane == 0) {
    red[wave][0] = nll;
#pragma unroll
    for (int k = 0; k < 6; ++k) red[wave][1 + k] = count[k];
  }
  if (row0 < rows) keep_train_bits(mask, row0, rows, bits);
  __syncthreads();
  if (threadIdx.x < kStats) {
    const int k = threadIdx.x;
    part[(int64_t)blockIdx.x * kStats + k] = ((red[0][k] + red[1][k]) + red[2][k]) + red[3][k];
  }
}

// C > 64: one wavefront per row (lanes over columns), 64 rows per wavefront
// of a 256-row workgroup.
__global__ __launch_bounds__(256) void xent_rows_wide(const float* __restrict__ x, int64_t ld,
                                                      int64_t rows, int C,
                                                      const int64_t* __restrict__ labels,
                                                      const uint8_t* __restrict__ mask,
                                                      float* __restrict__ lse_out,
                                                      float* __restrict__ grad, int64_t ldg,
                                                      double* __restrict__ part,
                                                      uint64_t* __restrict__ bits) {
  const int lane = threadIdx.x & 63;
  const int64_t row0 = (int64_t)blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6) * 64;
  double acc[kStats];
#pragma unroll
  for (int k = 0; k < kStats; ++k) acc[k] = 0.0;
  for (int64_t r = row0; r < row0 + 64 && r < rows; ++r) {
    const float* row = x + r * ld;
    float m = -INFINITY;
    for (int c = lane; c < C; c += 64) m = fmaxf(m, row[c]);
    m = group_max<64>(m);
    float s = 0.f;
    int first = C;
    for (int c = lane; c < C; c += 64) {
      const float v = row[c];
      s += expf(v - m);
      if (v == m && c < first) first = c;
    }
    s = group_sum<64>(s);
    first = group_min_int<64>(first);
    const float lse = m + logf(s);
    const uint8_t mk = mask[r];
    const int64_t y = labels[r];
    const bool ok_label = y >= 0 && y < C;
    const bool train = mk & 1;
    if (grad != nullptr && (train || bits == nullptr)) {
      float* g = grad + r * ldg;
      for (int c = lane; c < C; c += 64)
        g[c] = ok_label && train ? expf(row[c] - lse) - (c == (int)y ? 1.f : 0.f) : 0.f;
    }
    if (lane == 0) {
      if (lse_out != nullptr) lse_out[r] = lse;
      add_row_stats(acc, mk, ok_label, lse, ok_label ? row[y] : 0.f, first == (int)y);
    }
  }
  if (row0 < rows) keep_train_bits(mask, row0, rows, bits);
  block_stats(acc, part);
}

// out = grad * scale on train rows, 0 on the others (whose grad is not read),
// scale = *gloss / max(train rows, 1) when the loss is a mean (n_train not
// NULL).  SMALL: C <= 64, rows by a multiplication.  A workgroup takes 256 rows;
// both matrices are dense, so a block starts on a 16-byte boundary and a thread
// takes 16-byte pieces, each in one or (at a row's end) several rows: bound by
// memory, 301 MB in 58 us at 1M rows of 47 classes, 60% train.
template <bool SMALL>
__global__ __launch_bounds__(256) void xent_backward(const float* __restrict__ grad,
                                                     int64_t rows, int C,
                                                     const uint64_t* __restrict__ bits,
                                                     const float* __restrict__ gloss,
                                                     const int64_t* __restrict__ n_train,
                                                     float* __restrict__ out) {
  const int64_t row0 = (int64_t)blockIdx.x * kRowsPerBlock;
  const int nr = (int)min<int64_t>(kRowsPerBlock, rows - row0);
  float sc = *gloss;
  if (n_train != nullptr) sc /= (float)max<int64_t>(*n_train, 1);
  const int t = threadIdx.x;
  __shared__ uint8_t train[kRowsPerBlock];
  train[t] = t < nr && ((bits[(row0 + t) / 64] >> (t & 63)) & 1);
  __syncthreads();
  const int64_t base = row0 * C;
  const int64_t n = (int64_t)nr * C;
  const bool vec = ((reinterpret_cast<uintptr_t>(grad) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
  const int64_t n4 = vec ? n / 4 : 0;
  const float4* g4 = reinterpret_cast<const float4*>(grad + base);
  float4* o4 = reinterpret_cast<float4*>(out + base);
  const RowOf row_of(SMALL ? C : 1);
  auto row_at = [&](uint32_t e) {
    if constexpr (SMALL) {
      return row_of(e);
    } else {
      return e / (uint32_t)C;
    }
  };
#pragma unroll 4
  for (int64_t i = t; i < n4; i += 256) {
    // Rows of the piece's first and last element: 256 rows of up to 2^24
    // columns are indexed in 32 bits.
    const uint32_t e = (uint32_t)(4 * i);
    const uint32_t r0 = row_at(e), r1 = row_at(e + 1), r2 = row_at(e + 2), r3 = row_at(e + 3);
    const bool t0 = train[r0], t1 = train[r1], t2 = train[r2], t3 = train[r3];
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (t0 | t1 | t2 | t3) {
      const float4 g = g4[i];
      v.x = t0 ? g.x * sc : 0.f;
      v.y = t1 ? g.y * sc : 0.f;
      v.z = t2 ? g.z * sc : 0.f;
      v.w = t3 ? g.w * sc : 0.f;
    }
    o4[i] = v;
  }
  for (int64_t i = 4 * n4 + t; i < n; i += 256) {
    const int64_t r = i / C;
    out[base + i] = train[r] ? grad[base + i] * sc : 0.f;
  }
}

// Sums the per-workgroup partials: thread t adds workgroups t, t+256, ... in
// order, then a fixed tree over the 256 threads; writes the loss (sum, or
// mean over train rows when `mean`) and the integer statistics.
__global__ __launch_bounds__(256) void xent_finish(const double* __restrict__ part, int64_t nblk,
                                                   int mean, float* __restrict__ loss,
                                                   int64_t* __restrict__ stats) {
  double acc[kStats];
#pragma unroll
  for (int k = 0; k < kStats; ++k) acc[k] = 0.0;
  for (int64_t b = threadIdx.x; b < nblk; b += 256) {
#pragma unroll
    for (int k = 0; k < kStats; ++k) acc[k] += part[b * kStats + k];
  }
  __shared__ double red[kStats][256];
#pragma unroll
  for (int k = 0; k < kStats; ++k) red[k][threadIdx.x] = acc[k];
  __syncthreads();
  for (int w = 128; w >= 1; w >>= 1) {
    if ((int)threadIdx.x < w) {
#pragma unroll
      for (int k = 0; k < kStats; ++k) red[k][threadIdx.x] += red[k][threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double n_train = red[1][0];
    *loss = (float)((mean && n_train > 0.0) ? red[0][0] / n_train : red[0][0]);
  } else if (threadIdx.x < kStats) {
    stats[threadIdx.x - 1] = (int64_t)red[threadIdx.x][0];
  }
}

}  // namespace gr_loss

namespace gr_loss {

// bits: NULL, or where the train rows' bits go; the gradient's other rows are
// then left to gr_xent_backward.
static int forward(const float* logits, int64_t ld, int64_t rows, int64_t classes,
                   const int64_t* labels, const uint8_t* mask, int32_t mean, float* lse,
                   float* grad, int64_t ldg, uint64_t* bits, float* loss, int64_t* stats,
                   double* workspace, int64_t workspace_doubles, void* stream) {
  GR_REQUIRE(rows >= 0 && classes >= 1 && classes <= (1 << 24) && ld >= classes,
             "xent_forward: bad shape (%lld rows, %lld classes, ld %lld)", (long long)rows,
             (long long)classes, (long long)ld);
  GR_REQUIRE(loss && stats && workspace, "xent_forward: NULL output");
  GR_REQUIRE(rows == 0 || (logits && labels && mask), "xent_forward: NULL input");
  GR_REQUIRE(grad == nullptr || ldg >= classes, "xent_forward: ldg < classes");
  const int64_t nblk = std::max<int64_t>(1, (rows + kRowsPerBlock - 1) / kRowsPerBlock);
  GR_REQUIRE(nblk <= INT32_MAX, "xent_forward: too many rows");
  GR_REQUIRE(workspace_doubles >= nblk * kStats, "xent_forward: workspace of %lld doubles, "
             "%lld needed", (long long)workspace_doubles, (long long)(nblk * kStats));
  hipStream_t s = gr::as_stream(stream);
  const int c = (int)classes;
  // With rows == 0 the single workgroup writes zero partials.
#define GR_XENT(G, R, V)                                                                 \
  hipLaunchKernelGGL((xent_rows_narrow<G, R, V>), dim3((unsigned)nblk), dim3(256), 0, s,   \
                     logits, ld, rows, c, labels, mask, lse, grad, ldg, workspace, bits)
  if (c < 4) GR_XENT(4, 1, 1);
  else if (c <= 16) GR_XENT(4, 1, 4);
  else if (c <= 32) GR_XENT(4, 2, 4);
  else if (c <= 48) GR_XENT(4, 3, 4);
  else if (c <= kSmallC) GR_XENT(4, 4, 4);
  else
    hipLaunchKernelGGL(xent_rows_wide, dim3((unsigned)nblk), dim3(256), 0, s, logits, ld, rows, c,
                       labels, mask, lse, grad, ldg, workspace, bits);
#undef GR_XENT
  GR_HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(xent_finish, dim3(1), dim3(256), 0, s, workspace, nblk, (int)mean, loss,
                     stats);
  GR_HIP_CHECK(hipGetLastError());
  return GR_OK;
}

}  // namespace gr_loss

extern "C" int gr_xent_forward(const float* logits, int64_t ld, int64_t rows, int64_t classes,
                               const int64_t* labels, const uint8_t* mask, int32_t mean,
                               float* lse, float* grad, int64_t ldg, float* loss,
                               int64_t* stats, double* workspace, int64_t workspace_doubles,
                               void* stream) {
  gr::clear_error();
  return gr_loss::forward(logits, ld, rows, classes, labels, mask, mean, lse, grad, ldg, nullptr,
                          loss, stats, workspace, workspace_doubles, stream);
}

extern "C" int gr_xent_forward_train(const float* logits, int64_t ld, int64_t rows,
                                     int64_t classes, const int64_t* labels, const uint8_t* mask,
                                     int32_t mean, float* grad, int64_t ldg, uint64_t* train,
                                     float* loss, int64_t* stats, double* workspace,
                                     int64_t workspace_doubles, void* stream) {
  gr::clear_error();
  GR_REQUIRE(rows == 0 || (grad != nullptr && train != nullptr),
             "xent_forward_train: NULL output");
  return gr_loss::forward(logits, ld, rows, classes, labels, mask, mean, nullptr, grad, ldg, train,
                          loss, stats, workspace, workspace_doubles, stream);
}

extern "C" int gr_xent_backward(const float* grad, int64_t rows, int64_t classes,
                                const uint64_t* train, const float* gloss, const int64_t* n_train,
                                float* out, void* stream) {
  using namespace gr_loss;
  gr::clear_error();
  GR_REQUIRE(rows >= 0 && classes >= 1 && classes <= (1 << 24), "xent_backward: bad shape");
  if (rows == 0) return GR_OK;
  GR_REQUIRE(grad && train && gloss && out, "xent_backward: NULL pointer");
  const int64_t nblk = (rows + kRowsPerBlock - 1) / kRowsPerBlock;
  GR_REQUIRE(nblk <= INT32_MAX, "xent_backward: too many rows");
  hipStream_t s = gr::as_stream(stream);
  if (classes <= kSmallC)
    hipLaunchKernelGGL((xent_backward<true>), dim3((unsigned)nblk), dim3(256), 0, s, grad, rows,
                       (int)classes, train, gloss, n_train, out);
  else
    hipLaunchKernelGGL((xent_backward<false>), dim3((unsigned)nblk), dim3(256), 0, s, grad, rows,
                       (int)classes, train, gloss, n_train, out);
  GR_HIP_CHECK(hipGetLastError());
  return GR_OK;
}
