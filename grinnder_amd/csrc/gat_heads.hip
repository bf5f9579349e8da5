// GAT attention with several heads, or one of 36 to 64 channels, for gfx950:
// one pass over the edges each way (semantics as gat.hip: PyG GATConv,
// grinnder/nn/gat.py:54-61,69-78).
//
// Lanes are laid out by head: head h owns LPH consecutive lane positions (LPH
// the power of two at or above its C / 4 vectors), so a head's softmax state
// is held by its own lanes, its dot products are reduced over an aligned lane
// group, and no loop runs over the heads.  A wavefront takes one plan unit
// (row, edge range, slot) at a time; for narrow rows (up to 32 lane positions)
// 64 / G edge slots of G lanes work on the unit's edges side by side.
//
// Forward: an online softmax.  Per block of U edges a lane takes its head's
// logits s_j + d_i (the H values of a source row are one 4H-byte piece of a
// line), the running maximum, sum and weighted row sum, rescaled once a block.
// No alpha is stored.  For the backward it also keeps, per row and head,
//   N_i = sum_{t_ij <= 0} alpha_ij Hs_j  and  S_i = sum_{t_ij <= 0} alpha_ij.
// Backward, destination rows: c_i = <G_i, O_i> and
//   dd_i = -0.8 (<G_i, N_i> - c_i S_i) + c_i 1e-16 / den_i,
// the sum of the logit gradients over the row's edges (softmax is invariant to
// a shift of the row, so the plain sum is c_i 1e-16 / den_i, and LeakyReLU
// takes off 0.8 of the part with t <= 0); and a record rec_ih = (d, m, 1 / den,
// c).  Backward, source columns: an edge costs its row of G and its record
// (16 H bytes, one line for eight heads); alpha is formed again from it.
//
// Bound by the gathers of 4 H C-byte rows: 8 heads of 32 over 4M edges, 100k
// rows and 200k sources take 0.64 ms forward (6.4 TB/s of rows) and 0.63 + 0.06
// ms backward, against 1.29 and 1.31 ms for statistics, alpha and aggregation
// as three passes that loop over the heads with an exchange across the
// wavefront for each, with alpha and the logit gradients written per edge and
// head (a line each way for 32 bytes).  8 heads of 8 over 1M edges: 0.047 ms
// forward against 0.20.
#include <algorithm>
#include <cfloat>

#include "gr_internal.h"
#include "wave.h"

namespace gr_gath {

__device__ __forceinline__ float leaky(float t) { return t > 0.f ? t : 0.2f * t; }

__device__ __forceinline__ int64_t wave_id() {
  return (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}

// Four floats at any 4-byte boundary: one access, as aligned ones (a head's
// rows start anywhere when its channels are not a multiple of 4; 8 heads of 27
// and 2 of 95 took 2 to 4 times as long with 4-byte accesses).
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));

template <int VEC>
__device__ __forceinline__ void ld(const float* __restrict__ p, float (&r)[VEC]) {
  if constexpr (VEC == 4) {
    const float4u t = *reinterpret_cast<const float4u*>(p);
    r[0] = t.x; r[1] = t.y; r[2] = t.z; r[3] = t.w;
  } else {
    r[0] = *p;
  }
}

template <int VEC>
__device__ __forceinline__ void st(float* __restrict__ p, const float (&r)[VEC]) {
  if constexpr (VEC == 4) *reinterpret_cast<float4u*>(p) = float4u{r[0], r[1], r[2], r[3]};
  else *p = r[0];
}

// A lane's place in chunk ch of a row: head, feature and whether it holds any
// (lanes that do not read head 0's first vector and count as 0).  The last
// vector of a head whose channels are not a multiple of 4 ends with the head:
// its first `dup` features are its neighbour's too.  Both hold and store the
// same values for them; sums over the head leave them out here, by a select and
// not by a factor of 0, which an infinity or NaN of head 0 would turn into NaN
// in a lane of another head.
struct Place {
  int head, feat, dup;
  bool ok, lead;  // lead: the first lane of its head
};
template <int VEC>
__device__ __forceinline__ Place place(int p, int lph, int H, int C) {
  const int h = p / lph, v = p & (lph - 1);
  const bool ok = h < H && v * VEC < C;
  const int c = v * VEC + VEC <= C ? v * VEC : C - VEC;
  return Place{ok ? h : 0, ok ? h * C + c : 0, ok ? v * VEC - c : VEC, ok, ok && v == 0};
}

// t[u][ch] summed over the lanes of its head, for U edges at once: one uniform
// branch for all of them.
template <int U, int NCH>
__device__ __forceinline__ void head_sums(float (&t)[U][NCH], int lph) {
#define GR_EACH(N)                                 \
  {                                                \
    _Pragma("unroll") for (int u = 0; u < U; ++u)  \
    _Pragma("unroll") for (int c = 0; c < NCH; ++c) t[u][c] = gr_wave::group_sum<N>(t[u][c]); \
  }
  if (lph >= 64) {
    // A head over lph / 64 chunks.
    const int span = lph >> 6;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (span == 2) {
#pragma unroll
        for (int c = 0; c + 1 < NCH; c += 2) t[u][c] = t[u][c + 1] = t[u][c] + t[u][c + 1];
      } else if (span == 4) {
#pragma unroll
        for (int c = 0; c + 3 < NCH; c += 4)
          t[u][c] = t[u][c + 1] = t[u][c + 2] = t[u][c + 3] =
              (t[u][c] + t[u][c + 1]) + (t[u][c + 2] + t[u][c + 3]);
      }
    }
    GR_EACH(64)
  } else if (lph == 32) GR_EACH(32)
  else if (lph == 16) GR_EACH(16)
  else if (lph == 8) GR_EACH(8)
  else if (lph == 4) GR_EACH(4)
  else if (lph == 2) GR_EACH(2)
#undef GR_EACH
}

// Workspace of one split unit: acc [HC4] (| N [HC4]) | m [H4] | sum [H4] | S [H4].
__host__ __device__ inline int pad4(int n) { return (n + 3) & ~3; }

// ------------------------------------------------------------- forward --

// NEG: also N and S, the state of a backward.
template <int VEC, int G, int NCH, int U, bool NEG>
__global__ __launch_bounds__(256) void gat_heads_fwd(
    const int4* __restrict__ units, int64_t n_units, const int32_t* __restrict__ idx,
    const float* __restrict__ hs, int64_t ldh, const float* __restrict__ s,
    const float* __restrict__ d, int H, int C, int lph, const float* __restrict__ bias,
    float4* __restrict__ state, float* __restrict__ nrow, float* __restrict__ o,
    float* __restrict__ y, float* __restrict__ ws) {
  constexpr int EPI = 64 / G;
  static_assert(EPI == 1 || NCH == 1, "edge slots hold one chunk");
  const int lane = threadIdx.x & 63;
  const int64_t wid = wave_id();
  if (wid >= n_units) return;
  const int4 w = units[wid];
  const int64_t i = w.x;
  const int HC = H * C;
  const int slot = EPI == 1 ? 0 : lane / G;
  const int li = EPI == 1 ? lane : lane % G;
  Place pl[NCH];
  float di[NCH], m[NCH], sum[NCH], sneg[NCH], acc[NCH][VEC], neg[NCH][VEC];
#pragma unroll
  for (int ch = 0; ch < NCH; ++ch) {
    pl[ch] = place<VEC>(ch * 64 + li, lph, H, C);
    di[ch] = d[i * H + pl[ch].head];
    m[ch] = -FLT_MAX;
    sum[ch] = sneg[ch] = 0.f;
#pragma unroll
    for (int q = 0; q < VEC; ++q) acc[ch][q] = neg[ch][q] = 0.f;
  }
  int cnext = w.y < w.z ? idx[min(w.y + lane, w.z - 1)] : 0;
  for (int b = w.y; b < w.z; b += 64) {
    const int n = min(64, w.z - b);
    const int cl = cnext;
    if (b + 64 < w.z) cnext = idx[min(b + 64 + lane, w.z - 1)];
    for (int k = 0; k < n; k += EPI * U) {
      float r[U][NCH][VEC], t[U][NCH];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = EPI == 1 ? __builtin_amdgcn_readlane(cl, k + u)
                               : __shfl(cl, k + u * EPI + slot, 64);
        const float* row = hs + (int64_t)c * ldh;
        const float* sr = s + (int64_t)c * H;
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) t[u][ch] = sr[pl[ch].head];
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) ld<VEC>(row + pl[ch].feat, r[u][ch]);
      }
#pragma unroll
      for (int ch = 0; ch < NCH; ++ch) {
        float top = m[ch];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          t[u][ch] += di[ch];
          if (k + u * EPI + slot < n) top = fmaxf(top, leaky(t[u][ch]));
        }
        const float scale = expf(m[ch] - top);
        m[ch] = top;
        sum[ch] *= scale;
        if constexpr (NEG) sneg[ch] *= scale;
#pragma unroll
        for (int q = 0; q < VEC; ++q) {
          acc[ch][q] *= scale;
          if constexpr (NEG) neg[ch][q] *= scale;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const float p = k + u * EPI + slot < n ? expf(leaky(t[u][ch]) - top) : 0.f;
          sum[ch] += p;
#pragma unroll
          for (int q = 0; q < VEC; ++q) acc[ch][q] = fmaf(p, r[u][ch][q], acc[ch][q]);
          if constexpr (NEG) {
            const float pn = t[u][ch] > 0.f ? 0.f : p;
            sneg[ch] += pn;
#pragma unroll
            for (int q = 0; q < VEC; ++q) neg[ch][q] = fmaf(pn, r[u][ch][q], neg[ch][q]);
          }
        }
      }
    }
  }
  if constexpr (EPI > 1) {
    // The slots' states, in a fixed exchange order.
    float top = m[0];
#pragma unroll
    for (int x = G; x < 64; x <<= 1) top = fmaxf(top, __shfl_xor(top, x, 64));
    const float scale = expf(m[0] - top);
    m[0] = top;
    sum[0] = gr_wave::slot_sum<G>(sum[0] * scale);
    if constexpr (NEG) sneg[0] = gr_wave::slot_sum<G>(sneg[0] * scale);
#pragma unroll
    for (int q = 0; q < VEC; ++q) {
      acc[0][q] = gr_wave::slot_sum<G>(acc[0][q] * scale);
      if constexpr (NEG) neg[0][q] = gr_wave::slot_sum<G>(neg[0][q] * scale);
    }
    if (slot != 0) return;
  }
  if (w.w < 0) {
    const bool empty = w.z <= w.y;
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) {
      if (!pl[ch].ok) continue;
      const float den = empty ? 1.f : sum[ch] + 1e-16f;
      const float inv = 1.f / den;
      const int f = pl[ch].feat;
      if (NEG && pl[ch].lead)
        state[i * H + pl[ch].head] =
            make_float4(di[ch], empty ? 0.f : m[ch], den, sneg[ch] * inv);
      float v[VEC];
#pragma unroll
      for (int q = 0; q < VEC; ++q) v[q] = acc[ch][q] * inv;
      if (o != nullptr) st<VEC>(o + i * HC + f, v);
      if (y != nullptr) {
        float bv[VEC];
        ld<VEC>(bias + f, bv);
#pragma unroll
        for (int q = 0; q < VEC; ++q) v[q] += bv[q];
        st<VEC>(y + i * HC + f, v);
      }
      if constexpr (NEG) {
#pragma unroll
        for (int q = 0; q < VEC; ++q) v[q] = neg[ch][q] * inv;
        st<VEC>(nrow + i * HC + f, v);
      }
    }
  } else {
    const int hc4 = pad4(HC), h4 = pad4(H);
    float* p = ws + (int64_t)w.w * ((NEG ? 2 : 1) * hc4 + 3 * h4);
    float* q4 = p + (NEG ? 2 : 1) * hc4;
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) {
      if (!pl[ch].ok) continue;
      st<VEC>(p + pl[ch].feat, acc[ch]);
      if constexpr (NEG) st<VEC>(p + hc4 + pl[ch].feat, neg[ch]);
      if (pl[ch].lead) {
        q4[pl[ch].head] = m[ch];
        q4[h4 + pl[ch].head] = sum[ch];
        q4[2 * h4 + pl[ch].head] = sneg[ch];
      }
    }
  }
}

// Split rows: one workgroup a row, a thread per feature; slots in order.
__global__ __launch_bounds__(256) void gat_heads_fwd_fixup(
    const int32_t* __restrict__ fix, const float* __restrict__ ws, int neg, int H, int C,
    const float* __restrict__ d, const float* __restrict__ bias, float4* __restrict__ state,
    float* __restrict__ nrow, float* __restrict__ o, float* __restrict__ y) {
  const int64_t row = fix[3 * (int64_t)blockIdx.x + 0];
  const int first = fix[3 * (int64_t)blockIdx.x + 1], n = fix[3 * (int64_t)blockIdx.x + 2];
  const int HC = H * C, hc4 = pad4(HC), h4 = pad4(H);
  const int ns = (neg ? 2 : 1) * hc4, stride = ns + 3 * h4;
  const float* base = ws + (int64_t)first * stride;
  for (int f = threadIdx.x; f < HC; f += 256) {
    const int h = f / C;
    float m = -FLT_MAX;
    for (int k = 0; k < n; ++k) m = fmaxf(m, base[(int64_t)k * stride + ns + h]);
    float sum = 0.f, s0 = 0.f, acc = 0.f, nacc = 0.f;
    for (int k = 0; k < n; ++k) {
      const float* p = base + (int64_t)k * stride;
      const float sc = expf(p[ns + h] - m);
      sum = fmaf(p[ns + h4 + h], sc, sum);
      s0 = fmaf(p[ns + 2 * h4 + h], sc, s0);
      acc = fmaf(p[f], sc, acc);
      if (neg) nacc = fmaf(p[hc4 + f], sc, nacc);
    }
    const float den = sum + 1e-16f, inv = 1.f / den;
    if (o != nullptr) o[row * HC + f] = acc * inv;
    if (y != nullptr) y[row * HC + f] = acc * inv + bias[f];
    if (neg) {
      nrow[row * HC + f] = nacc * inv;
      if (f == h * C) state[row * H + h] = make_float4(d[row * H + h], m, den, s0 * inv);
    }
  }
}

// ---------------------------------------------------- backward, rows --

// Per row and head: c, dd and the record.  64 / G rows a wavefront.
template <int VEC, int G, int NCH>
__global__ __launch_bounds__(256) void gat_heads_bwd_dst(
    const float* __restrict__ go, const float* __restrict__ o, const float* __restrict__ nrow,
    const float4* __restrict__ state, int64_t rows, int H, int C, int lph,
    float4* __restrict__ rec, float* __restrict__ dd) {
  constexpr int RPW = 64 / G;
  const int lane = threadIdx.x & 63;
  const int slot = RPW == 1 ? 0 : lane / G;
  const int li = RPW == 1 ? lane : lane % G;
  const int HC = H * C;
  Place pl[NCH];
#pragma unroll
  for (int ch = 0; ch < NCH; ++ch) pl[ch] = place<VEC>(ch * 64 + li, lph, H, C);
  const int64_t nwaves = (int64_t)gridDim.x * 4;
  for (int64_t r0 = wave_id() * RPW; r0 < rows; r0 += nwaves * RPW) {
    const bool in = r0 + slot < rows;
    const int64_t i = in ? r0 + slot : r0;
    float t[2][NCH];
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) {
      float g[VEC], a[VEC], b[VEC];
      ld<VEC>(go + i * HC + pl[ch].feat, g);
      ld<VEC>(o + i * HC + pl[ch].feat, a);
      ld<VEC>(nrow + i * HC + pl[ch].feat, b);
      t[0][ch] = t[1][ch] = 0.f;
#pragma unroll
      for (int q = 0; q < VEC; ++q) {
        if (q >= pl[ch].dup) {
          t[0][ch] = fmaf(g[q], a[q], t[0][ch]);
          t[1][ch] = fmaf(g[q], b[q], t[1][ch]);
        }
      }
    }
    head_sums<2, NCH>(t, lph);
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) {
      if (!in || !pl[ch].lead) continue;
      const float4 f = state[i * H + pl[ch].head];
      const float c = t[0][ch];
      dd[i * H + pl[ch].head] = -0.8f * (t[1][ch] - c * f.w) + c * (1e-16f / f.z);
      rec[i * H + pl[ch].head] = make_float4(f.x, f.y, 1.f / f.z, c);
    }
  }
}

// -------------------------------------------------- backward, columns --

template <int VEC, int G, int NCH, int U>
__global__ __launch_bounds__(256) void gat_heads_bwd_src(
    const int4* __restrict__ units, int64_t n_units, const int32_t* __restrict__ row_idx,
    const float* __restrict__ hs, int64_t ldh, const float* __restrict__ s,
    const float* __restrict__ go, const float4* __restrict__ rec, int H, int C, int lph,
    int64_t n_dst, const float* __restrict__ att_src, const float* __restrict__ att_dst,
    const float* __restrict__ dd, float* __restrict__ dhs, float* __restrict__ ds,
    float* __restrict__ ws) {
  constexpr int EPI = 64 / G;
  static_assert(EPI == 1 || NCH == 1, "edge slots hold one chunk");
  const int lane = threadIdx.x & 63;
  const int64_t wid = wave_id();
  if (wid >= n_units) return;
  const int4 w = units[wid];
  const int64_t j = w.x;
  const int HC = H * C;
  const int slot = EPI == 1 ? 0 : lane / G;
  const int li = EPI == 1 ? lane : lane % G;
  Place pl[NCH];
  float hsj[NCH][VEC], sj[NCH], acc[NCH][VEC], dsl[NCH];
#pragma unroll
  for (int ch = 0; ch < NCH; ++ch) {
    pl[ch] = place<VEC>(ch * 64 + li, lph, H, C);
    ld<VEC>(hs + j * ldh + pl[ch].feat, hsj[ch]);
    sj[ch] = s[j * H + pl[ch].head];
    dsl[ch] = 0.f;
#pragma unroll
    for (int q = 0; q < VEC; ++q) acc[ch][q] = 0.f;
  }
  int inext = w.y < w.z ? row_idx[min(w.y + lane, w.z - 1)] : 0;
  for (int b = w.y; b < w.z; b += 64) {
    const int n = min(64, w.z - b);
    const int il = inext;
    if (b + 64 < w.z) inext = row_idx[min(b + 64 + lane, w.z - 1)];
    for (int k = 0; k < n; k += EPI * U) {
      float g[U][NCH][VEC], t[U][NCH];
      float4 rc[U][NCH];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t i = EPI == 1 ? __builtin_amdgcn_readlane(il, k + u)
                                   : __shfl(il, k + u * EPI + slot, 64);
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) {
          rc[u][ch] = rec[i * H + pl[ch].head];
          ld<VEC>(go + i * HC + pl[ch].feat, g[u][ch]);
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) {
          t[u][ch] = 0.f;
#pragma unroll
          for (int q = 0; q < VEC; ++q)
            t[u][ch] = q >= pl[ch].dup ? fmaf(g[u][ch][q], hsj[ch][q], t[u][ch]) : t[u][ch];
        }
      head_sums<U, NCH>(t, lph);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool in = k + u * EPI + slot < n;
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) {
          const float tt = sj[ch] + rc[u][ch].x;
          const float a = in ? expf(leaky(tt) - rc[u][ch].y) * rc[u][ch].z : 0.f;
          const float ge = in ? a * (t[u][ch] - rc[u][ch].w) : 0.f;
          dsl[ch] += tt > 0.f ? ge : 0.2f * ge;
#pragma unroll
          for (int q = 0; q < VEC; ++q)
            if (in) acc[ch][q] = fmaf(a, g[u][ch][q], acc[ch][q]);
        }
      }
    }
  }
  if constexpr (EPI > 1) {
    dsl[0] = gr_wave::slot_sum<G>(dsl[0]);
#pragma unroll
    for (int q = 0; q < VEC; ++q) acc[0][q] = gr_wave::slot_sum<G>(acc[0][q]);
    if (slot != 0) return;
  }
  const int hc4 = pad4(HC);
  float* p = w.w < 0 ? nullptr : ws + (int64_t)w.w * (hc4 + pad4(H));
#pragma unroll
  for (int ch = 0; ch < NCH; ++ch) {
    if (!pl[ch].ok) continue;
    const int f = pl[ch].feat;
    if (w.w < 0) {
      float av[VEC], bv[VEC];
      ld<VEC>(att_src + f, av);
#pragma unroll
      for (int q = 0; q < VEC; ++q) av[q] = fmaf(dsl[ch], av[q], acc[ch][q]);
      if (j < n_dst) {
        const float v = dd[j * H + pl[ch].head];
        ld<VEC>(att_dst + f, bv);
#pragma unroll
        for (int q = 0; q < VEC; ++q) av[q] = fmaf(v, bv[q], av[q]);
      }
      st<VEC>(dhs + j * HC + f, av);
      if (pl[ch].lead) ds[j * H + pl[ch].head] = dsl[ch];
    } else {
      st<VEC>(p + f, acc[ch]);
      if (pl[ch].lead) p[hc4 + pl[ch].head] = dsl[ch];
    }
  }
}

// Split columns: one workgroup a column, slots in order.
__global__ __launch_bounds__(256) void gat_heads_bwd_fixup(
    const int32_t* __restrict__ fix, const float* __restrict__ ws, int H, int C, int64_t n_dst,
    const float* __restrict__ att_src, const float* __restrict__ att_dst,
    const float* __restrict__ dd, float* __restrict__ dhs, float* __restrict__ ds) {
  const int64_t row = fix[3 * (int64_t)blockIdx.x + 0];
  const int first = fix[3 * (int64_t)blockIdx.x + 1], n = fix[3 * (int64_t)blockIdx.x + 2];
  const int HC = H * C, hc4 = pad4(HC), stride = hc4 + pad4(H);
  for (int f = threadIdx.x; f < HC; f += 256) {
    const int h = f / C;
    float acc = 0.f, dsum = 0.f;
    for (int k = 0; k < n; ++k) {
      const float* p = ws + (int64_t)(first + k) * stride;
      acc += p[f];
      dsum += p[hc4 + h];
    }
    float v = fmaf(dsum, att_src[f], acc);
    if (row < n_dst) v = fmaf(dd[row * H + h], att_dst[f], v);
    dhs[row * HC + f] = v;
    if (f == h * C) ds[row * H + h] = dsum;
  }
}

// ------------------------------------------------------------ dispatch --

// Vector width, lanes per head, chunks of a row and lanes a slot.  Heads of at
// least 4 channels take 16-byte accesses; H * C <= 1024 then needs at most 512
// lanes.
struct Shape {
  int vec, lph, nch, g;
};
bool shape_of(int64_t H, int64_t C, Shape* s) {
  if (H < 1 || H > 16 || C < 1 || H * C > 1024) return false;
  s->vec = C >= 4 ? 4 : 1;
  int lph = 1;
  while (lph * s->vec < C) lph *= 2;
  const int lanes = (int)H * lph;
  s->lph = lph;
  s->nch = 1;
  while (64 * s->nch < lanes) s->nch *= 2;
  if (s->nch > 8 || lph > 256) return false;  // a head spans at most four chunks
  s->g = lanes <= 16 ? 16 : lanes <= 32 ? 32 : 64;
  return true;
}

inline unsigned blocks_for(int64_t waves) { return (unsigned)((waves + 3) / 4); }

// Edges in flight a lane, by chunks and vector width: at most 32 registers of
// rows (the state takes as many again).
template <int VEC, int NCH>
constexpr int edges() {
  return NCH * VEC >= 32 ? 1 : NCH * VEC >= 16 ? 2 : NCH * VEC >= 8 ? 4 : 8;
}

}  // namespace gr_gath

using namespace gr_gath;

#define GR_HEADS_SHAPES(VEC_, CALL)                     \
  do {                                                  \
    if (sh.nch == 1) {                                  \
      if (sh.g == 16) CALL(VEC_, 16, 1);                \
      else if (sh.g == 32) CALL(VEC_, 32, 1);           \
      else CALL(VEC_, 64, 1);                           \
    } else if (sh.nch == 2) CALL(VEC_, 64, 2);          \
    else if (sh.nch == 4) CALL(VEC_, 64, 4);            \
    else CALL(VEC_, 64, 8);                             \
  } while (0)
#define GR_HEADS(CALL)                                  \
  do {                                                  \
    if (sh.vec == 4) GR_HEADS_SHAPES(4, CALL);          \
    else if (sh.g == 16) CALL(1, 16, 1);                \
    else if (sh.g == 32) CALL(1, 32, 1);                \
    else CALL(1, 64, 1);                                \
  } while (0)

extern "C" int gr_gat_heads_workspace(int64_t H, int64_t C, int32_t with_state,
                                      int64_t* floats_per_slot) {
  gr::clear_error();
  GR_REQUIRE(H >= 1 && C >= 1 && H * C <= 1024 && floats_per_slot != nullptr,
             "gat_heads_workspace: bad arguments");
  *floats_per_slot = (with_state ? 2 : 1) * pad4((int)(H * C)) + 3 * pad4((int)H);
  return GR_OK;
}

extern "C" int gr_gat_heads_forward(const int32_t* units, int64_t n_units, const int32_t* fixups,
                                    int64_t n_fix, const int32_t* idx, const float* hs,
                                    int64_t ldh, const float* s, const float* d, int64_t H,
                                    int64_t C, const float* bias, float* state, float* nrow,
                                    float* o, float* y, float* ws, int64_t ws_floats,
                                    int64_t n_slots, void* stream) {
  gr::clear_error();
  Shape sh;
  GR_REQUIRE(n_units >= 0 && n_fix >= 0 && n_slots >= 0, "gat_heads_forward: negative count");
  GR_REQUIRE(ldh >= H * C, "gat_heads_forward: leading dimension too small");
  const bool with_bias = y != nullptr;
  GR_REQUIRE(shape_of(H, C, &sh),
             "gat_heads_forward: %lld heads of %lld channels", (long long)H, (long long)C);
  GR_REQUIRE((state != nullptr) == (nrow != nullptr) && (o != nullptr || y != nullptr) &&
                 (!with_bias || bias != nullptr),
             "gat_heads_forward: state and nrow go together, and y with a bias");
  GR_REQUIRE(n_units <= int64_t(INT32_MAX) * 4, "gat_heads_forward: too many units");
  if (n_units == 0) return GR_OK;
  GR_REQUIRE(units && idx && hs && s && d && (n_fix == 0 || fixups),
             "gat_heads_forward: NULL pointer");
  const int64_t stride = (nrow ? 2 : 1) * pad4((int)(H * C)) + 3 * pad4((int)H);
  GR_REQUIRE(n_slots == 0 || (ws != nullptr && ws_floats >= n_slots * stride),
             "gat_heads_forward: workspace too small");
  hipStream_t st = gr::as_stream(stream);
  const int4* u4 = reinterpret_cast<const int4*>(units);
  const dim3 grid(blocks_for(n_units)), blk(256);
#define GR_CALL(V, G, N)                                                                         \
  do {                                                                                           \
    if (nrow != nullptr)                                                                         \
      hipLaunchKernelGGL((gat_heads_fwd<V, G, N, edges<V, N>(), true>), grid, blk, 0, st, u4,    \
                         n_units, idx, hs, ldh, s, d, (int)H, (int)C, sh.lph, bias,              \
                         reinterpret_cast<float4*>(state), nrow, o, y, ws);                      \
    else                                                                                         \
      hipLaunchKernelGGL((gat_heads_fwd<V, G, N, edges<V, N>(), false>), grid, blk, 0, st, u4,   \
                         n_units, idx, hs, ldh, s, d, (int)H, (int)C, sh.lph, bias,              \
                         (float4*)nullptr, (float*)nullptr, o, y, ws);                           \
  } while (0)
  GR_HEADS(GR_CALL);
#undef GR_CALL
  GR_HIP_CHECK(hipGetLastError());
  if (n_fix > 0) {
    hipLaunchKernelGGL(gat_heads_fwd_fixup, dim3((unsigned)n_fix), blk, 0, st, fixups, ws,
                       nrow != nullptr ? 1 : 0, (int)H, (int)C, d, bias,
                       reinterpret_cast<float4*>(state), nrow, o, y);
    GR_HIP_CHECK(hipGetLastError());
  }
  return GR_OK;
}

extern "C" int gr_gat_heads_backward(const int32_t* units, int64_t n_units,
                                     const int32_t* fixups, int64_t n_fix,
                                     const int32_t* row_idx, const float* hs, int64_t ldh,
                                     const float* s, const float* go, const float* o,
                                     const float* nrow, const float* state, int64_t n_dst,
                                     int64_t H, int64_t C, const float* att_src,
                                     const float* att_dst, float* rec, float* dd, float* dhs,
                                     float* ds, float* ws, int64_t ws_floats, int64_t n_slots,
                                     void* stream) {
  gr::clear_error();
  Shape sh;
  GR_REQUIRE(n_units >= 0 && n_fix >= 0 && n_slots >= 0 && n_dst >= 0,
             "gat_heads_backward: negative count");
  GR_REQUIRE(ldh >= H * C, "gat_heads_backward: leading dimension too small");
  GR_REQUIRE(shape_of(H, C, &sh),
             "gat_heads_backward: %lld heads of %lld channels", (long long)H, (long long)C);
  GR_REQUIRE(n_units <= int64_t(INT32_MAX) * 4, "gat_heads_backward: too many units");
  const int64_t stride = pad4((int)(H * C)) + pad4((int)H);
  GR_REQUIRE(n_slots == 0 || (ws != nullptr && ws_floats >= n_slots * stride),
             "gat_heads_backward: workspace too small");
  hipStream_t st = gr::as_stream(stream);
  const dim3 blk(256);
  if (n_dst > 0) {
    GR_REQUIRE(go && o && nrow && state && rec && dd, "gat_heads_backward: NULL pointer");
    // Enough wavefronts for every SIMD to hold eight.
    const unsigned grid = (unsigned)std::min<int64_t>(2048, (n_dst + 3) / 4);
#define GR_CALL(V, G, N)                                                                        \
  hipLaunchKernelGGL((gat_heads_bwd_dst<V, G, N>), dim3(grid), blk, 0, st, go, o, nrow,         \
                     reinterpret_cast<const float4*>(state), n_dst, (int)H, (int)C, sh.lph,     \
                     reinterpret_cast<float4*>(rec), dd)
    GR_HEADS(GR_CALL);
#undef GR_CALL
    GR_HIP_CHECK(hipGetLastError());
  }
  if (n_units == 0) return GR_OK;
  GR_REQUIRE(units && row_idx && hs && s && go && rec && att_src && att_dst && dhs && ds &&
                 (n_fix == 0 || fixups),
             "gat_heads_backward: NULL pointer");
  const int4* u4 = reinterpret_cast<const int4*>(units);
  const dim3 grid(blocks_for(n_units));
#define GR_CALL(V, G, N)                                                                        \
  hipLaunchKernelGGL((gat_heads_bwd_src<V, G, N, edges<V, N>() / (N > 1 ? 1 : 2)>), grid, blk, 0, \
                     st, u4, n_units, row_idx, hs, ldh, s, go,                                  \
                     reinterpret_cast<const float4*>(rec), (int)H, (int)C, sh.lph, n_dst,       \
                     att_src, att_dst, dd, dhs, ds, ws)
  GR_HEADS(GR_CALL);
#undef GR_CALL
  GR_HIP_CHECK(hipGetLastError());
  if (n_fix > 0) {
    hipLaunchKernelGGL(gat_heads_bwd_fixup, dim3((unsigned)n_fix), blk, 0, st, fixups, ws, (int)H,
                       (int)C, n_dst, att_src, att_dst, dd, dhs, ds);
    GR_HIP_CHECK(hipGetLastError());
  }
  return GR_OK;
}
