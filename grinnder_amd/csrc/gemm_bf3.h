// Tiled fp32 products on the bf16 matrix cores (three-way split, bf16x3.h).
#ifndef GR_GEMM_BF3_H
#define GR_GEMM_BF3_H

#include "bf16x3.h"
#include "wave.h"

namespace gr_bf3 {

constexpr int kXcds = 8;

// LDS image of one 16-k chunk: 16-byte units (8 consecutive k of one row of A
// or column of B), unit (piece p, k half q, row) at (2 p + q) (ROWS + 8) + row.
// A lane's fragment of a 32 x 32 x 16 step is one unit; the 32 rows of a
// fragment are 512 contiguous bytes, and the 8 pad units put the two k halves
// 32 banks apart, so reads and writes are free of bank conflicts.
template <int ROWS>
constexpr int chunk_units() {
  return 6 * (ROWS + 8);
}

template <int ROWS>
__device__ __forceinline__ int unit_of(int p, int q, int row) {
  return (2 * p + q) * (ROWS + 8) + row;
}

// t, or NaN where a sum of the block is infinite or NaN.  (A lane holds column
// lane % 32 of a 32 x 32 block, rows 8 (e / 4) + 4 (lane / 32) + e % 4, e < 16.)
__device__ __forceinline__ float nonfinite(const floatx16& acc, float t) {
#pragma unroll
  for (int e = 0; e < 16; ++e) t = fmaf(acc[e], 0.f, t);
  return t;
}

// C[M, N] = A[M, K] B[N, K]^T (+ bias[N]), all row-major: the dense transform's
// forward y = x W^T + b and input gradient dx = dy W (B = W^T).  Workgroup:
// WM x WN wavefronts, each MI x NJ blocks of 32 x 32; K in chunks of 16 through two LDS buffers,
// one barrier a chunk; chunk c + 2 is loaded and chunk c + 1 split and written
// while chunk c's products run.  The column tiles of one row tile are
// consecutive workgroups of one XCD, so A is read from HBM once and from that
// XCD's L2 after.  KN: B is [K, N] (dx = dy W from W itself), its pieces read as
// four rows' elements.  VEC: 4 with 16-byte rows of A (and B), else 1; TAIL: K is
// not a multiple of 16; store: 2 with 16-byte rows of C, 1 with any rows up to
// 2^21 floats apart, else 0.  Each output is one wavefront's sum in a fixed order.
//
// Bound by the matrix cores' power: at 250k x 256 x 1024 they are busy 71% of
// the cycles at 1.5 GHz (203 TFLOP/s of fp32 work; 115 with the fp32 matrix
// instructions).  Dealing the split out between the products gained 5% over
// leaving it in front of them; holding W's pieces from one workgroup to the
// next would take 1.5 times the LDS there is.
template <int WM, int WN, int MI, int NJ, int VEC, bool TAIL, bool KN>
__global__ __launch_bounds__(WM* WN * 64, 2) void gemm_nt_bf3(
    const float* __restrict__ A, int64_t lda, const float* __restrict__ B, int64_t ldb,
    const float* __restrict__ bias, float* __restrict__ C, int64_t ldc, int64_t M, int N, int K,
    int tiles_n, int store) {
  constexpr int T = WM * WN * 64, BM = WM * MI * 32, BN = WN * NJ * 32, R = BM + BN;
  constexpr int SA = BM * 4 / T, SB = BN * 4 / T;  // 4-k pieces a thread stages
  static_assert(BM * 4 % T == 0 && BN * 4 % T == 0, "staging slots");
  constexpr int UNITS = chunk_units<R>();
  // Two arrays, not one of twice the size: the compiler then knows that a
  // chunk's fragment reads and the next chunk's writes do not overlap.
  __shared__ __align__(16) uint4 lds0[UNITS];
  __shared__ __align__(16) uint4 lds1[UNITS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  const int r32 = lane & 31, q = lane >> 5;
  const int g = blockIdx.x, slot = g / kXcds;
  const int64_t m0 = ((int64_t)(slot / tiles_n) * kXcds + g % kXcds) * BM;
  if (m0 >= M) return;  // whole workgroup
  const int n0 = (slot % tiles_n) * BN;
  const int rows = (int)(M - m0 < BM ? M - m0 : BM);  // rows of this tile
  const int cols = N - n0 < BN ? N - n0 : BN;
  const float* Ab = A + m0 * lda;
  const float* Bb = B + (int64_t)n0 * ldb;
  const int nch = (K + 15) / 16;

  // Rows past the tile's end re-read its first row; what they give is not
  // stored.  k past K reads as 0.
  const float* pa[SA];
  const float* pb[SB];
  const int kq = tid & 3;
#pragma unroll
  for (int i = 0; i < SA; ++i) {
    const int row = (tid + i * T) >> 2;
    pa[i] = Ab + (int64_t)(row < rows ? row : 0) * lda;
  }
#pragma unroll
  for (int i = 0; i < SB; ++i) {
    const int row = (tid + i * T) >> 2;
    pb[i] = KN ? B + n0 + (row < cols ? row : 0) : Bb + (int64_t)(row < cols ? row : 0) * ldb;
  }
  // Loads are unconditional (one basic block a chunk): past the last chunk they
  // re-read it.  With TAIL (K not a multiple of 16) a piece past K reads the
  // row's start, and A's is made 0 in put, so the products there are 0.
  const int kend = nch * 16 - 16 + kq * 4;
  auto load_piece = [&](const float* p, int k) {
    float4 v;
    if constexpr (VEC == 4) {
      v = *reinterpret_cast<const float4*>(p + (TAIL && k >= K ? 0 : k));
    } else {
      v.x = p[k + 0 < K ? k + 0 : 0];
      v.y = p[k + 1 < K ? k + 1 : 0];
      v.z = p[k + 2 < K ? k + 2 : 0];
      v.w = p[k + 3 < K ? k + 3 : 0];
    }
    return v;
  };
  // Staged piece i of this thread: i < SA of A, else of B.
  constexpr int SP = SA + SB;
  float4 reg[SP];
  auto load_one = [&](int i, int c) {
    int k = c * 16 + kq * 4;
    k = k < kend ? k : kend;
    if (i < SA) {
      reg[i] = load_piece(pa[i < SA ? i : 0], k);
      if constexpr (TAIL) {
        reg[i].x = k + 0 < K ? reg[i].x : 0.f;
        reg[i].y = k + 1 < K ? reg[i].y : 0.f;
        reg[i].z = k + 2 < K ? reg[i].z : 0.f;
        reg[i].w = k + 3 < K ? reg[i].w : 0.f;
      }
    } else {
      const float* p = pb[i < SA ? 0 : i - SA];
      if constexpr (KN) {
        const int top = K - 1;
        reg[i].x = p[(int64_t)(TAIL && k + 0 > top ? top : k + 0) * ldb];
        reg[i].y = p[(int64_t)(TAIL && k + 1 > top ? top : k + 1) * ldb];
        reg[i].z = p[(int64_t)(TAIL && k + 2 > top ? top : k + 2) * ldb];
        reg[i].w = p[(int64_t)(TAIL && k + 3 > top ? top : k + 3) * ldb];
      } else {
        reg[i] = load_piece(p, k);
      }
    }
  };
  // Odd rows of A are negated (and their sums again at the end): see the
  // bias note in bf16x3.h.  A thread's rows have one parity (T / 4 is even).
  const unsigned odd = (unsigned)(tid & 4) << 29;
  auto val = [&](int i, float x) {
    return i < SA ? __builtin_bit_cast(float, __builtin_bit_cast(unsigned, x) ^ odd) : x;
  };
  auto put_one = [&](int i, uint4* buf, const uint2& h, const uint2& m, const uint2& l) {
    const int row = i < SA ? (tid + i * T) >> 2 : BM + ((tid + (i - SA) * T) >> 2);
    uint2* p = reinterpret_cast<uint2*>(buf + unit_of<R>(0, kq >> 1, row)) + (kq & 1);
    constexpr int PS = 2 * 2 * (R + 8);  // uint2 between pieces
    p[0] = h;
    p[PS] = m;
    p[2 * PS] = l;
  };

  floatx16 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = floatx16{};

  // One chunk: the products of `cur` in NS slots of MI matrix instructions,
  // with the split of chunk c + 1 (into nxt) and the loads of chunk c + 2
  // dealt out between them, a half piece (two k) at a time.  A matrix
  // instruction holds the matrix core for 8 issue slots, which the vector
  // instructions then fill; left to itself the compiler puts the whole split
  // in front of the products.
  auto step = [&](int c, const uint4* cur, uint4* nxt) {
    constexpr int NS = 6 * NJ, NH = 2 * SP;
    bf16x8 a[MI][3], b[2][3];
    uint2 h, m, l;
    auto frag = [&](int p, int row) {
      return *reinterpret_cast<const bf16x8*>(cur + unit_of<R>(p, q, row));
    };
#pragma unroll
    for (int p = 0; p < 3; ++p) b[0][p] = frag(p, BM + wn * NJ * 32 + r32);
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int p = 2; p >= 0; --p) a[i][p] = frag(p, wm * MI * 32 + i * 32 + r32);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int j = s / 6, t = s % 6;
      if (t == 0 && j + 1 < NJ) {
#pragma unroll
        for (int p = 0; p < 3; ++p)
          b[(j + 1) & 1][p] = frag(p, BM + wn * NJ * 32 + (j + 1) * 32 + r32);
      }
#pragma unroll
      for (int i = 0; i < MI; ++i)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][kPieceA[t]], b[j & 1][kPieceB[t]],
                                                            acc[i][j], 0, 0, 0);
#pragma unroll
      for (int e = 0; e < NH; ++e) {
        if (e * NS / NH != s) continue;
        const int i = e / 2;
        if (e % 2 == 0) {
          split2(val(i, reg[i].x), val(i, reg[i].y), h.x, m.x, l.x);
        } else {
          split2(val(i, reg[i].z), val(i, reg[i].w), h.y, m.y, l.y);
          put_one(i, nxt, h, m, l);  // the last chunk's writes are read by nobody
          load_one(i, c + 2);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
  };
#pragma unroll
  for (int i = 0; i < SP; ++i) load_one(i, 0);
#pragma unroll
  for (int i = 0; i < SP; ++i) {
    uint2 h, m, l;
    split2(val(i, reg[i].x), val(i, reg[i].y), h.x, m.x, l.x);
    split2(val(i, reg[i].z), val(i, reg[i].w), h.y, m.y, l.y);
    put_one(i, lds0, h, m, l);
    load_one(i, 1);
  }
  __syncthreads();
  int c = 0;
  for (; c + 1 < nch; c += 2) {
    step(c, lds0, lds1);
    step(c + 1, lds1, lds0);
  }
  if (c < nch) step(c, lds0, lds1);

  // Non-finite sums: the wavefront forms its blocks again in fp32.
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) t = nonfinite(acc[i][j], t);
  const bool redo = __any(t != t);
  if (redo) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = floatx16{};
    for (int k = 0; k < K; k += 2) {
      const bool in = k + q < K;
      float a[MI], b[NJ];
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const int row = wm * MI * 32 + i * 32 + r32;
        a[i] = in ? Ab[(int64_t)(row < rows ? row : 0) * lda + k + q] : 0.f;
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int col = wn * NJ * 32 + j * 32 + r32;
        const int64_t at = col < cols ? col : 0;
        b[j] = !in ? 0.f : KN ? B[(int64_t)(k + q) * ldb + n0 + at] : Bb[at * ldb + k + q];
      }
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
    }
  }

  const float sgn = redo ? 1.f : -1.f;  // odd rows were summed negated
  const int qc = lane & 3, qa = r32 >> 2;
  float* Cb = C + m0 * ldc + n0;
  // This lane's bias in block column j.  Loaded between the stores, which
  // paces them: 300k x 256 x 128 takes 144 us so, 154 with it loaded before
  // the loop.
  auto bias_of = [&](int j) {
    const int col = (wn * NJ + j) * 32 + r32;
    return bias != nullptr && col < cols ? bias[n0 + col] : 0.f;
  };
  if (store == 2) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const float bv = bias_of(j);
      const int col = (wn * NJ + j) * 32 + 4 * qa;
      float* p = Cb + (int64_t)(wm * MI * 32 + 4 * q + qc) * ldc + col;
      const int left = col < cols ? rows - (wm * MI * 32 + 4 * q + qc) : 0;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float v0 = acc[i][j][4 * e + 0] + bv, v1 = sgn * acc[i][j][4 * e + 1] + bv,
                v2 = acc[i][j][4 * e + 2] + bv, v3 = sgn * acc[i][j][4 * e + 3] + bv;
          gr_wave::quad_transpose(v0, v1, v2, v3, qc);
          if (i * 32 + 8 * e < left)
            *reinterpret_cast<float4*>(p + (i * 32 + 8 * e) * ldc) = make_float4(v0, v1, v2, v3);
        }
    }
    return;
  }
  if (store == 1) {
    // 4-byte stores go through a buffer resource over the tile's rows, which
    // drops rows past the matrix by itself, and lanes past its last column
    // have an offset past the resource: no branch around a store.  (With one
    // around each of these many stores 100k x 66 x 8 took 23 us, 11 now.)
    const uint32_t ldb4 = (uint32_t)ldc * 4u;
    const auto rs = gr_wave::buffer(Cb, (uint32_t)(rows - 1) * ldb4 + (uint32_t)cols * 4u);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const float bv = bias_of(j);
      const uint32_t col = (uint32_t)((wn * NJ + j) * 32 + r32);
      const uint32_t off =
          col < (uint32_t)cols ? (uint32_t)(wm * MI * 32 + 4 * q) * ldb4 + col * 4u
                               : gr_wave::kBufferDrop;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          gr_wave::buffer_store(rs, off + (uint32_t)(i * 32 + 8 * (e / 4) + e % 4) * ldb4,
                                (e % 2 ? sgn * acc[i][j][e] : acc[i][j][e]) + bv);
    }
    return;
  }
  // Rows too far apart for 32-bit offsets within a tile.
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const float bv = bias_of(j);
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = (wm * MI + i) * 32 + 8 * (e / 4) + 4 * q + e % 4;
        const int col = (wn * NJ + j) * 32 + r32;
        if (row < rows && col < cols)
          Cb[row * ldc + col] = (e % 2 ? sgn * acc[i][j][e] : acc[i][j][e]) + bv;
      }
  }
}

// part[z][M, N] = A[k rows of z]^T B[k rows of z] for A [K, M], B [K, N]
// row-major (the weight gradient's split-K product).  Tiles, LDS image and
// step as gemm_nt_bf3; a thread stages 4 consecutive k of one column, read as
// four rows' elements (32 columns, 128 bytes, a row and instruction), so the
// operands need no alignment.  The tiles of one K chunk are consecutive
// workgroups of one XCD: the chunk's rows come from HBM once.  LONG: rows so
// long (2^25 floats) that 32-bit offsets within 16 of them would not do.
//
// 1M rows of 256 x 256 in 256 chunks: 0.76 ms (172 TFLOP/s), against 1.23 ms
// with the fp32 matrix instructions.
template <int WM, int WN, int MI, int NJ, bool LONG>
__global__ __launch_bounds__(WM* WN * 64, 2) void gemm_tn_bf3(
    const float* __restrict__ A, int64_t lda, const float* __restrict__ B, int64_t ldb, int M,
    int N, int64_t K, int64_t kchunk, int nchunks, int tiles_m, int tiles,
    float* __restrict__ part) {
  constexpr int T = WM * WN * 64, BM = WM * MI * 32, BN = WN * NJ * 32, R = BM + BN;
  constexpr int SLOTS = 4 * R, SP = (SLOTS + T - 1) / T;
  constexpr int UNITS = chunk_units<R>();
  __shared__ __align__(16) uint4 lds0[UNITS];
  __shared__ __align__(16) uint4 lds1[UNITS];
  const int w = blockIdx.x, slot = w / kXcds, tile = slot % tiles;
  const int z = (slot / tiles) * kXcds + w % kXcds;
  if (z >= nchunks) return;  // whole workgroup
  const int m0 = (tile % tiles_m) * BM, n0 = (tile / tiles_m) * BN;
  const int64_t k_begin = (int64_t)z * kchunk;
  const int krows = (int)(k_begin + kchunk < K ? kchunk : K - k_begin);
  const int nch = (krows + 15) / 16;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  const int r32 = lane & 31, q = lane >> 5;
  const float* Ab = A + k_begin * lda;
  const float* Bb = B + k_begin * ldb;

  // Slot e of this thread: column `row` of the tile (of A below BM, of B
  // above; one or the other for a whole wavefront), k quad kq of the chunk.
  // Loads go through buffer resources over the chunk's rows: k past the
  // chunk's end and columns past the matrix read as 0 without an access.
  int row[SP], kq[SP];
  unsigned off[SP];
  bool isa[SP];
#pragma unroll
  for (int e = 0; e < SP; ++e) {
    const int idx = tid + e * T < SLOTS ? tid + e * T : SLOTS - 1;
    const int rem = idx % (2 * R);
    row[e] = rem >> 1;
    kq[e] = idx / (2 * R) * 2 + (rem & 1);
    const int first = (wave * 64 + e * T) % (2 * R) >> 1;  // the wavefront's first column
    isa[e] = first < BM;
    const int c = isa[e] ? m0 + row[e] : n0 + row[e] - BM;
    if constexpr (LONG) off[e] = (unsigned)c;
    else
      off[e] = c < (isa[e] ? M : N)
                   ? 4u * ((unsigned)kq[e] * 4u * (unsigned)(isa[e] ? lda : ldb) + (unsigned)c)
                   : gr_wave::kBufferDrop;
  }
  float4 reg[SP];
  auto load_one = [&](int e, int c) {
    const int left = krows - c * 16 < 16 ? krows - c * 16 : 16;
    const int64_t ld = isa[e] ? lda : ldb;
    if constexpr (LONG) {
      const float* p = (isa[e] ? Ab : Bb) + (int64_t)c * 16 * ld + off[e];
      const bool in = off[e] < (unsigned)(isa[e] ? M : N);
      auto at = [&](int k) { return in && k < left ? p[k * ld] : 0.f; };
      reg[e] = make_float4(at(4 * kq[e]), at(4 * kq[e] + 1), at(4 * kq[e] + 2),
                           at(4 * kq[e] + 3));
      return;
    }
    const auto rs = gr_wave::buffer((isa[e] ? Ab : Bb) + (int64_t)c * 16 * ld,
                                    left > 0 ? (uint32_t)left * (uint32_t)ld * 4u : 0u);
    auto at = [&](int j) {
      return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                           rs, off[e] + 4u * (uint32_t)ld * j, 0, 0));
    };
    reg[e] = make_float4(at(0), at(1), at(2), at(3));
  };
  // Odd K chunks sum -A (and store the sum negated): see the bias note in
  // bf16x3.h.
  const unsigned odd = (unsigned)(z & 1) << 31;
  auto val = [&](int e, float x) {
    return isa[e] ? __builtin_bit_cast(float, __builtin_bit_cast(unsigned, x) ^ odd) : x;
  };
  auto put_one = [&](int e, uint4* buf, const uint2& h, const uint2& m, const uint2& l) {
    if (SLOTS % T != 0 && tid + e * T >= SLOTS) return;
    uint2* p = reinterpret_cast<uint2*>(buf + unit_of<R>(0, kq[e] >> 1, row[e])) + (kq[e] & 1);
    constexpr int PS = 2 * 2 * (R + 8);
    p[0] = h;
    p[PS] = m;
    p[2 * PS] = l;
  };

  floatx16 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = floatx16{};

  auto step = [&](int c, const uint4* cur, uint4* nxt) {
    constexpr int NS = 6 * NJ, NH = 2 * SP;
    bf16x8 a[MI][3], b[2][3];
    uint2 h, m, l;
    auto frag = [&](int p, int r) {
      return *reinterpret_cast<const bf16x8*>(cur + unit_of<R>(p, q, r));
    };
#pragma unroll
    for (int p = 0; p < 3; ++p) b[0][p] = frag(p, BM + wn * NJ * 32 + r32);
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int p = 2; p >= 0; --p) a[i][p] = frag(p, wm * MI * 32 + i * 32 + r32);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int j = s / 6, t = s % 6;
      if (t == 0 && j + 1 < NJ) {
#pragma unroll
        for (int p = 0; p < 3; ++p)
          b[(j + 1) & 1][p] = frag(p, BM + wn * NJ * 32 + (j + 1) * 32 + r32);
      }
#pragma unroll
      for (int i = 0; i < MI; ++i)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][kPieceA[t]], b[j & 1][kPieceB[t]],
                                                            acc[i][j], 0, 0, 0);
#pragma unroll
      for (int e2 = 0; e2 < NH; ++e2) {
        if (e2 * NS / NH != s) continue;
        const int e = e2 / 2;
        if (e2 % 2 == 0) {
          split2(val(e, reg[e].x), val(e, reg[e].y), h.x, m.x, l.x);
        } else {
          split2(val(e, reg[e].z), val(e, reg[e].w), h.y, m.y, l.y);
          put_one(e, nxt, h, m, l);
          load_one(e, c + 2);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
  };
#pragma unroll
  for (int e = 0; e < SP; ++e) load_one(e, 0);
#pragma unroll
  for (int e = 0; e < SP; ++e) {
    uint2 h, m, l;
    split2(val(e, reg[e].x), val(e, reg[e].y), h.x, m.x, l.x);
    split2(val(e, reg[e].z), val(e, reg[e].w), h.y, m.y, l.y);
    put_one(e, lds0, h, m, l);
    load_one(e, 1);
  }
  __syncthreads();
  int c = 0;
  for (; c + 1 < nch; c += 2) {
    step(c, lds0, lds1);
    step(c + 1, lds1, lds0);
  }
  if (c < nch) step(c, lds0, lds1);

  float t = 0.f;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) t = nonfinite(acc[i][j], t);
  const bool redo = __any(t != t);
  if (redo) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = floatx16{};
    for (int k = 0; k < krows; k += 2) {
      const bool in = k + q < krows;
      float a[MI], b[NJ];
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const int m = m0 + wm * MI * 32 + i * 32 + r32;
        a[i] = in && m < M ? Ab[(int64_t)(k + q) * lda + m] : 0.f;
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int n = n0 + wn * NJ * 32 + j * 32 + r32;
        b[j] = in && n < N ? Bb[(int64_t)(k + q) * ldb + n] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
    }
  }

  const float sgn = !redo && (z & 1) ? -1.f : 1.f;
  float* out = part + (int64_t)z * M * N;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int n = n0 + wn * NJ * 32 + j * 32 + r32;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + wm * MI * 32 + i * 32 + 8 * (e / 4) + 4 * q + e % 4;
        if (m < M && n < N) out[(int64_t)m * N + n] = sgn * acc[i][j][e];
      }
    }
}

}  // namespace gr_bf3

#endif
