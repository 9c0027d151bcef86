// mlp.hip -- the block-proposal network: a small MLP trained and run with
// hand-written BF16 MFMA kernels (FP32 accumulation) on gfx950.
//
// No counterpart in the reference: it ranks the (generator, hole-pair)
// blocks of select_singles_and_doubles (plugins/Full_CI_ZMQ/selection.irp.f:
// 412-575) -- the same unit the reference's `subset` / fragment_count filter
// acts on (:561-562) -- by predicted log|PT2 contribution|.
//
// Network: x (D_IN features) -> 256 -> 256 -> 256 (ReLU) -> 1.  Features of a
// block: learned 32-d embeddings of h1 and h2 (one table over orbitals),
// h_11 and h_22 orbital energies, log|c| of the generator, one-hot spin
// class (aa, bb, ab), one-hot excitation degree of the generator from HF
// (0..4), zero padding to D_IN = 80.
//
// A row's way through the network, forward and backward, needs no other row:
// mlp_rows_kernel takes 16 RT rows from their descriptors to the prediction
// (and, in training, on to the bias, head and embedding gradients) with the
// activations in LDS and the weights streamed from L2 in operand order.  A
// training step is that kernel, one launch for the sums over the batch (the
// three weight gradients, cut along it, and the column sums) and one that sums
// their slices and makes the Adam step.  It was 28 launches, with every activation and its
// gradient written and read in FP32 and bf16: 235 us a step at batch 4096.
//
// The weight gradients' product (gemm_tile, launched by grad_kernel; the plain
// GEMM around it serves the checks of the tile's lane layout):
// C(MxN) = A(MxK) B(KxN), A and B bf16 with arbitrary row/column
// strides (so A^T, B^T need no copies), C fp32; workgroup tile 64x64, four
// wavefronts each owning 32x32 = 2x2 tiles of v_mfma_f32_16x16x32_bf16
// (CDNA4's bf16 MFMA with K = 32, one per tile and K-tile of 32).
// Lane layout of the 16x16x32 MFMA: lane l holds A[l%16][8(l/16)+0..7],
// B[8(l/16)+0..7][l%16] and D[4(l/16)+0..3][l%16].  Both tiles sit in LDS
// with k contiguous (A as [i][k], B as [j][k]), so each lane's MFMA operand
// is one 16-byte read; they are staged in runs of 8 elements (16-byte loads)
// along whichever index of the operand is contiguous in memory.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <cstdio>
#include <mutex>
#include <type_traits>
#include <vector>
#include <hip/hip_bf16.h>
#include "qpx_internal.h"

using namespace qpx;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ inline uint16_t f2bf(float x) {  // round to nearest even
  uint32_t u = __float_as_uint(x);
  if ((u & 0x7fffffff) > 0x7f800000) return 0x7fc0;  // NaN
  u += 0x7fff + ((u >> 16) & 1);
  return (uint16_t)(u >> 16);
}
__device__ inline float bf2f(uint16_t b) { return __uint_as_float(((uint32_t)b) << 16); }

struct GemmArgs {
  const uint16_t *A;  // bf16
  int64_t a_rs, a_cs; // A(i,k) = A[i*a_rs + k*a_cs]
  const uint16_t *B;
  int64_t b_rs, b_cs; // B(k,j) = B[k*b_rs + j*b_cs]
  float *C;           // C(i,j) = C[i*c_rs + j]
  int64_t c_rs;
  int M, N, K;
  float *part;        // split-K partial products (ksplit x M x N), or null
  int ksplit;         // K is cut into ksplit chunks (blockIdx.z); 1 = no split
  int a_run, b_run;   // staging: 1 = runs along k, 2 = along i (A) / j (B), 0 = element by element
  int to_part;        // write slices to part whatever their number
};

// LDK pads a tile row to 80 bytes: rows stay 16-byte aligned for the staging
// stores and 8-byte aligned for the operand reads
constexpr int TM = 64, TN = 64, TK = 32, LDK = TK + 8;

// Stages the rows x TK tile X(r, k) = P[r*rs + k*cs], r in [r0, r0+64),
// k in [k0, k0+TK), into T[r - r0][k - k0]; entries outside r < rmax,
// k < kmax are zero.  Each of the 256 threads moves one run of 8 elements:
// run = 1 reads it along k (cs == 1), run = 2 along r (rs == 1), run = 0
// element by element (any strides).  A run entirely in bounds is one
// 16-byte load; the host picks run 1 or 2 only for 16-byte-aligned runs.
__device__ inline void stage_tile(uint16_t (*T)[LDK], const uint16_t *__restrict__ P, int64_t rs, int64_t cs,
                                  int run, int r0, int k0, int rmax, int kmax, int tid) {
  u32x4 v = {0u, 0u, 0u, 0u};   // the run, two elements per word, element e in bits 16(e&1) of word e>>1
  if (run == 2) {
    const int kk = tid >> 3, rr = (tid & 7) * 8;
    const int gk = k0 + kk, gr = r0 + rr;
    if (gk < kmax) {
      if (gr + 8 <= rmax) {
        v = *(const u32x4 *)(P + (int64_t)gk * cs + gr);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (gr + e < rmax) v[e >> 1] |= (uint32_t)P[(int64_t)gk * cs + gr + e] << (16 * (e & 1));
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) T[rr + e][kk] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
  } else {
    const int rr = tid >> 2, kk = (tid & 3) * 8;
    const int gr = r0 + rr, gk = k0 + kk;
    if (gr < rmax) {
      if (run == 1 && gk + 8 <= kmax) {
        v = *(const u32x4 *)(P + (int64_t)gr * rs + gk);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (gk + e < kmax) v[e >> 1] |= (uint32_t)P[(int64_t)gr * rs + (int64_t)(gk + e) * cs] << (16 * (e & 1));
      }
    }
    *(u32x4 *)&T[rr][kk] = v;
  }
}

// the 64 x 64 tile (by, bx) of slice bz
__device__ inline void gemm_tile(const GemmArgs &g, int bx, int by, int bz) {
  __shared__ __align__(16) uint16_t As[TM][LDK];   // As[i][k]
  __shared__ __align__(16) uint16_t Bs[TN][LDK];   // Bs[j][k]
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int i0 = by * TM, j0 = bx * TN;
  const int wi = (wv >> 1) * 32, wj = (wv & 1) * 32;
  floatx4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = floatx4{0.f, 0.f, 0.f, 0.f};
  // this workgroup's slice of K (all of it without a split); slices are
  // whole multiples of TK
  const int kc = ((g.K + g.ksplit - 1) / g.ksplit + TK - 1) / TK * TK;
  const int k_lo = bz * kc, k_hi = min(g.K, k_lo + kc);
  // A and B operands of v_mfma_f32_16x16x32_bf16: lane (r, g = lane / 16)
  // supplies row r of the tile at k = 8 g .. 8 g + 7; the result rows are
  // 4 g .. 4 g + 3 of column r
  const int r = lane & 15, q = (lane >> 4) * 4, qk = (lane >> 4) * 8;
  for (int k0 = k_lo; k0 < k_hi; k0 += TK) {
    __syncthreads();
    // B(k, j) = B[k*b_rs + j*b_cs] is staged as the tile X(j, k)
    stage_tile(As, g.A, g.a_rs, g.a_cs, g.a_run, i0, k0, g.M, k_hi, tid);
    stage_tile(Bs, g.B, g.b_cs, g.b_rs, g.b_run, j0, k0, g.N, k_hi, tid);
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < TK; ks += 32) {
      bf16x8 av[2], bv[2];
#pragma unroll
      for (int a = 0; a < 2; ++a) av[a] = *(const bf16x8 *)&As[wi + 16 * a + r][ks + qk];
#pragma unroll
      for (int b = 0; b < 2; ++b) bv[b] = *(const bf16x8 *)&Bs[wj + 16 * b + r][ks + qk];
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[a], bv[b], acc[a][b], 0, 0, 0);
    }
  }
  // epilogue: lane holds D[q+0..3][r] of each 16x16 tile
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        int gi = i0 + wi + 16 * a + q + t, gj = j0 + wj + 16 * b + r;
        if (gi < g.M && gj < g.N && (g.ksplit > 1 || g.to_part)) {
          g.part[((int64_t)bz * g.M + gi) * g.N + gj] = acc[a][b][t];
        } else if (gi < g.M && gj < g.N) {
          g.C[gi * g.c_rs + gj] = acc[a][b][t];
        }
      }
}

__global__ __launch_bounds__(256) void gemm_bf16_kernel(GemmArgs g) {
  gemm_tile(g, (int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z);
}

// split-K: C = sum of the partial products in slice order
__global__ void gemm_splitk_reduce_kernel(GemmArgs g) {
  const int64_t mn = (int64_t)g.M * g.N;
  for (int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; x < mn; x += (int64_t)gridDim.x * blockDim.x) {
    const int gi = (int)(x / g.N), gj = (int)(x - (int64_t)gi * g.N);
    float v = 0.f;
    // unrolled so that the slice loads are in flight together; the adds stay in slice order
#pragma unroll 8
    for (int z = 0; z < g.ksplit; ++z) v += g.part[(int64_t)z * mn + x];
    g.C[gi * g.c_rs + gj] = v;
  }
}

__global__ void to_bf16_kernel(const float *__restrict__ x, uint16_t *__restrict__ y, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    y[i] = f2bf(x[i]);
}

constexpr int kDin = 80, kHid = 256;

// Weights in operand order: an MFMA step of 32 k and a block of 16 columns is
// 64 lanes x 8 elements, so a lane's operand is one 16-byte read and a
// wavefront's is 1 KiB in a row.  Position of element (k, n) of a K x 16 nb
// right factor.
__host__ __device__ inline int packed_at(int k, int n, int nb) {
  return ((((k >> 5) * nb + (n >> 4)) * 64 + ((k >> 3) & 3) * 16 + (n & 15)) << 3) + (k & 7);
}
constexpr int kPack1 = 3 * 16 * 512, kPack = 8 * 16 * 512, kPack1t = 8 * 5 * 512;

__device__ inline void store_packed(uint16_t *f, uint16_t *t, int rows, int i, float w) {
  const int k = i / kHid, n = i - k * kHid;
  const uint16_t b = f2bf(w);
  f[packed_at(k, n, kHid / 16)] = b;
  t[packed_at(n, k, rows / 16)] = b;   // the transpose, for the gradient of the layer's input
}
__global__ void pack_kernel(const float *__restrict__ W, int rows, uint16_t *__restrict__ f, uint16_t *__restrict__ t) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < rows * kHid; i += gridDim.x * blockDim.x)
    store_packed(f, t, rows, i, W[i]);
}

struct RowArgs {
  const int *perm;      // rows of the training set (null: rows 0, 1, ...)
  const int *desc;      // (h1, h2 (0-based), spin class 0..2, degree 0..4) per row
  const float *fdesc;   // (eps1, eps2, log|c|) per row
  const float *tgt;
  const float *emb;
  const uint16_t *p1, *p2, *p3, *p3t, *p2t, *p1t;
  const float *b1, *b2, *b3, *w4, *b4;
  int n;
  float *y;
  // training: operands of the weight gradients, what the column sums need in
  // FP32, the output's errors and gradient per row, the gradient of the
  // embedding features
  uint16_t *Xb, *H1b, *H2b, *dZ3b, *dZ2b, *dZ1b;
  float *Z3, *dZ2, *dZ1, *err, *dy, *dX;
};

constexpr int LDA = kHid + 8;   // LDS row stride: the 16 rows of an operand read fall on different banks

// 16 RT rows per workgroup; wavefront w computes the column blocks w, w + 4,
// w + 8, w + 12 of every layer, which is the order the output sum wants
// (column c belongs to lane c % 64 of a row's 64-lane sum).
// Bound: in training a workgroup reads 600 KB of weights from L2, 4 us at 64
// bytes a cycle, against 1 us of products per 16 rows at half the matrix peak.
template <int RT, bool TRAIN>
__global__ __launch_bounds__(256, 2) void mlp_rows_kernel(RowArgs A) {
  constexpr int R = 16 * RT;
  __shared__ __align__(16) uint16_t act[R][LDA];
  __shared__ float sred[R][65];
  __shared__ float dys[R];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, j = lane & 15, q = lane >> 4;
  const int r0 = (int)blockIdx.x * R;
  // features, eight at a time: the embeddings of h1 and h2, then the numbers
  // and the one-hot spin class and degree, then padding
  for (int x = tid; x < R * 12; x += 256) {
    const int r = x / 12, f = x - r * 12, row = r0 + r;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 0.f;
    if (row < A.n && f < 10) {
      const int64_t i = A.perm ? A.perm[row] : row;
      const int4 d = reinterpret_cast<const int4 *>(A.desc)[i];
      if (f < 8) {
        const int h = f < 4 ? d.x : d.y;
        const float4 *e = reinterpret_cast<const float4 *>(A.emb + h * 32 + (f & 3) * 8);
        const float4 e0 = e[0], e1 = e[1];
        v[0] = e0.x; v[1] = e0.y; v[2] = e0.z; v[3] = e0.w;
        v[4] = e1.x; v[5] = e1.y; v[6] = e1.z; v[7] = e1.w;
      } else if (f == 8) {
#pragma unroll
        for (int e = 0; e < 3; ++e) v[e] = A.fdesc[3 * i + e];
#pragma unroll
        for (int e = 3; e < 6; ++e) v[e] = d.z == e - 3 ? 1.f : 0.f;
        v[6] = d.w == 0 ? 1.f : 0.f;
        v[7] = d.w == 1 ? 1.f : 0.f;
      } else {
#pragma unroll
        for (int e = 0; e < 3; ++e) v[e] = d.w == e + 2 ? 1.f : 0.f;
      }
    }
    u32x4 p;
#pragma unroll
    for (int e = 0; e < 4; ++e) p[e] = (uint32_t)f2bf(v[2 * e]) | ((uint32_t)f2bf(v[2 * e + 1]) << 16);
    *reinterpret_cast<u32x4 *>(&act[r][8 * f]) = p;
    if (TRAIN && row < A.n && f < 10) *reinterpret_cast<u32x4 *>(A.Xb + (int64_t)row * kDin + 8 * f) = p;
  }
  __syncthreads();

  floatx4 acc[RT][4];
  // The operands of a whole layer are requested at once, as soon as the
  // previous layer's products have read theirs: they arrive during its
  // epilogue.  Column blocks w, w + 4, ... (nc of them) of `steps` steps.
  bf16x8 bv[8][4];
  auto fetch = [&](const uint16_t *P, auto steps, auto nb, auto nc) {
    constexpr int S = decltype(steps)::value, NB = decltype(nb)::value, NC = decltype(nc)::value;
    const bf16x8 *p = reinterpret_cast<const bf16x8 *>(P) + w * 64 + lane;
#pragma unroll
    for (int ks = 0; ks < S; ++ks)
#pragma unroll
      for (int c = 0; c < NC; ++c) bv[ks][c] = p[(ks * NB + 4 * c) * 64];
  };
  // acc = act times the fetched operands
  auto product = [&](auto steps, auto nc) {
    constexpr int S = decltype(steps)::value, NC = decltype(nc)::value;
#pragma unroll
    for (int a = 0; a < RT; ++a)
#pragma unroll
      for (int c = 0; c < NC; ++c) acc[a][c] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < S; ++ks)
#pragma unroll
      for (int a = 0; a < RT; ++a) {
        const bf16x8 av = *reinterpret_cast<const bf16x8 *>(&act[16 * a + j][32 * ks + 8 * q]);
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv[ks][c], acc[a][c], 0, 0, 0);
      }
  };
  using I3 = std::integral_constant<int, 3>;
  using I5 = std::integral_constant<int, 5>;
  using I8 = std::integral_constant<int, 8>;
  using I16 = std::integral_constant<int, 16>;
  using I4 = std::integral_constant<int, 4>;
  using I1 = std::integral_constant<int, 1>;
  // rows of LDS to memory, 16 bytes a thread
  auto save = [&](uint16_t *to) {
    for (int x = tid; x < R * (kHid / 8); x += 256) {
      const int r = x / (kHid / 8), c = (x - r * (kHid / 8)) * 8;
      if (r0 + r < A.n) *reinterpret_cast<u32x4 *>(to + (int64_t)(r0 + r) * kHid + c) = *reinterpret_cast<const u32x4 *>(&act[r][c]);
    }
  };
  // act = relu(acc + bias); bit 16 a + 4 c + t of the returned mask: positive
  auto relu = [&](const float *bias, bool keep) {
    uint64_t m = 0;
    __syncthreads();
#pragma unroll
    for (int a = 0; a < RT; ++a)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int col = 16 * (w + 4 * c) + j;
        const float b = bias[col];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          float v = acc[a][c][t] + b;
          v = v > 0.f ? v : 0.f;
          if (v > 0.f) m |= 1ull << (16 * a + 4 * c + t);
          if (keep) acc[a][c][t] = v;
          else act[16 * a + 4 * q + t][col] = f2bf(v);
        }
      }
    __syncthreads();
    return m;
  };
  fetch(A.p1, I3{}, I16{}, I4{});
  product(I3{}, I4{});
  fetch(A.p2, I8{}, I16{}, I4{});
  const uint64_t m1 = relu(A.b1, false);
  if (TRAIN) save(A.H1b);
  product(I8{}, I4{});
  fetch(A.p3, I8{}, I16{}, I4{});
  const uint64_t m2 = relu(A.b2, false);
  if (TRAIN) save(A.H2b);
  product(I8{}, I4{});
  if (TRAIN) fetch(A.p3t, I8{}, I16{}, I4{});
  relu(A.b3, true);
  // output: 64 sums over columns l, l + 64, l + 128, l + 192 per row, then a fixed tree
  float w4c[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) w4c[c] = A.w4[16 * (w + 4 * c) + j];
#pragma unroll
  for (int a = 0; a < RT; ++a)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      float s = 0.f;
#pragma unroll
      for (int c = 0; c < 4; ++c) s = fmaf(acc[a][c][t], w4c[c], s);
      sred[16 * a + 4 * q + t][16 * w + j] = s;
    }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < R / 4; ++i) {
    const int r = w * (R / 4) + i, row = r0 + r;
    float s = sred[r][lane];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    s += *A.b4;
    if (lane == 0) {
      float d = 0.f;
      if (row < A.n) {
        A.y[row] = s;
        if (TRAIN) {
          const float e = s - A.tgt[A.perm ? A.perm[row] : row];
          d = 2.f * e / A.n;
          A.err[row] = e;
          A.dy[row] = d;
        }
      }
      if (TRAIN) dys[r] = d;
    }
  }
  if constexpr (TRAIN) {
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int col = 16 * (w + 4 * c) + j;
#pragma unroll
      for (int a = 0; a < RT; ++a)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int r = 16 * a + 4 * q + t;
          const float v = acc[a][c][t];
          if (r0 + r < A.n) A.Z3[(int64_t)(r0 + r) * kHid + col] = v;
          act[r][col] = f2bf(v > 0.f ? dys[r] * w4c[c] : 0.f);
        }
    }
    __syncthreads();
    save(A.dZ3b);
    // act = acc where the layer's output was positive
    auto masked = [&](uint64_t m, float *to) {
      __syncthreads();
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int col = 16 * (w + 4 * c) + j;
#pragma unroll
        for (int a = 0; a < RT; ++a)
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const int r = 16 * a + 4 * q + t;
            const float v = (m >> (16 * a + 4 * c + t)) & 1 ? acc[a][c][t] : 0.f;
            if (r0 + r < A.n) to[(int64_t)(r0 + r) * kHid + col] = v;
            act[r][col] = f2bf(v);
          }
      }
      __syncthreads();
    };
    product(I8{}, I4{});
    fetch(A.p2t, I8{}, I16{}, I4{});
    masked(m2, A.dZ2);
    save(A.dZ2b);
    product(I8{}, I4{});
    fetch(A.p1t, I8{}, I5{}, I1{});
    masked(m1, A.dZ1);
    save(A.dZ1b);
    // gradient of the 64 embedding features; the others are data
    product(I8{}, I1{});
    const int f = 16 * w + j;
#pragma unroll
    for (int a = 0; a < RT; ++a)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = 16 * a + 4 * q + t;
        if (r0 + r < A.n) A.dX[(int64_t)(r0 + r) * 64 + f] = acc[a][0][t];
      }
  }
}

// The sums over the batch, in one launch: the slices of the three weight
// gradients, the column sums (gradients of w4, b3, b2, b1) by row chunks, the
// embedding gradient and the output bias.  Every sum but the embeddings' has a fixed order: a small change of a gradient
// that nearly cancels changes the sign of its first Adam step.
struct GradArgs {
  GemmArgs g[3];
  int blocks[3];              // of each product: tiles x slices, slice-major
  const float *Z3, *dZ2, *dZ1, *dy, *w4;
  int n, chunk, np;           // rows per chunk, chunks
  float *part;                // [4][np][256]
  float *gb4;
  const float *dX;            // [n][64]
  const int *perm, *desc;
  float *demb;
  int n_orb, ne;              // ne: chunks of kEmbRows rows
};
constexpr int kEmbRows = 256, kMaxOrb = 256;
__global__ __launch_bounds__(256) void grad_kernel(GradArgs S) {
  __shared__ float red[256];
  __shared__ double es[kMaxOrb * 8];
  int t = (int)blockIdx.x;
#pragma unroll
  for (int w = 0; w < 3; ++w) {
    if (t < S.blocks[w]) {
      const GemmArgs &g = S.g[w];
      const int nbx = (g.N + TN - 1) / TN, nby = (g.M + TM - 1) / TM, z = t / (nbx * nby);
      t -= z * nbx * nby;
      gemm_tile(g, t % nbx, t / nbx, z);
      return;
    }
    t -= S.blocks[w];
  }
  const int tid = threadIdx.x;
  if (t < 16 * S.np) {
    // sum `which` of 64 columns over a chunk: four row phases per column, combined in phase order
    const int which = t / (4 * S.np), u = t - which * 4 * S.np, p = u >> 2, k = (u & 3) * 64 + (tid & 63), g = tid >> 6;
    const int r0 = p * S.chunk, r1 = min(S.n, r0 + S.chunk);
    const float w4 = S.w4[k];
    float s = 0.f;
    if (which == 0) {
#pragma unroll 4
      for (int i = r0 + g; i < r1; i += 4) s = fmaf(S.Z3[(int64_t)i * kHid + k], S.dy[i], s);
    } else if (which == 1) {
#pragma unroll 4
      for (int i = r0 + g; i < r1; i += 4) {
#pragma clang fp contract(off)
        const float d = S.dy[i] * w4;
        s += S.Z3[(int64_t)i * kHid + k] > 0.f ? d : 0.f;
      }
    } else {
      const float *A = which == 2 ? S.dZ2 : S.dZ1;
#pragma unroll 4
      for (int i = r0 + g; i < r1; i += 4) s += A[(int64_t)i * kHid + k];
    }
    red[tid] = s;
    __syncthreads();
    if (g == 0) S.part[((int64_t)which * S.np + p) * kHid + k] = (red[tid] + red[64 + tid]) + (red[128 + tid] + red[192 + tid]);
    return;
  }
  t -= 16 * S.np;
  if (t < 4 * S.ne) {
    // embedding gradient of 8 of the 32 components over a chunk of rows: both
    // holes' features of a row go to its orbitals' sums, in FP64 (ds_add_f64 is
    // 17 times as fast as ds_add_f32), and one atomic per component and orbital
    // leaves the workgroup (one per row and feature took 21 us at 4096 rows)
    const int g = t & 3, r0 = (t >> 2) * kEmbRows, r1 = min(S.n, r0 + kEmbRows);
    for (int x = tid; x < S.n_orb * 8; x += 256) es[x] = 0.0;
    __syncthreads();
    for (int x = tid; x < (r1 - r0) * 16; x += 256) {
      const int row = r0 + (x >> 4), which = (x >> 3) & 1, f = x & 7;
      const int64_t i = S.perm ? S.perm[row] : row;
      const int h = S.desc[4 * i + which];
      unsafeAtomicAdd(&es[h * 8 + f], (double)S.dX[(int64_t)row * 64 + which * 32 + g * 8 + f]);
    }
    __syncthreads();
    for (int x = tid; x < S.n_orb * 8; x += 256) {
      const float v = (float)es[x];
      if (v != 0.f) atomicAdd(&S.demb[(x >> 3) * 32 + g * 8 + (x & 7)], v);
    }
    return;
  }
  float s = 0.f;
  for (int i = tid; i < S.n; i += 256) s += S.dy[i];
  red[tid] = s;
  __syncthreads();
  if (tid == 0) {
    float b = 0.f;
    for (int i = 0; i < 256; ++i) b += red[i];
    *S.gb4 = b;
  }
}

// The step after a batch: sums the weight gradients' slices and the column
// sums' chunks, takes the embedding gradient, and (lr > 0) makes the Adam step
// m = b1 m + (1 - b1) g, v = b2 v + (1 - b2) g^2,
// p -= lr (m / c1) / (sqrt(v / c2) + eps), c1, c2 the bias corrections
// 1 - b1^t, 1 - b2^t; the packed bf16 weights are refreshed.
// Blocks [0, nelem) take 256 elements of W1, W2, W3, emb, the next a column
// (w4, b3, b2, b1, b4) per wavefront: lane l adds chunks l, l + 64, ..., then
// a fixed tree; the last one the loss.
struct Param {
  float *p, *g, *m, *v;
};
struct AdamArgs {
  Param W[3], emb, col[4], b4;   // col: w4, b3, b2, b1
  const float *wpart[3];
  int ks[3], wrows[3];
  uint16_t *pf[3], *pt[3];
  float *demb;          // accumulated by atomics; taken and cleared here
  int n_emb, nelem;
  const float *part, *err;
  int np, n;
  float *loss_out;
  float lr, b1, b2, eps, c1, c2;
};

__device__ inline float adam(const AdamArgs &A, const Param &P, int i, float g) {
  P.g[i] = g;
  float p = P.p[i];
  if (A.lr > 0.f) {
    const float mi = fmaf(1.f - A.b1, g, A.b1 * P.m[i]);
    const float vi = fmaf(g, (1.f - A.b2) * g, A.b2 * P.v[i]);
    P.m[i] = mi;
    P.v[i] = vi;
    p -= A.lr * (mi / A.c1) / (sqrtf(vi / A.c2) + A.eps);
    P.p[i] = p;
  }
  return p;
}

__global__ __launch_bounds__(256) void adam_kernel(AdamArgs A) {
  if ((int)blockIdx.x < A.nelem) {
    int i = (int)blockIdx.x * 256 + (int)threadIdx.x;
#pragma unroll
    for (int w = 0; w < 3; ++w) {
      const int cnt = A.wrows[w] * kHid;
      if (i < cnt) {
        float g = 0.f;
#pragma unroll 8
        for (int z = 0; z < A.ks[w]; ++z) g += A.wpart[w][(int64_t)z * cnt + i];
        const float p = adam(A, A.W[w], i, g);
        if (A.lr > 0.f) store_packed(A.pf[w], A.pt[w], A.wrows[w], i, p);
        return;
      }
      i -= cnt;
    }
    if (i < A.n_emb) {
      const float g = A.demb[i];
      A.demb[i] = 0.f;
      adam(A, A.emb, i, g);
    }
    return;
  }
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int k = ((int)blockIdx.x - A.nelem) * 4 + wv;
  if ((int)blockIdx.x == (int)gridDim.x - 1) {
    __shared__ float red[4];
    float s = 0.f;
    for (int i = threadIdx.x; i < A.n; i += 256) s = fmaf(A.err[i], A.err[i], s);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) red[wv] = s;
    __syncthreads();
    if (threadIdx.x == 0) *A.loss_out = ((red[0] + red[1]) + (red[2] + red[3])) / (float)A.n;
    return;
  }
  if (k > 4 * kHid) return;
  float s = 0.f;
  if (k < 4 * kHid) {
    const float *src = A.part + (int64_t)(k / kHid) * A.np * kHid + k % kHid;
    for (int z = lane; z < A.np; z += 64) s += src[(int64_t)z * kHid];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  } else {
    s = A.b4.g[0];
  }
  if (lane == 0) adam(A, k < 4 * kHid ? A.col[k / kHid] : A.b4, k < 4 * kHid ? k % kHid : 0, s);
}

}  // namespace

// ---------------------------------------------------------------------------
// Scratch of the allocation-free prediction (qpx_mlp_predict_static): the
// staged descriptors and the predictions of at most kStaticRows blocks, in
// one file-scope device array.  Each GPU the library runs on holds its own
// copy until the process ends; its device address is looked up once per
// device (scratch_address) and only that address is handed to kernels and
// copies.
namespace {
constexpr int kStaticRows = 2048;
constexpr size_t al256(size_t x) { return (x + 255) & ~size_t(255); }
constexpr size_t kScratchBytes = al256(sizeof(int) * 4 * kStaticRows) + al256(sizeof(float) * 3 * kStaticRows) +
                                 al256(sizeof(float) * kStaticRows);
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_dev[kMaxDevices] = {};

// device address of this device's scratch (the current device must be
// `device`); looked up once per device
void *scratch_address(int device) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  QPX_REQUIRE(device >= 0 && device < kMaxDevices, "device index out of range");
  if (!g_scratch_dev[device]) {
    void *p = nullptr;
    QPX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    QPX_REQUIRE(p != nullptr, "no device address for the prediction scratch");
    g_scratch_dev[device] = p;
  }
  return g_scratch_dev[device];
}
}  // namespace

// ---------------------------------------------------------------------------
struct qpx_mlp {
  int din = 80, hid = 256, n_orb = 0;
  hipStream_t st = nullptr;
  int device = 0;
  // parameters (fp32 master; layer l: W (in x out) row-major) and the weights
  // packed as right factors, straight and transposed
  DBuf<float> W1, W2, W3, b1, b2, b3, w4, emb;
  DBuf<uint16_t> p1, p2, p3, p1t, p2t, p3t;
  DBuf<float> gW1, gW2, gW3, gb1, gb2, gb3, gw4, gemb, gb4;
  DBuf<float> demb;                     // embedding gradient being accumulated; zero between steps
  DBuf<float> ws1, ws2, ws3;            // slices of the weight gradients
  DBuf<float> mW1, mW2, mW3, mb1, mb2, mb3, mw4, memb, vW1, vW2, vW3, vb1, vb2, vb3, vw4, vemb;
  DBuf<float> b4, mb4, vb4;   // the output bias and its Adam moments (one element each, on the device)
  int step = 0;
  int cap = 0, tcap = 0;      // rows held: descriptors and predictions; training operands
  DBuf<float> y, part, Z3, dZ2, dZ1, dX, rerr, dy, lossp;
  DBuf<uint16_t> Xb, H1b, H2b, dZ3b, dZ2b, dZ1b;
  DBuf<int> desc;
  DBuf<float> fdesc, tgt;
  void *scratch = nullptr;   // device address of this device's prediction scratch
  std::string err;
};

namespace {

// C = A B by the weight gradients' tile, in every operand layout the tile can
// stage; the network itself launches the tile from grad_kernel, with runs along
// i and j and slices that adam_kernel sums.  Called by the checks alone
// (qpx_mlp_gemm_check, qpx_debug_mlp_gemm).  With a workspace, a product whose
// tile grid leaves most CUs idle and whose K is long is cut along K across
// workgroups and reduced in slice order.
void gemm(hipStream_t st, const uint16_t *A, int64_t ars, int64_t acs, const uint16_t *B, int64_t brs, int64_t bcs,
          float *C, int64_t crs, int M, int N, int K, DBuf<float> *ws = nullptr) {
  // 16-byte runs need a 16-byte-aligned base and a multiple-of-8 stride
  // across runs
  const auto run_of = [](const uint16_t *P, int64_t rs, int64_t cs) {
    if (((uintptr_t)P & 15) != 0) return 0;
    if (cs == 1 && rs % 8 == 0) return 1;
    if (rs == 1 && cs % 8 == 0) return 2;
    return 0;
  };
  GemmArgs g{A, ars, acs, B, brs, bcs, C, crs, M, N, K, nullptr, 1,
             run_of(A, ars, acs), run_of(B, bcs, brs), 0};
  dim3 grid((N + TN - 1) / TN, (M + TM - 1) / TM);
  const int tiles = (int)(grid.x * grid.y);
  constexpr int kGrain = 16;   // split-K sizing unit (slices are then rounded up to TK)
  if (ws && tiles < 128 && K >= 8 * kGrain) {
    g.ksplit = std::max(1, std::min({256 / tiles, K / (4 * kGrain), 32}));
    if (g.ksplit > 1 && ws->n >= (size_t)g.ksplit * M * N) {
      g.part = ws->p;
      grid.z = g.ksplit;
    } else {
      g.ksplit = 1;
    }
  }
  hipLaunchKernelGGL(gemm_bf16_kernel, grid, dim3(256), 0, st, g);
  QPX_HIP(hipGetLastError());
  if (g.ksplit > 1) {
    const int64_t mn = (int64_t)M * N;
    hipLaunchKernelGGL(gemm_splitk_reduce_kernel, dim3((unsigned)std::min<int64_t>((mn + 255) / 256, 4096)), dim3(256),
                       0, st, g);
    QPX_HIP(hipGetLastError());
  }
}

constexpr int kSlices = 32;      // most slices of a weight gradient
constexpr int kChunks = 64;      // most row chunks of a column sum

void ensure(qpx_mlp *m, int n) {
  if (n <= m->cap) return;
  m->cap = 0;   // should one of the allocations fail
  m->desc.alloc((size_t)4 * n);
  m->fdesc.alloc((size_t)3 * n);
  m->tgt.alloc(n);
  m->y.alloc(n);
  m->cap = n;
}

void ensure_train(qpx_mlp *m, int n) {
  ensure(m, n);
  if (n <= m->tcap) return;
  m->tcap = 0;
  const int Hd = m->hid;
  m->Xb.alloc((size_t)n * m->din);
  for (DBuf<uint16_t> *b : {&m->H1b, &m->H2b, &m->dZ1b, &m->dZ2b, &m->dZ3b}) b->alloc((size_t)n * Hd);
  for (DBuf<float> *b : {&m->Z3, &m->dZ2, &m->dZ1}) b->alloc((size_t)n * Hd);
  m->dX.alloc((size_t)n * 64);
  m->rerr.alloc(n);
  m->dy.alloc(n);
  m->part.alloc((size_t)4 * kChunks * Hd);
  m->lossp.alloc(1);
  m->ws1.alloc((size_t)kSlices * m->din * Hd);
  m->ws2.alloc((size_t)kSlices * Hd * Hd);
  m->ws3.alloc((size_t)kSlices * Hd * Hd);
  m->tcap = n;
}

// the rows of the given arrays (rows perm[0..n) of them with perm)
RowArgs row_args(qpx_mlp *m, int n, const int *perm, const int *desc, const float *fdesc, const float *tgt, float *y) {
  RowArgs A{};
  A.perm = perm; A.desc = desc; A.fdesc = fdesc; A.tgt = tgt; A.emb = m->emb.p;
  A.p1 = m->p1.p; A.p2 = m->p2.p; A.p3 = m->p3.p; A.p1t = m->p1t.p; A.p2t = m->p2t.p; A.p3t = m->p3t.p;
  A.b1 = m->b1.p; A.b2 = m->b2.p; A.b3 = m->b3.p; A.w4 = m->w4.p; A.b4 = m->b4.p;
  A.n = n; A.y = y;
  A.Xb = m->Xb.p; A.H1b = m->H1b.p; A.H2b = m->H2b.p; A.dZ3b = m->dZ3b.p; A.dZ2b = m->dZ2b.p; A.dZ1b = m->dZ1b.p;
  A.Z3 = m->Z3.p; A.dZ2 = m->dZ2.p; A.dZ1 = m->dZ1.p; A.err = m->rerr.p; A.dy = m->dy.p; A.dX = m->dX.p;
  return A;
}

// predictions of n rows: 64 rows per workgroup where that still fills the
// chip twice over (half the weight traffic of 32 or 16), fewer below
void predict_rows(qpx_mlp *m, int n, const int *desc, const float *fdesc, float *y) {
  const RowArgs A = row_args(m, n, nullptr, desc, fdesc, nullptr, y);
  if (n >= 64 * 512) hipLaunchKernelGGL((mlp_rows_kernel<4, false>), dim3((n + 63) / 64), dim3(256), 0, m->st, A);
  else if (n >= 32 * 256) hipLaunchKernelGGL((mlp_rows_kernel<2, false>), dim3((n + 31) / 32), dim3(256), 0, m->st, A);
  else hipLaunchKernelGGL((mlp_rows_kernel<1, false>), dim3((n + 15) / 16), dim3(256), 0, m->st, A);
  QPX_HIP(hipGetLastError());
}

// One Adam step on n rows, enqueued on the network's stream without waiting
// for it; the batch's mean squared error goes to *loss_out (device memory).
void train_step_async(qpx_mlp *m, int n, const int *perm, const int *desc, const float *fdesc, const float *tgt,
                      float lr, float *loss_out) {
  hipStream_t st = m->st;
  const int D = m->din, Hd = m->hid;
  // 16 rows per workgroup until every CU has one, 32 above
  const RowArgs R = row_args(m, n, perm, desc, fdesc, tgt, m->y.p);
  if (n <= 16 * 256) hipLaunchKernelGGL((mlp_rows_kernel<1, true>), dim3((n + 15) / 16), dim3(256), 0, st, R);
  else hipLaunchKernelGGL((mlp_rows_kernel<2, true>), dim3((n + 31) / 32), dim3(256), 0, st, R);
  // weight gradients dW1 = X^T dZ1, dW2 = H1^T dZ2, dW3 = H2^T dZ3 over the
  // batch, in slices of at least 64 rows, up to 256 workgroups a product;
  // column sums in chunks of at least 64 rows, up to kChunks of them
  GradArgs S{};
  const uint16_t *a[3] = {m->Xb.p, m->H1b.p, m->H2b.p}, *b[3] = {m->dZ1b.p, m->dZ2b.p, m->dZ3b.p};
  float *ws[3] = {m->ws1.p, m->ws2.p, m->ws3.p};
  const int rows[3] = {D, Hd, Hd};
  int ks[3], blocks = 0;
  for (int w = 0; w < 3; ++w) {
    const int tiles = ((rows[w] + TM - 1) / TM) * (Hd / TN);
    ks[w] = n >= 128 ? std::max(1, std::min({256 / tiles, n / 64, kSlices})) : 1;
    // one slice, too, goes through the slices' buffer
    S.g[w] = GemmArgs{a[w], 1, rows[w], b[w], Hd, 1, nullptr, Hd, rows[w], Hd, n, ws[w],
                      ks[w], 2, 2, 1};
    S.blocks[w] = tiles * ks[w];
    blocks += S.blocks[w];
  }
  S.Z3 = m->Z3.p; S.dZ2 = m->dZ2.p; S.dZ1 = m->dZ1.p; S.dy = m->dy.p; S.w4 = m->w4.p;
  S.n = n;
  S.np = std::max(1, std::min(kChunks, (n + 63) / 64));
  S.chunk = (n + S.np - 1) / S.np;
  S.np = (n + S.chunk - 1) / S.chunk;
  S.part = m->part.p;
  S.gb4 = m->gb4.p;
  S.dX = m->dX.p; S.perm = perm; S.desc = desc; S.demb = m->demb.p;
  S.n_orb = m->n_orb;
  S.ne = (n + kEmbRows - 1) / kEmbRows;
  hipLaunchKernelGGL(grad_kernel, dim3(blocks + 16 * S.np + 4 * S.ne + 1), dim3(256), 0, st, S);
  AdamArgs P{};
  auto par = [](DBuf<float> &p, DBuf<float> &g, DBuf<float> &mm, DBuf<float> &v) { return Param{p.p, g.p, mm.p, v.p}; };
  P.W[0] = par(m->W1, m->gW1, m->mW1, m->vW1);
  P.W[1] = par(m->W2, m->gW2, m->mW2, m->vW2);
  P.W[2] = par(m->W3, m->gW3, m->mW3, m->vW3);
  P.emb = par(m->emb, m->gemb, m->memb, m->vemb);
  P.col[0] = par(m->w4, m->gw4, m->mw4, m->vw4);
  P.col[1] = par(m->b3, m->gb3, m->mb3, m->vb3);
  P.col[2] = par(m->b2, m->gb2, m->mb2, m->vb2);
  P.col[3] = par(m->b1, m->gb1, m->mb1, m->vb1);
  P.b4 = par(m->b4, m->gb4, m->mb4, m->vb4);
  uint16_t *pf[3] = {m->p1.p, m->p2.p, m->p3.p}, *pt[3] = {m->p1t.p, m->p2t.p, m->p3t.p};
  int elems = 0;
  for (int w = 0; w < 3; ++w) {
    P.wpart[w] = ws[w];
    P.wrows[w] = rows[w];
    P.pf[w] = pf[w];
    P.pt[w] = pt[w];
    elems += rows[w] * Hd;
  }
  for (int w = 0; w < 3; ++w) P.ks[w] = ks[w];
  P.demb = m->demb.p;
  P.n_emb = (int)m->emb.n;
  P.nelem = (elems + P.n_emb + 255) / 256;
  P.part = m->part.p;
  P.err = m->rerr.p;
  P.np = S.np;
  P.n = n;
  P.loss_out = loss_out;
  P.lr = lr;
  if (lr > 0.f) {
    m->step++;
    P.b1 = 0.9f; P.b2 = 0.999f; P.eps = 1e-8f;
    P.c1 = 1.f - std::pow(P.b1, (float)m->step);
    P.c2 = 1.f - std::pow(P.b2, (float)m->step);
  }
  hipLaunchKernelGGL(adam_kernel, dim3(P.nelem + (4 * Hd + 1 + 3) / 4 + 1), dim3(256), 0, st, P);
  QPX_HIP(hipGetLastError());
}

template <typename F>
int mguard(qpx_mlp *m, F &&f) {
  if (!m) return 1;
  try {
    f();
    return 0;
  } catch (const qpx::Error &e) {
    m->err = e.what();
    return e.code;
  } catch (const std::exception &e) {
    m->err = e.what();
    return 3;
  }
}

// The descriptors index the embedding table and the one-hot slots: a row
// outside {h1, h2 in [0, n_orb), spin class in 0..2, degree in 0..4} would
// make the feature and embedding-gradient kernels read or write out of
// bounds, so it is rejected on the host before anything is uploaded.
void check_desc(const qpx_mlp *m, int64_t n, const int *desc) {
  QPX_REQUIRE(desc, "null descriptor array");
  const unsigned lim[4] = {(unsigned)m->n_orb, (unsigned)m->n_orb, 3u, 5u};   // negative values wrap above them
  unsigned bad = 0;
  for (int64_t i = 0; i < 4 * n; ++i) bad |= (unsigned)desc[i] >= lim[i & 3];   // no early exit: this vectorises
  if (!bad) return;
  for (int64_t i = 0; i < n; ++i) {
    const int *d = desc + 4 * i;
    if ((unsigned)d[0] >= lim[0] || (unsigned)d[1] >= lim[1] || (unsigned)d[2] >= lim[2] || (unsigned)d[3] >= lim[3]) {
      char buf[160];
      std::snprintf(buf, sizeof buf, "descriptor row %lld = (%d, %d, %d, %d) out of range (n_orb = %d)",
                    (long long)i, d[0], d[1], d[2], d[3], m->n_orb);
      QPX_REQUIRE(false, buf);
    }
  }
}

uint64_t sm64(uint64_t &s) {
  uint64_t z = (s += 0x9E3779B97F4A7C15ULL);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return z ^ (z >> 31);
}

}  // namespace

// ---------------------------------------------------------------------------
// C-ABI (no counterpart in the reference)
// ---------------------------------------------------------------------------
extern "C" int qpx_mlp_create(int device, int n_orb, uint64_t seed, qpx_mlp **out) {
  if (!out) return 1;
  qpx_mlp *m = new qpx_mlp();
  int rc = mguard(m, [&] {
    QPX_REQUIRE(n_orb > 0 && n_orb <= kMaxOrb, "n_orb must be in 1..256");
    QPX_HIP(hipSetDevice(device));
    m->device = device;
    m->n_orb = n_orb;
    QPX_REQUIRE(m->din == kDin && m->hid == kHid, "network shape differs from the prediction scratch layout");
    m->scratch = scratch_address(device);
    QPX_HIP(hipStreamCreateWithFlags(&m->st, hipStreamNonBlocking));
    const int D = m->din, Hd = m->hid;
    uint64_t s = seed;
    auto init = [&](DBuf<float> &p, size_t n, float scale) {
      std::vector<float> h(n);
      for (auto &x : h) {
        double u1 = 1.0 - (double)(sm64(s) >> 11) / 9007199254740992.0, u2 = (double)(sm64(s) >> 11) / 9007199254740992.0;
        x = (float)(scale * std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2));
      }
      p.upload(h, m->st);
    };
    init(m->W1, (size_t)D * Hd, std::sqrt(2.0f / 75.f));
    init(m->W2, (size_t)Hd * Hd, std::sqrt(2.0f / Hd));
    init(m->W3, (size_t)Hd * Hd, std::sqrt(2.0f / Hd));
    init(m->w4, Hd, std::sqrt(1.0f / Hd));
    init(m->emb, (size_t)n_orb * 32, 0.3f);
    std::vector<float> z(Hd, 0.f);
    m->b1.upload(z, m->st);
    m->b2.upload(z, m->st);
    m->b3.upload(z, m->st);
    m->p1.alloc(kPack1); m->p2.alloc(kPack); m->p3.alloc(kPack);
    m->p1t.alloc(kPack1t); m->p2t.alloc(kPack); m->p3t.alloc(kPack);
    QPX_HIP(hipMemsetAsync(m->p1.p, 0, sizeof(uint16_t) * kPack1, m->st));   // features 80..95 of the last step
    hipLaunchKernelGGL(pack_kernel, dim3(64), dim3(256), 0, m->st, m->W1.p, D, m->p1.p, m->p1t.p);
    hipLaunchKernelGGL(pack_kernel, dim3(64), dim3(256), 0, m->st, m->W2.p, Hd, m->p2.p, m->p2t.p);
    hipLaunchKernelGGL(pack_kernel, dim3(64), dim3(256), 0, m->st, m->W3.p, Hd, m->p3.p, m->p3t.p);
    auto zero = [&](DBuf<float> &p, size_t n) {
      p.alloc(n);
      QPX_HIP(hipMemsetAsync(p.p, 0, sizeof(float) * n, m->st));
    };
    zero(m->gW1, (size_t)D * Hd); zero(m->gW2, (size_t)Hd * Hd); zero(m->gW3, (size_t)Hd * Hd);
    zero(m->gb1, Hd); zero(m->gb2, Hd); zero(m->gb3, Hd); zero(m->gw4, Hd); zero(m->gb4, 1);
    zero(m->b4, 1); zero(m->mb4, 1); zero(m->vb4, 1);
    zero(m->gemb, (size_t)n_orb * 32); zero(m->demb, (size_t)n_orb * 32);
    zero(m->mW1, (size_t)D * Hd); zero(m->mW2, (size_t)Hd * Hd); zero(m->mW3, (size_t)Hd * Hd);
    zero(m->vW1, (size_t)D * Hd); zero(m->vW2, (size_t)Hd * Hd); zero(m->vW3, (size_t)Hd * Hd);
    zero(m->mb1, Hd); zero(m->mb2, Hd); zero(m->mb3, Hd); zero(m->mw4, Hd);
    zero(m->vb1, Hd); zero(m->vb2, Hd); zero(m->vb3, Hd); zero(m->vw4, Hd);
    zero(m->memb, (size_t)n_orb * 32); zero(m->vemb, (size_t)n_orb * 32);
    QPX_HIP(hipGetLastError());
    QPX_HIP(hipStreamSynchronize(m->st));
  });
  if (rc) {
    delete m;
    return rc;
  }
  *out = m;
  return 0;
}

extern "C" int qpx_mlp_destroy(qpx_mlp *m) {
  if (!m) return 0;
  (void)hipSetDevice(m->device);
  if (m->st) {
    (void)hipStreamSynchronize(m->st);
    (void)hipStreamDestroy(m->st);
  }
  delete m;
  return 0;
}

extern "C" int qpx_mlp_last_error(qpx_mlp *m, char *buf, int len) {
  if (!m || !buf || len <= 0) return 1;
  std::strncpy(buf, m->err.c_str(), (size_t)len - 1);
  buf[len - 1] = 0;
  return 0;
}

// One Adam step on a batch.  desc (n x 4 int32: h1, h2 0-based, spin class,
// degree), fdesc (n x 3 float: eps1, eps2, log|c|), target (n) = label.
// lr = 0 computes loss and gradients only.  *loss = mean squared error.
extern "C" int qpx_mlp_train_step(qpx_mlp *m, int n, const int *desc, const float *fdesc, const float *target,
                                  float lr, float *loss) {
  return mguard(m, [&] {
    QPX_HIP(hipSetDevice(m->device));
    QPX_REQUIRE(n > 0, "empty batch");
    QPX_REQUIRE(fdesc && target, "null argument");
    check_desc(m, n, desc);
    ensure_train(m, n);
    QPX_HIP(hipMemcpyAsync(m->desc.p, desc, sizeof(int) * 4 * n, hipMemcpyHostToDevice, m->st));
    QPX_HIP(hipMemcpyAsync(m->fdesc.p, fdesc, sizeof(float) * 3 * n, hipMemcpyHostToDevice, m->st));
    QPX_HIP(hipMemcpyAsync(m->tgt.p, target, sizeof(float) * n, hipMemcpyHostToDevice, m->st));
    train_step_async(m, n, nullptr, m->desc.p, m->fdesc.p, m->tgt.p, lr, m->lossp.p);
    float l = 0.f;
    QPX_HIP(hipMemcpyAsync(&l, m->lossp.p, sizeof(float), hipMemcpyDeviceToHost, m->st));
    QPX_HIP(hipStreamSynchronize(m->st));
    if (loss) *loss = l;
  });
}

extern "C" int qpx_mlp_train_epochs(qpx_mlp *m, int n, const int *desc, const float *fdesc, const float *target,
                                    float lr, int epochs, int batch, uint64_t seed, float *epoch_loss) {
  return mguard(m, [&] {
    QPX_HIP(hipSetDevice(m->device));
    QPX_REQUIRE(n > 0 && batch >= 1 && batch <= n && epochs >= 1, "need 1 <= batch <= n and epochs >= 1");
    QPX_REQUIRE(desc && fdesc && target && epoch_loss, "null argument");
    check_desc(m, n, desc);
    ensure_train(m, batch);
    DBuf<int> desc_all, perm_d;
    DBuf<float> fdesc_all, tgt_all;
    desc_all.upload(desc, (size_t)4 * n, m->st);
    fdesc_all.upload(fdesc, (size_t)3 * n, m->st);
    tgt_all.upload(target, (size_t)n, m->st);
    perm_d.alloc(n);
    const int steps = n / batch;
    DBuf<float> step_loss;   // one loss per step of an epoch, read back once per epoch
    step_loss.alloc(steps);
    std::vector<float> sl(steps);
    std::vector<int> perm(n);
    uint64_t s = seed;
    for (int ep = 0; ep < epochs; ++ep) {
      for (int i = 0; i < n; ++i) perm[i] = i;
      for (int i = n - 1; i > 0; --i) {   // Fisher-Yates
        const int j = (int)(sm64(s) % (uint64_t)(i + 1));
        std::swap(perm[i], perm[j]);
      }
      QPX_HIP(hipMemcpyAsync(perm_d.p, perm.data(), sizeof(int) * n, hipMemcpyHostToDevice, m->st));
      for (int q = 0; q < steps; ++q) {
        train_step_async(m, batch, perm_d.p + (size_t)q * batch, desc_all.p, fdesc_all.p, tgt_all.p, lr,
                         step_loss.p + q);
      }
      QPX_HIP(hipMemcpyAsync(sl.data(), step_loss.p, sizeof(float) * steps, hipMemcpyDeviceToHost, m->st));
      QPX_HIP(hipStreamSynchronize(m->st));
      double lsum = 0.0;
      for (float x : sl) lsum += x;
      epoch_loss[ep] = (float)(lsum / steps);
    }
  });
}

// Predictions for n blocks (processed in chunks of up to 65536).
extern "C" int qpx_mlp_predict(qpx_mlp *m, int n, const int *desc, const float *fdesc, float *out) {
  return mguard(m, [&] {
    QPX_HIP(hipSetDevice(m->device));
    QPX_REQUIRE(n >= 0 && (n == 0 || (fdesc && out)), "bad prediction arguments");
    check_desc(m, n, desc);
    const int chunk = 65536;
    for (int i0 = 0; i0 < n; i0 += chunk) {
      int c = std::min(chunk, n - i0);
      ensure(m, c);
      QPX_HIP(hipMemcpyAsync(m->desc.p, desc + 4 * (size_t)i0, sizeof(int) * 4 * c, hipMemcpyHostToDevice, m->st));
      QPX_HIP(hipMemcpyAsync(m->fdesc.p, fdesc + 3 * (size_t)i0, sizeof(float) * 3 * c, hipMemcpyHostToDevice, m->st));
      predict_rows(m, c, m->desc.p, m->fdesc.p, m->y.p);
      QPX_HIP(hipMemcpyAsync(out + i0, m->y.p, sizeof(float) * c, hipMemcpyDeviceToHost, m->st));
    }
    QPX_HIP(hipStreamSynchronize(m->st));
  });
}

// Prediction without any allocation: the descriptors and the predictions are
// staged in this device's file-scope scratch (kStaticRows rows at most; the
// activations live in LDS).  Every call on a GPU shares that scratch: calls that overlap on one
// GPU (from several threads or networks) race.
extern "C" int qpx_mlp_predict_static(qpx_mlp *m, int n, const int *desc, const float *fdesc, float *out) {
  return mguard(m, [&] {
    QPX_REQUIRE(n >= 1 && n <= kStaticRows, "n must be in 1..2048 (the rows the static scratch holds)");
    QPX_REQUIRE(fdesc && out, "null argument");
    check_desc(m, n, desc);
    QPX_HIP(hipSetDevice(m->device));
    QPX_REQUIRE(m->scratch, "no prediction scratch on this device");
    unsigned char *base = static_cast<unsigned char *>(m->scratch);
    int *dd = reinterpret_cast<int *>(base);
    float *df = reinterpret_cast<float *>(base + al256(sizeof(int) * 4 * kStaticRows));
    float *dy = reinterpret_cast<float *>(base + al256(sizeof(int) * 4 * kStaticRows) + al256(sizeof(float) * 3 * kStaticRows));
    QPX_HIP(hipMemcpyAsync(dd, desc, sizeof(int) * 4 * n, hipMemcpyHostToDevice, m->st));
    QPX_HIP(hipMemcpyAsync(df, fdesc, sizeof(float) * 3 * n, hipMemcpyHostToDevice, m->st));
    predict_rows(m, n, dd, df, dy);
    QPX_HIP(hipMemcpyAsync(out, dy, sizeof(float) * n, hipMemcpyDeviceToHost, m->st));
    QPX_HIP(hipStreamSynchronize(m->st));
  });
}

// Parameter exchange (fp32), for checkpoints and the gradient checks:
// which = 0 W1 (80x256), 1 W2, 2 W3 (256x256), 3 b1, 4 b2, 5 b3, 6 w4 (256),
// 7 emb (n_orb x 32), 8 b4 (1); the matching gradients with grad = 1.
extern "C" int qpx_mlp_param(qpx_mlp *m, int which, int grad, int set, float *data, int64_t n) {
  return mguard(m, [&] {
    QPX_HIP(hipSetDevice(m->device));
    DBuf<float> *P[8] = {&m->W1, &m->W2, &m->W3, &m->b1, &m->b2, &m->b3, &m->w4, &m->emb};
    DBuf<float> *G[8] = {&m->gW1, &m->gW2, &m->gW3, &m->gb1, &m->gb2, &m->gb3, &m->gw4, &m->gemb};
    if (which == 8) {
      QPX_REQUIRE(n == 1, "b4 has one element");
      if (grad) {
        QPX_HIP(hipMemcpyAsync(data, m->gb4.p, sizeof(float), hipMemcpyDeviceToHost, m->st));
        QPX_HIP(hipStreamSynchronize(m->st));
      } else if (set) {
        QPX_HIP(hipMemcpyAsync(m->b4.p, data, sizeof(float), hipMemcpyHostToDevice, m->st));
        QPX_HIP(hipStreamSynchronize(m->st));
      } else {
        QPX_HIP(hipMemcpyAsync(data, m->b4.p, sizeof(float), hipMemcpyDeviceToHost, m->st));
        QPX_HIP(hipStreamSynchronize(m->st));
      }
      return;
    }
    QPX_REQUIRE(which >= 0 && which < 8, "unknown parameter");
    DBuf<float> &b = grad ? *G[which] : *P[which];
    QPX_REQUIRE((size_t)n == b.n, "parameter size mismatch");
    if (set) {
      QPX_REQUIRE(!grad, "gradients are read-only");
      QPX_HIP(hipMemcpyAsync(b.p, data, sizeof(float) * n, hipMemcpyHostToDevice, m->st));
      uint16_t *pf[3] = {m->p1.p, m->p2.p, m->p3.p}, *pt[3] = {m->p1t.p, m->p2t.p, m->p3t.p};
      if (which < 3) hipLaunchKernelGGL(pack_kernel, dim3(64), dim3(256), 0, m->st, b.p, (int)(n / m->hid), pf[which], pt[which]);
    } else {
      QPX_HIP(hipMemcpyAsync(data, b.p, sizeof(float) * n, hipMemcpyDeviceToHost, m->st));
    }
    QPX_HIP(hipStreamSynchronize(m->st));
  });
}

// Test entry: C = A B through the weight gradients' tile in every operand layout
// it can stage.  ta = 0: A given (M x K) row-major; ta = 1: A given as its
// transpose, (K x M) row-major.  tb = 0: B (K x N) row-major; tb = 1: (N x K).
// split = 1 passes a workspace, so K is cut across workgroups where the tile
// grid is small.
extern "C" int qpx_debug_mlp_gemm(qpx_mlp *m, int M, int N, int K, const float *A, const float *B, int ta, int tb,
                                  int split, float *C) {
  if (M < 1 || N < 1 || K < 1 || !A || !B || !C) return 1;
  return mguard(m, [&] {
    QPX_HIP(hipSetDevice(m->device));
    DBuf<float> a, b, c, ws;
    DBuf<uint16_t> ab, bb;
    a.upload(A, (size_t)M * K, m->st);
    b.upload(B, (size_t)K * N, m->st);
    ab.alloc((size_t)M * K);
    bb.alloc((size_t)K * N);
    c.alloc((size_t)M * N);
    if (split) ws.alloc((size_t)32 * M * N);
    hipLaunchKernelGGL(to_bf16_kernel, dim3(64), dim3(256), 0, m->st, a.p, ab.p, (int64_t)M * K);
    hipLaunchKernelGGL(to_bf16_kernel, dim3(64), dim3(256), 0, m->st, b.p, bb.p, (int64_t)K * N);
    const int64_t ars = ta ? 1 : K, acs = ta ? M : 1;
    const int64_t brs = tb ? 1 : N, bcs = tb ? K : 1;
    gemm(m->st, ab.p, ars, acs, bb.p, brs, bcs, c.p, N, M, N, K, split ? &ws : nullptr);
    QPX_HIP(hipMemcpyAsync(C, c.p, sizeof(float) * M * N, hipMemcpyDeviceToHost, m->st));
    QPX_HIP(hipStreamSynchronize(m->st));
  });
}

// Plain bf16 GEMM C = A B (row-major A n x k, B k x m, fp32 inputs rounded
// to bf16), for the lane-layout and accuracy checks of the MFMA tiles.
extern "C" int qpx_mlp_gemm_check(qpx_mlp *m, int M, int N, int K, const float *A, const float *B, float *C) {
  return mguard(m, [&] {
    QPX_HIP(hipSetDevice(m->device));
    DBuf<float> a, b, c;
    DBuf<uint16_t> ab, bb;
    a.upload(A, (size_t)M * K, m->st);
    b.upload(B, (size_t)K * N, m->st);
    ab.alloc((size_t)M * K);
    bb.alloc((size_t)K * N);
    c.alloc((size_t)M * N);
    hipLaunchKernelGGL(to_bf16_kernel, dim3(64), dim3(256), 0, m->st, a.p, ab.p, (int64_t)M * K);
    hipLaunchKernelGGL(to_bf16_kernel, dim3(64), dim3(256), 0, m->st, b.p, bb.p, (int64_t)K * N);
    gemm(m->st, ab.p, K, 1, bb.p, N, 1, c.p, N, M, N, K);
    QPX_HIP(hipMemcpyAsync(C, c.p, sizeof(float) * M * N, hipMemcpyDeviceToHost, m->st));
    QPX_HIP(hipStreamSynchronize(m->st));
  });
}
