// sigma_fci.hip -- v = H u, s = S^2 u over a product space of spin strings
// (full CI, CAS): every alpha string with every beta string.
//
// Reference: H_S2_u_0_nstates_openmp_work (src/Davidson/u0Hu0.irp.f:97-458),
// which walks connected pairs one by one.  The dense-map kernels (sigma.hip)
// do the same from LDS and are bound by those gathers: one u row and one
// integral per alpha/beta pair.  In a product space the sums are contractions
// instead, and they run on the matrix cores:
//
//   alpha/beta doubles (sigma_fci_ab_kernel).  For a beta string b and its
//     singles b' (hole h, particle p, sign t), sum over r = (hp):
//       G[pq, a'] = sum_r (pq|r) t_r u(a', b'_r)
//     is a matrix product whose right factor is rows of u as they lie in
//     memory.  An orbital pair (pq) with one of p, q occupied in a' names one
//     single of a', so  v(a, b) += sign * G[pq, a']  places each element once
//     in the column b of v, which stays in LDS.  One LDS access per
//     (alpha string, pair) replaces one per (alpha single, beta single).
//   same-spin singles and doubles (sigma_fci_spin_kernel).  The strings are
//     taken 16 at a time; the partners of the 16 are listed once and their
//     matrix elements are stored as dense 16 x partners blocks: again a
//     matrix product with rows of u.
//   S^2: spin exchanges, one hole/particle swap of the singly occupied
//     orbitals at a time, by wavefronts that share the SIMDs with the products.
//
// FP64 products use v_mfma_f64_16x16x4 (77.8 TFLOP/s measured on this card
// with one wavefront per SIMD), FP32 ones v_mfma_f32_16x16x4 (150 TFLOP/s).
#include <algorithm>
#include <type_traits>
#include <vector>
#include "qpx_internal.h"
#include "qpx_device.h"

using namespace qpx;

namespace {

// 16x16x4 matrix instruction: lane l = (j = l % 16, q = l / 16) supplies
// A[j][q] and B[q][j] and holds D[row(q, r)][j], r = 0..3.
template <typename T>
struct Mfma;
template <>
struct Mfma<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mma(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __host__ __device__ constexpr int row(int q, int r) { return 4 * r + q; }
};
template <>
struct Mfma<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mma(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __host__ __device__ constexpr int row(int q, int r) { return 4 * q + r; }
};

template <typename T>
struct Prec;
template <>
struct Prec<double> {
  static const double *V(const Ham &H) { return H.V.p; }
  static const double *sval(const SpinConn &c) { return c.s_val.p; }
  static const double *dval(const SpinConn &c) { return c.d_val.p; }
  static FciTables<double> &tab(FciPlan &P) { return P.t64; }
};
template <>
struct Prec<float> {
  static const float *V(const Ham &H) { return H.Vf.p; }
  static const float *sval(const SpinConn &c) { return c.s_valf.p; }
  static const float *dval(const SpinConn &c) { return c.d_valf.p; }
  static FciTables<float> &tab(FciPlan &P) { return P.t32; }
};

__device__ __forceinline__ double flip_sign(double x, uint32_t bit31) {
  return __hiloint2double(__double2hiint(x) ^ (int)bit31, __double2loint(x));
}
__device__ __forceinline__ float flip_sign(float x, uint32_t bit31) {
  return __uint_as_float(__float_as_uint(x) ^ bit31);
}

// workgroups are dealt round-robin to the 8 XCDs: give each XCD a contiguous
// run of logical blocks, so that blocks that read the same rows share an L2
__device__ __forceinline__ int xcd_block() {
  const int n = (int)gridDim.x, base = n >> 3, rem = n & 7, x = (int)(blockIdx.x & 7);
  return x * base + min(x, rem) + (int)(blockIdx.x >> 3);
}

// off-diagonal orbital pair p < q (0-based) -> 0 .. M(M-1)/2 - 1
__host__ __device__ inline int off_pair(int p, int q) {
  const int lo = p < q ? p : q, hi = p < q ? q : p;
  return hi * (hi - 1) / 2 + lo;
}

constexpr uint32_t kNone = 0xffffffffu;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- tables
// A set-up kernel does both spins, blocks [0, n of alpha) and the rest: in a
// small space launches, allocations and waits are the time to the first result
// (4900 determinants, 4 vectors: 395 us; 655 with a launch per table and spin, an
// allocation per array and the partners' numbers read back, 480 with the dense
// map, which needs no tables).
struct SpinArgs {
  const int *s_ptr, *s_idx, *d_ptr, *d_idx;
  const uint32_t *s_info;
  int n, ntile, room;   // room: chunks of 8 partners at a tile's disposal, 0 = as many as it needs
  uint32_t *map;
  int2 *range;
  int *idx;
};

// map[i * npo + pair] = partner of string i through the single excitation
// between the pair's orbitals | sign << 31; kNone when both or neither are
// occupied
__global__ void fci_map_kernel(SpinArgs A, SpinArgs B, int npo) {
  int i = blockIdx.x;
  const bool beta = i >= A.n;
  if (beta) i -= A.n;
  const int *s_ptr = beta ? B.s_ptr : A.s_ptr, *s_idx = beta ? B.s_idx : A.s_idx;
  const uint32_t *s_info = beta ? B.s_info : A.s_info;
  uint32_t *map = beta ? B.map : A.map;
  for (int x = threadIdx.x; x < npo; x += blockDim.x) map[(int64_t)i * npo + x] = kNone;
  __syncthreads();
  for (int e = s_ptr[i] + (int)threadIdx.x; e < s_ptr[i + 1]; e += blockDim.x) {
    const uint32_t inf = s_info[e];
    map[(int64_t)i * npo + off_pair(inf & 0xff, (inf >> 8) & 0xff)] = (uint32_t)s_idx[e] | (((inf >> 16) & 1) << 31);
  }
}

// Targets in the order a lane of the product reads them: entry
// [(tile * ldt + a) * 4 + q] holds for r = 0..3 the target of pair row
// 16 tile + row(q, r) from alpha string a, as index | sign << 31 (a word
// each: its address is then one 24-bit multiply-add away; vector arithmetic
// does not overlap the matrix instructions of the same wavefront).  A row
// without a target points at the lane's own spare word behind the column, so
// that the placement needs no branch.  Rows npo + p are the diagonal pairs
// (pp): their target is the string itself when it holds p.
// Behind the targets, in the same launch: gb[i * npo + row], the sum over the
// orbitals k of beta string i of (row|kk), and vo[npo][nr], the integrals of each
// off-diagonal pair with all pairs.
template <typename T>
struct TableArgs {
  const uint32_t *map_a;
  const uint64_t *astr, *bstr;
  const T *V;
  int n_a, n_b, ldt, M, npo, nr, npair;
  int64_t n_tgt, n_gb, n_vo;
  uint4 *tgt;
  T *gb, *vo;
  FciConn conn, *conn_to;
};
// packed pair of row: off-diagonal pairs first, then the diagonal ones
__device__ inline int64_t pair_of_row(int row, int npo) {
  if (row >= npo) return pair_index(row - npo, row - npo);
  int q = (int)((1.0 + sqrt(1.0 + 8.0 * row)) / 2.0);
  while (q * (q - 1) / 2 > row) --q;
  while ((q + 1) * q / 2 <= row) ++q;
  return pair_index(row - q * (q - 1) / 2, q);
}
template <typename T>
__global__ __launch_bounds__(256) void fci_tables_kernel(TableArgs<T> A) {
  const int64_t n = A.n_tgt + A.n_gb + A.n_vo;
  if (blockIdx.x == 0 && threadIdx.x == 0) *A.conn_to = A.conn;
  for (int64_t y = blockIdx.x * (int64_t)256 + threadIdx.x; y < n; y += (int64_t)gridDim.x * 256) {
    int64_t x = y;
    if (x < A.n_tgt) {
      const int q = (int)(x & 3);
      const int a = (int)((x >> 2) % A.ldt), tile = (int)((x >> 2) / A.ldt);
      uint32_t w[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * tile + Mfma<T>::row(q, r);
        w[r] = (a < A.n_a && row < A.npo) ? A.map_a[(int64_t)a * A.npo + row] : kNone;
        if (a < A.n_a && row >= A.npo && row < A.npo + A.M && ((A.astr[a] >> (row - A.npo)) & 1)) w[r] = (uint32_t)a;
        if (w[r] == kNone) w[r] = (uint32_t)(A.n_a + 16 * q + (a & 15));
      }
      A.tgt[x] = make_uint4(w[0], w[1], w[2], w[3]);
      continue;
    }
    x -= A.n_tgt;
    if (x < A.n_gb) {
      const int i = (int)(x / A.npo), row = (int)(x - (int64_t)i * A.npo);
      const int64_t P = pair_of_row(row, A.npo);
      T g = T(0);
      for (uint64_t z = A.bstr[i]; z; z &= z - 1) {
        const int k = __ffsll((unsigned long long)z) - 1;
        g += A.V[P * A.npair + pair_index(k, k)];
      }
      A.gb[x] = g;
      continue;
    }
    x -= A.n_gb;
    A.vo[x] = A.V[pair_of_row((int)(x / A.nr), A.npo) * A.npair + pair_of_row((int)(x % A.nr), A.npo)];
  }
}

// Partners of 16 consecutive strings: a bitmap of the string set in LDS
// collects the singles and doubles of the 16; their number, rounded up to pairs
// of chunks of 8, gives the tile's range and the ascending list (padded with its
// first entry) goes to it.  With room for every tile one pass does both; without,
// a first pass (write = false) leaves the numbers in range[].y and the host the
// ranges for a second.
__global__ __launch_bounds__(256) void fci_union_kernel(SpinArgs A, SpinArgs B, bool write) {
  extern __shared__ uint32_t bits[];
  __shared__ int part[256];
  int tile = blockIdx.x;
  const SpinArgs &S = tile < A.ntile ? A : B;
  if (tile >= A.ntile) tile -= A.ntile;
  const int *s_ptr = S.s_ptr, *s_idx = S.s_idx, *d_ptr = S.d_ptr, *d_idx = S.d_idx;
  const int n = S.n, tid = threadIdx.x, nw = (n + 31) >> 5;
  for (int x = tid; x < nw; x += 256) bits[x] = 0;
  __syncthreads();
  const int i0 = 16 * tile, i1 = min(n, i0 + 16);
  for (int e = s_ptr[i0] + tid; e < s_ptr[i1]; e += 256) atomicOr(&bits[s_idx[e] >> 5], 1u << (s_idx[e] & 31));
  for (int e = d_ptr[i0] + tid; e < d_ptr[i1]; e += 256) atomicOr(&bits[d_idx[e] >> 5], 1u << (d_idx[e] & 31));
  __syncthreads();
  // each thread counts a contiguous run of words; the counts before it
  const int per = (nw + 255) / 256, w0 = min(nw, tid * per), w1 = min(nw, w0 + per);
  int c = 0;
  for (int w = w0; w < w1; ++w) c += __popc(bits[w]);
  part[tid] = c;
  __syncthreads();
  int before = 0, total = 0;
  for (int x = 0; x < 256; ++x) {
    if (x < tid) before += part[x];
    total += part[x];
  }
  const int nch = (total + 15) / 16 * 2;   // an even number: the product takes two at a time
  if (S.room && tid == 0) S.range[tile] = make_int2(tile * S.room, tile * S.room + nch);
  if (!write) {
    if (tid == 0) S.range[tile].y = nch;
    return;
  }
  int *out = S.idx + (int64_t)8 * (S.room ? tile * S.room : S.range[tile].x);
  for (int w = w0; w < w1; ++w)
    for (uint32_t y = bits[w]; y; y &= y - 1) out[before++] = 32 * w + __ffs(y) - 1;
  __syncthreads();
  for (int x = total + tid; x < 8 * nch; x += 256) out[x] = out[0];
}

// matrix elements of a tile: coef[(8 chunk + pos) * 16 + i % 16], zero where
// string i and the partner are not connected
template <typename T>
struct CoefArgs {
  const T *s_val, *d_val;
  T *coef;
};
template <typename T>
__global__ __launch_bounds__(256) void fci_coef_kernel(SpinArgs A, CoefArgs<T> CA, SpinArgs B, CoefArgs<T> CB) {
  int tile = blockIdx.x;
  const bool beta = tile >= A.ntile;
  if (beta) tile -= A.ntile;
  const SpinArgs &S = beta ? B : A;
  const CoefArgs<T> &C = beta ? CB : CA;
  const int *s_ptr = S.s_ptr, *s_idx = S.s_idx, *d_ptr = S.d_ptr, *d_idx = S.d_idx, *idx = S.idx;
  const T *s_val = C.s_val, *d_val = C.d_val;
  T *coef = C.coef;
  const int n = S.n, tid = threadIdx.x;
  const int2 range = S.range[tile];
  const int64_t c0 = (int64_t)8 * range.x;
  const int np = 8 * (range.y - range.x);
  for (int x = tid; x < 16 * np; x += 256) coef[c0 * 16 + x] = T(0);
  __syncthreads();
  const int i0 = 16 * tile, i1 = min(n, i0 + 16);
  auto place = [&](int i, int j, T v) {
    // the list ascends but for its padding, which repeats its first entry:
    // the last entry <= j below the padding is j itself
    int lo = 0, hi = np - 1;
    while (hi > 0 && idx[c0 + hi] == idx[c0]) --hi;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (idx[c0 + mid] < j) lo = mid + 1;
      else hi = mid;
    }
    coef[(c0 + lo) * 16 + (i - i0)] = v;
  };
  for (int i = i0; i < i1; ++i) {
    for (int e = s_ptr[i] + tid; e < s_ptr[i + 1]; e += 256) place(i, s_idx[e], s_val[e]);
    for (int e = d_ptr[i] + tid; e < d_ptr[i + 1]; e += 256) place(i, d_idx[e], d_val[e]);
  }
}

// ---------------------------------------------------------------- layouts
// u (beta-major, state-fastest) -> one plane per state, with the alpha
// strings contiguous (pb[st][b][lda]) and with the beta strings contiguous
// (pa[st][a][ldb]); the padding of the rows is zero.
template <typename T>
__global__ __launch_bounds__(256) void fci_planes_kernel(const T *__restrict__ u, int n_a, int n_b, int lda, int ldb,
                                                         int nst, T *__restrict__ pb, T *__restrict__ pa) {
  extern __shared__ __align__(16) unsigned char raw[];
  T *t = reinterpret_cast<T *>(raw);   // [st][b % 32][33]
  const int nba = (max(lda, n_a) + 31) / 32;
  const int a0 = 32 * (int)(blockIdx.x % nba), b0 = 32 * (int)(blockIdx.x / nba);
  for (int x = threadIdx.x; x < 32 * 32 * nst; x += 256) {
    const int b = x / (32 * nst), y = x - b * 32 * nst, a = y / nst, st = y - a * nst;
    T v = T(0);
    if (a0 + a < n_a && b0 + b < n_b) v = u[((int64_t)(b0 + b) * n_a + a0 + a) * nst + st];
    t[(st * 32 + b) * 33 + a] = v;
  }
  __syncthreads();
  for (int x = threadIdx.x; x < 32 * 32 * nst; x += 256) {
    const int st = x >> 10, i = (x >> 5) & 31, j = x & 31;
    if (b0 + i < n_b && a0 + j < lda) pb[((int64_t)st * n_b + b0 + i) * lda + a0 + j] = t[(st * 32 + i) * 33 + j];
    if (a0 + i < n_a && b0 + j < ldb) pa[((int64_t)st * n_a + a0 + i) * ldb + b0 + j] = t[(st * 32 + j) * 33 + i];
  }
}

// ---------------------------------------------------------------- same spin
// y(string, column) (+)= sum over the partners of H(string, partner)
// x(partner, column).  A wavefront owns 16 strings and 16 NT columns of one
// state's plane; the partners go by in chunks of 8 (two matrix instructions
// deep), the next chunk's rows in flight while one is multiplied.  A lane
// reads W neighbouring columns at once (16 bytes with many columns), so block
// t of the product holds the columns 16 W (t / W) + W j + t % W.  With ALPHA the planes are pa (columns
// are beta strings) and the product is formed transposed, so that both spins
// write the same layout y[st][b][lda]; the beta pass adds to what the alpha
// pass wrote.
// The four wavefronts of a workgroup, and neighbouring workgroups, take the
// string tiles of one column block, whose rows (n x 16 NT values) stay in L2.
template <typename T, int NT, int W, bool ALPHA>
__global__ __launch_bounds__(256, 2) void sigma_fci_spin_kernel(const int2 *__restrict__ range,
                                                                const int *__restrict__ idx,
                                                                const T *__restrict__ coef, int n, int ntile,
                                                                int ld, int ncol, int ngrp, int nblk,
                                                                const T *__restrict__ x, T *__restrict__ y, int lda,
                                                                int n_b) {
  typedef typename Mfma<T>::v4 v4;
  typedef T vw __attribute__((ext_vector_type(W)));
  static_assert(NT % W == 0, "columns come in runs of W blocks");
  constexpr int NP = NT / W;
  const int logical = xcd_block();
  if (logical >= nblk) return;
  const int lane = threadIdx.x & 63, j = lane & 15, q = lane >> 4;
  const int nt4 = (ntile + 3) >> 2;
  const int grp = logical / nt4, tile = 4 * (logical - grp * nt4) + (int)(threadIdx.x >> 6);
  if (tile >= ntile) return;
  const int st = grp / ngrp, c0 = (grp - st * ngrp) * 16 * NT;
  const T *xs = x + (int64_t)st * n * ld;
  uint32_t col[NP];
#pragma unroll
  for (int t = 0; t < NP; ++t) col[t] = min(c0 + 16 * W * t, ld - 16 * W) + W * j;   // past the end: the last columns again
  const int k0 = range[tile].x, k1 = range[tile].y;
  v4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = v4{T(0), T(0), T(0), T(0)};
  if (k0 < k1) {
    // a chunk: rows of the 8 partners, elements; the row offsets of the chunk after it
    struct Chunk {
      vw b[2][NP];
      T a[2];
    } X, Y;
    uint32_t id[2];
    auto ids = [&](int k) {
#pragma unroll
      for (int s = 0; s < 2; ++s) id[s] = (uint32_t)idx[8 * (int64_t)k + 4 * s + q] * (uint32_t)ld;
    };
    auto load = [&](Chunk &C, int k) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        C.a[s] = coef[(8 * (int64_t)k + 4 * s) * 16 + lane];
#pragma unroll
        for (int t = 0; t < NP; ++t) C.b[s][t] = *reinterpret_cast<const vw *>(xs + (id[s] + col[t]));
      }
    };
    auto multiply = [&](const Chunk &C) {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int t = 0; t < NT; ++t)
          acc[t] = ALPHA ? Mfma<T>::mma(C.b[s][t / W][t % W], C.a[s], acc[t])
                         : Mfma<T>::mma(C.a[s], C.b[s][t / W][t % W], acc[t]);
    };
    // FP64: the loads go out before the products (4.85 -> 4.44 ms for both
    // spins at 9.0M determinants, 4 states); FP32, with half the time per
    // product, is faster with them in between (3.46 -> 3.02 ms)
    auto fence = [] {
      if constexpr (sizeof(T) == 8) __builtin_amdgcn_sched_barrier(0);
    };
    ids(k0);
    load(X, k0);
    ids(k0 + 1);
    for (int k = k0; k < k1; k += 2) {
      load(Y, k + 1);
      const int k2 = min(k + 2, k1 - 2);   // past the end: the last pair again, not used
      ids(k2);
      fence();
      multiply(X);
      fence();
      load(X, k2);
      ids(k2 + 1);
      fence();
      multiply(Y);
      fence();
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int cb = c0 + 16 * W * (t / W) + t % W;
    if (c0 + 16 * W * (t / W) >= ld) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int w = Mfma<T>::row(q, r);
      if (ALPHA) {   // rows are beta strings, columns the tile's alpha strings
        const int bb = cb + W * w, aa = 16 * tile + j;
        if (bb < ncol && aa < n) y[((int64_t)st * n_b + bb) * lda + aa] = acc[t][r];
      } else {
        const int bb = 16 * tile + w;
        if (bb < n) y[((int64_t)st * n_b + bb) * lda + cb + W * j] += acc[t][r];
      }
    }
  }
}

// ---------------------------------------------------------------- alpha/beta
struct FciArgs {
  const uint64_t *bstr;
  const int *bs_ptr, *bs_idx;
  const uint32_t *bs_info;
  const uint4 *tgt;
  const uint64_t *astr;
  const uint32_t *map_a, *map_b;
  const double *hdiag, *sdiag;
  const FciConn *conn;
  const void *vo, *gbs;   // integrals of off-diagonal pairs with all pairs [npo][nr]; Coulomb sums of the beta strings [n_b][npo]
  int n_a, n_b, lda, ldt, npo, nr, mt, nst, nrow;   // nrow: wavefronts per state, each with every nrow-th pair tile
  template <typename T>
  __device__ const T *Vo() const { return static_cast<const T *>(vo); }
  template <typename T>
  __device__ const T *Gb() const { return static_cast<const T *>(gbs); }
};

// v(a, b) of state st, connected determinant by connected determinant.  The
// products multiply an infinity or NaN of u by the zeros of elements that are
// not there; a sum that came out not finite is formed again from those that are.
template <typename T>
__device__ __forceinline__ double fci_element(const FciArgs &A, int b, int a, int st, const T *__restrict__ u) {
  auto at = [&](int bb, int aa) { return (double)u[((int64_t)bb * A.n_a + aa) * A.nst + st]; };
  auto val = [](const void *x, int e) { return (double)static_cast<const T *>(x)[e]; };
  const FciConn C = *A.conn;
  const T *vo = A.Vo<T>(), *gb = A.Gb<T>() + (int64_t)b * A.npo;
  double t = A.hdiag[(int64_t)b * A.n_a + a] * at(b, a);
  for (int e = C.ad_ptr[a]; e < C.ad_ptr[a + 1]; ++e) t += val(C.ad_val, e) * at(b, C.ad_idx[e]);
  for (int e = C.bd_ptr[b]; e < C.bd_ptr[b + 1]; ++e) t += val(C.bd_val, e) * at(C.bd_idx[e], a);
  for (int e = C.as_ptr[a]; e < C.as_ptr[a + 1]; ++e) {
    const uint32_t inf = C.as_info[e];
    const double g = (double)gb[off_pair(inf & 0xff, (inf >> 8) & 0xff)];
    t += (val(C.as_val, e) + ((inf >> 16) & 1 ? -g : g)) * at(b, C.as_idx[e]);
  }
  for (int f = A.bs_ptr[b]; f < A.bs_ptr[b + 1]; ++f) {
    const uint32_t inf = A.bs_info[f];
    const T *row = vo + (int64_t)off_pair(inf & 0xff, (inf >> 8) & 0xff) * A.nr;
    const uint32_t neg = (inf >> 16) & 1;
    double g = 0.0;
    for (uint64_t y = A.astr[a]; y; y &= y - 1) g += (double)row[A.npo + __ffsll((unsigned long long)y) - 1];
    t += (val(C.bs_val, f) + (neg ? -g : g)) * at(A.bs_idx[f], a);
    for (int e = C.as_ptr[a]; e < C.as_ptr[a + 1]; ++e) {
      const uint32_t ia = C.as_info[e];
      const double h = (double)row[off_pair(ia & 0xff, (ia >> 8) & 0xff)];
      t += (neg ^ ((ia >> 16) & 1) ? -h : h) * at(A.bs_idx[f], C.as_idx[e]);
    }
  }
  return t;
}

// One workgroup per beta string b; wavefront w < nst nrow owns state w % nst
// and the pair tiles w / nst, w / nst + nrow, ... and adds into a column of
// its own, so that every sum has a fixed order.  Per 16 NT alpha strings it
// holds the rows u(a', b'_r) of all singles (4 KS of them) in registers,
// multiplies them by each tile of 16 orbital pairs, whose integrals sit in
// LDS with the beta signs, and places the previous tile's results between
// the matrix instructions; the next tile's integrals and the next rows are in
// flight meanwhile.  The alpha singles' Coulomb terms are the accumulators'
// start; the beta singles' ones are the diagonal pairs (pp), whose results
// stay in place (one more tile of pairs, or none where the last tile has
// room; a plain sum over the same rows by other wavefronts took longer: its
// loads delay the products').  The kHelp last wavefronts share the SIMDs with
// the matrix products and do what is no contraction: S^2.
// The columns are FP64 in both precisions: ds_add_f64 takes 11.5 cycles a
// wavefront here, ds_add_f32 194 (measured, no conflicts).
// Registers are kept within 256 (two wavefronts per SIMD allowed): above
// that the compiler moves every accumulator through the AGPRs.
constexpr int kHelp = 4;

// s(a, b) = sdiag u(a, b) - sum over the orbitals h of b alone and p of a
// alone of the sign of the exchange times u(a: p -> h, b: h -> p): about
// (n/2)^2 exchanges of a determinant, found from the two strings' bits, kX in
// flight.
template <typename T, int NST>
__device__ __forceinline__ void spin_exchange(const FciArgs &A, int b, uint64_t bw, int a0, const T *__restrict__ u,
                                              T *__restrict__ s) {
  constexpr int kX = 8;
  const uint32_t *mb = A.map_b + (int64_t)b * A.npo;
  for (int a = a0; a < A.n_a; a += 64 * kHelp) {
    const uint64_t aw = A.astr[a];
    const uint32_t *ma = A.map_a + (int64_t)a * A.npo;
    const int64_t e = (int64_t)b * A.n_a + a;
    double acc[NST];   // FP64 in both precisions: these wavefronts have the time
#pragma unroll
    for (int st = 0; st < NST; ++st) acc[st] = A.sdiag[e] * (double)u[e * NST + st];
    uint64_t y = aw & ~bw, z = bw & ~aw;
    const uint64_t z0 = z;
    if (z0 == 0) y = 0;
    while (y) {
      const T *src[kX];
      uint32_t sg[kX];
      bool on[kX];
#pragma unroll
      for (int i = 0; i < kX; ++i) {
        on[i] = y != 0;
        const int p = on[i] ? __ffsll((unsigned long long)y) - 1 : 1;
        const int h = on[i] ? __ffsll((unsigned long long)z) - 1 : 0;
        const int pr = off_pair(h, p);
        uint32_t x = ma[pr], w = mb[pr];
        on[i] = on[i] && x != kNone && w != kNone;   // a partner string outside the space
        if (!on[i]) x = w = 0;
        sg[i] = (~(x ^ w)) & 0x80000000u;   // minus the sign of the pair of singles
        src[i] = u + ((int64_t)(w & 0x7fffffffu) * A.n_a + (x & 0x7fffffffu)) * NST;
        z &= z - 1;
        if (z == 0) {
          z = z0;
          y &= y - 1;
        }
      }
      T t[kX][NST];
#pragma unroll
      for (int i = 0; i < kX; ++i)
#pragma unroll
        for (int st = 0; st < NST; ++st) t[i][st] = src[i][st];
#pragma unroll
      for (int i = 0; i < kX; ++i)
        if (on[i])
#pragma unroll
          for (int st = 0; st < NST; ++st) acc[st] += (double)flip_sign(t[i][st], sg[i]);
    }
#pragma unroll
    for (int st = 0; st < NST; ++st) s[e * NST + st] = (T)acc[st];
  }
}

// what a matrix wavefront keeps of a tile of 16 pairs: integrals, Coulomb
// starts, targets and sums
template <typename T, int KS, int NT>
struct FciTile {
  T a[KS], g[4];
  u32x4 tg[NT];
  typename Mfma<T>::v4 acc[NT];
};

template <typename T, int KS, int NT>
__global__ __launch_bounds__(512, 2) void sigma_fci_ab_kernel(FciArgs A, const T *__restrict__ pb, const T *__restrict__ y, const T *__restrict__ u,
                                                              T *__restrict__ v, T *__restrict__ s) {
  typedef typename Mfma<T>::v4 v4;
  extern __shared__ __align__(16) unsigned char raw[];
  const int nw = A.nst * A.nrow;
  const int ldc = A.n_a + 64;
  double *col = reinterpret_cast<double *>(raw);   // [nw][ldc]
  T *vb = reinterpret_cast<T *>(col + (size_t)nw * ldc);   // [mt][4 KS][16]: a read of 4 singles x 16 pairs is contiguous
  T *gb = vb + (size_t)4 * KS * 16 * A.mt;         // [16 mt]
  uint32_t *orow = reinterpret_cast<uint32_t *>(gb + 16 * A.mt);   // [4 KS] rows of u of the singles
  uint32_t *grow = orow + 4 * KS;                  // [4 KS] their Coulomb rows | sign << 31
  const int b = xcd_block(), tid = threadIdx.x, nth = blockDim.x;
  const int s0 = A.bs_ptr[b], kb = A.bs_ptr[b + 1] - s0;
  const uint64_t bw = A.bstr[b];
  for (int x = tid; x < nw * ldc; x += nth) col[x] = 0.0;
  // rows of the singles; a padding single reads the row of b itself, against zero integrals
  for (int k = tid; k < 4 * KS; k += nth) {
    orow[k] = (uint32_t)(k < kb ? A.bs_idx[s0 + k] : b) * A.lda;
    grow[k] = kNone;
    if (k < kb) {
      const uint32_t inf = A.bs_info[s0 + k];
      grow[k] = (uint32_t)off_pair(inf & 0xff, (inf >> 8) & 0xff) | (((inf >> 16) & 1) << 31);
    }
  }
  __syncthreads();
  // integrals of the singles of b with every pair, signs included
  for (int x0 = tid; x0 < 4 * KS * 16 * A.mt; x0 += 4 * nth) {
    T val[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int x = x0 + i * nth, k = x / (16 * A.mt), row = x - k * 16 * A.mt;
      const uint32_t gk = k < 4 * KS ? grow[k] : kNone;
      val[i] = T(0);
      if (gk != kNone && row < A.nr) val[i] = flip_sign(A.Vo<T>()[(gk & 0x7fffffffu) * A.nr + row], gk & 0x80000000u);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int x = x0 + i * nth, k = x / (16 * A.mt), row = x - k * 16 * A.mt;
      if (k < 4 * KS) vb[((row >> 4) * 4 * KS + k) * 16 + (row & 15)] = val[i];
    }
  }
  for (int row = tid; row < 16 * A.mt; row += nth) gb[row] = row < A.npo ? A.Gb<T>()[(int64_t)b * A.npo + row] : T(0);
  __syncthreads();

  const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (wv >= nw) {
    const int a0 = 64 * (wv - nw) + lane;
    switch (A.nst) {
      case 1: spin_exchange<T, 1>(A, b, bw, a0, u, s); break;
      case 2: spin_exchange<T, 2>(A, b, bw, a0, u, s); break;
      case 3: spin_exchange<T, 3>(A, b, bw, a0, u, s); break;
      default: spin_exchange<T, 4>(A, b, bw, a0, u, s); break;
    }
  } else {
    const int j = lane & 15, q = lane >> 4;
    const int part = __builtin_amdgcn_readfirstlane(wv / A.nst);
    const int st = wv - part * A.nst;
    double *mine = col + (size_t)wv * ldc;
    const T *pst = pb + (int64_t)st * A.n_b * A.lda;
    const uint32_t own = (uint32_t)b * A.lda + j;
    const int ngrp = (A.lda + 16 * NT - 1) / (16 * NT);
    // blocks past the end repeat the last one: their targets are spare words
    auto a_of = [&](int g, int t) { return (uint32_t)min(16 * (g * NT + t), A.lda - 16); };
    const T *av = vb + lane;
    const uint32_t tlane = 4 * j + q;
    T B[KS][NT], ub[NT];
    FciTile<T, KS, NT> X, Y;
    auto load_tile = [&](FciTile<T, KS, NT> &N, int m) {
#pragma unroll
      for (int r = 0; r < 4; ++r) N.g[r] = gb[16 * m + Mfma<T>::row(q, r)];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) N.a[ks] = av[(m * KS + ks) * 64];
    };
    auto load_tg = [&](u32x4 *to, int g, int m) {
      const u32x4 *base = reinterpret_cast<const u32x4 *>(A.tgt) + ((int64_t)m * A.ldt + 16 * NT * g) * 4;
#pragma unroll
      for (int t = 0; t < NT; ++t) to[t] = base[64 * t + tlane];
    };
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      ub[t] = pst[own + a_of(0, t)];
      Y.tg[t] = u32x4{1, 1, 1, 1} * (uint32_t)(A.n_a + lane);
      Y.acc[t] = v4{T(0), T(0), T(0), T(0)};
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const uint32_t o = orow[4 * ks + q] + j;
#pragma unroll
      for (int t = 0; t < NT; ++t) B[ks][t] = pst[o + a_of(0, t)];
    }
    load_tile(X, part);
    load_tg(X.tg, 0, part);
    // element i % 4 of block i / 4 of a finished tile to its column
    auto place = [&](const FciTile<T, KS, NT> &D, int i) {
      const int t = i >> 2, r = i & 3;
      const uint32_t w = D.tg[t][r];
      double *to = reinterpret_cast<double *>(reinterpret_cast<char *>(mine) + __umul24(w, 8));
      unsafeAtomicAdd(to, flip_sign((double)D.acc[t][r], w & 0x80000000u));
    };
    // multiply tile C, place what O holds, and load the next tile (gn, mn) into O
    auto step = [&](FciTile<T, KS, NT> &C, FciTile<T, KS, NT> &O, int gn, int mn, auto &&also) {
      u32x4 tn[NT];
      load_tg(tn, gn, mn);
      also();
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) C.acc[t][r] = C.g[r] * ub[t];
      load_tile(O, mn);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
        for (int t = 0; t < NT; ++t) C.acc[t] = Mfma<T>::mma(C.a[ks], B[ks][t], C.acc[t]);
#pragma unroll
        for (int i = 0; i < 4 * NT; ++i)
          if (i * KS / (4 * NT) == ks) place(O, i);
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) O.tg[t] = tn[t];
    };
    const int cnt = (A.mt - part + A.nrow - 1) / A.nrow;   // this wavefront's tiles
    for (int g = 0; g < ngrp; ++g) {
      T Bn[KS][NT], un[NT];
      const int gn = min(g + 1, ngrp - 1);
      // the next rows are requested behind the first step's own loads, which
      // are waited for first
      auto rows = [&] {
#pragma unroll
        for (int t = 0; t < NT; ++t) un[t] = pst[own + a_of(gn, t)];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const uint32_t o = orow[4 * ks + q] + j;
#pragma unroll
          for (int t = 0; t < NT; ++t) Bn[ks][t] = pst[o + a_of(gn, t)];
        }
      };
      auto none = [] {};
      auto m_of = [&](int i) { return i < cnt ? part + i * A.nrow : part; };   // tile i, or the next group's first
      auto g_of = [&](int i) { return i < cnt ? g : gn; };
      step(X, Y, g_of(1), m_of(1), rows);
      int i = 1;
      for (; i + 1 < cnt; i += 2) {
        step(Y, X, g, m_of(i + 1), none);
        step(X, Y, g_of(i + 2), m_of(i + 2), none);
      }
      if (i < cnt) {
        step(Y, X, gn, part, none);
      } else {   // an odd number of tiles: the roles are exchanged once per group
        auto swap = [](auto &x, auto &z) { auto w = x; x = z; z = w; };
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) swap(X.a[ks], Y.a[ks]);
#pragma unroll
        for (int r = 0; r < 4; ++r) swap(X.g[r], Y.g[r]);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          swap(X.tg[t], Y.tg[t]);
          swap(X.acc[t], Y.acc[t]);
        }
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        ub[t] = un[t];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) B[ks][t] = Bn[ks][t];
      }
    }
#pragma unroll
    for (int i = 0; i < 4 * NT; ++i) place(Y, i);
  }
  __syncthreads();
  // column of v: the wavefronts' parts in order, the same-spin part, the
  // diagonal; a thread takes an alpha string with all its states
  const int64_t plane = (int64_t)A.n_b * A.lda;
  for (int a = tid; a < A.n_a; a += nth) {
    const int64_t e = (int64_t)b * A.n_a + a;
    const T hd = (T)A.hdiag[e];
    T uu[4], yy[4];
#pragma unroll
    for (int st = 0; st < 4; ++st)
      if (st < A.nst) {
        uu[st] = u[e * A.nst + st];
        yy[st] = y[st * plane + (int64_t)b * A.lda + a];
      }
#pragma unroll
    for (int st = 0; st < 4; ++st)
      if (st < A.nst) {
        double t = 0.0;
        for (int r = 0; r < A.nrow; ++r) t += col[(size_t)(r * A.nst + st) * ldc + a];
        t += (double)yy[st] + (double)(hd * uu[st]);
        if (!isfinite(t)) t = fci_element<T>(A, b, a, st, u);
        v[e * A.nst + st] = (T)t;
      }
  }
}

// ---------------------------------------------------------------- host
int round_up(int x, int m) { return (x + m - 1) / m * m; }

// steps of 4 singles the alpha/beta kernel is instantiated for
constexpr int kSteps[] = {2, 4, 6, 8, 9, 10, 12, 14, 16, 20, 24};

int steps_for(int singles) {
  for (int k : kSteps)
    if (4 * k >= singles) return k;
  return 0;
}

struct Shape {
  int ks = 0, mt = 0, nrow = 0;
  size_t lds = 0;
};

// LDS of the alpha/beta kernel, with as many wavefronts per state as it takes
// to give each SIMD one (four in all) and as fit; ks = 0: it does not fit
Shape ab_shape(const qpx_ctx *c, int nst, size_t ts, int max_singles) {
  Shape S;
  const int npo = c->H.M * (c->H.M - 1) / 2;
  S.mt = (npo + c->H.M + 15) / 16;
  const int ks = steps_for(std::max(1, max_singles));
  if (!ks) return S;
  S.nrow = std::max(1, std::min(4 / nst, S.mt));
  for (; S.nrow >= 1; --S.nrow) {
    S.lds = ((size_t)4 * ks * 16 * S.mt + 16 * S.mt) * ts + sizeof(double) * nst * S.nrow * (c->W.n_a + 64) +
            2 * sizeof(uint32_t) * 4 * ks;
    if (S.lds <= (size_t)c->lds_per_block) {
      S.ks = ks;
      return S;
    }
  }
  return S;
}

SpinArgs spin_args(const SpinConn &cc, int n, const SpinTiles &t, int room, const View<uint32_t> &map) {
  return SpinArgs{cc.s_ptr.p, cc.s_idx.p, cc.d_ptr.p, cc.d_idx.p, cc.s_info.p, n, t.ntile, room, map.p, t.range.p, t.idx.p};
}

// most chunks of 8 partners (an even number, not 0) the 16 strings of a tile have
int most_chunks(const SpinConn &cc, int n) {
  return std::max(2, (int)((std::min<int64_t>(n, 16 * ((int64_t)cc.max_singles + cc.max_doubles)) + 15) / 16 * 2));
}

// Enqueued on the context's stream, as build_tables; the caller waits.
void build_plan(qpx_ctx *c) {
  Wfn &W = c->W;
  FciPlan &P = W.fci;
  if (P.valid) return;
  hipStream_t s = c->stream;
  const int M = c->H.M, npo = M * (M - 1) / 2;
  // whole runs of 16 W columns; the padding of small sets stays small
  P.lda = round_up(W.n_a, W.n_a >= 256 ? 64 : 32);
  P.ldb = round_up(W.n_b, W.n_b >= 256 ? 64 : 32);
  P.ldt = round_up(W.n_a, 64);
  P.a.ntile = (W.n_a + 15) / 16;
  P.b.ntile = (W.n_b + 15) / 16;
  P.mem.layout([&] {
    P.mem.lay(P.map_a, (size_t)W.n_a * npo);
    P.mem.lay(P.map_b, (size_t)W.n_b * npo);
    P.mem.lay(P.a.range, P.a.ntile);
    P.mem.lay(P.b.range, P.b.ntile);
  });
  // Room for the most partners a tile can have, where the FP64 elements (1 KB a
  // chunk) then take at most 4 MB: the partners are listed without a look at
  // their number.
  int room_a = most_chunks(W.ca, W.n_a), room_b = most_chunks(W.cb, W.n_b);
  P.a.nchunk = (int64_t)P.a.ntile * room_a;
  P.b.nchunk = (int64_t)P.b.ntile * room_b;
  const size_t lds = sizeof(uint32_t) * ((std::max(W.n_a, W.n_b) + 31) / 32);
  const dim3 grid(P.a.ntile + P.b.ntile), block(256);
  auto args = [&](bool beta) {
    return beta ? spin_args(W.cb, W.n_b, P.b, room_b, P.map_b) : spin_args(W.ca, W.n_a, P.a, room_a, P.map_a);
  };
  if (P.a.nchunk + P.b.nchunk > 4096) {
    room_a = room_b = 0;
    hipLaunchKernelGGL(fci_union_kernel, grid, block, lds, s, args(false), args(true), false);
    QPX_HIP(hipGetLastError());
    for (SpinTiles *t : {&P.a, &P.b}) {
      std::vector<int2> r(t->ntile);
      QPX_HIP(hipMemcpyAsync(r.data(), t->range.p, sizeof(int2) * t->ntile, hipMemcpyDeviceToHost, s));
      QPX_HIP(hipStreamSynchronize(s));
      int64_t at = 0;
      for (int2 &x : r) {
        x = make_int2((int)at, (int)at + x.y);
        at = x.y;
      }
      t->nchunk = at;
      QPX_HIP(hipMemcpyAsync(t->range.p, r.data(), sizeof(int2) * t->ntile, hipMemcpyHostToDevice, s));
      QPX_HIP(hipStreamSynchronize(s));   // r goes out of scope
    }
  }
  P.lists.layout([&] {
    P.lists.lay(P.a.idx, (size_t)8 * P.a.nchunk);
    P.lists.lay(P.b.idx, (size_t)8 * P.b.nchunk);
  });
  hipLaunchKernelGGL(fci_map_kernel, dim3(W.n_a + W.n_b), dim3(64), 0, s, args(false), args(true), npo);
  hipLaunchKernelGGL(fci_union_kernel, grid, block, lds, s, args(false), args(true), true);
  QPX_HIP(hipGetLastError());
  P.valid = true;
}

template <typename T>
void build_tables(qpx_ctx *c) {
  Wfn &W = c->W;
  FciPlan &P = W.fci;
  FciTables<T> &t = Prec<T>::tab(P);
  if (t.valid) return;
  hipStream_t s = c->stream;
  const int M = c->H.M, npo = M * (M - 1) / 2, nr = npo + M, mt = (nr + 15) / 16;
  t.mem.layout([&] {
    t.mem.lay(t.coef_a, (size_t)128 * P.a.nchunk);
    t.mem.lay(t.coef_b, (size_t)128 * P.b.nchunk);
    t.mem.lay(t.tgt, (size_t)mt * P.ldt * 4);
    t.mem.lay(t.gb, (size_t)npo * W.n_b);
    t.mem.lay(t.vo, (size_t)npo * nr);
    t.mem.lay(t.conn, 1);
  });
  const SpinArgs a = spin_args(W.ca, W.n_a, P.a, 0, P.map_a), b = spin_args(W.cb, W.n_b, P.b, 0, P.map_b);
  hipLaunchKernelGGL(fci_coef_kernel<T>, dim3(P.a.ntile + P.b.ntile), dim3(256), 0, s, a,
                     CoefArgs<T>{Prec<T>::sval(W.ca), Prec<T>::dval(W.ca), t.coef_a.p}, b,
                     CoefArgs<T>{Prec<T>::sval(W.cb), Prec<T>::dval(W.cb), t.coef_b.p});
  const TableArgs<T> A{P.map_a.p, W.astr.p, W.bstr.p, Prec<T>::V(c->H), W.n_a, W.n_b, P.ldt, M, npo, nr, c->H.npair,
                       (int64_t)mt * P.ldt * 4, (int64_t)npo * W.n_b, (int64_t)npo * nr, t.tgt.p, t.gb.p, t.vo.p,
                       FciConn{W.ca.s_ptr.p, W.ca.s_idx.p, W.ca.d_ptr.p, W.ca.d_idx.p, W.cb.d_ptr.p, W.cb.d_idx.p,
                               W.ca.s_info.p, Prec<T>::sval(W.ca), Prec<T>::dval(W.ca), Prec<T>::sval(W.cb),
                               Prec<T>::dval(W.cb)},
                       t.conn.p};
  hipLaunchKernelGGL(fci_tables_kernel<T>, dim3((unsigned)std::min<int64_t>((A.n_tgt + A.n_gb + A.n_vo + 255) / 256, 4096)),
                     dim3(256), 0, s, A);
  QPX_HIP(hipGetLastError());
  QPX_HIP(hipStreamSynchronize(s));   // the call may be on another stream
  t.valid = true;
}

template <typename T, int KS>
void launch_ab(qpx_ctx *c, const Shape &S, int nst, const T *pb, T *y, const T *u, T *v, T *s, hipStream_t st) {
  Wfn &W = c->W;
  FciPlan &P = W.fci;
  FciTables<T> &t = Prec<T>::tab(P);
  // blocks of 16 alpha strings at a time: what two sets of KS x NT rows and
  // two of KS integrals leave of the 256 registers
  constexpr int NT = KS * (int)sizeof(T) <= (sizeof(T) == 8 ? 16 : 40) ? 4 : KS * (int)sizeof(T) <= 96 ? 2 : 1;
  FciArgs A{W.bstr.p, W.cb.s_ptr.p, W.cb.s_idx.p, W.cb.s_info.p, t.tgt.p, W.astr.p, P.map_a.p,
            P.map_b.p, W.hdiag.p, W.sdiag.p, t.conn.p, t.vo.p, t.gb.p, W.n_a, W.n_b, P.lda, P.ldt,
            c->H.M * (c->H.M - 1) / 2, c->H.M * (c->H.M + 1) / 2, S.mt, nst, S.nrow};
  auto k = sigma_fci_ab_kernel<T, KS, NT>;
  QPX_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S.lds));
  hipLaunchKernelGGL(k, dim3(W.n_b), dim3(64 * (nst * S.nrow + kHelp)), S.lds, st, A, pb, y, u, v, s);
  QPX_HIP(hipGetLastError());
}

template <typename T, int NT, int W>
void launch_spin(qpx_ctx *c, int nst, const T *pa, const T *pb, T *y, hipStream_t st) {
  Wfn &F = c->W;
  FciPlan &P = F.fci;
  FciTables<T> &t = Prec<T>::tab(P);
  const int ga = (P.ldb + 16 * NT - 1) / (16 * NT), gb = (P.lda + 16 * NT - 1) / (16 * NT);
  const int na = nst * ga * ((P.a.ntile + 3) / 4), nb = nst * gb * ((P.b.ntile + 3) / 4);
  hipLaunchKernelGGL((sigma_fci_spin_kernel<T, NT, W, true>), dim3(na), dim3(256), 0, st, P.a.range.p, P.a.idx.p,
                     t.coef_a.p, F.n_a, P.a.ntile, P.ldb, F.n_b, ga, na, pa, y, P.lda, F.n_b);
  hipLaunchKernelGGL((sigma_fci_spin_kernel<T, NT, W, false>), dim3(nb), dim3(256), 0, st, P.b.range.p, P.b.idx.p,
                     t.coef_b.p, F.n_b, P.b.ntile, P.lda, F.n_a, gb, nb, pb, y, P.lda, F.n_b);
  QPX_HIP(hipGetLastError());
}

// scratch of a call: two planes per state over the beta strings, one over the alpha strings
template <typename T>
char *scratch_for(qpx_ctx *c, int nst, hipStream_t st) {
  const Wfn &W = c->W;
  const FciPlan &P = W.fci;
  return c->ws_fci.get(sizeof(T) * (size_t)nst * (2 * (size_t)W.n_b * P.lda + (size_t)W.n_a * P.ldb), st);
}

template <typename T>
void run(qpx_ctx *c, const Shape &S, char *ws, int nst, const T *u, T *v, T *s, hipStream_t st) {
  Wfn &W = c->W;
  FciPlan &P = W.fci;
  const int64_t plane_b = (int64_t)W.n_b * P.lda;
  T *pb = (T *)ws, *y = pb + nst * plane_b, *pa = y + nst * plane_b;
  const int nba = (P.lda + 31) / 32, nbb = (P.ldb + 31) / 32;
  const size_t lds_t = sizeof(T) * nst * 32 * 33;
  auto kp = fci_planes_kernel<T>;
  QPX_HIP(hipFuncSetAttribute((const void *)kp, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_t));
  hipLaunchKernelGGL(kp, dim3(nba * nbb), dim3(256), lds_t, st, u, W.n_a, W.n_b, P.lda, P.ldb, nst, pb, pa);
  QPX_HIP(hipGetLastError());
  if (c->ktiming) QPX_HIP(hipEventRecord(c->kev[0], st));
  // 128 columns per wavefront where that still gives every SIMD two of them
  if (P.lda % 64 == 0 && P.ldb % 64 == 0 && (int64_t)nst * (P.lda / 128) * P.b.ntile >= 2048)
    launch_spin<T, 8, 16 / (int)sizeof(T)>(c, nst, pa, pb, y, st);
  else
    launch_spin<T, 2, 2>(c, nst, pa, pb, y, st);
  if (c->ktiming) QPX_HIP(hipEventRecord(c->kev[1], st));
  switch (S.ks) {
    case 2: launch_ab<T, 2>(c, S, nst, pb, y, u, v, s, st); break;
    case 4: launch_ab<T, 4>(c, S, nst, pb, y, u, v, s, st); break;
    case 6: launch_ab<T, 6>(c, S, nst, pb, y, u, v, s, st); break;
    case 8: launch_ab<T, 8>(c, S, nst, pb, y, u, v, s, st); break;
    case 9: launch_ab<T, 9>(c, S, nst, pb, y, u, v, s, st); break;
    case 10: launch_ab<T, 10>(c, S, nst, pb, y, u, v, s, st); break;
    case 12: launch_ab<T, 12>(c, S, nst, pb, y, u, v, s, st); break;
    case 14: launch_ab<T, 14>(c, S, nst, pb, y, u, v, s, st); break;
    case 16: launch_ab<T, 16>(c, S, nst, pb, y, u, v, s, st); break;
    case 20: launch_ab<T, 20>(c, S, nst, pb, y, u, v, s, st); break;
    default: launch_ab<T, 24>(c, S, nst, pb, y, u, v, s, st); break;
  }
  if (c->ktiming) QPX_HIP(hipEventRecord(c->kev[2], st));
  c->ws_fci.used(st);
}

}  // namespace

namespace qpx {

// The string-driven path takes a product space (every alpha string with every
// beta string) whose column of v, with the integrals of one beta string, fits
// the LDS of a workgroup.
bool fci_ok(qpx_ctx *c, int nst, size_t ts) {
  const Wfn &W = c->W;
  if (W.nint != 1 || nst > 4 || c->H.M < 2) return false;
  if (W.n_det != (int64_t)W.n_a * W.n_b) return false;
  if (W.n_a + 64 > 0x7fff || W.n_b > 65535) return false;
  // 32-bit row offsets within a plane
  if ((int64_t)W.n_b * round_up(W.n_a, 64) >= (1LL << 31) || (int64_t)W.n_a * round_up(W.n_b, 64) >= (1LL << 31))
    return false;
  // cheap bound before the connectivity is built: at most n (M - n) singles
  const int most = std::max(c->H.na * (c->H.M - c->H.na), c->H.nb * (c->H.M - c->H.nb));
  if (!ab_shape(c, nst, ts, most).ks) return false;
  return true;
}

// Whether the string-driven kernels are the faster ones for a space that the
// dense map could take too.  They give a beta string one workgroup of four
// matrix wavefronts, the dense map one workgroup per 1024 alpha strings, and
// their work does not shrink with the connections that an incomplete set
// lacks: with fewer beta strings than CUs, many alpha strings and several
// vectors the dense map can win (20 orbitals, 4a1b, 4845 x 20 strings, FP32, 2
// vectors: 433 against 935 us; 14 orbitals, 6a1b, 3003 x 14, FP64, 1 vector: 263
// against 206).  The two times, in microseconds, are fitted to 1072 spaces of
// 1 to 256 beta strings (4 to 30 orbitals, 1, 2 and 4 vectors, both
// precisions) within about 10 %.  By them no space is more than 8 % slower than
// with the dense map, and the mean is 1 % above the faster of the two.  With more beta strings
// the string-driven kernels were at most 4 % behind in incomplete sets, and 1.5
// to 4 times as fast in complete ones.
bool fci_pays(qpx_ctx *c, int nst, size_t ts) {
  const Wfn &W = c->W;
  if (W.n_b > 256 || W.n_a < 128) return true;
  ensure_conn(c);
  const Shape S = ab_shape(c, nst, ts, W.cb.max_singles);
  if (!S.ks) return true;
  const bool f64 = ts == 8;
  const double n_a = W.n_a, n_b = W.n_b, groups = (W.n_a + 63) / 64, tiles = (double)S.mt / S.nrow;
  const double strings = (f64 ? 18.4 : 20.6) + 5.0e-5 * nst * n_a * n_b +
                         groups * (tiles * (f64 ? 0.103 + 0.161 * S.ks : 0.291 + 0.078 * S.ks) + (f64 ? 2.8 : 2.4));
  // per string: beta singles k, alpha singles and same-spin partners
  const double k = W.cb.n_singles / n_b, sa = W.ca.n_singles / n_a, same_a = sa + W.ca.n_doubles / n_a;
  const double same_b = k + W.cb.n_doubles / n_b, rows = std::min(1.0, n_a / 1024);
  const double rounds = (W.n_b * ((W.n_a + 1023) / 1024) + 255) / 256, row_rounds = n_a / 256;
  const double stage = nst * n_a / 1024;
  const double dense =
      f64 ? 6.7 + 9.2 * nst + rounds * (k * (1.54 + 0.056 * stage + sa * rows * (0.014 + 0.067 * nst)) + 0.325 * rows * same_a) +
                row_rounds * 0.110 * same_b
          : 12.5 + 3.1 * nst + rounds * (k * (1.46 + 0.156 * stage + sa * rows * (0.110 + 0.016 * nst)) + 0.222 * rows * same_a) +
                row_rounds * (1.72 + 0.054 * same_b);
  return strings < 0.95 * dense;
}

// False when the tables or the scratch do not fit the device's memory: the
// caller then takes a path that needs none.  What the call began and could not
// finish goes again; what is complete stays, for the calls and captured graphs
// that use it.
bool sigma_fci(qpx_ctx *c, int prec, int nst, const void *u, void *v, void *s, hipStream_t st) {
  ensure_conn(c);
  FciPlan &P = c->W.fci;
  auto drop = [&] {
    if (prec == QPX_FP64 && !P.t64.valid) P.t64.release();
    if (prec != QPX_FP64 && !P.t32.valid) P.t32.release();
    if (!P.valid) P.release();
  };
  char *ws = nullptr;
  try {
    build_plan(c);
    if (prec == QPX_FP64) build_tables<double>(c);
    else build_tables<float>(c);
    ws = prec == QPX_FP64 ? scratch_for<double>(c, nst, st) : scratch_for<float>(c, nst, st);
  } catch (const OutOfMemory &) {
    drop();
    return false;
  } catch (...) {
    drop();
    throw;
  }
  if (prec == QPX_FP64)
    run<double>(c, ab_shape(c, nst, 8, c->W.cb.max_singles), ws, nst, (const double *)u, (double *)v, (double *)s, st);
  else
    run<float>(c, ab_shape(c, nst, 4, c->W.cb.max_singles), ws, nst, (const float *)u, (float *)v, (float *)s, st);
  return true;
}

}  // namespace qpx
