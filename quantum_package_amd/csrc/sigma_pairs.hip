// sigma_pairs.hip -- v = H u, s = S^2 u for selected wavefunctions, bucket by
// bucket.
//
// Reference: H_S2_u_0_nstates_openmp_work (src/Davidson/u0Hu0.irp.f:97-458).
// As in sigma_sparse.hip, connected determinants are found as members of the
// same bucket: two spin strings are single (double) excitations of each other
// iff they share an (n-1)- ((n-2)-) electron sub-string, and that sub-string
// is unique.  That file walks, for every determinant, the buckets of all its
// slots; every visit then reads the partner's entry, its row of u and an
// integral from addresses of their own, and works out a phase.
//
// Here the work is laid out by bucket.  A lane owns one entry m of a bucket
// (a determinant with its removed orbitals) and runs over the bucket's
// members n:
//   - the members and their rows of u are the same for all lanes of the
//     bucket: a wavefront brings them to LDS once;
//   - the integral sits at table[base(n) + offset(m)], the offset (the removed
//     orbitals of m) running along the table, so neighbouring lanes read
//     neighbouring words; the table holds zero where m and n share a removed
//     orbital, so the loop has no tests;
//   - the phase is the product of a sign of m and one of n (the parity of
//     the electrons below the removed orbitals in the common sub-string).
// The sums of an entry go to memory once, and one pass per determinant adds
// its entries' sums in slot order, the diagonal and S^2 (whose few spin
// exchanges per determinant are listed at set-up).  Buckets with one member
// have no pairs and are dropped (38-55 % of the entries of a selected
// wavefunction).  The others are ordered by size: those of 256 and more
// (kSplit) get a workgroup per 64 entries, which cuts the chain of the largest
// ones to a quarter; those of 64 and more a wavefront per 64 entries; of the
// smaller ones a wavefront takes as many of one size as fit, and there every
// integral is read once for both of its determinants.
//
// 262,144 determinants, 96 orbitals, 10 + 10 electrons, FP64, 4 states: 7.6 ms
// by determinant, here 2.3 (doubles 1.59, singles 0.21, collection 0.46);
// 40,003, 50 orbitals, FP32, 2 states: 459 and 125 us.  The doubles read 7.5 GB
// from HBM, at 4.7 TB/s (an integral table of 0.85 GB in an order with little
// reuse: half the occupancy or twice the loads in flight changes nothing; at 2.1M
// determinants, with longer buckets, they reach 7.6 TB/s), the collection 3.2 GB
// at 7 TB/s.  The table
// packed by pair symmetry (0.34 GB) was slower, 1.82 ms: neighbouring lanes
// no longer read neighbouring words.
#include <algorithm>
#include <type_traits>
#include <vector>
#include <hipcub/hipcub.hpp>
#include "qpx_internal.h"
#include "qpx_device.h"

using namespace qpx;

namespace {

constexpr int kMaxElec = 32, kMaxState = 8;
constexpr uint32_t kSign = 0x80000000u;
constexpr uint32_t kSplit = 256;   // members from which on a workgroup shares the lanes' sums

__device__ __forceinline__ double flip(double x, uint32_t bit31) {
  return __hiloint2double(__double2hiint(x) ^ (int)bit31, __double2loint(x));
}
__device__ __forceinline__ float flip(float x, uint32_t bit31) { return __uint_as_float(__float_as_uint(x) ^ bit31); }

__host__ __device__ inline int lower_pair(int p, int q) { return q * (q - 1) / 2 + p; }   // p < q

// electrons of a string below orbital o
template <int NI>
__device__ inline int below(const uint64_t *x, int o) {
  int c = 0;
#pragma unroll
  for (int w = 0; w < NI; ++w) {
    const int n = o - 64 * w;
    if (n >= 64) c += __popcll(x[w]);
    else if (n > 0) c += __popcll(x[w] & ((1ULL << n) - 1));
  }
  return c;
}

// ---------------------------------------------------------------- sub-strings
struct Removed {
  int i, j;   // orbitals; j = -1 when one is removed
};
template <int NI>
__device__ inline Removed removed_of(const uint64_t *x, int ne, int drop, int slot) {
  if (drop == 1) return Removed{kth_bit<NI>(x, slot), -1};
  int a, b;
  pair_of(slot, ne, &a, &b);
  return Removed{kth_bit<NI>(x, a), kth_bit<NI>(x, b)};
}
template <int NI>
__device__ inline uint64_t sub_word(const uint64_t *str, int ne, int drop, int nslot, int e, int w) {
  const uint64_t *x = str + (int64_t)(e / nslot) * NI;
  const Removed r = removed_of<NI>(x, ne, drop, e % nslot);
  uint64_t y = x[w];
  if ((r.i >> 6) == w) y &= ~(1ULL << (r.i & 63));
  if (r.j >= 0 && (r.j >> 6) == w) y &= ~(1ULL << (r.j & 63));
  return y;
}

template <int NI>
__global__ void sub_key_kernel(const uint64_t *__restrict__ str, int ne, int drop, int nslot, int n, int w,
                               const int *__restrict__ ord, uint64_t *__restrict__ key) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x)
    key[t] = sub_word<NI>(str, ne, drop, nslot, ord[t], w);
}
__global__ void iota_kernel(int *__restrict__ v, int64_t n) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x) v[t] = (int)t;
}
template <int NI>
__global__ void sub_head_kernel(const uint64_t *__restrict__ str, int ne, int drop, int nslot, int n,
                                const int *__restrict__ ord, int *__restrict__ head) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x) {
    bool h = t == 0;
    for (int w = 0; w < NI && !h; ++w)
      h = sub_word<NI>(str, ne, drop, nslot, ord[t], w) != sub_word<NI>(str, ne, drop, nslot, ord[t - 1], w);
    head[t] = h;
  }
}
__global__ void sub_id_kernel(const int *__restrict__ ord, const int *__restrict__ sid, int n, int *__restrict__ id) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x) id[ord[t]] = sid[t] - 1;
}

int grid_for(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 1 << 16)); }

// scratch of the set-up, taken piece by piece from one block; the block is
// sized by a first pass over the same calls (base null)
struct Arena {
  char *base = nullptr;
  size_t used = 0;
  char *tmp = nullptr;   // hipCUB's temporary storage
  size_t tmp_n = 0;
  DBuf<char> more;       // where a smaller count asks for more than its bound did
  template <typename T>
  T *take(size_t n) {
    T *p = reinterpret_cast<T *>(base + used);
    used += (n * sizeof(T) + 255) / 256 * 256;
    return p;
  }
  // f(storage, bytes): a hipCUB call
  template <typename F>
  void cub(F f) {
    size_t need = 0;
    QPX_HIP(f((char *)nullptr, need));
    if (!base) {
      tmp_n = std::max(tmp_n, need);
    } else if (need <= tmp_n) {
      QPX_HIP(f(tmp, need));
    } else {
      if (more.n < need) more.alloc(need);
      QPX_HIP(f(more.p, need));
    }
  }
};
template <typename K>
void sort_pairs(Arena &A, const K *k, K *k2, const int *v, int *v2, int64_t n, int bits, hipStream_t s, bool down = false) {
  A.cub([&](char *p, size_t &need) {
    return down ? hipcub::DeviceRadixSort::SortPairsDescending(p, need, k, k2, v, v2, (int)n, 0, bits, s)
                : hipcub::DeviceRadixSort::SortPairs(p, need, k, k2, v, v2, (int)n, 0, bits, s);
  });
}
template <bool INCL>
void scan(Arena &A, const int *in, int *out, int64_t n, hipStream_t s) {
  A.cub([&](char *p, size_t &need) {
    return INCL ? hipcub::DeviceScan::InclusiveSum(p, need, in, out, (int)n, s)
                : hipcub::DeviceScan::ExclusiveSum(p, need, in, out, (int)n, s);
  });
}
void read_ints(const int *p, int n, int *v, hipStream_t s) {
  QPX_HIP(hipMemcpyAsync(v, p, sizeof(int) * n, hipMemcpyDeviceToHost, s));
  QPX_HIP(hipStreamSynchronize(s));
}
void copy_int(const int *from, int *to, hipStream_t s) {
  QPX_HIP(hipMemcpyAsync(to, from, sizeof(int), hipMemcpyDeviceToDevice, s));
}
int bits_of(uint64_t x) {   // bits of the values 0..x
  int b = 1;
  while (b < 64 && (x >> b) != 0) ++b;
  return b;
}

struct SortScratch {
  uint64_t *k1, *k2;
  int *v1, *v2;
};

// ids of the (ne - drop)-electron sub-strings of n strings, id[string * nslot
// + slot], their number to *count
template <int NI>
void substring_ids(Arena &A, const SortScratch &Z, const uint64_t *str, int n, int M, int ne, int drop, int *id,
                   int *count, hipStream_t s) {
  const int nslot = drop == 1 ? ne : ne * (ne - 1) / 2;
  const int64_t m = (int64_t)n * nslot;
  if (m == 0) return;
  int *v1 = Z.v1, *v2 = Z.v2;
  const int g = grid_for(m);
  if (A.base) hipLaunchKernelGGL(iota_kernel, dim3(g), dim3(256), 0, s, v1, m);
  for (int w = 0; w < NI; ++w) {   // stable passes, word by word
    if (A.base) {
      hipLaunchKernelGGL(sub_key_kernel<NI>, dim3(g), dim3(256), 0, s, str, ne, drop, nslot, (int)m, w, v1, Z.k1);
      QPX_HIP(hipGetLastError());
    }
    sort_pairs(A, Z.k1, Z.k2, v1, v2, m, std::max(1, std::min(64, M - 64 * w)), s);
    std::swap(v1, v2);
  }
  int *sid = reinterpret_cast<int *>(Z.k1);
  if (A.base) hipLaunchKernelGGL(sub_head_kernel<NI>, dim3(g), dim3(256), 0, s, str, ne, drop, nslot, (int)m, v1, v2);
  scan<true>(A, v2, sid, m, s);
  if (!A.base) return;
  hipLaunchKernelGGL(sub_id_kernel, dim3(g), dim3(256), 0, s, v1, sid, (int)m, id);
  QPX_HIP(hipGetLastError());
  copy_int(sid + (m - 1), count, s);
}

// ---------------------------------------------------------------- buckets
// classes: 0 ab (alpha minus one, beta minus one), 1 a2, 2 b2 (one spin minus
// two), 3 a1, 4 b1 (one spin minus one)
struct ClassArgs {
  int cls, nslot;
  const int *sa, *sb;   // sub-string ids (null: the string's own id)
  int nsa, nsb;
  int64_t mult;         // key = hi * mult + lo
  int slot0, S;         // first of the class's slots, all slots of a determinant
  int M, npo, ne_a, ne_b;
  uint32_t tab2;        // offset of the same-spin table
};

__global__ void pair_key_kernel(ClassArgs C, const int *__restrict__ csc_a, const int *__restrict__ csc_b, int64_t n,
                                uint64_t *__restrict__ key, int *__restrict__ orig) {
  for (int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; x < n; x += (int64_t)gridDim.x * blockDim.x) {
    const int64_t k = x / C.nslot;
    const int sl = (int)(x - k * C.nslot);
    const int a = csc_a[k], b = csc_b[k];
    uint64_t hi = (uint64_t)a, lo = (uint64_t)b;
    if (C.cls == 0) {
      hi = (uint64_t)C.sa[(int64_t)a * C.nsa + sl / C.nsb];
      lo = (uint64_t)C.sb[(int64_t)b * C.nsb + sl % C.nsb];
    } else if (C.sa) {
      hi = (uint64_t)C.sa[(int64_t)a * C.nsa + sl];
    } else {
      lo = (uint64_t)C.sb[(int64_t)b * C.nsb + sl];
    }
    key[x] = hi * (uint64_t)C.mult + lo;
    orig[x] = (int)x;
  }
}
__global__ void pair_head_kernel(const uint64_t *__restrict__ key, int64_t n, int *__restrict__ head) {
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x)
    head[p] = p == 0 || key[p] != key[p - 1];
}
__global__ void pair_start_kernel(const int *__restrict__ head, const int *__restrict__ sid, int64_t n,
                                  int *__restrict__ start) {
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x)
    if (head[p]) start[sid[p] - 1] = (int)p;
}
// sizes of the buckets; buckets of one are given size 0 (dropped)
__global__ void pair_size_kernel(const int *__restrict__ start, int nseg, int64_t n, uint32_t *__restrict__ size,
                                 int *__restrict__ id) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < nseg; q += (int64_t)gridDim.x * blockDim.x) {
    const int64_t len = (q + 1 < nseg ? (int64_t)start[q + 1] : n) - start[q];
    size[q] = len > 1 ? (uint32_t)len : 0;
    id[q] = (int)q;
  }
}
// Positions of the buckets, in the order of decreasing size: one of 64 and
// more starts on a wavefront; of the smaller ones a wavefront takes as many of
// one size as fit.  first: number of the first bucket of each size below 64.
__global__ void pair_first_kernel(const uint32_t *__restrict__ size, int nseg, int *__restrict__ first) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < nseg; q += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t z = size[q];
    if (z < 64 && (q == 0 || size[q - 1] != z)) first[z] = (int)q;
  }
}
__global__ void pair_room_kernel(const uint32_t *__restrict__ size, int nseg, const int *__restrict__ first,
                                 int *__restrict__ room) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < nseg; q += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t z = size[q];
    if (z >= 64) room[q] = (int)((z + 63) & ~63u);
    else room[q] = z && ((uint32_t)q - (uint32_t)first[z]) % (64 / z) == 0 ? 64 : 0;
  }
}
__global__ void pair_place_kernel(const int *__restrict__ id, const int *__restrict__ at, const int *__restrict__ room,
                                  const uint32_t *__restrict__ size, int nseg, const int *__restrict__ first,
                                  int *__restrict__ place, int *__restrict__ total) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < nseg; q += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t z = size[q];
    int p = -1;
    if (z < kSplit && (q == 0 || size[q - 1] >= kSplit)) total[1] = at[q];
    if (z >= 64) p = at[q];
    else if (z) {
      const uint32_t r = ((uint32_t)q - (uint32_t)first[z]) % (64 / z);
      p = at[q] + (r ? (int)(r * z) - 64 : 0);
    }
    place[id[q]] = p;
    if (q == nseg - 1) {
      total[0] = at[q] + room[q];
      if (z >= kSplit) total[1] = total[0];
    }
  }
}

struct EntryArrays {
  uint2 *ent;        // determinant | sign << 31; table base (ab, a2, b2) or particle (a1, b1)
  uint32_t *off;     // table offset, or hole
  int2 *wave;        // 64 and more members: first, number; fewer: lanes in use, number
  int *slotpos;      // [determinant][slot]: position of its entry, -1: none
};

template <int NI>
__global__ void pair_fill_kernel(ClassArgs C, const int *__restrict__ orig, const int *__restrict__ sid,
                                 const int *__restrict__ start, const int *__restrict__ place, int64_t n, int nseg,
                                 const int *__restrict__ csc_a, const int *__restrict__ csc_b,
                                 const uint64_t *__restrict__ astr, const uint64_t *__restrict__ bstr, int base_big,
                                 int base_small, EntryArrays E) {
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x) {
    const int o = orig[p];
    const int64_t k = o / C.nslot;
    const int sl = o - (int)(k * C.nslot);
    const int s = sid[p] - 1, first = place[s];
    int *to = E.slotpos + k * C.S + C.slot0 + sl;
    if (first < 0) {
      *to = -1;
      continue;
    }
    const int len = (s + 1 < nseg ? start[s + 1] : (int)n) - start[s];
    const int b0 = (len >= (int)kSplit ? base_big : base_small) + first, at = b0 + (int)p - start[s];
    *to = at;
    const uint64_t *aw = astr + (int64_t)csc_a[k] * NI, *bw = bstr + (int64_t)csc_b[k] * NI;
    uint32_t base, off;
    int par;
    if (C.cls == 0) {
      const int i = kth_bit<NI>(aw, sl / C.nsb), j = kth_bit<NI>(bw, sl % C.nsb);
      par = below<NI>(aw, i) + below<NI>(bw, j);
      off = (uint32_t)(j * C.M + i);
      base = (uint32_t)(i * C.M + j) * (uint32_t)(C.M * C.M);
    } else if (C.cls <= 2) {
      const uint64_t *x = C.cls == 1 ? aw : bw;
      const Removed r = removed_of<NI>(x, C.cls == 1 ? C.ne_a : C.ne_b, 2, sl);
      par = below<NI>(x, r.i) + below<NI>(x, r.j);
      off = (uint32_t)lower_pair(r.i, r.j);
      base = C.tab2 + off * (uint32_t)C.npo;
    } else {
      const uint64_t *x = C.cls == 3 ? aw : bw;
      const int i = kth_bit<NI>(x, sl);
      par = below<NI>(x, i);
      off = base = (uint32_t)i;
    }
    E.ent[at] = make_uint2((uint32_t)k | ((par & 1) ? kSign : 0u), base);
    E.off[at] = off;
    if (len >= 64) {
      E.wave[at >> 6] = make_int2(b0, len);
    } else {
      atomicMax(&E.wave[at >> 6].x, (at & 63) + 1);
      E.wave[at >> 6].y = len;
    }
  }
}

// ---------------------------------------------------------------- S^2
// spin exchanges of determinant k (orbitals i of alpha alone and j of beta
// alone trade places) that are in the wavefunction: determinant | sign << 31.
// Pass 0 counts, pass 1 writes.
template <int NI>
__device__ inline bool key_less(const uint64_t *x, const uint64_t *y) {
  uint64_t kx = 0, ky = 0;
#pragma unroll
  for (int w = 0; w < NI; ++w) {
    kx ^= x[w];
    ky ^= y[w];
  }
  if (kx != ky) return kx < ky;
#pragma unroll
  for (int w = 0; w < NI; ++w)
    if (x[w] != y[w]) return x[w] < y[w];
  return false;
}
// index of string x among the n unique ones (ordered by the exclusive-or of
// their words, then the words), or -1
template <int NI>
__device__ inline int find_string(const uint64_t *str, int n, const uint64_t *x) {
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (key_less<NI>(str + (int64_t)mid * NI, x)) lo = mid + 1;
    else hi = mid;
  }
  if (lo == n) return -1;
#pragma unroll
  for (int w = 0; w < NI; ++w)
    if (str[(int64_t)lo * NI + w] != x[w]) return -1;
  return lo;
}
template <int NI>
__global__ void exchange_kernel(const int *__restrict__ csc_a, const int *__restrict__ csc_b,
                                const int *__restrict__ col_ptr, const uint64_t *__restrict__ astr, int n_a,
                                const uint64_t *__restrict__ bstr, int n_b, int64_t n, const int *__restrict__ ptr,
                                int *__restrict__ count, uint32_t *__restrict__ list) {
  for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
    uint64_t a[NI], b[NI];
#pragma unroll
    for (int w = 0; w < NI; ++w) {
      a[w] = astr[(int64_t)csc_a[k] * NI + w];
      b[w] = bstr[(int64_t)csc_b[k] * NI + w];
    }
    int c = 0;
    for (int wi = 0; wi < NI; ++wi)
      for (uint64_t y = a[wi] & ~b[wi]; y; y &= y - 1) {
        const int i = 64 * wi + __ffsll((unsigned long long)y) - 1;
        for (int wj = 0; wj < NI; ++wj)
          for (uint64_t z = b[wj] & ~a[wj]; z; z &= z - 1) {
            const int j = 64 * wj + __ffsll((unsigned long long)z) - 1;
            uint64_t a2[NI], b2[NI];
#pragma unroll
            for (int w = 0; w < NI; ++w) {
              const uint64_t mi = w == (i >> 6) ? 1ULL << (i & 63) : 0, mj = w == (j >> 6) ? 1ULL << (j & 63) : 0;
              a2[w] = (a[w] & ~mi) | mj;
              b2[w] = (b[w] & ~mj) | mi;
            }
            const int ib = find_string<NI>(bstr, n_b, b2);
            if (ib < 0) continue;
            const int ia = find_string<NI>(astr, n_a, a2);
            if (ia < 0) continue;
            int lo = col_ptr[ib], hi = col_ptr[ib + 1];
            const int end = hi;
            while (lo < hi) {
              const int mid = (lo + hi) >> 1;
              if (csc_a[mid] < ia) lo = mid + 1;
              else hi = mid;
            }
            if (lo == end || csc_a[lo] != ia) continue;
            if (list) {
              const int par = between_parity<NI>(a, i, j) ^ between_parity<NI>(b, i, j);
              list[ptr[k] + c] = (uint32_t)lo | (par ? 0u : kSign);   // minus the phase of the double excitation
            }
            ++c;
          }
      }
    if (!list) count[k] = c;
  }
}

// ---------------------------------------------------------------- tables
// [((x M + y) M + j) M + i] = (x i|y j), zero where x = i or y = j; behind it
// [pair(x < y)][pair(i < j)] = (i x|j y) - (i y|j x), zero where they share an orbital
template <typename T>
__global__ void pair_table_kernel(const double *__restrict__ V, int M, int npair, int npo, T *__restrict__ tab) {
  const int64_t n4 = (int64_t)M * M * M * M, n = n4 + (int64_t)npo * npo;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x) {
    double v = 0.0;
    if (q < n4) {
      const int i = (int)(q % M);
      int64_t t = q / M;
      const int j = (int)(t % M);
      t /= M;
      const int y = (int)(t % M), x = (int)(t / M);
      if (x != i && y != j) v = V[pair_index(x, i) * npair + pair_index(y, j)];
    } else {
      const int64_t t = q - n4;
      auto split = [](int r, int *p, int *s) {
        int u = (int)((1.0 + sqrt(1.0 + 8.0 * r)) / 2.0);
        while (u * (u - 1) / 2 > r) --u;
        while ((u + 1) * u / 2 <= r) ++u;
        *s = u;
        *p = r - u * (u - 1) / 2;
      };
      int x, y, i, j;
      split((int)(t / npo), &x, &y);
      split((int)(t % npo), &i, &j);
      if (x != i && x != j && y != i && y != j)
        v = V[pair_index(i, x) * npair + pair_index(j, y)] - V[pair_index(i, y) * npair + pair_index(j, x)];
    }
    tab[q] = (T)v;
  }
}
// single excitation i -> x from the HF occupation: h + sum over HF's orbitals,
// [spin][x M + i]
__global__ void fock_table_kernel(const double *__restrict__ hcore, const double *__restrict__ GS,
                                  const double *__restrict__ GO, int M, int na, int nb,
                                  double *__restrict__ f) {
  for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < 2 * M * M; q += gridDim.x * blockDim.x) {
    const int sp = q / (M * M), r = q - sp * M * M, x = r / M, i = r - x * M;
    const int ns = sp ? nb : na, no = sp ? na : nb;
    const int64_t row = ((int64_t)i * M + x) * M;
    double v = hcore[i * M + x];
    for (int k = 0; k < ns; ++k) v += GS[row + k];
    for (int k = 0; k < no; ++k) v += GO[row + k];
    f[q] = v;
  }
}

// ---------------------------------------------------------------- kernels
// orders the LDS accesses of one wavefront's lanes
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Sums and the rows of u in LDS are FP64 in both precisions: a chain over a
// bucket that holds one large coefficient (HF's) rounds every later term
// against it.

// adds members [c, end) of one bucket, 64 at a time: their rows of u, with the
// members' signs, go to LDS (ru, this wavefront's)
template <typename T, int NST>
__device__ __forceinline__ void add_members(const uint2 *ent, int c, int end, const T *row, const T *u,
                                            double *ru, double (&acc)[NST]) {
  constexpr int B = 16;   // integrals in flight
  const int lane = threadIdx.x & 63;
  for (; c < end; c += 64) {
    const int n = min(64, end - c);
    const uint2 e = ent[c + min(lane, n - 1)];
    const T *src = u + (int64_t)(e.x & ~kSign) * NST;
#pragma unroll
    for (int st = 0; st < NST; ++st) ru[lane * NST + st] = lane < n ? (double)flip(src[st], e.x & kSign) : 0.0;
    wave_fence();
    for (int r = 0; r < n; r += B) {
      T g[B];
#pragma unroll
      for (int i = 0; i < B; ++i) g[i] = row[(uint32_t)__builtin_amdgcn_readlane((int)e.y, r + i)];
#pragma unroll
      for (int i = 0; i < B; ++i)
#pragma unroll
        for (int st = 0; st < NST; ++st) acc[st] += (double)g[i] * ru[(r + i) * NST + st];
    }
    wave_fence();
  }
}

// sums of the double excitations of every entry
template <typename T, int NST>
__global__ __launch_bounds__(256) void pair_doubles_kernel(const uint2 *__restrict__ ent, const uint32_t *__restrict__ off,
                                                           const int2 *__restrict__ wave, int nbig, int nwave,
                                                           const T *__restrict__ tab, const T *__restrict__ u,
                                                           T *__restrict__ part) {
  __shared__ double row_u[256 * NST];
  // 16 workgroups in a row to an XCD: they share a bucket's members and rows of the
  // table in its L2 (1.62 -> 1.59 ms above; 2.1M determinants, the call 113 -> 107 ms)
  int blk = (int)blockIdx.x;
  if ((blk | 127) < (int)gridDim.x) blk = (blk & ~127) | (blk & 7) << 4 | (blk & 127) >> 3;
  __shared__ uint32_t row_base[256];
  const int lane = threadIdx.x & 63;
  const int sub = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  double *ru = row_u + sub * 64 * NST;
  double acc[NST];
#pragma unroll
  for (int st = 0; st < NST; ++st) acc[st] = 0.0;
  if (blk < nbig) {
    // 64 entries of a bucket of kSplit and more: a quarter of the members each
    const int64_t p = (int64_t)blk * 64 + lane;
    const int2 d = wave[blk];
    add_members<T, NST>(ent, d.x + (int)((int64_t)d.y * sub / 4), d.x + (int)((int64_t)d.y * (sub + 1) / 4), tab + off[p],
                        u, ru, acc);
#pragma unroll
    for (int st = 0; st < NST; ++st) ru[st * 64 + lane] = acc[st];
    __syncthreads();
    if (sub || p >= d.x + d.y) return;
    const uint32_t own = ent[p].x;
#pragma unroll
    for (int st = 0; st < NST; ++st) {
#pragma unroll
      for (int q = 1; q < 4; ++q) acc[st] += row_u[q * 64 * NST + st * 64 + lane];
      part[p * NST + st] = (T)flip(acc[st], own & kSign);
    }
    return;
  }
  const int wv = nbig + (blk - nbig) * 4 + sub;
  if (wv >= nwave) return;
  const int2 d = wave[wv];
  if (d.y == 0) return;
  const int64_t p = (int64_t)wv * 64 + lane;
  const uint2 own = ent[p];
  const T *row = tab + off[p];
  if (d.y >= 64) {
    add_members<T, NST>(ent, d.x, d.x + d.y, row, u, ru, acc);
    if (p >= d.x + d.y) return;
#pragma unroll
    for (int st = 0; st < NST; ++st) part[p * NST + st] = (T)flip(acc[st], own.x & kSign);
    return;
  }
  // buckets of one size: their rows of u, with the members' signs, and table
  // bases to LDS.  The element of a pair is the same both ways, so lane m
  // reads those of m + 1 .. m + size / 2 (round the bucket) and hands each on.
  const int z = d.y, half = z >> 1;
  const bool on = lane < d.x;
  uint32_t *rb = row_base + sub * 64;
  rb[lane] = own.y;
  const T *src = u + (int64_t)(own.x & ~kSign) * NST;
  T x[NST], g[4];
#pragma unroll
  for (int st = 0; st < NST; ++st) x[st] = src[st];
  wave_fence();
  const int m = lane % z;
  auto load = [&](int r0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = r0 + i;
      g[i] = T(0);
      if (r <= half && on) g[i] = row[rb[m + r < z ? lane + r : lane + r - z]];
    }
  };
  load(1);   // beside the rows of u
#pragma unroll
  for (int st = 0; st < NST; ++st) ru[lane * NST + st] = (double)flip(x[st], own.x & kSign);
  wave_fence();
  for (int r0 = 1;;) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = r0 + i;
      if (r > half) break;
      const int up = !on ? lane : m + r < z ? lane + r : lane + r - z;
      const int dn = !on ? lane : m >= r ? lane - r : lane - r + z;
#pragma unroll
      for (int st = 0; st < NST; ++st) acc[st] += (double)g[i] * ru[up * NST + st];
      if (2 * r < z) {
        const double h = (double)__shfl(g[i], dn);
#pragma unroll
        for (int st = 0; st < NST; ++st) acc[st] += h * ru[dn * NST + st];
      }
    }
    r0 += 4;
    if (r0 > half) break;
    load(r0);
  }
  if (!on) return;
#pragma unroll
  for (int st = 0; st < NST; ++st) part[p * NST + st] = (T)flip(acc[st], own.x & kSign);
}

struct SingleArgs {
  const int *csc_a, *csc_b;
  const uint64_t *astr, *bstr;
  int64_t n_alpha;   // end of the alpha entries
  int M, na, nb;
};

// sums of the single excitations: HF's element plus the change of the
// occupations (a few orbitals) instead of a sum over all electrons; elements in
// FP64 in both precisions, what HF's occupation adds being taken off again
template <typename T, int NI, int NST>
__global__ __launch_bounds__(256) void pair_singles_kernel(SingleArgs A, int64_t first, const uint2 *__restrict__ ent,
                                                           const uint32_t *__restrict__ off,
                                                           const int2 *__restrict__ wave, const double *__restrict__ fock,
                                                           const T *__restrict__ GS, const T *__restrict__ GO,
                                                           const T *__restrict__ u, T *__restrict__ part) {
  const int64_t p = first + blockIdx.x * (int64_t)256 + threadIdx.x;
  const int2 d2 = wave[p >> 6];
  const int lane = threadIdx.x & 63;
  if (d2.y == 0 || (d2.y >= 64 ? p >= d2.x + d2.y : lane >= d2.x)) return;
  const int b0 = d2.y >= 64 ? d2.x : (int)p - lane % d2.y, b1 = b0 + d2.y;
  const uint32_t own = ent[p].x;
  const int64_t d = own & ~kSign;
  const int i = (int)off[p], M = A.M;
  const bool beta = p >= A.n_alpha;
  const uint64_t *a = A.astr + (int64_t)A.csc_a[d] * NI, *b = A.bstr + (int64_t)A.csc_b[d] * NI;
  uint64_t same[NI], other[NI];   // changes from HF: the sub-string of this spin, the other spin
  uint64_t hs[NI], ho[NI];        // HF's occupations
#pragma unroll
  for (int w = 0; w < NI; ++w) {
    const int ns = (beta ? A.nb : A.na) - 64 * w, no = (beta ? A.na : A.nb) - 64 * w;
    hs[w] = ns <= 0 ? 0ULL : ns >= 64 ? ~0ULL : (1ULL << ns) - 1;
    ho[w] = no <= 0 ? 0ULL : no >= 64 ? ~0ULL : (1ULL << no) - 1;
    const uint64_t x = beta ? b[w] : a[w], y = beta ? a[w] : b[w];
    same[w] = (w == (i >> 6) ? x & ~(1ULL << (i & 63)) : x) ^ hs[w];
    other[w] = y ^ ho[w];
  }
  double acc[NST];
#pragma unroll
  for (int st = 0; st < NST; ++st) acc[st] = 0.0;
  const double *f = fock + (beta ? M * M : 0) + i;
  for (int k = b0; k < b1; k += 4) {
    uint2 e[4];
    double h[4];
    const T *gs[4], *go[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      e[q] = ent[min(k + q, b1 - 1)];
      const int64_t row = ((int64_t)i * M + e[q].y) * M;
      gs[q] = GS + row;
      go[q] = GO + row;
      h[q] = f[e[q].y * M];
    }
#pragma unroll
    for (int w = 0; w < NI; ++w) {
      for (uint64_t y = same[w]; y; y &= y - 1) {
        const int o = __ffsll((unsigned long long)y) - 1;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double g = (double)gs[q][64 * w + o];
          h[q] += (hs[w] >> o) & 1 ? -g : g;
        }
      }
      for (uint64_t y = other[w]; y; y &= y - 1) {
        const int o = __ffsll((unsigned long long)y) - 1;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double g = (double)go[q][64 * w + o];
          h[q] += (ho[w] >> o) & 1 ? -g : g;
        }
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (k + q >= b1 || (int)e[q].y == i) continue;
      const double t = flip(h[q], e[q].x & kSign);
      const T *src = u + (int64_t)(e[q].x & ~kSign) * NST;
#pragma unroll
      for (int st = 0; st < NST; ++st) acc[st] += t * (double)src[st];
    }
  }
#pragma unroll
  for (int st = 0; st < NST; ++st) part[p * NST + st] = (T)flip(acc[st], own & kSign);
}

// what a sum that is not finite is formed again from
template <typename T>
struct EntryTable {
  const uint2 *ent;
  const uint32_t *off;
  const int2 *wave;
  const T *tab;
  int64_t n_dbl;
  int M, npo;
  uint32_t tab2;
};

// Sum of the off-diagonal terms of a determinant's state, without the pairs that
// are not connected: the doubles kernel multiplies an infinity or NaN of u by
// their zeros.
template <typename T, int NST>
__device__ __forceinline__ double entry_sums(const EntryTable<T> &E, const int *sp, int S, const T *__restrict__ u,
                                             const T *__restrict__ part, int st) {
  auto split = [](uint32_t r, uint32_t *p, uint32_t *q) {   // pair r = (p < q)
    uint32_t t = 1;
    while ((t + 1) * t / 2 <= r) ++t;
    *q = t;
    *p = r - t * (t - 1) / 2;
  };
  double sum = 0.0;
  for (int t = 0; t < S; ++t) {
    const int at = sp[t];
    if (at < 0) continue;
    double x = (double)part[(int64_t)at * NST + st];
    if (at < E.n_dbl && !isfinite(x)) {
      const int2 d = E.wave[at >> 6];
      const int first = d.y >= 64 ? d.x : at - (at & 63) % d.y;
      const uint32_t own = E.ent[at].x, off = E.off[at], M = (uint32_t)E.M, M2 = M * M;
      const bool ab = E.ent[at].y < E.tab2;
      uint32_t i = off % M, j = off / M;
      if (!ab) split(off, &i, &j);
      x = 0.0;
      for (int n = first; n < first + d.y; ++n) {
        const uint2 e = E.ent[n];
        uint32_t a, b;
        if (ab) {
          a = e.y / (M2 * M);
          b = e.y / M2 % M;
          if (a == i || b == j) continue;
        } else {
          split((e.y - E.tab2) / (uint32_t)E.npo, &a, &b);
          if (a == i || a == j || b == i || b == j) continue;
        }
        x += (double)E.tab[e.y + off] * (double)flip(u[(int64_t)(e.x & ~kSign) * NST + st], e.x & kSign);
      }
      x = flip(x, own & kSign);
    }
    sum += x;
  }
  return sum;
}

// v and s of a determinant: 16 lanes add its entries' sums, slots l, l + 16,
// ..., then a fixed tree.  In FP64 in both precisions: an FP32 call's error
// would otherwise be that of hundreds of sums and of the list of spin exchanges
// added one by one.
template <typename T, int NST>
__global__ __launch_bounds__(256) void pair_collect_kernel(const int *__restrict__ slotpos, int S, int64_t n,
                                                           const T *__restrict__ part, const int *__restrict__ xptr,
                                                           const uint32_t *__restrict__ xlist,
                                                           const double *__restrict__ hdiag,
                                                           const double *__restrict__ sdiag, const T *__restrict__ u,
                                                           EntryTable<T> E, T *__restrict__ v, T *__restrict__ s) {
  const int64_t k = blockIdx.x * (int64_t)16 + (threadIdx.x >> 4);
  const int l = threadIdx.x & 15;
  const bool on = k < n;
  double acc[NST];
#pragma unroll
  for (int st = 0; st < NST; ++st) acc[st] = 0.0;
  if (on) {
    const int *sp = slotpos + k * S;
    for (int t = l; t < S; t += 64) {
      int at[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) at[q] = t + 16 * q < S ? sp[t + 16 * q] : -1;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (at[q] >= 0)
#pragma unroll
          for (int st = 0; st < NST; ++st) acc[st] += (double)part[(int64_t)at[q] * NST + st];
    }
  }
#pragma unroll
  for (int st = 0; st < NST; ++st)
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) acc[st] += __shfl_xor(acc[st], o, 16);
  if (!on) return;
  // lane st writes state st of v, lane 8 + st of s
#pragma unroll
  for (int st = 0; st < NST; ++st) {
    const double x = (double)u[k * NST + st];
    if (l == st) {
      double t = acc[st];
      if (!isfinite(t)) t = entry_sums<T, NST>(E, slotpos + k * S, S, u, part, st);
      v[k * NST + st] = (T)(t + hdiag[k] * x);
    }
    if (l == 8 + st) {
      double t = sdiag[k] * x;
      for (int q = xptr[k]; q < xptr[k + 1]; ++q) {
        const uint32_t e = xlist[q];
        t += (double)flip(u[(int64_t)(e & ~kSign) * NST + st], e & kSign);
      }
      s[k * NST + st] = (T)t;
    }
  }
}

// ---------------------------------------------------------------- host
// room for n: an earlier wavefunction's if it is not far too much
template <typename T>
void reserve(DBuf<T> &b, size_t n) {
  if (b.n < n || b.n / 4 > n) b.alloc(n);
}

struct ClassBuild {
  ClassArgs C;
  int64_t n = 0;
  int *orig, *sid, *start, *place;
};

// sorts one class's entries by bucket; the number of buckets to *count
void sort_class(qpx_ctx *c, Arena &A, const SortScratch &Z, ClassBuild &B, uint64_t max_key, int *count) {
  Wfn &W = c->W;
  hipStream_t s = c->stream;
  const int64_t n = B.n;
  if (n == 0) return;
  const int g = grid_for(n);
  if (A.base) {
    hipLaunchKernelGGL(pair_key_kernel, dim3(g), dim3(256), 0, s, B.C, W.csc_a.p, W.csc_b.p, n, Z.k1, Z.v1);
    QPX_HIP(hipGetLastError());
  }
  sort_pairs(A, Z.k1, Z.k2, Z.v1, B.orig, n, bits_of(max_key), s);
  if (A.base) hipLaunchKernelGGL(pair_head_kernel, dim3(g), dim3(256), 0, s, Z.k2, n, Z.v1);
  scan<true>(A, Z.v1, B.sid, n, s);
  if (!A.base) return;
  hipLaunchKernelGGL(pair_start_kernel, dim3(g), dim3(256), 0, s, Z.v1, B.sid, n, B.start);
  QPX_HIP(hipGetLastError());
  copy_int(B.sid + (n - 1), count, s);
}

// positions of its nseg buckets; the room they take, and of it that of the
// buckets of kSplit and more, to count[0], count[1]
void place_class(Arena &A, const SortScratch &Z, ClassBuild &B, int nseg, int *first, int *count, hipStream_t s) {
  const int64_t n = B.n;
  if (n == 0) return;
  uint32_t *sz = reinterpret_cast<uint32_t *>(Z.k1), *sz2 = sz + nseg;
  int *id = reinterpret_cast<int *>(Z.k2), *id2 = id + nseg;
  const int g = grid_for(nseg);
  if (A.base) {
    hipLaunchKernelGGL(pair_size_kernel, dim3(g), dim3(256), 0, s, B.start, nseg, n, sz, id);
    QPX_HIP(hipGetLastError());
  }
  sort_pairs(A, sz, sz2, id, id2, nseg, bits_of((uint64_t)n), s, true);
  if (A.base) {
    hipLaunchKernelGGL(pair_first_kernel, dim3(g), dim3(256), 0, s, sz2, nseg, first);
    hipLaunchKernelGGL(pair_room_kernel, dim3(g), dim3(256), 0, s, sz2, nseg, first, id);
  }
  scan<false>(A, id, Z.v1, nseg, s);
  if (!A.base) return;
  hipLaunchKernelGGL(pair_place_kernel, dim3(g), dim3(256), 0, s, id2, Z.v1, id, sz2, nseg, first, B.place, count);
  QPX_HIP(hipGetLastError());
}

template <int NI>
bool build(qpx_ctx *c) {
  Wfn &W = c->W;
  PairIdx &X = W.pr;
  hipStream_t s = c->stream;
  const int na = c->H.na, nb = c->H.nb, M = c->H.M, npo = M * (M - 1) / 2;
  const int na2 = na * (na - 1) / 2, nb2 = nb * (nb - 1) / 2;
  const int nslot[5] = {na * nb, na2, nb2, na, nb};
  X.S = nslot[0] + nslot[1] + nslot[2] + nslot[3] + nslot[4];
  int64_t nmax = 1;
  ClassBuild B[5];
  const uint32_t tab2 = (uint32_t)((int64_t)M * M * M * M);
  int slot0 = 0;
  for (int q = 0; q < 5; ++q) {
    B[q].n = W.n_det * nslot[q];
    if (B[q].n >= ((int64_t)1 << 31)) return false;
    nmax = std::max(nmax, B[q].n);
    B[q].C = ClassArgs{q, nslot[q], nullptr, nullptr, 0, 0, 1, slot0, X.S, M, npo, na, nb, tab2};
    slot0 += nslot[q];
  }
  if (W.n_det * (int64_t)X.S >= ((int64_t)1 << 33)) return false;
  int cnt[4] = {0, 0, 0, 0}, nseg[5] = {0, 0, 0, 0, 0}, room[10] = {0};
  Arena A;
  int *d_cnt, *first, *sa1, *sa2, *sb1, *sb2, *cx;
  SortScratch Z;
  // the first pass only adds up the scratch
  for (int pass = 0; pass < 2; ++pass) {
    if (pass) {
      const size_t bytes = A.used + A.tmp_n + 256;
      A.base = c->ws_pairs.get(bytes, s);
      A.used = 0;
    }
    d_cnt = A.take<int>(32);
    first = A.take<int>(64);
    sa1 = A.take<int>((size_t)W.n_a * na);
    sa2 = A.take<int>((size_t)W.n_a * na2);
    sb1 = A.take<int>((size_t)W.n_b * nb);
    sb2 = A.take<int>((size_t)W.n_b * nb2);
    cx = A.take<int>(W.n_det + 1);
    Z.k1 = A.take<uint64_t>(nmax);
    Z.k2 = A.take<uint64_t>(nmax);
    Z.v1 = A.take<int>(nmax);
    Z.v2 = A.take<int>(nmax);
    for (int q = 0; q < 5; ++q) {
      B[q].orig = A.take<int>(B[q].n);
      B[q].sid = A.take<int>(B[q].n);
      B[q].start = A.take<int>(B[q].n);
      B[q].place = A.take<int>(B[q].n);
    }
    if (pass) {
      A.tmp = A.take<char>(A.tmp_n);
      QPX_HIP(hipMemsetAsync(d_cnt, 0, sizeof(int) * 32, s));
    }
    substring_ids<NI>(A, Z, W.astr.p, W.n_a, M, na, 1, sa1, d_cnt, s);
    substring_ids<NI>(A, Z, W.astr.p, W.n_a, M, na, 2, sa2, d_cnt + 1, s);
    substring_ids<NI>(A, Z, W.bstr.p, W.n_b, M, nb, 1, sb1, d_cnt + 2, s);
    substring_ids<NI>(A, Z, W.bstr.p, W.n_b, M, nb, 2, sb2, d_cnt + 3, s);
    if (pass) read_ints(d_cnt, 4, cnt, s);
    auto ids = [](ClassArgs &C, const int *sa, int nsa, const int *sb, int nsb, int64_t mult) {
      C.sa = sa; C.nsa = nsa; C.sb = sb; C.nsb = nsb; C.mult = std::max<int64_t>(1, mult);
    };
    ids(B[0].C, sa1, na, sb1, nb, cnt[2]);
    ids(B[1].C, sa2, na2, nullptr, 0, W.n_b);
    ids(B[2].C, nullptr, 0, sb2, nb2, cnt[3]);
    ids(B[3].C, sa1, na, nullptr, 0, W.n_b);
    ids(B[4].C, nullptr, 0, sb1, nb, cnt[2]);
    const int hi[5] = {cnt[0], cnt[1], W.n_a, cnt[0], W.n_a};
    for (int q = 0; q < 5; ++q)
      sort_class(c, A, Z, B[q], pass ? (uint64_t)std::max(1, hi[q]) * (uint64_t)B[q].C.mult : ~0ULL, d_cnt + 4 + q);
    if (pass) read_ints(d_cnt + 4, 5, nseg, s);
    for (int q = 0; q < 5; ++q) place_class(A, Z, B[q], pass ? nseg[q] : (int)B[q].n, first, d_cnt + 9 + 2 * q, s);
    if (pass) {
      read_ints(d_cnt + 9, 10, room, s);
      for (int q = 0; q < 5; ++q)
        if (room[2 * q] < 0) return false;   // less than twice the entries, but 2^31 and more
    }
    if (!pass) scan<false>(A, cx, cx, W.n_det + 1, s);
  }
  // the doubles' large buckets, their small ones, the singles
  int64_t total = 0, big[5], small[5];
  for (int q = 0; q < 3; ++q) {
    big[q] = total;
    total += room[2 * q + 1];
  }
  const int64_t n_big = total;
  for (int q = 0; q < 5; ++q) {
    if (q >= 3) {
      total = (total + 255) / 256 * 256;   // a workgroup of the singles has one spin
      if (q == 3) X.n_dbl = total;
      else X.alpha_end = total;
      big[q] = total;
      total += room[2 * q + 1];
    }
    small[q] = total - room[2 * q + 1];
    total += room[2 * q] - room[2 * q + 1];
  }
  total = (total + 255) / 256 * 256;
  if (total >= ((int64_t)1 << 31)) return false;
  // what stays for this wavefunction, beside what its callers still need
  size_t free_b = 0, total_b = 0;
  QPX_HIP(hipMemGetInfo(&free_b, &total_b));
  const size_t keep = (size_t)total * (sizeof(uint2) + sizeof(uint32_t) + sizeof(double) * kMaxState) +
                      sizeof(int) * (size_t)W.n_det * X.S;
  if (keep > free_b / 2) return false;
  X.n_big = n_big;
  X.n_all = total;
  const size_t n1 = std::max<int64_t>(total, 256);
  reserve(X.ent, n1);
  reserve(X.off, n1);
  reserve(X.wave, n1 / 64);
  reserve(X.slotpos, (size_t)W.n_det * X.S);
  reserve(X.xptr, W.n_det + 1);
  QPX_HIP(hipMemsetAsync(X.wave.p, 0, sizeof(int2) * (n1 / 64), s));
  QPX_HIP(hipMemsetAsync(X.ent.p, 0, sizeof(uint2) * n1, s));   // positions without an entry
  QPX_HIP(hipMemsetAsync(X.off.p, 0, sizeof(uint32_t) * n1, s));
  for (int q = 0; q < 5; ++q)
    if (B[q].n) {
      hipLaunchKernelGGL(pair_fill_kernel<NI>, dim3(grid_for(B[q].n)), dim3(256), 0, s, B[q].C, B[q].orig, B[q].sid,
                         B[q].start, B[q].place, B[q].n, nseg[q], W.csc_a.p, W.csc_b.p, W.astr.p, W.bstr.p,
                         (int)big[q], (int)small[q], EntryArrays{X.ent.p, X.off.p, X.wave.p, X.slotpos.p});
      QPX_HIP(hipGetLastError());
    }
  // spin exchanges
  const int g = grid_for(W.n_det);
  hipLaunchKernelGGL(exchange_kernel<NI>, dim3(g), dim3(256), 0, s, W.csc_a.p, W.csc_b.p, W.col_ptr.p, W.astr.p, W.n_a,
                     W.bstr.p, W.n_b, W.n_det, (const int *)nullptr, cx, (uint32_t *)nullptr);
  QPX_HIP(hipMemsetAsync(cx + W.n_det, 0, sizeof(int), s));
  QPX_HIP(hipGetLastError());
  scan<false>(A, cx, X.xptr.p, W.n_det + 1, s);
  int nx = 0;   // at most as many as alpha/beta slots
  read_ints(X.xptr.p + W.n_det, 1, &nx, s);
  reserve(X.xlist, std::max(nx, 1));
  hipLaunchKernelGGL(exchange_kernel<NI>, dim3(g), dim3(256), 0, s, W.csc_a.p, W.csc_b.p, W.col_ptr.p, W.astr.p, W.n_a,
                     W.bstr.p, W.n_b, W.n_det, (const int *)X.xptr.p, cx, X.xlist.p);
  QPX_HIP(hipGetLastError());
  QPX_HIP(hipStreamSynchronize(s));
  X.valid = true;
  return true;
}

template <typename T>
void build_table(qpx_ctx *c, DBuf<T> &tab) {
  Ham &H = c->H;
  if (tab.p) return;
  const int M = H.M, npo = M * (M - 1) / 2;
  const int64_t n = (int64_t)M * M * M * M + (int64_t)npo * npo;
  tab.alloc(n);
  if (!H.Pf.p) {
    H.Pf.alloc((size_t)2 * M * M);
    hipLaunchKernelGGL(fock_table_kernel, dim3(64), dim3(256), 0, c->stream, H.hcore.p, H.GS.p, H.GO.p, M, H.na, H.nb,
                       H.Pf.p);
  }
  hipLaunchKernelGGL(pair_table_kernel<T>, dim3(grid_for(n)), dim3(256), 0, c->stream, H.V.p, M, H.npair, npo, tab.p);
  QPX_HIP(hipGetLastError());
  QPX_HIP(hipStreamSynchronize(c->stream));
}

template <typename T, int NI, int NST>
void launch(qpx_ctx *c, char *ws, const T *tab, const double *fock, const T *u, T *v, T *s, hipStream_t st) {
  Wfn &W = c->W;
  PairIdx &X = W.pr;
  const bool f64 = std::is_same<T, double>::value;
  const T *GS = f64 ? (const T *)c->H.GS.p : (const T *)c->H.GSf.p;
  const T *GO = f64 ? (const T *)c->H.GO.p : (const T *)c->H.GOf.p;
  T *part = (T *)ws;
  const int64_t nbig = X.n_big / 64, nsmall = (X.n_dbl - X.n_big + 255) / 256;
  if (X.n_dbl)
    hipLaunchKernelGGL((pair_doubles_kernel<T, NST>), dim3((unsigned)(nbig + nsmall)), dim3(256), 0, st, X.ent.p, X.off.p,
                       X.wave.p, (int)nbig, (int)(X.n_dbl / 64), tab, u, part);
  const int64_t ns = X.n_all - X.n_dbl;
  if (ns) {
    SingleArgs A{W.csc_a.p, W.csc_b.p, W.astr.p, W.bstr.p, X.alpha_end, c->H.M, c->H.na, c->H.nb};
    hipLaunchKernelGGL((pair_singles_kernel<T, NI, NST>), dim3((unsigned)(ns / 256)), dim3(256), 0, st, A, X.n_dbl,
                       X.ent.p, X.off.p, X.wave.p, fock, GS, GO, u, part);
  }
  const int M = c->H.M;
  const EntryTable<T> E{X.ent.p, X.off.p, X.wave.p, tab, X.n_dbl, M, M * (M - 1) / 2, (uint32_t)((int64_t)M * M * M * M)};
  hipLaunchKernelGGL((pair_collect_kernel<T, NST>), dim3((unsigned)((W.n_det + 15) / 16)), dim3(256), 0, st, X.slotpos.p,
                     X.S, W.n_det, part, X.xptr.p, X.xlist.p, W.hdiag.p, W.sdiag.p, u, E, v, s);
  QPX_HIP(hipGetLastError());
}

template <typename T, int NI>
void launch_nst(qpx_ctx *c, int nst, char *ws, const T *tab, const double *fock, const T *u, T *v, T *s, hipStream_t st) {
  switch (nst) {
    case 1: launch<T, NI, 1>(c, ws, tab, fock, u, v, s, st); break;
    case 2: launch<T, NI, 2>(c, ws, tab, fock, u, v, s, st); break;
    case 3: launch<T, NI, 3>(c, ws, tab, fock, u, v, s, st); break;
    case 4: launch<T, NI, 4>(c, ws, tab, fock, u, v, s, st); break;
    case 5: launch<T, NI, 5>(c, ws, tab, fock, u, v, s, st); break;
    case 6: launch<T, NI, 6>(c, ws, tab, fock, u, v, s, st); break;
    case 7: launch<T, NI, 7>(c, ws, tab, fock, u, v, s, st); break;
    default: launch<T, NI, 8>(c, ws, tab, fock, u, v, s, st); break;
  }
}

template <typename T>
void launch_ni(qpx_ctx *c, int nst, char *ws, const T *tab, const double *fock, const T *u, T *v, T *s, hipStream_t st) {
  switch (c->W.nint) {
    case 1: launch_nst<T, 1>(c, nst, ws, tab, fock, u, v, s, st); break;
    case 2: launch_nst<T, 2>(c, nst, ws, tab, fock, u, v, s, st); break;
    default: launch_nst<T, 3>(c, nst, ws, tab, fock, u, v, s, st); break;
  }
}

}  // namespace

namespace qpx {

// False when the entries, their sums or the integral table do not fit: the
// caller then walks the buckets determinant by determinant (sigma_sparse.hip).
// What the call began and could not finish goes again; what is complete stays,
// for the calls and captured graphs that use it (the walk's set-up gives it up
// if it needs the room).  Entries that do not fit are not tried again for this
// wavefunction; a table or sums (of a precision, of a number of states) are,
// which costs an allocation.
bool sigma_pairs(qpx_ctx *c, int prec, int nst, const void *u, void *v, void *s, hipStream_t st) {
  Wfn &W = c->W;
  Ham &H = c->H;
  // a wavefront per determinant is the faster one for few entries (20,000: 28
  // against 33 us, 42,000: 96 against 76, 60,000: 53 against 22)
  if (c->force_path == 0 && W.n_det * (int64_t)(H.na * H.nb + H.na * (H.na + 1) / 2 + H.nb * (H.nb + 1) / 2) < 32768)
    return false;
  if (H.M > kG4MaxOrb || nst > kMaxState || H.na > kMaxElec || H.nb > kMaxElec || H.na < 1 || H.nb < 1) return false;
  if (W.pr.failed) return false;
  const bool f64 = prec == QPX_FP64;
  const bool had_entries = W.pr.valid;
  bool table = f64 ? H.Pt.p != nullptr : H.Ptf.p != nullptr, entries = had_entries;
  auto drop = [&] {
    if (!entries) {
      W.pr.release();
      c->ws_pairs.release();
    }
    if (table) return;
    if (f64) H.Pt.release();
    else H.Ptf.release();
  };
  char *ws = nullptr;
  bool ok = false, failed = false;   // failed: the entries do not fit
  try {
    if (f64) build_table<double>(c, H.Pt);
    else build_table<float>(c, H.Ptf);
    table = true;
    if (!entries) {
      failed = true;
      switch (W.nint) {
        case 1: entries = build<1>(c); break;
        case 2: entries = build<2>(c); break;
        default: entries = build<3>(c); break;
      }
      failed = !entries;
    }
    ok = entries;
    const size_t sums = (f64 ? 8 : 4) * (size_t)nst * std::max<int64_t>(W.pr.n_all, 1);
    if (ok && !had_entries) c->ws_pairs.trim(std::max(kKeepBytes, sums));   // the set-up's scratch
    if (ok) ws = c->ws_pairs.get(sums, st);
  } catch (const OutOfMemory &) {
    ok = false;
  } catch (...) {
    drop();
    throw;
  }
  if (!ok) {
    drop();
    W.pr.failed = failed;
    return false;
  }
  if (c->ktiming) QPX_HIP(hipEventRecord(c->kev[0], st));
  if (f64)
    launch_ni<double>(c, nst, ws, H.Pt.p, H.Pf.p, (const double *)u, (double *)v, (double *)s, st);
  else
    launch_ni<float>(c, nst, ws, H.Ptf.p, H.Pf.p, (const float *)u, (float *)v, (float *)s, st);
  if (c->ktiming) {
    QPX_HIP(hipEventRecord(c->kev[1], st));
    QPX_HIP(hipEventRecord(c->kev[2], st));
  }
  c->ws_pairs.used(st);
  return true;
}

}  // namespace qpx
