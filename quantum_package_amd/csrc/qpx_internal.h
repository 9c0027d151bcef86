// qpx_internal.h -- shared state of libqpx (MI355X / gfx950).
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdint>
#include <string>
#include <memory>
#include <vector>
#include <stdexcept>
#include "../../include/qpx.h"

namespace qpx {

struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};

// No device memory for an allocation: a sigma call then takes a path that
// needs less.  Every other error reaches the caller.
struct OutOfMemory : Error {
  using Error::Error;
};

#define QPX_HIP(call)                                                                          \
  do {                                                                                         \
    hipError_t e_ = (call);                                                                    \
    if (e_ != hipSuccess)                                                                      \
      throw ::qpx::Error(2, std::string("HIP error ") + hipGetErrorString(e_) + " at " +       \
                                __FILE__ + ":" + std::to_string(__LINE__) + " (" #call ")");   \
  } while (0)

#define QPX_REQUIRE(cond, msg)                                                                 \
  do {                                                                                         \
    if (!(cond)) throw ::qpx::Error(1, std::string(msg));                                      \
  } while (0)

constexpr int NINT_MAX = 4;
// largest orbital count for which the M^4 integral table (Ham::G4) is built:
// 8 + 4 bytes per entry, 7.9 GB at 160 orbitals; above it the kernels read
// the pair matrix
constexpr int kG4MaxOrb = 160;

// Test hook (qpx_debug_fail_alloc): allocations of this thread above
// fail_above bytes end with fail_with.
inline thread_local size_t fail_above = SIZE_MAX;
inline thread_local hipError_t fail_with = hipErrorOutOfMemory;

inline void device_alloc(void **p, size_t bytes) {
  const hipError_t e = bytes > fail_above ? fail_with : hipMalloc(p, bytes);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    *p = nullptr;
    throw OutOfMemory(2, "HIP error out of memory: " + std::to_string(bytes) + " bytes of device memory");
  }
  QPX_HIP(e);
}

// Waits for the device.  hipDeviceSynchronize would fail while any thread of the
// process captures a stream, and break its capture; hipFree, which waits too, is
// refused only where an allocation is (a capture in the global mode).
inline void wait_device() {
  void *p = nullptr;
  device_alloc(&p, 256);
  QPX_HIP(hipFree(p));
}

// What a context keeps of one wavefunction's arrays and scratch for the next, of
// the bucket kernels and of the string-driven ones; more costs less to allocate
// again than the set-up it serves (some 10^8 entries to sort).
constexpr size_t kKeepBytes = (size_t)4 << 30;
constexpr size_t kKeepFci = (size_t)64 << 20;   // tables of a product space: what allocations cost shows in small ones

// Device buffer with RAII.
template <typename T>
struct DBuf {
  T *p = nullptr;
  size_t n = 0;
  DBuf() = default;
  DBuf(const DBuf &) = delete;
  DBuf &operator=(const DBuf &) = delete;
  ~DBuf() { release(); }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  void alloc(size_t count) {
    if (count == n && p) return;
    release();
    if (count == 0) return;
    device_alloc((void **)&p, count * sizeof(T));
    n = count;
  }
  void upload(const T *h, size_t count, hipStream_t s) {
    alloc(count);
    if (count) QPX_HIP(hipMemcpyAsync(p, h, count * sizeof(T), hipMemcpyHostToDevice, s));
  }
  void upload(const std::vector<T> &v, hipStream_t s) { upload(v.data(), v.size(), s); }
};

// Hamiltonian tables on the device.
//   V[P*npair + R] = (pq|rs) with P = pair(p,q), R = pair(r,s) (0-based
//   packed pair index P = max(max+1)/2 + min over 0-based p,q).
struct Ham {
  int M = 0, na = 0, nb = 0, nint = 0, npair = 0;
  std::vector<double> h;          // M*M column-major
  std::vector<double> eri;        // packed n8
  DBuf<double> V;                 // npair^2
  DBuf<float> Vf;
  DBuf<double> hcore;             // M*M
  DBuf<float> hcoref;
  DBuf<double> Jd, Kd;            // M*M: J_ij=(ii|jj), K_ij=(ij|ji)
  DBuf<double> JAd;               // M*M: J_ij - K_ij (mo_bielec_integral_jj_anti)
  DBuf<double> fock_cs;           // M*M fock_operator_closed_shell_ref_bitmask
  DBuf<int> ptab;                 // M*M pair index
  DBuf<double> GS, GO;            // M^3 single-excitation tables (context.hip)
  DBuf<float> GSf, GOf;
  // M^4 table G4[((i*M + j)*M + y)*M + x] = (ix|jy), built on first use by
  // the sparse sigma path when M <= kG4MaxOrb (ensure_g4)
  DBuf<double> G4;
  DBuf<float> G4f;
  // integrals (per precision, on first use) and HF elements of the
  // bucket-by-bucket sparse sigma (sigma_pairs.hip)
  DBuf<double> Pt, Pf;
  DBuf<float> Ptf;
  void release_pair_tables() {
    Pt.release();
    Pf.release();
    Ptf.release();
  }
  double ref_energy = 0.0;        // ref_bitmask_energy of the HF determinant
};

// Small arrays laid out one after another in one allocation: a dozen allocations
// cost as much as ten sigma calls of a small space.  Arrays of 1 MB and more get
// memory of their own (one block of several MB took 0.2 ms longer).  lay() runs
// twice, first to add up the size, then to hand out the addresses.
template <typename T>
struct View {
  T *p = nullptr;
};
struct Block {
  DBuf<char> mem;
  std::vector<std::unique_ptr<DBuf<char>>> own;
  size_t used = 0, n_own = 0;
  bool sizing = true;
  // memory that is large enough stays, unless it is far too large
  static void reserve(DBuf<char> &b, size_t n) {
    if (b.n < n || b.n / 4 > std::max(n, (size_t)1 << 20)) b.alloc(n);
  }
  template <typename T>
  void lay(View<T> &v, size_t count) {
    const size_t n = (std::max<size_t>(count, 1) * sizeof(T) + 255) / 256 * 256;
    if (n >= (size_t)1 << 20) {
      if (n_own == own.size()) own.push_back(std::make_unique<DBuf<char>>());
      DBuf<char> &b = *own[n_own++];
      if (sizing) reserve(b, n);
      else v.p = reinterpret_cast<T *>(b.p);
      return;
    }
    if (!sizing) v.p = reinterpret_cast<T *>(mem.p + used);
    used += n;
  }
  size_t bytes() const {
    size_t n = mem.n;
    for (const auto &b : own) n += b->n;
    return n;
  }
  void release() {
    mem.release();
    own.clear();
  }
  template <typename F>
  void layout(F f) {   // f(): the lay() calls
    for (bool first : {true, false}) {
      sizing = first;
      used = n_own = 0;
      f();
      if (first) {
        reserve(mem, used);
        own.resize(n_own);
      }
    }
  }
};

// Connectivity of unique spin strings (within the unique set).
struct SpinConn {
  View<int> s_ptr, s_idx;         // singles: CSR over strings
  View<uint32_t> s_info;          // h | p<<8 | (phase<0)<<16 (0-based orbitals)
  View<double> s_val;             // same-spin part of the single element, phase included
  View<float> s_valf;
  View<int> d_ptr, d_idx;         // doubles
  View<double> d_val;             // full same-spin double element, phase included
  View<float> d_valf;
  int max_singles = 0, max_doubles = 0;
  int64_t n_singles = 0, n_doubles = 0;
};

// Sub-string buckets of the sparse sigma path (sigma_sparse.hip): per
// excitation class, the sorted entries (determinant | removed orbitals) and,
// per (determinant, slot), the range of its bucket.
struct Buckets {
  int nslot = 0;
  int64_t visited = 0;   // sum of squared bucket sizes
  DBuf<uint64_t> pay;
  DBuf<int2> range;
};
struct SparseIdx {
  bool valid = false;
  DBuf<int> a1, a2, b1, b2;   // sub-string ids per unique string
  Buckets cls[5];             // ab, a1, a2, b1, b2
  void clear() {
    valid = false;
    a1.release(); a2.release(); b1.release(); b2.release();
    for (auto &b : cls) { b.pay.release(); b.range.release(); b.nslot = 0; }
  }
};

// Tables of the string-driven sigma of product spaces (sigma_fci.hip), built
// on first use: partners of 16 strings at a time, their matrix elements and
// the placement tables, per precision.
struct FciConn {   // connections and elements, for sums that are not finite
  const int *as_ptr, *as_idx, *ad_ptr, *ad_idx, *bd_ptr, *bd_idx;
  const uint32_t *as_info;
  const void *as_val, *ad_val, *bs_val, *bd_val;
};
struct SpinTiles {
  int ntile = 0;
  int64_t nchunk = 0;    // room for the partners of all tiles, in chunks of 8
  View<int2> range;      // chunks of a tile
  View<int> idx;
};
template <typename T>
struct FciTables {
  bool valid = false;
  Block mem;
  View<T> coef_a, coef_b, gb, vo;
  View<uint4> tgt;
  View<FciConn> conn;
  void release() {
    valid = false;
    mem.release();
  }
};
struct FciPlan {
  bool valid = false;
  int lda = 0, ldb = 0, ldt = 0;
  Block mem, lists;      // maps and ranges; partners
  View<uint32_t> map_a, map_b;
  SpinTiles a, b;
  FciTables<double> t64;
  FciTables<float> t32;
  void clear() {   // the next wavefunction may take the memory
    valid = t64.valid = t32.valid = false;
    if (mem.bytes() + lists.bytes() + t64.mem.bytes() + t32.mem.bytes() > kKeepFci) release();
  }
  void release() {
    valid = false;
    mem.release();
    lists.release();
    t64.release();
    t32.release();
  }
};

// Entries of the bucket-by-bucket sparse sigma (sigma_pairs.hip): double
// excitations [0, n_dbl), those of buckets of 64 and more in front, alpha singles [n_dbl, alpha_end), beta singles
// [alpha_end, n_all).
struct PairIdx {
  bool valid = false, failed = false;
  int64_t n_big = 0, n_dbl = 0, alpha_end = 0, n_all = 0;
  int S = 0;                  // slots of a determinant
  DBuf<uint2> ent;
  DBuf<uint32_t> off, xlist;
  DBuf<int2> wave;            // buckets of a wavefront's 64 entries
  DBuf<int> slotpos, xptr;    // entry of each slot; spin exchanges of each determinant
  void clear() { valid = failed = false; }   // the next wavefunction may take the arrays
  size_t bytes() const {
    return ent.n * sizeof(uint2) + wave.n * sizeof(int2) + (off.n + xlist.n + slotpos.n + xptr.n) * sizeof(int);
  }
  void release() {
    clear();
    ent.release(); off.release(); xlist.release(); wave.release(); slotpos.release(); xptr.release();
  }
};

struct Wfn {
  int64_t n_det = 0;
  int nint = 0;
  int n_a = 0, n_b = 0;
  bool valid = false;
  std::vector<uint64_t> astr_h, bstr_h;   // unique strings (n*nint)
  std::vector<int64_t> perm;              // bilinear position -> psi index
  DBuf<uint64_t> psi;                     // determinants in psi order (n_det, 2, nint)
  DBuf<uint64_t> astr, bstr;
  DBuf<int> col_ptr, csc_a, csc_b;        // CSC by beta column; entries sorted by alpha
  DBuf<int> row_ptr, csr_b, csr2csc;      // CSR by alpha row; entries sorted by beta
  DBuf<int64_t> perm_d;                   // bilinear position -> psi index
  SpinConn ca, cb;               // built on first use by the dense-map or scan path (ensure_conn)
  bool conn_valid = false;
  DBuf<double> hdiag, sdiag;              // bilinear order
  // per-string scan costs for the generic alpha/beta kernel
  View<int64_t> cost_a, cost_b;
  DBuf<int> conn_count;                   // singles and doubles per string
  Block conn;                             // ca, cb and the costs
  std::vector<int> col_len_h, row_len_h;
  int max_col = 0, max_row = 0;
  SparseIdx sp;                           // built on first use of the sparse path
  PairIdx pr;                             // built on first use of the sparse path
  FciPlan fci;                            // built on first use of the product-space path
};

struct Workspace {
  DBuf<char> buf;
  char *get(size_t bytes) {
    if (buf.n < bytes) buf.alloc(bytes + (bytes >> 3));
    return buf.p;
  }
};

inline bool capturing(hipStream_t s, unsigned long long *id = nullptr) {
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  unsigned long long x = 0;
  if (hipStreamGetCaptureInfo(s, &cs, &x) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  if (id) *id = x;
  return cs != hipStreamCaptureStatusNone;
}

// While s is captured, lets this thread allocate and wait on other streams:
// tables and scratch that a captured call is the first to need are made beside
// the graph.
struct RelaxedCapture {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  bool on;
  explicit RelaxedCapture(hipStream_t s) : on(capturing(s)) {
    if (on) QPX_HIP(hipThreadExchangeStreamCaptureMode(&mode));
  }
  ~RelaxedCapture() {
    if (on) (void)hipThreadExchangeStreamCaptureMode(&mode);
  }
  RelaxedCapture(const RelaxedCapture &) = delete;
  RelaxedCapture &operator=(const RelaxedCapture &) = delete;
};

// Scratch of calls that are enqueued on a caller's stream and return before
// they have run: every call first waits for the last user.  On one stream that
// costs nothing; handles are not compared, since hipStreamPerThread stands for a
// stream of each thread.
struct StreamWorkspace {
  DBuf<char> buf;
  hipEvent_t done = nullptr;
  bool pending = false;
  ~StreamWorkspace() {
    if (done) (void)hipEventDestroy(done);
  }
  // A captured graph owns its scratch (one buffer per capture and stream, till
  // the wavefunction it was captured for goes or qpx_release_captured): it may be
  // replayed on any stream, beside other calls and after calls that need more.
  // The runtime tells nobody that a graph is gone: a user object retained by one
  // is not released with its last executable.
  struct Captured {
    hipStream_t s;
    unsigned long long id;
    DBuf<char> buf;
  };
  std::vector<std::unique_ptr<Captured>> graphs;
  char *get(size_t bytes, hipStream_t s) {
    unsigned long long id = 0;
    if (capturing(s, &id)) {
      for (auto &g : graphs)
        if (g->s == s && g->id == id && g->buf.n >= bytes) return g->buf.p;
      auto g = std::make_unique<Captured>();
      g->s = s;
      g->id = id;
      g->buf.alloc(bytes);
      graphs.push_back(std::move(g));
      return graphs.back()->buf.p;
    }
    if (pending) QPX_HIP(hipStreamWaitEvent(s, done, 0));
    // hipFree waits for the device, so the old buffer is not in use any more
    if (buf.n < bytes) buf.alloc(bytes);
    return buf.p;
  }
  void release() {
    buf.release();
    pending = false;
  }
  void trim(size_t keep) {
    if (buf.n > keep) release();
  }
  void used(hipStream_t s) {
    if (capturing(s)) return;
    if (!done) QPX_HIP(hipEventCreateWithFlags(&done, hipEventDisableTiming));
    QPX_HIP(hipEventRecord(done, s));
    pending = true;
  }
};

}  // namespace qpx

struct qpx_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  qpx::Ham H;
  qpx::Wfn W;
  bool ham_set = false;
  int lds_per_block = 65536;
  int n_cu = 256;
  qpx::Workspace ws_sigma_io;   // host-order u/v/s staging for qpx_sigma
  qpx::Workspace ws_sigma_t;    // transposed u_t/v_t/s_t
  qpx::Workspace ws_misc;
  qpx::StreamWorkspace ws_pairs;  // sums of the entries (sigma_pairs.hip)
  qpx::StreamWorkspace ws_fci;  // planes of u and the same-spin part (sigma_fci.hip)
  int64_t sel_stats[4] = {0, 0, 0, 0};
  std::vector<int64_t> sel_ticks;   // per-block durations of the last selection (benchmark hook)
  int sigma_path = 0;           // last sigma path: 1 = string-driven or dense map, 2 = generic scan, 3 = sparse buckets
  int sigma_kernels = 0;        // its kernels, numbered as the forced paths (qpx_debug.h)
  int force_path = 0;           // 0 auto, else the path to use (tests)
  int verbosity = 0;            // 1: Davidson iteration table on stderr
  hipEvent_t kev[3] = {nullptr, nullptr, nullptr};  // per-kernel timing (benchmark hook)
  bool ktiming = false;
};

namespace qpx {
// implemented in context.hip: builds Ham::G4/G4f if M <= kG4MaxOrb and
// returns whether the table exists
bool ensure_g4(qpx_ctx *c);
// implemented in wavefunction.hip; ensure_conn builds the spin-string
// connectivity and scan costs of the current wavefunction if needed
void build_wavefunction(qpx_ctx *c, int n_int, int64_t n_det, const uint64_t *psi_det);
void ensure_conn(qpx_ctx *c);
// implemented in sigma.hip
void sigma_device(qpx_ctx *c, int prec, int n_st, const void *u_t, void *v_t, void *s_t, hipStream_t s);
// implemented in sigma_pairs.hip
bool sigma_pairs(qpx_ctx *c, int prec, int n_st, const void *u_t, void *v_t, void *s_t, hipStream_t s);
// implemented in sigma_fci.hip
bool fci_ok(qpx_ctx *c, int n_st, size_t tsize);
bool fci_pays(qpx_ctx *c, int n_st, size_t tsize);
bool sigma_fci(qpx_ctx *c, int prec, int n_st, const void *u_t, void *v_t, void *s_t, hipStream_t s);
// implemented in sigma_sparse.hip
bool sparse_ok(qpx_ctx *c, int n_st);
void sigma_sparse(qpx_ctx *c, int prec, int n_st, const void *u_t, void *v_t, void *s_t, hipStream_t s);
}  // namespace qpx

// Run a body, translating exceptions into return codes.
template <typename F>
static inline int qpx_guard(qpx_ctx *c, F &&f) {
  if (!c) return 1;
  try {
    f();
    return 0;
  } catch (const qpx::Error &e) {
    c->err = e.what();
    return e.code;
  } catch (const std::exception &e) {
    c->err = e.what();
    return 3;
  }
}
