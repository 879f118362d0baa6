// kpm_capi.hip -- implementation of the C-ABI in include/fastkpm_hip.h.
//
// Owns device memory and the HIP stream of one engine handle, validates every
// shape on the host before a launch, picks the kernel geometry, and sequences
// the per-step launches of the Chebyshev recursions.  The algorithms follow
// Engine_CPU (src/engine_cpu.cpp) and Engine_cuSPARSE (src/engine_cusparse.cpp)
// of the reference; the kernels are in kpm_kernels.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <type_traits>
#include <vector>


#include "fastkpm_hip.h"
#include "kpm_dispatch.h"
#include "kpm_internal.h"
// this unit defines the non-template helper kernels
#define FKD_DEFINE_HELPERS
#include "kpm_kernels.h"
#include "kpm_dots.h"
#define FKD_RES_SHARED
#include "kpm_resident.h"

namespace {

thread_local std::string g_last_error;

int fail(int code, const char* fmt, ...) {
  char buf[1024];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

#define HIPCHK(x)                                                                    \
  do {                                                                               \
    hipError_t e_ = (x);                                                             \
    if (e_ != hipSuccess) return fail(FKPM_E_HIP, "%s failed: %s (%s:%d)", #x,       \
                                      hipGetErrorString(e_), __FILE__, __LINE__);    \
  } while (0)

#define CHK(x)              \
  do {                      \
    int rc_ = (x);          \
    if (rc_ != 0) return rc_; \
  } while (0)

template <class T>
struct TypeId {
  typedef T type;
};

// One recorded kernel launch: entry, grid, block and the argument bytes.
struct LaunchRec {
  const void* fn = nullptr;
  dim3 grid, block;
  std::vector<size_t> offs;
  std::vector<unsigned char> args;
};

// While a recorder is active on this thread for a stream, launch() on that
// stream appends to it instead of launching (LaunchRecorder below replays the
// run directly or as a cached hipGraph).
struct RecSink {
  hipStream_t stream = nullptr;
  std::vector<LaunchRec>* recs = nullptr;
};
thread_local RecSink g_rec;

// Launch a kernel through its host stub with exactly its parameter types.
template <typename... P>
int launch(void (*fp)(P...), dim3 grid, dim3 block, hipStream_t st,
           typename TypeId<P>::type... args) {
  void* argv[] = {(void*)&args...};
  if (g_rec.recs != nullptr && g_rec.stream == st) {
    static constexpr size_t sz[] = {sizeof(P)...};
    static constexpr size_t al[] = {alignof(P)...};
    LaunchRec r;
    r.fn = (const void*)fp;
    r.grid = grid;
    r.block = block;
    size_t off = 0;
    for (size_t k = 0; k < sizeof...(P); k++) {
      off = (off + al[k] - 1) / al[k] * al[k];
      r.offs.push_back(off);
      off += sz[k];
    }
    r.args.resize(off);
    for (size_t k = 0; k < sizeof...(P); k++) memcpy(r.args.data() + r.offs[k], argv[k], sz[k]);
    g_rec.recs->push_back(std::move(r));
    return 0;
  }
  hipError_t e = hipLaunchKernel((const void*)fp, grid, block, argv, 0, st);
  if (e != hipSuccess) return fail(FKPM_E_HIP, "kernel launch failed: %s", hipGetErrorString(e));
  return 0;
}

// The same with dynamic LDS (never recorded: these kernels run whole loops).
template <typename... P>
int launch_lds(void (*fp)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t st,
               typename TypeId<P>::type... args) {
  if (lds > 65536) {
    const hipError_t e = hipFuncSetAttribute((const void*)fp,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return fail(FKPM_E_HIP, "%zu bytes of LDS: %s", lds, hipGetErrorString(e));
  }
  void* argv[] = {(void*)&args...};
  const hipError_t e = hipLaunchKernel((const void*)fp, grid, block, argv, lds, st);
  if (e != hipSuccess) return fail(FKPM_E_HIP, "kernel launch failed: %s", hipGetErrorString(e));
  return 0;
}

int replay_direct(const std::vector<LaunchRec>& recs, hipStream_t st) {
  std::vector<void*> argv;
  for (const LaunchRec& r : recs) {
    argv.resize(r.offs.size());
    for (size_t k = 0; k < r.offs.size(); k++)
      argv[k] = const_cast<unsigned char*>(r.args.data() + r.offs[k]);
    hipError_t e = hipLaunchKernel(r.fn, r.grid, r.block, argv.data(), 0, st);
    if (e != hipSuccess) return fail(FKPM_E_HIP, "kernel launch failed: %s", hipGetErrorString(e));
  }
  return 0;
}

// Identity of a recorded run: every launch's entry, grid and argument bytes.
uint64_t rec_hash(const std::vector<LaunchRec>& recs) {
  uint64_t x = 1469598103934665603ull;  // FNV-1a
  auto mix = [&](const void* p, size_t n) {
    const unsigned char* b = static_cast<const unsigned char*>(p);
    for (size_t i = 0; i < n; i++) x = (x ^ b[i]) * 1099511628211ull;
  };
  for (const LaunchRec& r : recs) {
    mix(&r.fn, sizeof(r.fn));
    const unsigned g[6] = {r.grid.x, r.grid.y, r.grid.z, r.block.x, r.block.y, r.block.z};
    mix(g, sizeof(g));
    mix(r.args.data(), r.args.size());
  }
  return x;
}

bool rec_equal(const std::vector<LaunchRec>& a, const std::vector<LaunchRec>& b) {
  if (a.size() != b.size()) return false;
  for (size_t k = 0; k < a.size(); k++) {
    const LaunchRec &x = a[k], &y = b[k];
    if (x.fn != y.fn || x.grid.x != y.grid.x || x.grid.y != y.grid.y || x.grid.z != y.grid.z ||
        x.block.x != y.block.x || x.block.y != y.block.y || x.block.z != y.block.z ||
        x.args != y.args)
      return false;
  }
  return true;
}

// Instantiated graphs of recorded runs, most recently used first.
struct GraphCache {
  struct Entry {
    uint64_t key;
    std::vector<LaunchRec> recs;
    hipGraphExec_t exec;
  };
  std::vector<Entry> entries;
  static constexpr size_t kMax = 16;
  void clear() {
    for (Entry& e : entries) (void)hipGraphExecDestroy(e.exec);
    entries.clear();
  }
  ~GraphCache() { clear(); }
};

struct DevBuf {
  void* p = nullptr;
  size_t bytes = 0;
  int ensure(size_t n) {
    if (n <= bytes && p != nullptr) return 0;
    if (p) {
      hipError_t e = hipFree(p);
      p = nullptr;
      bytes = 0;
      if (e != hipSuccess) return fail(FKPM_E_HIP, "hipFree: %s", hipGetErrorString(e));
    }
    if (n == 0) return 0;
    hipError_t e = hipMalloc(&p, n);
    if (e != hipSuccess) {
      p = nullptr;
      return fail(FKPM_E_HIP, "hipMalloc(%zu bytes): %s", n, hipGetErrorString(e));
    }
    bytes = n;
    return 0;
  }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
  }
  template <class T>
  T* as() const {
    return static_cast<T*>(p);
  }
};

// Pinned host memory the kernels read and write directly (small operands and
// results of a call); grows only.
struct PinBuf {
  void* p = nullptr;
  size_t bytes = 0;
  int ensure(size_t n) {
    if (n <= bytes && p != nullptr) return 0;
    release();
    const hipError_t e = hipHostMalloc(&p, n, hipHostMallocDefault);
    if (e != hipSuccess) {
      p = nullptr;
      return fail(FKPM_E_HIP, "hipHostMalloc(%zu bytes): %s", n, hipGetErrorString(e));
    }
    bytes = n;
    return 0;
  }
  void release() {
    if (p) (void)hipHostFree(p);
    p = nullptr;
    bytes = 0;
  }
};

size_t host_elem_bytes(int dtype) {
  switch (dtype) {
    case FKPM_F32: return 4;
    case FKPM_F64: return 8;
    case FKPM_C32: return 8;
    case FKPM_C64: return 16;
  }
  return 0;
}
bool dtype_complex(int dtype) { return dtype == FKPM_C32 || dtype == FKPM_C64; }
bool dtype_single(int dtype) { return dtype == FKPM_F32 || dtype == FKPM_C32; }

int grid_for(size_t n, int per_block = 256) {
  size_t g = (n + per_block - 1) / per_block;
  if (g < 1) g = 1;
  if (g > 4096) g = 4096;
  return (int)g;
}

// Validate a BSR/COO block pattern on the host.
int check_pattern(const char* what, int nb, int nnzb, const int* row_ptr, const int* row_idx,
                  const int* col_idx) {
  if (nb <= 0 || nnzb < 0) return fail(FKPM_E_ARG, "%s: bad sizes nb=%d nnzb=%d", what, nb, nnzb);
  if (!row_ptr || (nnzb > 0 && !col_idx))
    return fail(FKPM_E_ARG, "%s: null pattern array", what);
  if (row_ptr[0] != 0 || row_ptr[nb] != nnzb)
    return fail(FKPM_E_ARG, "%s: row_ptr[0]=%d row_ptr[nb]=%d, expected 0 and %d", what,
                row_ptr[0], row_ptr[nb], nnzb);
  for (int i = 0; i < nb; i++) {
    if (row_ptr[i + 1] < row_ptr[i]) return fail(FKPM_E_ARG, "%s: row_ptr not monotone at %d", what, i);
    for (int p = row_ptr[i]; p < row_ptr[i + 1]; p++) {
      if (col_idx[p] < 0 || col_idx[p] >= nb)
        return fail(FKPM_E_ARG, "%s: col_idx[%d]=%d out of range [0,%d)", what, p, col_idx[p], nb);
      if (row_idx && row_idx[p] != i)
        return fail(FKPM_E_ARG, "%s: row_idx[%d]=%d inconsistent with row_ptr (row %d)", what, p,
                    row_idx[p], i);
    }
  }
  return 0;
}

// Kernel kinds with a geometry of their own.
// K_MOMT / K_ADS: the forward step writing the table of forward vectors and
// the backward step reading it (tuned apart: a step that writes a fresh
// vector per launch meets the caches differently from one cycling a ring).
enum KKind { K_MOM = 0, K_XI = 1, K_AD = 2, K_OUT = 3, K_MOMT = 4, K_ADS = 5, NKIND = 6 };

// Geometry of one kernel kind: lanes per block row, packets per lane,
// workgroup cap and nontemporal bits; nwg/chunk derived from them.
struct KCfg {
  int L = 0, KQ = 0, maxwg = 0, nt = 0;
  int mfma = 0;  // matrix-core kernel (one wave per block row: L = 64, KQ = 1):
                 // 1 general, 2 row-resident (rows of <= 8 blocks, vectors < 4 GiB)
  int sweep = 0;  // rows: 0 per-XCD regions, s >= 1 one front in segments of s passes
                  // per XCD (chunk = -s, workgroups a multiple of 8 s)
  int dm = 8;     // row-resident matrix-core kernels: block slots per row (7 when no
                  // row has more than 7 blocks, else 8); set by set_kind
  int nwg = 0, chunk = 0;
};

// Most blocks per row of the row-resident matrix-core kernels (fkd::MF_DM).
constexpr int kRowResidentMax = 8;

template <class S>
fkd::RSource<S> no_rsource() {
  fkd::RSource<S> r;
  r.rd = nullptr;
  r.rcol = nullptr;
  r.rval = nullptr;
  r.cr = 0.0;
  return r;
}

}  // namespace

struct fkpm_handle {
  int device = 0;
  size_t total_bytes = 0;  // memory of the device (0: not asked yet)
  hipStream_t stream = nullptr;
  int dtype = FKPM_C64;
  int prec = FKPM_PREC_FP64;
  bool cx = true;
  bool single = false;  // storage is FP32

  // --- H (scaled) ---
  int nb = 0, b = 0, nnzb = 0, max_deg = 0;
  bool h_set = false;
  DevBuf rp, ci, hv, rowblk, hraw;
  double avg = 0.0, mag = 1.0;
  std::vector<int> h_rp, h_ci;
  bool pattern_set = false;  // the device holds the pattern of h_rp, h_ci

  // --- R and recursion state ---
  int n = 0, s = 0;
  bool r_set = false, r_dirty = true;
  DevBuf rraw;             // R as given (host layout and type)
  bool r_compact = false;  // at most one nonzero per row (probing colours)
  DevBuf rcol, rval, rflag;
  int qp = 0, sp = 0, wmax = 0, geo_b = 0;
  KCfg kc[NKIND];
  fkd::KSet<double> kd[NKIND];
  fkd::KSet<float> kf[NKIND];
  int force_L = 0, force_KQ = 0, max_wg = 0;
  bool tuned = false;
  bool autotune_on_use = false;
  bool mfma_on = true;  // matrix-core kernels where the block shape has them
  bool rr_force = false;  // FKPM_OPT_MFMA 2: row-resident ones by default wherever they exist
  int stoch_method = FKPM_STOCH_AUTO;
  int stoch_used = -1;  // method the last stoch_matrix ran (FKPM_STOCH_*)
  DevBuf R, A[3], Bv[3], xi, partial, tune_dacc;
  PinBuf psum;             // moment sums, written by the reducing kernel
  int alpha_M = 0;  // M of the moments whose final state is held, 0 if none
  DevBuf atab;            // alpha_1 .. alpha_{M/2} of the last moments(M), when it fits
  int a_slots = 0;        // moments state: alpha_1 .. alpha_{a_slots} live in atab, later ones
                          // in the ring A[3]
  int tab_K = 0;          // atab holds alpha_1 .. alpha_tab_K of the current H and R,
  int tab_M = 0;          // kept by moments(tab_M)
  int unread = 0;         // moments in a row by the step kernels that no autodiff_matrix or
                          // stoch_matrix followed
  DevBuf tabc;            // stoch_matrix weights of the table vectors
  std::vector<double> tabc_host;
  int store_alpha = 1;    // FKPM_OPT_STORE_ALPHA: 0 never, 1 auto, 2 whenever the table fits
  int sweep_force = -1;  // FKPM_OPT_SWEEP: row sweep of every kind (-1: per configuration)
  int slice_force = -1;  // FKPM_OPT_SLICE: column-pass loop order (-1: per configuration)
  int order_force = -1;  // FKPM_OPT_ROW_ORDER: lattice row order (-1: per configuration)
  bool has_order = false;  // rdesc holds a row order for the current pattern
  DevBuf rdesc;            // {row, first block, end block} per sweep position
  long long table_cap_mb = -1;  // FKPM_OPT_ALPHA_TABLE_MB (-1: the default budget)

  // --- whole-recursion kernels of small lattices (kpm_resident.h) ---
  struct Resident {
    bool packed = false;  // hval / hoff hold the current H
    int rpt = 0, threads = 0, nt = 0;
    DevBuf hval, hoff, atab, btab, xi, coef, part;
    PinBuf pin;           // coefficients in, moment sums out
    fkd::ResSet<double> kd;
    fkd::ResSet<float> kf;
    bool state = false;   // the held moments state (alpha_M) is atab's
    int K = 0;            // atab holds alpha_0 .. alpha_K of the current H and R
  } res;

  // --- D ---
  int nbD = 0, nnzbD = 0;
  bool d_set = false, d_sym = false, d_fused = false, d_valid = false;
  DevBuf drp, dci, tpos, dacc, dout;
  DevBuf dout_f;  // D rounded to float for single-precision engines
  std::vector<int> hd_rp, hd_ci;

  // --- pinned staging of host arrays ---
  PinBuf stage;             // H values on their way in (upload_H_t)
  bool stage_busy = false;  // a copy from it may still be queued
  PinBuf dpin;              // chunks of a large D on their way out (copy_to_host)
  std::vector<hipEvent_t> dpin_ev;

  // --- two-current moments (moments2) ---
  DevBuf j_rp[2], j_ci[2], j_rb[2], j_raw[2], j_val[2], m2_a, m2_b, m2_ring, m2_c, m2_part;

  // --- hipGraph replay of the step loops (short steps) ---
  int graph_mode = -1;  // FKPM_OPT_GRAPH: -1 automatic, 0 never, 1 always
  GraphCache gcache;
  long long n_graph_launches = 0, n_graph_captures = 0;

  // --- timing ---
  bool timing = false;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  double ms_mom = 0, ms_stoch = 0, ms_ad = 0;
  int n_mom = 0, n_stoch = 0, n_ad = 0;

  ~fkpm_handle() {
    (void)hipSetDevice(device);
    if (stream) (void)hipStreamSynchronize(stream);
    DevBuf* bufs[] = {&rp,    &ci,    &hv,      &rowblk, &hraw, &rraw,  &rcol,     &rval,
                      &rflag, &R,     &A[0],    &A[1],   &A[2], &Bv[0], &Bv[1],    &Bv[2],
                      &xi,    &partial, &tune_dacc, &drp, &dci,  &tpos,     &dacc,
                      &dout,  &dout_f, &atab,  &tabc, &rdesc};
    for (DevBuf* d : bufs) d->release();
    DevBuf* m2bufs[] = {&j_rp[0], &j_ci[0], &j_rb[0], &j_raw[0], &j_val[0], &j_rp[1], &j_ci[1],
                        &j_rb[1], &j_raw[1], &j_val[1], &m2_a, &m2_b, &m2_ring, &m2_c, &m2_part};
    for (DevBuf* d : m2bufs) d->release();
    DevBuf* rbufs[] = {&res.hval, &res.hoff, &res.atab, &res.btab, &res.xi, &res.coef, &res.part};
    for (DevBuf* d : rbufs) d->release();
    res.pin.release();
    psum.release();
    stage.release();
    dpin.release();
    for (hipEvent_t e : dpin_ev) (void)hipEventDestroy(e);
    gcache.clear();
    if (ev0) (void)hipEventDestroy(ev0);
    if (ev1) (void)hipEventDestroy(ev1);
    if (stream) (void)hipStreamDestroy(stream);
  }

  size_t vbytes() const { return (size_t)n * sp * (cx ? 2 : 1) * (single ? 4 : 8); }
  size_t accbytes() const { return (size_t)n * sp * (cx ? 2 : 1) * 8; }
  int ne() const { return (single ? 4 : 2) / (cx ? 2 : 1); }  // elements per 16-byte packet
  // forward-phase alpha_k: R, then the table's alpha_1 .. alpha_{a_slots}, then the
  // ring of three
  void* vec_a(int k) {
    if (k == 0) return R.p;
    if (k <= a_slots) return static_cast<char*>(atab.p) + (size_t)(k - 1) * vbytes();
    return A[k % 3].p;
  }
  template <class S>
  const fkd::KSet<S>& ks(int kind) const;
  template <class S>
  fkd::ResSet<S>& rset();
};

template <>
fkd::ResSet<double>& fkpm_handle::rset<double>() {
  return res.kd;
}
template <>
fkd::ResSet<float>& fkpm_handle::rset<float>() {
  return res.kf;
}

template <>
const fkd::KSet<double>& fkpm_handle::ks<double>(int kind) const {
  return kd[kind];
}
template <>
const fkd::KSet<float>& fkpm_handle::ks<float>(int kind) const {
  return kf[kind];
}

namespace {

// Vectors of at most this many scalars count as short steps: their launches,
// not HBM, set the time of a step loop, so the loop is replayed as a hipGraph.
constexpr size_t kGraphMaxScalars = (size_t)1 << 22;

// Records the kernel launches of one step loop on the handle's stream; run()
// then launches them directly or, for short steps (FKPM_OPT_GRAPH), replays
// the cached hipGraph of exactly the same launches, capturing it the first
// time.  A graph replays launches with identical entries, grids and argument
// bytes, so it computes what the direct launches compute.
class LoopRecorder {
 public:
  explicit LoopRecorder(fkpm_handle* h) : h_(h) {
    g_rec.stream = h->stream;
    g_rec.recs = &recs_;
  }
  ~LoopRecorder() { stop(); }
  int run() {
    stop();
    const bool graph = h_->graph_mode == 1 ||
                       (h_->graph_mode == -1 && recs_.size() >= 8 &&
                        (size_t)h_->n * h_->sp * (h_->cx ? 2 : 1) <= kGraphMaxScalars);
    if (!graph) return replay_direct(recs_, h_->stream);
    GraphCache& gc = h_->gcache;
    const uint64_t key = rec_hash(recs_);
    for (size_t k = 0; k < gc.entries.size(); k++) {
      if (gc.entries[k].key == key && rec_equal(gc.entries[k].recs, recs_)) {
        std::rotate(gc.entries.begin(), gc.entries.begin() + k, gc.entries.begin() + k + 1);
        HIPCHK(hipGraphLaunch(gc.entries[0].exec, h_->stream));
        h_->n_graph_launches++;
        return 0;
      }
    }
    HIPCHK(hipStreamBeginCapture(h_->stream, hipStreamCaptureModeThreadLocal));
    const int rc = replay_direct(recs_, h_->stream);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(h_->stream, &g);
    if (rc != 0 || e != hipSuccess) {
      if (g) (void)hipGraphDestroy(g);
      return rc != 0 ? rc : fail(FKPM_E_HIP, "graph capture: %s", hipGetErrorString(e));
    }
    hipGraphExec_t ex = nullptr;
    const hipError_t ei = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (ei != hipSuccess) return fail(FKPM_E_HIP, "graph instantiate: %s", hipGetErrorString(ei));
    if (gc.entries.size() >= GraphCache::kMax) {
      HIPCHK(hipStreamSynchronize(h_->stream));  // no replay of the evicted graph in flight
      (void)hipGraphExecDestroy(gc.entries.back().exec);
      gc.entries.pop_back();
    }
    gc.entries.insert(gc.entries.begin(), GraphCache::Entry{key, std::move(recs_), ex});
    h_->n_graph_captures++;
    HIPCHK(hipGraphLaunch(ex, h_->stream));
    h_->n_graph_launches++;
    return 0;
  }

 private:
  void stop() {
    if (g_rec.recs == &recs_) {
      g_rec.recs = nullptr;
      g_rec.stream = nullptr;
    }
  }
  fkpm_handle* h_;
  std::vector<LaunchRec> recs_;
};

bool lookup_kset(fkpm_handle* h, int kind, int B, int L, int KQ) {
  if (h->single)
    return h->cx ? fkd::find_kset_fc(B, L, KQ, &h->kf[kind]) : fkd::find_kset_fr(B, L, KQ, &h->kf[kind]);
  return h->cx ? fkd::find_kset_dc(B, L, KQ, &h->kd[kind]) : fkd::find_kset_dr(B, L, KQ, &h->kd[kind]);
}

bool compiled(int b, int L, int KQ) {
  fkd::GeomChoice gs[64];
  const int ng = fkd::geometries_for_block(b, gs, 64);
  for (int k = 0; k < ng; k++)
    if (gs[k].L == L && gs[k].KQ == KQ) return true;
  return false;
}

void derive_grid(int nb, KCfg& c) {
  const int gwg = (fkd::WG / fkd::WAVE) * (fkd::WAVE / c.L);
  const int cap = c.maxwg > 0 ? c.maxwg : 4096;
  int nwg = (nb + gwg - 1) / gwg;
  if (nwg > cap) nwg = cap;
  if (nwg < 1) nwg = 1;
  int chunk = (nb + nwg - 1) / nwg;
  chunk = ((chunk + gwg - 1) / gwg) * gwg;
  c.nwg = (nb + chunk - 1) / chunk;
  c.chunk = chunk;
  if (c.sweep > 0) {
    // one front: a multiple of 8 s workgroups (the extra ones find no rows)
    const int q = 8 * c.sweep;
    c.nwg = (c.nwg + q - 1) / q * q;
    c.chunk = -c.sweep;
  }
}

// Matrix-core kernels exist for complex 8x8 blocks (forward/Clenshaw steps,
// also into the table, and both autodiff steps).
bool mfma_avail(const fkpm_handle* h, int kind) {
  return h->mfma_on && h->cx && h->b == 8 &&
         (kind == K_MOM || kind == K_MOMT || kind == K_AD || kind == K_ADS);
}

// The row-resident variants: rows of at most kRowResidentMax blocks (MF_DM of
// kpm_mfma.h), byte offsets of a vector within 32 bits.
bool mfma_rr_avail(const fkpm_handle* h, int kind) {
  return mfma_avail(h, kind) && h->max_deg <= kRowResidentMax && h->vbytes() < (size_t(1) << 32);
}

int set_kind(fkpm_handle* h, int kind, KCfg c) {
  if (c.mfma) {
    if (!mfma_avail(h, kind) || (c.mfma == 2 && !mfma_rr_avail(h, kind)))
      return fail(FKPM_E_UNSUP, "no matrix-core kernel for block %d (kind %d)", h->b, kind);
    c.L = 64;  // one wave per block row
    c.KQ = 1;
    c.nt = 0;
    c.dm = h->max_deg <= 7 ? 7 : 8;
  }
  if (!lookup_kset(h, kind, h->b, c.L, c.KQ))
    return fail(FKPM_E_UNSUP, "no kernel for block %d, lanes %d, packets %d", h->b, c.L, c.KQ);
  if (h->sweep_force >= 0) c.sweep = h->sweep_force;
  if (h->slice_force >= 0 && !c.mfma)
    c.nt = (c.nt & ~fkd::NT_SLICE) | (h->slice_force ? fkd::NT_SLICE : 0);
  if (h->order_force >= 0 && !c.mfma && kind != K_OUT)
    c.nt = (c.nt & ~fkd::NT_ORDER) | (h->order_force ? fkd::NT_ORDER : 0);
  // the order exists for lattice patterns only; its sweep is one range per XCD
  if (!h->has_order || c.mfma || kind == K_OUT) c.nt &= ~fkd::NT_ORDER;
  if (c.nt & fkd::NT_ORDER) c.sweep = 0;
  derive_grid(h->nb, c);
  h->kc[kind] = c;
  return 0;
}

// The row order in the chosen configurations after the pattern or the
// FKPM_OPT_ROW_ORDER switch changed: off where the pattern has none, forced
// on or off by the switch, else as chosen (its sweep is one range per XCD).
void apply_row_order(fkpm_handle* h) {
  for (int k = 0; k < NKIND; k++) {
    KCfg& c = h->kc[k];
    if (c.L <= 0) continue;
    const bool can = h->has_order && !c.mfma && k != K_OUT;
    if (!can || h->order_force == 0) c.nt &= ~fkd::NT_ORDER;
    else if (h->order_force == 1) c.nt |= fkd::NT_ORDER;
    if (c.nt & fkd::NT_ORDER) c.sweep = 0;
    derive_grid(h->nb, c);
  }
}

// The row array a step kernel of configuration c reads: the row offsets, or
// the row order's descriptors (NT_ORDER).
const int* rp_for(const fkpm_handle* h, const KCfg& c) {
  return (c.nt & fkd::NT_ORDER) ? h->rdesc.as<const int>() : h->rp.as<const int>();
}

// The nt argument of a step kernel on H's pattern: the configuration's, with the
// row length where all rows share one (row_ptr).
int nt_for(const fkpm_handle* h, const KCfg& c) {
  const bool same = !(c.nt & fkd::NT_ORDER) && (long long)h->nb * h->max_deg == h->nnzb &&
                    h->max_deg < 1 << 16;
  return same ? c.nt | h->max_deg << fkd::NT_DEG : c.nt;
}

// Whether a row much longer than the others sets the time of a step: its blocks are one
// chain of gathers in a lane group, longer by a third with two packets a lane than with
// one, while the other rows stream past.  moments of M = 40 (us), two packets a lane /
// one, rows of 5 blocks and one of 65: 30000 x 2 FP64 (15 MB a vector) 554 / 462, x 4 FP32
// (31 MB) 1462 / 1118; one of 25: 9000 x 2 FP32 (5 MB) 273 / 218, 30000 x 4 FP32 (31 MB) 686 / 568,
// but 30000 x 2 FP64 (15 MB) 308 / 352, x 4 (61 MB) 960 / 1265.
bool long_rows(int nb, int nnzb, int max_deg) { return (long long)max_deg * nb > 2ll * nnzb; }

bool chain_bound(const fkpm_handle* h) {
  return long_rows(h->nb, h->nnzb, h->max_deg) &&
         h->vbytes() < (size_t)h->max_deg * h->b * ((h->single ? 320 : 192) << 10);
}

// Column passes side by side in the forward method's step.  Rows of complex 8x8 blocks
// are padded to tiles of the matrix cores, which leaves this vector-unit step passes as
// narrow as one tile (144 columns FP64: nine); one after another in the workgroup of the
// row they are one long chain, and few rows leave the chip idle meanwhile.  So with
// blocks of 4 and 8 the passes of a sweep of up to 128 workgroups run side by side.
// stoch_matrix of M = 32 (us), in turn / side by side: 12x12 x 8 FP64, S = 129 3674 / 911,
// 10^3 5679 / 3052, 45x45 (127 workgroups) 4824 / 3875; 15^3 (211) S = 65 4594 / 4989, FP32
// S = 129 4201 / 4484.  Smaller blocks have few passes of many rows (60x60 x 1 FP32, S = 150
// 256 / 271).
constexpr int kXiPassWgs = 128;

int xi_apart(const fkpm_handle* h, const KCfg& c) {
  return h->b >= 4 && c.nwg <= kXiPassWgs ? h->qp / (c.L * c.KQ) : 1;
}
template <class S>
auto xi_fn(const fkpm_handle* h, const fkd::KSet<S>& ks, const KCfg& c) {
  return xi_apart(h, c) > 1 ? ks.xi_apart : ks.xi;
}

// Kernel entry of a kind under its configuration.
template <class S>
auto mom_fn(const fkpm_handle* h, const fkd::KSet<S>& ks, const KCfg& c) {
  if (c.mfma == 2 && ks.mfma_mom_rr2 != nullptr && h->qp % 16 == 0)
    return c.dm == 7 ? ks.mfma_mom_rr2_7 : ks.mfma_mom_rr2;
  if (c.mfma == 2) return c.dm == 7 ? ks.mfma_mom_rr7 : ks.mfma_mom_rr;
  return c.mfma ? ks.mfma_mom : fkd::step_fn(ks, h->nb, chain_bound(h));
}
// The row-resident autodiff step in FP32 takes column tiles in pairs when the
// padded width allows (16 packets, two 16-column tiles, divide it): C4 FP32
// 1747 -> 1561 us per step.
template <class S>
auto adf_fn(const fkpm_handle* h, const fkd::KSet<S>& ks, const KCfg& c) {
  if (c.mfma == 2 && ks.mfma_ad_rr2 != nullptr && h->qp % 16 == 0)
    return c.dm == 7 ? ks.mfma_ad_rr2_7 : ks.mfma_ad_rr2;
  return c.mfma == 2 ? (c.dm == 7 ? ks.mfma_ad_rr7 : ks.mfma_ad_rr)
                      : c.mfma ? ks.mfma_ad_fused : ks.ad_fused;
}
template <class S>
auto adp_fn(const fkd::KSet<S>& ks, const KCfg& c) {
  return c.mfma ? ks.mfma_ad_plain : ks.ad_plain;
}
// The backward steps reading the table, as adf_fn / adp_fn choose.
template <class S>
auto ads_fn(const fkpm_handle* h, const fkd::KSet<S>& ks, const KCfg& c) {
  if (c.mfma == 2 && ks.mfma_ads[fkd::ADS_RR2] != nullptr && h->qp % 16 == 0)
    return ks.mfma_ads[c.dm == 7 ? fkd::ADS_RR2_7 : fkd::ADS_RR2];
  if (c.mfma == 2) return ks.mfma_ads[c.dm == 7 ? fkd::ADS_RR7 : fkd::ADS_RR];
  return c.mfma ? ks.mfma_ads[fkd::ADS_FUSED] : ks.ad_stored;
}
template <class S>
auto adsp_fn(const fkd::KSet<S>& ks, const KCfg& c) {
  return c.mfma ? ks.mfma_ads[fkd::ADS_PLAIN] : ks.ad_stored_plain;
}

// Last-level cache of the device (MI355X: 256 MB).
constexpr size_t kLlcBytes = (size_t)256 << 20;

// Default geometry of a kernel kind when nothing is tuned: one pass of width
// wmax.  From 64 packets on, whole waves per row (wave-uniform rows, scalar
// offsets and H); below, two packets per lane, which keeps more loads in
// flight per wave than twice the lanes, where that leaves a workgroup for each
// of the 256 CUs.  Forward step (us), 64 x 1 / 16 x 4 / 32 x 2 lanes x packets on 64:
// 256^2 x 2 FP64 81 / 98 / 110, 20^3 x 2 12.9 / 14.9 / 16.2; 16 x 2 / 32 x 1 on
// 32: 256^2 x 2 FP32 37 / 47, 128^2 x 2 FP64 14.4 / 18.1; 8 x 2 / 16 x 1 on 16:
// 31x29x27 real 7.2 / 10.6, but 37x52 x 2 (61 / 121 workgroups) 8.4 / 7.9.  The
// backward step reading the table takes four packets per lane while its vectors
// stay in the last-level cache (16 x 4 / 64 x 1: 20^3 x 2 23.4 / 26, past it 256^2 x 2
// 171 / 165; 8 x 4 / 16 x 2: 128^2 x 2 22.0 / 24.5).
KCfg default_cfg(fkpm_handle* h, int kind) {
  static const int wide[] = {64, 32, 16, 8, 4};
  static const int reduce[] = {16, 8, 32, 4, 64};
  // vectors a step touches; one that writes a fresh table slot meets the ones
  // of the steps before it in the cache too
  const int nvec = kind == K_AD || kind == K_ADS ? 6 : kind == K_XI || kind == K_MOMT ? 5 : 3;
  const bool cached = (size_t)nvec * h->vbytes() <= kLlcBytes;
  KCfg c;
  auto packets = [&](int kq) {
    const int L = h->wmax / kq;
    if (c.L > 0 || h->wmax % kq != 0 || !compiled(h->b, L, kq) || chain_bound(h) ||
        h->nb < 256 * (fkd::WG / fkd::WAVE) * (fkd::WAVE / L))
      return;
    c.L = L;
    c.KQ = kq;
  };
  if (kind == K_ADS && cached) packets(4);
  if (kind != K_OUT && h->wmax < 64) packets(2);
  const int* pref = kind == K_OUT ? reduce : wide;
  for (int t = 0; t < 5 && c.L == 0; t++) {
    const int L = pref[t];
    if (h->wmax % L == 0 && compiled(h->b, L, h->wmax / L)) {
      c.L = L;
      c.KQ = h->wmax / L;
    }
  }
  if (c.L == 0) {  // any compiled geometry of width <= wmax, widest first
    fkd::GeomChoice gs[64];
    const int ng = fkd::geometries_for_block(h->b, gs, 64);
    for (int k = 0; k < ng; k++) {
      const int w = gs[k].L * gs[k].KQ;
      if (w <= h->wmax && (c.L == 0 || w > c.L * c.KQ)) {
        c.L = gs[k].L;
        c.KQ = gs[k].KQ;
      }
    }
  }
  // One pass over the rows: with several, a workgroup's next rows lie far off and
  // an XCD sweeps as many windows at once, each with its share of the L2 (FP64
  // forward step 256^2 x 2: 81 us, 4096 workgroups 87; 64^3 x 2 in lattice row
  // order: 687 us, 16384 workgroups 772; its autodiff step 1590 and 1690).
  c.maxwg = 65536;
  c.nt = 0;
  // While a step's vectors stay in the last-level cache each XCD sweeps its own
  // region, whose neighbour rows its L2 then holds (128^2 x 2 FP64 forward step
  // 13.2 us against 16.6 in one front, 20^3 x 2 12.9 / 17.8, autodiff 25 / 30);
  // past it one front in segments of two passes keeps far neighbours in the
  // shared cache (256^2 x 2 FP64: 81 us, per XCD 92).  A sweep of fewer than
  // 64 workgroups has no regions to speak of.
  const int gwg = (fkd::WG / fkd::WAVE) * (fkd::WAVE / (c.L > 0 ? c.L : fkd::WAVE));
  c.sweep = cached && h->nb / gwg >= 64 ? 0 : 2;
  // The lattice row order where the vectors miss the cache and a tile plane of
  // 128 sites (512 KB a vector) fills the L2 better than a plane of the lattice
  // (64^3 x 2, S = 128 FP64: 687 against 762 us); with half the bytes a site the two
  // sweeps measured the same (FP32: 377 and 366).
  if (h->has_order && !cached && kind != K_OUT &&
      h->vbytes() / (size_t)h->nb >= 4096)
    c.nt |= fkd::NT_ORDER;
  if (mfma_avail(h, kind)) {
    c.mfma = 1;
    // row-resident: the forward step always, the autodiff step in FP64 and in
    // FP32 where its column tiles pair up (adf_fn)
    if (mfma_rr_avail(h, kind) && (kind == K_MOM || kind == K_MOMT || !h->single ||
                                   h->qp % 16 == 0 || h->rr_force))
      c.mfma = 2;
    // per XCD while three vectors stay in the last-level cache (forward step at
    // 18x15x13 x 8 FP64, 65 MB vectors: 52 us, one front 65), else one front of
    // single passes (32^3 x 8 FP32: 447, segments of two 466, per XCD 555)
    if (h->nb / gwg >= 64) c.sweep = 3 * h->vbytes() <= kLlcBytes ? 0 : 1;
  }
  return c;
}

// Whether moments(M) keeps the forward vectors (when they fit).  The backward
// steps then gather one vector instead of two and stoch_matrix takes half the
// steps; the forward step pays a write-back to a fresh slot.  M = 128, us per
// call, ring / table: 60x40 x 2 FP64 set_H + moments + autodiff_matrix 1168 / 1101
// and moments + autodiff_matrix + stoch_matrix 1827 / 1445; 140x120 x 1 1672 / 1667
// and 2321 / 1921; 256^2 x 2 FP32 forward step 35 / 38, autodiff 107 / 91.
bool table_wanted(const fkpm_handle* h) { return h->store_alpha != 0; }

// By default not from the third moments on that nothing followed (a density of states,
// a Monte Carlo walk on energies): the writes to fresh slots cost moments up to 15 %
// (us, table / ring: 46x46 x 2, S = 8, M = 1024 3053 / 2658; 200x200 real, S = 16, M = 128
// 465 / 399; 128^2 x 2 FP32, S = 32, M = 256 1089 / 940; the matrix-core steps lose nothing, 12^3 x 8
// FP32 255 / 292).  Only where the forward step has one launch configuration either
// way, so that the moments are bitwise the same.
constexpr int kUnread = 2;

bool table_idle(const fkpm_handle* h) {
  const KCfg &a = h->kc[K_MOM], &b = h->kc[K_MOMT];
  return h->store_alpha == 1 && h->unread >= kUnread && a.L == b.L && a.KQ == b.KQ &&
         a.nwg == b.nwg && a.chunk == b.chunk && a.nt == b.nt && !a.mfma && !b.mfma;
}

// Process-wide cache of tuned geometries, keyed by the problem shape.
std::mutex g_tune_mu;
std::map<std::string, std::array<KCfg, NKIND>> g_tune_cache;

std::string tune_key(const fkpm_handle* h) {
  char k[128];
  snprintf(k, sizeof(k), "%d/%d/%d/%d/%d/%d/%d/%d/%d/%d", h->dtype, h->prec, h->b, h->s, h->nb,
           h->nnzb, h->mfma_on ? (h->rr_force ? 2 : 1) : 0,
           h->max_deg <= 7 ? 2 : h->max_deg <= kRowResidentMax ? 1 : 0, table_wanted(h) ? 1 : 0,
           h->has_order ? 1 : 0);
  return k;
}

// Packed width: qp packets per row, a multiple of wmax, the smallest compiled
// pass width that covers the row (or the widest, with several passes).
int choose_geometry(fkpm_handle* h) {
  const int ne = h->ne();
  const int qp0 = (h->s + ne - 1) / ne;
  fkd::GeomChoice gs[64];
  const int ng = fkd::geometries_for_block(h->b, gs, 64);
  if (ng == 0) return fail(FKPM_E_UNSUP, "block size %d is not supported", h->b);
  int wmax = 0, widest = 0;
  for (int k = 0; k < ng; k++) {
    const int w = gs[k].L * gs[k].KQ;
    widest = std::max(widest, w);
    if (w >= qp0 && (wmax == 0 || w < wmax)) wmax = w;
  }
  if (wmax == 0) wmax = widest;
  // Matrix-core tiles are 16 complex columns wide (FP32 takes them in pairs) and
  // a row may hold any number of them: of the compiled widths that are whole
  // tiles, the one that pads the row least (144 columns: 144 instead of 192).
  if (h->mfma_on && h->cx && h->b == 8) {
    const int tile = qp0 <= 16 / ne ? 16 / ne : 16;
    int best = 0;
    for (int k = 0; k < ng; k++) {
      const int w = gs[k].L * gs[k].KQ;
      if (w % tile != 0) continue;
      const int pad = (qp0 + w - 1) / w * w;
      if (best == 0 || pad < best || (pad == best && w > wmax)) {
        best = pad;
        wmax = w;
      }
    }
  }
  if (h->force_L > 0) {
    const int fkq = h->force_KQ > 0 ? h->force_KQ : 1;
    if (!compiled(h->b, h->force_L, fkq))
      return fail(FKPM_E_UNSUP, "geometry lanes=%d kq=%d not compiled for block %d", h->force_L,
                  fkq, h->b);
    wmax = std::max(wmax, h->force_L * fkq);
  }
  h->wmax = wmax;
  h->qp = ((qp0 + wmax - 1) / wmax) * wmax;
  h->sp = h->qp * ne;
  h->geo_b = h->b;
  bool cached = false;
  std::array<KCfg, NKIND> cc;
  if (h->force_L == 0) {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tune_cache.find(tune_key(h));
    if (it != g_tune_cache.end()) {
      cc = it->second;
      cached = true;
    }
  }
  for (int kind = 0; kind < NKIND; kind++) {
    KCfg c;
    if (h->force_L > 0) {
      c.L = h->force_L;
      c.KQ = h->force_KQ > 0 ? h->force_KQ : 1;
      c.maxwg = h->max_wg;
    } else if (cached) {
      c = cc[kind];
    } else {
      c = default_cfg(h, kind);
      if (h->max_wg > 0) c.maxwg = h->max_wg;
    }
    CHK(set_kind(h, kind, c));
  }
  h->tuned = cached;
  return 0;
}

template <class TH, class S, bool CX>
int pack_R_t(fkpm_handle* h) {
  dim3 grid((h->n + 63) / 64, (h->sp + 15) / 16);
  CHK(launch(&fkd::k_pack_R<TH, S, CX>, grid, dim3(fkd::WG), h->stream, h->rraw.as<const TH>(),
             h->R.as<S>(), h->n, h->s, h->sp));
  // compact form when every row holds at most one nonzero
  CHK(h->rcol.ensure(sizeof(int) * (size_t)h->n));
  CHK(h->rval.ensure(sizeof(S) * (size_t)h->n * (CX ? 2 : 1)));
  CHK(h->rflag.ensure(16));
  CHK(launch(&fkd::k_zero, dim3(1), dim3(64), h->stream, (double*)h->rflag.p, (size_t)2));
  CHK(launch(&fkd::k_compact_R<TH, S, CX>, dim3((h->n + fkd::WG - 1) / fkd::WG), dim3(fkd::WG),
             h->stream, h->rraw.as<const TH>(), h->n, h->s, h->rcol.as<int>(), h->rval.as<S>(),
             h->rflag.as<int>()));
  int flag = 1;
  HIPCHK(hipMemcpyAsync(&flag, h->rflag.p, sizeof(int), hipMemcpyDeviceToHost, h->stream));
  HIPCHK(hipStreamSynchronize(h->stream));
  h->r_compact = (flag == 0);
  return 0;
}

template <class S>
int pack_R_s(fkpm_handle* h) {
  switch (h->dtype) {
    case FKPM_F32: return pack_R_t<float, S, false>(h);
    case FKPM_F64: return pack_R_t<double, S, false>(h);
    case FKPM_C32: return pack_R_t<float, S, true>(h);
    default: return pack_R_t<double, S, true>(h);
  }
}

template <class S>
fkd::RSource<S> rsource(fkpm_handle* h, double cr) {
  fkd::RSource<S> r = no_rsource<S>();
  r.cr = cr;
  if (h->r_compact) {
    r.rcol = h->rcol.as<const int>();
    r.rval = h->rval.as<const S>();
  } else {
    r.rd = h->R.as<const S>();
  }
  return r;
}

int tune(fkpm_handle* h);

// Make geometry, vectors and packed R consistent with the current H and R.
int ensure_ready(fkpm_handle* h) {
  if (!h->h_set) return fail(FKPM_E_STATE, "set_H has not been called");
  if (!h->r_set) return fail(FKPM_E_STATE, "R has not been set (set_R / transfer_R)");
  if (h->n != h->nb * h->b)
    return fail(FKPM_E_ARG, "R has %d rows but H has %d = %d blocks x %d", h->n, h->nb * h->b,
                h->nb, h->b);
  bool stale = h->r_dirty || h->geo_b != h->b;
  // backstop: a row-resident matrix-core kernel on a pattern with longer rows
  // would read only the first kRowResidentMax blocks of each row
  for (int k = 0; k < NKIND && !stale; k++)
    stale = h->kc[k].mfma == 2 && (!mfma_rr_avail(h, k) || (h->kc[k].dm == 7 && h->max_deg > 7));
  if (!stale) return 0;
  CHK(choose_geometry(h));
  const size_t vb = h->vbytes();
  CHK(h->R.ensure(vb));
  for (int k = 0; k < 3; k++) CHK(h->A[k].ensure(vb));
  if (h->single)
    CHK(pack_R_s<float>(h));
  else
    CHK(pack_R_s<double>(h));
  // A-buffers: every element is written by the recursion before it is read.
  h->r_dirty = false;
  h->alpha_M = 0;
  h->tab_K = 0;
  h->res.K = 0;
  if (h->autotune_on_use && !h->tuned && h->force_L == 0) CHK(tune(h));
  return 0;
}

// Steps whose moment partials are held before they are reduced: 64 MiB of them
// (a step of 65536 workgroups leaves 1 MiB).
int partial_steps(int nsteps, int nwg) {
  const size_t per = (size_t)std::max(nwg, 1) * 2 * sizeof(double);
  return (int)std::min<size_t>(nsteps, std::max<size_t>(1, ((size_t)64 << 20) / per));
}

int ensure_partials(fkpm_handle* h, int nsteps) {
  // the wider grid may hold fewer steps and less memory in all
  size_t rows = 0;
  for (int kind : {K_MOM, K_MOMT}) {
    const int nwg = h->kc[kind].nwg;
    rows = std::max(rows, (size_t)partial_steps(nsteps, nwg) * nwg);
  }
  CHK(h->partial.ensure(rows * 2 * sizeof(double)));
  CHK(h->psum.ensure((size_t)nsteps * 2 * sizeof(double)));
  return 0;
}

int zero_doubles(fkpm_handle* h, void* p, size_t n) {
  return launch(&fkd::k_zero, dim3(grid_for(n)), dim3(256), h->stream, (double*)p, n);
}

int timing_begin(fkpm_handle* h) {
  if (h->timing) HIPCHK(hipEventRecord(h->ev0, h->stream));
  return 0;
}
int timing_end(fkpm_handle* h, double* ms, int* cnt, int launches) {
  if (!h->timing) return 0;
  HIPCHK(hipEventRecord(h->ev1, h->stream));
  HIPCHK(hipEventSynchronize(h->ev1));
  float t = 0.f;
  HIPCHK(hipEventElapsedTime(&t, h->ev0, h->ev1));
  *ms = t;
  *cnt = launches;
  return 0;
}

// ---------------------------------------------------------------------------
// Autotuner: times every compiled geometry of pass width wmax or wmax/2, three
// workgroup caps (where they differ) and the nontemporal choice, per kernel kind, on the current
// H and R; keeps the fastest and caches it for this problem shape.
// ---------------------------------------------------------------------------
template <class S>
int tune_t(fkpm_handle* h) {
  h->tab_K = 0;  // the table may serve as tuning slots below
  h->alpha_M = 0;
  const int HS = h->cx ? 2 : 1;
  const size_t vb = h->vbytes();
  CHK(h->Bv[0].ensure(vb));
  CHK(h->xi.ensure(h->accbytes()));
  CHK(h->tune_dacc.ensure((size_t)(h->nnzb > 0 ? h->nnzb : 1) * h->b * h->b * HS * sizeof(double)));
  CHK(h->partial.ensure(((size_t)(h->nb + 3) / 4 + 8 * 64) * 2 * sizeof(double)));
  const int* rp = h->rp.as<const int>();
  const int* ci = h->ci.as<const int>();
  const S* hv = h->hv.as<const S>();
  const S* R = h->R.as<const S>();
  S* A0 = h->A[0].as<S>();
  S* A1 = h->A[1].as<S>();
  S* A2 = h->A[2].as<S>();
  S* B0 = h->Bv[0].as<S>();
  CHK(h->Bv[1].ensure(vb));
  CHK(h->Bv[2].ensure(vb));
  S* B1 = h->Bv[1].as<S>();
  S* B2 = h->Bv[2].as<S>();
  // finite inputs for every candidate: every ring buffer = Hs R
  {
    const KCfg& c = h->kc[K_MOM];
    const auto& ks = h->ks<S>(K_MOM);
    S* outs[] = {A0, A1, A2, B0, B1, B2};
    for (S* o : outs)
      CHK(launch(mom_fn(h, ks, c), dim3(c.nwg), dim3(fkd::WG), h->stream, rp, ci, hv, R, (const S*)nullptr,
                 o, h->nb, h->qp, c.chunk, 1.0, 0.0, (double*)nullptr, 0, no_rsource<S>()));
    CHK(zero_doubles(h, h->tune_dacc.p, (size_t)h->nnzb * h->b * h->b * HS));
  }
  S* ring[3] = {A0, A1, A2};
  S* bring[3] = {B0, B1, B2};
  const bool log = getenv("FKPM_TUNE_LOG") != nullptr;
  int step = 0;
  fkd::GeomChoice gs[64];
  const int ng = fkd::geometries_for_block(h->b, gs, 64);
  static const int caps[] = {4096, 16384, 65536};
  static const int nts[] = {0, fkd::NT_LOAD | fkd::NT_STORE};
  static const int sweeps[] = {0, 1, 2, 8};
  // The table kinds are timed on ns slots (at least 512 MB, more than the
  // last-level cache holds) walked as the recursions walk the table: a fresh
  // slot per forward step, the kept vectors backwards.  Without a table in
  // prospect they take the ring kinds' choice.
  int ns = 0;
  int tstep = 0;
  auto slot = [&](int k) { return (S*)((char*)h->atab.p + (size_t)k * vb); };
  const int kinds[] = {K_MOM, K_XI, K_AD, K_MOMT, K_ADS};
  for (int kind : kinds) {
    if (kind == K_MOMT) {
      if (table_wanted(h)) {
        const size_t want = ((size_t)512 << 20) / vb + 1;
        const int n = (int)std::min<size_t>(64, std::max<size_t>(8, want));
        size_t free_b = 0, total_b = 0;
        HIPCHK(hipMemGetInfo(&free_b, &total_b));
        if ((size_t)n * vb <= free_b / 4 + h->atab.bytes) {
          CHK(h->atab.ensure((size_t)n * vb));
          ns = n;
          const KCfg& c = h->kc[K_MOM];
          const auto& ks = h->ks<S>(K_MOM);
          for (int k = 0; k < ns; k++)  // every slot = Hs R
            CHK(launch(mom_fn(h, ks, c), dim3(c.nwg), dim3(fkd::WG), h->stream, rp, ci, hv, R,
                       (const S*)nullptr, slot(k), h->nb, h->qp, c.chunk, 1.0, 0.0,
                       (double*)nullptr, 0, no_rsource<S>()));
        }
      }
      if (ns == 0) {
        CHK(set_kind(h, K_MOMT, h->kc[K_MOM]));
        CHK(set_kind(h, K_ADS, h->kc[K_AD]));
        break;
      }
    }
    KCfg best = h->kc[kind];
    float best_ms = 1e30f;
    std::vector<KCfg> cands;
    for (int g = 0; g < ng; g++) {
      const int w = gs[g].L * gs[g].KQ;
      if (w > h->wmax || 2 * w < h->wmax) continue;
      // the column passes as the outer loop (NT_SLICE) when a row takes
      // several passes of this width
      const int nsl = h->qp / w >= 2 ? 2 : 1;
      for (int cap : caps)
        for (int nt : nts)
          for (int sl = 0; sl < nsl; sl++) {
            KCfg c;
            c.L = gs[g].L;
            c.KQ = gs[g].KQ;
            c.maxwg = cap;
            c.nt = nt | (sl ? fkd::NT_SLICE : 0);
            for (int sw : sweeps) {
              c.sweep = sw;
              cands.push_back(c);
            }
            if (h->has_order && kind != K_OUT) {  // the lattice row order, one range per XCD
              c.nt |= fkd::NT_ORDER;
              c.sweep = 0;
              cands.push_back(c);
            }
          }
    }
    if (mfma_avail(h, kind))
      for (int v = 1; v <= (mfma_rr_avail(h, kind) ? 2 : 1); v++)
        for (int cap : caps)
          for (int sw : sweeps) {
            KCfg c;
            c.mfma = v;
            c.maxwg = cap;
            c.sweep = sw;
            cands.push_back(c);
          }
    // every candidate timed over 6 launches, then the closest few again over
    // 24, so that one noisy short timing does not decide the kernel for every
    // later solve of this shape
    auto time_cfg = [&](const KCfg& c, int reps, float* us) -> int {
          CHK(set_kind(h, kind, c));
          const KCfg& k = h->kc[kind];
          const auto& ks = h->ks<S>(kind);
          // steps rotate their buffers as the recursions do (one continuous
          // recurrence over all candidates keeps the values bounded)
          auto run = [&]() -> int {
            if (kind == K_MOMT) {  // alpha_{t+2} = 2 Hs alpha_{t+1} - alpha_t into a fresh slot
              const int t = tstep++;
              return launch(mom_fn(h, ks, k), dim3(k.nwg), dim3(fkd::WG), h->stream, rp_for(h, k), ci, hv,
                            (const S*)slot((t + 1) % ns), (const S*)slot(t % ns),
                            slot((t + 2) % ns), h->nb, h->qp, k.chunk, 2.0, -1.0,
                            h->partial.as<double>(), nt_for(h, k), no_rsource<S>());
            }
            if (kind == K_ADS) {  // backward over slots ns-2 .. 1, beta in the ring
              const int t = tstep++;
              const int m = ns - 2 - t % (ns - 2);
              return launch(ads_fn(h, ks, k), dim3(k.nwg), dim3(fkd::WG), h->stream, rp_for(h, k), ci,
                            hv, (const S*)slot(m), (const S*)slot(m + 1),
                            (const S*)bring[(t + 1) % 3], (const S*)bring[t % 3],
                            (const S*)slot(m - 1), bring[(t + 2) % 3], h->tune_dacc.as<double>(),
                            h->nb, h->qp, k.chunk, 0.1, 0.1, 0.1, 1.0, 0.0, 2.0, nt_for(h, k));
            }
            const int t = step++;
            S* x = ring[(t + 1) % 3];
            S* z = ring[t % 3];
            S* y = ring[(t + 2) % 3];
            // recurrences keep |x| bounded: y = 2 Hs x - z stays within the spectrum scale.
            // The forward kernel also runs stoch_matrix's Clenshaw steps (with
            // the source term c_k R, without the moment dots): every other
            // launch here is one, so both forms weigh in the choice
            if (kind == K_MOM) {
              const bool cl = t & 1;
              return launch(mom_fn(h, ks, k), dim3(k.nwg), dim3(fkd::WG), h->stream, rp_for(h, k), ci, hv,
                            (const S*)x, (const S*)z, y, h->nb, h->qp, k.chunk, 2.0, -1.0,
                            cl ? (double*)nullptr : h->partial.as<double>(), nt_for(h, k),
                            cl ? rsource<S>(h, 0.25) : no_rsource<S>());
            }
            if (kind == K_XI)
              return launch(xi_fn(h, ks, k), dim3(k.nwg, xi_apart(h, k)), dim3(fkd::WG),
                            h->stream, rp_for(h, k), ci, hv, (const S*)x, (const S*)z, y,
                            h->xi.as<double>(), h->nb, h->qp, k.chunk, 2.0, -1.0, 0.0, 0.5,
                            t == 0 ? 1 : 0, nt_for(h, k));
            // backward step: reads alpha_m, alpha_{m+1}, beta_{m+1}, beta_{m+2};
            // writes alpha_{m-1}, beta_m into the third buffers
            return launch(adf_fn(h, ks, k), dim3(k.nwg), dim3(fkd::WG), h->stream, rp_for(h, k), ci, hv,
                          (const S*)x, (const S*)z, (const S*)bring[(t + 1) % 3],
                          (const S*)bring[t % 3], y, bring[(t + 2) % 3], h->tune_dacc.as<double>(),
                          h->nb, h->qp, k.chunk, 0.1, 0.1, 0.1, 1.0, 0.0, 2.0, nt_for(h, k));
          };
          CHK(run());
          HIPCHK(hipEventRecord(h->ev0, h->stream));
          for (int r = 0; r < reps; r++) CHK(run());
          HIPCHK(hipEventRecord(h->ev1, h->stream));
          HIPCHK(hipEventSynchronize(h->ev1));
          float ms = 0.f;
          HIPCHK(hipEventElapsedTime(&ms, h->ev0, h->ev1));
          *us = 1e3f * ms / reps;
          if (log)
            fprintf(stderr,
                    "[fkpm tune] kind=%d L=%d KQ=%d mfma=%d maxwg=%d nwg=%d nt=%d sweep=%d: %.2f us%s\n",
                    kind, k.L, k.KQ, k.mfma, k.maxwg, k.nwg, k.nt, k.sweep, *us,
                    reps > 6 ? " (final)" : "");
          return 0;
    };
    // caps that give the same grid are one candidate
    std::vector<KCfg> distinct;
    for (KCfg c : cands) {
      KCfg d = c;
      if (d.mfma) {
        d.L = 64;
        d.KQ = 1;
      }
      derive_grid(h->nb, d);
      bool seen = false;
      for (const KCfg& o : distinct)
        seen |= o.L == c.L && o.KQ == c.KQ && o.nt == c.nt && o.mfma == c.mfma &&
                o.sweep == c.sweep && o.nwg == d.nwg && o.chunk == d.chunk;
      if (seen) continue;
      c.nwg = d.nwg;
      c.chunk = d.chunk;
      distinct.push_back(c);
    }
    std::vector<std::pair<float, KCfg>> timed;
    for (const KCfg& c : distinct) {
      float us = 0.f;
      CHK(time_cfg(c, 6, &us));
      timed.push_back({us, h->kc[kind]});
    }
    std::stable_sort(timed.begin(), timed.end(),
                     [](const std::pair<float, KCfg>& a, const std::pair<float, KCfg>& b) {
                       return a.first < b.first;
                     });
    const size_t nfinal = std::min<size_t>(4, timed.size());
    for (size_t f = 0; f < nfinal; f++) {
      float us = 0.f;
      CHK(time_cfg(timed[f].second, 24, &us));
      if (us < best_ms) {
        best_ms = us;
        best = h->kc[kind];
      }
    }
    CHK(set_kind(h, kind, best));
  }
  // outer products: once per call, the autodiff geometry (a vector-unit
  // geometry of full pass width when autodiff runs on the matrix cores)
  KCfg outc = h->kc[K_AD].mfma ? default_cfg(h, K_OUT) : h->kc[K_AD];
  outc.nt = 0;
  CHK(set_kind(h, K_OUT, outc));
  h->alpha_M = 0;
  h->tab_K = 0;  // the table slots held tuning data
  h->tuned = true;
  std::array<KCfg, NKIND> cc;
  for (int k = 0; k < NKIND; k++) cc[k] = h->kc[k];
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_tune_cache[tune_key(h)] = cc;
  return 0;
}

int tune(fkpm_handle* h) { return h->single ? tune_t<float>(h) : tune_t<double>(h); }

// mu from the dots of each step, sums[2m] = |alpha_m|^2 and sums[2m+1] =
// Re<alpha_{m+1}, alpha_m>.
void moments_from_sums(const double* ps, int nsteps, double* mu) {
  mu[0] = ps[0];
  mu[1] = ps[1];
  for (int m = 1; m < nsteps; m++) {
    mu[2 * m] = 2 * ps[2 * m] - mu[0];
    mu[2 * m + 1] = 2 * ps[2 * m + 1] - mu[1];
  }
}

// Packets of a vector up to which k_table_sums splits the slots (us, split / one
// thread a packet; 250 slots FP64: 16384 packets 23 / 37, 32768 29 / 40, 65536 69 /
// 43; 64 slots: 6 / 8, 9 / 12, 19 / 13).
constexpr size_t kSumsSplit = 32768;

// Weights of the table vectors in stoch_matrix (stoch_table): d_0 .. d_K of v,
// then e_0 .. e_K of u.
void stoch_table_weights(int M, const double* c, std::vector<double>& w) {
  const int K = (M + 1) / 2;
  auto cm = [&](int m) { return m < M ? c[m] : 0.0; };
  w.assign(2 * (size_t)(K + 1), 0.0);
  for (int i = 0; i <= K; i++) {
    w[i] = (i < K ? cm(i) : 0.0) - (i >= 1 ? cm(2 * K - i) : 0.0);  // d_i
    w[K + 1 + i] = i < K ? cm(K + i) : 0.0;                         // e_i
  }
}

// The NO sums of stoch_matrix from K table slots of n scalars (k_table_sums).
template <class S, int NO>
int table_sums(fkpm_handle* h, const S* R, const S* tab, size_t n, int K, const double* w, S* o0,
               S* o1, S* o2 = nullptr) {
  const size_t np = n * sizeof(S) / 16;
  if (np <= kSumsSplit)
    return launch(&fkd::k_table_sums<S, 8, NO>, dim3((unsigned)((np + 31) / 32)), dim3(fkd::WG),
                  h->stream, R, tab, n, K, w, o0, o1, o2, n);
  return launch(&fkd::k_table_sums<S, 1, NO>, dim3(4096), dim3(fkd::WG), h->stream, R, tab, n, K, w,
                o0, o1, o2, n);
}

// out = (add ? out : 0) + the ny rows of part, cnt values each (k_sum_parts).
int sum_parts(fkpm_handle* h, const double* part, int ny, size_t cnt, double* out, bool add) {
  const size_t wgs = (cnt + fkd::SUM_X - 1) / fkd::SUM_X;
  return launch(&fkd::k_sum_parts, dim3((unsigned)std::min<size_t>(std::max<size_t>(wgs, 1), 65536)),
                dim3(fkd::WG), h->stream, part, ny, cnt, out, add ? 1 : 0);
}

// dacc += f A B^+ on D's pattern: complex 8x8 blocks on the matrix cores (us, vector
// units / matrix cores: 32^3 sites, S = 256 FP32 4384 / 1264; 18x15x13, S = 144 FP64
// 286 / 175).
template <class S>
int add_outer(fkpm_handle* h, const S* A, const S* B, double f) {
  const auto& ks = h->ks<S>(K_OUT);
  KCfg c = h->kc[K_OUT];
  auto fn = ks.outer_ss;
  if (mfma_avail(h, K_AD) && h->qp % (4 * fkd::MO_U) == 0) {
    fn = ks.mfma_outer;
    c.L = fkd::WAVE;  // one wave per block row
    derive_grid(h->nb, c);
  }
  return launch(fn, dim3(c.nwg), dim3(fkd::WG), h->stream, h->drp.as<const int>(),
                h->dci.as<const int>(), A, B, h->dacc.as<double>(), h->nb, h->qp, c.chunk, f);
}

// Weights of the table vectors where the table holds a third of the orders
// (stoch_table3, K = ceil(M/3)): v, w_1, w_2.
void stoch_table3_weights(int M, const double* c, std::vector<double>& w) {
  const int K = (M + 2) / 3, n = K + 1;
  std::vector<double> a(3 * (size_t)K, 0.0);  // coefficients of T_{jK+i} at j K + i
  std::copy(c, c + M, a.begin());
  w.assign(3 * (size_t)n, 0.0);
  for (int j = 2; j >= 1; j--) {
    w[j * n] = a[j * K];
    for (int i = 1; i < K; i++) {
      w[j * n + i] = 2 * a[j * K + i];
      a[(j - 1) * K + K - i] -= a[j * K + i];
    }
  }
  for (int i = 0; i < K; i++) w[i] = a[i] - w[2 * n + i];
}

// ---------------------------------------------------------------------------
// Whole-recursion kernels of small lattices (kpm_resident.h): moments,
// autodiff_matrix and stoch_matrix as one launch per recursion.
// ---------------------------------------------------------------------------

// LDS of one workgroup.
constexpr size_t kLdsBytes = 160 << 10;
// Bytes of H beyond its registers that a workgroup of the backward recursion may
// read from the L2 in every step (most of H at a column that still fits the LDS twice).
constexpr size_t kResStream = 1024 << 10;

// 16-byte L2 loads of H (smaller blocks: one each) a thread may have in a forward
// step, where it owns four rows or more, or two of 4x4 blocks; with fewer rows the
// streamed loads of a step overlap.  Every row is padded to the longest one, so an
// uneven pattern streams far more than it holds.  moments / moments + autodiff_matrix
// of M = 128 (us), whole recursion against step kernels, by loads:
//   b = 1  2000 rows of 19, FP64        44    518 / 556     1235 / 1351
//          2000 rows of 27, FP32        48    541 / 629     1223 / 1703
//          2000 rows, hub of 21         52    580 / 420     1271 / 1108
//          4000 rows, hub of 11         64    460 / 357     1410 / 835
//          4000 rows of 13              80    534 / 446     1655 / 1029
//          3000 rows of 27, real       160   1379 / 589     3004 / 1509
//   b = 2  1000 rows, hub of 17 (two)   96    495 / 576     1061 / 1429
//          1500 rows of 9              112    452 / 379     1189 / 959
//          1100 rows, hub of 15        208    684 / 432     1450 / 1114
//   b = 4  900 rows of 9, FP32         112    536 / 829     1202 / 2437
//          600 rows of 5               128    506 / 429     1212 / 1193
constexpr int res_max_loads(int b) { return b == 1 ? 48 : b == 2 ? 104 : 120; }

bool find_res(fkpm_handle* h, int rpt) {
  if (h->single)
    return h->cx ? fkd::find_res_fc(h->b, rpt, &h->res.kf) : fkd::find_res_fr(h->b, rpt, &h->res.kf);
  return h->cx ? fkd::find_res_dc(h->b, rpt, &h->res.kd) : fkd::find_res_dr(h->b, rpt, &h->res.kd);
}

// Scalars between the orders of a resident table, and of one order.
size_t res_count(const fkpm_handle* h) { return (size_t)h->n * h->s * (h->cx ? 2 : 1); }
size_t res_slot(const fkpm_handle* h) { return (res_count(h) + 63) / 64 * 64; }

template <class S>
size_t res_lds(fkpm_handle* h) {
  return 2 * (((size_t)(h->nb + 1) * h->rset<S>().elem_bytes + 15) / 16 * 16);
}

// The kernel for rows of at most `deg` blocks, from the blocks each keeps.
int res_mode(int deg, const int (&dreg)[3]) {
  return deg <= dreg[fkd::RES_OWN] ? fkd::RES_OWN
         : deg <= dreg[fkd::RES_REG] ? fkd::RES_REG
                                     : fkd::RES_ST;
}

// Blocks of a row it streams.
int res_streamed(int deg, const int (&dreg)[3]) {
  return res_mode(deg, dreg) == fkd::RES_ST ? deg - dreg[fkd::RES_ST] : 0;
}

// The streamed 16-byte loads of a thread in a step, 0 where its rows are few enough
// for them to overlap.
template <class S>
int res_loads(fkpm_handle* h, int rpt, const int (&dreg)[3]) {
  if (rpt < (h->b == 4 ? 2 : 4)) return 0;
  return res_streamed(h->max_deg, dreg) * rpt * std::max(1, h->rset<S>().block_bytes / 16);
}

// The backward recursion's kernel: the thread's rows of the forward vectors in
// registers where the whole of H still fits beside them, else in LDS where
// four buffers fit (autodiff_matrix of M = 128, us, registers / LDS: 45x42 x 2 FP32 272 /
// 253, 35x36 x 2 FP64 534 / 439, 50x50 x 1 510 / 421, 15^3 x 1 real 422 / 354, 8^3 x 4 FP32
// 331 / 261, FP64 663 / 602).
struct ResBwd {
  int mode, la;  // fkd::ResMode; forward vectors in LDS
  size_t lds;
};

template <class S>
ResBwd res_bwd(fkpm_handle* h) {
  const fkd::ResSet<S>& rs = h->rset<S>();
  const size_t lds = res_lds<S>(h);
  if (h->max_deg <= rs.dreg_bwd[fkd::RES_OWN][0]) return ResBwd{fkd::RES_OWN, 0, lds};
  const int la = h->max_deg > rs.dreg_bwd[fkd::RES_REG][0] && 2 * lds <= kLdsBytes;
  return ResBwd{h->max_deg > rs.dreg_bwd[fkd::RES_REG][la] ? fkd::RES_ST : fkd::RES_REG, la,
                la ? 2 * lds : lds};
}

// Streamed blocks of a workgroup and step from which autodiff_matrix leaves the
// backward recursion to the step kernels, where the forward vectors do not fit the LDS
// beside its own (FP64 complex) and a thread has all its rows: it then streams nearly
// all of H.  autodiff_matrix of M = 128 (us), whole recursion / step kernels recomputing
// alpha from the last two forward vectors:
//   40x40 x 2       8000   478 / 494 (S = 4)   810 / 861 (S = 128)
//   11^3 x 2        9317   590 / 609           917 / 968
//   1500 x 2, 7     10500  612 / 536           673 / 601 (S = 32)
//   57x57 x 1       12996  506 / 399           834 / 772
//   64x64 x 1       16384  538 / 379          1722 / 1480 (S = 256)
//   15^3 x 1        20250  693 / 472 (S = 16) 1074 / 930
// Below an order the two transposed vectors and the outer products at both ends cost
// more than the steps gain (moments + autodiff_matrix, whole / step kernels: 57x57 x 1 M = 16
// 168 / 172, M = 24 212 / 206; 12^3 x 2 M = 64 593 / 597).
constexpr int kResBwdBlocks = 10240;

template <class S>
bool res_bwd_wanted(fkpm_handle* h, int M) {
  if (M < (h->b == 1 ? 24 : 96)) return true;
  const ResBwd rb = res_bwd<S>(h);
  if (rb.mode != fkd::RES_ST || rb.la || h->b == 4 || h->res.rpt < fkd::res_max_rpt(h->b))
    return true;
  const int d = h->max_deg - h->rset<S>().dreg_bwd[fkd::RES_ST][0];
  return (long long)d * h->nb <= kResBwdBlocks;
}

// Whether the whole-recursion kernels run for the current H and R: the
// defaults of every switch that names a step kernel or the table (a forced
// geometry, sweep, order, graph or table mode asks for the step kernels), and a
// column that fits the LDS twice with little of H left to stream (res_max_loads).
template <class S>
bool res_wanted(fkpm_handle* h) {
  if (h->force_L > 0 || h->max_wg > 0 || h->sweep_force >= 0 || h->slice_force >= 0 ||
      h->order_force >= 0 || h->graph_mode == 1 || h->store_alpha != 1 || h->table_cap_mb >= 0 ||
      !h->mfma_on || h->rr_force)
    return false;
  const int rmax = fkd::res_max_rpt(h->b);
  if (h->nb > fkd::RES_T * rmax) return false;
  int rpt = 1;
  while (h->nb > fkd::RES_T * rpt) rpt *= 2;
  if (!find_res(h, rpt)) return false;
  const fkd::ResSet<S>& rs = h->rset<S>();
  if (2 * ((size_t)(h->nb + 1) * rs.elem_bytes + 16) > kLdsBytes) return false;
  if (res_loads<S>(h, rpt, rs.dreg_fwd) > res_max_loads(h->b)) return false;
  const int threads = ((h->nb + rpt - 1) / rpt + 63) / 64 * 64;
  const ResBwd rb = res_bwd<S>(h);
  if (rb.mode == fkd::RES_ST) {
    const int d = h->max_deg - rs.dreg_bwd[fkd::RES_ST][rb.la];
    if ((size_t)d * (rs.block_bytes + 4) * h->nb > kResStream) return false;
  }
  if (rpt != h->res.rpt || threads != h->res.threads) h->res.packed = false;
  h->res.rpt = rpt;
  h->res.threads = threads;
  h->res.nt = rpt * threads;
  return true;
}

// Whether stoch_matrix without a table runs as one launch: not where a step waits for
// streamed blocks longer than the step kernels' launches and columns take.
// stoch_matrix by the Clenshaw recurrence with set_H, M = 128 (us), whole recursion /
// step kernels, by blocks streamed a row:
//   64x64 x 1    2   619 / 621 (S = 4)   627 / 857 (S = 64)
//   45x42 x 2    3   704 / 676 (16)      725 / 985 (128)
//   13^3 x 1     4   838 / 664 (4)       844 / 731 (32)    865 / 1125 (128)
//   12^3 x 2     5   890 / 807 (16)      895 / 904 (32)    896 / 1055 (64)
//   3000 x 1, 9  6  1127 / 748 (4)      1145 / 857 (32)
//   1500 x 1, 17 9   881 / 799 (4)       888 / 792 (32)
//   FP32 x 2 and b = 4 gained at every size: 1900 rows of 9 636 / 968, 8^3 x 4 1004 / 1142
// The step kernels' time grows with the vector from about 512 KiB a streamed block, and
// below M = 16 their start costs more than the steps gain (2197 x 1, 7, M = 8 93 / 121,
// M = 16 139 / 136; 12^3 x 2 171 / 171).
template <class S>
bool res_clenshaw_wanted(fkpm_handle* h, int M) {
  if (M < 16) return true;
  const int d = res_streamed(h->max_deg, h->rset<S>().dreg_xi);
  const int loads = res_loads<S>(h, h->res.rpt, h->rset<S>().dreg_xi);
  const bool waits = h->b == 1 ? loads >= 32 : h->b == 2 && !h->single && loads >= 80;
  return !waits || h->vbytes() >= (size_t)d * (512 << 10);
}

// Room for the tables of forward and (allocated by autodiff_matrix) backward vectors,
// within the budget of the step kernels' table (moments_t).
int res_tables(fkpm_handle* h, size_t abytes, size_t bbytes, bool* ok) {
  fkpm_handle::Resident& r = h->res;
  size_t budget = ~(size_t)0;
  if (abytes > r.atab.bytes) {
    size_t free_b = 0, total_b = 0;
    HIPCHK(hipMemGetInfo(&free_b, &total_b));
    budget = std::min(free_b / 2 + r.atab.bytes + r.btab.bytes, total_b / 4);
  }
  if (const char* e = getenv("FKPM_ALPHA_TABLE_BYTES")) budget = (size_t)strtoull(e, nullptr, 10);
  *ok = abytes + bbytes <= budget;
  if (!*ok) return 0;
  return r.atab.ensure(abytes);
}

template <class S>
fkd::ResH<S> res_H(const fkpm_handle* h) {
  fkd::ResH<S> H;
  H.val = h->res.hval.as<const S>();
  H.off = h->res.hoff.as<const int>();
  H.nb = h->nb;
  H.nt = h->res.nt;
  H.deg = h->max_deg;
  return H;
}

template <class S>
int res_pack(fkpm_handle* h) {
  if (h->res.packed) return 0;
  const fkd::ResSet<S>& rs = h->rset<S>();
  const size_t blocks = (size_t)h->res.nt * h->max_deg;
  CHK(h->res.hval.ensure(blocks * rs.block_bytes + 16));
  CHK(h->res.hoff.ensure(blocks * sizeof(int) + 16));
  if (blocks > 0)
    CHK(launch(rs.pack, dim3(grid_for(blocks)), dim3(fkd::WG), h->stream, h->rp.as<const int>(),
               h->ci.as<const int>(), h->hv.as<const S>(), h->nb, h->res.nt, h->max_deg,
               h->res.hval.as<S>(), h->res.hoff.as<int>()));
  h->res.packed = true;
  return 0;
}

// Coefficients to the device: pinned memory, read by a kernel on the stream.
int res_coef(fkpm_handle* h, const double* c, int M) {
  CHK(h->res.pin.ensure((size_t)M * sizeof(double)));
  CHK(h->res.coef.ensure((size_t)M * sizeof(double)));
  memcpy(h->res.pin.p, c, (size_t)M * sizeof(double));
  return launch(&fkd::k_res_coef, dim3((M + fkd::WG - 1) / fkd::WG), dim3(fkd::WG), h->stream,
                (const double*)h->res.pin.p, h->res.coef.as<double>(), M);
}

// *done = false when the table does not fit (nothing was launched).
template <class S>
int res_moments(fkpm_handle* h, int M, double* mu, bool* done) {
  const int nsteps = M / 2;
  const fkd::ResSet<S>& rs = h->rset<S>();
  const size_t slot = res_slot(h), cnt = res_count(h);
  *done = false;
  bool ok = false;
  h->res.K = 0;
  CHK(res_tables(h, (size_t)(nsteps + 1) * slot * sizeof(S), (size_t)nsteps * slot * sizeof(S), &ok));
  if (!ok) return 0;
  CHK(res_pack<S>(h));
  // about 2048 packets per workgroup of the dots
  const int ny = (int)std::min<size_t>(16, std::max<size_t>(1, cnt * sizeof(S) / 16 / 2048));
  CHK(h->partial.ensure((size_t)nsteps * ny * 2 * sizeof(double)));
  CHK(h->res.pin.ensure((size_t)nsteps * 2 * sizeof(double)));
  CHK(timing_begin(h));
  CHK(launch_lds(rs.fwd[res_mode(h->max_deg, rs.dreg_fwd)], dim3(h->s), dim3(h->res.threads), res_lds<S>(h), h->stream,
                 res_H<S>(h), h->R.as<const S>(), h->sp, h->res.atab.as<S>(), slot, nsteps));
  CHK(timing_end(h, &h->ms_mom, &h->n_mom, 1));
  CHK(launch(&fkd::k_res_dots<S>, dim3(nsteps, ny), dim3(fkd::WG), h->stream,
             h->res.atab.as<const S>(), slot, cnt, h->partial.as<double>()));
  double* ps = static_cast<double*>(h->res.pin.p);
  CHK(launch(&fkd::k_reduce_partials, dim3(nsteps), dim3(fkd::WG), h->stream,
             (const double*)h->partial.as<double>(), ny, ps));
  HIPCHK(hipStreamSynchronize(h->stream));
  moments_from_sums(ps, nsteps, mu);
  h->res.K = nsteps;
  h->res.state = true;
  h->a_slots = 0;
  h->alpha_M = M;
  *done = true;
  return 0;
}

// dst = the D sum over the terms T (nterm of them) on D's pattern.
template <class S>
int res_outer(fkpm_handle* h, const fkd::ResTerms<S>& T, int nterm, double* dst) {
  const size_t cnt = (size_t)h->nnzbD * h->b * h->b * (h->cx ? 2 : 1);
  if (cnt == 0) return 0;
  const int gx = (h->nnzbD + fkd::WG - 1) / fkd::WG;
  const long long pairs = (long long)nterm * h->s;
  // about 2048 workgroups, at least 16 products a thread, 64 MiB of partial sums
  long long ny = std::min<long long>({std::max(1, 2048 / gx), (pairs + 15) / 16,
                                      std::max<long long>(1, (64ll << 20) / (long long)(cnt * 8))});
  const int per = (int)((pairs + ny - 1) / ny);
  ny = (pairs + per - 1) / per;
  CHK(h->res.part.ensure((size_t)ny * cnt * sizeof(double)));
  const dim3 grid(gx, (int)ny), block(fkd::WG);
  auto go = [&](auto fn) {
    return launch(fn, grid, block, h->stream, h->drp.as<const int>(), h->dci.as<const int>(), h->nb,
                  h->nnzbD, T, nterm, h->s, per, h->res.part.as<double>());
  };
  int rc = FKPM_E_UNSUP;
  if (h->b == 1) rc = h->cx ? go(&fkd::k_res_outer<S, true, 1>) : go(&fkd::k_res_outer<S, false, 1>);
  if (h->b == 2) rc = h->cx ? go(&fkd::k_res_outer<S, true, 2>) : go(&fkd::k_res_outer<S, false, 2>);
  if (h->b == 4) rc = h->cx ? go(&fkd::k_res_outer<S, true, 4>) : go(&fkd::k_res_outer<S, false, 4>);
  CHK(rc);
  return sum_parts(h, h->res.part.as<const double>(), (int)ny, cnt, dst, false);
}

// alpha_{M/2-1} and alpha_{M/2} of the resident table into the step kernels' ring.
template <class S>
int res_to_ring(fkpm_handle* h, int M) {
  const dim3 grid((h->n + fkd::RES_TILE - 1) / fkd::RES_TILE,
                  (h->sp + fkd::RES_TILE - 1) / fkd::RES_TILE);
  for (int k = M / 2 - 1; k <= M / 2; k++)
    CHK(launch(h->cx ? &fkd::k_res_to_rows<S, true> : &fkd::k_res_to_rows<S, false>, grid,
               dim3(fkd::WG), h->stream, h->res.atab.as<const S>() + (size_t)k * res_slot(h), h->n,
               h->s, h->sp, h->A[k % 3].as<S>()));
  return 0;
}

// The backward recursion and D from the resident table, into dacc.
template <class S>
int res_autodiff(fkpm_handle* h, int M, const double* c, double diag) {
  const int M2 = M / 2;
  const fkd::ResSet<S>& rs = h->rset<S>();
  const size_t slot = res_slot(h);
  CHK(timing_begin(h));
  if (M2 > 1) {
    CHK(res_coef(h, c, M));
    const ResBwd rb = res_bwd<S>(h);
    CHK(launch_lds(rs.bwd[rb.mode][rb.la], dim3(h->s), dim3(h->res.threads), rb.lds, h->stream,
                   res_H<S>(h), h->res.atab.as<const S>(), h->res.btab.as<S>(), slot, M2,
                   h->res.coef.as<const double>(), 2 * c[M - 1]));
  }
  fkd::ResTerms<S> T{h->res.atab.as<const S>(), h->res.btab.as<const S>(), slot, M2, diag,
                     2 * c[M - 1]};
  CHK(res_outer<S>(h, T, M2 > 1 ? M2 + 1 : 1, h->dacc.as<double>()));
  return timing_end(h, &h->ms_ad, &h->n_ad, M2 > 1 ? 1 : 0);
}

// xi by the Clenshaw recurrence, or from the resident table, then D into dout.
template <class S>
int res_stoch(fkpm_handle* h, int M, const double* c, bool table) {
  const size_t slot = res_slot(h), vb = slot * sizeof(S);
  const fkd::ResSet<S>& rs = h->rset<S>();
  CHK(res_pack<S>(h));
  CHK(h->res.xi.ensure(3 * vb));
  S* u = h->res.xi.as<S>();
  S* v = u + slot;
  S* xi = v + slot;
  const int K = (M + 1) / 2;
  std::vector<double> w;
  if (table) {
    stoch_table_weights(M, c, w);
    CHK(res_coef(h, w.data(), (int)w.size()));
    CHK((table_sums<S, 2>(h, h->res.atab.as<const S>(), h->res.atab.as<const S>() + slot, slot, K,
                          h->res.coef.as<const double>(), v, u)));
  } else {
    CHK(res_coef(h, c, M));
  }
  const S* r0 = table ? h->res.atab.as<const S>() : u;
  CHK(launch_lds(rs.xi[res_mode(h->max_deg, rs.dreg_xi)], dim3(h->s), dim3(h->res.threads), res_lds<S>(h), h->stream,
                 res_H<S>(h), h->R.as<const S>(), h->sp, (const S*)(table ? u : nullptr),
                 (const S*)v, h->res.coef.as<const double>(), table ? K : M, u, xi));
  return res_outer<S>(h, fkd::ResTerms<S>{r0, xi, slot, 0, 0.0, 0.0}, 2, h->dout.as<double>());
}

// ---------------------------------------------------------------------------
// moments (engine_cpu.cpp:63-84; engine_cusparse.cpp:755-791)
// ---------------------------------------------------------------------------
template <class S>
int moments_t(fkpm_handle* h, int M, double* mu) {
  const int nsteps = M / 2;
  if (res_wanted<S>(h)) {
    bool done = false;
    CHK(res_moments<S>(h, M, mu, &done));
    if (done) return 0;
  }
  h->res.state = false;
  CHK(ensure_partials(h, nsteps));
  // Keep the alpha_k for autodiff_matrix (no backward recomputation of alpha) and
  // stoch_matrix when wanted (table_wanted): all of them where the table fits
  // half the free device memory (or the byte count in FKPM_ALPHA_TABLE_BYTES),
  // else as many as fit from a third of M on, the first ones (64^3 x 2 FP64, S = 128,
  // M = 160, 67 of 80 kept: moments + autodiff_matrix + stoch_matrix 305 -> 258 ms).
  h->a_slots = 0;
  if (table_wanted(h) && !table_idle(h)) {
    const size_t vb = h->vbytes(), need = (size_t)nsteps * vb;
    const int least = (M + 2) / 3;
    // default: half of what is free (the table already held counts as free),
    // never more than a quarter of the device, so that other engines and a
    // batch arena on the same device keep room whatever the order of calls
    size_t budget = h->total_bytes / 4;
    if (need > h->atab.bytes || h->total_bytes == 0) {  // else the held table is big enough
      size_t free_b = 0;
      HIPCHK(hipMemGetInfo(&free_b, &h->total_bytes));
      budget = std::min(free_b / 2 + h->atab.bytes, h->total_bytes / 4);
    }
    if (h->table_cap_mb >= 0) budget = (size_t)h->table_cap_mb << 20;
    if (const char* e = getenv("FKPM_ALPHA_TABLE_BYTES")) budget = (size_t)strtoull(e, nullptr, 10);
    size_t slots = std::min<size_t>(budget / vb, nsteps);
    // a held table that serves is not grown for a few slots more
    if (slots < (size_t)nsteps && h->atab.bytes / vb >= (size_t)least)
      slots = std::min(slots, h->atab.bytes / vb);
    if (slots >= (size_t)std::min(least, nsteps)) {
      h->tab_K = 0;  // rewritten below (and lost if the table grows)
      CHK(h->atab.ensure(slots * vb));
      h->a_slots = (int)slots;
    }
  }
  h->unread = std::min(h->unread + 1, kUnread);
  const dim3 block(fkd::WG);
  CHK(timing_begin(h));
  {
    LoopRecorder rec(h);
    // alpha_{m+1} = cx Hs alpha_m + cz alpha_{m-1}, into the table, then the ring
    for (int m0 = 0; m0 < nsteps;) {
      const int kind = m0 < h->a_slots ? K_MOMT : K_MOM;
      const KCfg& kc = h->kc[kind];
      const auto& ks = h->ks<S>(kind);
      const int m1 = std::min(m0 + partial_steps(nsteps, kc.nwg), kind == K_MOMT ? h->a_slots : nsteps);
      for (int m = m0; m < m1; m++) {
        const S* x = (const S*)h->vec_a(m);
        const S* z = m == 0 ? nullptr : (const S*)h->vec_a(m - 1);
        S* y = (S*)h->vec_a(m + 1);
        CHK(launch(mom_fn(h, ks, kc), dim3(kc.nwg), block, h->stream, rp_for(h, kc),
                   h->ci.as<const int>(), h->hv.as<const S>(), x, z, y, h->nb, h->qp, kc.chunk,
                   m == 0 ? 1.0 : 2.0, m == 0 ? 0.0 : -1.0,
                   h->partial.as<double>() + (size_t)(m - m0) * kc.nwg * 2, nt_for(h, kc),
                   no_rsource<S>()));
      }
      CHK(launch(&fkd::k_reduce_partials, dim3(m1 - m0), block, h->stream,
                 (const double*)h->partial.as<double>(), kc.nwg, (double*)h->psum.p + 2 * m0));
      m0 = m1;
    }
    CHK(rec.run());
  }
  CHK(timing_end(h, &h->ms_mom, &h->n_mom, nsteps));
  if (h->a_slots > 0) {
    h->tab_K = h->a_slots;
    h->tab_M = M;
  }
  HIPCHK(hipStreamSynchronize(h->stream));
  moments_from_sums((const double*)h->psum.p, nsteps, mu);
  h->alpha_M = M;
  return 0;
}

// A large copy to pageable memory runs at the rate of one core copying out of
// pinned memory (17 GB/s), a third of the link's: from kBigCopy on, four threads
// copy chunks out of a ring of pinned buffers while the next chunks arrive
// (117 MB: 6.9 -> 2.7 ms).  Memory that the runtime knows (pinned, registered) takes
// the link's full rate by itself (57 MB: 1.0 ms, through the ring 1.5).
constexpr size_t kBigCopy = 16 << 20, kCopyChunk = 2 << 20;
constexpr int kCopyThreads = 4;

bool pageable(const void* p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
  (void)hipGetLastError();  // not an address of the runtime's: no error of ours
  return true;
}

int copy_to_host(fkpm_handle* h, void* dst, const void* src, size_t bytes) {
  if (bytes < kBigCopy || !pageable(dst)) {
    HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, h->stream));
    HIPCHK(hipStreamSynchronize(h->stream));
    return 0;
  }
  CHK(h->dpin.ensure(2 * kCopyThreads * kCopyChunk));
  while (h->dpin_ev.size() < 2 * kCopyThreads) {
    hipEvent_t e = nullptr;
    HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    h->dpin_ev.push_back(e);
  }
  const size_t n = (bytes + kCopyChunk - 1) / kCopyChunk;
  std::atomic<int> err{hipSuccess};
  // thread w takes chunks w, w + kCopyThreads, ..., two of them under way
  auto work = [&](int w) {
    auto note = [&](hipError_t e) {
      if (e != hipSuccess) err = e;
      return e == hipSuccess;
    };
    if (!note(hipSetDevice(h->device))) return;
    auto slot = [&](size_t i) { return 2 * w + (int)(i / kCopyThreads & 1); };
    auto len = [&](size_t i) { return std::min(kCopyChunk, bytes - i * kCopyChunk); };
    auto fetch = [&](size_t i) {
      return i >= n ||
             (note(hipMemcpyAsync((char*)h->dpin.p + slot(i) * kCopyChunk,
                                  (const char*)src + i * kCopyChunk, len(i), hipMemcpyDeviceToHost,
                                  h->stream)) &&
              note(hipEventRecord(h->dpin_ev[slot(i)], h->stream)));
    };
    if (!fetch(w) || !fetch(w + kCopyThreads)) return;
    for (size_t i = w; i < n; i += kCopyThreads) {
      if (!note(hipEventSynchronize(h->dpin_ev[slot(i)]))) return;
      memcpy((char*)dst + i * kCopyChunk, (const char*)h->dpin.p + slot(i) * kCopyChunk, len(i));
      if (!fetch(i + 2 * kCopyThreads)) return;
    }
  };
  std::thread pool[kCopyThreads];
  int started = 1;
  try {
    for (; started < kCopyThreads; started++) pool[started] = std::thread(work, started);
  } catch (const std::exception&) {
    // no thread to be had: this one takes the remaining chunks below
  }
  work(0);
  for (int w = started; w < kCopyThreads; w++) work(w);
  for (int w = 1; w < started; w++) pool[w].join();
  HIPCHK((hipError_t)err.load());
  HIPCHK(hipStreamSynchronize(h->stream));
  return 0;
}

// D to the host in the engine type.  Single-precision engines round on the
// device (k_round_D), so half the bytes cross PCIe and no host pass follows.
int copy_D_out(fkpm_handle* h, void* D_val) {
  const size_t cnt = (size_t)h->nnzbD * h->b * h->b * (h->cx ? 2 : 1);
  const void* src = h->dout.p;
  size_t bytes = cnt * sizeof(double);
  if (dtype_single(h->dtype)) {
    bytes = cnt * sizeof(float);
    CHK(h->dout_f.ensure(bytes > 0 ? bytes : 16));
    CHK(launch(&fkd::k_round_D, dim3(grid_for(cnt)), dim3(256), h->stream,
               (const double*)h->dout.as<double>(), h->dout_f.as<float>(), cnt));
    src = h->dout_f.p;
  }
  return copy_to_host(h, D_val, src, bytes);
}

int check_D_ready(fkpm_handle* h) {
  if (!h->d_set) return fail(FKPM_E_STATE, "D pattern has not been set");
  if (h->nbD != h->nb)
    return fail(FKPM_E_ARG, "D has %d block rows but H has %d", h->nbD, h->nb);
  const size_t dbytes = (size_t)h->nnzbD * h->b * h->b * (h->cx ? 2 : 1) * sizeof(double);
  CHK(h->dacc.ensure(dbytes > 0 ? dbytes : 16));
  CHK(h->dout.ensure(dbytes > 0 ? dbytes : 16));
  h->d_fused = (h->hd_rp == h->h_rp && h->hd_ci == h->h_ci);
  return 0;
}

// ---------------------------------------------------------------------------
// stoch_matrix (engine_cpu.cpp:229-253; engine_cusparse.cpp:910-953)
// ---------------------------------------------------------------------------

// xi = sum_{m<M} c_m T_m(Hs) R by the Clenshaw recurrence
//   b_{M-1} = c_{M-1} R, b_M = 0,
//   b_k = c_k R + 2 Hs b_{k+1} - b_{k+2}   (k = M-2 .. 1),
//   xi = c_0 R + Hs b_1 - b_2,
// one SpMM pass per step reading two vectors (no FP64 accumulator traffic);
// b_{M-1} stays virtual (a multiple of R).  Returns xi's buffer.
template <class S>
int stoch_clenshaw(fkpm_handle* h, int M, const double* c, const S** xi_out) {
  const KCfg& kc = h->kc[K_MOM];
  const auto& ks = h->ks<S>(K_MOM);
  const dim3 grid(kc.nwg), block(fkd::WG);
  const S* R = (const S*)h->R.p;
  struct Vb {
    const S* p;
    double s;
  };
  Vb b1{R, c[M - 1]}, b2{nullptr, 0.0};
  int slot = 0, launches = 0;
  auto step = [&](double xfac, double cr, S* y) -> int {
    return launch(mom_fn(h, ks, kc), grid, block, h->stream, rp_for(h, kc), h->ci.as<const int>(),
                  h->hv.as<const S>(), b1.p, b2.p, y, h->nb, h->qp, kc.chunk, xfac * b1.s,
                  b2.p ? -b2.s : 0.0, (double*)nullptr, nt_for(h, kc), rsource<S>(h, cr));
  };
  for (int k = M - 2; k >= 1; k--) {
    S* y = (S*)h->A[slot].p;
    slot = (slot + 1) % 3;
    CHK(step(2.0, c[k], y));
    launches++;
    b2 = b1;
    b1 = Vb{y, 1.0};
  }
  S* y = (S*)h->A[slot].p;
  CHK(step(1.0, c[0], y));
  *xi_out = y;
  return launches + 1;
}

// f T_K(Hs) x + add for the vector x in A[*slot], by K Chebyshev steps
// (y_0 = x, y_1 = Hs x, y_{k+1} = 2 Hs y_k - y_{k-1}, the last one scaled by f with
// `add` as its source); *slot is then the result's place in the ring.
template <class S>
int chebyshev_of(fkpm_handle* h, int K, double f, const S* add, int* slot) {
  const KCfg& kc = h->kc[K_MOM];
  const auto& ks = h->ks<S>(K_MOM);
  fkd::RSource<S> src = no_rsource<S>();
  src.rd = add;
  src.cr = 1.0;
  const S* x = (const S*)h->A[*slot].p;
  const S* z = nullptr;
  for (int k = 0; k < K; k++) {
    *slot = (*slot + 1) % 3;
    S* y = (S*)h->A[*slot].p;
    const double g = k == K - 1 ? f : 1.0;
    CHK(launch(mom_fn(h, ks, kc), dim3(kc.nwg), dim3(fkd::WG), h->stream, rp_for(h, kc),
               h->ci.as<const int>(), h->hv.as<const S>(), x, z, y, h->nb, h->qp, kc.chunk,
               (k == 0 ? 1.0 : 2.0) * g, k == 0 ? 0.0 : -g, (double*)nullptr, nt_for(h, kc),
               k == K - 1 ? src : no_rsource<S>()));
    z = x;
    x = y;
  }
  return 0;
}

// xi from the kept forward vectors alpha_0 .. alpha_K (K = ceil(M/2), coefficients
// padded with zeros to 2K): by T_{K+j} = 2 T_K T_j - T_{K-j},
//   xi = sum_{m<2K} c_m T_m(Hs) R = v + 2 T_K(Hs) u,
//   v = sum_{i=0..K} ([i<K] c_i - [i>=1] c_{2K-i}) alpha_i,
//   u = sum_{i<K} c_{K+i} alpha_i,
// one streaming pass over the table (k_table_sums) and K Chebyshev steps
// from u, the last adding v as its source term: about 4K + 4 vector
// transfers instead of the 3(M - 1) of the Clenshaw recurrence.  Returns
// xi's buffer.
template <class S>
int stoch_table(fkpm_handle* h, int M, const double* c, const S** xi_out) {
  const int K = (M + 1) / 2;
  const size_t n = h->vbytes() / sizeof(S);
  std::vector<double>& w = h->tabc_host;
  stoch_table_weights(M, c, w);
  CHK(h->tabc.ensure(w.size() * sizeof(double)));
  HIPCHK(hipMemcpyAsync(h->tabc.p, w.data(), w.size() * sizeof(double), hipMemcpyHostToDevice,
                        h->stream));
  CHK(h->Bv[0].ensure(h->vbytes()));
  S* u = (S*)h->A[0].p;
  S* v = (S*)h->Bv[0].p;
  CHK((table_sums<S, 2>(h, (const S*)h->R.p, (const S*)h->atab.p, n, K, h->tabc.as<const double>(),
                        v, u)));
  int slot = 0;
  CHK(chebyshev_of<S>(h, K, 2.0, v, &slot));
  *xi_out = (const S*)h->A[slot].p;
  return K + 1;
}

// xi from the first forward vectors alpha_0 .. alpha_{K-1} only, K = ceil(M/3)
// (coefficients padded with zeros to 3K): by T_{jK+i} = 2 T_{jK} T_i - T_{(j-1)K+(K-i)},
// from j = 2 down,
//   xi = w_0 + T_K(Hs) w_1 + T_{2K}(Hs) w_2 = (w_0 - w_2) + T_K(Hs) (w_1 + 2 T_K(Hs) w_2),
// w_j sums of the alpha_i: 2K steps and one pass over K vectors instead of M - 1
// steps.  Returns xi's buffer.
template <class S>
int stoch_table3(fkpm_handle* h, int M, const double* c, const S** xi_out) {
  const int K = (M + 2) / 3;
  const size_t n = h->vbytes() / sizeof(S);
  std::vector<double>& w = h->tabc_host;
  stoch_table3_weights(M, c, w);
  CHK(h->tabc.ensure(w.size() * sizeof(double)));
  HIPCHK(hipMemcpyAsync(h->tabc.p, w.data(), w.size() * sizeof(double), hipMemcpyHostToDevice,
                        h->stream));
  for (int k = 0; k < 2; k++) CHK(h->Bv[k].ensure(h->vbytes()));
  S* v = (S*)h->Bv[0].p;
  S* w1 = (S*)h->Bv[1].p;
  CHK((table_sums<S, 3>(h, (const S*)h->R.p, (const S*)h->atab.p, n, K, h->tabc.as<const double>(),
                        v, w1, (S*)h->A[0].p)));
  int slot = 0;
  CHK(chebyshev_of<S>(h, K, 2.0, w1, &slot));
  CHK(chebyshev_of<S>(h, K, 1.0, v, &slot));
  *xi_out = (const S*)h->A[slot].p;
  return 2 * K + 1;
}

template <class S>
int stoch_t(fkpm_handle* h, int M, const double* c) {
  h->a_slots = 0;  // the forward method's alpha_k go to the ring
  h->unread = 0;
  const dim3 block(fkd::WG);
  const int* rp = h->rp.as<const int>();
  const int* ci = h->ci.as<const int>();
  const S* hv = h->hv.as<const S>();
  const size_t dcount = (size_t)h->nnzbD * h->b * h->b * (h->cx ? 2 : 1);
  const KCfg& ko = h->kc[K_OUT];
  const auto& kso = h->ks<S>(K_OUT);
  const bool res_table = h->stoch_method == FKPM_STOCH_AUTO && h->res.K >= (M + 1) / 2;
  if (h->stoch_method != FKPM_STOCH_FORWARD && res_wanted<S>(h) &&
      (res_table || res_clenshaw_wanted<S>(h, M))) {
    const bool table = res_table;
    h->stoch_used = table ? FKPM_STOCH_TABLE : FKPM_STOCH_CLENSHAW;
    CHK(timing_begin(h));
    CHK(res_stoch<S>(h, M, c, table));
    CHK(timing_end(h, &h->ms_stoch, &h->n_stoch, table ? 2 : 1));
    h->alpha_M = 0;
    return 0;
  }
  CHK(timing_begin(h));
  const bool table = h->stoch_method == FKPM_STOCH_AUTO && h->tab_K >= (M + 1) / 2;
  // a table cut short by the memory, up to the order it was kept for
  const bool table3 = !table && h->stoch_method == FKPM_STOCH_AUTO && M <= h->tab_M &&
                      h->tab_K >= (M + 2) / 3;
  h->stoch_used = table || table3 ? FKPM_STOCH_TABLE
                        : h->stoch_method == FKPM_STOCH_FORWARD ? FKPM_STOCH_FORWARD
                                                                : FKPM_STOCH_CLENSHAW;
  if (h->stoch_used != FKPM_STOCH_FORWARD) {
    const S* xi = nullptr;
    int launches = 0;
    {
      LoopRecorder rec(h);
      launches = table    ? stoch_table<S>(h, M, c, &xi)
                 : table3 ? stoch_table3<S>(h, M, c, &xi)
                          : stoch_clenshaw<S>(h, M, c, &xi);
      if (launches < 0) return launches;
      CHK(rec.run());
    }
    CHK(timing_end(h, &h->ms_stoch, &h->n_stoch, launches));
    CHK(zero_doubles(h, h->dacc.p, dcount));
    // D = (1/2) R xi^+ + (1/2) xi R^+
    CHK(add_outer<S>(h, (const S*)h->R.p, xi, 0.5));
    CHK(add_outer<S>(h, xi, (const S*)h->R.p, 0.5));
  } else {
    // the reference's order: forward recursion, xi accumulated in FP64
    CHK(h->xi.ensure(h->accbytes()));
    const KCfg& kx = h->kc[K_XI];
    const auto& ksx = h->ks<S>(K_XI);
    const dim3 grid(kx.nwg, xi_apart(h, kx));
    {
      LoopRecorder rec(h);
      // alpha_1 = Hs R, xi = c0 R + c1 alpha_1
      CHK(launch(xi_fn(h, ksx, kx), grid, block, h->stream, rp_for(h, kx), ci, hv,
                 (const S*)h->vec_a(0), (const S*)nullptr, (S*)h->vec_a(1),
                 h->xi.as<double>(), h->nb, h->qp, kx.chunk, 1.0, 0.0, c[0], c[1], 1,
                 nt_for(h, kx)));
      for (int m = 2; m < M; m++) {
        // alpha_m = 2 Hs alpha_{m-1} - alpha_{m-2}; xi += c_m alpha_m
        CHK(launch(xi_fn(h, ksx, kx), grid, block, h->stream, rp_for(h, kx), ci, hv,
                   (const S*)h->vec_a(m - 1),
                   (const S*)h->vec_a(m - 2), (S*)h->vec_a(m), h->xi.as<double>(), h->nb, h->qp,
                   kx.chunk, 2.0, -1.0, 0.0, c[m], 0, nt_for(h, kx)));
      }
      CHK(rec.run());
    }
    CHK(timing_end(h, &h->ms_stoch, &h->n_stoch, M - 1));
    CHK(zero_doubles(h, h->dacc.p, dcount));
    CHK(launch(kso.outer_sd, dim3(ko.nwg), block, h->stream, h->drp.as<const int>(),
               h->dci.as<const int>(), (const S*)h->vec_a(0), (const double*)h->xi.as<double>(),
               h->dacc.as<double>(), h->nb, h->qp, ko.chunk, 0.5));
    CHK(launch(kso.outer_ds, dim3(ko.nwg), block, h->stream, h->drp.as<const int>(),
               h->dci.as<const int>(), (const double*)h->xi.as<double>(), (const S*)h->vec_a(0),
               h->dacc.as<double>(), h->nb, h->qp, ko.chunk, 0.5));
  }
  HIPCHK(hipMemcpyAsync(h->dout.p, h->dacc.p, dcount * sizeof(double), hipMemcpyDeviceToDevice,
                        h->stream));
  h->alpha_M = 0;  // engine_cpu.cpp:250-252
  return 0;
}

// ---------------------------------------------------------------------------
// autodiff_matrix (engine_cpu.cpp:255-304; engine_cusparse.cpp:955-1039)
// ---------------------------------------------------------------------------
// D = (symmetrized dacc) / mag into dout; the end of autodiff_matrix.
int finish_autodiff(fkpm_handle* h) {
  const double* dacc = h->dacc.as<const double>();
  // symmetrize + scale(1/mag)
  const size_t dcnt = (size_t)h->nnzbD * h->b * h->b;
  if (h->cx)
    CHK(launch(&fkd::k_symmetrize_scale<true>, dim3(grid_for(dcnt)), dim3(256), h->stream,
               (const double*)dacc, h->dout.as<double>(), h->tpos.as<const int>(), h->nnzbD, h->b,
               1.0 / h->mag));
  else
    CHK(launch(&fkd::k_symmetrize_scale<false>, dim3(grid_for(dcnt)), dim3(256), h->stream,
               (const double*)dacc, h->dout.as<double>(), h->tpos.as<const int>(), h->nnzbD, h->b,
               1.0 / h->mag));
  h->alpha_M = 0;  // engine_cpu.cpp:301-303
  return 0;
}

// Whether the fused backward steps compute alpha_{m-1} anew although the table holds
// it.  Real 8-row blocks on a wave a row: of the step that recomputes one wave fits a
// SIMD, of the one that reads two, and while the rows are one wave for each of 1024
// SIMDs the first is the shorter chain.  autodiff_matrix of M = 64, recomputed / read
// (us): FP64 x 128 6^3 1852 / 2170, 10^3 2177 / 2484, 32x32 1640 / 1870, 11^3 (1331 rows)
// 3925 / 3052; FP32 x 256 32x32 1542 / 1739, 36x36 2751 / 2142.  On D's own pattern
// reading is the faster everywhere (10^3 FP64 1091 / 1013).
constexpr int kOneWaveRows = 1024;

bool ad_recomputes(const fkpm_handle* h) {
  const KCfg& a = h->kc[K_AD];
  return h->store_alpha == 1 && h->b == 8 && !h->cx && a.L == fkd::WAVE && h->d_fused &&
         h->nb <= kOneWaveRows;
}

template <class S>
int autodiff_t(fkpm_handle* h, int M, const double* c) {
  const dim3 block(fkd::WG);
  const KCfg& ka = h->kc[K_AD];
  const KCfg& kt = h->kc[K_ADS];
  const auto& ksa = h->ks<S>(K_AD);
  const auto& kst = h->ks<S>(K_ADS);
  const int* rp = h->rp.as<const int>();
  const int* ci = h->ci.as<const int>();
  const S* hv = h->hv.as<const S>();
  double* dacc = h->dacc.as<double>();
  const size_t dcount = (size_t)h->nnzbD * h->b * h->b * (h->cx ? 2 : 1);

  double diag = c[1];
  for (int m = 1; m < M / 2; m++) diag -= c[2 * m + 1];
  h->unread = 0;
  if (h->res.state) {
    // without room for the backward vectors (taken since moments) too, the ring serves
    const size_t bytes = (size_t)(M / 2) * res_slot(h) * sizeof(S);
    if (M == 2 || (res_bwd_wanted<S>(h, M) && h->res.btab.ensure(bytes) == 0)) {
      CHK(res_autodiff<S>(h, M, c, diag));
      return finish_autodiff(h);
    }
    CHK(res_to_ring<S>(h, M));  // and on with the ring's steps
  }
  CHK(zero_doubles(h, dacc, dcount));
  // D = diag R R^+
  CHK(add_outer<S>(h, (const S*)h->vec_a(0), (const S*)h->vec_a(0), diag));
  int launches = 0;
  if (M > 2)
    for (int k = 0; k < 3; k++) CHK(h->Bv[k].ensure(h->vbytes()));
  CHK(timing_begin(h));
  LoopRecorder rec(h);
  if (M > 2) {
    const bool again = ad_recomputes(h);
    const double sb = 2 * c[M - 1];  // beta_{M/2} = 2 c_{M-1} alpha_{M/2-1}
    for (int m = M / 2 - 1; m >= 1; m--) {
      // alpha_{m-1}: from the table, or recomputed into the ring by the step
      const bool stored = h->a_slots > 0 && m - 1 <= h->a_slots && !again;
      const S* am = (const S*)h->vec_a(m);
      const S* am1 = (const S*)h->vec_a(m + 1);
      S* aout = stored ? (S*)h->vec_a(m - 1) : (S*)h->A[(m - 1) % 3].p;
      const bool first = (m == M / 2 - 1);
      const bool second = (m == M / 2 - 2);
      const S* bm1 = first ? nullptr : (const S*)h->Bv[(m + 1) % 3].p;
      const S* bm2 = (first || second) ? nullptr : (const S*)h->Bv[(m + 2) % 3].p;
      const double sb2 = second ? sb : 0.0;
      S* bout = (S*)h->Bv[m % 3].p;
      const double c4 = 4 * c[2 * m], c2 = 2 * c[2 * m + 1];
      const double w = m > 1 ? 2 * c[2 * m - 1] : 0.0;
      if (stored) {
        if (!h->d_fused)  // D += 2 alpha_m beta_{m+1}^+ on D's own pattern
          CHK(add_outer<S>(h, am, first ? am : bm1, first ? 2.0 * sb : 2.0));
        CHK(launch(h->d_fused ? ads_fn(h, kst, kt) : adsp_fn(kst, kt), dim3(kt.nwg), block,
                   h->stream, rp_for(h, kt), ci, hv, am, am1, bm1, bm2, (const S*)aout, bout, dacc,
                   h->nb, h->qp, kt.chunk, c4, c2, w, sb, sb2, 2.0, nt_for(h, kt)));
      } else if (h->d_fused) {
        CHK(launch(adf_fn(h, ksa, ka), dim3(ka.nwg), block, h->stream, rp_for(h, ka), ci, hv, am, am1,
                   bm1, bm2,
                   aout, bout, dacc, h->nb, h->qp, ka.chunk, c4, c2, w, sb, sb2, 2.0, nt_for(h, ka)));
      } else {
        // D += 2 alpha_m beta_{m+1}^+ on D's own pattern, then the step.
        CHK(add_outer<S>(h, am, first ? am : bm1, first ? 2.0 * sb : 2.0));
        CHK(launch(adp_fn(ksa, ka), dim3(ka.nwg), block, h->stream, rp_for(h, ka), ci, hv, am, am1,
                   bm1, bm2,
                   aout, bout, dacc, h->nb, h->qp, ka.chunk, c4, c2, w, sb, sb2, 2.0, nt_for(h, ka)));
      }
      launches++;
    }
    // D += alpha_0 beta_1^+ (alpha_0 = R kept, or recomputed into A[0])
    CHK(add_outer<S>(h, (const S*)(h->a_slots > 0 ? h->R.p : h->A[0].p), (const S*)h->Bv[1].p, 1.0));
  }
  CHK(rec.run());
  CHK(timing_end(h, &h->ms_ad, &h->n_ad, launches));
  return finish_autodiff(h);
}

// ---------------------------------------------------------------------------
// Two-current moments (Engine_CPU::moments2_v1, engine_cpu.cpp:86-160;
// engine_cusparse.cpp:793-902):
//   mu[m1][m2] = sum_k <alpha_m1(k), j2 atild_m2(k)>,
//   alpha_m(k) = T_m(Hs) r_k,  atild_m(k) = T_m(Hs) j1 r_k.
// For a chunk of probe columns all M alpha_m and all M j2 atild_m are kept in
// HBM as the columns of two K x M matrices (K = n * padded columns), built by
// the step kernels (j1, j2 on their own block patterns), and the M x M block
// of dots A^H B is formed on the matrix cores (kpm_dots.h), accumulated in
// FP64 over chunks.
// ---------------------------------------------------------------------------

// The kernel set and geometry for a pass width of W packets (a compiled
// (L, KQ) with L * KQ == W, widest lane groups first).
template <class S>
bool kset_for_width(fkpm_handle* h, int W, fkd::KSet<S>* ks, int* L, int* KQ);
template <>
bool kset_for_width<double>(fkpm_handle* h, int W, fkd::KSet<double>* ks, int* L, int* KQ) {
  fkd::GeomChoice gs[64];
  const int ng = fkd::geometries_for_block(h->b, gs, 64);
  for (int want = 64; want >= 1; want /= 2)
    for (int k = 0; k < ng; k++)
      if (gs[k].L == want && gs[k].L * gs[k].KQ == W) {
        *L = gs[k].L;
        *KQ = gs[k].KQ;
        return h->cx ? fkd::find_kset_dc(h->b, *L, *KQ, ks) : fkd::find_kset_dr(h->b, *L, *KQ, ks);
      }
  return false;
}
template <>
bool kset_for_width<float>(fkpm_handle* h, int W, fkd::KSet<float>* ks, int* L, int* KQ) {
  fkd::GeomChoice gs[64];
  const int ng = fkd::geometries_for_block(h->b, gs, 64);
  for (int want = 64; want >= 1; want /= 2)
    for (int k = 0; k < ng; k++)
      if (gs[k].L == want && gs[k].L * gs[k].KQ == W) {
        *L = gs[k].L;
        *KQ = gs[k].KQ;
        return h->cx ? fkd::find_kset_fc(h->b, *L, *KQ, ks) : fkd::find_kset_fr(h->b, *L, *KQ, ks);
      }
  return false;
}

// C (M x M, FP64, row-major (m1, m2)) = [C +] A^H B for K x M matrices A, B
// of the storage type (column m at A + m * ld): k_dot_block over slices of
// 512 k interleaved across about 2048 workgroups, then k_sum_parts adding
// the grid rows' partial blocks in order (at most 1 GiB of them).
template <class S>
int dot_block_acc(fkpm_handle* h, const S* A, const S* B, long long K, long long ld, int M,
                  bool first) {
  const int HS = h->cx ? 2 : 1;
  const int nbm = (M + fkd::DOT_BM - 1) / fkd::DOT_BM;
  const int nblk = nbm * nbm;
  const long long kslice = 512;
  const size_t cnt = (size_t)M * M * HS;
  const long long nslices = (K + kslice - 1) / kslice;
  long long ny = std::max(1, 2048 / nblk);
  ny = std::min(ny, nslices);
  ny = std::min<long long>(ny, std::max<long long>(1, ((size_t)1 << 30) / (cnt * sizeof(double))));
  ny = std::min<long long>(ny, 65535);
  CHK(h->m2_part.ensure((size_t)ny * cnt * sizeof(double)));
  double* part = h->m2_part.as<double>();
  if (h->cx)
    CHK(launch(&fkd::k_dot_block<S, true>, dim3(nblk, (int)ny), dim3(fkd::WG), h->stream, A, B,
               ld, 0LL, K, kslice, M, part));
  else
    CHK(launch(&fkd::k_dot_block<S, false>, dim3(nblk, (int)ny), dim3(fkd::WG), h->stream, A, B,
               ld, 0LL, K, kslice, M, part));
  return sum_parts(h, part, (int)ny, cnt, h->m2_c.as<double>(), !first);
}

template <class TH, class S, bool CX>
int upload_current(fkpm_handle* h, int which, int nnzb, const int* rp, const int* ci,
                   const void* val) {
  const int nb = h->nb, b = h->b;
  std::vector<int> rb(nnzb > 0 ? nnzb : 1);
  for (int i = 0; i < nb; i++)
    for (int p = rp[i]; p < rp[i + 1]; p++) rb[p] = i;
  DevBuf &drp = h->j_rp[which], &dci = h->j_ci[which], &drb = h->j_rb[which];
  DevBuf &draw = h->j_raw[which], &dval = h->j_val[which];
  const size_t cnt = (size_t)nnzb * b * b;
  CHK(drp.ensure(sizeof(int) * (nb + 1)));
  CHK(dci.ensure(sizeof(int) * (nnzb > 0 ? nnzb : 1)));
  CHK(drb.ensure(sizeof(int) * rb.size()));
  CHK(draw.ensure(cnt * sizeof(TH) * (CX ? 2 : 1) + 16));
  CHK(dval.ensure(cnt * sizeof(S) * (CX ? 2 : 1) + 16));
  HIPCHK(hipMemcpyAsync(drp.p, rp, sizeof(int) * (nb + 1), hipMemcpyHostToDevice, h->stream));
  if (nnzb > 0) {
    HIPCHK(hipMemcpyAsync(dci.p, ci, sizeof(int) * nnzb, hipMemcpyHostToDevice, h->stream));
    HIPCHK(hipMemcpyAsync(draw.p, val, cnt * sizeof(TH) * (CX ? 2 : 1), hipMemcpyHostToDevice,
                          h->stream));
  }
  HIPCHK(hipMemcpyAsync(drb.p, rb.data(), sizeof(int) * rb.size(), hipMemcpyHostToDevice,
                        h->stream));
  if (cnt > 0)
    CHK(launch(&fkd::k_scale_H<TH, S, CX>, dim3(grid_for(cnt)), dim3(256), h->stream,
               draw.as<const TH>(), dval.as<S>(), drb.as<const int>(), dci.as<const int>(), nnzb,
               b, 1.0, 0.0));
  HIPCHK(hipStreamSynchronize(h->stream));  // host arrays (rb, caller's) go out of scope
  return 0;
}

template <class S>
int upload_current_s(fkpm_handle* h, int which, int nnzb, const int* rp, const int* ci,
                     const void* val) {
  switch (h->dtype) {
    case FKPM_F32: return upload_current<float, S, false>(h, which, nnzb, rp, ci, val);
    case FKPM_F64: return upload_current<double, S, false>(h, which, nnzb, rp, ci, val);
    case FKPM_C32: return upload_current<float, S, true>(h, which, nnzb, rp, ci, val);
    default: return upload_current<double, S, true>(h, which, nnzb, rp, ci, val);
  }
}

template <class TH, class S, bool CX>
int pack_R_cols(fkpm_handle* h, int k0, int sc, int spc, S* dst) {
  const TH* src = h->rraw.as<const TH>() + (size_t)k0 * h->n * (CX ? 2 : 1);
  const dim3 grid((h->n + 63) / 64, (spc + 15) / 16);
  return launch(&fkd::k_pack_R<TH, S, CX>, grid, dim3(fkd::WG), h->stream, src, dst, h->n, sc, spc);
}

template <class S>
int pack_R_cols_s(fkpm_handle* h, int k0, int sc, int spc, S* dst) {
  switch (h->dtype) {
    case FKPM_F32: return pack_R_cols<float, S, false>(h, k0, sc, spc, dst);
    case FKPM_F64: return pack_R_cols<double, S, false>(h, k0, sc, spc, dst);
    case FKPM_C32: return pack_R_cols<float, S, true>(h, k0, sc, spc, dst);
    default: return pack_R_cols<double, S, true>(h, k0, sc, spc, dst);
  }
}

template <class S>
int moments2_t(fkpm_handle* h, int M, int col_chunk, size_t budget, double* mu) {
  const int HS = h->cx ? 2 : 1;
  const int ne = h->ne();
  const size_t es = sizeof(S);
  // columns per chunk: the requested count (or all), halved until 2M + 3
  // vectors fit the budget
  auto padded = [&](int sc, int* W) {
    const int need = (sc + ne - 1) / ne;
    fkd::GeomChoice gs[64];
    const int ng = fkd::geometries_for_block(h->b, gs, 64);
    int best = 0, widest = 0;
    for (int k = 0; k < ng; k++) {
      const int w = gs[k].L * gs[k].KQ;
      widest = std::max(widest, w);
      if (w >= need && (best == 0 || w < best)) best = w;
    }
    if (best == 0) best = widest;
    *W = best;
    return ((need + best - 1) / best) * best * ne;  // padded columns
  };
  int sc = col_chunk > 0 ? std::min(col_chunk, h->s) : h->s;
  int W = 0, spc = padded(sc, &W);
  auto vec_bytes = [&](int spc_) { return (size_t)h->n * spc_ * HS * es; };
  while (sc > 1 && (size_t)(2 * M + 3) * vec_bytes(spc) > budget) {
    sc = (sc + 1) / 2;
    spc = padded(sc, &W);
  }
  if ((size_t)(2 * M + 3) * vec_bytes(spc) > budget)
    return fail(FKPM_E_ARG, "moments2: M = %d vectors of %zu bytes exceed the %zu-byte budget", M,
                vec_bytes(spc), budget);
  // the engine's own forward-step configuration (tuned or default) when it
  // has this pass width, else the widest lane groups of that width
  fkd::KSet<S> ks;
  KCfg c;
  const KCfg& km = h->kc[K_MOM];
  if (!km.mfma && km.L * km.KQ == W) {
    ks = h->ks<S>(K_MOM);
    c = km;
    if (!h->tuned && h->sweep_force < 0 && !(c.nt & fkd::NT_ORDER)) {
      // every step writes a fresh column of A or B: one front, as past the
      // last-level cache (default_cfg)
      c.sweep = 2;
      derive_grid(h->nb, c);
    }
  } else {
    int L = 0, KQ = 0;
    if (!kset_for_width<S>(h, W, &ks, &L, &KQ))
      return fail(FKPM_E_UNSUP, "moments2: no kernel of width %d for block %d", W, h->b);
    c.L = L;
    c.KQ = KQ;
    c.maxwg = 4096;
    derive_grid(h->nb, c);
  }
  const int qpc = spc / ne;
  const size_t vb = vec_bytes(spc);
  // the columns of A and B are spaced by a vector plus 4352 bytes: with K a
  // power of two a plain spacing would put the same k of every column in the
  // same HBM channel
  const size_t vpad = 4352;
  CHK(h->m2_a.ensure((size_t)M * (vb + vpad)));
  CHK(h->m2_b.ensure((size_t)M * (vb + vpad)));
  CHK(h->m2_ring.ensure(3 * vb));
  CHK(h->m2_c.ensure((size_t)M * M * HS * sizeof(double)));
  const size_t vlen = vb / es;            // scalars per vector
  const size_t vs = (vb + vpad) / es;     // scalars between columns of A, B
  S* A = h->m2_a.as<S>();
  S* Bm = h->m2_b.as<S>();
  S* ring = h->m2_ring.as<S>();
  const int* rp = h->rp.as<const int>();
  const int* ci = h->ci.as<const int>();
  const S* hv = h->hv.as<const S>();
  const dim3 grid(c.nwg), block(fkd::WG);
  auto step = [&](const int* rp_, const int* ci_, const S* hv_, const S* x, const S* z, S* y,
                  double cx, double cz) {
    // the row order and the row length belong to H's pattern
    KCfg rows = c;
    rows.nt &= ~fkd::NT_ORDER;
    return launch(fkd::step_fn(ks, h->nb, chain_bound(h)), grid, block, h->stream, rp_, ci_, hv_, x, z, y,
                  h->nb, qpc, c.chunk, cx, cz, (double*)nullptr, rp_ == rp ? nt_for(h, rows) : rows.nt,
                  no_rsource<S>());
  };
  const int* j1rp = h->j_rp[0].as<const int>();
  const int* j1ci = h->j_ci[0].as<const int>();
  const S* j1v = h->j_val[0].as<const S>();
  const int* j2rp = h->j_rp[1].as<const int>();
  const int* j2ci = h->j_ci[1].as<const int>();
  const S* j2v = h->j_val[1].as<const S>();
  bool first = true;
  for (int k0 = 0; k0 < h->s; k0 += sc) {
    const int scc = std::min(sc, h->s - k0);
    CHK(pack_R_cols_s<S>(h, k0, scc, spc, A));
    // alpha_m = T_m(Hs) r into column m of A
    for (int m = 1; m < M; m++)
      CHK(step(rp, ci, hv, A + (m - 1) * vs, m >= 2 ? A + (m - 2) * vs : nullptr, A + m * vs,
               m == 1 ? 1.0 : 2.0, m == 1 ? 0.0 : -1.0));
    // atild_m = T_m(Hs) j1 r in a ring of three; column m of B = j2 atild_m
    CHK(step(j1rp, j1ci, j1v, A, nullptr, ring, 1.0, 0.0));
    for (int m = 0; m < M; m++) {
      S* t = ring + (m % 3) * vlen;
      if (m >= 1)
        CHK(step(rp, ci, hv, ring + ((m - 1) % 3) * vlen, m >= 2 ? ring + ((m - 2) % 3) * vlen : nullptr,
                 t, m == 1 ? 1.0 : 2.0, m == 1 ? 0.0 : -1.0));
      CHK(step(j2rp, j2ci, j2v, t, nullptr, Bm + m * vs, 1.0, 0.0));
    }
    CHK(dot_block_acc<S>(h, A, Bm, (long long)h->n * spc, (long long)(vs / HS), M, first));
    first = false;
  }
  std::vector<double> cm((size_t)M * M * HS);
  HIPCHK(hipMemcpyAsync(cm.data(), h->m2_c.p, cm.size() * sizeof(double), hipMemcpyDeviceToHost,
                        h->stream));
  HIPCHK(hipStreamSynchronize(h->stream));
  for (size_t x = 0; x < (size_t)M * M; x++) {
    mu[2 * x] = cm[x * HS];
    mu[2 * x + 1] = HS == 2 ? cm[x * HS + 1] : 0.0;
  }
  return 0;  // the buffers of moments / autodiff_matrix are untouched
}

// H values up to this size go through pinned staging, so that set_H returns
// without waiting for the device.
constexpr size_t kStageBytes = 512 << 10;

template <class TH, class S, bool CX>
int upload_H_t(fkpm_handle* h, DevBuf& dst, const void* val, double mag, double shift) {
  const size_t cnt = (size_t)h->nnzb * h->b * h->b, bytes = cnt * sizeof(TH) * (CX ? 2 : 1);
  if (bytes <= kStageBytes) {
    if (h->stage_busy) HIPCHK(hipStreamSynchronize(h->stream));
    CHK(h->stage.ensure(kStageBytes));
    memcpy(h->stage.p, val, bytes);
    val = h->stage.p;
    h->stage_busy = true;
  } else {
    h->stage_busy = false;  // set_H waits for the stream
  }
  HIPCHK(hipMemcpyAsync(h->hraw.p, val, bytes, hipMemcpyHostToDevice, h->stream));
  return launch(&fkd::k_scale_H<TH, S, CX>, dim3(grid_for(cnt)), dim3(256), h->stream,
                h->hraw.as<const TH>(), dst.as<S>(), h->rowblk.as<const int>(),
                h->ci.as<const int>(), h->nnzb, h->b, mag, shift);
}

template <class S>
int upload_H_s(fkpm_handle* h, DevBuf& dst, const void* val, double mag, double shift) {
  switch (h->dtype) {
    case FKPM_F32: return upload_H_t<float, S, false>(h, dst, val, mag, shift);
    case FKPM_F64: return upload_H_t<double, S, false>(h, dst, val, mag, shift);
    case FKPM_C32: return upload_H_t<float, S, true>(h, dst, val, mag, shift);
    default: return upload_H_t<double, S, true>(h, dst, val, mag, shift);
  }
}

// Pattern upload shared by set_H and energy_scale.
// A periodic 3-D lattice in natural order (block row x + n1 (y + n2 z)),
// recognised from H's block offsets: the three distances |j - i| (mod nb, the
// shorter way round) that at least half the rows have are 1 < n1 < n1 n2 with
// n1 n2 n3 = nb and every side at least 8.  Fills n[3]; false otherwise.
bool lattice_dims(int nb, const int* rp, const int* ci, int n[3]) {
  if (nb < 512) return false;
  std::vector<int> cnt(nb / 2 + 1, 0);  // blocks at each distance
  for (int i = 0; i < nb; i++)
    for (int p = rp[i]; p < rp[i + 1]; p++) {
      int d = ci[p] - i;
      if (d == 0) continue;
      if (d < 0) d += nb;
      cnt[std::min(d, nb - d)]++;
    }
  std::vector<int> dist;
  for (int d = 1; d <= nb / 2; d++)
    if (2ll * cnt[d] >= nb) dist.push_back(d);
  if (dist.size() != 3 || dist[0] != 1) return false;
  const long long n1 = dist[1], c = dist[2];
  if (c % n1 != 0 || nb % c != 0) return false;
  n[0] = (int)n1;
  n[1] = (int)(c / n1);
  n[2] = (int)(nb / c);
  return n[0] >= 8 && n[1] >= 8 && n[2] >= 8;
}

// Sweep order for an n1 x n2 x n3 lattice: one x-slab per XCD (x in
// [floor(k n1 / 8), floor((k+1) n1 / 8)) for XCD k: widths n1/8 rounded down
// or up, about one eighth of the sweep each, the same split into eighths that
// the per-XCD row ranges of the sweep make), each walked in y-tiles of ty rows
// (about 128 sites a plane of the tile) and, inside a tile, plane by plane
// along z.  A row's +-z neighbours are then one tile-plane away in the sweep
// instead of a whole slab-plane (on 64^3: 128 instead of 512 sites), so the
// neighbour rows of both vectors an autodiff step gathers stay in the XCD's
// L2.
bool lattice_order(int nb, const int* rp, const int* ci, std::vector<int>& order) {
  int n[3];
  if (!lattice_dims(nb, rp, ci, n)) return false;
  const int wmax = (n[0] + 7) / 8;
  int ty = 1;
  for (int t = 1; t <= n[1]; t++)
    if (n[1] % t == 0 && wmax * t <= 128) ty = t;
  order.clear();
  order.reserve(nb);
  for (int k = 0; k < 8; k++) {
    const int x0 = (int)((long long)k * n[0] / 8), x1 = (int)((long long)(k + 1) * n[0] / 8);
    for (int y0 = 0; y0 < n[1]; y0 += ty)
      for (int z = 0; z < n[2]; z++)
        for (int yo = 0; yo < ty; yo++)
          for (int x = x0; x < x1; x++) order.push_back(x + n[0] * ((y0 + yo) + n[1] * z));
  }
  return (int)order.size() == nb;
}

int upload_pattern(fkpm_handle* h, int nb, int b, int nnzb, const int* row_ptr,
                   const int* col_idx) {
  h->pattern_set = false;
  h->nb = nb;
  h->b = b;
  h->nnzb = nnzb;
  h->h_rp.assign(row_ptr, row_ptr + nb + 1);
  h->max_deg = 0;
  for (int i = 0; i < nb; i++) h->max_deg = std::max(h->max_deg, row_ptr[i + 1] - row_ptr[i]);
  h->h_ci.assign(col_idx, col_idx + nnzb);
  std::vector<int> rowblk(nnzb > 0 ? nnzb : 1);
  for (int i = 0; i < nb; i++)
    for (int p = row_ptr[i]; p < row_ptr[i + 1]; p++) rowblk[p] = i;
  CHK(h->rp.ensure(sizeof(int) * (nb + 1)));
  CHK(h->ci.ensure(sizeof(int) * (nnzb > 0 ? nnzb : 1)));
  CHK(h->rowblk.ensure(sizeof(int) * rowblk.size()));
  HIPCHK(hipMemcpyAsync(h->rp.p, row_ptr, sizeof(int) * (nb + 1), hipMemcpyHostToDevice, h->stream));
  if (nnzb > 0)
    HIPCHK(hipMemcpyAsync(h->ci.p, col_idx, sizeof(int) * nnzb, hipMemcpyHostToDevice, h->stream));
  HIPCHK(hipMemcpyAsync(h->rowblk.p, rowblk.data(), sizeof(int) * rowblk.size(),
                        hipMemcpyHostToDevice, h->stream));
  const size_t hvb = (size_t)nnzb * b * b * host_elem_bytes(h->dtype);
  CHK(h->hraw.ensure(hvb > 0 ? hvb : 16));
  std::vector<int> order, desc;
  h->has_order = lattice_order(nb, row_ptr, col_idx, order);
  if (h->has_order) {
    desc.resize(3 * (size_t)nb);
    for (int k = 0; k < nb; k++) {
      desc[3 * (size_t)k] = order[k];
      desc[3 * (size_t)k + 1] = row_ptr[order[k]];
      desc[3 * (size_t)k + 2] = row_ptr[order[k] + 1];
    }
    CHK(h->rdesc.ensure(sizeof(int) * desc.size()));
    HIPCHK(hipMemcpyAsync(h->rdesc.p, desc.data(), sizeof(int) * desc.size(),
                          hipMemcpyHostToDevice, h->stream));
  }
  apply_row_order(h);
  // the async copies above read host arrays owned by the caller (and desc):
  // finish them
  HIPCHK(hipStreamSynchronize(h->stream));
  h->pattern_set = true;
  return 0;
}

// Symmetric tridiagonal extreme eigenvalues by Sturm-sequence bisection
// (replaces arma::eig_sym on the Lanczos matrix, engine_cusparse.cpp:655-666).
int sturm_below(const std::vector<double>& a, const std::vector<double>& b2, double x) {
  int cnt = 0;
  double q = a[0] - x;
  if (q < 0) cnt++;
  for (size_t j = 1; j < a.size(); j++) {
    if (q == 0) q = 1e-300;
    q = a[j] - x - b2[j] / q;
    if (q < 0) cnt++;
  }
  return cnt;
}

void tridiag_extremes(const std::vector<double>& a, const std::vector<double>& beta,
                      double* emin, double* emax) {
  const size_t n = a.size();
  std::vector<double> b2(n, 0.0);
  double lo = a[0], hi = a[0];
  for (size_t j = 1; j < n; j++) b2[j] = beta[j] * beta[j];
  for (size_t j = 0; j < n; j++) {
    const double r = (j > 0 ? std::fabs(beta[j]) : 0.0) + (j + 1 < n ? std::fabs(beta[j + 1]) : 0.0);
    lo = std::min(lo, a[j] - r);
    hi = std::max(hi, a[j] + r);
  }
  const double pad = 1e-12 * (std::fabs(lo) + std::fabs(hi) + 1.0);
  auto kth = [&](int k) {
    double l = lo - pad, u = hi + pad;
    for (int it = 0; it < 200; it++) {
      const double mid = 0.5 * (l + u);
      if (mid == l || mid == u) break;
      if (sturm_below(a, b2, mid) > k) u = mid; else l = mid;
    }
    return 0.5 * (l + u);
  };
  *emin = kth(0);
  *emax = kth((int)n - 1);
}

// Lanczos on the device in FP64 (engine_cusparse.cpp:598-673).  Uses its own
// buffers, so the engine's H is untouched.  A diagonal block missing from H is
// inserted as an explicit zero block: the fused SpMM kernel takes the own-row
// operand of the dot from the diagonal block.
template <class TH, bool CX>
int lanczos_t(fkpm_handle* h, int nb, int b, int nnzb, const int* row_ptr, const int* col_idx,
              const void* val, double extend, int iters, const void* v_start, double* lo,
              double* hi) {
  fkd::KSet<double> ks;
  const int geoL = 4, geoKQ = 1;
  const bool ok = CX ? fkd::find_kset_dc(b, geoL, geoKQ, &ks) : fkd::find_kset_dr(b, geoL, geoKQ, &ks);
  if (!ok) return fail(FKPM_E_UNSUP, "no Lanczos kernel for block %d", b);
  const int HS = CX ? 2 : 1;
  const int bb = b * b;
  // pattern with every diagonal block present; when H has them all (the
  // usual case) its arrays are uploaded as they are
  int missing = 0;
  for (int i = 0; i < nb; i++) {
    bool diag = false;
    for (int p = row_ptr[i]; p < row_ptr[i + 1] && !diag; p++) diag = (col_idx[p] == i);
    missing += diag ? 0 : 1;
  }
  const bool direct = missing == 0 && std::is_same<TH, double>::value;
  std::vector<int> rp2, ci2;
  std::vector<double> hv2;
  if (!direct) {
    rp2.assign(nb + 1, 0);
    ci2.reserve((size_t)nnzb + missing);
    hv2.reserve(((size_t)nnzb + missing) * bb * HS);
    for (int i = 0; i < nb; i++) {
      bool diag = false;
      for (int p = row_ptr[i]; p < row_ptr[i + 1]; p++) diag |= (col_idx[p] == i);
      for (int p = row_ptr[i]; p < row_ptr[i + 1]; p++) {
        ci2.push_back(col_idx[p]);
        const TH* v = static_cast<const TH*>(val) + (size_t)p * bb * HS;
        for (int e = 0; e < bb * HS; e++) hv2.push_back((double)v[e]);
      }
      if (!diag) {
        ci2.push_back(i);
        for (int e = 0; e < bb * HS; e++) hv2.push_back(0.0);
      }
      rp2[i + 1] = (int)ci2.size();
    }
  }
  const int* up_rp = direct ? row_ptr : rp2.data();
  const int* up_ci = direct ? col_idx : ci2.data();
  const double* up_hv = direct ? static_cast<const double*>(val) : hv2.data();
  const int nnz2 = direct ? nnzb : (int)ci2.size();
  const int n = nb * b;
  const int qp = geoL * geoKQ;  // one probe column padded to one lane-group pass
  const int sp = qp * (2 / HS);
  const size_t len = (size_t)n * sp * HS;  // doubles per vector
  const int gwg = (fkd::WG / fkd::WAVE) * (fkd::WAVE / geoL);
  int nwg = std::min((nb + gwg - 1) / gwg, 1024);
  int chunk = (nb + nwg - 1) / nwg;
  chunk = ((chunk + gwg - 1) / gwg) * gwg;
  nwg = (nb + chunk - 1) / chunk;

  struct Bufs {
    DevBuf rp, ci, hv, v0, v1, w, part, ps, coef, used;
    ~Bufs() {
      DevBuf* all[] = {&rp, &ci, &hv, &v0, &v1, &w, &part, &ps, &coef, &used};
      for (DevBuf* d : all) d->release();
    }
  } B;
  const size_t hv_count = (size_t)nnz2 * bb * HS;
  CHK(B.rp.ensure(sizeof(int) * (nb + 1)));
  CHK(B.ci.ensure(sizeof(int) * std::max(nnz2, 1)));
  CHK(B.hv.ensure(sizeof(double) * std::max<size_t>(hv_count, 1)));
  CHK(B.v0.ensure(len * sizeof(double)));
  CHK(B.v1.ensure(len * sizeof(double)));
  CHK(B.w.ensure(len * sizeof(double)));
  CHK(B.part.ensure((size_t)nwg * 2 * sizeof(double)));
  CHK(B.ps.ensure(2 * sizeof(double)));
  HIPCHK(hipMemcpyAsync(B.rp.p, up_rp, sizeof(int) * (nb + 1), hipMemcpyHostToDevice, h->stream));
  if (nnz2 > 0) {
    HIPCHK(hipMemcpyAsync(B.ci.p, up_ci, sizeof(int) * nnz2, hipMemcpyHostToDevice, h->stream));
    HIPCHK(hipMemcpyAsync(B.hv.p, up_hv, sizeof(double) * hv_count, hipMemcpyHostToDevice,
                          h->stream));
  }
  CHK(zero_doubles(h, B.v0.p, len));
  CHK(zero_doubles(h, B.w.p, len));
  {
    std::vector<double> packed(len, 0.0);
    double nrm = 0.0;
    for (int r = 0; r < n; r++)
      for (int c = 0; c < HS; c++) {
        const double x = (double)static_cast<const TH*>(v_start)[(size_t)r * HS + c];
        nrm += x * x;
      }
    nrm = std::sqrt(nrm);
    if (!(nrm > 0) || !std::isfinite(nrm)) return fail(FKPM_E_ARG, "energy_scale: bad start vector");
    for (int r = 0; r < n; r++)
      for (int c = 0; c < HS; c++)
        packed[(size_t)r * sp * HS + c] = (double)static_cast<const TH*>(v_start)[(size_t)r * HS + c] / nrm;
    HIPCHK(hipMemcpyAsync(B.v1.p, packed.data(), len * sizeof(double), hipMemcpyHostToDevice, h->stream));
    HIPCHK(hipStreamSynchronize(h->stream));  // host staging vectors go out of scope
  }
  // the iteration runs on the stream without a host round trip: alpha, beta
  // and the invariant-subspace cut stay on the device until the end
  const dim3 grid(nwg), block(fkd::WG);
  CHK(B.coef.ensure(2 * (size_t)iters * sizeof(double)));
  CHK(B.used.ensure(sizeof(int)));
  double* coef = static_cast<double*>(B.coef.p);
  int* dused = static_cast<int*>(B.used.p);
  const double* dps = static_cast<const double*>(B.ps.p);
  auto spmv_dot = [&]() -> int {
    // w = H v1; ps = (|v1|^2, Re <w, v1>)
    CHK(launch(ks.mom, grid, block, h->stream, (const int*)B.rp.p, (const int*)B.ci.p,
               (const double*)B.hv.p, (const double*)B.v1.p, (const double*)nullptr,
               (double*)B.w.p, nb, qp, chunk, 1.0, 0.0, (double*)B.part.p, 0, no_rsource<double>()));
    return launch(&fkd::k_reduce_partials, dim3(1), block, h->stream, (const double*)B.part.p,
                  nwg, (double*)B.ps.p);
  };
  CHK(launch(&fkd::k_lanczos_edge, dim3(1), dim3(64), h->stream, dps, coef, iters, dused, 0));
  for (int j = 1; j < iters; j++) {
    CHK(spmv_dot());
    CHK(launch(&fkd::k_lanczos_orth, dim3(nwg), block, h->stream, (double*)B.w.p,
               (const double*)B.v1.p, (const double*)B.v0.p, len, dps, coef, iters, j,
               (double*)B.part.p));
    CHK(launch(&fkd::k_reduce_partials, dim3(1), block, h->stream, (const double*)B.part.p, nwg,
               (double*)B.ps.p));
    CHK(launch(&fkd::k_lanczos_next, dim3(grid_for(len)), dim3(256), h->stream, (double*)B.v0.p,
               (double*)B.v1.p, (const double*)B.w.p, len, dps, coef, iters, j, dused));
  }
  CHK(spmv_dot());
  CHK(launch(&fkd::k_lanczos_edge, dim3(1), dim3(64), h->stream, dps, coef, iters, dused, 1));
  std::vector<double> cf(2 * (size_t)iters);
  int used = iters;
  HIPCHK(hipMemcpyAsync(cf.data(), coef, cf.size() * sizeof(double), hipMemcpyDeviceToHost,
                        h->stream));
  HIPCHK(hipMemcpyAsync(&used, dused, sizeof(int), hipMemcpyDeviceToHost, h->stream));
  HIPCHK(hipStreamSynchronize(h->stream));
  std::vector<double> alpha(cf.begin(), cf.begin() + used), beta(cf.begin() + iters,
                                                                 cf.begin() + iters + used);
  double emin = 0, emax = 0;
  tridiag_extremes(alpha, beta, &emin, &emax);
  const double slack = extend * (emax - emin);
  *lo = emin - slack;
  *hi = emax + slack;
  return 0;
}


}  // namespace

// ===========================================================================
// C-ABI
// ===========================================================================
extern "C" {

const char* fkpm_last_error(void) { return g_last_error.c_str(); }

int fkpm_device_count(void) {
  int c = 0;
  if (hipGetDeviceCount(&c) != hipSuccess) return 0;
  return c;
}

int fkpm_dev_open(int device, int dtype, int prec, fkpm_handle** out) {
  if (!out) return fail(FKPM_E_ARG, "null handle pointer");
  *out = nullptr;
  if (dtype < FKPM_F32 || dtype > FKPM_C64) return fail(FKPM_E_ARG, "bad dtype %d", dtype);
  if (prec != FKPM_PREC_FP64 && prec != FKPM_PREC_FP32) return fail(FKPM_E_ARG, "bad prec %d", prec);
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess || count == 0)
    return fail(FKPM_E_NODEV, "no HIP device is available");
  if (device < 0 || device >= count)
    return fail(FKPM_E_NODEV, "invalid device #%d (%d available)", device, count);
  HIPCHK(hipSetDevice(device));
  fkpm_handle* h = new fkpm_handle();
  h->device = device;
  h->dtype = dtype;
  h->prec = prec;
  h->cx = dtype_complex(dtype);
  h->single = (prec == FKPM_PREC_FP32);
  // FKPM_AUTOTUNE=1: tune at the first use of a shape (FKPM_OPT_AUTOTUNE for
  // callers that cannot reach fkpm_set_option, such as the C++ API)
  if (const char* e = getenv("FKPM_AUTOTUNE")) h->autotune_on_use = e[0] != '\0' && e[0] != '0';
  // FKPM_GRAPH=0/1/-1: the FKPM_OPT_GRAPH default for handles opened afterwards
  if (const char* e = getenv("FKPM_GRAPH")) {
    const int v = atoi(e);
    if (v >= -1 && v <= 1) h->graph_mode = v;
  }
  if (hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&h->ev0) != hipSuccess || hipEventCreate(&h->ev1) != hipSuccess) {
    delete h;
    return fail(FKPM_E_HIP, "stream/event creation failed");
  }
  *out = h;
  return 0;
}

int fkpm_dev_close(fkpm_handle* h) {
  if (!h) return 0;
  delete h;
  return 0;
}

void* fkpm_stream(fkpm_handle* h) { return h ? (void*)h->stream : nullptr; }

int fkpm_synchronize(fkpm_handle* h) {
  if (!h) return fail(FKPM_E_ARG, "null handle");
  HIPCHK(hipSetDevice(h->device));
  HIPCHK(hipStreamSynchronize(h->stream));
  return 0;
}

int fkpm_set_H(fkpm_handle* h, int nb, int b, int nnzb, const int* row_ptr, const int* col_idx,
               const void* val, double avg, double mag) {
  if (!h) return fail(FKPM_E_ARG, "null handle");
  HIPCHK(hipSetDevice(h->device));
  if (b <= 0) return fail(FKPM_E_ARG, "bad block size %d", b);
  if (!fkd::block_supported(b)) return fail(FKPM_E_UNSUP, "block size %d has no kernels", b);
  if (!(mag > 0) || !std::isfinite(avg)) return fail(FKPM_E_ARG, "bad energy scale avg=%g mag=%g", avg, mag);
  if (nnzb > 0 && !val) return fail(FKPM_E_ARG, "null H values");
  // The pattern the handle already holds (compared by content, as in a loop
  // over Hamiltonians on one lattice) has been checked and is on the device.
  const bool same = h->pattern_set && nb == h->nb && b == h->b && nnzb == h->nnzb && row_ptr &&
                    (nnzb == 0 || col_idx) &&
                    memcmp(row_ptr, h->h_rp.data(), sizeof(int) * ((size_t)nb + 1)) == 0 &&
                    (nnzb == 0 || memcmp(col_idx, h->h_ci.data(), sizeof(int) * (size_t)nnzb) == 0);
  if (!same) {
    CHK(check_pattern("set_H", nb, nnzb, row_ptr, nullptr, col_idx));
    for (int i = 0; i < nb; i++) {  // engine_cusparse.cpp:716-727: every diagonal block present
      bool found = false;
      for (int p = row_ptr[i]; p < row_ptr[i + 1]; p++) found |= (col_idx[p] == i);
      if (!found) return fail(FKPM_E_ARG, "set_H: diagonal block (%d,%d) is missing", i, i);
    }
  }
  // The kernel choice depends on the block size, the block-row and block
  // counts (grids, tuned-shape key) and on whether every row has at most
  // kRowResidentMax blocks (row-resident matrix-core kernels read only that many),
  // or at most 7 (their instantiation without a padding slot), and on a row much
  // longer than the others: a change of any of them picks the kernels again at the
  // next use.
  const int old_b = h->b, old_nb = h->nb, old_nnzb = h->nnzb, old_deg = h->max_deg;
  if (!same) CHK(upload_pattern(h, nb, b, nnzb, row_ptr, col_idx));
  const bool geo_change = b != old_b || nb != old_nb || nnzb != old_nnzb ||
                          (old_deg <= kRowResidentMax) != (h->max_deg <= kRowResidentMax) ||
                          (old_deg <= 7) != (h->max_deg <= 7) ||
                          (old_deg != h->max_deg && (long_rows(nb, nnzb, old_deg) ||
                                                     long_rows(nb, nnzb, h->max_deg)));
  h->avg = avg;
  h->mag = mag;
  const size_t eb = h->single ? 4 : 8;
  CHK(h->hv.ensure((size_t)(nnzb > 0 ? nnzb : 1) * b * b * (h->cx ? 2 : 1) * eb));
  if (h->single)
    CHK(upload_H_s<float>(h, h->hv, val, mag, avg / mag));
  else
    CHK(upload_H_s<double>(h, h->hv, val, mag, avg / mag));
  if (!h->stage_busy) HIPCHK(hipStreamSynchronize(h->stream));  // the copy reads val itself
  h->h_set = true;
  h->alpha_M = 0;
  h->tab_K = 0;
  h->res.K = 0;
  h->res.packed = false;
  if (geo_change) h->r_dirty = true;
  return 0;
}

int fkpm_set_R(fkpm_handle* h, int n, int s, const void* R_colmajor) {
  if (!h) return fail(FKPM_E_ARG, "null handle");
  HIPCHK(hipSetDevice(h->device));
  if (n <= 0 || s <= 0 || !R_colmajor)  // engine_cusparse.cpp:678-681
    return fail(FKPM_E_ARG, "cannot handle an empty R matrix (n=%d, s=%d)", n, s);
  const size_t bytes = (size_t)n * s * host_elem_bytes(h->dtype);
  CHK(h->rraw.ensure(bytes));
  HIPCHK(hipMemcpyAsync(h->rraw.p, R_colmajor, bytes, hipMemcpyHostToDevice, h->stream));
  HIPCHK(hipStreamSynchronize(h->stream));
  h->n = n;
  h->s = s;
  h->r_set = true;
  h->r_dirty = true;
  h->alpha_M = 0;
  h->tab_K = 0;
  h->res.K = 0;
  return 0;
}

int fkpm_moments(fkpm_handle* h, int M, double* mu) {
  if (!h || !mu) return fail(FKPM_E_ARG, "null argument");
  HIPCHK(hipSetDevice(h->device));
  if (M < 2 || M % 2 != 0) return fail(FKPM_E_ARG, "moments: M=%d must be even and >= 2", M);
  CHK(ensure_ready(h));
  h->alpha_M = 0;
  if (h->single) return moments_t<float>(h, M, mu);
  return moments_t<double>(h, M, mu);
}

int fkpm_set_D_pattern(fkpm_handle* h, int nbD, int nnzbD, const int* row_ptr, const int* row_idx,
                       const int* col_idx) {
  if (!h) return fail(FKPM_E_ARG, "null handle");
  HIPCHK(hipSetDevice(h->device));
  CHK(check_pattern("D pattern", nbD, nnzbD, row_ptr, row_idx, col_idx));
  // block (i,j) -> index of block (j,i), or -1
  std::vector<int> tpos(nnzbD > 0 ? nnzbD : 1, -1);
  bool sym = true;
  for (int i = 0; i < nbD; i++)
    for (int p = row_ptr[i]; p < row_ptr[i + 1]; p++) {
      const int j = col_idx[p];
      int t = -1;
      for (int q = row_ptr[j]; q < row_ptr[j + 1]; q++)
        if (col_idx[q] == i) {
          t = q;
          break;
        }
      tpos[p] = t;
      if (t < 0 && i >= j) sym = false;  // the reference aborts only for these
    }
  CHK(h->drp.ensure(sizeof(int) * (nbD + 1)));
  CHK(h->dci.ensure(sizeof(int) * (nnzbD > 0 ? nnzbD : 1)));
  CHK(h->tpos.ensure(sizeof(int) * tpos.size()));
  HIPCHK(hipMemcpyAsync(h->drp.p, row_ptr, sizeof(int) * (nbD + 1), hipMemcpyHostToDevice, h->stream));
  if (nnzbD > 0)
    HIPCHK(hipMemcpyAsync(h->dci.p, col_idx, sizeof(int) * nnzbD, hipMemcpyHostToDevice, h->stream));
  HIPCHK(hipMemcpyAsync(h->tpos.p, tpos.data(), sizeof(int) * tpos.size(), hipMemcpyHostToDevice,
                        h->stream));
  HIPCHK(hipStreamSynchronize(h->stream));
  h->nbD = nbD;
  h->nnzbD = nnzbD;
  h->hd_rp.assign(row_ptr, row_ptr + nbD + 1);
  h->hd_ci.assign(col_idx, col_idx + nnzbD);
  h->d_set = true;
  h->d_sym = sym;
  h->d_valid = false;
  return 0;
}

int fkpm_stoch_matrix(fkpm_handle* h, int M, const double* c, void* D_val) {
  if (!h || !c) return fail(FKPM_E_ARG, "null argument");
  HIPCHK(hipSetDevice(h->device));
  if (M < 2) return fail(FKPM_E_ARG, "stoch_matrix: need at least 2 coefficients (M=%d)", M);
  CHK(ensure_ready(h));
  CHK(check_D_ready(h));
  h->d_valid = false;
  if (h->single)
    CHK(stoch_t<float>(h, M, c));
  else
    CHK(stoch_t<double>(h, M, c));
  h->d_valid = true;
  if (D_val) return copy_D_out(h, D_val);
  HIPCHK(hipStreamSynchronize(h->stream));
  return 0;
}

int fkpm_autodiff_matrix(fkpm_handle* h, int M, const double* c, void* D_val) {
  if (!h || !c) return fail(FKPM_E_ARG, "null argument");
  HIPCHK(hipSetDevice(h->device));
  if (M < 2 || M % 2 != 0) return fail(FKPM_E_ARG, "autodiff_matrix: M=%d must be even and >= 2", M);
  if (h->alpha_M != M)
    return fail(FKPM_E_STATE,
                "autodiff_matrix requires moments(M) with the same M (%d) immediately before "
                "(held: %d)", M, h->alpha_M);
  CHK(check_D_ready(h));
  if (!h->d_sym)
    return fail(FKPM_E_ARG, "autodiff_matrix: a block (i,j) with i >= j of D has no (j,i) partner");
  h->d_valid = false;
  if (h->single)
    CHK(autodiff_t<float>(h, M, c));
  else
    CHK(autodiff_t<double>(h, M, c));
  h->d_valid = true;
  if (D_val) return copy_D_out(h, D_val);
  HIPCHK(hipStreamSynchronize(h->stream));
  return 0;
}

int fkpm_moments2(fkpm_handle* h, int M, int nnzb1, const int* rp1, const int* ci1,
                  const void* v1, int nnzb2, const int* rp2, const int* ci2, const void* v2,
                  int col_chunk, double* mu) {
  if (!h || !mu || !rp1 || !ci1 || !v1 || !rp2 || !ci2 || !v2)
    return fail(FKPM_E_ARG, "moments2: null argument");
  if (M < 2 || M % 2 != 0) return fail(FKPM_E_ARG, "moments2: M = %d must be even and >= 2", M);
  HIPCHK(hipSetDevice(h->device));
  CHK(ensure_ready(h));
  CHK(check_pattern("j1", h->nb, nnzb1, rp1, nullptr, ci1));
  CHK(check_pattern("j2", h->nb, nnzb2, rp2, nullptr, ci2));
  if (h->single) {
    CHK(upload_current_s<float>(h, 0, nnzb1, rp1, ci1, v1));
    CHK(upload_current_s<float>(h, 1, nnzb2, rp2, ci2, v2));
  } else {
    CHK(upload_current_s<double>(h, 0, nnzb1, rp1, ci1, v1));
    CHK(upload_current_s<double>(h, 1, nnzb2, rp2, ci2, v2));
  }
  // vector budget: half the free device memory, at most 64 GiB, unless the
  // environment names one
  size_t free_b = 0, total_b = 0;
  HIPCHK(hipMemGetInfo(&free_b, &total_b));
  size_t budget = std::min((size_t)64 << 30, free_b / 2);
  if (const char* e = getenv("FKPM_MOMENTS2_BYTES")) budget = (size_t)strtoull(e, nullptr, 10);
  return h->single ? moments2_t<float>(h, M, col_chunk, budget, mu)
                   : moments2_t<double>(h, M, col_chunk, budget, mu);
}

int fkpm_get_D(fkpm_handle* h, void* D_val) {
  if (!h || !D_val) return fail(FKPM_E_ARG, "null argument");
  HIPCHK(hipSetDevice(h->device));
  if (!h->d_valid) return fail(FKPM_E_STATE, "no D has been computed");
  return copy_D_out(h, D_val);
}

int fkpm_energy_scale(fkpm_handle* h, int nb, int b, int nnzb, const int* row_ptr,
                      const int* col_idx, const void* val, double extend, int iters,
                      const void* v_start, double* lo, double* hi) {
  if (!h || !v_start || !lo || !hi) return fail(FKPM_E_ARG, "null argument");
  HIPCHK(hipSetDevice(h->device));
  if (b <= 0 || !fkd::block_supported(b)) return fail(FKPM_E_UNSUP, "block size %d has no kernels", b);
  if (iters < 1) return fail(FKPM_E_ARG, "energy_scale: iters=%d", iters);
  if (nnzb > 0 && !val) return fail(FKPM_E_ARG, "null H values");
  CHK(check_pattern("energy_scale", nb, nnzb, row_ptr, nullptr, col_idx));
  switch (h->dtype) {
    case FKPM_F32: return lanczos_t<float, false>(h, nb, b, nnzb, row_ptr, col_idx, val, extend, iters, v_start, lo, hi);
    case FKPM_F64: return lanczos_t<double, false>(h, nb, b, nnzb, row_ptr, col_idx, val, extend, iters, v_start, lo, hi);
    case FKPM_C32: return lanczos_t<float, true>(h, nb, b, nnzb, row_ptr, col_idx, val, extend, iters, v_start, lo, hi);
    default: return lanczos_t<double, true>(h, nb, b, nnzb, row_ptr, col_idx, val, extend, iters, v_start, lo, hi);
  }
}

int fkpm_set_timing(fkpm_handle* h, int on) {
  if (!h) return fail(FKPM_E_ARG, "null handle");
  h->timing = on != 0;
  return 0;
}

int fkpm_get_timing(fkpm_handle* h, double* ms_moments, int* n_moments, double* ms_stoch,
                    int* n_stoch, double* ms_autodiff, int* n_autodiff) {
  if (!h) return fail(FKPM_E_ARG, "null handle");
  if (ms_moments) *ms_moments = h->ms_mom;
  if (n_moments) *n_moments = h->n_mom;
  if (ms_stoch) *ms_stoch = h->ms_stoch;
  if (n_stoch) *n_stoch = h->n_stoch;
  if (ms_autodiff) *ms_autodiff = h->ms_ad;
  if (n_autodiff) *n_autodiff = h->n_ad;
  return 0;
}

int fkpm_get_config(fkpm_handle* h, int* lanes, int* kq, int* s_padded, int* n_wg,
                    int* fused_autodiff) {
  if (!h) return fail(FKPM_E_ARG, "null handle");
  if (lanes) *lanes = h->kc[K_MOM].L;
  if (kq) *kq = h->kc[K_MOM].KQ;
  if (s_padded) *s_padded = h->sp;
  if (n_wg) *n_wg = h->kc[K_MOM].nwg;
  if (fused_autodiff) *fused_autodiff = h->d_fused ? 1 : 0;
  return 0;
}

int fkpm_get_kernel_config(fkpm_handle* h, int kind, int* lanes, int* kq, int* n_wg, int* nt) {
  if (!h) return fail(FKPM_E_ARG, "null handle");
  if (kind < 0 || kind >= NKIND) return fail(FKPM_E_ARG, "bad kernel kind %d", kind);
  const KCfg& c = h->kc[kind];
  if (lanes) *lanes = c.L;
  if (kq) *kq = c.KQ;
  if (n_wg) *n_wg = c.nwg;
  if (nt) *nt = c.nt;
  return 0;
}

int fkpm_get_kernel_mfma(fkpm_handle* h, int kind, int* mfma) {
  if (!h || !mfma) return fail(FKPM_E_ARG, "null argument");
  if (kind < 0 || kind >= NKIND) return fail(FKPM_E_ARG, "bad kernel kind %d", kind);
  *mfma = h->kc[kind].mfma;
  return 0;
}

int fkpm_get_alpha_table(fkpm_handle* h, int* stored) {
  if (!h || !stored) return fail(FKPM_E_ARG, "null argument");
  *stored = (h->a_slots > 0 && h->alpha_M > 0) ? 1 : 0;
  return 0;
}

int fkpm_get_whole_recursion(fkpm_handle* h, int* on) {
  if (!h || !on) return fail(FKPM_E_ARG, "null argument");
  *on = h->res.state ? 1 : 0;
  return 0;
}

int fkpm_get_stoch_method(fkpm_handle* h, int* method) {
  if (!h || !method) return fail(FKPM_E_ARG, "null argument");
  *method = h->stoch_used;
  return 0;
}

int fkpm_get_kernel_sweep(fkpm_handle* h, int kind, int* sweep) {
  if (!h || !sweep) return fail(FKPM_E_ARG, "null argument");
  if (kind < 0 || kind >= NKIND) return fail(FKPM_E_ARG, "bad kernel kind %d", kind);
  *sweep = h->kc[kind].sweep;
  return 0;
}

int fkpm_lattice_order(int nb, int nnzb, const int* row_ptr, const int* col_idx, int* order,
                       int* dims) {
  if (nb <= 0 || nnzb < 0 || !row_ptr || (nnzb > 0 && !col_idx) || !order || !dims)
    return fail(FKPM_E_ARG, "lattice_order: bad arguments");
  CHK(check_pattern("lattice_order", nb, nnzb, row_ptr, nullptr, col_idx));
  std::vector<int> ord;
  if (!lattice_order(nb, row_ptr, col_idx, ord)) return 0;
  int n[3];
  lattice_dims(nb, row_ptr, col_idx, n);
  std::copy(ord.begin(), ord.end(), order);
  std::copy(n, n + 3, dims);
  return 1;
}

int fkpm_get_graph_stats(fkpm_handle* h, long long* launches, long long* captures) {
  if (!h) return fail(FKPM_E_ARG, "null handle");
  if (launches) *launches = h->n_graph_launches;
  if (captures) *captures = h->n_graph_captures;
  return 0;
}

int fkpm_get_state(fkpm_handle* h, int* r_compact, int* tuned, int* moments_M) {
  if (!h) return fail(FKPM_E_ARG, "null handle");
  if (r_compact) *r_compact = h->r_compact ? 1 : 0;
  if (tuned) *tuned = h->tuned ? 1 : 0;
  if (moments_M) *moments_M = h->alpha_M;
  return 0;
}

int fkpm_set_geometry(fkpm_handle* h, int lanes, int kq, int max_wg) {
  if (!h) return fail(FKPM_E_ARG, "null handle");
  if (lanes < 0 || kq < 0 || max_wg < 0) return fail(FKPM_E_ARG, "bad geometry");
  if (lanes != 0 && h->b > 0 && !compiled(h->b, lanes, kq > 0 ? kq : 1))
    return fail(FKPM_E_UNSUP, "geometry lanes=%d kq=%d not compiled for block %d", lanes, kq, h->b);
  h->force_L = lanes;
  h->force_KQ = kq;
  h->max_wg = max_wg;
  h->r_dirty = true;
  h->alpha_M = 0;
  return 0;
}

int fkpm_autotune(fkpm_handle* h) {
  if (!h) return fail(FKPM_E_ARG, "null handle");
  HIPCHK(hipSetDevice(h->device));
  CHK(ensure_ready(h));
  if (h->force_L > 0) return fail(FKPM_E_STATE, "a forced geometry is set (fkpm_set_geometry)");
  CHK(tune(h));
  HIPCHK(hipStreamSynchronize(h->stream));
  return 0;
}

int fkpm_set_option(fkpm_handle* h, int option, int value) {
  if (!h) return fail(FKPM_E_ARG, "null handle");
  switch (option) {
    case FKPM_OPT_STOCH_METHOD:
      if (value != FKPM_STOCH_CLENSHAW && value != FKPM_STOCH_FORWARD && value != FKPM_STOCH_AUTO)
        return fail(FKPM_E_ARG, "bad stoch_matrix method %d", value);
      h->stoch_method = value;
      return 0;
    case FKPM_OPT_AUTOTUNE:
      h->autotune_on_use = value != 0;
      return 0;
    case FKPM_OPT_STORE_ALPHA:
      if (value < 0 || value > 2) return fail(FKPM_E_ARG, "bad store-alpha mode %d", value);
      h->store_alpha = value;
      h->alpha_M = 0;  // moments(M) again before autodiff_matrix
      h->a_slots = 0;
      return 0;
    case FKPM_OPT_SWEEP:
      if (value < -1 || value > 64) return fail(FKPM_E_ARG, "bad sweep %d", value);
      h->sweep_force = value;
      if (value >= 0)
        for (int k = 0; k < NKIND; k++)
          if (h->kc[k].L > 0) {
            h->kc[k].sweep = (h->kc[k].nt & fkd::NT_ORDER) ? 0 : value;
            derive_grid(h->nb, h->kc[k]);
          }
      return 0;
    case FKPM_OPT_GRAPH:
      if (value < -1 || value > 1) return fail(FKPM_E_ARG, "bad graph switch %d", value);
      h->graph_mode = value;
      return 0;
    case FKPM_OPT_SLICE:
      if (value < -1 || value > 1) return fail(FKPM_E_ARG, "bad slice switch %d", value);
      h->slice_force = value;
      if (value >= 0)
        for (int k = 0; k < NKIND; k++)
          if (h->kc[k].L > 0 && !h->kc[k].mfma)
            h->kc[k].nt = (h->kc[k].nt & ~fkd::NT_SLICE) | (value ? fkd::NT_SLICE : 0);
      return 0;
    case FKPM_OPT_ROW_ORDER:
      if (value < -1 || value > 1) return fail(FKPM_E_ARG, "bad row-order switch %d", value);
      h->order_force = value;
      apply_row_order(h);
      return 0;
    case FKPM_OPT_ALPHA_TABLE_MB:
      if (value < -1) return fail(FKPM_E_ARG, "bad table budget %d MiB", value);
      h->table_cap_mb = value;
      return 0;
    case FKPM_OPT_MFMA:
      if (value < 0 || value > 2) return fail(FKPM_E_ARG, "bad MFMA switch %d", value);
      if (h->mfma_on != (value != 0) || h->rr_force != (value == 2)) {
        h->mfma_on = value != 0;
        h->rr_force = value == 2;
        h->r_dirty = true;  // geometry (and padded width) chosen again at next use
        h->alpha_M = 0;
        h->tuned = false;
      }
      return 0;
  }
  return fail(FKPM_E_ARG, "unknown option %d", option);
}

int fkpm_bandwidth_probe(fkpm_handle* h, size_t bytes, int reps, double* gbs) {
  if (!h || !gbs || bytes == 0 || bytes % 16 != 0 || reps < 1)
    return fail(FKPM_E_ARG, "bandwidth_probe: bad arguments");
  HIPCHK(hipSetDevice(h->device));
  DevBuf a, b;
  struct Rel {
    DevBuf *x, *y;
    ~Rel() {
      x->release();
      y->release();
    }
  } rel{&a, &b};
  CHK(a.ensure(bytes));
  CHK(b.ensure(bytes));
  const size_t n = bytes / 16;
  CHK(zero_doubles(h, a.p, n * 2));
  // the plain copy (1024 workgroups), then the streaming one (4096); the
  // faster of the two is the ceiling
  double best = 0.0;
  for (int v = 0; v < 2; v++) {
    auto fn = v == 0 ? &fkd::k_copy16 : &fkd::k_copy16_nt;
    const int grid = v == 0 ? 1024 : 4096;
    CHK(launch(fn, dim3(grid), dim3(fkd::WG), h->stream, (const double2*)a.p, (double2*)b.p, n));
    HIPCHK(hipEventRecord(h->ev0, h->stream));
    for (int r = 0; r < reps; r++)
      CHK(launch(fn, dim3(grid), dim3(fkd::WG), h->stream, (const double2*)a.p, (double2*)b.p,
                 n));
    HIPCHK(hipEventRecord(h->ev1, h->stream));
    HIPCHK(hipEventSynchronize(h->ev1));
    float ms = 0.f;
    HIPCHK(hipEventElapsedTime(&ms, h->ev0, h->ev1));
    best = std::max(best, 2.0 * (double)bytes * reps / (ms * 1e-3) / 1e9);
  }
  *gbs = best;
  return 0;
}

}  // extern "C"

namespace fkd {
int geometries_for_block(int b, GeomChoice* out, int cap) {
  int n = 0;
#define FKD_GEO(bb, l, kq) \
  if (bb == b && n < cap) out[n++] = GeomChoice{l, kq};
  FKD_FOR_EACH_GEOMETRY(FKD_GEO)
#undef FKD_GEO
  return n;
}
}  // namespace fkd

// ---------------------------------------------------------------------------
// Host functions for the batched engine (kpm_batch.hip).
// ---------------------------------------------------------------------------
namespace fkpm_internal {

int scale_H_cx(hipStream_t st, const double* raw, void* dst, bool single, const int* row_of_block,
               const int* ci, int nnzb, int b, double mag, double shift) {
  const size_t cnt = (size_t)nnzb * b * b;
  if (cnt == 0) return 0;
  if (single)
    return launch(&fkd::k_scale_H<double, float, true>, dim3(grid_for(cnt)), dim3(256), st, raw,
                  (float*)dst, row_of_block, ci, nnzb, b, mag, shift);
  return launch(&fkd::k_scale_H<double, double, true>, dim3(grid_for(cnt)), dim3(256), st, raw,
                (double*)dst, row_of_block, ci, nnzb, b, mag, shift);
}

int pack_R_cx(hipStream_t st, const double* raw, void* dst, bool single, int n, int s, int sp) {
  const dim3 grid((n + 63) / 64, (sp + 15) / 16);
  if (single)
    return launch(&fkd::k_pack_R<double, float, true>, grid, dim3(fkd::WG), st, raw, (float*)dst, n,
                  s, sp);
  return launch(&fkd::k_pack_R<double, double, true>, grid, dim3(fkd::WG), st, raw, (double*)dst,
                n, s, sp);
}

int set_error(int code, const char* msg) { return fail(code, "%s", msg); }

bool lattice_row_order(int nb, const int* rp, const int* ci, std::vector<int>& order) {
  return lattice_order(nb, rp, ci, order);
}

}  // namespace fkpm_internal
