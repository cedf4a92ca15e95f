// C-ABI of the MI355X FDTD engine (include/gmes_engine.h).
//
// Host side of the engine: device memory for one sim, validation of every
// index a kernel will use (so a bad table becomes an error code, never an
// out-of-bounds access), grouping of source operations per cell, the
// per-step launch sequence (gmes/fdtd.py:1099-1122), HIP-graph capture of
// one step, HIP-event kernel timing and batches of sims.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <numeric>
#include <shared_mutex>
#include <string>
#include <unordered_set>
#include <exception>
#include <thread>
#include <atomic>
#include <vector>

#include "engine_kernels.h"

using namespace gmes_engine;

// Partial sums of gmes_sim_field_sum_sq_noalloc: 65536 blocks of 2048
// cells (boxes of up to 2^27 cells) and the total, 512 KiB per GPU.
constexpr int64_t kScratchPartials = 65536;
static __device__ __align__(256) double scratch[kScratchPartials + 1];

namespace {

thread_local char g_err[512];

int set_error(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof g_err, fmt, ap);
  va_end(ap);
  return code;
}

#define HIP_TRY(expr)                                                                   \
  do {                                                                                  \
    hipError_t e_ = (expr);                                                             \
    if (e_ != hipSuccess)                                                               \
      return set_error(e_ == hipErrorOutOfMemory ? GMES_ENOMEM : GMES_EDEVICE, "%s: %s", \
                       #expr, hipGetErrorString(e_));                                   \
  } while (0)

// Engine calls made from several threads (a served request is built on a
// worker thread while the main thread captures the batch step) must not
// run inside a stream capture: a synchronous copy, memset or free issued
// meanwhile can invalidate it.  Every entry point holds this lock shared
// (once per thread, however deeply entry points nest); a capture holds it
// exclusively, so it runs while no other thread is inside the engine.
std::shared_mutex g_capture_mu;
thread_local int tl_api_depth = 0;

struct ApiGuard {
  ApiGuard() {
    if (tl_api_depth++ == 0) g_capture_mu.lock_shared();
  }
  ~ApiGuard() {
    if (--tl_api_depth == 0) g_capture_mu.unlock_shared();
  }
};

// Exclusive for the duration of a capture; the calling thread's own shared
// hold is released first and taken back afterwards.
struct CaptureGuard {
  bool held;
  CaptureGuard() : held(tl_api_depth > 0) {
    if (held) g_capture_mu.unlock_shared();
    g_capture_mu.lock();
  }
  ~CaptureGuard() {
    g_capture_mu.unlock();
    if (held) g_capture_mu.lock_shared();
  }
};

// f(0) .. f(n - 1) on a few threads (passes over all `cells` of a sim while
// it is being set up); f writes only what is its own.  Starting the threads
// takes 0.1 ms, a pass over 2^18 cells about as long.
template <class F>
void host_parallel(int n, int64_t cells, F f) {
  const int most = cells < (1 << 18) ? 1 : 8;
  const int nt = std::min<int>(n, std::min<unsigned>(most, std::max(1u, std::thread::hardware_concurrency())));
  std::atomic<int> next{0};
  std::atomic<bool> failed{false};
  auto work = [&] {
    try {
      for (int q = next++; q < n; q = next++) f(q);
    } catch (const std::bad_alloc&) {
      failed = true;
    }
  };
  std::vector<std::thread> t;
  try {
    t.reserve(nt);  // a vector that could not grow would take its threads with it
    for (int q = 1; q < nt; ++q) t.emplace_back(work);
  } catch (const std::exception&) {  // no more threads, or no memory for one: the ones there do it
  }
  work();
  for (auto& x : t) x.join();
  if (failed) throw std::bad_alloc();
}

// Pinned staging of large field reads and writes: at most kStageMax buffers,
// leased for one transfer each and freed with the last sim.
constexpr int64_t kStageBytes = 16 << 20;
constexpr int kStageMax = 4, kStageThreads = 4;
struct StagePool {
  std::mutex mu;
  std::vector<void*> idle;
  int total = 0, sims = 0;
} g_stage;

void* stage_lease() {
  std::lock_guard<std::mutex> lk(g_stage.mu);
  if (!g_stage.idle.empty()) {
    void* p = g_stage.idle.back();
    g_stage.idle.pop_back();
    return p;
  }
  if (g_stage.total == kStageMax) return nullptr;
  void* p = nullptr;
  if (hipHostMalloc(&p, kStageBytes, hipHostMallocPortable) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  ++g_stage.total;
  return p;
}

void stage_return(void* p) {
  std::lock_guard<std::mutex> lk(g_stage.mu);
  g_stage.idle.push_back(p);
}

// a sim is created (1) or gone (-1)
void stage_sims(int d) {
  std::lock_guard<std::mutex> lk(g_stage.mu);
  g_stage.sims += d;
  if (g_stage.sims) return;
  for (void* p : g_stage.idle) (void)hipHostFree(p);
  g_stage.total -= (int)g_stage.idle.size();
  g_stage.idle.clear();
}

hipError_t dev_release(void* p) { return hipFree(p); }
hipError_t device_drain() { return hipDeviceSynchronize(); }
hipError_t stream_release(hipStream_t st) { return hipStreamDestroy(st); }

const int kAx1[6] = {1, 2, 0, 1, 2, 0};
const int kAx2[6] = {2, 0, 1, 2, 0, 1};
const int kGhostOrder[6][2] = {{1, 2}, {2, 0}, {0, 1}, {1, 2}, {2, 0}, {0, 1}};

bool active(const gmes_sim* s, int c) { return (s->g.active >> c) & 1u; }
bool is3d(const gmes_sim* s) { return s->g.active == 0x3Fu; }
// 3-D sims with rows under 256 cells store their rows unpadded (gmes_sim::packed)
bool packed_rows(const gmes_grid_desc* d) { return d->active == 0x3Fu && d->nz < 256; }
// A 2-D mode with a collapsed z axis (TMz, TEz): every active component
// has rows of at most 2 elements and exactly one updated z plane (its own
// axis z has extent 1; a z extent of 2 holds one ghost plane).  Single-sim
// steps of such modes use k_main2z.
bool is_2z(const gmes_sim* s) {
  if (is3d(s)) return false;
  for (int c = 0; c < 6; ++c) {
    if (!active(s, c)) continue;
    const int64_t* sh = s->shape[c];
    if (sh[2] > 2 || (c % 3 == 2 && sh[2] != 1) || sh[0] < 2 || sh[1] < 2) return false;
  }
  return true;
}

// device element of logical (i,j,k) / of a logical C-order flat index
int64_t dev_index(const gmes_sim* s, int c, int64_t i, int64_t j, int64_t k) {
  return kPad + i * s->pi[c] + j * s->pitch[c] + k * s->pk[c] - s->koff[c];
}
int64_t dev_flat(const gmes_sim* s, int c, int64_t flat) {
  const int64_t sz = s->shape[c][2], sy = s->shape[c][1];
  return dev_index(s, c, flat / (sy * sz), (flat / sz) % sy, flat % sz);
}


// Device memory.  When there is none left, the second buffers of the one-sweep
// steps on the device make room: sims that have them never keep out what
// would fit without them.
void sweep_reclaim(int device);
hipError_t dev_malloc(int device, void** p, size_t bytes) {
  const hipError_t e = hipMalloc(p, bytes);
  if (e != hipErrorOutOfMemory) return e;
  (void)hipGetLastError();
  // alone until it is allocated: another thread may have made room, or be
  // about to take it
  CaptureGuard alone;
  sweep_reclaim(device);
  return hipMalloc(p, bytes);
}

int dev_alloc(gmes_sim* s, void** p, size_t bytes) {
  if (bytes == 0) bytes = 16;
  HIP_TRY(dev_malloc(s->device, p, bytes));
  s->bytes += (int64_t)bytes;
  return GMES_OK;
}

void dev_free(gmes_sim* s, void* p, size_t bytes) {
  if (p) {
    (void)dev_release(p);
    s->bytes -= (int64_t)bytes;
  }
}

int state_words(const gmes_mat_rec& r) {
  switch (r.cls) {
    case GMES_CLS_DRUDE: return 2 * r.n1;
    case GMES_CLS_DCP_ADE: return 1 + 2 * r.n1 + 2 * r.n2;
    case GMES_CLS_DCP_PLRC: return r.n1 + 2 * r.n2;
    case GMES_CLS_DM2: return 3 * r.n1;
    default: return 0;
  }
}

size_t real_size(const gmes_sim* s) { return s->fp64 ? 8 : 4; }

// bytes of one ADE state word of a class
size_t ade_word(const gmes_sim* s, int cls) {
  if (cls == GMES_CLS_DCP_PLRC) return 2 * real_size(s);
  if (cls == GMES_CLS_DM2) return real_size(s);
  return (size_t)s->esize;
}

void free_ade(gmes_sim* s) {
  for (int c = 0; c < 6; ++c)
    for (int k = 0; k < GMES_NCLS; ++k) {
      AdeList& L = s->ade[c][k];
      if (L.cell) (void)dev_release(L.cell);
      if (L.rec) (void)dev_release(L.rec);
      if (L.state) (void)dev_release(L.state);
      L = AdeList();
    }
}

// Byte copies of the material ids for the real-FP32 3-D main kernels,
// which then read 1 byte per cell and component instead of 2, when the
// record table has at most 256 entries (other sims and kernels read the
// 16-bit ids; for wider words the saving measured below the cost).
int upload_byte_ids(gmes_sim* s) {
  const bool narrow = is3d(s) && s->g.dtype == GMES_F32 && s->recs.size() <= 256;
  for (int c = 0; c < 6; ++c) {
    if (!narrow || !active(s, c)) {
      if (s->ids8[c]) { (void)dev_release(s->ids8[c]); s->ids8[c] = nullptr; }
      continue;
    }
    if (!s->ids8[c]) {
      int rc = dev_alloc(s, (void**)&s->ids8[c], (size_t)s->dsize[c]);
      if (rc) return rc;
    }
    launch_narrow_ids(s->ids[c], s->ids8[c], s->dsize[c], s->stream);  // pads included
    HIP_TRY(hipGetLastError());
  }
  HIP_TRY(hipStreamSynchronize(s->stream));
  return GMES_OK;
}

// Coordinates along `axis` where the CPML c coefficient of profile set p is
// exactly zero for every active component: the longest such run [lo, hi),
// packed as lo | hi << 16 (0 = empty: every coordinate keeps its psi).
// There psi stays +0, and the kernels neither read nor write it.
int32_t zero_c_run(const gmes_sim* s, int p, int axis) {
  int lo = 0, hi = INT32_MAX;
  for (int c = 0; c < 6; ++c) {
    if (!active(s, c)) continue;
    const std::vector<double>& v = s->prof_host[p][c][axis];
    if (s->prof_w[p][c][axis] != 3 || v.empty()) return 0;
    const int n = (int)(v.size() / 3);
    int best_a = 0, best_b = 0;
    for (int q = 0; q < n;) {
      if (v[3 * (size_t)q + 1] != 0.0) { ++q; continue; }
      int e = q;
      while (e < n && v[3 * (size_t)e + 1] == 0.0) ++e;
      if (e - q > best_b - best_a) { best_a = q; best_b = e; }
      q = e;
    }
    lo = std::max(lo, best_a);
    hi = std::min(hi, best_b);
  }
  if (lo >= hi || hi > 0x7FFF) return 0;
  return lo | (hi << 16);
}

// Real-FP32 3-D sims whose three components of a field type all have CPML
// cells: each axis is read by two of them (E: x by Ey and Ez, y by Ex and
// Ez, z by Ex and Ey; H: x by Hy and Hz, y by Hx and Hz, z by Hx and Hy),
// at the same coordinates.  When their set-0 rows are identical, and every
// row is (b, 0, 1) inside the zero-c run of its axis, the kernels load one
// row per axis with the cell's other operands (MainArgs::pp) instead of
// two rows per component after the cell's record.
void profile_prefetch(gmes_sim* s) {
  s->pp_ok[0] = s->pp_ok[1] = false;
  if (!is3d(s) || s->g.dtype != GMES_F32 || s->nprof < 1) return;
  for (int e = 0; e < 2; ++e) {
    const int c0 = e ? 3 : 0;
    bool ok = true;
    for (int c = c0; c < c0 + 3 && ok; ++c) ok = s->pml_state[c] && s->has_cls[c][GMES_CLS_CPML];
    const int pairs[3][2] = {{c0 + 1, c0 + 2}, {c0, c0 + 2}, {c0, c0 + 1}};
    for (int a = 0; a < 3 && ok; ++a) {
      const std::vector<double>& r0 = s->prof_host[0][pairs[a][0]][a];
      const std::vector<double>& r1 = s->prof_host[0][pairs[a][1]][a];
      ok = s->prof_w[0][pairs[a][0]][a] == 3 && s->prof_w[0][pairs[a][1]][a] == 3 && !r0.empty() && r0 == r1;
      const int lo = s->prun[a] & 0xFFFF, hi = s->prun[a] >> 16;
      for (int q = lo; ok && q < hi && 3 * (size_t)q + 2 < r0.size(); ++q)
        ok = r0[3 * (size_t)q + 1] == 0.0 && r0[3 * (size_t)q + 2] == 1.0;
    }
    s->pp_ok[e] = ok;
  }
}

// Real-FP32 3-D sims: the components with UPML (and no CPML) state whose
// state word the 3-D kernels load together with the cell's other operands,
// and a box of storage coordinates (per axis lo | hi << 16) holding no UPML
// cell of those components, inside which the kernels read the array's
// guard word instead (its value is unused there).  The box is the run of
// non-UPML cells through each component's centre along each axis,
// intersected over the components, and is kept only if no cell inside it
// is UPML; otherwise the kernels load the word after the cell's record.
void upml_box(gmes_sim* s) {
  s->upml_pre = 0;
  for (int a = 0; a < 3; ++a) s->ubox[a] = 0;
  if (!is3d(s) || s->g.dtype != GMES_F32) return;
  int64_t lo[3] = {0, 0, 0}, hi[3] = {0x7FFF, 0x7FFF, 0x7FFF};
  unsigned mask = 0;
  for (int c = 0; c < 6; ++c) {
    if (!active(s, c) || !s->pml_state[c] || s->has_cls[c][GMES_CLS_CPML] || !s->has_cls[c][GMES_CLS_UPML]) continue;
    mask |= 1u << c;
    const int64_t* n = s->shape[c];
    const std::vector<uint16_t>& ids = s->host_ids[c];
    for (int a = 0; a < 3; ++a) {
      int64_t ix[3] = {n[0] / 2, n[1] / 2, n[2] / 2};
      auto upml_at = [&](int64_t v) {
        ix[a] = v;
        return s->recs[ids[(ix[0] * n[1] + ix[1]) * n[2] + ix[2]]].cls == GMES_CLS_UPML;
      };
      const int64_t mid = n[a] / 2;
      if (upml_at(mid)) return;
      int64_t l = mid, h = mid + 1;
      while (l > 0 && !upml_at(l - 1)) --l;
      while (h < n[a] && !upml_at(h)) ++h;
      lo[a] = std::max(lo[a], l);
      hi[a] = std::min(hi[a], h);
    }
  }
  if (!mask) return;
  for (int a = 0; a < 3; ++a)
    if (lo[a] >= hi[a]) return;
  for (int c = 0; c < 6; ++c) {
    if (!((mask >> c) & 1u)) continue;
    const int64_t* n = s->shape[c];
    const std::vector<uint16_t>& ids = s->host_ids[c];
    for (int64_t i = lo[0]; i < std::min(hi[0], n[0]); ++i)
      for (int64_t j = lo[1]; j < std::min(hi[1], n[1]); ++j)
        for (int64_t k = lo[2]; k < std::min(hi[2], n[2]); ++k)
          if (s->recs[ids[(i * n[1] + j) * n[2] + k]].cls == GMES_CLS_UPML) return;
  }
  s->upml_pre = mask;
  for (int a = 0; a < 3; ++a) s->ubox[a] = (int32_t)(lo[a] | (hi[a] << 16));
}

// Real-FP32 3-D sims whose three components of a field type all get their
// UPML state prefetched (upml_pre): each axis is a curl axis of two of
// them (E: x of Ey and Ez, y of Ex and Ez, z of Ex and Ey; H: x of Hy and
// Hz, y of Hx and Hz, z of Hx and Hy), which take c1..c4 at the same
// coordinates, and the own axis of the third, which takes c5, c6.  When
// the two set-0 rows of each axis are identical, the kernels load that
// row and the owner's row with the cell's other operands (MainArgs::ur)
// instead of three rows per component after the cell's record.
void upml_rows(gmes_sim* s) {
  s->ur_ok[0] = s->ur_ok[1] = false;
  if (!is3d(s) || s->g.dtype != GMES_F32 || s->nprof < 1) return;
  for (int e = 0; e < 2; ++e) {
    const int c0 = e ? 3 : 0;
    bool ok = true;
    for (int c = c0; c < c0 + 3 && ok; ++c) ok = (s->upml_pre >> c) & 1u;
    const int pairs[3][2] = {{c0 + 1, c0 + 2}, {c0, c0 + 2}, {c0, c0 + 1}};
    for (int a = 0; a < 3 && ok; ++a) {
      const std::vector<double>& r0 = s->prof_host[0][pairs[a][0]][a];
      const std::vector<double>& r1 = s->prof_host[0][pairs[a][1]][a];
      ok = s->prof_w[0][pairs[a][0]][a] == 6 && s->prof_w[0][pairs[a][1]][a] == 6 &&
           s->prof_w[0][c0 + a][a] == 6 && !r0.empty() && r0 == r1 && !s->prof_host[0][c0 + a][a].empty();
    }
    s->ur_ok[e] = ok;
  }
}

template <class R>
int upload_tables(gmes_sim* s) {
  std::vector<DevRec<R>> dr(s->recs.size());
  for (size_t i = 0; i < s->recs.size(); ++i) {
    const gmes_mat_rec& r = s->recs[i];
    dr[i].cls = r.cls;
    dr[i].n1 = r.n1;
    dr[i].n2 = r.n2;
    dr[i].prof = r.prof;
    dr[i].coef_off = r.coef_off;
    if (r.cls == GMES_CLS_CPML && r.prof >= 0 && r.prof < s->nprof) {
      dr[i].n1 = zero_c_run(s, r.prof, 0);
      dr[i].n2 = zero_c_run(s, r.prof, 1);
      dr[i].coef_off = zero_c_run(s, r.prof, 2);
    }
    dr[i].c0 = (R)(s->g.dt / r.eps_mu);  // dt / eps_inf in FP64, rounded once
    dr[i].eps_mu = (R)r.eps_mu;
    dr[i].inv_eps = (R)(1.0 / r.eps_mu);
    dr[i].val_re = (R)r.value[0];
    dr[i].val_im = (R)r.value[1];
  }
  std::vector<R> cf(s->coef.size());
  for (size_t i = 0; i < cf.size(); ++i) cf[i] = (R)s->coef[i];
  // profiles into one buffer with offsets
  std::vector<int64_t> off(64 * 18, 0);
  std::vector<R> pr;
  for (int p = 0; p < s->nprof; ++p)
    for (int c = 0; c < 6; ++c)
      for (int a = 0; a < 3; ++a) {
        off[(p * 6 + c) * 3 + a] = (int64_t)pr.size();
        // FP32 tables hold 1/kappa in the CPML kappa column (the FP32 kernels
        // multiply); FP64 tables hold the reference's values unchanged.
        const std::vector<double>& src = s->prof_host[p][c][a];
        const bool recip = !s->fp64 && s->prof_w[p][c][a] == 3;
        for (size_t q = 0; q < src.size(); ++q)
          pr.push_back((R)(recip && q % 3 == 2 ? 1.0 / src[q] : src[q]));
      }
  if (pr.size() > (size_t)INT32_MAX) return set_error(GMES_EINVAL, "profile pool too large");
  for (int c = 0; c < 6; ++c)
    for (int a = 0; a < 3; ++a) s->prof_off0[c][a] = off[c * 3 + a];
  if (pr.empty()) pr.push_back(R(0));
  if (cf.empty()) cf.push_back(R(0));
  int rc;
  if ((rc = dev_alloc(s, &s->d_recs, dr.size() * sizeof(DevRec<R>)))) return rc;
  if ((rc = dev_alloc(s, &s->d_coef, cf.size() * sizeof(R)))) return rc;
  if ((rc = dev_alloc(s, &s->d_prof, pr.size() * sizeof(R)))) return rc;
  if ((rc = dev_alloc(s, (void**)&s->d_prof_off, off.size() * sizeof(int64_t)))) return rc;
  HIP_TRY(hipMemcpy(s->d_recs, dr.data(), dr.size() * sizeof(DevRec<R>), hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(s->d_coef, cf.data(), cf.size() * sizeof(R), hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(s->d_prof, pr.data(), pr.size() * sizeof(R), hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(s->d_prof_off, off.data(), off.size() * sizeof(int64_t), hipMemcpyHostToDevice));
  return GMES_OK;
}

template <class R>
int upload_sources(gmes_sim* s) {
  // stable grouping by (phase, comp, cell); E groups first
  std::vector<int64_t> order(s->ops.size());
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int64_t x, int64_t y) {
    const gmes_src_op &a = s->ops[x], &b = s->ops[y];
    const int pa = a.comp >= 3, pb = b.comp >= 3;
    if (pa != pb) return pa < pb;
    if (a.comp != b.comp) return a.comp < b.comp;
    return a.cell < b.cell;
  });
  std::vector<DevSrcOp<R>> dops(order.size());
  std::vector<SrcGroup> groups;
  s->ngroups_e = s->ngroups_h = 0;
  for (size_t n = 0; n < order.size(); ++n) {
    const gmes_src_op& o = s->ops[order[n]];
    DevSrcOp<R>& d = dops[n];
    d.kind = o.kind; d.wave = o.wave; d.aux = o.aux; d.aux_comp = o.aux_comp;
    d.i0 = o.i0; d.i1 = o.i1; d.k = (R)o.k; d.r0 = (R)o.r0; d.r1 = (R)o.r1;
    if (o.kind == GMES_SRC_AUX_ADD || o.kind == GMES_SRC_AUX_SUB) {
      d.i0 = dev_flat(s->aux[o.aux], o.aux_comp, o.i0);
      d.i1 = dev_flat(s->aux[o.aux], o.aux_comp, o.i1);
    }
    const int64_t dcell = dev_flat(s, o.comp, o.cell);
    if (groups.empty() || groups.back().comp != o.comp || groups.back().cell != dcell) {
      SrcGroup g;
      g.comp = o.comp; g.cell = dcell; g.begin = (int32_t)n; g.end = (int32_t)n + 1; g.pad_ = 0;
      groups.push_back(g);
      if (o.comp < 3) s->ngroups_e++; else s->ngroups_h++;
    } else {
      groups.back().end = (int32_t)n + 1;
    }
  }
  if (s->d_ops) { dev_free(s, s->d_ops, 0); s->d_ops = nullptr; }
  if (s->d_groups) { dev_free(s, s->d_groups, 0); s->d_groups = nullptr; }
  int rc;
  if ((rc = dev_alloc(s, &s->d_ops, std::max<size_t>(1, dops.size()) * sizeof(DevSrcOp<R>)))) return rc;
  if ((rc = dev_alloc(s, (void**)&s->d_groups, std::max<size_t>(1, groups.size()) * sizeof(SrcGroup)))) return rc;
  if (!dops.empty())
    HIP_TRY(hipMemcpy(s->d_ops, dops.data(), dops.size() * sizeof(DevSrcOp<R>), hipMemcpyHostToDevice));
  if (!groups.empty())
    HIP_TRY(hipMemcpy(s->d_groups, groups.data(), groups.size() * sizeof(SrcGroup), hipMemcpyHostToDevice));
  return GMES_OK;
}

// ------------------------------------------------------------ launching
template <class T>
FieldArgs<T> field_args(const gmes_sim* s) {
  FieldArgs<T> a;
  for (int c = 0; c < 6; ++c) {
    a.f[c] = static_cast<T*>(s->f[c]);
    for (int d = 0; d < 3; ++d) a.s[c][d] = (int)s->shape[c][d];
    a.pi[c] = s->pi[c];
    a.p[c] = s->pitch[c];
    a.pk[c] = s->pk[c];
    a.koff[c] = s->koff[c];
  }
  a.active = s->g.active;
  return a;
}

int next_pow2(int v) {
  int p = 1;
  while (p < v) p <<= 1;
  return p;
}

void time_begin(gmes_sim* s, int fam, hipStream_t st) {
  if (!s->timing.on) return;
  hipEvent_t a, b;
  (void)hipEventCreate(&a);
  (void)hipEventCreate(&b);
  (void)hipEventRecord(a, st);
  s->timing.pending.push_back({fam, {a, b}});
}

void time_end(gmes_sim* s, hipStream_t st) {
  if (!s->timing.on) return;
  (void)hipEventRecord(s->timing.pending.back().second.second, st);
}

// Ghost-copy arguments of one field type; total = ghost points.
template <class T>
GhostArgs<T> ghost_args(const gmes_sim* s, bool electric, int tick, int64_t& total) {
  using R = typename real_of<T>::type;
  GhostArgs<T> g{};
  g.fa = field_args<T>(s);
  g.ncomp = 0;
  total = 0;
  for (int c = electric ? 0 : 3; c < (electric ? 3 : 6); ++c) {
    if (!active(s, c)) continue;
    const int t = g.ncomp++;
    const int a1 = kGhostOrder[c][0], a2 = kGhostOrder[c][1], a0 = c % 3;
    g.comp[t] = c;
    g.ax[t][0] = a1; g.ax[t][1] = a2; g.ax[t][2] = a0;
    const int64_t p1 = s->shape[c][a0] * s->shape[c][a2], p2 = s->shape[c][a0] * (s->shape[c][a1] - 1);
    g.count[t] = p1 + p2;
    g.skip[t] = 0;
    if (!electric && s->fuse_hz && s->shape[c][2] == 2) {  // the z plane is the E kernel's
      if (a2 == 2) g.count[t] = p1;
      else if (a1 == 2) { g.skip[t] = p1; g.count[t] = p2; }
    }
    g.ph[t][0] = cplx<R>{(R)s->g.phase[c][a1][0], (R)s->g.phase[c][a1][1]};
    g.ph[t][1] = cplx<R>{(R)s->g.phase[c][a2][0], (R)s->g.phase[c][a2][1]};
    total += g.count[t];
  }
  g.tick = tick;
  g.ctl = reinterpret_cast<Ctl*>(s->d_clock);
  return g;
}

template <class T>
void enqueue_ghost(gmes_sim* s, bool electric, int tick, hipStream_t st) {
  int64_t total = 0;
  GhostArgs<T> g = ghost_args<T>(s, electric, tick, total);
  time_begin(s, 4, st);
  launch_ghost<T>(g, total, st);
  time_end(s, st);
}

// Main-kernel arguments of one field type; ext = the largest storage extent
// of its components.  False when the field type has no active component.
template <class T>
bool main_args(const gmes_sim* s, bool electric, MainArgs<T>& m, int ext[3]) {
  using R = typename real_of<T>::type;
  m = MainArgs<T>{};
  m.fa = field_args<T>(s);
  ext[0] = ext[1] = ext[2] = 0;
  bool any = false;
  for (int c = electric ? 0 : 3; c < (electric ? 3 : 6); ++c) {
    if (!active(s, c)) continue;
    any = true;
    for (int d = 0; d < 3; ++d) ext[d] = std::max<int>(ext[d], (int)s->shape[c][d]);
  }
  if (!any) return false;
  m.kloop = !is3d(s) && ext[2] <= 2;
  m.kext = ext[2];
  m.cpml_mask = 0;
  for (int c = 0; c < 6; ++c)
    if (s->pml_state[c] && s->has_cls[c][GMES_CLS_CPML]) m.cpml_mask |= 1u << c;
  for (int a = 0; a < 3; ++a) m.prun[a] = s->prun[a];
  m.upml_mask = s->upml_pre;
  for (int a = 0; a < 3; ++a) m.ubox[a] = s->ubox[a];
  m.hzg = electric && s->fuse_hz;
  if (m.hzg) {
    m.hzph[0] = cplx<R>{(R)s->g.phase[3][2][0], (R)s->g.phase[3][2][1]};
    m.hzph[1] = cplx<R>{(R)s->g.phase[4][2][0], (R)s->g.phase[4][2][1]};
    m.hyxph = cplx<R>{(R)s->g.phase[4][0][0], (R)s->g.phase[4][0][1]};
  }
  for (int c = 0; c < 6; ++c)
    for (int a = 0; a < 3; ++a) m.po0[c][a] = (int)s->prof_off0[c][a];
  m.ur = 0;
  if (s->ur_ok[electric ? 0 : 1]) {
    // shared rows: x of the 2nd component, y and z of the 1st; own rows:
    // axis a of component a
    const int c0 = electric ? 0 : 3;
    m.ur = 1;
    m.urs[0] = m.po0[c0 + 1][0];
    m.urs[1] = m.po0[c0][1];
    m.urs[2] = m.po0[c0][2];
    for (int a = 0; a < 3; ++a) m.uro[a] = m.po0[c0 + a][a];
  }
  m.pp = 0;
  if (s->pp_ok[electric ? 0 : 1]) {
    // axis x: 2nd component (Ey / Hy), axis y and z: 1st component (Ex / Hx)
    const int c0 = electric ? 0 : 3;
    m.pp = 1;
    m.pprow[0] = m.po0[c0 + 1][0];
    m.pprow[1] = m.po0[c0][1];
    m.pprow[2] = m.po0[c0][2];
  }
  m.narrow = 1;
  for (int c = 0; c < 6; ++c) {
    m.ids[c] = s->ids[c];
    m.ids8[c] = s->ids8[c];
    if (active(s, c) && !s->ids8[c]) m.narrow = 0;
    m.pml[c] = s->pml_state[c];
    m.dsize[c] = (int)s->dsize[c];
  }
  m.recs = static_cast<const DevRec<R>*>(s->d_recs);
  m.prof = static_cast<const R*>(s->d_prof);
  m.prof_off = s->d_prof_off;
  m.d[0] = (R)s->g.dx; m.d[1] = (R)s->g.dy; m.d[2] = (R)s->g.dz;
  m.inv_d[0] = (R)(1.0 / s->g.dx); m.inv_d[1] = (R)(1.0 / s->g.dy); m.inv_d[2] = (R)(1.0 / s->g.dz);
  m.nrec = (int)s->recs.size();
  m.n[0] = s->g.nx; m.n[1] = s->g.ny; m.n[2] = s->g.nz;
  m.fuse = electric && s->fuse_e;
  for (int c = 0; c < 3; ++c)
    for (int t = 0; t < 2; ++t) {
      const int a = kGhostOrder[c][t];
      m.gax[c][t] = a;
      m.gph[c][t] = cplx<R>{(R)s->g.phase[c][a][0], (R)s->g.phase[c][a][1]};
    }
  return true;
}


// Tile (bx along k, by along j) of the main kernels: the sim's own setting
// (gmes_sim_set_tile, gmes_sim_autotune) or the default.  3-D: (j,k) tiles
// of one i plane, 128 x 2 for long rows; on packed rows (gmes_sim::packed)
// 256 x 1 means flat blocks of 256 consecutive (j, k) points of a plane,
// the default there.  Other modes: a k x j tile of one i plane.
void tile_of(const gmes_sim* s, const int ext[3], int& bx, int& by) {
  bx = s->tile_bx;
  by = s->tile_by;
  if (bx > 0 && by > 0 && (is3d(s) || (bx <= next_pow2(ext[2]) && ext[2] > 2))) return;
  if (is3d(s) && s->packed) {
    bx = 256;
    by = 1;
  } else if (is3d(s)) {
    // real FP32: whole 256-cell rows per block when they divide the row
    // (256^3: E launch 0.1708 to 0.1675 ms, H unchanged; FP64 0.5% slower
    // that way), else 128 x 2
    bx = s->esize == 4 && s->g.nz % 256 == 0 ? 256 : std::min(128, next_pow2(s->g.nz));
    by = std::max(1, 256 / bx);
  } else if (ext[2] <= 2) {
    bx = 1;  // short rows: a thread per (i, j) walks k (MainArgs::kloop)
    by = std::min(256, next_pow2(ext[1]));
  } else {
    bx = std::min(64, next_pow2(ext[2]));
    by = std::max(1, std::min(256 / bx, next_pow2(ext[1])));
  }
}

template <class T>
void launch_main_tile(const gmes_sim* s, bool electric, const MainArgs<T>& m, int ext[3], int bx, int by,
                      hipStream_t st) {
  if (is3d(s) && s->packed && bx == 256 && by == 1) {
    launch_main3d_flat<T>(electric, m, st);
  } else if (is3d(s)) {
    launch_main3d<T>(electric, m, bx, by, s->tile_ic > 0 ? s->tile_ic : 1, st);
  } else {
    launch_main<T>(electric, m, ext, bx, by, st);
  }
}

template <class T>
void enqueue_main(gmes_sim* s, bool electric, hipStream_t st) {
  MainArgs<T> m;
  int ext[3];
  if (!main_args<T>(s, electric, m, ext)) return;
  time_begin(s, electric ? 0 : 1, st);
  if (is_2z(s)) {
    launch_main2z<T>(electric, m, ext, st);
  } else {
    int bx, by;
    tile_of(s, ext, bx, by);
    launch_main_tile<T>(s, electric, m, ext, bx, by, st);
  }
  time_end(s, st);
}

template <class T>
AdeArgs<T> ade_args(const gmes_sim* s, int c, int cls) {
  using R = typename real_of<T>::type;
  const AdeList& L = s->ade[c][cls];
  AdeArgs<T> a{};
  a.fa = field_args<T>(s);
  a.cell = L.cell; a.rec = L.rec; a.state = L.state; a.n = (int)L.n;
  a.recs = static_cast<const DevRec<R>*>(s->d_recs);
  a.coef = static_cast<const R*>(s->d_coef);
  a.d[0] = (R)s->g.dx; a.d[1] = (R)s->g.dy; a.d[2] = (R)s->g.dz;
  a.dt = (R)s->g.dt;
  a.ctl = reinterpret_cast<Ctl*>(s->d_clock);
  return a;
}

template <class T>
void enqueue_ade(gmes_sim* s, hipStream_t st) {
  for (int c = 0; c < 3; ++c)
    for (int cls = GMES_CLS_DRUDE; cls < GMES_NCLS; ++cls) {
      if (s->ade[c][cls].n == 0) continue;
      const AdeArgs<T> a = ade_args<T>(s, c, cls);
      time_begin(s, 2, st);
      launch_ade<T>(cls, c, a, st);
      time_end(s, st);
    }
}

template <class T>
SrcArgs<T> src_args(const gmes_sim* s, bool electric) {
  using R = typename real_of<T>::type;
  SrcArgs<T> a{};
  a.fa = field_args<T>(s);
  a.groups = s->d_groups + (electric ? 0 : s->ngroups_e);
  a.ngroups = electric ? s->ngroups_e : s->ngroups_h;
  a.ops = static_cast<const DevSrcOp<R>*>(s->d_ops);
  a.waves = s->d_waves;
  a.aux = static_cast<void* const*>(s->d_aux_ptrs);
  a.ctl = reinterpret_cast<Ctl*>(s->d_clock);
  return a;
}

template <class T>
void enqueue_src(gmes_sim* s, bool electric, hipStream_t st) {
  const SrcArgs<T> a = src_args<T>(s, electric);
  if (a.ngroups == 0) return;
  time_begin(s, 3, st);
  launch_src<T>(a, st);
  time_end(s, st);
}

// Records the probes of one field type or, after a one-sweep step, of both.
constexpr int kProbeH = 0, kProbeE = 1, kProbeBoth = 2;
template <class T>
void enqueue_probe(gmes_sim* s, int types, hipStream_t st) {
  if (s->probes.empty()) return;
  ProbeArgs<T> a{};
  a.fa = field_args<T>(s);
  a.cells = s->d_probe_cells;
  a.comps = s->d_probe_comps;
  a.n = (int)s->probes.size();
  a.types = types;
  a.buf = s->d_probe_buf;
  a.cap = s->probe_cap;
  a.ctl = reinterpret_cast<Ctl*>(s->d_clock);
  launch_probe<T>(a, st);
}

// DFT monitor jobs of a sim, first block numbered block0.
template <class T>
void dft_jobs(const gmes_sim* s, std::vector<DftJob<T>>& out, int64_t& block0) {
  for (const auto& d : s->dfts) {
    DftJob<T> J{};
    J.f = static_cast<T*>(s->f[d.comp]);
    J.pi = s->pi[d.comp];
    J.p = s->pitch[d.comp];
    J.pk = s->pk[d.comp];
    J.koff = s->koff[d.comp];
    J.comp = d.comp;
    for (int a = 0; a < 3; ++a) { J.lo[a] = (int)d.lo[a]; J.n[a] = (int)d.n[a]; }
    J.nfreq = d.nfreq;
    J.decim = d.decim;
    J.electric = d.comp < 3;
    J.ncells = d.ncells;
    J.acc = d.acc;
    J.w = s->d_dft_w;
    J.ctl = reinterpret_cast<Ctl*>(s->d_clock);
    J.block0 = block0;
    block0 += (d.ncells + 255) / 256;
    out.push_back(J);
  }
}

// The device table holds the jobs on the buffers of either parity
// (gmes_sim::par), half after half.
template <class T>
int upload_dft_jobs_t(gmes_sim* s) {
  std::vector<DftJob<T>> jobs;
  for (int p = 0; p < 2; ++p) {
    int64_t nb = 0;
    std::vector<DftJob<T>> half;
    dft_jobs<T>(s, half, nb);
    if (p != s->par && s->sweep_ok)
      for (auto& J : half) J.f = static_cast<T*>(s->f_alt[J.comp]);
    s->dft_blocks = nb;
    jobs.insert(jobs.end(), half.begin(), half.end());
  }
  if (jobs.empty()) return GMES_OK;
  // capacity for 16 monitors on two buffer sets: adding monitors rarely reallocates (a free
  // would wait for every kernel on the device)
  const int64_t need = std::max<int64_t>(32, (int64_t)jobs.size());
  if (need > s->dft_jobs_cap) {
    if (s->d_dft_jobs) HIP_TRY(dev_release(s->d_dft_jobs));
    s->d_dft_jobs = nullptr;
    HIP_TRY(dev_malloc(s->device, &s->d_dft_jobs, (size_t)need * sizeof(DftJob<T>)));
    s->dft_jobs_cap = need;
  }
  HIP_TRY(hipMemcpy(s->d_dft_jobs, jobs.data(), jobs.size() * sizeof(DftJob<T>), hipMemcpyHostToDevice));
  return GMES_OK;
}

int upload_dft_jobs(gmes_sim* s) {
  switch (s->g.dtype) {
    case GMES_F32: return upload_dft_jobs_t<float>(s);
    case GMES_F64: return upload_dft_jobs_t<double>(s);
    case GMES_C64: return upload_dft_jobs_t<cplx<float>>(s);
    default: return upload_dft_jobs_t<cplx<double>>(s);
  }
}

template <class T>
void enqueue_dft(gmes_sim* s, hipStream_t st) {
  if (s->dfts.empty()) return;
  launch_dft_batch<T>(static_cast<const DftJob<T>*>(s->d_dft_jobs) + s->par * s->dfts.size(), (int)s->dfts.size(),
                      s->dft_blocks, st);
}

void enqueue_step(gmes_sim* s, hipStream_t st);

// One whole step of each auxiliary (TFSF) grid of s, between the E and H
// half steps of s; sweep: the step of s is a one-sweep step.
void enqueue_aux_steps(gmes_sim* s, bool sweep, hipStream_t st);

bool on_ghost_copy_plane(const gmes_sim* s, int c, int64_t x, bool source, bool ghost);
int sweep_sources(gmes_sim* s);
void destroy_graph(gmes_sim* s);
hipError_t sync_exec(gmes_sim* s);

// ---- one-sweep steps (step3d.hip)
//
// A real FP32 or FP64, or complex FP32, 3-D sim takes them when
//   * it holds no DM2 cells, and one kind of absorber with one profile set,
//     whose two rows per axis agree (a single Shell),
//   * three whole (j, k) rows fit a block, with some absorbers more
//     (sweep_min_rows): nz <= 341; 256 with 8-byte words and an absorber along
//     x or y; at most half of the E work is done twice,
//   * its distinct triples of records fit a block's LDS,
//   * its sources are off the ghost planes, and no E probe sits on a ghost
//     plane (it reads the plane before the copy),
//   * with dispersive cells, an auxiliary grid or sources on more than
//     kSweepMaxSrc cells: what stepfix.hip and sweep_fix_build ask, and not too
//     many of them (sweep_list_limit),
//   * a component's CPML state is under 4 GiB (32-bit byte offsets),
//   * its second buffers leave the device half empty, or are a small part of
//     what is idle (sweep_room), and
//   * the caller asked for no tile and did not turn ghost fusion off.
// Other sims keep the two-kernel step.
constexpr int kSweepMinRows = 3;
constexpr int64_t kSweepMaxTab = 24 * 1024;  // bytes of entries in LDS
constexpr int kSweepMaxSrc = 16;
constexpr int kSweepFloor = 20;        // waves whose plane takes as long as the latency of one
constexpr int64_t kSweepLds = 160 * 1024;
constexpr size_t kSweepAlign = 4096;

// The two rows read along each axis by one field type agree; CPML: inside
// the run without live state every row is (b, 0, 1).
bool sweep_rows_agree(const gmes_sim* s, int width) {
  for (int e = 0; e < 2; ++e) {
    const int32_t* run = e ? s->sweep_run_h : s->sweep_run_e;
    const int c0 = e ? 3 : 0;
    const int pairs[3][2] = {{c0 + 1, c0 + 2}, {c0, c0 + 2}, {c0, c0 + 1}};
    for (int a = 0; a < 3; ++a) {
      const std::vector<double>& r0 = s->prof_host[0][pairs[a][0]][a];
      const std::vector<double>& r1 = s->prof_host[0][pairs[a][1]][a];
      if (s->prof_w[0][pairs[a][0]][a] != width || r0.empty() || r0 != r1 || s->prof_w[0][pairs[a][1]][a] != width)
        return false;
      if (width == 6 && (s->prof_w[0][c0 + a][a] != 6 || s->prof_host[0][c0 + a][a].empty())) return false;
      if (width == 3)
        for (int q = run[a] & 0xFFFF; q < (run[a] >> 16) && 3 * (size_t)q + 2 < r0.size(); ++q)
          if (r0[3 * (size_t)q + 1] != 0.0 || r0[3 * (size_t)q + 2] != 1.0) return false;
    }
  }
  return true;
}

// A box of storage coordinates (per axis lo | hi << 16) holding no UPML cell
// of any component, from the runs of non-UPML cells through the centres;
// empty runs when the box is not free.
void upml_free_box(const gmes_sim* s, int32_t box[3]) {
  for (int a = 0; a < 3; ++a) box[a] = 0;
  int64_t lo[3] = {0, 0, 0}, hi[3] = {0x7FFF, 0x7FFF, 0x7FFF};
  for (int c = 0; c < 6; ++c) {
    const int64_t* n = s->shape[c];
    const std::vector<uint16_t>& ids = s->host_ids[c];
    for (int a = 0; a < 3; ++a) {
      int64_t ix[3] = {n[0] / 2, n[1] / 2, n[2] / 2};
      auto upml_at = [&](int64_t v) {
        ix[a] = v;
        return s->recs[ids[(ix[0] * n[1] + ix[1]) * n[2] + ix[2]]].cls == GMES_CLS_UPML;
      };
      const int64_t mid = n[a] / 2;
      if (upml_at(mid)) return;
      int64_t l = mid, h = mid + 1;
      while (l > 0 && !upml_at(l - 1)) --l;
      while (h < n[a] && !upml_at(h)) ++h;
      lo[a] = std::max(lo[a], l);
      hi[a] = std::min(hi[a], h);
    }
  }
  for (int a = 0; a < 3; ++a)
    if (lo[a] >= hi[a]) return;
  for (int c = 0; c < 6; ++c) {
    const int64_t* n = s->shape[c];
    const std::vector<uint16_t>& ids = s->host_ids[c];
    std::vector<char> upml(s->recs.size());
    for (size_t r = 0; r < upml.size(); ++r) upml[r] = s->recs[r].cls == GMES_CLS_UPML;
    for (int64_t i = lo[0]; i < std::min(hi[0], n[0]); ++i)
      for (int64_t j = lo[1]; j < std::min(hi[1], n[1]); ++j)
        for (int64_t k = lo[2]; k < std::min(hi[2], n[2]); ++k)
          if (upml[ids[(i * n[1] + j) * n[2] + k]]) return;
  }
  for (int a = 0; a < 3; ++a) box[a] = (int32_t)(lo[a] | (hi[a] << 16));
}

// The coordinates lo | hi << 16 along an axis where the CPML rows that E (or
// H) components read there have no live state: c = 0 on the longest run.
// (The H rows of the two components are read at storage index i + 1, up to
// the last one.)
int32_t sweep_dead_run(const gmes_sim* s, bool electric, int axis) {
  const int c = (electric ? 0 : 3) + (axis == 0 ? 1 : 0);  // a component with that curl axis
  const std::vector<double>& v = s->prof_host[0][c][axis];
  if (s->prof_w[0][c][axis] != 3 || v.empty()) return 0;
  const int len = (int)(v.size() / 3);
  int lo = 0, hi = 0;
  for (int q = 0; q < len;) {
    if (v[3 * (size_t)q + 1] != 0.0) { ++q; continue; }
    int e = q;
    while (e < len && v[3 * (size_t)e + 1] == 0.0) ++e;
    if (e - q > hi - lo) { lo = q; hi = e; }
    q = e;
  }
  return hi > 0x7FFF ? 0 : lo | (hi << 16);
}

// Whether every cell with live CPML state is a CPML cell (or a flagged one):
// the sweep takes the update from the coordinate.
bool sweep_live_cells_cpml(const gmes_sim* s) {
  std::vector<char> ok(s->recs.size());
  for (size_t r = 0; r < ok.size(); ++r) {
    const int cls = s->recs[r].cls;
    ok[r] = cls == GMES_CLS_CPML || cls == GMES_CLS_DUMMY || cls == GMES_CLS_CONST;
  }
  std::atomic<bool> all{true};
  host_parallel(12, s->ncell[0], [&](int q) {
    const int c = q / 2, a = q % 2 ? kAx2[c] : kAx1[c];
    const int64_t* n = s->shape[c];
    const int run = c < 3 ? s->sweep_run_e[a] : s->sweep_run_h[a], lo = run & 0xFFFF, hi = run >> 16;
    int64_t ix[3];
    for (ix[0] = 0; ix[0] < n[0] && all; ++ix[0]) {
      if (a == 0 && ix[0] >= lo && ix[0] < hi) continue;
      for (ix[1] = 0; ix[1] < n[1]; ++ix[1]) {
        if (a == 1 && ix[1] >= lo && ix[1] < hi) continue;
        const uint16_t* row = s->host_ids[c].data() + (ix[0] * n[1] + ix[1]) * n[2];
        for (int64_t k = 0; k < n[2]; ++k) {
          if (a == 2 && k >= lo && k < hi) { k = hi - 1; continue; }
          if (!ok[row[k]]) all = false;
        }
      }
    }
  });
  return all;
}

// The distinct triples of records of the cells one thread owns, of one field
// type; entries[id] are the record ids of a triple's three components.
// False when there are more than `most`.
bool sweep_triples(const gmes_sim* s, bool electric, size_t most, std::vector<std::array<uint16_t, 3>>& entries) {
  const int c0 = electric ? 0 : 3;
  const int64_t nx = s->g.nx, ny = s->g.ny, nz = s->g.nz;
  constexpr int kParts = 16;
  std::vector<uint64_t> found[kParts];  // in the order of the cells
  host_parallel(kParts, s->ncell[0], [&](int part) {
    std::unordered_set<uint64_t> seen;
    uint64_t last = ~0ull;
    const uint16_t* src[3];
    for (int64_t i = nx * part / kParts; i < nx * (part + 1) / kParts; ++i)
      for (int64_t j = 0; j < ny; ++j) {
        for (int t = 0; t < 3; ++t) {
          const int64_t* n = s->shape[c0 + t];
          // H cells sit one up along the axes across their own
          const int64_t ii = i + (!electric && t != 0), jj = j + (!electric && t != 1), kk = !electric && t != 2;
          src[t] = s->host_ids[c0 + t].data() + (ii * n[1] + jj) * n[2] + kk;
        }
        for (int64_t k = 0; k < nz; ++k) {
          const uint64_t key = step_key(src[0][k], src[1][k], src[2][k]);
          if (key == last) continue;
          last = key;
          if (seen.size() <= most && seen.insert(key).second) found[part].push_back(key);
        }
      }
  });
  std::unordered_set<uint64_t> seen;
  for (const auto& part : found)
    for (const uint64_t key : part) {
      if (!seen.insert(key).second) continue;
      if (entries.size() >= most) return false;
      entries.push_back({(uint16_t)key, (uint16_t)(key >> 16), (uint16_t)(key >> 32)});
    }
  return true;
}

// Writes the entry ids of every cell on the device, from the material ids
// there and hash tables of the triples (building them on the host and
// copying them took 40 ms at 256^3).
std::vector<StepKey> sweep_keys(const std::vector<std::array<uint16_t, 3>>& ent) {
  size_t cap = 64;
  while (cap < 4 * ent.size()) cap *= 2;
  std::vector<StepKey> tab(cap, StepKey{~0ull, 0});
  for (size_t e = 0; e < ent.size(); ++e) {
    const uint64_t key = step_key(ent[e][0], ent[e][1], ent[e][2]);
    uint32_t at = step_hash(key, (uint32_t)cap - 1);
    while (tab[at].key != ~0ull) at = (at + 1) & ((uint32_t)cap - 1);
    tab[at] = StepKey{key, (uint64_t)e};
  }
  return tab;
}

int sweep_ids(gmes_sim* s, const std::vector<StepKey> (&tab)[2], char* d) {
  StepIdArgs a{};
  for (int c = 0; c < 6; ++c) {
    a.ids[c] = s->ids[c];
    a.first[c] = dev_index(s, c, c >= 3 && c != 3, c >= 3 && c != 4, c >= 3 && c != 5);
    a.plane[c] = s->pi[c];
    a.row[c] = s->pitch[c];
  }
  a.n[0] = s->g.nx; a.n[1] = s->g.ny; a.n[2] = s->g.nz;
  a.pitch = s->pitch[0];
  a.types = 2;
  a.shift = s->step_eb;
  if (s->step_idw == 2) a.out16 = static_cast<uint16_t*>(s->d_step_ids);
  else a.out = static_cast<uint32_t*>(s->d_step_ids);
  const size_t b0 = tab[0].size() * sizeof(StepKey), b1 = tab[1].size() * sizeof(StepKey);
  HIP_TRY(hipMemcpy(d, tab[0].data(), b0, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(d + b0, tab[1].data(), b1, hipMemcpyHostToDevice));
  for (int h = 0; h < 2; ++h) {
    a.tab[h] = reinterpret_cast<const StepKey*>(d + (h ? b0 : 0));
    a.mask[h] = (uint32_t)tab[h].size() - 1;
  }
  launch_step_ids(a, s->stream);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(s->stream));
  return GMES_OK;
}

template <class R>
void sweep_entry(const gmes_sim* s, const std::array<uint16_t, 3>& rec, StepEnt<R>& e, StepRare rare[3]) {
  e = StepEnt<R>{};
  for (int t = 0; t < 3; ++t) {
    const gmes_mat_rec& r = s->recs[rec[t]];
    const bool upml = r.cls == GMES_CLS_UPML;
    rare[t] = StepRare{r.cls == GMES_CLS_DUMMY ? 1 : r.cls == GMES_CLS_CONST ? 2 : 0, -1, GMES_SRC_SET, 0,
                       r.value[0], r.value[1]};
    if (r.cls >= GMES_CLS_DRUDE) e.c[t] = 0;  // keeps its value: see stepfix.hip
    else if (rare[t].keep) e.meta |= kStepRareCell;
    else e.c[t] = upml ? (s->fp64 ? (R)r.eps_mu : (R)(1.0 / r.eps_mu)) : (R)(s->g.dt / r.eps_mu);
    if (upml || r.cls == GMES_CLS_CPML) e.meta |= 2u << t;
  }
}

// CPML with live state along x or y: blocks without it take a body without
// those words, blocks with one of the two a body that loads its words a plane
// ahead, in one launch; from 5 MB a component (us per step, one body for all
// against this: 96^3 FP32 26.6, 34; 112^3 39, 36; 256^3 293, 255; FP64 80^3
// 31, 35; 96^3 58, 50; 160^3 177, 153; 171 x 150 x 139 153, 145).  Few planes
// per block: a plane takes its loads' latency, which only more blocks hide
// (256^3, planes of blocks with and without x or y words: 6 and 9 255, 16 and
// 29 259, 24 and 39 277; 128^3 6 and 9 49, 16 and 29 61).
constexpr int64_t kSweepSplitBytes = 5 << 20;
constexpr int kSweepOuterPlanes = 6, kSweepInnerPlanes = 9;

// Whole rows that have to fit a block, so that the rim row, whose E it computes
// again, is worth it (it may take fewer, three at least: 181 x 203 x 225 FP32 UPML
// 168 us with three, 238 with four): three; with UPML, or in complex sims CPML along x or y, whose
// bodies hold few waves, five of 8-byte words and four of 4-byte ones, unless
// the launches bound the two-kernel step (us per step, that one against this:
// complex FP32 CPML 120 x 30 x 200 46, 58; 160^3 163, 168; 144^3, five rows,
// 122, 116; UPML 160^3 FP64 182, 215; 144^3 136, 138; 96 x 96 x 256 FP64 106,
// 119; FP32, three rows, 160 x 200 x 310 221, 240; 40 x 40 x 341 28, 23; FP64
// CPML 96 x 96 x 256 118, 99).
constexpr int64_t kSweepLongBytes = 4 << 20;
int sweep_min_rows(const gmes_sim* s, int absorber) {
  if (s->ncell[0] * s->esize < kSweepLongBytes || absorber == kPmlNone || absorber == kPmlZ) return kSweepMinRows;
  if (absorber == kUpml) return s->esize == 8 ? 5 : 4;
  return s->complex_ ? 5 : kSweepMinRows;
}

// The launches of a step.  A block's march costs its planes and two more (the
// rim plane, the prologue); blocks run in rounds over the 256 CUs, a last
// incomplete round costing about half of one; a CU with few waves still pays
// the latency of a plane (kSweepFloor).  256^3 CPML, rows of 256, blocks of 3
// rows: 64 planes (one full round) 285 us, 32 planes 303, 16 planes 312; 181 x
// 203 x 225 UPML: 3 rows 190 us, 4 rows (one block per CU) 204.
//
// Rows and planes per block of a launch over ni planes of nj rows; returns its
// cost (0: no shape fits).
template <class T>
double sweep_shape(const gmes_sim* s, int nent, int absorber, int ni, int nj, gmes_sim::SweepPart& part, int& ch_out) {
  const int nz = s->g.nz;
  double best = 0;
  part.absorber = absorber;
  if (sweep_min_rows(s, absorber) * nz > step3_max_threads<T>(absorber)) return 0;
  for (int rows = kSweepMinRows; rows <= nj + 1; ++rows) {
    const int threads = (rows * nz + 63) / 64 * 64, most = step3_max_threads<T>(absorber);
    if (threads > most) break;
    const int64_t lds = (int64_t)step3_lds<T>(threads, nent, rows, nz, absorber);
    if (lds > kSweepLds) break;
    // waves a CU holds: registers (see StepWaves)
    const bool full = absorber != kPmlNone && absorber != kPmlZ;
    const int waves = threads / 64, held = sizeof(T) == 4 ? (absorber ? 24 : 32) : full ? 12 : absorber ? 16 : 20;
    const int per_cu = std::max<int>(1, (int)std::min<int64_t>(held / waves, kSweepLds / lds));
    const int tiles = (nj + rows - 2) / (rows - 1);
    const double plane = std::max(per_cu * waves, kSweepFloor);
    for (int nch = 1; nch <= ni; ++nch) {
      const int ch = (ni + nch - 1) / nch;
      const double x = (double)tiles * ((ni + ch - 1) / ch) / (256.0 * per_cu);
      const double rounds = x <= 1 ? 1 : x + (std::ceil(x) > x ? 0.5 : 0);
      const double cost = rounds * (ch + 2.0) * plane;
      if (best == 0 || cost < best * 0.999) {
        best = cost;
        part.rows = rows;
        part.threads = threads;
        ch_out = ch;
      }
    }
  }
  return best;
}

// The longest run of thread coordinates along axis a (0 x, 1 y), n of them,
// whose E, H and the E after the last have no live CPML state: lo, hi.
void sweep_quiet(const gmes_sim* s, int a, int n, int& lo, int& hi) {
  const int re = s->sweep_run_e[a], rh = s->sweep_run_h[a];
  auto dead_e = [&](int q) { q = q == n ? 0 : q; return q >= (re & 0xFFFF) && q < (re >> 16); };
  auto dead_h = [&](int q) { return q + 1 >= (rh & 0xFFFF) && q + 1 < (rh >> 16); };  // storage index
  lo = hi = 0;
  for (int q = 0; q < n;) {
    if (!dead_e(q) || !dead_h(q)) { ++q; continue; }
    int e = q;
    while (e < n && dead_e(e) && dead_h(e)) ++e;
    while (e > q && !dead_e(e)) --e;
    if (e - q > hi - lo) { lo = q; hi = e; }
    q = std::max(e, q + 1);
  }
}

void sweep_rect(gmes_sim::SweepPart& part, int i0, int i1, int j0, int j1, int most, int kind) {
  if (i0 >= i1 || j0 >= j1) return;
  const int len = i1 - i0, n = (len + most - 1) / most;
  const int r[6] = {i0, i1, j0, j1, (len + n - 1) / n, kind};
  std::copy(r, r + 6, part.rect[part.nrect++]);
}

// Blocks by their CPML words; [ia, ib) x [ja, jb) has none along x and y.
void sweep_rects(gmes_sim::SweepPart& part, int nx, int ny, int ia, int ib, int ja, int jb, int out, int in) {
  const int xs[4] = {0, ia, ib, nx}, ys[4] = {0, ja, jb, ny};
  for (int x : {0, 2})
    for (int y : {0, 2}) sweep_rect(part, xs[x], xs[x + 1], ys[y], ys[y + 1], out, kPmlXYZ);
  for (int x : {0, 2}) sweep_rect(part, xs[x], xs[x + 1], ja, jb, out, kPmlXZ);
  for (int y : {0, 2}) sweep_rect(part, ia, ib, ys[y], ys[y + 1], out, kPmlYZ);
  sweep_rect(part, ia, ib, ja, jb, in, kPmlZ);
}

// The shape of a member of a batch: blocks of one size for all, and at most ch
// planes.  lean: as step3_batch_threads has it.
bool sweep_lean(const gmes_sim* s, int& ia, int& ib, int& ja, int& jb) {
  ia = ib = ja = jb = 0;
  if (s->sweep_absorber == kPmlXYZ) {
    sweep_quiet(s, 0, s->g.nx, ia, ib);
    sweep_quiet(s, 1, s->g.ny, ja, jb);
  }
  return s->sweep_absorber == kPmlNone || (ib - ia == s->g.nx && jb - ja == s->g.ny);
}

bool sweep_batch_part(const gmes_sim* s, gmes_sim::SweepPart& part, bool& lean, int ch) {
  const int nx = s->g.nx, ny = s->g.ny, nz = s->g.nz;
  int ia, ib, ja, jb;
  lean = sweep_lean(s, ia, ib, ja, jb);
  part = gmes_sim::SweepPart{};
  part.threads = s->esize == 8 ? step3_batch_threads<double>(lean) : step3_batch_threads<float>(lean);
  part.rows = std::min(part.threads / nz, ny + 1);
  if (part.rows < kSweepMinRows) return false;
  part.absorber = s->sweep_absorber;
  if (lean) sweep_rect(part, 0, nx, 0, ny, ch, s->sweep_absorber ? kPmlZ : kPmlNone);
  else if (ib > ia && jb > ja) sweep_rects(part, nx, ny, ia, ib, ja, jb, std::min(ch, kSweepOuterPlanes), ch);
  else sweep_rect(part, 0, nx, 0, ny, ch, s->sweep_absorber);
  return true;
}

template <class T>
void sweep_plan_t(gmes_sim* s, int nent) {
  const int nx = s->g.nx, ny = s->g.ny;
  gmes_sim::SweepPart& part = s->sweep_part;
  part = gmes_sim::SweepPart{};
  int ia = 0, ib = 0, ja = 0, jb = 0, ch = 0, kind = s->sweep_absorber;
  if (kind == 1) {
    sweep_quiet(s, 0, nx, ia, ib);
    sweep_quiet(s, 1, ny, ja, jb);
    if (ib - ia == nx && jb - ja == ny) kind = kPmlZ;
    else if (s->ncell[0] * s->esize >= kSweepSplitBytes && ib > ia && jb > ja) kind = kPmlMixed;
  }
  if (sweep_shape<T>(s, nent, kind, nx, ny, part, ch) == 0) {
    part.rows = 0;
    return;
  }
  if (kind != kPmlMixed) {
    sweep_rect(part, 0, nx, 0, ny, ch, kind);
    return;
  }
  sweep_rects(part, nx, ny, ia, ib, ja, jb, kSweepOuterPlanes, kSweepInnerPlanes);
}

void sweep_plan(gmes_sim* s) {
  const int nent = (int)(s->step_e.size() + s->step_h.size()) + 2 * kSweepMaxSrc;
  switch (s->g.dtype) {
    case GMES_F32: sweep_plan_t<float>(s, nent); break;
    case GMES_F64: sweep_plan_t<double>(s, nent); break;
    default: sweep_plan_t<cplx<float>>(s, nent); break;
  }
}

void fix_release(gmes_sim* s) {
  dev_free(s, s->d_fix_items, (size_t)s->fix_bytes);
  s->sweep_bytes -= s->fix_bytes;
  s->d_fix_items = nullptr;
  s->fix_bytes = 0;
}

void sweep_swap(gmes_sim* s);

// Gives back what one-sweep steps hold (the device is idle as far as s goes).
// After an odd number of them the current buffers are the ones to be given back:
// keep: their contents move to the sim's own.
void sweep_release(gmes_sim* s, bool keep = true) {
  if (s->sweep_mem && s->par != s->sweep_par0) {
    auto move = [&](void* to, const void* from, size_t bytes) {
      if (keep && to) (void)hipMemcpyAsync(to, from, bytes, hipMemcpyDeviceToDevice, s->stream);
    };
    for (int c = 0; c < 6; ++c) {
      const size_t b = (size_t)s->dsize[c] * s->esize;
      move(s->f_alt[c], s->f[c], b);
      if (c >= 3) continue;
      move(s->pml_alt[c], s->pml_state[c], (s->has_cls[c][GMES_CLS_CPML] ? 2 : 1) * b);
      for (int k = 0; k < GMES_NCLS; ++k) {
        const AdeList& L = s->ade[c][k];
        move(s->ade_alt[c][k], L.state, (size_t)L.nstate * L.n * ade_word(s, k));
      }
    }
    if (keep) (void)hipStreamSynchronize(s->stream);
    sweep_swap(s);
  }
  s->clk_stale = true;  // Ctl::clk is by parity
  if (s->sweep_mem) (void)dev_release(s->sweep_mem);
  s->sweep_mem = nullptr;
  for (void*& p : s->f_alt) p = nullptr;
  for (int c = 0; c < 3; ++c) {
    s->pml_alt[c] = nullptr;
    s->d_adeq[c] = nullptr;
    for (void*& p : s->ade_alt[c]) p = nullptr;
  }
  s->d_step_ids = s->d_step_tab = nullptr;
  s->d_rare = nullptr;
  fix_release(s);
  s->sweep_fix = false;
  s->sweep_1d = s->sweep_2d = false;
  s->bytes -= s->sweep_bytes;
  s->sweep_bytes = 0;
  s->sweep_ok = false;
  s->step_tab_cap = 0;
}

// What one-sweep steps hold, in one allocation (a dozen of them took 1 ms of
// setting up a small sim): parts to be cleared, the others.
struct SweepParts {
  struct Part {
    void** p;
    size_t bytes;
  };
  std::vector<Part> cleared, other;
  // E state of component c: its CPML or UPML words
  void state(gmes_sim* s, int c) {
    if (s->pml_state[c])
      cleared.push_back({&s->pml_alt[c], (size_t)(s->has_cls[c][GMES_CLS_CPML] ? 2 : 1) * s->dsize[c] * s->esize});
  }
  // and that of its dispersive cells, with their places in the lists
  void ade(gmes_sim* s, int c) {
    bool any = false;
    for (int k = GMES_CLS_DRUDE; k < GMES_CLS_DM2; ++k) {
      const AdeList& L = s->ade[c][k];
      if (!L.n) continue;
      any = true;
      cleared.push_back({&s->ade_alt[c][k], (size_t)L.nstate * L.n * ade_word(s, k)});
    }
    if (any) other.push_back({(void**)&s->d_adeq[c], (size_t)s->dsize[c] * sizeof(int32_t)});
  }
};

// (plain hipMalloc: a sim that finds no room does without)
int sweep_take(gmes_sim* s, const SweepParts& v) {
  auto up = [](size_t b) { return (std::max<size_t>(b, 1) + kSweepAlign - 1) / kSweepAlign * kSweepAlign; };
  size_t zero = 0, total = 0;
  for (const auto& x : v.cleared) zero += up(x.bytes);
  for (const auto& x : v.other) total += up(x.bytes);
  total += zero;
  HIP_TRY(hipMalloc(&s->sweep_mem, total));
  s->bytes += (int64_t)total;
  s->sweep_bytes += (int64_t)total;
  s->sweep_par0 = s->par;
  char* d = static_cast<char*>(s->sweep_mem);
  for (const auto* list : {&v.cleared, &v.other})
    for (const auto& x : *list) {
      *x.p = d;
      d += up(x.bytes);
    }
  if (zero) HIP_TRY(hipMemsetAsync(s->sweep_mem, 0, zero, s->stream));
  return GMES_OK;
}

// Every sim, for sweep_reclaim.
std::mutex g_sims_mu;
std::unordered_set<gmes_sim*> g_sims;
void known_sim(gmes_sim* s, bool there) {
  std::lock_guard<std::mutex> lk(g_sims_mu);
  if (there) g_sims.insert(s);
  else g_sims.erase(s);
}

// Releases the second buffers of every sim on a device, with no other thread
// inside the engine: between two calls, and where a call has let go of its
// hold (it captures a graph, or is here itself), the current buffers hold the
// whole state, and the two-kernel step goes on from there.
void sweep_reclaim(int device) {
  std::lock_guard<std::mutex> lk(g_sims_mu);
  for (gmes_sim* s : g_sims) {
    if (s->device != device || s->sweep_bytes == 0) continue;
    (void)sync_exec(s);
    destroy_graph(s);
    sweep_release(s);
  }
}

// Whether the second buffers of s leave the device at least half empty: sims
// that fill it keep the two-kernel step, and other users of the device find
// room (the engine's own sims take it from here when there is none left, see
// sweep_reclaim).  Lines and small planes take them on a fuller device too: at
// most 1/256 of what is idle each, so never all of it.  Held until they are
// allocated: sims set up at once count each other's.
std::mutex g_room_mu;
bool sweep_room(const gmes_sim* s) {
  int64_t need = (int64_t)s->g.nx * s->g.ny * s->g.nz * 4;
  for (int c = 0; c < 6; ++c) {
    if (!active(s, c)) continue;
    need += s->dsize[c] * s->esize;
    if (c < 3 && s->pml_state[c]) need += (s->has_cls[c][GMES_CLS_CPML] ? 2 : 1) * s->dsize[c] * s->esize;
  }
  size_t idle = 0, total = 0;
  if (hipMemGetInfo(&idle, &total) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return (int64_t)idle - need >= (int64_t)(total / 2) || need <= (int64_t)(idle / 256);
}

// Uploads the entry tables, those of source cells (after the step_net /
// step_nht plain ones) included.
template <class R>
int sweep_upload_tab(gmes_sim* s, const std::vector<std::array<int, 3>>& se, const std::vector<std::array<int, 3>>& sh) {
  // se, sh: (base entry, component 0..2, op index) of each source cell
  const int net = (int)(s->step_e.size() + se.size()), nht = (int)(s->step_h.size() + sh.size());
  std::vector<StepEnt<R>> tab((size_t)(net + nht));
  std::vector<StepRare> rare((size_t)(net + nht) * 3);
  for (size_t e = 0; e < s->step_e.size(); ++e) sweep_entry<R>(s, s->step_e[e], tab[e], &rare[3 * e]);
  for (size_t e = 0; e < s->step_h.size(); ++e) sweep_entry<R>(s, s->step_h[e], tab[net + e], &rare[3 * (net + e)]);
  for (int h = 0; h < 2; ++h) {
    const auto& src = h ? sh : se;
    const size_t base = h ? (size_t)net : 0, first = h ? (size_t)net + s->step_h.size() : s->step_e.size();
    for (size_t q = 0; q < src.size(); ++q) {
      const gmes_src_op& o = s->ops[src[q][2]];
      const size_t d = first + q, b = base + src[q][0];
      tab[d] = tab[b];
      for (int t = 0; t < 3; ++t) rare[3 * d + t] = rare[3 * b + t];
      tab[d].meta |= kStepRareCell;
      rare[3 * d + src[q][1]].wave = o.wave;
      rare[3 * d + src[q][1]].kind = o.kind;
    }
  }
  HIP_TRY(hipMemcpy(s->d_step_tab, tab.data(), tab.size() * sizeof(StepEnt<R>), hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(s->d_rare, rare.data(), rare.size() * sizeof(StepRare), hipMemcpyHostToDevice));
  s->step_net = net;
  s->step_nht = nht;
  return GMES_OK;
}

// ---- one-sweep steps of TEM lines (step1d.hip)
//
// Taken when every absorber cell is of one kind and one profile set, in both
// components or none, CPML has no live state along the collapsed axes, no cell
// is of the DM2 class, and for sources and probes what the 2-D modes ask.
// Direction e of the E component of a line of components e and e + 1 along
// axis e + 2; -1: not such a line.
int line_dir(const gmes_sim* s) {
  const int64_t n[3] = {s->g.nx, s->g.ny, s->g.nz};
  for (int e = 0; e < 3; ++e) {
    const int h = (e + 1) % 3, l = (e + 2) % 3;
    if (s->g.active == ((1u << e) | (8u << h)) && n[e] == 1 && n[h] == 1 && n[l] > 1) return e;
  }
  return -1;
}
int64_t stride_of(const gmes_sim* s, int c, int axis) {
  return axis == 0 ? s->pi[c] : axis == 1 ? s->pitch[c] : s->pk[c];
}

int sweep1_build(gmes_sim* s) {
  const int e = line_dir(s), comp[2] = {e, 3 + (e + 1) % 3}, line = (e + 2) % 3;
  if (s->naux) return GMES_OK;
  bool cpml = false, upml = false;
  for (const int c : comp) {
    cpml |= s->has_cls[c][GMES_CLS_CPML];
    upml |= s->has_cls[c][GMES_CLS_UPML];
    if (s->has_cls[c][GMES_CLS_DM2]) return GMES_OK;
  }
  if ((cpml && upml) || ((cpml || upml) && s->nprof != 1)) return GMES_OK;
  s->sweep_absorber = cpml ? 1 : upml ? 2 : 0;
  for (const int c : comp) {
    if (!s->sweep_absorber) break;
    if (!s->pml_state[c]) return GMES_OK;
    for (int a = 0; a < 3; ++a) {
      const std::vector<double>& v = s->prof_host[0][c][a];
      const int w = cpml ? 3 : 6;
      if (s->prof_w[0][c][a] != w || (int64_t)v.size() != s->shape[c][a] * w) return GMES_OK;
      for (size_t q = 1; cpml && a != line && q < v.size(); q += 3)
        if (v[q] != 0.0) return GMES_OK;
    }
  }
  std::unique_lock<std::mutex> room(g_room_mu);
  if (!sweep_room(s)) return GMES_OK;
  SweepParts parts;
  for (const int c : comp) parts.other.push_back({&s->f_alt[c], (size_t)s->dsize[c] * s->esize});
  parts.state(s, e);
  parts.ade(s, e);
  const int rc = sweep_take(s, parts);
  room.unlock();
  if (rc) {
    (void)hipGetLastError();
    sweep_release(s);
    return GMES_OK;
  }
  for (int k = GMES_CLS_DRUDE; k < GMES_CLS_DM2; ++k) {
    const AdeList& L = s->ade[e][k];
    if (L.n)
      launch_list_places({L.cell, (int)L.n, (int)s->shape[e][1], (int)s->shape[e][2], s->pi[e], s->pitch[e], s->pk[e],
                          s->d_adeq[e] + (kPad - s->koff[e])}, s->stream);
  }
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(s->stream));
  s->sweep_1d = true;
  s->sweep_ok = true;
  return GMES_OK;
}

int sweep1_sources(gmes_sim* s) {
  const int e = line_dir(s), line = (e + 2) % 3;
  s->step2_src.clear();
  s->sweep_src_ok = (int)s->ops.size() <= kStep2Src;
  const int64_t n[3] = {s->g.nx, s->g.ny, s->g.nz};
  for (const gmes_src_op& o : s->ops) {
    const int64_t sy = s->shape[o.comp][1], sz = s->shape[o.comp][2];
    const int64_t ix[3] = {o.cell / (sy * sz), (o.cell / sz) % sy, o.cell % sz};
    int64_t q = 0;
    if (o.kind != GMES_SRC_SET && o.kind != GMES_SRC_SUB) s->sweep_src_ok = false;
    for (int a = 0; a < 3; ++a) {
      const int64_t x = ix[a] - (o.comp >= 3 && a != o.comp - 3);
      if (x < 0 || x >= n[a]) s->sweep_src_ok = false;  // a ghost cell
      if (a == line) q = x;
    }
    s->step2_src.push_back({o.comp >= 3, (int)q, 0, o.wave, o.kind});
  }
  return GMES_OK;
}

template <class T>
Step1Args<T> step1_args(const gmes_sim* s) {
  using R = typename real_of<T>::type;
  Step1Args<T> m{};
  const int e = line_dir(s), hd = (e + 1) % 3, line = (e + 2) % 3, comp[2] = {e, 3 + hd};
  const int w = s->sweep_absorber == 1 ? 3 : 6;
  for (int f = 0; f < 2; ++f) {
    const int c = comp[f], collapsed = f ? e : hd;
    int64_t x[3] = {0, 0, 0};  // storage of cell 0
    if (f) x[collapsed] = x[line] = 1;
    const int64_t o = dev_index(s, c, x[0], x[1], x[2]);
    m.fi[f] = static_cast<const T*>(s->f[c]) + o;
    m.fo[f] = static_cast<T*>(s->f_alt[c]) + o;
    m.st[f] = (int)stride_of(s, c, line);
    m.gc[f] = (f ? -1 : 1) * stride_of(s, c, collapsed);
    m.ids[f] = s->ids[c] + o;
    if (s->sweep_absorber) {
      // CPML: E's line is its second curl axis, H's its first
      const int64_t word = s->sweep_absorber == 1 && f == 0 ? s->dsize[c] : 0;
      m.si[f] = static_cast<const T*>(s->pml_state[c]) + o + word;
      m.so[f] = static_cast<T*>(f ? s->pml_state[c] : s->pml_alt[c]) + o + word;
      const int axes[3] = {kAx1[c], kAx2[c], c % 3};
      for (int a = 0; a < 3; ++a)
        m.row[f][a] = static_cast<const R*>(s->d_prof) + s->prof_off0[c][axes[a]] + x[axes[a]] * w;
    }
    m.ph[f][0] = cplx<R>{(R)s->g.phase[c][collapsed][0], (R)s->g.phase[c][collapsed][1]};
    m.ph[f][1] = cplx<R>{(R)s->g.phase[c][line][0], (R)s->g.phase[c][line][1]};
  }
  const double d[3] = {s->g.dx, s->g.dy, s->g.dz};
  const int axes[3] = {e, hd, line};
  for (int a = 0; a < 3; ++a) {
    m.d[a] = (R)d[axes[a]];
    m.inv_d[a] = (R)(1.0 / d[axes[a]]);
  }
  const int64_t n[3] = {s->g.nx, s->g.ny, s->g.nz};
  m.n = (int)n[line];
  m.recs = static_cast<const DevRec<R>*>(s->d_recs);
  m.coef = static_cast<const R*>(s->d_coef);
  if (s->d_adeq[e]) m.adeq = s->d_adeq[e] + dev_index(s, e, 0, 0, 0);
  for (int k = 0; k < 3; ++k) {
    m.ade_in[k] = s->ade[e][GMES_CLS_DRUDE + k].state;
    m.ade_out[k] = s->ade_alt[e][GMES_CLS_DRUDE + k];
    m.ade_n[k] = (int)s->ade[e][GMES_CLS_DRUDE + k].n;
  }
  m.nsrc = (int)s->step2_src.size();
  for (int q = 0; q < m.nsrc; ++q) {
    const auto& v = s->step2_src[q];
    m.src[q] = {v[0], v[1], v[3], v[4]};
  }
  m.waves = s->d_waves;
  m.ctl = reinterpret_cast<Ctl*>(s->d_clock);
  m.par = s->par;
  // the operations of a parent may sample ghost cells
  m.ghosts = s->sweep_ghosts || s->parent;
  m.absorber = s->sweep_absorber;
  return m;
}

// ---- one-sweep steps of collapsed-z 2-D modes (step2d.hip)
//
// Taken when
//   * all absorber cells are of one kind and one profile set, in every
//     component or none, and CPML has no live state along z,
//   * no cell is of the DM2 class,
//   * the distinct triples of records fit a block's LDS (kSweepMaxTab) and a
//     component 4 GiB (32-bit byte offsets),
//   * every source is a point operation off the ghost planes, at most
//     kStep2Src of them, and no E probe sits on a ghost plane, and
//   * the caller asked for no tile and did not turn ghost fusion off.
bool step2_tm(const gmes_sim* s) { return active(s, 2); }
// component of direction a of the mode
int step2_comp(const gmes_sim* s, int a) { return step2_tm(s) ? (a == 2 ? 2 : 3 + a) : (a == 2 ? 5 : a); }
// storage coordinate along axis x of thread coordinate 0
int step2_first(int c, int x) { return c >= 3 && c - 3 != x; }

// Columns per block and rows per block.  Whole rows up to 512 columns;
// longer ones in stretches of 224 columns (whole lines of 128 bytes; 226
// lanes of 256), which beat 448 (1200^2 FP32 14.2 against 14.9 us) and whole
// rows of 640 (7.5 against 8.2).  Rows: a block pays one more than it owns,
// and fewer, longer blocks leave the last ones running alone: the best
// count grew with the square root of the tiles per CU (us per step at 1, 2,
// 3, 4, 6 rows: 640^2 FP32 8.6, 7.5, 8.4; 1200^2 FP32 18.6, 15.2, 14.2,
// 15.5, 14.5; 2048^2 FP32 5 rows 30.3, 4 31.7, 10 33.2; 300^2 5.6, 6.8;
// 512^2 complex FP64 7.7, 6.2, 7.1).
void sweep2_shape(gmes_sim* s) {
  const int nx = s->g.nx, ny = s->g.ny;
  s->sweep_whole = ny <= 512;
  s->sweep_w = s->sweep_whole ? ny : 224;
  const double waves = (double)nx * ((ny + s->sweep_w - 1) / s->sweep_w) * step2_threads(s->sweep_w, s->sweep_whole) / 64;
  s->sweep_ch = std::max(1, std::min(nx, (int)std::ceil(std::sqrt(waves / 4096))));
}

// Entries, their cells' details, the key table of the entry ids and the ids
// themselves are one part of a sim's second buffers, filled by one copy and one
// launch: what is copied, and where its pieces begin.
struct Sweep2Tables {
  std::vector<char> host;
  size_t cells_at, keys_at, ids_at, nkeys;
};
template <class R>
Sweep2Tables sweep2_host(const gmes_sim* s) {
  const size_t n = s->step_e.size();
  const std::vector<StepKey> keys = sweep_keys(s->step_e);
  const size_t cells_at = n * sizeof(Step2Ent<R>), keys_at = cells_at + 3 * n * sizeof(Step2Cell),
               ids_at = keys_at + keys.size() * sizeof(StepKey);
  static_assert(sizeof(Step2Ent<R>) % 16 == 0 && sizeof(Step2Cell) % 8 == 0 && sizeof(StepKey) % 16 == 0, "alignment");
  std::vector<char> host(ids_at, 0);
  Step2Ent<R>* tab = reinterpret_cast<Step2Ent<R>*>(host.data());
  Step2Cell* cells = reinterpret_cast<Step2Cell*>(host.data() + cells_at);
  for (size_t e = 0; e < n; ++e)
    for (int t = 0; t < 3; ++t) {
      const gmes_mat_rec& r = s->recs[s->step_e[e][t]];
      const bool absorber = r.cls == GMES_CLS_CPML || r.cls == GMES_CLS_UPML;
      const int kind = r.cls == GMES_CLS_DUMMY ? 1 : r.cls == GMES_CLS_CONST ? 2 : r.cls >= GMES_CLS_DRUDE ? 3 : 0;
      cells[3 * e + t] = Step2Cell{kind, s->step_e[e][t], r.value[0], r.value[1]};
      if (kind) tab[e].meta |= 2u << (2 * t);
      else if (absorber) tab[e].meta |= 1u << (2 * t);
      if (!kind)
        tab[e].c[t] = r.cls == GMES_CLS_UPML ? (s->fp64 ? (R)r.eps_mu : (R)(1.0 / r.eps_mu)) : (R)(s->g.dt / r.eps_mu);
    }
  memcpy(host.data() + keys_at, keys.data(), keys.size() * sizeof(StepKey));
  return {std::move(host), cells_at, keys_at, ids_at, keys.size()};
}

int sweep2_tables(gmes_sim* s, const Sweep2Tables& v) {
  const int64_t pi = s->pi[step2_comp(s, 0)];
  char* d = static_cast<char*>(s->d_step_tab);
  s->step2_cells = d + v.cells_at;
  s->step2_ids = reinterpret_cast<uint16_t*>(d + v.ids_at);
  HIP_TRY(hipMemcpy(d, v.host.data(), v.ids_at, hipMemcpyHostToDevice));
  StepIdArgs a{};
  for (int x = 0; x < 3; ++x) {
    const int c = step2_comp(s, x);
    a.ids[x] = s->ids[c];
    a.first[x] = dev_index(s, c, step2_first(c, 0), step2_first(c, 1), s->shape[c][2] == 2 ? step2_first(c, 2) : 0);
    a.plane[x] = s->pi[c];
  }
  a.tab[0] = reinterpret_cast<const StepKey*>(d + v.keys_at);
  a.mask[0] = (uint32_t)v.nkeys - 1;
  a.n[0] = s->g.nx; a.n[1] = 1; a.n[2] = s->g.ny;
  a.pitch = (int)pi;
  a.types = 1;
  a.out16 = s->step2_ids;
  launch_step_ids(a, s->stream);
  for (int c = 0; c < 3; ++c)
    for (int k = GMES_CLS_DRUDE; k < GMES_CLS_DM2; ++k) {
      const AdeList& L = s->ade[c][k];
      if (!L.n) continue;
      launch_list_places({L.cell, (int)L.n, (int)s->shape[c][1], (int)s->shape[c][2], s->pi[c], s->pitch[c], s->pk[c],
                          s->d_adeq[c] + (kPad - s->koff[c])}, s->stream);
    }
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(s->stream));
  return GMES_OK;
}

int sweep2_build(gmes_sim* s) {
  const int64_t nx = s->g.nx, ny = s->g.ny;
  const bool tm = step2_tm(s);
  if (s->g.nz != 1 || s->g.active != (tm ? 0x1Cu : 0x23u)) return GMES_OK;
  for (int a = 0; a < 3; ++a)  // 32-bit byte offsets
    if (s->dsize[step2_comp(s, a)] * s->esize > (int64_t)0xFFFFFFFF) return GMES_OK;
  bool cpml = false, upml = false;
  for (int a = 0; a < 3; ++a) {
    const int c = step2_comp(s, a);
    cpml |= s->has_cls[c][GMES_CLS_CPML];
    upml |= s->has_cls[c][GMES_CLS_UPML];
    if (s->has_cls[c][GMES_CLS_DM2]) return GMES_OK;
  }
  if ((cpml && upml) || ((cpml || upml) && s->nprof != 1)) return GMES_OK;
  s->sweep_absorber = cpml ? 1 : upml ? 2 : 0;
  const uint16_t* ids[3];
  for (int a = 0; a < 3; ++a) {
    const int c = step2_comp(s, a);
    if (s->sweep_absorber) {
      if (!s->pml_state[c]) return GMES_OK;
      for (int x = 0; x < 3; ++x)
        if (s->prof_w[0][c][x] != (cpml ? 3 : 6) ||
            (int64_t)s->prof_host[0][c][x].size() != s->shape[c][x] * (cpml ? 3 : 6))
          return GMES_OK;
    }
    if (cpml) {
      for (size_t q = 1; q < s->prof_host[0][c][2].size(); q += 3)
        if (s->prof_host[0][c][2][q] != 0.0) return GMES_OK;
      for (int x = 0; x < 2; ++x) {  // the longest run with c = 0
        const std::vector<double>& v = s->prof_host[0][c][x];
        const int len = (int)(v.size() / 3);
        int lo = 0, hi = 0;
        for (int q = 0; q < len;) {
          if (v[3 * (size_t)q + 1] != 0.0) { ++q; continue; }
          int e = q;
          while (e < len && v[3 * (size_t)e + 1] == 0.0) ++e;
          if (e - q > hi - lo) { lo = q; hi = e; }
          q = e;
        }
        lo = std::max(0, lo - step2_first(c, x));
        hi = std::max(0, hi - step2_first(c, x));
        s->sweep_run2[a][x] = hi > 0x7FFF ? 0 : lo | (hi << 16);
      }
    }
    // record of thread (i, j): [(i * s1 + j) * s2] from here
    ids[a] = s->host_ids[c].data() + (step2_first(c, 0) * s->shape[c][1] + step2_first(c, 1)) * s->shape[c][2] +
             (s->shape[c][2] == 2 ? step2_first(c, 2) : 0);
  }
  auto rec = [&](int a, int64_t i, int64_t j) {
    const int64_t* n = s->shape[step2_comp(s, a)];
    return ids[a][(i * n[1] + j) * n[2]];
  };
  if (upml) {
    // a box without UPML cells: the free runs through the centre, if no cell
    // inside is one
    std::vector<char> is(s->recs.size());
    for (size_t r = 0; r < is.size(); ++r) is[r] = s->recs[r].cls == GMES_CLS_UPML;
    auto at = [&](int64_t i, int64_t j) { return is[rec(0, i, j)] || is[rec(1, i, j)] || is[rec(2, i, j)]; };
    int64_t lo[2] = {nx / 2, ny / 2}, hi[2] = {nx / 2, ny / 2};
    while (lo[0] > 0 && !at(lo[0] - 1, ny / 2)) --lo[0];
    while (hi[0] < nx && !at(hi[0], ny / 2)) ++hi[0];
    while (lo[1] > 0 && !at(nx / 2, lo[1] - 1)) --lo[1];
    while (hi[1] < ny && !at(nx / 2, hi[1])) ++hi[1];
    bool free = hi[0] <= 0x7FFF && hi[1] <= 0x7FFF;
    for (int64_t i = lo[0]; free && i < hi[0]; ++i)
      for (int a = 0; a < 3; ++a) {
        const int64_t* n = s->shape[step2_comp(s, a)];
        const uint16_t* r = ids[a] + i * n[1] * n[2];
        char any = 0;
        for (int64_t j = lo[1]; j < hi[1]; ++j) any |= is[r[j * n[2]]];
        free = free && !any;
      }
    for (int x = 0; x < 2; ++x) s->sweep_run2[0][x] = free ? (int32_t)(lo[x] | (hi[x] << 16)) : 0;
  }
  auto pow2 = [](double v) { int e; return std::frexp(v, &e) == 0.5; };
  bool exact = pow2(s->g.dx) && pow2(s->g.dy) && pow2(s->g.dz);
  for (int a = 0; a < 3 && cpml; ++a)
    for (int x = 0; x < 3; ++x) {
      const std::vector<double>& v = s->prof_host[0][step2_comp(s, a)][x];
      for (size_t q = 2; q < v.size(); q += 3) exact = exact && v[q] == 1.0;
    }
  s->sweep_exact = exact;
  s->step_e.clear();
  s->step_h.clear();
  const size_t most = (size_t)kSweepMaxTab / (s->fp64 ? sizeof(Step2Ent<double>) : sizeof(Step2Ent<float>));
  std::unordered_set<uint64_t> seen;
  uint64_t last = ~0ull;
  int64_t step[3];
  for (int a = 0; a < 3; ++a) step[a] = s->shape[step2_comp(s, a)][2];
  for (int64_t i = 0; i < nx; ++i) {
    const uint16_t* r[3];
    for (int a = 0; a < 3; ++a) r[a] = ids[a] + i * s->shape[step2_comp(s, a)][1] * step[a];
    for (int64_t j = 0; j < ny; ++j) {
      const uint16_t x = r[0][j * step[0]], y = r[1][j * step[1]], z = r[2][j * step[2]];
      const uint64_t key = step_key(x, y, z);
      if (key == last) continue;
      last = key;
      if (!seen.insert(key).second) continue;
      if (s->step_e.size() >= most) return GMES_OK;
      s->step_e.push_back({x, y, z});
    }
  }
  std::unique_lock<std::mutex> room(g_room_mu);
  if (!sweep_room(s)) return GMES_OK;
  sweep2_shape(s);
  const Sweep2Tables tables = s->fp64 ? sweep2_host<double>(s) : sweep2_host<float>(s);
  SweepParts parts;
  for (int a = 0; a < 3; ++a) {
    const int c = step2_comp(s, a);
    parts.other.push_back({&s->f_alt[c], (size_t)s->dsize[c] * s->esize});
    if (c >= 3) continue;
    parts.state(s, c);
    parts.ade(s, c);
  }
  parts.other.push_back({&s->d_step_tab, tables.ids_at + (size_t)s->g.nx * s->pi[step2_comp(s, 0)] * sizeof(uint16_t)});
  int rc = sweep_take(s, parts);
  room.unlock();
  if (!rc) rc = sweep2_tables(s, tables);
  if (rc) {  // no room for a second set of buffers
    (void)hipGetLastError();
    sweep_release(s);
    return GMES_OK;
  }
  s->sweep_2d = true;
  s->sweep_ok = true;
  return GMES_OK;
}

int sweep2_sources(gmes_sim* s) {
  s->step2_src.clear();
  s->sweep_src_ok = (int)s->ops.size() <= kStep2Src;
  s->has_waves = !s->ops.empty();
  const int64_t n[3] = {s->g.nx, s->g.ny, 1};
  for (size_t q = 0; s->sweep_src_ok && q < s->ops.size(); ++q) {
    const gmes_src_op& o = s->ops[q];
    const int64_t sy = s->shape[o.comp][1], sz = s->shape[o.comp][2];
    int64_t ix[3] = {o.cell / (sy * sz), (o.cell / sz) % sy, o.cell % sz};
    bool ok = o.kind == GMES_SRC_SET || o.kind == GMES_SRC_SUB;
    for (int a = 0; a < 3; ++a) {
      if (s->shape[o.comp][a] > n[a]) ix[a] -= step2_first(o.comp, a);
      if (ix[a] < 0 || ix[a] >= n[a]) ok = false;  // a ghost cell
    }
    if (!ok) s->sweep_src_ok = false;
    s->step2_src.push_back({o.comp % 3, (int)ix[0], (int)ix[1], o.wave, o.kind});
  }
  return GMES_OK;
}

template <class T>
Step2Args<T> step2_args(const gmes_sim* s) {
  using R = typename real_of<T>::type;
  Step2Args<T> m{};
  const int width = s->sweep_absorber == 1 ? 3 : 6;
  for (int a = 0; a < 3; ++a) {
    const int c = step2_comp(s, a);
    const bool two = s->shape[c][2] == 2;
    const int64_t o = dev_index(s, c, step2_first(c, 0), step2_first(c, 1), two ? step2_first(c, 2) : 0);
    m.fi[a] = static_cast<const T*>(s->f[c]) + o;
    m.fo[a] = static_cast<T*>(s->f_alt[c]) + o;
    m.pi = s->pi[c];
    m.pk[a] = two ? (c < 3 ? (int64_t)s->pk[c] : -(int64_t)s->pk[c]) : 0;
    if (s->sweep_absorber) {
      const T* in = static_cast<const T*>(s->pml_state[c]) + o;
      T* out = static_cast<T*>(c < 3 ? s->pml_alt[c] : s->pml_state[c]) + o;
      for (int x = 0; x < 2; ++x) {
        // CPML: the first word goes with the first curl axis
        const int64_t w = s->sweep_absorber == 1 && kAx2[c] == x ? s->dsize[c] : 0;
        m.si[a][x] = in + w;
        m.so[a][x] = out + w;
      }
      for (int x = 0; x < 3; ++x)
        m.row[a][x] = static_cast<const R*>(s->d_prof) + s->prof_off0[c][x] +
                      (s->shape[c][x] > (x == 2 ? 1 : 0) ? step2_first(c, x) * width : 0);
    }
    for (int x = 0; x < 2; ++x) m.run[a][x] = s->sweep_run2[a][x];
    for (int x = 0; x < 3; ++x) m.ph[a][x] = cplx<R>{(R)s->g.phase[c][x][0], (R)s->g.phase[c][x][1]};
    if (c < 3) {
      m.adeq[a] = s->d_adeq[c] ? s->d_adeq[c] + o : nullptr;
      for (int k = 0; k < 3; ++k) {
        m.ade_in[a][k] = s->ade[c][GMES_CLS_DRUDE + k].state;
        m.ade_out[a][k] = s->ade_alt[c][GMES_CLS_DRUDE + k];
        m.ade_n[a][k] = (int)s->ade[c][GMES_CLS_DRUDE + k].n;
      }
    }
  }
  m.ids = s->step2_ids;
  m.n[0] = s->g.nx; m.n[1] = s->g.ny;
  m.tab = static_cast<const Step2Ent<R>*>(s->d_step_tab);
  m.cells = static_cast<const Step2Cell*>(s->step2_cells);
  m.nent = (int)s->step_e.size();
  m.d[0] = (R)s->g.dx; m.d[1] = (R)s->g.dy; m.d[2] = (R)s->g.dz;
  m.inv_d[0] = (R)(1.0 / s->g.dx); m.inv_d[1] = (R)(1.0 / s->g.dy); m.inv_d[2] = (R)(1.0 / s->g.dz);
  m.recs = static_cast<const DevRec<R>*>(s->d_recs);
  m.coef = static_cast<const R*>(s->d_coef);
  m.nsrc = (int)s->step2_src.size();
  for (int q = 0; q < m.nsrc; ++q) {
    const auto& v = s->step2_src[q];
    m.src[q] = {v[0], v[1], v[2], v[3], v[4]};
  }
  m.w = s->sweep_w;
  m.whole = s->sweep_whole;
  m.ch = s->sweep_ch;
  m.nj = (s->g.ny + m.w - 1) / m.w;
  m.nblk = m.nj * ((s->g.nx + m.ch - 1) / m.ch);
  m.waves = s->d_waves;
  m.ctl = reinterpret_cast<Ctl*>(s->d_clock);
  m.par = s->par;
  m.exact = s->sweep_exact;
  m.ghosts = s->sweep_ghosts;
  return m;
}

bool step2_ade(const gmes_sim* s) { return s->d_adeq[0] || s->d_adeq[1] || s->d_adeq[2]; }

// Bytes of the cells that a step may finish after the sweep (dispersive E, and
// the H cells listed): those move twice, while the sweep saves a third of the
// whole grid's, and more where the two-kernel step has absorber words to read
// again.  us per step, that one against this, small Drude or critical-point
// blocks all over: no absorber, FP64 160^3 41 MB 166, 161; 82 MB 185, 191;
// 96^3 31 MB 63, 62; complex FP32 128^3 21 MB 102, 102; 37 MB 112, 119; FP32
// 160^3 36 MB 129, 125; 59 MB 151, 162; CPML FP64 160^3 34 MB 234, 230; FP32
// 192^3 30 MB 210, 191; CPML on z alone, complex FP32 384 x 384 x 192 173 MB
// (13 % of the cells) 1489, 1450.
double sweep_list_limit(const gmes_sim* s) {
  switch (s->sweep_part.absorber) {
    case kPmlNone: return s->esize == 8 ? 20e6 : 35e6;
    case kUpml: return s->esize == 8 ? 12e6 : 35e6;
    case kPmlZ: return std::max(72e6, 0.15 * 6 * s->ncell[0] * s->esize);
    default: return 35e6;
  }
}
int64_t ade_cells(const gmes_sim* s) {
  int64_t n = 0;
  for (int c = 0; c < 3; ++c)
    for (int k = GMES_CLS_DRUDE; k < GMES_CLS_DM2; ++k) n += s->ade[c][k].n;
  return n;
}

// Lists the H cells that a step finishes after the sweep (stepfix.hip).
// sweep_src_ok is false, and the sim keeps the two-kernel step, when an
// operation acts on a ghost cell or on a dispersive one (its order after the
// medium's update would need another launch), when one of those H cells has
// live absorber state, or when they are too many (sweep_list_limit).
int sweep_fix_build(gmes_sim* s) {
  HIP_TRY(sync_exec(s));
  fix_release(s);
  for (int& n : s->fix_nitem) n = 0;
  s->sweep_src_ok = false;
  const int64_t n[3] = {s->g.nx, s->g.ny, s->g.nz};
  if (n[0] * n[1] * n[2] >= INT32_MAX / 4) return GMES_OK;  // 32-bit items
  for (const gmes_src_op& o : s->ops) {
    const int64_t sy = s->shape[o.comp][1], sz = s->shape[o.comp][2];
    const int64_t ix[3] = {o.cell / (sy * sz), (o.cell / sz) % sy, o.cell % sz};
    for (int a = 0; a < 3; ++a) {
      const int64_t x = ix[a] - (o.comp >= 3 && a != o.comp - 3);
      if (x < 0 || x >= n[a]) return GMES_OK;  // a ghost cell
    }
    if (o.comp < 3 && s->recs[s->host_ids[o.comp][o.cell]].cls >= GMES_CLS_DRUDE) return GMES_OK;
  }
  FixBuild b{};
  for (int a = 0; a < 3; ++a) {
    b.n[a] = (int)n[a];
    // storage coordinates of H lie one up
    const int lo = s->sweep_run_h[a] & 0xFFFF, hi = s->sweep_run_h[a] >> 16;
    b.run_h[a] = std::max(0, lo - 1) | (std::max(0, hi - 1) << 16);
  }
  b.cells = n[0] * n[1] * n[2];
  b.nblk = (int)((b.cells + kFixMark - 1) / kFixMark);
  for (int c = 0; c < 6; ++c) {
    b.base[c] = dev_index(s, c, 0, 0, 0);
    b.pi[c] = s->pi[c];
    b.p[c] = s->pitch[c];
    if (c >= 3) b.hid[c - 3] = s->ids[c] + dev_index(s, c, c != 3, c != 4, c != 5);
  }
  b.groups = s->d_groups;
  b.nge = s->ngroups_e;
  b.ngroups = s->ngroups_e + s->ngroups_h;
  std::vector<int32_t> cls(s->recs.size());
  for (size_t r = 0; r < cls.size(); ++r) cls[r] = s->recs[r].cls;
  const size_t mark = ((size_t)(3 * b.cells) + 15) / 16 * 16, count = (size_t)3 * b.nblk * sizeof(int32_t),
               rec = cls.size() * sizeof(int32_t);
  char* tmp = nullptr;
  std::vector<int32_t> counts((size_t)3 * b.nblk);
  int bad = 0;
  auto build = [&]() -> hipError_t {
    hipError_t e = hipMalloc((void**)&tmp, mark + count + rec + 16);
    if (e != hipSuccess) return e;
    b.mark = reinterpret_cast<uint8_t*>(tmp);
    b.count = reinterpret_cast<int32_t*>(tmp + mark);
    b.cls = reinterpret_cast<int32_t*>(tmp + mark + count);
    b.bad = reinterpret_cast<int*>(tmp + mark + count + rec);
    if ((e = hipMemset(tmp, 0, mark + count + rec + 16)) != hipSuccess) return e;
    if ((e = hipMemcpy(const_cast<int32_t*>(b.cls), cls.data(), rec, hipMemcpyHostToDevice)) != hipSuccess) return e;
    for (int c = 0; c < 3; ++c)
      for (int k = GMES_CLS_DRUDE; k < GMES_CLS_DM2; ++k) {
        const AdeList& L = s->ade[c][k];
        if (!L.n) continue;
        b.ade_cell = L.cell;
        b.ade_n = (int)L.n;
        b.comp = c;
        b.s1 = (int)s->shape[c][1];
        b.s2 = (int)s->shape[c][2];
        launch_fix_mark_ade(b, nullptr);
      }
    if (b.ngroups) launch_fix_mark_src(b, nullptr);
    launch_fix_count(b, nullptr);
    if ((e = hipMemcpy(counts.data(), b.count, count, hipMemcpyDeviceToHost)) != hipSuccess) return e;
    int total = 0;
    for (int c = 0; c < 3; ++c) {
      b.first_item[c] = total;
      for (int q = 0; q < b.nblk; ++q) {
        const int m = counts[(size_t)c * b.nblk + q];
        counts[(size_t)c * b.nblk + q] = total;
        total += m;
      }
      b.nitem[c] = total - b.first_item[c];
    }
    if (!total) return hipSuccess;
    if ((double)(total + ade_cells(s)) * s->esize > sweep_list_limit(s)) {
      bad = 1;
      return hipSuccess;
    }
    if ((e = hipMalloc(&s->d_fix_items, (size_t)total * sizeof(FixItem))) != hipSuccess) return e;
    s->fix_bytes = (int64_t)total * sizeof(FixItem);
    s->bytes += s->fix_bytes;
    s->sweep_bytes += s->fix_bytes;
    b.items = static_cast<FixItem*>(s->d_fix_items);
    if ((e = hipMemcpy(b.count, counts.data(), count, hipMemcpyHostToDevice)) != hipSuccess) return e;
    launch_fix_fill(b, nullptr);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    return hipMemcpy(&bad, b.bad, sizeof bad, hipMemcpyDeviceToHost);
  };
  const hipError_t e = build();
  if (tmp) (void)dev_release(tmp);
  if (e == hipErrorOutOfMemory) {  // no room for the lists: the two-kernel step needs none
    (void)hipGetLastError();
    return GMES_OK;
  }
  HIP_TRY(e);
  for (int c = 0; c < 3; ++c) s->fix_nitem[c] = b.nitem[c];
  s->sweep_src_ok = !bad;
  return GMES_OK;
}

template <class T>
FixArgs<T> fix_args(const gmes_sim* s) {
  using R = typename real_of<T>::type;
  FixArgs<T> m{};
  for (int c = 0; c < 6; ++c) {
    const int64_t o = dev_index(s, c, c >= 3 && c != 3, c >= 3 && c != 4, c >= 3 && c != 5);
    const T* old = static_cast<const T*>(s->f_alt[c]) + o;  // the sweep has swapped the sets
    T* now = static_cast<T*>(s->f[c]) + o;
    const int a = c % 3;
    (c < 3 ? m.ei : m.hi)[a] = old;
    (c < 3 ? m.eo : m.ho)[a] = now;
    (c < 3 ? m.pe : m.ph)[a] = s->pi[c];
    (c < 3 ? m.re : m.rh)[a] = s->pitch[c];
    for (int x = 0; x < 3; ++x)
      (c < 3 ? m.phe : m.phh)[a][x] = cplx<R>{(R)s->g.phase[c][x][0], (R)s->g.phase[c][x][1]};
    m.base[c] = static_cast<T*>(s->f[c]);
    if (c >= 3) m.hid[a] = s->ids[c] + o;
  }
  m.n[0] = s->g.nx; m.n[1] = s->g.ny; m.n[2] = s->g.nz;
  m.d[0] = (R)s->g.dx; m.d[1] = (R)s->g.dy; m.d[2] = (R)s->g.dz;
  m.inv_d[0] = (R)(1.0 / s->g.dx); m.inv_d[1] = (R)(1.0 / s->g.dy); m.inv_d[2] = (R)(1.0 / s->g.dz);
  m.recs = static_cast<const DevRec<R>*>(s->d_recs);
  m.coef = static_cast<const R*>(s->d_coef);
  for (int c = 0; c < 3; ++c)
    for (int k = GMES_CLS_DRUDE; k < GMES_CLS_DM2; ++k) {
      const AdeList& L = s->ade[c][k];
      if (!L.n) continue;
      m.ade[m.nade++] = {L.cell, L.rec, L.state, (int)L.n, c, k, m.eblocks, (int)s->shape[c][1], (int)s->shape[c][2]};
      m.eblocks += (int)((L.n + kFixBlock - 1) / kFixBlock);
    }
  m.first_src = m.eblocks;
  m.groups = s->d_groups;
  m.nge = s->ngroups_e;
  m.eblocks += (m.nge + kFixBlock - 1) / kFixBlock;
  m.ops = static_cast<const DevSrcOp<R>*>(s->d_ops);
  m.waves = s->d_waves;
  for (int i = 0; i < s->naux; ++i)
    for (int c = 0; c < 6; ++c) m.aux[i][c] = s->aux[i] ? s->aux[i]->f[c] : nullptr;
  m.ctl = reinterpret_cast<Ctl*>(s->d_clock);
  m.items = static_cast<const FixItem*>(s->d_fix_items);
  for (int c = 0, at = 0; c < 3; ++c) {
    m.nitem[c] = s->fix_nitem[c];
    m.first_item[c] = at;
    m.item_blk[c] = m.hblocks;
    at += m.nitem[c];
    m.hblocks += (m.nitem[c] + kFixBlock - 1) / kFixBlock;
  }
  return m;
}

// Marks the cells of the sim's source operations in the sweep's ids, when
// all of them can be applied there (sweep_src_ok).  Of a committed sim only
// (commit itself calls it): records or material ids set since are neither
// checked nor those that the tables were built from.
int sweep_sources(gmes_sim* s) {
  if (!s->sweep_ok) return GMES_OK;
  if (s->sweep_1d) return sweep1_sources(s);
  if (s->sweep_2d) return sweep2_sources(s);
  HIP_TRY(sync_exec(s));
  const size_t idw = (size_t)s->step_idw;
  char* const ids = static_cast<char*>(s->d_step_ids);
  for (const auto& x : s->src_ids) HIP_TRY(hipMemcpy(ids + x.first * idw, &x.second, idw, hipMemcpyHostToDevice));
  s->src_ids.clear();
  s->has_waves = false;
  s->sweep_fix = s->sweep_ade || s->naux || (int)s->ops.size() > kSweepMaxSrc;
  if (s->sweep_fix) {
    if (int rc = sweep_fix_build(s)) return rc;
    return s->fp64 ? sweep_upload_tab<double>(s, {}, {}) : sweep_upload_tab<float>(s, {}, {});
  }
  s->sweep_src_ok = true;
  std::vector<std::array<int, 3>> src[2];
  std::vector<int64_t> cell(s->ops.size());
  const int64_t n[3] = {s->g.nx, s->g.ny, s->g.nz};
  for (size_t q = 0; s->sweep_src_ok && q < s->ops.size(); ++q) {
    const gmes_src_op& o = s->ops[q];
    const int c = o.comp, h = c >= 3;
    const int64_t sy = s->shape[c][1], sz = s->shape[c][2];
    int64_t ix[3] = {o.cell / (sy * sz), (o.cell / sz) % sy, o.cell % sz};
    bool ok = o.kind == GMES_SRC_SET || o.kind == GMES_SRC_SUB;
    for (int a = 0; a < 3; ++a) {
      if (h && a != c % 3) --ix[a];
      if (ix[a] < 0 || ix[a] >= n[a]) ok = false;  // a ghost cell
    }
    cell[q] = (ix[0] * n[1] + ix[1]) * s->pitch[0] + ix[2];
    for (size_t p = 0; p < q; ++p)
      if (cell[p] == cell[q]) ok = false;  // two operations on one thread's cells
    if (!ok) s->sweep_src_ok = false;
  }
  if (!s->sweep_src_ok) return GMES_OK;
  for (size_t q = 0; q < s->ops.size(); ++q) {
    const int h = s->ops[q].comp >= 3;
    uint32_t w = 0;
    HIP_TRY(hipMemcpy(&w, ids + cell[q] * idw, idw, hipMemcpyDeviceToHost));
    s->src_ids.push_back({cell[q], w});
    const uint32_t id = (uint32_t)((h ? s->step_h.size() : s->step_e.size()) + src[h].size());
    const uint32_t low = (1u << s->step_eb) - 1u;
    src[h].push_back({(int)(h ? w >> s->step_eb : w & low), s->ops[q].comp % 3, (int)q});
    w = h ? (w & low) | id << s->step_eb : (w & ~low) | id;
    HIP_TRY(hipMemcpy(ids + cell[q] * idw, &w, idw, hipMemcpyHostToDevice));
  }
  s->has_waves = !s->ops.empty();
  return s->fp64 ? sweep_upload_tab<double>(s, src[0], src[1]) : sweep_upload_tab<float>(s, src[0], src[1]);
}

// Builds what one-sweep steps need (at commit, which has released the old);
// leaves sweep_ok false when the sim does not qualify.
int sweep_build(gmes_sim* s) {
  if (line_dir(s) >= 0) return sweep1_build(s);
  if (is_2z(s)) return s->naux ? GMES_OK : sweep2_build(s);
  if (!is3d(s) || s->g.dtype == GMES_C128) return GMES_OK;
  const int nz = s->g.nz;
  if (kSweepMinRows * nz > kStepMaxThreads || s->g.ny < 2) return GMES_OK;
  for (int c = 0; c < 6; ++c)  // 32-bit byte offsets, both state words included
    if (2 * s->dsize[c] * s->esize >= (int64_t)0xFFFFFF00) return GMES_OK;
  bool cpml = false, upml = false;
  s->sweep_ade = false;
  for (int c = 0; c < 6; ++c) {
    cpml |= s->has_cls[c][GMES_CLS_CPML];
    upml |= s->has_cls[c][GMES_CLS_UPML];
    if (s->has_cls[c][GMES_CLS_DM2]) return GMES_OK;
    for (int k = GMES_CLS_DRUDE; k < GMES_CLS_DM2; ++k) s->sweep_ade |= s->has_cls[c][k];
  }
  if ((cpml && upml) || ((cpml || upml) && s->nprof != 1)) return GMES_OK;
  // the kernels keep every component's absorber state
  if (cpml || upml) {
    for (int c = 0; c < 6; ++c)
      if (!s->pml_state[c]) return GMES_OK;
  }
  s->sweep_absorber = cpml ? 1 : upml ? 2 : 0;
  if (cpml)
    for (int a = 0; a < 3; ++a) {
      s->sweep_run_e[a] = sweep_dead_run(s, true, a);
      s->sweep_run_h[a] = sweep_dead_run(s, false, a);
    }
  if (upml) {
    upml_free_box(s, s->sweep_run_e);
    for (int a = 0; a < 3; ++a) s->sweep_run_h[a] = s->sweep_run_e[a];
  }
  if (s->sweep_absorber && !sweep_rows_agree(s, cpml ? 3 : 6)) return GMES_OK;
  if (cpml && !sweep_live_cells_cpml(s)) return GMES_OK;
  // FP64: divisions by powers of two are exact multiplications
  auto pow2 = [](double v) { int e; return std::frexp(v, &e) == 0.5; };
  bool exact = pow2(s->g.dx) && pow2(s->g.dy) && pow2(s->g.dz);
  for (int c = 0; c < 6 && cpml; ++c)
    for (int a = 0; a < 3; ++a)
      for (size_t q = 2; q < s->prof_host[0][c][a].size(); q += 3) exact = exact && s->prof_host[0][c][a][q] == 1.0;
  s->sweep_exact = exact;
  s->step_e.clear();
  s->step_h.clear();
  const size_t ent = s->fp64 ? sizeof(StepEnt<double>) : sizeof(StepEnt<float>);
  const size_t most = (size_t)kSweepMaxTab / ent - 2 * kSweepMaxSrc;
  if (!sweep_triples(s, true, most, s->step_e) || !sweep_triples(s, false, most, s->step_h) ||
      s->step_e.size() + s->step_h.size() > most)
    return GMES_OK;
  sweep_plan(s);
  if (!s->sweep_part.rows) return GMES_OK;
  // (they are read by at least as many H cells)
  if (2.0 * ade_cells(s) * s->esize > sweep_list_limit(s)) return GMES_OK;
  std::unique_lock<std::mutex> room(g_room_mu);
  if (!sweep_room(s)) return GMES_OK;
  // E and H entries, those of source cells included, in one 16-bit word when
  // they fit (256^3 FP32: at 4 bytes they are 67 of 1250 MB a step, 256 us; at 2
  // 248.  181 x 203 x 225 UPML 173, 168)
  auto bits = [](size_t n) {
    int b = 1;
    while ((size_t(1) << b) < n) ++b;
    return b;
  };
  const int eb = bits(s->step_e.size() + kSweepMaxSrc), hb = bits(s->step_h.size() + kSweepMaxSrc);
  s->step_idw = eb + hb <= 16 ? 2 : 4;
  s->step_eb = eb + hb <= 16 ? eb : 16;
  s->step_tab_cap = (int64_t)(s->step_e.size() + s->step_h.size()) + 2 * kSweepMaxSrc;
  const std::vector<StepKey> keys[2] = {sweep_keys(s->step_e), sweep_keys(s->step_h)};
  void* d_keys = nullptr;
  SweepParts parts;
  for (int c = 0; c < 6; ++c) parts.other.push_back({&s->f_alt[c], (size_t)s->dsize[c] * s->esize});
  for (int c = 0; c < 3; ++c) parts.state(s, c);
  parts.other.push_back({&s->d_step_ids, (size_t)s->g.nx * s->g.ny * s->pitch[0] * s->step_idw});
  parts.other.push_back({&s->d_step_tab, (size_t)s->step_tab_cap * ent});
  parts.other.push_back({(void**)&s->d_rare, (size_t)s->step_tab_cap * 3 * sizeof(StepRare)});
  parts.other.push_back({&d_keys, (keys[0].size() + keys[1].size()) * sizeof(StepKey)});
  int rc = sweep_take(s, parts);
  room.unlock();
  if (rc) {  // no room for a second set of buffers: the two-kernel step needs none
    (void)hipGetLastError();
    sweep_release(s);
    return GMES_OK;
  }
  if ((rc = sweep_ids(s, keys, static_cast<char*>(d_keys)))) return rc;
  s->src_ids.clear();
  s->sweep_ok = true;
  return GMES_OK;
}

// Whether an auxiliary grid takes one-sweep steps when its parent does.
bool aux_sweeps(const gmes_sim* a) {
  return a->sweep_1d && a->sweep_ok && a->sweep_src_ok && a->allow_fuse && a->probes.empty() && a->dfts.empty();
}

// Whether the next step of s is a one-sweep step.
bool sweeps(const gmes_sim* s) {
  if (!s->sweep_ok || !s->sweep_src_ok || !s->allow_fuse || (s->naux && !s->sweep_fix) || s->parent) return false;
  if (s->tile_bx > 0 && !s->tile_tuned) return false;
  for (const auto& p : s->probes)
    if (p.comp < 3 && on_ghost_copy_plane(s, p.comp, p.cell, false, true)) return false;
  return true;
}

// Whether something reads ghost planes between the steps of one call (else
// only its last step writes them).
bool sweep_ghosts(const gmes_sim* s) {
  auto on_ghost = [&](int c, int a, int64_t lo, int64_t hi) {
    return a != c % 3 && (c < 3 ? hi > s->shape[c][a] - 1 : lo < 1);
  };
  for (const auto& p : s->probes) {
    const int64_t sy = s->shape[p.comp][1], sz = s->shape[p.comp][2];
    const int64_t ix[3] = {p.cell / (sy * sz), (p.cell / sz) % sy, p.cell % sz};
    for (int a = 0; a < 3; ++a)
      if (on_ghost(p.comp, a, ix[a], ix[a] + 1)) return true;
  }
  for (const auto& d : s->dfts)
    for (int a = 0; a < 3; ++a)
      if (on_ghost(d.comp, a, d.lo[a], d.lo[a] + d.n[a])) return true;
  return false;
}

template <class T>
Step3Args<T> step3_args(const gmes_sim* s, const gmes_sim::SweepPart& part) {
  using R = typename real_of<T>::type;
  Step3Args<T> m{};
  auto rsrc = [](const void* p, int64_t bytes) {
    const uint64_t a = (uint64_t)(uintptr_t)p;
    // raw buffer: stride 0, 32-bit data format
    return i4_t{(int)(uint32_t)a, (int)(uint32_t)(a >> 32), (int)(uint32_t)bytes, 0x00020000};
  };
  for (int c = 0; c < 6; ++c) {
    const int64_t o = (int64_t)(kPad - s->koff[c]) * s->esize, b = s->dsize[c] * s->esize - o;
    const int64_t sb = b + (s->sweep_absorber == 1 ? s->dsize[c] * s->esize : 0);
    auto at = [&](const void* p, int64_t n) { return p ? rsrc(static_cast<const char*>(p) + o, n) : i4_t{0, 0, 0, 0}; };
    (c < 3 ? m.ei[c] : m.hi[c - 3]) = at(s->f[c], b);
    (c < 3 ? m.eo[c] : m.ho[c - 3]) = at(s->f_alt[c], b);
    if (c < 3) {
      m.si[c] = at(s->pml_state[c], sb);
      m.so[c] = at(s->pml_alt[c], sb);
    } else {
      m.sh[c - 3] = at(s->pml_state[c], sb);
    }
    m.ds[c] = (unsigned)(s->dsize[c] * s->esize);
    for (int a = 0; a < 3; ++a) {
      const cplx<R> ph{(R)s->g.phase[c][a][0], (R)s->g.phase[c][a][1]};
      if (c < 3) m.pe[c][a] = ph;
      else m.ph[c - 3][a] = ph;
    }
  }
  m.W0 = s->pitch[0];
  m.W2 = s->pitch[2];
  m.n[0] = s->g.nx; m.n[1] = s->g.ny; m.n[2] = s->g.nz;
  m.ids = rsrc(s->d_step_ids, (int64_t)s->g.nx * s->g.ny * s->pitch[0] * s->step_idw);
  m.idw = s->step_idw;
  m.eb = s->step_eb;
  m.exact = s->sweep_exact;
  m.ghosts = s->sweep_ghosts;
  m.tab = s->d_step_tab;
  m.rare = s->d_rare;
  m.net = s->step_net;
  m.nht = s->step_nht;
  m.d[0] = (R)s->g.dx; m.d[1] = (R)s->g.dy; m.d[2] = (R)s->g.dz;
  m.inv_d[0] = (R)(1.0 / s->g.dx); m.inv_d[1] = (R)(1.0 / s->g.dy); m.inv_d[2] = (R)(1.0 / s->g.dz);
  const R* prof = static_cast<const R*>(s->d_prof);
  // rows two components share: x of the 2nd, y and z of the 1st; own rows
  const int sc[3] = {1, 0, 0};
  for (int a = 0; a < 3; ++a) {
    m.re[a] = prof + s->prof_off0[sc[a]][a];
    m.rh[a] = prof + s->prof_off0[3 + sc[a]][a];
    m.oe[a] = prof + s->prof_off0[a][a];
    m.oh[a] = prof + s->prof_off0[3 + a][a];
    m.run_e[a] = s->sweep_run_e[a];
    m.run_h[a] = s->sweep_run_h[a];
  }
  m.rows = part.rows;
  m.nrect = part.nrect;
  for (int q = 0; q < part.nrect; ++q) {
    const int* r = part.rect[q];
    const int tiles = (r[3] - r[2] + m.rows - 2) / (m.rows - 1), nblk = tiles * ((r[1] - r[0] + r[4] - 1) / r[4]);
    m.rect[q] = {r[0], r[1], r[2], r[3], r[4], tiles, nblk, (nblk + 7) / 8, m.slots, r[5]};
    m.slots += (nblk + 7) / 8;
  }
  m.waves = s->has_waves ? s->d_waves : nullptr;
  m.ctl = reinterpret_cast<Ctl*>(s->d_clock);
  m.par = s->par;
  return m;
}

// The current buffers become the other set.
void sweep_swap(gmes_sim* s) {
  for (int c = 0; c < 6; ++c)
    if (s->f_alt[c]) std::swap(s->f[c], s->f_alt[c]);
  for (int c = 0; c < 3; ++c)
    if (s->pml_alt[c]) std::swap(s->pml_state[c], s->pml_alt[c]);
  for (int c = 0; c < 3; ++c)
    for (int k = 0; k < GMES_NCLS; ++k)
      if (s->ade_alt[c][k]) std::swap(s->ade[c][k].state, s->ade_alt[c][k]);
  s->par ^= 1;
}

template <class T>
void enqueue_sweep(gmes_sim* s, hipStream_t st) {
  time_begin(s, 0, st);
  if (s->sweep_1d) {
    launch_step1d<T>(step1_args<T>(s), st);
  } else if (s->sweep_2d) {
    launch_step2d<T>(step2_args<T>(s), step2_tm(s), s->sweep_absorber, step2_ade(s), st);
  } else if constexpr (!std::is_same<T, cplx<double>>::value) {
    launch_step3d<T>(step3_args<T>(s, s->sweep_part), s->sweep_part.absorber, s->sweep_part.threads, st);
  }
  time_end(s, st);
  sweep_swap(s);
}

template <class T>
void enqueue_step_t(gmes_sim* s, hipStream_t st) {
  if (sweeps(s)) {
    enqueue_sweep<T>(s, st);
    if constexpr (!std::is_same<T, cplx<double>>::value) {
      if (s->sweep_fix) {
        time_begin(s, 2, st);
        launch_fix_e<T>(fix_args<T>(s), st);  // reads the auxiliary grids before their step
        time_end(s, st);
        enqueue_aux_steps(s, true, st);
        if (s->sweep_ghosts) enqueue_ghost<T>(s, true, 0, st);
        time_begin(s, 3, st);
        launch_fix_h<T>(fix_args<T>(s), st);
        time_end(s, st);
        enqueue_probe<T>(s, kProbeBoth, st);
        enqueue_dft<T>(s, st);
        return;
      }
    }
    enqueue_probe<T>(s, kProbeBoth, st);
    enqueue_dft<T>(s, st);
    return;
  }
  enqueue_ghost<T>(s, false, 1, st);
  enqueue_main<T>(s, true, st);
  enqueue_ade<T>(s, st);
  enqueue_src<T>(s, true, st);
  enqueue_probe<T>(s, kProbeE, st);
  enqueue_aux_steps(s, false, st);
  if (!s->fuse_e) enqueue_ghost<T>(s, true, 0, st);
  enqueue_main<T>(s, false, st);
  enqueue_src<T>(s, false, st);
  enqueue_probe<T>(s, kProbeH, st);
  enqueue_dft<T>(s, st);
}

void enqueue_aux_steps(gmes_sim* s, bool sweep, hipStream_t st) {
  for (int i = 0; i < s->naux; ++i) {
    gmes_sim* a = s->aux[i];
    if (!a) continue;
    time_begin(s, 5, st);
    if (!(sweep && aux_sweeps(a))) {
      enqueue_step(a, st);
    } else {
      switch (a->g.dtype) {
        case GMES_F32: enqueue_sweep<float>(a, st); break;
        case GMES_F64: enqueue_sweep<double>(a, st); break;
        case GMES_C64: enqueue_sweep<cplx<float>>(a, st); break;
        default: enqueue_sweep<cplx<double>>(a, st); break;
      }
    }
    time_end(s, st);
  }
}

void enqueue_step(gmes_sim* s, hipStream_t st) {
  switch (s->g.dtype) {
    case GMES_F32: enqueue_step_t<float>(s, st); break;
    case GMES_F64: enqueue_step_t<double>(s, st); break;
    case GMES_C64: enqueue_step_t<cplx<float>>(s, st); break;
    default: enqueue_step_t<cplx<double>>(s, st); break;
  }
}

void advance_host_clock(gmes_sim* s, int64_t n) {
  s->step += n;
  s->probe_n = s->step - s->probe_base;
  for (int i = 0; i < s->naux; ++i)
    if (s->aux[i]) advance_host_clock(s->aux[i], n);
}

// Waits for all work that may touch s: its own stream, for an aux sim the
// stream of the sim that advances it, and the stream of s's batch.
hipError_t sync_exec(gmes_sim* s) {
  hipError_t e = hipStreamSynchronize(s->stream);
  if (e == hipSuccess && s->parent) e = sync_exec(s->parent);
  if (e == hipSuccess && s->batch_stream) e = hipStreamSynchronize(s->batch_stream);
  return e;
}

// Checks that every step in [s->step, s->step + n) is covered by the
// waveform window and the probe buffer (recursively for aux sims).
int check_windows(gmes_sim* s, int64_t n) {
  bool waves = false;
  for (const auto& o : s->ops)
    if (o.kind == GMES_SRC_SET || o.kind == GMES_SRC_SUB || o.wave >= 0) waves = true;
  if (waves && (s->step < s->wave_step0 || s->step + n > s->wave_step0 + s->wave_n))
    return set_error(GMES_EINVAL, "waveforms cover steps [%lld, %lld), need [%lld, %lld)",
                     (long long)s->wave_step0, (long long)(s->wave_step0 + s->wave_n),
                     (long long)s->step, (long long)(s->step + n));
  if (!s->dfts.empty() && (s->step < s->dft_step0 || s->step + n > s->dft_step0 + s->dft_n))
    return set_error(GMES_EINVAL, "DFT weights cover steps [%lld, %lld), need [%lld, %lld)",
                     (long long)s->dft_step0, (long long)(s->dft_step0 + s->dft_n), (long long)s->step,
                     (long long)(s->step + n));
  for (int i = 0; i < s->naux; ++i) {
    if (!s->aux[i]) continue;
    int rc = check_windows(s->aux[i], n);
    if (rc) return rc;
  }
  return GMES_OK;
}

int ensure_probe_capacity(gmes_sim* s, int64_t n) {
  for (int i = 0; i < s->naux; ++i) {
    if (!s->aux[i]) continue;
    int rc = ensure_probe_capacity(s->aux[i], n);
    if (rc) return rc;
  }
  if (s->probes.empty()) return GMES_OK;
  const int64_t need = (s->step - s->probe_base) + n;
  if (need <= s->probe_cap) return GMES_OK;
  int64_t cap = std::max<int64_t>(1024, s->probe_cap);
  while (cap < need) cap *= 2;
  double* nb = nullptr;
  int rc = dev_alloc(s, (void**)&nb, (size_t)cap * s->probes.size() * 2 * sizeof(double));
  if (rc) return rc;
  HIP_TRY(sync_exec(s));
  if (s->d_probe_buf) {
    const int64_t used = s->step - s->probe_base;
    for (size_t p = 0; p < s->probes.size(); ++p)
      HIP_TRY(hipMemcpy(nb + p * cap * 2, s->d_probe_buf + p * s->probe_cap * 2, used * 2 * sizeof(double),
                        hipMemcpyDeviceToDevice));
    dev_free(s, s->d_probe_buf, (size_t)s->probe_cap * s->probes.size() * 2 * sizeof(double));
  }
  s->d_probe_buf = nb;
  s->probe_cap = cap;
  s->graph_dirty = true;
  ++s->gen;
  if (s->parent) {
    s->parent->graph_dirty = true;
    ++s->parent->gen;
  }
  return GMES_OK;
}

void destroy_graph(gmes_sim* s) {
  if (s->graph_exec) {
    (void)hipGraphExecDestroy(s->graph_exec);
    s->graph_exec = nullptr;
  }
  s->graph_dirty = true;
  ++s->gen;
  // the parent's graph holds this aux sim's kernels and their arguments
  if (s->parent) destroy_graph(s->parent);
}

int build_graph(gmes_sim* s) {
  destroy_graph(s);
  hipGraph_t graph;
  hipError_t e;
  {
    CaptureGuard capture;
    HIP_TRY(hipStreamBeginCapture(s->stream, hipStreamCaptureModeThreadLocal));
    // one-sweep steps swap the buffers: a graph of two returns them
    s->graph_par = s->par;
    s->graph_steps = sweeps(s) ? 2 : 1;
    s->sweep_ghosts = sweep_ghosts(s);
    for (int t = 0; t < s->graph_steps; ++t) enqueue_step(s, s->stream);
    HIP_TRY(hipStreamEndCapture(s->stream, &graph));
    e = hipGraphInstantiate(&s->graph_exec, graph, nullptr, nullptr, 0);
    s->graph_dirty = e != hipSuccess;
  }
  (void)hipGraphDestroy(graph);
  if (e != hipSuccess) return set_error(GMES_EDEVICE, "hipGraphInstantiate: %s", hipGetErrorString(e));
  return GMES_OK;
}

int collect_timing(gmes_sim* s) {
  for (auto& p : s->timing.pending) {
    float ms = 0.f;
    HIP_TRY(hipEventSynchronize(p.second.second));
    HIP_TRY(hipEventElapsedTime(&ms, p.second.first, p.second.second));
    s->timing.ms[p.first] += ms;
    s->timing.launches[p.first] += 1;
    (void)hipEventDestroy(p.second.first);
    (void)hipEventDestroy(p.second.second);
  }
  s->timing.pending.clear();
  return GMES_OK;
}

bool any_graph_blocker(gmes_sim* s) { return s->timing.on; }

// The clock as one-sweep steps pass it on (Ctl::clk), brought up to date before
// the first of them after other steps.
void sweep_clock(gmes_sim* s, bool sweep, hipStream_t st) {
  if (sweep && s->clk_stale) launch_clock_copy(reinterpret_cast<Ctl*>(s->d_clock), st);
  s->clk_stale = !sweep;
}

// The table of the auxiliary grids' buffers that source launches read; their
// one-sweep steps swap those.
int aux_pointers(gmes_sim* s) {
  for (int i = 0; i < s->naux; ++i) {
    if (!s->aux[i] || !memcmp(s->aux_ptr[i], s->aux[i]->f, sizeof s->aux_ptr[i])) continue;
    HIP_TRY(sync_exec(s));
    memcpy(s->aux_ptr[i], s->aux[i]->f, sizeof s->aux_ptr[i]);
    HIP_TRY(hipMemcpy(static_cast<void**>(s->d_aux_ptrs) + i * 6, s->aux_ptr[i], sizeof s->aux_ptr[i], hipMemcpyHostToDevice));
  }
  return GMES_OK;
}

int do_step(gmes_sim* s, int64_t n) {
  if (!s->committed) return set_error(GMES_EINVAL, "sim is not committed");
  if (n < 0) return set_error(GMES_EINVAL, "negative step count");
  if (s->parent) return set_error(GMES_EINVAL, "an auxiliary grid is advanced by its parent");
  if (s->aux_lost) return set_error(GMES_EINVAL, "an auxiliary grid of this sim was destroyed");
  if (s->batch_stream) HIP_TRY(hipStreamSynchronize(s->batch_stream));
  int rc = check_windows(s, n);
  if (rc) return rc;
  if ((rc = ensure_probe_capacity(s, n))) return rc;
  HIP_TRY(hipSetDevice(s->device));
  // a capture waits until it is alone in the engine: what another thread does
  // before or after it (sweep_reclaim) may call for another graph
  const bool graph = s->use_graph && !any_graph_blocker(s);
  while (graph && (s->graph_dirty || !s->graph_exec || s->graph_steps != (sweeps(s) ? 2 : 1)))
    if ((rc = build_graph(s))) return rc;
  const bool sweep = sweeps(s);
  if (n > 0) {
    sweep_clock(s, sweep, s->stream);
    for (int i = 0; i < s->naux; ++i)
      if (s->aux[i]) sweep_clock(s->aux[i], sweep && aux_sweeps(s->aux[i]), s->stream);
    if (!sweep && (rc = aux_pointers(s))) return rc;
  }
  const int par = s->par;
  if (graph) {
    int64_t t = 0;
    const int64_t last = sweep ? 1 : 0;  // the step that writes the ghost planes
    if (s->par != s->graph_par && t + last < n) { enqueue_step(s, s->stream); ++t; }
    for (; t + s->graph_steps + last <= n; t += s->graph_steps) HIP_TRY(hipGraphLaunch(s->graph_exec, s->stream));
    for (; t < n; ++t) {
      s->sweep_ghosts = sweep_ghosts(s) || t == n - 1;
      enqueue_step(s, s->stream);
    }
    HIP_TRY(hipGetLastError());
  } else {
    for (int64_t t = 0; t < n; ++t) {
      s->sweep_ghosts = sweep_ghosts(s) || t == n - 1;
      enqueue_step(s, s->stream);
    }
    HIP_TRY(hipGetLastError());
  }
  if (s->par != par) ++s->gen;  // a batch's graph may hold the other set's pointers
  advance_host_clock(s, n);
  s->probe_n = s->step - s->probe_base;
  if (s->timing.on && s->timing.pending.size() > 4096) return collect_timing(s);
  return GMES_OK;
}

// ---- tile autotuner
// Times the E main kernel of a sim under each candidate tile and keeps the
// fastest, per size class (device, storage type, mode, log2 of the
// extents) for the life of the process.  The fields and CPML state the
// trial launches touch are saved first and restored afterwards, so tuning
// leaves the simulation unchanged.
std::mutex g_tune_mu;
std::map<std::string, std::pair<int, int>> g_tune_cache;

int ceil_log2(int v) {
  int l = 0;
  while ((1 << l) < v) ++l;
  return l;
}

template <class T>
int autotune_t(gmes_sim* s, int& best_bx, int& best_by) {
  MainArgs<T> m;
  int ext[3];
  best_bx = best_by = 0;
  if (!main_args<T>(s, true, m, ext)) return GMES_OK;
  if (!is3d(s)) return GMES_OK;  // the 2-D/1-D tile follows each field type's rows
  char key[96];
  snprintf(key, sizeof key, "%d/%d/%x/%d/%d/%d", s->device, s->g.dtype, s->g.active, ceil_log2(ext[0]),
           ceil_log2(ext[1]), ceil_log2(ext[2]));
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tune_cache.find(key);
    if (it != g_tune_cache.end()) {
      best_bx = it->second.first;
      best_by = it->second.second;
      return GMES_OK;
    }
  }
  std::vector<int> cand;
  const int row = next_pow2(ext[2]);
  for (int bx = 1; bx <= 256; bx *= 2) {
    if (bx == 256 && s->packed) { cand.push_back(bx); continue; }  // flat blocks
    if (bx > std::max(row, 1) && bx > 1) continue;          // wider than a row: idle lanes
    if (row >= 32 && bx < 32) continue;                      // narrower than a 128-byte line
    cand.push_back(bx);
  }
  if (cand.empty()) cand.push_back(std::min(256, row));
  HIP_TRY(sync_exec(s));
  // save what the E kernel writes: E fields and E-side PML state
  std::vector<std::pair<void*, std::pair<void*, size_t>>> saved;
  for (int c = 0; c < 3; ++c) {
    if (!active(s, c)) continue;
    const size_t fb = (size_t)s->dsize[c] * s->esize;
    void* tmp = nullptr;
    HIP_TRY(dev_malloc(s->device, &tmp, fb));
    HIP_TRY(hipMemcpy(tmp, s->f[c], fb, hipMemcpyDeviceToDevice));
    saved.push_back({tmp, {s->f[c], fb}});
    if (s->pml_state[c]) {
      const int pw = s->has_cls[c][GMES_CLS_CPML] ? 2 : 1;
      const size_t pb = (size_t)pw * s->dsize[c] * s->esize;
      HIP_TRY(dev_malloc(s->device, &tmp, pb));
      HIP_TRY(hipMemcpy(tmp, s->pml_state[c], pb, hipMemcpyDeviceToDevice));
      saved.push_back({tmp, {s->pml_state[c], pb}});
    }
  }
  hipEvent_t e0, e1;
  HIP_TRY(hipEventCreate(&e0));
  HIP_TRY(hipEventCreate(&e1));
  float best = 1e30f;
  const int reps = 5;
  for (int bx : cand) {
    const int by = std::max(1, 256 / bx);
    launch_main_tile<T>(s, true, m, ext, bx, by, s->stream);
    HIP_TRY(hipEventRecord(e0, s->stream));
    for (int r = 0; r < reps; ++r) launch_main_tile<T>(s, true, m, ext, bx, by, s->stream);
    HIP_TRY(hipEventRecord(e1, s->stream));
    HIP_TRY(hipEventSynchronize(e1));
    float ms = 0;
    HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
    if (ms < best) {
      best = ms;
      best_bx = bx;
      best_by = by;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  for (auto& x : saved) {
    HIP_TRY(hipMemcpy(x.second.first, x.first, x.second.second, hipMemcpyDeviceToDevice));
    HIP_TRY(dev_release(x.first));
  }
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_tune_cache[key] = {best_bx, best_by};
  return GMES_OK;
}

// Whether the 3-D (or 2-D collapsed-z) E kernel may write the E ghost
// planes itself instead of the separate copy that runs later in the step
// (after the dispersive updates, the E sources and the E probes).  The results are the same when
// none of those touches a plane involved in the copy: no dispersive cell
// on a source plane (plane 0 of a transverse axis), no E source operation
// on a source or ghost plane, no E probe on a ghost plane (it would read
// the ghost before the copy).  gmes_sim_set_ghost_fusion(sim, 0) turns it off.
bool on_ghost_copy_plane(const gmes_sim* s, int c, int64_t x, bool source, bool ghost) {
  const int64_t sy = s->shape[c][1], sz = s->shape[c][2];
  const int64_t ix[3] = {x / (sy * sz), (x / sz) % sy, x % sz};
  for (int t = 0; t < 2; ++t) {
    const int a = kGhostOrder[c][t];
    if ((source && ix[a] == 0) || (ghost && ix[a] == s->shape[c][a] - 1)) return true;
  }
  return false;
}

//
// In a 2-D mode with a collapsed z axis where Ez is the only E component
// (TMz), the z ghost plane (k = 0) of Hx and Hy is read by no E update
// (Ez reads k = 1), and nothing runs between the H ghost copy and the E
// kernel; the 2-D E kernel then writes that plane itself from k = 1, with
// the copy's phases and corner order, and the H copy leaves it out.
void decide_fusion(gmes_sim* s) {
  const bool prev = s->fuse_e, prev_hz = s->fuse_hz;
  bool f = s->allow_fuse && (is3d(s) || is_2z(s)) && s->committed && !s->ade_on_ghost_source;
  for (size_t n = 0; f && n < s->ops.size(); ++n)
    if (s->ops[n].comp < 3 && on_ghost_copy_plane(s, s->ops[n].comp, s->ops[n].cell, true, true)) f = false;
  for (size_t n = 0; f && n < s->probes.size(); ++n)
    if (s->probes[n].comp < 3 && on_ghost_copy_plane(s, s->probes[n].comp, s->probes[n].cell, false, true)) f = false;
  s->fuse_e = f;
  bool hz = s->allow_fuse && s->committed && is_2z(s) && active(s, 2) && !active(s, 0) && !active(s, 1);
  bool any = false;
  for (int c = 3; hz && c < 5; ++c) {
    if (!active(s, c) || s->shape[c][2] != 2) continue;
    any = true;
    // the E kernel's threads span Ez's (i, j) extent
    if (s->shape[c][0] > s->shape[2][0] || s->shape[c][1] > s->shape[2][1]) hz = false;
  }
  s->fuse_hz = hz && any;
  if (f != prev || s->fuse_hz != prev_hz) destroy_graph(s);
}

int ctl_write(gmes_sim* s) {
  Ctl c;
  HIP_TRY(sync_exec(s));
  HIP_TRY(hipMemcpyAsync(&c, s->d_clock, sizeof c, hipMemcpyDeviceToHost, s->stream));
  HIP_TRY(sync_exec(s));
  c.wave_step0 = s->wave_step0;
  c.wave_n = s->wave_n;
  c.probe_base = s->probe_base;
  c.dft_step0 = s->dft_step0;
  c.dft_n = s->dft_n;
  HIP_TRY(hipMemcpyAsync(s->d_clock, &c, sizeof c, hipMemcpyHostToDevice, s->stream));
  HIP_TRY(sync_exec(s));
  return GMES_OK;
}

// ---- sum of |F|^2 over a box
// No-allocation variant: the partial sums live in this file-scope device
// array (one copy per GPU, held until the process ends).  Host code never
// passes the array's name to a kernel or copy: it uses the device address
// that hipGetSymbolAddress returns, looked up once per device with that
// device current.
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu[kMaxDevices];   // serialises no-allocation calls per device
double* g_scratch_ptr[kMaxDevices] = {};

static int sq_check(const gmes_sim* s, int32_t c, const int64_t lo[3], const int64_t hi[3], const double* out,
                    int64_t& ncells) {
  if (!s || !lo || !hi || !out) return set_error(GMES_EINVAL, "null argument");
  if (c < 0 || c > 5) return set_error(GMES_EINVAL, "bad component");
  ncells = 1;
  for (int a = 0; a < 3; ++a) {
    if (lo[a] < 0 || hi[a] > s->shape[c][a] || hi[a] <= lo[a]) return set_error(GMES_ERANGE, "box out of bounds");
    ncells *= hi[a] - lo[a];
  }
  return GMES_OK;
}

template <class T>
static void sq_launch(const gmes_sim* s, int c, const int64_t lo[3], const int64_t hi[3], double* partial) {
  SqBox<T> b;
  b.f = static_cast<const T*>(s->f[c]);
  b.pi = s->pi[c];
  b.p = s->pitch[c];
  b.pk = s->pk[c];
  b.koff = s->koff[c];
  b.ncells = 1;
  for (int a = 0; a < 3; ++a) {
    b.lo[a] = (int)lo[a];
    b.n[a] = (int)(hi[a] - lo[a]);
    b.ncells *= b.n[a];
  }
  launch_sum_sq<T>(b, partial, s->stream);
}

// Runs the two passes on the sim's stream into partial[0 .. nblocks] and
// copies partial[nblocks] to *out.
static int sq_run(gmes_sim* s, int32_t c, const int64_t lo[3], const int64_t hi[3], double* out, double* partial,
                  int64_t ncells) {
  HIP_TRY(sync_exec(s));  // steps of a batch or a parent write these fields on their streams
  switch (s->g.dtype) {
    case GMES_F32: sq_launch<float>(s, c, lo, hi, partial); break;
    case GMES_F64: sq_launch<double>(s, c, lo, hi, partial); break;
    case GMES_C64: sq_launch<cplx<float>>(s, c, lo, hi, partial); break;
    default: sq_launch<cplx<double>>(s, c, lo, hi, partial); break;
  }
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpyAsync(out, partial + sq_blocks(ncells), sizeof(double), hipMemcpyDeviceToHost, s->stream));
  HIP_TRY(hipStreamSynchronize(s->stream));
  return GMES_OK;
}

}  // namespace

// =============================================================== C-ABI
extern "C" {

const char* gmes_last_error(void) { return g_err; }
int gmes_abi_version(void) { return GMES_ABI_VERSION; }

int gmes_device_count(int32_t* count) {
  ApiGuard api;
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) n = 0;
  *count = n;
  return GMES_OK;
}

int gmes_sim_create(const gmes_grid_desc* desc, gmes_sim** out) {
  ApiGuard api;
  if (!desc || !out) return set_error(GMES_EINVAL, "null argument");
  if (desc->dtype < GMES_F32 || desc->dtype > GMES_C128) return set_error(GMES_ETYPE, "bad dtype");
  if (desc->nx < 1 || desc->ny < 1 || desc->nz < 1) return set_error(GMES_EINVAL, "grid sizes must be positive");
  // Kernels index a component with 32-bit offsets (and ADE cell lists hold
  // 32-bit cells): refuse any component of 2^31 device elements or more,
  // before touching the device.
  for (int c = 0; c < 6; ++c) {
    if (!((desc->active >> c) & 1u)) continue;
    const int64_t ext[3] = {(int64_t)desc->nx + (c % 3 != 0), (int64_t)desc->ny + (c % 3 != 1),
                            (int64_t)desc->nz + (c % 3 != 2)};
    const int64_t row = ext[2] >= 32 && !packed_rows(desc) ? (ext[2] + 31) / 32 * 32 : ext[2];
    const double elems = 2.0 * kPad + (double)ext[0] * (double)ext[1] * (double)row;
    if (elems >= 2147483648.0)
      return set_error(GMES_EINVAL, "component %d would hold %.0f device elements; the limit is 2^31 - 1", c, elems);
  }
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return set_error(GMES_EDEVICE, "no GPU visible");
  if (desc->device < 0 || desc->device >= ndev) return set_error(GMES_EINVAL, "bad device ordinal");
  HIP_TRY(hipSetDevice(desc->device));
  gmes_sim* s = new gmes_sim();
  stage_sims(1);
  known_sim(s, true);
  s->g = *desc;
  s->device = desc->device;
  s->complex_ = desc->dtype == GMES_C64 || desc->dtype == GMES_C128;
  s->fp64 = desc->dtype == GMES_F64 || desc->dtype == GMES_C128;
  s->esize = (s->fp64 ? 8 : 4) * (s->complex_ ? 2 : 1);
  const int64_t n[3] = {desc->nx, desc->ny, desc->nz};
  // 3-D sims with rows under 256 cells store their rows back to back:
  // with 128-byte lines, padding short rows to 32 words left a part-used
  // line at every row end (the batched 64-instance workload's 3-D main
  // launches: 1.112 to 1.049 ms (E), 1.058 to 1.002 ms (H) unpadded; the
  // c64 dispersive cell's E launch 0.558 to 0.491 ms); their single-sim
  // launches then take flat blocks (tile_of).
  s->packed = packed_rows(desc);
  for (int c = 0; c < 6; ++c) {
    if (!active(s, c)) {
      s->shape[c][0] = s->shape[c][1] = s->shape[c][2] = 1;
    } else {
      for (int a = 0; a < 3; ++a) s->shape[c][a] = n[a] + 1;
      s->shape[c][c % 3] = n[c % 3];
    }
    s->ncell[c] = s->shape[c][0] * s->shape[c][1] * s->shape[c][2];
  }
  for (int c = 0; c < 6; ++c) {
    const int64_t s0 = s->shape[c][0], s1 = s->shape[c][1], s2 = s->shape[c][2];
    if (is_2z(s) && active(s, c)) {  // one piece per z plane
      const bool padded = n[1] >= 31;
      const int64_t row = padded ? (n[1] + 32) / 32 * 32 : n[1] + 1;  // the same for every component
      s->pitch[c] = 1;
      s->pi[c] = (int32_t)row;
      s->pk[c] = (int32_t)std::min<int64_t>(s0 * row, INT32_MAX);
      s->koff[c] = padded && (c == GMES_HX || c == GMES_HZ) ? 1 : 0;
      s->dsize[c] = 2 * kPad + s0 * row * s2;
    } else {
      const bool padded = s2 >= 32 && !s->packed;
      const int64_t row = padded ? (s2 + 31) / 32 * 32 : s2;
      s->pitch[c] = (int32_t)row;
      s->pi[c] = (int32_t)std::min<int64_t>(s1 * row, INT32_MAX);
      s->pk[c] = 1;
      s->koff[c] = padded && (c == GMES_HX || c == GMES_HY) ? 1 : 0;
      s->dsize[c] = 2 * kPad + s0 * s1 * row;
    }
    if (s->dsize[c] >= (int64_t(1) << 31)) {
      known_sim(s, false);
      delete s;
      stage_sims(-1);
      return set_error(GMES_EINVAL, "component %d has more than 2^31 cells", c);
    }
  }
  int rc = GMES_OK;
  for (int c = 0; c < 6 && !rc; ++c) {
    rc = dev_alloc(s, &s->f[c], (size_t)(s->dsize[c] * s->esize));
    if (!rc && hipMemset(s->f[c], 0, (size_t)(s->dsize[c] * s->esize)) != hipSuccess)
      rc = set_error(GMES_EDEVICE, "hipMemset failed");
  }
  if (!rc) rc = dev_alloc(s, (void**)&s->d_clock, sizeof(Ctl));
  if (!rc && hipMemset(s->d_clock, 0, sizeof(Ctl)) != hipSuccess) rc = set_error(GMES_EDEVICE, "hipMemset failed");
  if (!rc) rc = dev_alloc(s, &s->d_aux_ptrs, 48 * sizeof(void*));
  if (!rc && hipStreamCreate(&s->stream) != hipSuccess) rc = set_error(GMES_EDEVICE, "hipStreamCreate failed");
  if (rc) {
    gmes_sim_destroy(s);
    return rc;
  }
  *out = s;
  return GMES_OK;
}

int gmes_sim_destroy(gmes_sim* s) {
  ApiGuard api;
  if (!s) return GMES_OK;
  // a batch's job tables and graph hold this sim's buffers
  if (s->batch_stream) return set_error(GMES_EINVAL, "sim is a batch member: destroy the batch first");
  (void)hipSetDevice(s->device);
  if (s->stream) (void)hipStreamSynchronize(s->stream);
  // an aux sim is advanced on its parent's stream: drain that too.  The
  // parent's source operations read this grid, so the parent refuses to
  // step from now on.
  if (gmes_sim* p = s->parent) {
    if (p->stream) (void)hipStreamSynchronize(p->stream);
    if (p->batch_stream) (void)hipStreamSynchronize(p->batch_stream);
    for (int i = 0; i < p->naux; ++i)
      if (p->aux[i] == s) p->aux[i] = nullptr;
    p->aux_lost = true;
    ++p->gen;
    destroy_graph(p);
  }
  for (int i = 0; i < s->naux; ++i)
    if (s->aux[i]) s->aux[i]->parent = nullptr;
  destroy_graph(s);
  collect_timing(s);
  sweep_release(s, false);
  for (int c = 0; c < 6; ++c) {
    if (s->f[c]) (void)dev_release(s->f[c]);
    if (s->ids[c]) (void)dev_release(s->ids[c]);
    if (s->ids8[c]) (void)dev_release(s->ids8[c]);
    if (s->pml_state[c]) (void)dev_release(s->pml_state[c]);
  }
  free_ade(s);
  for (auto& d : s->dfts)
    if (d.acc) (void)dev_release(d.acc);
  void* bufs[] = {s->d_recs, s->d_coef, s->d_prof, s->d_prof_off, s->d_ops, s->d_groups, s->d_waves,
                  s->d_aux_ptrs, s->d_probe_cells, s->d_probe_comps, s->d_probe_buf, s->d_clock,
                  s->d_dft_w, s->d_dft_jobs, s->d_sq, s->d_stage};
  for (void* b : bufs)
    if (b) (void)dev_release(b);
  if (s->stream) (void)stream_release(s->stream);
  known_sim(s, false);
  delete s;
  stage_sims(-1);
  return GMES_OK;
}

int gmes_sim_shape(const gmes_sim* s, int32_t c, int64_t shape[3]) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  if (c < 0 || c > 5) return set_error(GMES_EINVAL, "bad component");
  for (int a = 0; a < 3; ++a) shape[a] = s->shape[c][a];
  return GMES_OK;
}

int gmes_sim_footprint(const gmes_sim* s, int64_t* bytes) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  *bytes = s->bytes;
  return GMES_OK;
}

int gmes_sim_set_materials(gmes_sim* s, const gmes_mat_rec* recs, int32_t nrec, const double* coef,
                           int64_t ncoef) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  if (nrec < 1 || nrec > 65536) return set_error(GMES_EINVAL, "record count must be in [1, 65536]");
  if (ncoef < 0) return set_error(GMES_EINVAL, "negative coefficient count");
  s->recs.assign(recs, recs + nrec);
  s->coef.assign(coef, coef + ncoef);
  for (int r = 0; r < nrec; ++r) {
    const gmes_mat_rec& m = recs[r];
    if (m.cls < 0 || m.cls >= GMES_NCLS) return set_error(GMES_EINVAL, "record %d: bad class", r);
    if (m.n1 < 0 || m.n2 < 0) return set_error(GMES_EINVAL, "record %d: bad pole count", r);
    int64_t need = 0;
    switch (m.cls) {
      case GMES_CLS_DRUDE: need = 3 * (int64_t)m.n1 + 3; break;
      case GMES_CLS_DCP_ADE: need = 3 * (int64_t)m.n1 + 5 * (int64_t)m.n2 + 4; break;
      case GMES_CLS_DCP_PLRC: need = 3 * (int64_t)m.n1 + 6 * (int64_t)m.n2 + 3; break;
      case GMES_CLS_DM2: need = 2 * (int64_t)m.n1 + 6; break;
      default: break;
    }
    if (need && (m.coef_off < 0 || m.coef_off + need > ncoef))
      return set_error(GMES_EINVAL, "record %d: coefficients out of the pool", r);
    if (m.cls == GMES_CLS_DM2 && s->complex_) return set_error(GMES_EINVAL, "Dm2 class supports real fields only");
    if (m.cls == GMES_CLS_DM2 && (m.n1 < 1 || m.n1 > kDm2Max))
      return set_error(GMES_EINVAL, "record %d: DM2 supports 1..%d transitions", r, kDm2Max);
    if ((m.cls == GMES_CLS_CPML || m.cls == GMES_CLS_UPML) && (m.prof < 0 || m.prof >= 64))
      return set_error(GMES_EINVAL, "record %d: bad profile set", r);
    if (m.cls != GMES_CLS_DUMMY && m.cls != GMES_CLS_CONST && !(m.eps_mu != 0.0))
      return set_error(GMES_EINVAL, "record %d: zero permittivity/permeability", r);
  }
  s->committed = false;
  return GMES_OK;
}

int gmes_sim_set_material_ids(gmes_sim* s, int32_t c, const uint16_t* ids, int64_t count) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  if (c < 0 || c > 5) return set_error(GMES_EINVAL, "bad component");
  if (count != s->ncell[c]) return set_error(GMES_EINVAL, "id count %lld != cells %lld", (long long)count,
                                             (long long)s->ncell[c]);
  s->host_ids[c].assign(ids, ids + count);
  if (!s->ids[c]) {
    int rc = dev_alloc(s, (void**)&s->ids[c], (size_t)s->dsize[c] * sizeof(uint16_t));
    if (rc) return rc;
  }
  // the device layout (pads included) is assembled on the host and copied
  // in one contiguous transfer: a strided 2-D copy would wait for every
  // kernel running on the device, including other sims' batches
  std::vector<uint16_t> dev((size_t)s->dsize[c], 0);
  const int64_t n0 = s->shape[c][0], n1 = s->shape[c][1], n2 = s->shape[c][2];
  for (int64_t i = 0; i < n0; ++i) {
    const uint16_t* h = ids + i * n1 * n2;
    if (s->pk[c] == 1) {
      for (int64_t j = 0; j < n1; ++j)
        memcpy(dev.data() + dev_index(s, c, i, j, 0), h + j * n2, (size_t)n2 * sizeof(uint16_t));
    } else {  // collapsed z: rows along j, a plane for each k
      for (int64_t k = 0; k < n2; ++k) {
        uint16_t* d = dev.data() + dev_index(s, c, i, 0, k);
        for (int64_t j = 0; j < n1; ++j) d[j] = h[j * n2 + k];
      }
    }
  }
  HIP_TRY(hipMemcpy(s->ids[c], dev.data(), dev.size() * sizeof(uint16_t), hipMemcpyHostToDevice));
  s->committed = false;
  return GMES_OK;
}

int gmes_sim_set_profile(gmes_sim* s, int32_t p, int32_t c, int32_t axis, const double* vals, int32_t n,
                         int32_t width) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  if (p < 0 || p >= 64 || c < 0 || c > 5 || axis < 0 || axis > 2)
    return set_error(GMES_EINVAL, "bad profile address");
  if (n != s->shape[c][axis] || (width != 3 && width != 6)) return set_error(GMES_EINVAL, "bad profile size");
  s->prof_host[p][c][axis].assign(vals, vals + (size_t)n * width);
  s->prof_w[p][c][axis] = width;
  s->nprof = std::max(s->nprof, p + 1);
  s->committed = false;
  return GMES_OK;
}

int gmes_sim_commit(gmes_sim* s) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  if (s->recs.empty()) return set_error(GMES_EINVAL, "materials not set");
  HIP_TRY(hipSetDevice(s->device));
  HIP_TRY(sync_exec(s));
  s->committed = false;
  sweep_release(s);
  free_ade(s);
  s->ade_on_ghost_source = false;
  std::vector<int64_t> counts[6];  // cells per record; empty: an id is out of range
  host_parallel(6, s->ncell[0] + s->ncell[2] + s->ncell[5], [&](int c) {
    if (!active(s, c)) return;
    counts[c].assign(s->recs.size(), 0);
    for (const uint16_t id : s->host_ids[c]) {
      if (id >= counts[c].size()) {
        counts[c].clear();
        return;
      }
      ++counts[c][id];
    }
  });
  for (int c = 0; c < 6; ++c) {
    for (int k = 0; k < GMES_NCLS; ++k) s->has_cls[c][k] = false;
    if (!active(s, c)) continue;
    const std::vector<uint16_t>& ids = s->host_ids[c];
    if ((int64_t)ids.size() != s->ncell[c]) return set_error(GMES_EINVAL, "ids of component %d not set", c);
    const int64_t s0 = s->shape[c][0], sy = s->shape[c][1], sz = s->shape[c][2];
    std::vector<std::vector<int32_t>> cells(GMES_NCLS);
    std::vector<std::vector<uint16_t>> recs(GMES_NCLS);
    std::vector<int> words(GMES_NCLS, 0);
    // records in use
    const std::vector<int64_t>& count = counts[c];
    if (count.empty()) return set_error(GMES_ERANGE, "material id out of range");
    bool any_ade = false;
    for (size_t id = 0; id < s->recs.size(); ++id) {
      if (!count[id]) continue;
      const gmes_mat_rec& r = s->recs[id];
      s->has_cls[c][r.cls] = true;
      if (r.cls >= GMES_CLS_DRUDE) {
        if (c >= 3) return set_error(GMES_EINVAL, "dispersive class on a magnetic component");
        any_ade = true;
        words[r.cls] = std::max(words[r.cls], state_words(r));
      }
      if (r.cls == GMES_CLS_CPML || r.cls == GMES_CLS_UPML) {
        const int w = r.cls == GMES_CLS_CPML ? 3 : 6;
        for (int a = 0; a < 3; ++a)
          if ((int64_t)s->prof_host[r.prof][c][a].size() != s->shape[c][a] * w)
            return set_error(GMES_EINVAL, "profile %d of component %d axis %d missing", r.prof, c, a);
      }
    }
    // Ghost planes must be Dummy: a kernel never reads past them
    // (gmes/fdtd.py:365-366 and the analogous lines).  E: the last plane
    // of each transverse axis; H: plane 0.
    const int64_t n3[3] = {s0, sy, sz};
    for (int a = 0; a < 3; ++a) {
      if (a == c % 3) continue;
      const int64_t g = c < 3 ? n3[a] - 1 : 0;
      int64_t ix[3];
      for (ix[0] = 0; ix[0] < s0; ++ix[0])
        for (ix[1] = 0; ix[1] < sy; ++ix[1]) {
          if (a == 0 && ix[0] != g) break;
          if (a == 1 && ix[1] != g) continue;
          for (ix[2] = (a == 2 ? g : 0); ix[2] < (a == 2 ? g + 1 : sz); ++ix[2]) {
            const int64_t x = (ix[0] * sy + ix[1]) * sz + ix[2];
            if (s->recs[ids[x]].cls != GMES_CLS_DUMMY)
              return set_error(GMES_EINVAL, "component %d: ghost cell %lld is not Dummy", c, (long long)x);
          }
        }
    }
    if (any_ade)
      for (int64_t x = 0; x < s->ncell[c]; ++x) {
        const gmes_mat_rec& r = s->recs[ids[x]];
        if (r.cls >= GMES_CLS_DRUDE) {
          cells[r.cls].push_back((int32_t)x);
          recs[r.cls].push_back(ids[x]);
          if (c < 3 && on_ghost_copy_plane(s, c, x, true, false)) s->ade_on_ghost_source = true;
        }
      }
    // full-grid CPML (2 words) / UPML (1 word) state
    const int pw = s->has_cls[c][GMES_CLS_CPML] ? 2 : (s->has_cls[c][GMES_CLS_UPML] ? 1 : 0);
    if (s->pml_state[c]) { dev_free(s, s->pml_state[c], 0); s->pml_state[c] = nullptr; }
    if (pw) {
      const size_t b = (size_t)pw * s->dsize[c] * s->esize;
      int rc = dev_alloc(s, &s->pml_state[c], b);
      if (rc) return rc;
      HIP_TRY(hipMemset(s->pml_state[c], 0, b));
    }
    for (int k = GMES_CLS_DRUDE; k < GMES_NCLS; ++k) {
      AdeList& L = s->ade[c][k];
      L.n = (int64_t)cells[k].size();
      if (!L.n) continue;
      L.nstate = words[k];
      HIP_TRY(dev_malloc(s->device, (void**)&L.cell, L.n * sizeof(int32_t)));
      HIP_TRY(dev_malloc(s->device, (void**)&L.rec, L.n * sizeof(uint16_t)));
      const size_t sb = std::max<size_t>(1, (size_t)L.nstate * L.n * ade_word(s, k));
      HIP_TRY(dev_malloc(s->device, &L.state, sb));
      s->bytes += L.n * 6 + (int64_t)sb;
      HIP_TRY(hipMemcpy(L.cell, cells[k].data(), L.n * sizeof(int32_t), hipMemcpyHostToDevice));
      HIP_TRY(hipMemcpy(L.rec, recs[k].data(), L.n * sizeof(uint16_t), hipMemcpyHostToDevice));
      HIP_TRY(hipMemset(L.state, 0, sb));
    }
  }
  if (s->d_recs) { (void)dev_release(s->d_recs); s->d_recs = nullptr; }
  if (s->d_coef) { (void)dev_release(s->d_coef); s->d_coef = nullptr; }
  if (s->d_prof) { (void)dev_release(s->d_prof); s->d_prof = nullptr; }
  if (s->d_prof_off) { (void)dev_release(s->d_prof_off); s->d_prof_off = nullptr; }
  int rc = s->fp64 ? upload_tables<double>(s) : upload_tables<float>(s);
  if (rc) return rc;
  if ((rc = upload_byte_ids(s))) return rc;
  // the coordinate runs where no CPML record's psi can be nonzero
  for (int a = 0; a < 3; ++a) {
    int lo = 0, hi = 0x7FFF;
    bool any = false;
    for (const gmes_mat_rec& r : s->recs) {
      if (r.cls != GMES_CLS_CPML) continue;
      const int32_t run = (r.prof >= 0 && r.prof < s->nprof) ? zero_c_run(s, r.prof, a) : 0;
      any = true;
      lo = std::max(lo, (int)(run & 0xFFFF));
      hi = std::min(hi, (int)(run >> 16));
    }
    s->prun[a] = (any && lo < hi) ? (lo | (hi << 16)) : 0;
  }
  profile_prefetch(s);
  upml_box(s);
  upml_rows(s);
  if ((rc = sweep_build(s))) return rc;
  if ((rc = sweep_sources(s))) return rc;
  s->committed = true;
  destroy_graph(s);
  decide_fusion(s);
  return s->dfts.empty() ? GMES_OK : upload_dft_jobs(s);  // the jobs hold the buffers' addresses
}

int gmes_sim_set_sources(gmes_sim* s, const gmes_src_op* ops, int64_t nops, int32_t nwaves) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  if (nops < 0 || nwaves < 0) return set_error(GMES_EINVAL, "negative count");
  if (nops > (1 << 30)) return set_error(GMES_EINVAL, "too many source operations");
  for (int64_t i = 0; i < nops; ++i) {
    const gmes_src_op& o = ops[i];
    if (o.comp < 0 || o.comp > 5 || !active(s, o.comp)) return set_error(GMES_EINVAL, "source on an inactive component");
    if (o.cell < 0 || o.cell >= s->ncell[o.comp]) return set_error(GMES_ERANGE, "field index is out of bounds");
    if (o.kind == GMES_SRC_SET || o.kind == GMES_SRC_SUB) {
      if (o.wave < 0 || o.wave >= nwaves) return set_error(GMES_EINVAL, "bad waveform row");
    } else if (o.kind == GMES_SRC_AUX_ADD || o.kind == GMES_SRC_AUX_SUB) {
      if (o.aux < 0 || o.aux >= s->naux) return set_error(GMES_EINVAL, "auxiliary grid %d not attached", o.aux);
      if (o.wave < -1 || o.wave >= nwaves) return set_error(GMES_EINVAL, "bad envelope row");
      if (o.aux_comp < 0 || o.aux_comp > 5) return set_error(GMES_EINVAL, "bad aux component");
      const gmes_sim* a = s->aux[o.aux];
      if (!((a->g.active >> o.aux_comp) & 1u)) return set_error(GMES_EINVAL, "inactive aux component");
      if (o.i0 < 0 || o.i1 < 0 || o.i0 >= a->ncell[o.aux_comp] || o.i1 >= a->ncell[o.aux_comp])
        return set_error(GMES_ERANGE, "aux sample index out of bounds");
    } else {
      return set_error(GMES_EINVAL, "bad source kind");
    }
  }
  HIP_TRY(hipSetDevice(s->device));
  HIP_TRY(sync_exec(s));
  s->ops.assign(ops, ops + nops);
  s->nwaves = nwaves;
  int rc = s->fp64 ? upload_sources<double>(s) : upload_sources<float>(s);
  if (!rc && s->committed) rc = sweep_sources(s);
  destroy_graph(s);
  decide_fusion(s);
  return rc;
}

int gmes_sim_set_waveforms(gmes_sim* s, int64_t step0, int64_t nsteps, const double* values) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  if (nsteps < 0) return set_error(GMES_EINVAL, "negative step count");
  HIP_TRY(hipSetDevice(s->device));
  const int64_t need = std::max<int64_t>(1, (int64_t)s->nwaves * nsteps * 2);
  HIP_TRY(sync_exec(s));
  if (need > s->wave_cap) {
    if (s->d_waves) dev_free(s, s->d_waves, (size_t)s->wave_cap * sizeof(double));
    s->d_waves = nullptr;
    int rc = dev_alloc(s, (void**)&s->d_waves, (size_t)need * sizeof(double));
    if (rc) return rc;
    s->wave_cap = need;
    destroy_graph(s);
  }
  if (s->nwaves && nsteps)
    HIP_TRY(hipMemcpy(s->d_waves, values, (size_t)s->nwaves * nsteps * 2 * sizeof(double), hipMemcpyHostToDevice));
  s->wave_step0 = step0;
  s->wave_n = nsteps;
  return ctl_write(s);
}

int gmes_sim_attach_aux(gmes_sim* s, gmes_sim* aux, int32_t* slot) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  if (!aux || aux == s) return set_error(GMES_EINVAL, "bad auxiliary sim");
  if (s->naux >= 8) return set_error(GMES_EINVAL, "too many auxiliary grids");
  if (aux->g.dtype != s->g.dtype) return set_error(GMES_ETYPE, "aux dtype mismatch");
  if (aux->device != s->device) return set_error(GMES_EINVAL, "aux sim on another device");
  if (aux->naux) return set_error(GMES_EINVAL, "an auxiliary grid cannot have its own");
  if (aux->parent) return set_error(GMES_EINVAL, "auxiliary grid already attached");
  HIP_TRY(hipSetDevice(s->device));
  HIP_TRY(sync_exec(s));
  if (s->sweep_1d || s->sweep_2d) sweep_release(s);  // a 1-D or 2-D sim with one takes two-kernel steps: no second buffers
  s->aux[s->naux] = aux;
  aux->parent = s;
  *slot = s->naux++;
  if (int rc = aux_pointers(s)) return rc;
  destroy_graph(s);
  return s->committed ? sweep_sources(s) : GMES_OK;
}

int gmes_sim_add_probe(gmes_sim* s, int32_t c, int64_t cell, int32_t* id) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  if (c < 0 || c > 5 || !active(s, c) || cell < 0 || cell >= s->ncell[c])
    return set_error(GMES_ERANGE, "probe index out of bounds");
  if (s->step != s->probe_base) return set_error(GMES_EINVAL, "read pending probe values first");
  HIP_TRY(hipSetDevice(s->device));
  HIP_TRY(sync_exec(s));
  s->probes.push_back({c, cell});
  std::vector<int64_t> cells;
  std::vector<int32_t> comps;
  for (auto& p : s->probes) { cells.push_back(dev_flat(s, p.comp, p.cell)); comps.push_back(p.comp); }
  if (s->d_probe_cells) (void)dev_release(s->d_probe_cells);
  if (s->d_probe_comps) (void)dev_release(s->d_probe_comps);
  if (s->d_probe_buf) (void)dev_release(s->d_probe_buf);
  s->d_probe_buf = nullptr;
  s->probe_cap = 0;
  HIP_TRY(dev_malloc(s->device, (void**)&s->d_probe_cells, cells.size() * sizeof(int64_t)));
  HIP_TRY(dev_malloc(s->device, (void**)&s->d_probe_comps, comps.size() * sizeof(int32_t)));
  HIP_TRY(hipMemcpy(s->d_probe_cells, cells.data(), cells.size() * sizeof(int64_t), hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(s->d_probe_comps, comps.data(), comps.size() * sizeof(int32_t), hipMemcpyHostToDevice));
  *id = (int32_t)s->probes.size() - 1;
  destroy_graph(s);
  decide_fusion(s);
  return GMES_OK;
}

int gmes_sim_read_probe(gmes_sim* s, int32_t id, double* out, int64_t max, int64_t* n) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  if (id < 0 || id >= (int32_t)s->probes.size()) return set_error(GMES_EINVAL, "bad probe id");
  HIP_TRY(hipSetDevice(s->device));
  HIP_TRY(sync_exec(s));
  std::vector<int64_t>& cur = s->probe_read;
  cur.resize(s->probes.size(), 0);
  const int64_t avail = s->probe_n - cur[id];
  const int64_t m = std::min(avail, max);
  if (m > 0)
    HIP_TRY(hipMemcpy(out, s->d_probe_buf + (id * s->probe_cap + cur[id]) * 2, m * 2 * sizeof(double),
                      hipMemcpyDeviceToHost));
  cur[id] += m;
  *n = m;
  bool all = true;
  for (size_t p = 0; p < cur.size(); ++p) all = all && cur[p] == s->probe_n;
  if (all) {
    s->probe_base = s->step;
    s->probe_n = 0;
    std::fill(cur.begin(), cur.end(), 0);
    return ctl_write(s);
  }
  return GMES_OK;
}

int gmes_sim_add_dft(gmes_sim* s, int32_t c, const int64_t lo[3], const int64_t hi[3], int32_t nfreq,
                     int32_t decim, int32_t* id) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  if (c < 0 || c > 5 || !active(s, c)) return set_error(GMES_EINVAL, "DFT of an inactive component");
  if (nfreq < 1 || decim < 1) return set_error(GMES_EINVAL, "nfreq and decim must be positive");
  if (!s->dfts.empty() && nfreq != s->dft_nfreq)
    return set_error(GMES_EINVAL, "all DFT monitors of a sim share one frequency list");
  gmes_sim::Dft d{};
  d.comp = c;
  d.ncells = 1;
  for (int a = 0; a < 3; ++a) {
    if (lo[a] < 0 || hi[a] > s->shape[c][a] || hi[a] <= lo[a]) return set_error(GMES_ERANGE, "DFT box out of bounds");
    d.lo[a] = lo[a];
    d.n[a] = hi[a] - lo[a];
    d.ncells *= d.n[a];
  }
  d.nfreq = nfreq;
  d.decim = decim;
  HIP_TRY(hipSetDevice(s->device));
  HIP_TRY(sync_exec(s));
  // sums [nfreq][ncells][re, im], then their compensations, same layout
  const size_t bytes = 2 * (size_t)nfreq * d.ncells * 2 * sizeof(double);
  HIP_TRY(dev_malloc(s->device, (void**)&d.acc, bytes));
  HIP_TRY(hipMemset(d.acc, 0, bytes));
  s->dfts.push_back(d);
  s->dft_nfreq = nfreq;
  s->bytes += (int64_t)bytes;
  *id = (int32_t)s->dfts.size() - 1;
  destroy_graph(s);
  return upload_dft_jobs(s);
}

int gmes_sim_set_dft_weights(gmes_sim* s, int64_t step0, int64_t nsteps, const double* w) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  if (s->dfts.empty()) return set_error(GMES_EINVAL, "no DFT monitor");
  if (nsteps < 0) return set_error(GMES_EINVAL, "negative step count");
  HIP_TRY(hipSetDevice(s->device));
  HIP_TRY(sync_exec(s));
  const int64_t need = std::max<int64_t>(1, nsteps * s->dft_nfreq * 4);
  if (need > s->dft_w_cap) {
    if (s->d_dft_w) HIP_TRY(dev_release(s->d_dft_w));
    s->d_dft_w = nullptr;
    HIP_TRY(dev_malloc(s->device, (void**)&s->d_dft_w, (size_t)need * sizeof(double)));
    s->dft_w_cap = need;
    int rc = upload_dft_jobs(s);  // the jobs hold the weight pointer
    if (rc) return rc;
    ++s->gen;
  }
  if (nsteps) HIP_TRY(hipMemcpy(s->d_dft_w, w, (size_t)nsteps * s->dft_nfreq * 4 * sizeof(double), hipMemcpyHostToDevice));
  s->dft_step0 = step0;
  s->dft_n = nsteps;
  return ctl_write(s);
}

int gmes_sim_read_dft(gmes_sim* s, int32_t id, double* out, int64_t count) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  if (id < 0 || id >= (int32_t)s->dfts.size()) return set_error(GMES_EINVAL, "bad DFT id");
  const auto& d = s->dfts[id];
  if (count != (int64_t)d.nfreq * d.ncells * 2) return set_error(GMES_EINVAL, "size mismatch");
  HIP_TRY(hipSetDevice(s->device));
  HIP_TRY(sync_exec(s));
  HIP_TRY(hipMemcpy(out, d.acc, (size_t)count * sizeof(double), hipMemcpyDeviceToHost));
  return GMES_OK;
}

// Whether a component's device layout is the host's, after kPad elements.
static bool dense_layout(const gmes_sim* s, int c) {
  const int64_t s1 = s->shape[c][1], s2 = s->shape[c][2];
  return s->koff[c] == 0 && (s2 == 1 || s->pk[c] == 1) && s->pitch[c] == s2 && s->pi[c] == s1 * s2;
}

static LayoutArgs layout_of(const gmes_sim* s, int c) {
  return {s->ncell[c], (int)s->shape[c][1], (int)s->shape[c][2], s->pi[c], s->pitch[c], s->pk[c]};
}

// The staging buffer of field reads and writes of padded rows, at least
// `bytes` long (grown on demand; the sim's stream is idle when it grows).
static int stage_reserve(gmes_sim* s, int64_t bytes) {
  if (bytes <= s->stage_cap) return GMES_OK;
  HIP_TRY(sync_exec(s));
  if (s->d_stage) dev_free(s, s->d_stage, (size_t)s->stage_cap);
  s->d_stage = nullptr;
  s->stage_cap = 0;
  for (int c = 0; c < 6; ++c) bytes = std::max(bytes, s->ncell[c] * s->esize);  // once for all components
  int rc = dev_alloc(s, &s->d_stage, (size_t)bytes);
  if (rc) return rc;
  s->stage_cap = bytes;
  return GMES_OK;
}

// Copies contiguous device memory from or to the caller's array, on the stream
// of s, and waits.  The caller's memory is pageable: the runtime copies it
// through its own buffers on one thread.  Large copies go through pinned
// buffers here, a few threads each moving a part of the array while the next
// piece is on the link (67 MB: reading 17.3 -> 37 GB/s, writing 28 -> 36; 11 MB:
// reading 17.2 -> 26, writing 27 -> 25.5; below, starting the threads costs as
// much as it gains).
constexpr int64_t kStageRead = 8 << 20, kStageWrite = 16 << 20;
static int host_copy(gmes_sim* s, char* dev, char* host, int64_t bytes, bool to_device) {
  void* const pinned = bytes >= (to_device ? kStageWrite : kStageRead) ? stage_lease() : nullptr;
  if (!pinned) {
    HIP_TRY(to_device ? hipMemcpyAsync(dev, host, (size_t)bytes, hipMemcpyHostToDevice, s->stream)
                      : hipMemcpyAsync(host, dev, (size_t)bytes, hipMemcpyDeviceToHost, s->stream));
    HIP_TRY(sync_exec(s));
    return GMES_OK;
  }
  constexpr int64_t piece = kStageBytes / kStageThreads / 2;
  std::atomic<int> error{(int)hipSuccess};
  auto part = [&](int t) {
    const int64_t lo = bytes / 64 * t / kStageThreads * 64,
                  hi = t == kStageThreads - 1 ? bytes : bytes / 64 * (t + 1) / kStageThreads * 64;
    char* const buf = static_cast<char*>(pinned) + 2 * piece * t;
    hipEvent_t done[2] = {};
    auto ok = [&](hipError_t e) {
      if (e != hipSuccess) error = (int)e;
      return e == hipSuccess;
    };
    auto move = [&](int64_t k) {  // piece k of the part over the link
      const int64_t o = lo + k * piece, n = std::min(piece, hi - o);
      char* const b = buf + (k & 1) * piece;
      return ok(to_device ? hipMemcpyAsync(dev + o, b, (size_t)n, hipMemcpyHostToDevice, s->stream)
                          : hipMemcpyAsync(b, dev + o, (size_t)n, hipMemcpyDeviceToHost, s->stream)) &&
             ok(hipEventRecord(done[k & 1], s->stream));
    };
    const int64_t n = (hi - lo + piece - 1) / piece;
    bool good = ok(hipSetDevice(s->device));
    for (hipEvent_t& e : done) good = good && ok(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    if (good && !to_device && n > 0) good = move(0);
    for (int64_t k = 0; k < n && good; ++k) {
      char* const h = host + lo + k * piece;
      const size_t m = (size_t)std::min(piece, hi - lo - k * piece);
      if (to_device) {
        if (k >= 2) good = ok(hipEventSynchronize(done[k & 1]));
        if (good) memcpy(buf + (k & 1) * piece, h, m);
        good = good && move(k);
      } else {
        if (k + 1 < n) good = move(k + 1);
        good = good && ok(hipEventSynchronize(done[k & 1]));
        if (good) memcpy(h, buf + (k & 1) * piece, m);
      }
    }
    if (!good) (void)hipStreamSynchronize(s->stream);
    for (hipEvent_t e : done)
      if (e) (void)hipEventDestroy(e);
  };
  host_parallel(kStageThreads, bytes, part);
  const hipError_t e = hipStreamSynchronize(s->stream);
  stage_return(pinned);
  if (e != hipSuccess) error = (int)e;
  HIP_TRY((hipError_t)error.load());
  HIP_TRY(sync_exec(s));
  return GMES_OK;
}

int gmes_sim_write_field(gmes_sim* s, int32_t c, const void* host, int64_t bytes) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  if (c < 0 || c > 5) return set_error(GMES_EINVAL, "bad component");
  if (bytes != s->ncell[c] * s->esize) return set_error(GMES_EINVAL, "size mismatch");
  HIP_TRY(hipSetDevice(s->device));
  HIP_TRY(sync_exec(s));  // steps queued on the sim's (or its batch's) stream come first
  if (dense_layout(s, c)) {
    return host_copy(s, static_cast<char*>(s->f[c]) + (size_t)kPad * s->esize,
                     const_cast<char*>(static_cast<const char*>(host)), bytes, true);
  }
  // one contiguous upload, then rows moved to their pitched places
  int rc = stage_reserve(s, bytes);
  if (rc) return rc;
  if ((rc = host_copy(s, static_cast<char*>(s->d_stage), const_cast<char*>(static_cast<const char*>(host)), bytes, true)))
    return rc;
  launch_layout_copy(true, s->d_stage, static_cast<char*>(s->f[c]) + (size_t)(kPad - s->koff[c]) * s->esize,
                     layout_of(s, c), s->esize, s->stream);
  HIP_TRY(hipGetLastError());
  HIP_TRY(sync_exec(s));
  return GMES_OK;
}

int gmes_sim_read_field(gmes_sim* s, int32_t c, void* host, int64_t bytes) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  if (c < 0 || c > 5) return set_error(GMES_EINVAL, "bad component");
  if (bytes != s->ncell[c] * s->esize) return set_error(GMES_EINVAL, "size mismatch");
  HIP_TRY(hipSetDevice(s->device));
  HIP_TRY(sync_exec(s));  // steps queued on the sim's (or its batch's) stream come first
  if (dense_layout(s, c)) {
    return host_copy(s, static_cast<char*>(s->f[c]) + (size_t)kPad * s->esize, static_cast<char*>(host), bytes, false);
  }
  // rows packed on the device, then one contiguous download
  int rc = stage_reserve(s, bytes);
  if (rc) return rc;
  launch_layout_copy(false, s->d_stage, static_cast<char*>(s->f[c]) + (size_t)(kPad - s->koff[c]) * s->esize,
                     layout_of(s, c), s->esize, s->stream);
  HIP_TRY(hipGetLastError());
  return host_copy(s, static_cast<char*>(s->d_stage), static_cast<char*>(host), bytes, false);
}

// ---- snapshot / restore
// The blob of a sim: a header (magic, step), the CPML/UPML and ADE state,
// the DFT accumulators, and for every attached auxiliary grid its six
// fields followed by its own blob.  The sim's own six fields are not in
// it: the caller keeps them (gmes_sim_read_field / gmes_sim_write_field).
// Restore sets the step clock back to the snapshot's and drops unread
// probe values, so the next step records and injects at the restored time.
constexpr int64_t kSnapMagic = 0x31504e5353454d47LL;  // "GMESSNP1"

// Arrays laid out like a component are in it in the order of (i, j, k): as
// one piece of device memory, except that collapsed-z modes keep k fastest
// (their device layout is converted), with kPad elements before and after.
struct StateBlock {
  void* dev;
  size_t bytes;  // in the blob
  int comp;      // component whose layout it has, -1: plain bytes
  int words;
};

static void grid_block(const gmes_sim* s, std::vector<StateBlock>& out, void* dev, int c, int words) {
  if (is_2z(s)) out.push_back({dev, (size_t)words * (2 * kPad + s->ncell[c]) * s->esize, c, words});
  else out.push_back({dev, (size_t)words * s->dsize[c] * s->esize, -1, words});
}

static int block_copy(const gmes_sim* s, const StateBlock& b, char* p, bool save) {
  if (b.comp < 0) {
    if (save) HIP_TRY(hipMemcpy(p, b.dev, b.bytes, hipMemcpyDeviceToHost));
    else HIP_TRY(hipMemcpy(b.dev, p, b.bytes, hipMemcpyHostToDevice));
    return GMES_OK;
  }
  const int c = b.comp;
  const size_t e = (size_t)s->esize;
  const int64_t n1 = s->shape[c][1], n2 = s->shape[c][2];
  std::vector<char> dev((size_t)b.words * s->dsize[c] * e, 0);
  if (save) {
    HIP_TRY(hipMemcpy(dev.data(), b.dev, dev.size(), hipMemcpyDeviceToHost));
    memset(p, 0, b.bytes);
  }
  for (int w = 0; w < b.words; ++w)
    for (int64_t x = 0; x < s->ncell[c]; ++x) {
      char* d = dev.data() + (w * s->dsize[c] + dev_index(s, c, x / (n1 * n2), x / n2 % n1, x % n2)) * e;
      char* h = p + (w * (2 * kPad + s->ncell[c]) + kPad + x) * e;
      if (save) memcpy(h, d, e);
      else memcpy(d, h, e);
    }
  if (!save) HIP_TRY(hipMemcpy(b.dev, dev.data(), dev.size(), hipMemcpyHostToDevice));
  return GMES_OK;
}

static void state_blocks(gmes_sim* s, std::vector<StateBlock>& out) {
  for (int c = 0; c < 6; ++c) {
    if (s->pml_state[c]) grid_block(s, out, s->pml_state[c], c, s->has_cls[c][GMES_CLS_CPML] ? 2 : 1);
    for (int k = GMES_CLS_DRUDE; k < GMES_NCLS; ++k)
      if (s->ade[c][k].n)
        out.push_back({s->ade[c][k].state, (size_t)s->ade[c][k].nstate * s->ade[c][k].n * ade_word(s, k), -1, 0});
  }
  for (auto& d : s->dfts) out.push_back({d.acc, 2 * (size_t)d.nfreq * d.ncells * 2 * sizeof(double), -1, 0});
}

// the fields of an auxiliary grid
static void field_blocks(gmes_sim* a, std::vector<StateBlock>& out) {
  for (int c = 0; c < 6; ++c) {
    if (active(a, c)) grid_block(a, out, a->f[c], c, 1);
    else out.push_back({a->f[c], (size_t)a->dsize[c] * a->esize, -1, 1});
  }
}

static int64_t blob_bytes(gmes_sim* s) {
  std::vector<StateBlock> b;
  state_blocks(s, b);
  for (int i = 0; i < s->naux; ++i)
    if (s->aux[i]) field_blocks(s->aux[i], b);
  int64_t t = 2 * sizeof(int64_t);
  for (auto& x : b) t += (int64_t)x.bytes;
  for (int i = 0; i < s->naux; ++i)
    if (s->aux[i]) t += blob_bytes(s->aux[i]);
  return t;
}

// Copies the blob of s to or from host memory at p (the streams of s are
// idle); returns the bytes done.
static int blob_copy(gmes_sim* s, char* p, bool save, int64_t& done) {
  int64_t head[2] = {kSnapMagic, s->step};
  if (save) {
    memcpy(p, head, sizeof head);
  } else {
    memcpy(head, p, sizeof head);
    if (head[0] != kSnapMagic || head[1] < 0) return set_error(GMES_EINVAL, "not a snapshot of this engine");
  }
  done = sizeof head;
  std::vector<StateBlock> b;
  state_blocks(s, b);
  for (auto& x : b) {
    if (int rc = block_copy(s, x, p + done, save)) return rc;
    done += (int64_t)x.bytes;
  }
  for (int i = 0; i < s->naux; ++i) {
    gmes_sim* a = s->aux[i];
    if (!a) continue;
    b.clear();
    field_blocks(a, b);
    for (auto& x : b) {
      if (int rc = block_copy(a, x, p + done, save)) return rc;
      done += (int64_t)x.bytes;
    }
    int64_t sub = 0;
    int rc = blob_copy(a, p + done, save, sub);
    if (rc) return rc;
    done += sub;
  }
  if (!save) {
    s->step = head[1];
    s->probe_base = s->step;
    s->probe_n = 0;
    std::fill(s->probe_read.begin(), s->probe_read.end(), 0);
    Ctl c;
    HIP_TRY(hipMemcpy(&c, s->d_clock, sizeof c, hipMemcpyDeviceToHost));
    c.clock = s->step;
    s->clk_stale = true;
    c.probe_base = s->probe_base;
    c.err = 0;
    HIP_TRY(hipMemcpy(s->d_clock, &c, sizeof c, hipMemcpyHostToDevice));
  }
  return GMES_OK;
}

int gmes_sim_state_bytes(const gmes_sim* s, int64_t* bytes) {
  ApiGuard api;
  if (!s || !bytes) return set_error(GMES_EINVAL, "null argument");
  *bytes = blob_bytes(const_cast<gmes_sim*>(s));
  return GMES_OK;
}

int gmes_sim_snapshot(gmes_sim* s, void* host, int64_t bytes) {
  ApiGuard api;
  if (!s || !host) return set_error(GMES_EINVAL, "null argument");
  if (blob_bytes(s) != bytes) return set_error(GMES_EINVAL, "size mismatch");
  HIP_TRY(hipSetDevice(s->device));
  HIP_TRY(sync_exec(s));
  int64_t done = 0;
  return blob_copy(s, static_cast<char*>(host), true, done);
}

int gmes_sim_restore(gmes_sim* s, const void* host, int64_t bytes) {
  ApiGuard api;
  if (!s || !host) return set_error(GMES_EINVAL, "null argument");
  if (s->parent) return set_error(GMES_EINVAL, "an auxiliary grid is restored with its parent");
  if (blob_bytes(s) != bytes) return set_error(GMES_EINVAL, "size mismatch");
  HIP_TRY(hipSetDevice(s->device));
  HIP_TRY(sync_exec(s));
  int64_t done = 0;
  return blob_copy(s, const_cast<char*>(static_cast<const char*>(host)), false, done);
}

int gmes_sim_field_sum_sq(gmes_sim* s, int32_t c, const int64_t lo[3], const int64_t hi[3], double* out) {
  ApiGuard api;
  int64_t ncells = 0;
  int rc = sq_check(s, c, lo, hi, out, ncells);
  if (rc) return rc;
  HIP_TRY(hipSetDevice(s->device));
  const int64_t need = sq_blocks(ncells) + 1;
  if (need > s->sq_cap) {
    HIP_TRY(sync_exec(s));
    if (s->d_sq) dev_free(s, s->d_sq, (size_t)s->sq_cap * sizeof(double));
    s->d_sq = nullptr;
    s->sq_cap = 0;
    if ((rc = dev_alloc(s, (void**)&s->d_sq, (size_t)need * sizeof(double)))) return rc;
    s->sq_cap = need;
  }
  return sq_run(s, c, lo, hi, out, s->d_sq, ncells);
}

int gmes_sim_field_sum_sq_noalloc(gmes_sim* s, int32_t c, const int64_t lo[3], const int64_t hi[3], double* out) {
  ApiGuard api;
  int64_t ncells = 0;
  int rc = sq_check(s, c, lo, hi, out, ncells);
  if (rc) return rc;
  if (sq_blocks(ncells) > kScratchPartials)
    return set_error(GMES_EINVAL, "box of %lld cells exceeds the no-allocation limit of %lld cells",
                     (long long)ncells, (long long)(kScratchPartials * kSqBlockCells));
  if (s->device < 0 || s->device >= kMaxDevices) return set_error(GMES_EINVAL, "device ordinal beyond %d", kMaxDevices);
  HIP_TRY(hipSetDevice(s->device));
  std::lock_guard<std::mutex> lk(g_scratch_mu[s->device]);
  if (!g_scratch_ptr[s->device]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return set_error(GMES_EDEVICE, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
    g_scratch_ptr[s->device] = static_cast<double*>(p);
  }
  return sq_run(s, c, lo, hi, out, g_scratch_ptr[s->device], ncells);
}

int gmes_sim_step(gmes_sim* s, int64_t nsteps) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  return do_step(s, nsteps);
}

int gmes_sim_sync(gmes_sim* s) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  HIP_TRY(hipSetDevice(s->device));
  HIP_TRY(sync_exec(s));
  Ctl c;
  HIP_TRY(hipMemcpy(&c, s->d_clock, sizeof c, hipMemcpyDeviceToHost));
  if (c.err == 1) return set_error(GMES_ERUNTIME, "Dm2 corrector produced an invalid error");
  if (c.err == 2) return set_error(GMES_ERUNTIME, "Dm2 corrector failed to converge");
  for (int i = 0; i < s->naux; ++i) {
    if (!s->aux[i]) continue;
    int rc = gmes_sim_sync(s->aux[i]);
    if (rc) return rc;
  }
  if (s->timing.on) return collect_timing(s);
  return GMES_OK;
}

int gmes_sim_get_step(const gmes_sim* s, int64_t* step) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  *step = s->step;
  return GMES_OK;
}

int gmes_sim_set_graph(gmes_sim* s, int32_t enable) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  s->use_graph = enable != 0;
  destroy_graph(s);
  return GMES_OK;
}

int gmes_sim_set_ghost_fusion(gmes_sim* s, int32_t enable, int32_t* fused) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  HIP_TRY(hipSetDevice(s->device));
  HIP_TRY(sync_exec(s));
  s->allow_fuse = enable != 0;
  destroy_graph(s);  // one-sweep steps end or begin with it
  decide_fusion(s);
  if (fused) *fused = (s->fuse_e || s->fuse_hz) ? 1 : 0;
  return GMES_OK;
}

int gmes_sim_set_tile(gmes_sim* s, int32_t bx, int32_t by) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  if (bx < 0 || by < 0 || bx * by > 256 || (bx && (bx & (bx - 1))))
    return set_error(GMES_EINVAL, "bad tile: bx must be a power of two and bx*by <= 256");
  s->tile_bx = bx;
  s->tile_by = by;
  s->tile_tuned = false;
  const char* ic = getenv("GMES_ICHUNK");
  s->tile_ic = ic ? atoi(ic) : 0;
  destroy_graph(s);
  return GMES_OK;
}

int gmes_sim_autotune(gmes_sim* s, int32_t* bx, int32_t* by) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  if (!s->committed) return set_error(GMES_EINVAL, "sim is not committed");
  HIP_TRY(hipSetDevice(s->device));
  int tbx = 0, tby = 0, rc;
  switch (s->g.dtype) {
    case GMES_F32: rc = autotune_t<float>(s, tbx, tby); break;
    case GMES_F64: rc = autotune_t<double>(s, tbx, tby); break;
    case GMES_C64: rc = autotune_t<cplx<float>>(s, tbx, tby); break;
    default: rc = autotune_t<cplx<double>>(s, tbx, tby); break;
  }
  if (rc) return rc;
  if (tbx > 0) {
    s->tile_bx = tbx;
    s->tile_by = tby;
    s->tile_tuned = true;
    destroy_graph(s);
  }
  if (bx) *bx = tbx;
  if (by) *by = tby;
  return GMES_OK;
}

int gmes_sim_profile(gmes_sim* s, int32_t enable) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  HIP_TRY(hipSetDevice(s->device));
  HIP_TRY(sync_exec(s));
  collect_timing(s);
  s->timing.on = enable != 0;
  for (int i = 0; i < 6; ++i) { s->timing.ms[i] = 0; s->timing.launches[i] = 0; }
  return GMES_OK;
}

int gmes_sim_read_profile(gmes_sim* s, double ms[6], int64_t launches[6]) {
  ApiGuard api;
  if (!s) return set_error(GMES_EINVAL, "null sim handle");
  HIP_TRY(hipSetDevice(s->device));
  HIP_TRY(sync_exec(s));
  int rc = collect_timing(s);
  if (rc) return rc;
  for (int i = 0; i < 6; ++i) { ms[i] = s->timing.ms[i]; launches[i] = s->timing.launches[i]; }
  return GMES_OK;
}

// ----------------------------------------------------------------- batches
}  // extern "C"

struct gmes_batch {
  std::vector<gmes_sim*> sims;
  int device = 0;
  int dtype = 0;
  hipStream_t stream = nullptr;
  bool use_graph = true;
  // Captured steps.  Without one-sweep members: one step ([0][0]).  With them,
  // by the buffer set they start from (theirs swap with every step): two steps,
  // and the last one or two of an odd or even call, which write the ghost planes.
  hipGraphExec_t graphs[2][3] = {};
  std::vector<uint64_t> gens;  // member generations they were captured with
  // job tables: one device buffer, rebuilt on the host for every call
  void* d_jobs = nullptr;
  size_t jobs_cap = 0;
  std::vector<char> h_jobs;
  struct Launch {
    size_t off = 0;
    int njobs = 0;
    int64_t nblocks = 0;
  };
  // the launches of one step of a group of sims
  struct JobSet {
    Launch main3d[2], main2z[2], mainnd[2], src[2], ghost[2];  // [0] E, [1] H
    Launch main3d_pp[2];  // 3-D jobs with the CPML row prefetch (kBatch3dPP)
    Launch main3d_ur[2];  // 3-D jobs with the UPML row prefetch (kBatch3dUR)
    bool lds3d[2] = {false, false};  // every 3-D job stages its records in LDS
    bool lds2z[2] = {false, false};  // every collapsed-z job does
    Launch ade[GMES_NCLS];                                      // by dispersive class
    Launch dft;
  };
  // one-sweep members: the launches of a step, for the first and second step
  // of a call (their buffers swap), then the same writing the ghost planes
  struct SweepSet {
    Launch s3[4], s2, s1, aux, fix_e, fix_h, ghost, dft;  // s3: exact divisions (1), lean (2)
    size_t lds3[4] = {}, lds2 = 0;
  };
  SweepSet sweep[4];
  std::vector<gmes_sim*> sweepers, others;
  JobSet set;                      // the other members
  JobSet aux_set;                  // their auxiliary (TFSF) grids, stepped inside the members' step
  std::vector<gmes_sim*> aux_sims;
  std::vector<int64_t> shape_sig;  // launch shapes the graph was captured with
  // kernel timing (gmes_batch_profile): [E 3-D main, H 3-D main, E 2-D/1-D
  // main, H 2-D/1-D main, dispersive, the rest]
  gmes_engine::Timing timing;
};

namespace {

size_t append_table(std::vector<char>& h, const void* p, size_t bytes) {
  const size_t off = (h.size() + 255) / 256 * 256;
  h.resize(off + bytes);
  if (bytes) memcpy(h.data() + off, p, bytes);
  return off;
}

// Job tables of every batched launch.  The tiles follow each member's own
// setting (gmes_sim_set_tile / gmes_sim_autotune), with by = 256 / bx.
template <class T>
void build_jobs(gmes_batch* b, const std::vector<gmes_sim*>& sims, gmes_batch::JobSet& out) {
  for (int e = 0; e < 2; ++e) {
    const bool electric = e == 0;
    std::vector<MainJob<T>> j3, j2, jn, j3p, j3u;
    int64_t nb3 = 0, nb2 = 0, nbn = 0, nb3p = 0, nb3u = 0;
    bool lds3d = true, lds2z = true;
    // the block-wide record staging of the main tiles (RecStage::use_lds)
    constexpr int chunks = (int)(sizeof(DevRec<typename real_of<T>::type>) / 16);
    std::vector<SrcJob<T>> js;
    int64_t nbs = 0;
    std::vector<GhostJob<T>> jg;
    int64_t nbg = 0;
    for (gmes_sim* s : sims) {
      MainJob<T> J{};
      int ext[3];
      if (main_args<T>(s, electric, J.m, ext)) {
        int bx, by;
        tile_of(s, ext, bx, by);
        J.bx = bx;
        const int tby = 256 / bx;
        if (is3d(s)) {
          const bool fits = J.m.nrec <= kRecLds && J.m.nrec * chunks <= 256;
          J.gx = (int)(((int64_t)s->g.ny * s->g.nz + 255) / 256);
          J.gy = 1;
          if (std::is_same<T, float>::value && J.m.pp && fits) {
            J.block0 = nb3p;
            nb3p += (int64_t)J.gx * J.gy * s->g.nx;
            j3p.push_back(J);
          } else if (std::is_same<T, float>::value && J.m.ur && fits) {
            J.block0 = nb3u;
            nb3u += (int64_t)J.gx * J.gy * s->g.nx;
            j3u.push_back(J);
          } else {
            if (!fits) lds3d = false;
            J.block0 = nb3;
            nb3 += (int64_t)J.gx * J.gy * s->g.nx;
            j3.push_back(J);
          }
        } else if (is_2z(s)) {
          if (J.m.nrec > kRecLds || J.m.nrec * chunks > 256) lds2z = false;
          J.bx = ext[1];
          J.gx = (int)(((int64_t)ext[0] * ext[1] + 255) / 256);
          J.gy = 1;
          J.block0 = nb2;
          nb2 += (int64_t)J.gx * J.gy;
          j2.push_back(J);
        } else {
          J.gx = J.m.kloop ? 1 : (ext[2] + bx - 1) / bx;
          J.gy = (ext[1] + tby - 1) / tby;
          J.block0 = nbn;
          nbn += (int64_t)J.gx * J.gy * ext[0];
          jn.push_back(J);
        }
      }
      SrcJob<T> S{};
      S.a = src_args<T>(s, electric);
      if (S.a.ngroups > 0) {
        S.block0 = nbs;
        nbs += (S.a.ngroups + 255) / 256;
        js.push_back(S);
      }
      if (electric && s->fuse_e) continue;  // E ghosts written by the 3-D E kernel
      GhostJob<T> G{};
      int64_t total = 0;
      G.g = ghost_args<T>(s, electric, 0, total);
      G.block0 = nbg;
      nbg += std::max<int64_t>(1, (total + 255) / 256);  // >= 1: the block that ticks the clock
      jg.push_back(G);
    }
    out.main3d[e] = {append_table(b->h_jobs, j3.data(), j3.size() * sizeof(MainJob<T>)), (int)j3.size(), nb3};
    out.main3d_pp[e] = {append_table(b->h_jobs, j3p.data(), j3p.size() * sizeof(MainJob<T>)), (int)j3p.size(), nb3p};
    out.main3d_ur[e] = {append_table(b->h_jobs, j3u.data(), j3u.size() * sizeof(MainJob<T>)), (int)j3u.size(), nb3u};
    out.lds3d[e] = lds3d;
    out.lds2z[e] = lds2z;
    out.main2z[e] = {append_table(b->h_jobs, j2.data(), j2.size() * sizeof(MainJob<T>)), (int)j2.size(), nb2};
    out.mainnd[e] = {append_table(b->h_jobs, jn.data(), jn.size() * sizeof(MainJob<T>)), (int)jn.size(), nbn};
    out.src[e] = {append_table(b->h_jobs, js.data(), js.size() * sizeof(SrcJob<T>)), (int)js.size(), nbs};
    out.ghost[e] = {append_table(b->h_jobs, jg.data(), jg.size() * sizeof(GhostJob<T>)), (int)jg.size(), nbg};
  }
  for (int cls = GMES_CLS_DRUDE; cls < GMES_NCLS; ++cls) {
    std::vector<AdeJob<T>> ja;
    int64_t nba = 0;
    for (gmes_sim* s : sims)
      for (int c = 0; c < 3; ++c) {
        if (s->ade[c][cls].n == 0) continue;
        AdeJob<T> A{};
        A.a = ade_args<T>(s, c, cls);
        A.comp = c;
        A.block0 = nba;
        nba += (A.a.n + 255) / 256;
        ja.push_back(A);
      }
    out.ade[cls] = {append_table(b->h_jobs, ja.data(), ja.size() * sizeof(AdeJob<T>)), (int)ja.size(), nba};
  }
  std::vector<DftJob<T>> jd;
  int64_t nbd = 0;
  for (gmes_sim* s : sims) dft_jobs<T>(s, jd, nbd);
  out.dft = {append_table(b->h_jobs, jd.data(), jd.size() * sizeof(DftJob<T>)), (int)jd.size(), nbd};
}

template <class J>
const J* job_ptr(const gmes_batch* b, size_t off) {
  return reinterpret_cast<const J*>(static_cast<const char*>(b->d_jobs) + off);
}

// Whether a member takes one-sweep steps in a batch.
bool batch_sweeps(const gmes_sim* s) {
  if (!sweeps(s)) return false;
  for (int i = 0; i < s->naux; ++i)
    if (s->aux[i] && !aux_sweeps(s->aux[i])) return false;
  gmes_sim::SweepPart part;
  bool lean;
  return s->sweep_1d || s->sweep_2d || sweep_batch_part(s, part, lean, kSweepInnerPlanes);
}

// A member's buffers, and those of its auxiliary grids, become the other set.
void sweep_swap_aux(gmes_sim* s) {
  for (int i = 0; i < s->naux; ++i)
    if (s->aux[i]) sweep_swap(s->aux[i]);
}

// The buffers of the one-sweep members become the other set.
void batch_swap(gmes_batch* b) {
  for (gmes_sim* s : b->sweepers) {
    sweep_swap(s);
    sweep_swap_aux(s);
  }
}

// Planes (rows) per block of a batch's one-sweep members, from its tiles times
// planes (rows).  As in sweep2_shape, fewer while they fill the chip badly (us
// per step at 3, 5, 7, 9, 16 planes: 476 tile planes 36, 43, 48, 54, 63; 2199
// 79, 89, 83, 93, 115; 4315 99, 99, 103, 111, 118; 12303 224, 217, 217, 223,
// 237; at 1, 2, 3, 5 rows: 965 tile rows 107, 108, 111, 115; 5852 274, 266,
// 264, 266).
int batch_ch3(double work) { return std::max(3, std::min(9, (int)std::lround(std::sqrt(work / 300)))); }
int batch_ch2(double work) { return std::max(1, std::min(5, (int)std::ceil(std::sqrt(work / 1500)))); }

// Job tables of the one-sweep members.  The arguments of a step are taken
// from the sims as that step finds them: the host's pointers are swapped
// on the way and end where they were.  A call of one step leaves out the second
// one's (gmes_batch::sweep [1] and [3] stay as they were, at the end of the
// tables).
template <class T>
void build_sweep_jobs(gmes_batch* b, int64_t nsteps) {
  std::vector<Step3Job<T>> j3[2][4];
  std::vector<Step2Job<T>> j2[2];
  std::vector<Step1Job<T>> j1[2], ja;
  // planes (rows in 2-D) per block: a few rounds of blocks over the chip
  double work3 = 0, work2 = 0;
  for (const gmes_sim* s : b->sweepers) {
    if (s->sweep_2d) work2 += (double)s->g.nx * ((s->g.ny + 255) / 256);
    else if (!s->sweep_1d) work3 += (double)s->g.nx * s->g.ny / std::max(1, 768 / s->g.nz - 1);
  }
  const int ch3 = batch_ch3(work3), ch2 = batch_ch2(work2);
  const int steps = nsteps > 1 ? 2 : 1;
  for (int t = 0; t < steps; ++t) {
    std::vector<FixJob<T>> je, jh;
    std::vector<GhostJob<T>> jg[2];
    std::vector<DftJob<T>> jd;
    int64_t n3[4] = {}, n2 = 0, n1 = 0, na = 0, ne = 0, nh = 0, ng[2] = {0, 0}, nd = 0;
    size_t lds3[4] = {}, lds2 = 0;
    for (int g = 0; g < 2; ++g) {
      for (auto& v : j3[g]) v.clear();
      j2[g].clear();
      j1[g].clear();
    }
    ja.clear();
    for (gmes_sim* s : b->sweepers) {
      const bool always = sweep_ghosts(s);
      s->sweep_ghosts = true;
      auto add = [&](auto& v, auto& J) {  // with the ghost planes, and without
        v[1].push_back(J);
        J.a.ghosts = always;
        v[0].push_back(J);
      };
      if (s->sweep_1d) {
        Step1Job<T> J{step1_args<T>(s), n1};
        n1 += (J.a.n + kStep1Threads - 2) / (kStep1Threads - 1);
        add(j1, J);
      } else if (s->sweep_2d) {
        Step2Job<T> J{step2_args<T>(s), step2_tm(s), s->sweep_absorber, n2};
        // blocks of kStep2BatchThreads threads, a few rows each
        J.a.whole = J.a.n[1] <= kStep2BatchThreads;
        J.a.w = J.a.whole ? J.a.n[1] : 224;
        J.a.ch = std::min(ch2, J.a.n[0]);
        J.a.nj = (J.a.n[1] + J.a.w - 1) / J.a.w;
        J.a.nblk = J.a.nj * ((J.a.n[0] + J.a.ch - 1) / J.a.ch);
        n2 += (J.a.nblk + 7) / 8 * 8;
        lds2 = std::max(lds2, step2_lds<T>(kStep2BatchThreads, J.a.nent));
        add(j2, J);
      } else if constexpr (!std::is_same<T, cplx<double>>::value) {
        gmes_sim::SweepPart part;
        bool lean;
        (void)sweep_batch_part(s, part, lean, ch3);
        Step3Job<T> J{step3_args<T>(s, part), 0};
        const int x = (std::is_same<T, double>::value && J.a.exact) + 2 * lean;
        J.block0 = n3[x];
        n3[x] += 8 * (int64_t)J.a.slots;
        lds3[x] = std::max(lds3[x], step3_lds<T>(part.threads, J.a.net + J.a.nht, part.rows, s->g.nz, s->sweep_absorber));
        j3[1][x].push_back(J);
        J.a.ghosts = always;
        j3[0][x].push_back(J);
      }
      sweep_swap(s);
      if constexpr (!std::is_same<T, cplx<double>>::value) {
        if (s->sweep_fix && !s->sweep_1d && !s->sweep_2d) {
          FixJob<T> F{fix_args<T>(s), ne};
          ne += F.a.eblocks;
          if (F.a.eblocks) je.push_back(F);
          for (int i = 0; i < s->naux; ++i) {
            if (!s->aux[i]) continue;
            Step1Job<T> A{step1_args<T>(s->aux[i]), na};
            na += (A.a.n + kStep1Threads - 2) / (kStep1Threads - 1);
            ja.push_back(A);
          }
          sweep_swap_aux(s);
          FixJob<T> H{fix_args<T>(s), nh};
          nh += H.a.hblocks;
          if (H.a.hblocks) jh.push_back(H);
          for (int g = 0; g < 2; ++g) {
            if (!always && !g) continue;
            GhostJob<T> G{};
            int64_t total = 0;
            G.g = ghost_args<T>(s, true, 0, total);
            G.block0 = ng[g];
            ng[g] += std::max<int64_t>(1, (total + 255) / 256);
            jg[g].push_back(G);
          }
        }
      }
      dft_jobs<T>(s, jd, nd);
    }
    auto put = [&](const auto& v, int64_t blocks) {
      using J = typename std::decay<decltype(v[0])>::type;
      return gmes_batch::Launch{append_table(b->h_jobs, v.data(), v.size() * sizeof(J)), (int)v.size(), blocks};
    };
    const gmes_batch::Launch la = put(ja, na), le = put(je, ne), lh = put(jh, nh), ld = put(jd, nd);
    for (int g = 0; g < 2; ++g) {
      gmes_batch::SweepSet& S = b->sweep[t + 2 * g];
      for (int x = 0; x < 4; ++x) {
        S.s3[x] = put(j3[g][x], n3[x]);
        S.lds3[x] = lds3[x];
      }
      S.s2 = put(j2[g], n2);
      S.s1 = put(j1[g], n1);
      S.aux = la;
      S.fix_e = le;
      S.fix_h = lh;
      S.ghost = put(jg[g], ng[g]);
      S.dft = ld;
      S.lds2 = lds2;
    }
  }
  if (steps == 1) batch_swap(b);
}

// One step of a group of sims (the members, or their auxiliary grids)
// with one launch per kernel kind.
template <class T>
void build_tables(gmes_batch* b, int64_t nsteps) {
  build_jobs<T>(b, b->others, b->set);
  build_jobs<T>(b, b->aux_sims, b->aux_set);
  build_sweep_jobs<T>(b, nsteps);
}

// HIP events around the launches of one kernel family of a batch step
// (members only; the auxiliary grids count as "the rest").
void btime_begin(gmes_batch* b, bool on, int fam, hipStream_t st) {
  if (!on || !b->timing.on) return;
  hipEvent_t x, y;
  (void)hipEventCreate(&x);
  (void)hipEventCreate(&y);
  (void)hipEventRecord(x, st);
  b->timing.pending.push_back({fam, {x, y}});
}

void btime_end(gmes_batch* b, bool on, hipStream_t st) {
  if (!on || !b->timing.on) return;
  (void)hipEventRecord(b->timing.pending.back().second.second, st);
}

template <class T>
void enqueue_set_step_t(gmes_batch* b, const gmes_batch::JobSet& js, const std::vector<gmes_sim*>& sims,
                        bool with_aux, hipStream_t st) {
  const bool tm = with_aux;  // timing covers the members' launches
  const auto& H = js.ghost[1];
  btime_begin(b, tm, 5, st);
  launch_ghost_batch<T>(job_ptr<GhostJob<T>>(b, H.off), H.njobs, H.nblocks, 1, st);
  btime_end(b, tm, st);
  for (int e = 0; e < 2; ++e) {
    const bool electric = e == 0;
    if (!electric) {
      const auto& G = js.ghost[0];
      btime_begin(b, tm, 5, st);
      launch_ghost_batch<T>(job_ptr<GhostJob<T>>(b, G.off), G.njobs, G.nblocks, 0, st);
      btime_end(b, tm, st);
    }
    btime_begin(b, tm, e, st);
    launch_main_batch<T>(electric, kBatch3dPP, job_ptr<MainJob<T>>(b, js.main3d_pp[e].off), js.main3d_pp[e].njobs,
                         js.main3d_pp[e].nblocks, st);
    launch_main_batch<T>(electric, kBatch3dUR, job_ptr<MainJob<T>>(b, js.main3d_ur[e].off), js.main3d_ur[e].njobs,
                         js.main3d_ur[e].nblocks, st);
    launch_main_batch<T>(electric, js.lds3d[e] ? kBatch3dLds : kBatch3d, job_ptr<MainJob<T>>(b, js.main3d[e].off),
                         js.main3d[e].njobs,
                         js.main3d[e].nblocks, st);
    btime_end(b, tm, st);
    btime_begin(b, tm, 2 + e, st);
    launch_main_batch<T>(electric, js.lds2z[e] ? kBatch2zLds : kBatch2z, job_ptr<MainJob<T>>(b, js.main2z[e].off),
                         js.main2z[e].njobs,
                         js.main2z[e].nblocks, st);
    launch_main_batch<T>(electric, kBatchGeneric, job_ptr<MainJob<T>>(b, js.mainnd[e].off), js.mainnd[e].njobs,
                         js.mainnd[e].nblocks, st);
    btime_end(b, tm, st);
    if (electric) {
      btime_begin(b, tm, 4, st);
      for (int cls = GMES_CLS_DRUDE; cls < GMES_NCLS; ++cls)
        launch_ade_batch<T>(cls, job_ptr<AdeJob<T>>(b, js.ade[cls].off), js.ade[cls].njobs, js.ade[cls].nblocks, st);
      btime_end(b, tm, st);
    }
    btime_begin(b, tm, 5, st);
    launch_src_batch<T>(job_ptr<SrcJob<T>>(b, js.src[e].off), js.src[e].njobs, js.src[e].nblocks, st);
    for (gmes_sim* s : sims) enqueue_probe<T>(s, electric, st);
    // every member's auxiliary grids advance one whole step here, all of
    // them in one launch per kernel kind (as each single sim does it with
    // its own grids)
    if (electric && with_aux && !b->aux_sims.empty()) enqueue_set_step_t<T>(b, b->aux_set, b->aux_sims, false, st);
    btime_end(b, tm, st);
  }
  btime_begin(b, tm, 5, st);
  launch_dft_batch<T>(job_ptr<DftJob<T>>(b, js.dft.off), js.dft.njobs, js.dft.nblocks, st);
  btime_end(b, tm, st);
}

// One step of the one-sweep members, in the order of their own step.
template <class T>
void enqueue_sweep_set(gmes_batch* b, int variant, hipStream_t st) {
  const gmes_batch::SweepSet& S = b->sweep[variant];
  if constexpr (!std::is_same<T, cplx<double>>::value) {
    btime_begin(b, true, 0, st);
    for (int x = 0; x < 4; ++x)
      launch_step3d_batch<T>(job_ptr<Step3Job<T>>(b, S.s3[x].off), S.s3[x].njobs, S.s3[x].nblocks, x & 1, x & 2,
                             S.lds3[x], st);
    btime_end(b, true, st);
  }
  btime_begin(b, true, 2, st);
  launch_step2d_batch<T>(job_ptr<Step2Job<T>>(b, S.s2.off), S.s2.njobs, S.s2.nblocks, S.lds2, st);
  launch_step1d_batch<T>(job_ptr<Step1Job<T>>(b, S.s1.off), S.s1.njobs, S.s1.nblocks, st);
  btime_end(b, true, st);
  for (gmes_sim* s : b->sweepers) sweep_swap(s);
  btime_begin(b, true, 4, st);
  if constexpr (!std::is_same<T, cplx<double>>::value)
    launch_fix_batch<T>(true, job_ptr<FixJob<T>>(b, S.fix_e.off), S.fix_e.njobs, S.fix_e.nblocks, st);
  btime_end(b, true, st);
  btime_begin(b, true, 5, st);
  launch_step1d_batch<T>(job_ptr<Step1Job<T>>(b, S.aux.off), S.aux.njobs, S.aux.nblocks, st);
  for (gmes_sim* s : b->sweepers) sweep_swap_aux(s);
  if (S.ghost.njobs)
    launch_ghost_batch<T>(job_ptr<GhostJob<T>>(b, S.ghost.off), S.ghost.njobs, S.ghost.nblocks, 0, st);
  if constexpr (!std::is_same<T, cplx<double>>::value)
    launch_fix_batch<T>(false, job_ptr<FixJob<T>>(b, S.fix_h.off), S.fix_h.njobs, S.fix_h.nblocks, st);
  for (gmes_sim* s : b->sweepers) enqueue_probe<T>(s, kProbeBoth, st);
  if (S.dft.njobs) launch_dft_batch<T>(job_ptr<DftJob<T>>(b, S.dft.off), S.dft.njobs, S.dft.nblocks, st);
  btime_end(b, true, st);
}

// One step of every member, in the single-sim order, with the kernels of all
// members batched into one launch of each kind.  variant: which tables of the
// one-sweep members (gmes_batch::sweep).
template <class T>
void enqueue_batch_step_t(gmes_batch* b, int variant, hipStream_t st) {
  if (!b->sweepers.empty()) enqueue_sweep_set<T>(b, variant, st);
  if (!b->others.empty()) enqueue_set_step_t<T>(b, b->set, b->others, true, st);
}

void enqueue_batch_step(gmes_batch* b, int variant, hipStream_t st) {
  switch (b->dtype) {
    case GMES_F32: enqueue_batch_step_t<float>(b, variant, st); break;
    case GMES_F64: enqueue_batch_step_t<double>(b, variant, st); break;
    case GMES_C64: enqueue_batch_step_t<cplx<float>>(b, variant, st); break;
    default: enqueue_batch_step_t<cplx<double>>(b, variant, st); break;
  }
}

void destroy_batch_graph(gmes_batch* b) {
  for (auto& set : b->graphs)
    for (hipGraphExec_t& g : set) {
      if (g) (void)hipGraphExecDestroy(g);
      g = nullptr;
    }
}

std::vector<uint64_t> batch_gens(const gmes_batch* b) {
  std::vector<uint64_t> gens;
  for (const gmes_sim* s : b->sims) {
    gens.push_back(s->gen);
    for (int i = 0; i < s->naux; ++i)
      if (s->aux[i]) gens.push_back(s->aux[i]->gen);
  }
  return gens;
}

hipGraphExec_t& batch_graph(gmes_batch* b, int kind) {
  return b->graphs[b->sweepers.empty() ? 0 : b->sweepers[0]->par][kind];
}

// Whether a call of nsteps replays the graph of a kind (gmes_batch::graphs).
bool batch_uses(const gmes_batch* b, int kind, int64_t nsteps) {
  if (b->sweepers.empty()) return kind == 0;
  return kind == 0 ? nsteps > 2 : kind == 1 ? nsteps % 2 == 1 : nsteps % 2 == 0;
}

// The job tables of a call of nsteps on the device, and its graphs; ready is
// false when a member changed meanwhile, where this call waited to be alone
// in the engine (dev_malloc, the capture).
int batch_ready(gmes_batch* b, int64_t nsteps, bool& ready) {
  const std::vector<uint64_t> gens = batch_gens(b);
  b->sweepers.clear();
  b->others.clear();
  for (gmes_sim* s : b->sims) {
    const bool sweep = batch_sweeps(s);
    if (!sweep)
      if (int rc = aux_pointers(s)) return rc;
    sweep_clock(s, sweep, b->stream);
    for (int i = 0; i < s->naux; ++i)
      if (s->aux[i]) sweep_clock(s->aux[i], sweep, b->stream);
    (sweep ? b->sweepers : b->others).push_back(s);
  }
  // the job tables are read by kernels still in flight: wait before rewriting
  HIP_TRY(hipStreamSynchronize(b->stream));
  b->aux_sims.clear();
  for (gmes_sim* s : b->others)
    for (int i = 0; i < s->naux; ++i)
      if (s->aux[i]) b->aux_sims.push_back(s->aux[i]);
  b->h_jobs.clear();
  switch (b->dtype) {
    case GMES_F32: build_tables<float>(b, nsteps); break;
    case GMES_F64: build_tables<double>(b, nsteps); break;
    case GMES_C64: build_tables<cplx<float>>(b, nsteps); break;
    default: build_tables<cplx<double>>(b, nsteps); break;
  }
  if (b->h_jobs.size() > b->jobs_cap) {
    destroy_batch_graph(b);
    if (b->d_jobs) HIP_TRY(dev_release(b->d_jobs));
    b->d_jobs = nullptr;
    b->jobs_cap = 0;
    HIP_TRY(dev_malloc(b->device, &b->d_jobs, b->h_jobs.size()));
    b->jobs_cap = b->h_jobs.size();
  }
  HIP_TRY(hipMemcpy(b->d_jobs, b->h_jobs.data(), b->h_jobs.size(), hipMemcpyHostToDevice));
  // launch shapes and per-member captured arguments decide whether the
  // graph is still valid; table contents are read at run time
  std::vector<int64_t> sig;
  for (const gmes_batch::JobSet* js : {&b->set, &b->aux_set}) {
    for (int e = 0; e < 2; ++e)
      for (const auto* L : {&js->main3d[e], &js->main3d_pp[e], &js->main3d_ur[e], &js->main2z[e], &js->mainnd[e], &js->src[e],
                            &js->ghost[e]}) {
        sig.push_back((int64_t)L->off);
        sig.push_back(L->njobs);
        sig.push_back(L->nblocks);
      }
    for (const auto& L : js->ade) {
      sig.push_back((int64_t)L.off);
      sig.push_back(L.njobs);
      sig.push_back(L.nblocks);
    }
    sig.push_back((int64_t)js->dft.off);
    sig.push_back(js->dft.njobs);
    sig.push_back(js->dft.nblocks);
  }
  for (const gmes_batch::SweepSet& S : b->sweep) {
    for (const auto* L : {&S.s3[0], &S.s3[1], &S.s3[2], &S.s3[3], &S.s2, &S.s1, &S.aux, &S.fix_e, &S.fix_h, &S.ghost, &S.dft}) {
      sig.push_back((int64_t)L->off);
      sig.push_back(L->njobs);
      sig.push_back(L->nblocks);
    }
    for (const size_t l : S.lds3) sig.push_back((int64_t)l);
    sig.push_back((int64_t)S.lds2);
  }
  if (sig != b->shape_sig || gens != b->gens) destroy_batch_graph(b);
  b->shape_sig = sig;
  b->gens = gens;
  for (int kind = 0; kind < 3 && b->use_graph && !b->timing.on; ++kind) {
    hipGraphExec_t& exec = batch_graph(b, kind);
    if (exec || !batch_uses(b, kind, nsteps)) continue;
    hipGraph_t graph;
    hipError_t e;
    {
      CaptureGuard capture;
      if (gens != batch_gens(b)) return GMES_OK;
      HIP_TRY(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
      const int first = kind == 1 ? 2 : 0;  // the tables (gmes_batch::sweep) of its steps
      enqueue_batch_step(b, first, b->stream);
      if (!b->sweepers.empty() && kind != 1) enqueue_batch_step(b, kind == 0 ? 1 : 3, b->stream);
      HIP_TRY(hipStreamEndCapture(b->stream, &graph));
      if (kind == 1) batch_swap(b);
      e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    }
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) return set_error(GMES_EDEVICE, "hipGraphInstantiate: %s", hipGetErrorString(e));
  }
  ready = gens == batch_gens(b);
  return GMES_OK;
}

}  // namespace

extern "C" {

int gmes_batch_create(gmes_sim* const* sims, int32_t n, gmes_batch** out) {
  ApiGuard api;
  if (n < 1) return set_error(GMES_EINVAL, "empty batch");
  for (int i = 0; i < n; ++i) {
    gmes_sim* s = sims[i];
    if (!s) return set_error(GMES_EINVAL, "null batch member");
    if (s->device != sims[0]->device) return set_error(GMES_EINVAL, "batch members must share a device");
    if (s->g.dtype != sims[0]->g.dtype) return set_error(GMES_ETYPE, "batch members must share a storage type");
    if (s->batch_stream) return set_error(GMES_EINVAL, "sim %d is already in a batch", i);
    if (s->parent) return set_error(GMES_EINVAL, "an auxiliary grid cannot be a batch member");
    if (!s->committed) return set_error(GMES_EINVAL, "sim %d is not committed", i);
    for (int k = 0; k < i; ++k)
      if (sims[k] == s) return set_error(GMES_EINVAL, "sim %d appears twice", i);
  }
  HIP_TRY(hipSetDevice(sims[0]->device));
  gmes_batch* b = new gmes_batch();
  b->sims.assign(sims, sims + n);
  b->device = sims[0]->device;
  b->dtype = sims[0]->g.dtype;
  // non-blocking: host threads that build other sims meanwhile issue
  // null-stream copies, which must not order against (or invalidate a
  // graph capture on) the batch stream; ordering with the members is
  // explicit (sync_exec waits on the batch stream)
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) {
    delete b;
    return set_error(GMES_EDEVICE, "hipStreamCreate failed");
  }
  for (gmes_sim* s : b->sims) {
    (void)sync_exec(s);
    s->batch_stream = b->stream;
  }
  // setup work of the members issued on the null stream (zero fills, table
  // uploads) is not ordered before the non-blocking batch stream: drain it
  HIP_TRY(device_drain());
  *out = b;
  return GMES_OK;
}

int gmes_batch_destroy(gmes_batch* b) {
  ApiGuard api;
  if (!b) return GMES_OK;
  (void)hipSetDevice(b->device);
  (void)hipStreamSynchronize(b->stream);
  destroy_batch_graph(b);
  for (auto& p : b->timing.pending) {
    (void)hipEventDestroy(p.second.first);
    (void)hipEventDestroy(p.second.second);
  }
  for (gmes_sim* s : b->sims) s->batch_stream = nullptr;
  if (b->d_jobs) (void)dev_release(b->d_jobs);
  (void)stream_release(b->stream);
  delete b;
  return GMES_OK;
}

int gmes_batch_set_graph(gmes_batch* b, int32_t enable) {
  ApiGuard api;
  if (!b) return set_error(GMES_EINVAL, "null batch handle");
  b->use_graph = enable != 0;
  destroy_batch_graph(b);
  return GMES_OK;
}

// Advance every member by nsteps: one batched launch per kernel kind (and half
// step, for members that take those), replayed from captured graphs.
int gmes_batch_step(gmes_batch* b, int64_t nsteps) {
  ApiGuard api;
  if (!b) return set_error(GMES_EINVAL, "null batch handle");
  if (nsteps < 0) return set_error(GMES_EINVAL, "negative step count");
  for (gmes_sim* s : b->sims) {
    if (s->timing.on) return set_error(GMES_EINVAL, "kernel timing is per sim; switch it off for batch members");
    if (s->aux_lost) return set_error(GMES_EINVAL, "an auxiliary grid of a batch member was destroyed");
    int rc = check_windows(s, nsteps);
    if (rc) return rc;
    if ((rc = ensure_probe_capacity(s, nsteps))) return rc;
  }
  if (nsteps == 0) return GMES_OK;
  HIP_TRY(hipSetDevice(b->device));
  // members that lose their second buffers meanwhile (sweep_reclaim) change
  // the tables
  bool ready = false;
  while (!ready)
    if (int rc = batch_ready(b, nsteps, ready)) return rc;
  if (!b->use_graph || b->timing.on) {
    for (int64_t t = 0; t < nsteps; ++t) enqueue_batch_step(b, (int)(t & 1) + (t == nsteps - 1 ? 2 : 0), b->stream);
    HIP_TRY(hipGetLastError());
  } else if (b->sweepers.empty()) {
    for (int64_t t = 0; t < nsteps; ++t) HIP_TRY(hipGraphLaunch(batch_graph(b, 0), b->stream));
  } else {
    for (int64_t t = 0; t + 2 < nsteps; t += 2) HIP_TRY(hipGraphLaunch(batch_graph(b, 0), b->stream));
    HIP_TRY(hipGraphLaunch(batch_graph(b, nsteps % 2 ? 1 : 2), b->stream));
    if (nsteps % 2) batch_swap(b);
  }
  for (gmes_sim* s : b->sims) advance_host_clock(s, nsteps);
  return GMES_OK;
}

int gmes_batch_profile(gmes_batch* b, int32_t enable) {
  ApiGuard api;
  if (!b) return set_error(GMES_EINVAL, "null batch handle");
  HIP_TRY(hipSetDevice(b->device));
  HIP_TRY(hipStreamSynchronize(b->stream));
  for (auto& p : b->timing.pending) {
    (void)hipEventDestroy(p.second.first);
    (void)hipEventDestroy(p.second.second);
  }
  b->timing = Timing();
  b->timing.on = enable != 0;
  return GMES_OK;
}

int gmes_batch_read_profile(gmes_batch* b, double ms[6], int64_t launches[6]) {
  ApiGuard api;
  if (!b || !ms || !launches) return set_error(GMES_EINVAL, "null argument");
  HIP_TRY(hipSetDevice(b->device));
  for (auto& p : b->timing.pending) {
    float t = 0.f;
    HIP_TRY(hipEventSynchronize(p.second.second));
    HIP_TRY(hipEventElapsedTime(&t, p.second.first, p.second.second));
    b->timing.ms[p.first] += t;
    b->timing.launches[p.first] += 1;
    (void)hipEventDestroy(p.second.first);
    (void)hipEventDestroy(p.second.second);
  }
  b->timing.pending.clear();
  for (int i = 0; i < 6; ++i) {
    ms[i] = b->timing.ms[i];
    launches[i] = b->timing.launches[i];
  }
  return GMES_OK;
}

int gmes_batch_sync(gmes_batch* b) {
  ApiGuard api;
  if (!b) return set_error(GMES_EINVAL, "null batch handle");
  HIP_TRY(hipSetDevice(b->device));
  HIP_TRY(hipStreamSynchronize(b->stream));
  for (gmes_sim* s : b->sims) {
    int rc = gmes_sim_sync(s);
    if (rc) return rc;
  }
  return GMES_OK;
}

}  // extern "C"
