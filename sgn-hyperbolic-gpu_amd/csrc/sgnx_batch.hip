// =============================================================================
// sgnx_batch.hip -- many independent solvers of uneven sizes advanced together.
//
// Every RHS launch of an adaptive step covers all running members: the
// row-sweep workgroups of every member follow each other (a per-member offset
// table) in one launch per stage kind, followed by one launch that folds each
// member's error partials. Each member keeps its own state buffers, time, step
// size and controller (the same RkCtl as sgnx_integrate) and its own error
// partials, so its results are bit for bit those of sgnx_integrate on it
// alone. The reference's counterpart is a parameter sweep run as separate jobs
// (scripts/shoal_sweep.sbatch).
//
// Members recording an adjoint tape (sgnx_tape_begin) record it here as in
// sgnx_integrate: snapshot copies on the batch stream ahead of a step, the
// accepted steps after it.
//
// A step is: member arguments (pinned host -> device), three stage launches,
// the fold, which posts the (sum, max) pairs to mapped host memory; optionally
// captured once into a hipGraph and replayed while the set of running members
// is unchanged (the copy reads the same pinned buffer, which the host refills
// before each replay).
// =============================================================================

#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <iterator>
#include <string>
#include <vector>

#include "sgnx_handle.h"
#include "sgnx_tape.h"

struct sgnx_batch {
  std::vector<sgnx_solver*> m;
  int n = 0;
  int device = 0, cus = 1;
  int waves3 = 0x2;                    // bit k: launch kind k built for 3 waves/SIMD
  int rows = 0;                        // the packed launches' height from the autotuner
                                       // (0: by the rule for the running members)
  hipStream_t stream = nullptr;
  // argument tables, [4 launch kinds][n slots], then the tile offsets, then the
  // attempt's sequence number, in one block (one copy takes a step's part)
  BatchMember* h_mem = nullptr;        // pinned
  BatchMember* d_mem = nullptr;
  long long* h_ts = nullptr;           // n + 1, behind h_mem
  long long* d_ts = nullptr;
  // what the attempt's last launch writes for the host: per slot sum, max and
  // the sequence number, for which the host polls
  double* h_post = nullptr;            // pinned, mapped, 3 n
  double* d_post = nullptr;            // its device address
  unsigned long long seq = 0;
  // the captured step and the running set it was captured for
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  std::vector<int> graphSet;
  bool graphKeep = false;   // the captured step keeps stage inputs
  // the launch shape baked into the captured step: its grid (the members'
  // tiles in all) and each running member's tile height, so that a change of
  // either (sgnx_set_rhs_kernel or sgnx_autotune on a member) forces a capture
  long long graphTotal = 0;
  std::vector<int> graphRows;
  // argument arena of the batched reverse sweep (pinned host, device)
  char* h_adj = nullptr;
  char* d_adj = nullptr;
  size_t adjCap = 0;
  std::string err;
};

namespace {

thread_local std::string g_batch_create_error;

int bfail(sgnx_batch* b, int code, const std::string& msg) {
  if (b) b->err = msg;
  else g_batch_create_error = msg;
  return code;
}

#define BCHK(b, call)                                                                 \
  do {                                                                                \
    hipError_t e_ = (call);                                                           \
    if (e_ != hipSuccess)                                                             \
      return bfail((b), e_ == hipErrorOutOfMemory ? SGNX_ENOMEM : SGNX_EDEVICE,       \
                   std::string(#call) + ": " + hipGetErrorString(e_));                \
  } while (0)

void drop_graph(sgnx_batch* b) {
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  b->exec = nullptr;
  b->graph = nullptr;
  b->graphSet.clear();
  b->graphRows.clear();
  b->graphTotal = 0;
}

BatchMember member_args(const sgnx_solver* s, const double* U, double* dU, const Stage& sa,
                        double t, int times = 1) {
  return sweep_member(s->g, s->ph, U, dU, ghost_time(s, t), sa, times);
}

// A member's own tile height suits a launch of its own; packed with others it
// would make more and shorter workgroups than the device needs (24 grids of
// 34x17 to 126x63, heights 1 and 2, or 4 for all: stages 2, 3 and 4 103, 142 and
// 106 us, or 96, 128 and 109; ten accepted steps 5.25 ms, or 5.03).
// So the members in `set` take the multiple of their own that is nearest to the
// height for all their tiles together, by the rule or by the batch's autotuner;
// a height set from outside or by an autotuner is taken as it is.
int packed_rows(const sgnx_batch* b, const std::vector<int>& set) {
  std::vector<const Geometry*> gs;
  for (int i : set) gs.push_back(&b->m[i]->g);
  return sweep_rows(gs.data(), (int)gs.size(), b->cus);
}
int row_multiple(const sgnx_solver* s, int rows) {
  return s->rowsSet ? 1 : std::max(1, (2 * rows + s->g.rows) / (2 * s->g.rows));
}
std::vector<int> row_multiples(const sgnx_batch* b, const std::vector<int>& set) {
  const int rows = b->rows ? b->rows : packed_rows(b, set);
  std::vector<int> times;
  for (int i : set) times.push_back(row_multiple(b->m[i], rows));
  return times;
}

// tile offsets of the members in `set` (slot order; their entries of h_mem from
// `mem` on filled) into h_ts; returns the total
long long fill_offsets(sgnx_batch* b, const std::vector<int>& set, const BatchMember* mem) {
  long long acc = 0;
  for (size_t i = 0; i < set.size(); ++i) {
    b->h_ts[i] = acc;
    acc += packed_tiles(mem[i].nTiles);
  }
  b->h_ts[set.size()] = acc;
  return acc;
}

// whether every member's Hx, Hy are (D Hnod) / J bit for bit, so that the
// batched sweep may form them from Hnod (otherwise it reads them, which is
// right for every member)
bool batch_hxr(const sgnx_batch* b) {
  for (const sgnx_solver* s : b->m)
    if (!s->g.hxr) return false;
  return true;
}

// the device work of one attempted step for the members in `set` (slots
// 0..A-1 of kinds 1..3 of h_mem filled by the caller); `keep`: stages 2 and 3
// also write their inputs where a member's stage names a buffer for them
int enqueue_step(sgnx_batch* b, const std::vector<int>& set, long long total, bool keep) {
  const int A = (int)set.size();
  const size_t n = (size_t)b->n;
  BCHK(b, hipMemcpyAsync(b->d_mem + n, b->h_mem + n,
                         3 * n * sizeof(BatchMember) + (n + 2) * sizeof(long long),
                         hipMemcpyHostToDevice, b->stream));
  for (int k = 1; k <= 3; ++k)
    BCHK(b, launch_rhs_stage_batch(b->d_mem + k * n, b->d_ts, A, total, k,
                                   (b->waves3 >> k) & 1, b->stream, keep && k < 3, batch_hxr(b)));
  BCHK(b, launch_finish_batch(b->d_mem + 3 * n, A, b->d_post, b->d_ts + n + 1, b->stream));
  return SGNX_OK;
}

// The posts of an attempt's A slots: polled for a millisecond, which spares a
// short attempt the copy and the wake-up of a synchronization (an attempt of three
// grids of 32x16 to 64x32: 57 -> 45 us, of 24 of 34x17 to 126x63: 375 -> 362);
// longer ones end by it.
int wait_posts(sgnx_batch* b, int A) {
  auto posted = [&](int slot) {
    const auto* q = reinterpret_cast<const volatile unsigned long long*>(b->h_post + 3 * slot + 2);
    return *q == b->seq;
  };
  const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(1);
  int slot = 0;
  for (int k = 0; slot < A; ++k) {
    if (posted(slot)) ++slot;
    else if ((k & 63) == 63 && std::chrono::steady_clock::now() > until) break;
  }
  if (slot < A) {
    BCHK(b, hipStreamSynchronize(b->stream));
    for (; slot < A; ++slot)
      if (!posted(slot)) return bfail(b, SGNX_EDEVICE, "batch step: error norm not posted");
  }
  std::atomic_thread_fence(std::memory_order_acquire);
  return SGNX_OK;
}

// tile heights tried by the autotuners (rows of elements per workgroup)
constexpr int kTuneRows[] = {2, 4, 8, 12, 16, 24, 32};

// a step size for the probe launches: any finite value times the same work
constexpr double kProbeDt = 1e-9;

struct EventPair {
  hipEvent_t a = nullptr, b = nullptr;
  ~EventPair() {
    if (a) (void)hipEventDestroy(a);
    if (b) (void)hipEventDestroy(b);
  }
};

}  // namespace

extern "C" {

const char* sgnx_batch_last_error(const sgnx_batch* b) {
  return b ? b->err.c_str() : g_batch_create_error.c_str();
}

int sgnx_batch_create(sgnx_solver* const* members, int n, sgnx_batch** out) {
  if (!out) return SGNX_EINVAL;
  *out = nullptr;
  if (!members || n < 1) return bfail(nullptr, SGNX_EINVAL, "batch: no members");
  int dev = -1;
  for (int i = 0; i < n; ++i) {
    const sgnx_solver* s = members[i];
    if (!s) return bfail(nullptr, SGNX_EINVAL, "batch: null member");
    if (s->g.variant != 1)
      return bfail(nullptr, SGNX_EINVAL,
                   s->ph.nManning != 0.0
                       ? "batch: members with Manning friction are not supported (no row sweep)"
                       : "batch: members must use the row-sweep kernel");
    if (dev < 0) dev = s->device;
    if (s->device != dev) return bfail(nullptr, SGNX_EINVAL, "batch: members on different devices");
    for (int j = 0; j < i; ++j)
      if (members[j] == s) return bfail(nullptr, SGNX_EINVAL, "batch: a member appears twice");
  }
  sgnx_batch* b = new (std::nothrow) sgnx_batch();
  if (!b) return bfail(nullptr, SGNX_ENOMEM, "batch: out of host memory");
  b->m.assign(members, members + n);
  b->n = n;
  b->device = dev;
  int rc = SGNX_OK;
  auto chk = [&](hipError_t e, const char* what) {
    if (e != hipSuccess && rc == SGNX_OK) {
      rc = (e == hipErrorOutOfMemory) ? SGNX_ENOMEM : SGNX_EDEVICE;
      g_batch_create_error = std::string(what) + ": " + hipGetErrorString(e);
    }
  };
  chk(hipSetDevice(dev), "hipSetDevice");
  chk(hipDeviceGetAttribute(&b->cus, hipDeviceAttributeMultiprocessorCount, dev),
      "hipDeviceGetAttribute");
  chk(hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking), "hipStreamCreate");
  const size_t tables = 4 * (size_t)n * sizeof(BatchMember);
  const size_t args = tables + ((size_t)n + 2) * sizeof(long long);
  chk(hipHostMalloc((void**)&b->h_mem, args), "hipHostMalloc");
  chk(hipMalloc((void**)&b->d_mem, args), "hipMalloc");
  chk(hipHostMalloc((void**)&b->h_post, 3 * (size_t)n * sizeof(double),
                    hipHostMallocMapped | hipHostMallocCoherent), "hipHostMalloc");
  if (rc == SGNX_OK) {
    b->h_ts = reinterpret_cast<long long*>(b->h_mem + 4 * (size_t)n);
    b->d_ts = reinterpret_cast<long long*>(b->d_mem + 4 * (size_t)n);
    std::memset(b->h_post, 0, 3 * (size_t)n * sizeof(double));
    chk(hipHostGetDevicePointer((void**)&b->d_post, b->h_post, 0), "hipHostGetDevicePointer");
  }
  if (rc != SGNX_OK) {
    sgnx_batch_destroy(b);
    return rc;
  }
  if (const char* w = std::getenv("SGNX_SWEEP_WAVES3")) b->waves3 = waves_mask_from_text(w);
  else b->waves3 = members[0]->g.waves3;
  *out = b;
  return SGNX_OK;
}

int sgnx_batch_destroy(sgnx_batch* b) {
  if (!b) return SGNX_EINVAL;
  drop_graph(b);
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  if (b->h_mem) (void)hipHostFree(b->h_mem);
  if (b->h_post) (void)hipHostFree(b->h_post);
  if (b->h_adj) (void)hipHostFree(b->h_adj);
  for (void* p : {(void*)b->d_mem, (void*)b->d_adj})
    if (p) (void)hipFree(p);
  if (b->stream) (void)hipStreamDestroy(b->stream);
  delete b;
  return SGNX_OK;
}

int sgnx_batch_set_waves(sgnx_batch* b, int waves3) {
  if (!b || waves3 < 0 || waves3 > 0xf) return SGNX_EINVAL;
  b->waves3 = waves3;
  drop_graph(b);
  return SGNX_OK;
}

int sgnx_batch_rhs(sgnx_batch* b, const double* const* U, double* const* dU, const double* t) {
  if (!b || !U || !dU || !t) return SGNX_EINVAL;
  const int n = b->n;
  BCHK(b, hipSetDevice(b->device));
  for (int i = 0; i < n; ++i) {
    if (!U[i] || !dU[i] || U[i] == dU[i]) return bfail(b, SGNX_EINVAL, "batch rhs: bad buffers");
    BCHK(b, hipStreamSynchronize(b->m[i]->stream));
  }
  std::vector<int> all(n);
  for (int i = 0; i < n; ++i) all[i] = i;
  const std::vector<int> times = row_multiples(b, all);
  for (int i = 0; i < n; ++i) {
    Stage sa{};
    sa.u = U[i];
    b->h_mem[i] = member_args(b->m[i], U[i], dU[i], sa, t[i], times[i]);
  }
  const long long total = fill_offsets(b, all, b->h_mem);
  BCHK(b, hipMemcpyAsync(b->d_mem, b->h_mem, (size_t)n * sizeof(BatchMember),
                         hipMemcpyHostToDevice, b->stream));
  BCHK(b, hipMemcpyAsync(b->d_ts, b->h_ts, ((size_t)n + 1) * sizeof(long long),
                         hipMemcpyHostToDevice, b->stream));
  BCHK(b, launch_rhs_stage_batch(b->d_mem, b->d_ts, n, total, kPlain, b->waves3 & 1, b->stream,
                                 false, batch_hxr(b)));
  BCHK(b, hipStreamSynchronize(b->stream));
  return SGNX_OK;
}

int sgnx_batch_integrate(sgnx_batch* b, const double* t0, const double* tEnd, const double* dt0,
                         const sgnx_rk_opts* opts, sgnx_rk_stats* stats, int flags) {
  if (!b || !t0 || !tEnd || !dt0 || !opts || !stats) return SGNX_EINVAL;
  const int n = b->n;
  const bool useGraph = (flags & SGNX_BATCH_GRAPH) != 0;
  BCHK(b, hipSetDevice(b->device));
  for (int i = 0; i < n; ++i) BCHK(b, hipStreamSynchronize(b->m[i]->stream));
  std::vector<RkCtl> ctl;
  ctl.reserve(n);
  for (int i = 0; i < n; ++i) ctl.emplace_back(&opts[i], t0[i], tEnd[i], dt0[i], b->m[i]->n(),
                                               nullptr, 0);
  // FSAL heads: k1 = R(U) of every member, one launch
  {
    std::vector<int> all(n);
    for (int i = 0; i < n; ++i) all[i] = i;
    const std::vector<int> times = row_multiples(b, all);
    for (int i = 0; i < n; ++i) {
      sgnx_solver* s = b->m[i];
      Stage sa{};
      sa.u = s->d_U;
      b->h_mem[i] = member_args(s, s->d_U, s->d_k1, sa, ctl[i].t, times[i]);
      ++ctl[i].S.rhsEvals;
    }
    const long long total = fill_offsets(b, all, b->h_mem);
    BCHK(b, hipMemcpyAsync(b->d_mem, b->h_mem, (size_t)n * sizeof(BatchMember),
                           hipMemcpyHostToDevice, b->stream));
    BCHK(b, hipMemcpyAsync(b->d_ts, b->h_ts, ((size_t)n + 1) * sizeof(long long),
                           hipMemcpyHostToDevice, b->stream));
    BCHK(b, launch_rhs_stage_batch(b->d_mem, b->d_ts, n, total, kPlain, b->waves3 & 1,
                                   b->stream, false, batch_hxr(b)));
    // the copies above read the pinned tables asynchronously; the steps below
    // refill them
    BCHK(b, hipStreamSynchronize(b->stream));
  }
  std::vector<int> set, lastSet, times;
  int rc = SGNX_OK;
  for (;;) {
    set.clear();
    for (int i = 0; i < n; ++i)
      if (ctl[i].next()) set.push_back(i);
    if (set.empty()) break;
    if (set != lastSet) {
      times = row_multiples(b, set);
      lastSet = set;
    }
    const int A = (int)set.size();
    // members recording a tape: whether the step's input state is due as a
    // snapshot, and the buffers its stage launches keep their inputs in
    bool taping = false;
    for (int slot = 0; slot < A; ++slot) {
      sgnx_solver* s = b->m[set[slot]];
      taping = taping || tape_recording(s);
      if (tape_recording(s) && tape_step_begin(s))
        return bfail(b, SGNX_EDEVICE, "batch: tape snapshot: " + s->err);
    }
    bool keep = false;
    for (int slot = 0; slot < A; ++slot) {
      const int i = set[slot];
      sgnx_solver* s = b->m[i];
      BS3Launch L[3];
      bs3_launches(s, ctl[i].t, ctl[i].dt, opts[i].atol, opts[i].rtol, L);
      keep = keep || L[0].sa.yOut != nullptr;
      for (int k = 0; k < 3; ++k)
        b->h_mem[(size_t)(k + 1) * n + slot] =
            member_args(s, L[k].sa.u, L[k].dU, L[k].sa, L[k].t, times[slot]);
    }
    const long long total = fill_offsets(b, set, b->h_mem + n);
    b->h_ts[n + 1] = (long long)++b->seq;
    if (useGraph) {
      std::vector<int> rowsNow(A);
      for (int slot = 0; slot < A; ++slot) rowsNow[slot] = times[slot] * b->m[set[slot]]->g.rows;
      if (!b->exec || b->graphSet != set || b->graphKeep != keep || b->graphTotal != total ||
          b->graphRows != rowsNow) {
        BCHK(b, hipStreamSynchronize(b->stream));
        drop_graph(b);
        BCHK(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
        rc = enqueue_step(b, set, total, keep);
        hipGraph_t g = nullptr;
        const hipError_t ec = hipStreamEndCapture(b->stream, &g);
        if (rc) {
          if (g) (void)hipGraphDestroy(g);
          return rc;
        }
        BCHK(b, ec);
        b->graph = g;
        BCHK(b, hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
        b->graphSet = set;
        b->graphKeep = keep;
        b->graphTotal = total;
        b->graphRows = rowsNow;
      }
      BCHK(b, hipGraphLaunch(b->exec, b->stream));
    } else {
      if ((rc = enqueue_step(b, set, total, keep))) return rc;
    }
    // (a tape allocates and frees between steps: it finds the stream at rest)
    if (taping) BCHK(b, hipStreamSynchronize(b->stream));
    if ((rc = wait_posts(b, A))) return rc;
    for (int slot = 0; slot < A; ++slot) {
      const int i = set[slot];
      sgnx_solver* s = b->m[i];
      ctl[i].S.rhsEvals += 3;
      const double tStep = ctl[i].t, dtStep = ctl[i].dt;
      if (ctl[i].finish(b->h_post[3 * slot], b->h_post[3 * slot + 1])) {
        std::swap(s->d_U, s->d_uNew);
        std::swap(s->d_k1, s->d_k4);
        const long rows = s->grows;
        BCHK(b, record_gauges(s, b->stream, ctl[i].t));
        if (tape_recording(s) && tape_accept(s, tStep, dtStep, s->grows > rows ? rows : -1))
          return bfail(b, SGNX_EDEVICE, "batch: tape: " + s->err);
      }
    }
  }
  BCHK(b, hipStreamSynchronize(b->stream));
  for (int i = 0; i < n; ++i) stats[i] = ctl[i].S;
  return SGNX_OK;
}

// ---- autotuning (no counterpart in the reference) --------------------------

int sgnx_autotune(sgnx_solver* s, int reps, int* rows_out, int* waves3_out) {
  if (!s || reps < 1) return SGNX_EINVAL;
  if (s->ph.nManning != 0.0) {
    s->err = "autotune: the row sweep has no Manning friction term";
    return SGNX_EUNSUPPORTED;
  }
  if (hipSetDevice(s->device) != hipSuccess || hipStreamSynchronize(s->stream) != hipSuccess)
    return SGNX_EDEVICE;
  EventPair ev;
  if (hipEventCreate(&ev.a) != hipSuccess || hipEventCreate(&ev.b) != hipSuccess)
    return SGNX_EDEVICE;
  const Geometry keep = s->g;
  const bool keepSet = s->rowsSet;
  auto failed = [&] {
    s->g = keep;
    s->rowsSet = keepSet;
    s->err = "autotune: probe launch failed";
    return SGNX_EDEVICE;
  };
  s->g.variant = 1;
  BS3Launch L[3];
  // ms of `reps` launches of kind k (0: R(U) into k2's buffer; 1..3: a BS3
  // stage at the probe step) with the kind built for three waves or two
  auto timed = [&](int k, bool three, float* ms) -> hipError_t {
    s->g.waves3 = three ? (1 << k) : 0;
    Stage sa{};
    sa.u = s->d_U;
    const Stage& st = (k == 0) ? sa : L[k - 1].sa;
    double* dU = (k == 0) ? s->d_k2 : L[k - 1].dU;
    const GhostTime gt = ghost_time(s, 0.0);
    hipError_t e = launch_rhs_stage(s->g, s->ph, k, st, dU, gt, s->stream);   // warm
    if (e != hipSuccess) return e;
    if ((e = hipEventRecord(ev.a, s->stream)) != hipSuccess) return e;
    for (int r = 0; r < reps; ++r)
      if ((e = launch_rhs_stage(s->g, s->ph, k, st, dU, gt, s->stream)) != hipSuccess) return e;
    if ((e = hipEventRecord(ev.b, s->stream)) != hipSuccess) return e;
    if ((e = hipEventSynchronize(ev.b)) != hipSuccess) return e;
    return hipEventElapsedTime(ms, ev.a, ev.b);
  };
  double best = 1e300;
  int bestRows = keep.rows, bestMask = keep.waves3;
  std::vector<int> heights(std::begin(kTuneRows), std::end(kTuneRows));
  // the default height too, unless it is among them or another one was set (that of
  // a larger grid, with its tall tiles, in any case)
  if ((s->ownTall > 1 || !s->rowsSet) &&
      std::find(heights.begin(), heights.end(), s->ownRows) == heights.end())
    heights.push_back(s->ownRows);
  for (int rows : heights) {
    if (rows > s->g.Ny && rows != kTuneRows[0]) continue;
    take_rows(s, rows);
    bs3_launches(s, 0.0, kProbeDt, 1.0, 0.0, L);
    double tot = 0.0;
    int mask = 0;
    for (int k = 1; k <= 3; ++k) {
      float t2 = 0.0f, t3 = 0.0f;
      if (timed(k, false, &t2) != hipSuccess || timed(k, true, &t3) != hipSuccess) return failed();
      tot += std::min(t2, t3);
      if (t3 < t2) mask |= 1 << k;
    }
    if (tot < best) {
      best = tot;
      bestRows = rows;
      bestMask = mask;
    }
  }
  take_rows(s, bestRows);
  float p2 = 0.0f, p3 = 0.0f;
  if (timed(0, false, &p2) != hipSuccess || timed(0, true, &p3) != hipSuccess) return failed();
  s->g.waves3 = bestMask | (p3 < p2 ? 1 : 0);
  if (rows_out) *rows_out = s->g.rows;
  if (waves3_out) *waves3_out = s->g.waves3;
  return SGNX_OK;
}

int sgnx_batch_autotune(sgnx_batch* b, int reps, int* rows_out, int* waves3_out) {
  if (!b || reps < 1) return SGNX_EINVAL;
  const int n = b->n;
  BCHK(b, hipSetDevice(b->device));
  for (int i = 0; i < n; ++i) BCHK(b, hipStreamSynchronize(b->m[i]->stream));
  drop_graph(b);
  EventPair ev;
  BCHK(b, hipEventCreate(&ev.a));
  BCHK(b, hipEventCreate(&ev.b));
  std::vector<int> all(n);
  for (int i = 0; i < n; ++i) all[i] = i;
  int maxNy = 1;
  for (sgnx_solver* s : b->m) maxNy = std::max(maxNy, s->g.Ny);
  const size_t nn = (size_t)n;
  // Fill the tables of every kind for a candidate height (0: the rule's). A member
  // with its default height takes the nearest multiple of it, as it will in the
  // batch; one whose height was set, the candidate.
  auto fill = [&](int rows) -> long long {
    const int packed = rows ? rows : packed_rows(b, all);
    for (int i = 0; i < n; ++i) {
      sgnx_solver* s = b->m[i];
      Geometry g = s->g;
      if (s->rowsSet && rows) g.rows = rows;
      const int times = row_multiple(s, packed);
      const GhostTime gt = ghost_time(s, 0.0);
      BS3Launch L[3];
      bs3_launches(s, 0.0, kProbeDt, 1.0, 0.0, L);
      Stage sa{};
      sa.u = s->d_U;
      b->h_mem[i] = sweep_member(g, s->ph, s->d_U, s->d_k2, gt, sa, times);
      for (int k = 0; k < 3; ++k)
        b->h_mem[(size_t)(k + 1) * nn + i] =
            sweep_member(g, s->ph, L[k].sa.u, L[k].dU, ghost_time(s, L[k].t), L[k].sa, times);
    }
    return fill_offsets(b, all, b->h_mem);
  };
  auto timed = [&](int k, bool three, long long total, float* ms) -> hipError_t {
    hipError_t e = launch_rhs_stage_batch(b->d_mem + k * nn, b->d_ts, n, total, k, three,
                                          b->stream, false, batch_hxr(b));
    if (e != hipSuccess) return e;
    if ((e = hipEventRecord(ev.a, b->stream)) != hipSuccess) return e;
    for (int r = 0; r < reps; ++r)
      if ((e = launch_rhs_stage_batch(b->d_mem + k * nn, b->d_ts, n, total, k, three,
                                      b->stream, false, batch_hxr(b))) != hipSuccess)
        return e;
    if ((e = hipEventRecord(ev.b, b->stream)) != hipSuccess) return e;
    if ((e = hipEventSynchronize(ev.b)) != hipSuccess) return e;
    return hipEventElapsedTime(ms, ev.a, ev.b);
  };
  // the rule's heights are a candidate where a member has its default one
  bool rule = false;
  for (const sgnx_solver* s : b->m) rule = rule || !s->rowsSet;
  std::vector<int> heights;
  if (rule) heights.push_back(0);
  for (int rows : kTuneRows)
    if (rows <= maxNy || rows == kTuneRows[0]) heights.push_back(rows);
  double best = 1e300;
  int bestRows = heights[0], bestMask = b->waves3;
  for (int rows : heights) {
    const long long total = fill(rows);
    BCHK(b, hipMemcpyAsync(b->d_mem, b->h_mem, 4 * nn * sizeof(BatchMember),
                           hipMemcpyHostToDevice, b->stream));
    BCHK(b, hipMemcpyAsync(b->d_ts, b->h_ts, (nn + 1) * sizeof(long long),
                           hipMemcpyHostToDevice, b->stream));
    double tot = 0.0;
    int mask = 0;
    for (int k = 1; k <= 3; ++k) {
      float t2 = 0.0f, t3 = 0.0f;
      BCHK(b, timed(k, false, total, &t2));
      BCHK(b, timed(k, true, total, &t3));
      tot += std::min(t2, t3);
      if (t3 < t2) mask |= 1 << k;
    }
    BCHK(b, hipStreamSynchronize(b->stream));
    if (tot < best) {
      best = tot;
      bestRows = rows;
      bestMask = mask;
    }
  }
  const long long total = fill(bestRows);
  BCHK(b, hipMemcpyAsync(b->d_mem, b->h_mem, 4 * nn * sizeof(BatchMember),
                         hipMemcpyHostToDevice, b->stream));
  BCHK(b, hipMemcpyAsync(b->d_ts, b->h_ts, (nn + 1) * sizeof(long long), hipMemcpyHostToDevice,
                         b->stream));
  float p2 = 0.0f, p3 = 0.0f;
  BCHK(b, timed(0, false, total, &p2));
  BCHK(b, timed(0, true, total, &p3));
  BCHK(b, hipStreamSynchronize(b->stream));
  b->rows = bestRows;
  b->waves3 = bestMask | (p3 < p2 ? 1 : 0);
  for (sgnx_solver* s : b->m) {
    // (a default height stays: alone, a member is faster with it, and its norm's
    // partial sums follow it in the batch too)
    if (s->rowsSet && bestRows) take_rows(s, bestRows);
    s->g.waves3 = b->waves3;
  }
  if (rows_out) *rows_out = bestRows ? bestRows : packed_rows(b, all);
  if (waves3_out) *waves3_out = b->waves3;
  return SGNX_OK;
}

// The reverse sweeps of every member's tape in lockstep, aligned at the last
// step: iteration k reverses step N_m - 1 - k of each member that has it, with
// one launch per kind over all of them (the gauge cotangents, the stage
// recomputation of members whose tape keeps no stage inputs: R(u), then the
// stage-2 launch that writes y2 and forms y3; the three products), each
// member on its own buffers. The arithmetic is that of sgnx_adjoint on each
// member alone, so the cotangents are bit for bit the same. Every member's
// tape must hold every step's snapshot. One member, and two large ones whose
// products would hardly end sooner in one launch each, are swept by their own
// calls back to back (same bits). A reversed step with kept stages and with
// recomputed ones, us, back to back -> in lockstep:
//   16 x 128x64   1143 ->  628  1604 ->  896     2 x 128x64   143 -> 120   199 -> 167
//    8 x 128x64    572 ->  354   802 ->  503     2 x 220x110  254 -> 245   359 -> 354
//    8 x 256x128  1301 -> 1140  1882 -> 1627     2 x 200x100  222 -> 218   314 -> 325
//    3 x 450x225  1255 -> 1200  1906 -> 1750     2 x 300x150  407 -> 404   591 -> 616
//    3 x 1024x512 6226 -> 5987  8991 -> 8810     2 x 450x225  857 -> 877  1304 -> 1283
// By vjp_step_cost the pairs take 1.37, 1.15, 1.11, 1.07 and 1.00 times the
// lockstep's time back to back; the line lies at 1.12. A pair with a small member
// (less than six one-row tiles per compute unit) hides that one's launches in the
// other's: 92x63 and 334x197 374 -> 355 and 541 -> 504. One of 64x32: 43 -> 60.
int sgnx_batch_adjoint(sgnx_batch* b, const double* const* Ubar_final,
                       const double* const* gauge_bar, double* const* U0bar,
                       double* const* theta_bar, int mem) {
  if (!b || !U0bar) return SGNX_EINVAL;
  if (mem != SGNX_MEM_HOST && mem != SGNX_MEM_DEVICE)
    return bfail(b, SGNX_EINVAL, "batch adjoint: bad memory kind");
  const int n = b->n;
  BCHK(b, hipSetDevice(b->device));
  // the products' tile heights for all members, unless set from outside
  std::vector<const Geometry*> gs;
  bool given = false;
  for (const sgnx_solver* s : b->m) {
    gs.push_back(&s->g);
    given = given || s->vrowsSet;
  }
  int vrows[2] = {0, 0};
  if (!given)
    for (int k = 0; k < 2; ++k) vrows[k] = vjp_rows(gs.data(), n, b->cus, k == 1);
  bool own = n == 1;
  if (n == 2 && std::min(vjp_row_tiles(*gs[0]), vjp_row_tiles(*gs[1])) >= 6LL * b->cus) {
    double alone = 0.0;
    for (const Geometry*& g : gs) alone += vjp_step_cost(&g, 1, b->cus, g->vrows);
    own = alone < 1.12 * vjp_step_cost(gs.data(), n, b->cus, vrows[0] ? vrows : gs[0]->vrows);
  }
  if (own) {
    for (int i = 0; i < n; ++i) {
      sgnx_solver* s = b->m[i];
      if (!U0bar[i]) return bfail(b, SGNX_EINVAL, "batch adjoint: U0bar missing for a member");
      AdjTape* t = nullptr;
      int rc = adjoint_begin(s, true, &t);
      if (!rc)
        rc = sgnx_adjoint(s, Ubar_final ? Ubar_final[i] : nullptr,
                          gauge_bar ? gauge_bar[i] : nullptr, U0bar[i],
                          theta_bar ? theta_bar[i] : nullptr, mem);
      if (rc) return bfail(b, rc, "batch adjoint, member " + std::to_string(i) + ": " + s->err);
    }
    return SGNX_OK;
  }
  // (work on the null stream that a member's own stream would wait for)
  if (mem == SGNX_MEM_DEVICE) BCHK(b, hipStreamSynchronize(nullptr));
  std::vector<AdjTape*> tp(n, nullptr);
  std::vector<const double*> gb(n, nullptr);
  long Nmax = 0;
  for (int i = 0; i < n; ++i) {
    sgnx_solver* s = b->m[i];
    if (!U0bar[i]) return bfail(b, SGNX_EINVAL, "batch adjoint: U0bar missing for a member");
    BCHK(b, hipStreamSynchronize(s->stream));
    int rc = adjoint_begin(s, true, &tp[i]);
    if (!rc)
      rc = adjoint_inputs(s, tp[i], Ubar_final ? Ubar_final[i] : nullptr,
                          gauge_bar ? gauge_bar[i] : nullptr, mem, b->stream, &gb[i]);
    if (rc) return bfail(b, rc, "batch adjoint, member " + std::to_string(i) + ": " + s->err);
    tp[i]->recomputed = tp[i]->peakSlots = 0;
    Nmax = std::max(Nmax, (long)tp[i]->t.size());
  }
  // argument arena: gauges, two RHS tables (R(u); the stage-2 launch keeping
  // y2 and forming y3) + offsets, three products + offsets
  auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
  const size_t nn = (size_t)n;
  const size_t oG = 0, oR1 = up(oG + nn * sizeof(GaugeMember));
  const size_t oR2 = up(oR1 + nn * sizeof(BatchMember)), oRT = up(oR2 + nn * sizeof(BatchMember));
  const size_t oV3 = up(oRT + (nn + 1) * sizeof(long long));
  const size_t oV2 = up(oV3 + nn * sizeof(VjpMember)), oV1 = up(oV2 + nn * sizeof(VjpMember));
  const size_t oVT = up(oV1 + nn * sizeof(VjpMember));
  const size_t oWT = up(oVT + (nn + 1) * sizeof(long long));   // the third product's offsets
  const size_t total = up(oWT + (nn + 1) * sizeof(long long));
  if (b->adjCap < total) {
    if (b->h_adj) (void)hipHostFree(b->h_adj);
    if (b->d_adj) (void)hipFree(b->d_adj);
    b->h_adj = nullptr;
    b->d_adj = nullptr;
    b->adjCap = 0;
    BCHK(b, hipHostMalloc((void**)&b->h_adj, total, hipHostMallocDefault));
    BCHK(b, hipMalloc((void**)&b->d_adj, total));
    b->adjCap = total;
  }
  auto* hG = reinterpret_cast<GaugeMember*>(b->h_adj + oG);
  auto* hR1 = reinterpret_cast<BatchMember*>(b->h_adj + oR1);
  auto* hR2 = reinterpret_cast<BatchMember*>(b->h_adj + oR2);
  auto* hRT = reinterpret_cast<long long*>(b->h_adj + oRT);
  auto* hV3 = reinterpret_cast<VjpMember*>(b->h_adj + oV3);
  auto* hV2 = reinterpret_cast<VjpMember*>(b->h_adj + oV2);
  auto* hV1 = reinterpret_cast<VjpMember*>(b->h_adj + oV1);
  auto* hVT = reinterpret_cast<long long*>(b->h_adj + oVT);
  auto* hWT = reinterpret_cast<long long*>(b->h_adj + oWT);
  auto dptr = [&](size_t off) { return b->d_adj + off; };
  std::vector<int> all(n);
  for (int i = 0; i < n; ++i) all[i] = i;
  const std::vector<int> times = row_multiples(b, all);
  for (long k = 0; k < Nmax; ++k) {
    int A = 0, Rn = 0;   // members in this step; of those, the ones that recompute stages
    long long rAcc = 0, vAcc = 0, wAcc = 0;
    for (int i = 0; i < n; ++i) {
      AdjTape* T = tp[i];
      const long m = (long)T->t.size() - 1 - k;
      if (m < 0) continue;
      sgnx_solver* s = b->m[i];
      const double t = T->t[m], dt = T->dt[m];
      const double* u = T->snap[m];
      GaugeMember gq{};
      if (gb[i] && T->row[m] >= 0 && T->row[m] < s->grows) {
        gq.Gb = gb[i] + (size_t)T->row[m] * s->nG;
        gq.nodes = s->d_gnodes;
        gq.n = s->nG;
        gq.lam = T->lam;
        gq.thetaBar = T->thb;
      }
      hG[A] = gq;
      // stage inputs y2, y3: kept by the taped run, or recomputed here
      const bool kept = m < (long)T->y2s.size();
      const double* y2 = kept ? T->y2s[m] : s->d_tmp;
      const double* y3 = kept ? T->y3s[m] : s->d_k3;
      if (!kept) {
        Stage s1{};
        s1.u = u;
        hR1[Rn] = member_args(s, u, s->d_k1, s1, t, times[i]);
        // the forward's stage-2 launch, keeping its input and forming the
        // next one: y2, k2 = R(y2) and y3 = u + 3dt/4 k2
        Stage s2{};
        s2.u = u;
        s2.k1 = s->d_k1;
        s2.a = 0.5 * dt;
        s2.yOut = s->d_tmp;
        s2.y3Out = s->d_k3;
        s2.a3 = 0.75 * dt;
        hR2[Rn] = member_args(s, u, nullptr, s2, t + 0.5 * dt, times[i]);
        hRT[Rn] = rAcc;
        rAcc += packed_tiles(hR1[Rn].nTiles);
        ++Rn;
      }
      VjpArgs p[3];
      step_products(T, u, y2, y3, dt, T->thb, p);
      Geometry vg = s->g;
      if (vrows[0]) std::memcpy(vg.vrows, vrows, sizeof vrows);
      hV3[A] = vjp_member(vg, s->ph, p[0], ghost_time(s, t + 0.75 * dt));
      hV2[A] = vjp_member(vg, s->ph, p[1], ghost_time(s, t + 0.5 * dt));
      hV1[A] = vjp_member(vg, s->ph, p[2], ghost_time(s, t));
      std::swap(T->lam, T->lamNew);   // (the tables hold this step's; the next reads its result)
      hVT[A] = vAcc;
      hWT[A] = wAcc;
      vAcc += packed_tiles(hV3[A].nTiles);
      wAcc += packed_tiles(hV1[A].nTiles);
      ++A;
    }
    hRT[Rn] = rAcc;
    hVT[A] = vAcc;
    hWT[A] = wAcc;
    BCHK(b, hipMemcpyAsync(b->d_adj, b->h_adj, total, hipMemcpyHostToDevice, b->stream));
    const auto* dR1 = reinterpret_cast<const BatchMember*>(dptr(oR1));
    const auto* dR2 = reinterpret_cast<const BatchMember*>(dptr(oR2));
    const auto* dRT = reinterpret_cast<const long long*>(dptr(oRT));
    BCHK(b, launch_gauge_bar_batch(reinterpret_cast<const GaugeMember*>(dptr(oG)), A, b->stream));
    if (Rn > 0) {
      BCHK(b, launch_rhs_stage_batch(dR1, dRT, Rn, rAcc, kPlain, b->waves3 & 1, b->stream, false,
                                     batch_hxr(b)));
      BCHK(b, launch_rhs_stage_batch(dR2, dRT, Rn, rAcc, kAxpy, (b->waves3 >> 1) & 1, b->stream,
                                     true, batch_hxr(b)));
    }
    const size_t oV[3] = {oV3, oV2, oV1};
    for (int k = 0; k < 3; ++k)
      BCHK(b, launch_rhs_vjp_batch(
                  reinterpret_cast<const VjpMember*>(dptr(oV[k])),
                  reinterpret_cast<const long long*>(dptr(k < 2 ? oVT : oWT)), A,
                  k < 2 ? vAcc : wAcc, k + 1, b->stream));
    // the arena is refilled for the next iteration
    BCHK(b, hipStreamSynchronize(b->stream));
  }
  for (int i = 0; i < n; ++i) {
    int rc = adjoint_outputs(b->m[i], tp[i], U0bar[i], theta_bar ? theta_bar[i] : nullptr, mem,
                             b->stream);
    if (rc) return bfail(b, rc, "batch adjoint: " + b->m[i]->err);
  }
  BCHK(b, hipStreamSynchronize(b->stream));
  return SGNX_OK;
}

}  // extern "C"
