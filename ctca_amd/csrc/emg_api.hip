// emg_api.hip -- the extern "C" entry points of libemgpu (include/emgpu.h).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "emg_internal.h"

namespace emg {

static thread_local std::string g_last_error;

int set_error(int code, const std::string &msg) {
  g_last_error = msg;
  // a failed allocation also sets HIP's last error, which the launch checks
  // of later calls read: the failure is reported here, so clear it
  if (code == EMG_ERR_NOMEM) (void)hipGetLastError();
  return code;
}

int hip_check(hipError_t e, const char *what) {
  if (e == hipSuccess) return EMG_OK;
  (void)hipGetLastError();  // reported now, not again by a later launch check
  return set_error(e == hipErrorOutOfMemory ? EMG_ERR_NOMEM : EMG_ERR_HIP,
                   std::string(what) + ": " + hipGetErrorString(e));
}

// ---- kernel timing: event pairs recorded around launches, accumulated lazily
namespace {
struct EvPair {
  hipEvent_t a, b;
  int kind;
};
struct TimerState {
  std::vector<EvPair> pending;
  std::vector<EvPair> free_pairs;
  EvPair open[kTNum];
  bool is_open[kTNum] = {false, false, false, false, false};
};
}  // namespace

static TimerState *tstate(emg_ctx *c);

static void timer_flush(emg_ctx *c) {
  TimerState *t = tstate(c);
  for (EvPair &p : t->pending) {
    float ms = 0.f;
    if (hipEventSynchronize(p.b) == hipSuccess && hipEventElapsedTime(&ms, p.a, p.b) == hipSuccess) {
      c->timers[p.kind].total_ms += ms;
      c->timers[p.kind].last_ms = ms;
      c->timers[p.kind].launches += 1;
    }
    t->free_pairs.push_back(p);
  }
  t->pending.clear();
}

void timer_begin(emg_ctx *c, int kind) {
  if (!c->timing) return;
  TimerState *t = tstate(c);
  if (t->pending.size() >= 512) timer_flush(c);
  EvPair p;
  if (!t->free_pairs.empty()) {
    p = t->free_pairs.back();
    t->free_pairs.pop_back();
  } else {
    if (hipEventCreate(&p.a) != hipSuccess || hipEventCreate(&p.b) != hipSuccess) return;
  }
  p.kind = kind;
  (void)hipEventRecord(p.a, c->stream);
  t->open[kind] = p;
  t->is_open[kind] = true;
}

void timer_end(emg_ctx *c, int kind) {
  if (!c->timing) return;
  TimerState *t = tstate(c);
  if (!t->is_open[kind]) return;
  EvPair p = t->open[kind];
  (void)hipEventRecord(p.b, c->stream);
  t->pending.push_back(p);
  t->is_open[kind] = false;
}

// declared in the other translation units
int init_device_into(emg_ctx *c, State64 &st, const emg_device_species *spec, int nspec,
                     uint64_t seed);
int64_t energy64_part_need(int nspec);

namespace {

constexpr int kFlagPreside = 8;
constexpr int kFlagPid = 16;
constexpr int kFlagDead = 32;  // a record with nid < 0 in an upload that expected none

// AoS pbuf records -> SoA FP64 state, validating each record
// (near += the records that lie in the 8^3 tile of the one before them, over
// every kNearSample-th block)
constexpr int kNearSample = 8;
__global__ __launch_bounds__(kBlock) void k_split(const emg_particle *rec, int64_t n, State64 st,
                                                  int64_t dst0, Grid g, int *flag, int need_pid0,
                                                  int *near) {
  int64_t m = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  const bool act = m < n;
  emg_particle r{};
  if (act) r = rec[m];
  if (blockIdx.x % kNearSample == 0) {
    const int tile = ((int)r.z >> 3) * 1048573 + ((int)r.y >> 3) * 1021 + ((int)r.x >> 3);
    const bool eq = __shfl_up(tile, 1) == tile;
    const int same = __popcll(__ballot(act && eq && __lane_id() != 0));
    if (__lane_id() == 0 && same) atomicAdd(near, same);
  }
  if (!act) return;
  if (r.nid < 0) {  // the host drops the dead records and uploads again
    atomicOr(flag, kFlagDead);
    return;
  }
  bool ok = (r.x >= 0.0) && (r.x <= g.slx) && (r.y >= 0.0) && (r.y <= g.sly) && (r.z >= 0.0) &&
            (r.z <= g.slz) && (r.vx == r.vx) && (r.vy == r.vy) && (r.vz == r.vz) &&
            (fabs(r.vx) < 1e300) && (fabs(r.vy) < 1e300) && (fabs(r.vz) < 1e300);
  if (!ok) atomicOr(flag, kFlagDomain);
  if (r.preside != 0) atomicOr(flag, kFlagPreside);
  if (need_pid0 && r.pid != 0) atomicOr(flag, kFlagPid);
  int64_t d = dst0 + m;
  st.x[d] = ok ? r.x : 0.0;
  st.y[d] = ok ? r.y : 0.0;
  st.z[d] = ok ? r.z : 0.0;
  st.vx[d] = ok ? r.vx : 0.0;
  st.vy[d] = ok ? r.vy : 0.0;
  st.vz[d] = ok ? r.vz : 0.0;
  st.pid[d] = r.pid;
}

__global__ __launch_bounds__(kBlock) void k_join(State64 st, int64_t src0, int64_t n, int spec,
                                                 emg_particle *rec) {
  int64_t m = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (m >= n) return;
  int64_t s = src0 + m;
  emg_particle r;
  r.x = st.x[s];
  r.y = st.y[s];
  r.z = st.z[s];
  r.vx = st.vx[s];
  r.vy = st.vy[s];
  r.vz = st.vz[s];
  r.pid = st.pid[s];
  r.preside = 0;
  r.nid = 0;
  r.spec = spec;
  rec[m] = r;
}

template <typename T>
int dalloc(emg_ctx *c, T **p, size_t count, const char *what) {
  if (count == 0) count = 1;
  if (dev_malloc(c, p, sizeof(T) * count)) return EMG_OK;
  return set_error(EMG_ERR_NOMEM, std::string("device allocation failed: ") + what);
}

void dfree(void *p) {
  if (p) (void)hipFree(p);
}

void free_state64(State64 &st) {
  dfree(st.x);
  dfree(st.y);
  dfree(st.z);
  dfree(st.vx);
  dfree(st.vy);
  dfree(st.vz);
  dfree(st.pid);
  st = State64{};
}

// all of a state's arrays or none
int alloc_state64(emg_ctx *c, State64 &st, int64_t cap) {
  int rc;
  if ((rc = dalloc(c, &st.x, cap, "x")) || (rc = dalloc(c, &st.y, cap, "y")) ||
      (rc = dalloc(c, &st.z, cap, "z")) || (rc = dalloc(c, &st.vx, cap, "vx")) ||
      (rc = dalloc(c, &st.vy, cap, "vy")) || (rc = dalloc(c, &st.vz, cap, "vz")) ||
      (rc = dalloc(c, &st.pid, cap, "pid")))
    free_state64(st);
  return rc;
}

}  // namespace

// The records of an upload with nid >= 0: how many come before a record, and a
// range of them without the others.
struct LivingRecords {
  static constexpr int64_t kStep = 1024;
  const emg_particle *rec = nullptr;
  std::vector<int64_t> at;  // living records before every kStep-th one
  int count(emg_ctx *c, const emg_particle *r, int64_t n) {
    rec = r;
    const int64_t steps = (n + kStep - 1) / kStep;
    try {
      at.assign((size_t)steps + 1, 0);
    } catch (const std::bad_alloc &) {
      return set_error(EMG_ERR_NOMEM, "host allocation failed");
    }
    const int rc = io_ranges(c, steps, sizeof(emg_particle) * kStep, [&](int64_t a, int64_t b) {
      for (int64_t k = a; k < b; k++) at[k + 1] = alive(k * kStep, std::min(n, (k + 1) * kStep));
    });
    for (int64_t k = 0; k < steps; k++) at[k + 1] += at[k];
    return rc;
  }
  int64_t alive(int64_t a, int64_t b) const {
    int64_t k = 0;
    for (; a < b; a++) k += rec[a].nid >= 0;
    return k;
  }
  int64_t before(int64_t m) const { return at[m / kStep] + alive(m / kStep * kStep, m); }
  // the living ones of n records from m on, to out; their bytes
  size_t copy(int64_t m, int64_t n, emg_particle *out) const {
    int64_t k = 0;
    for (int64_t a = m; a < m + n; a++)
      if (rec[a].nid >= 0) out[k++] = rec[a];
    return sizeof(emg_particle) * (size_t)k;
  }
};

int flags_error(emg_ctx *c) {
  const int f = *c->hflag;
  if (f == 0) return EMG_OK;
  launch_zero(c->dflag, sizeof(int), c->stream);
  (void)hipStreamSynchronize(c->stream);
  if (f & kFlagSpillLost)
    return set_error(EMG_ERR_CAPACITY, "re-bucketing overflowed the spill region: particles lost");
  if (f & kFlagDomain)
    return set_error(EMG_ERR_DOMAIN, "particle outside [0, L] or non-finite (clamped)");
  if (f & kFlagFar)
    return set_error(EMG_ERR_DOMAIN, "particle moved more than one box length in one step");
  if (f & kFlagPreside)
    return set_error(EMG_ERR_UNSUPPORTED, "only alive records (preside == 0) are supported");
  if (f & kFlagPid)
    return set_error(EMG_ERR_UNSUPPORTED, "EMG_FP32_FIXED does not carry pid: upload pid = 0");
  return set_error(EMG_ERR_HIP, "unknown device flag");
}

bool capturing(emg_ctx *c) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(c->stream, &st) == hipSuccess && st == hipStreamCaptureStatusNone)
    return false;
  (void)hipGetLastError();
  return true;
}

}  // namespace emg

using namespace emg;

struct emg_timer_holder {
  TimerState t;
};

namespace emg {
static TimerState *tstate(emg_ctx *c) {
  // the TimerState lives right after the context in one allocation
  return &reinterpret_cast<emg_timer_holder *>(c + 1)->t;
}
}  // namespace emg

// Staging of emg_get_rho_noalloc: a file-scope device array instead of a
// per-call allocation.  Every GPU that runs the library holds its own copy
// until the process ends; all calls on one GPU share it.  Host code uses the
// device address hipGetSymbolAddress gives for the current device (taken
// once per device, at the first emg_create on it), never the array's name.
namespace emg {
constexpr int64_t kScratchDoubles = int64_t(1) << 24;  // 128 MiB
static __device__ __align__(256) double scratch[kScratchDoubles];
static std::mutex g_scratch_mu;
static std::vector<double *> g_scratch_dev;  // per device id

// the scratch address on the current device (`dev`)
static int scratch_address(int dev, double **out) {
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (dev < 0) return set_error(EMG_ERR_ARG, "device id");
  if ((size_t)dev >= g_scratch_dev.size()) g_scratch_dev.resize((size_t)dev + 1, nullptr);
  if (!g_scratch_dev[dev]) {
    void *p = nullptr;
    int rc = hip_check(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "scratch address");
    if (rc) return rc;
    g_scratch_dev[dev] = static_cast<double *>(p);
  }
  *out = g_scratch_dev[dev];
  return EMG_OK;
}
}  // namespace emg

#define CTX_CHECK(c)                                                   \
  do {                                                                 \
    if (!(c)) return set_error(EMG_ERR_ARG, "null context");           \
    if (hipSetDevice((c)->device) != hipSuccess)                        \
      return set_error(EMG_ERR_HIP, "hipSetDevice failed");            \
  } while (0)

extern "C" {

int emg_last_error(char *buf, size_t len) {
  if (!buf || len == 0) return EMG_ERR_ARG;
  std::snprintf(buf, len, "%s", g_last_error.c_str());
  return EMG_OK;
}

int emg_create(const emg_config *cfg, emg_ctx **out) {
  if (!cfg || !out) return set_error(EMG_ERR_ARG, "null argument");
  *out = nullptr;
  if (cfg->nspec < 1 || cfg->nspec > EMG_MAX_SPECIES)
    return set_error(EMG_ERR_ARG, "nspec must be 1..EMG_MAX_SPECIES");
  for (int d = 0; d < 3; d++)
    if (cfg->n[d] < 2) return set_error(EMG_ERR_ARG, "need at least 2 cells per axis");
  if (cfg->precision != EMG_PLAIN_FP64 && cfg->precision != EMG_FP32_FIXED)
    return set_error(EMG_ERR_ARG, "unknown precision form");
  if (cfg->sort_every < 0) return set_error(EMG_ERR_ARG, "sort_every must be >= 0");
  if (cfg->sort_every != 0 && cfg->precision != EMG_PLAIN_FP64)
    return set_error(EMG_ERR_ARG, "sort_every applies to EMG_PLAIN_FP64 only");
  for (int s = 0; s < cfg->nspec; s++)
    if (cfg->capacity[s] < 0) return set_error(EMG_ERR_ARG, "negative capacity");

  void *mem = ::operator new(sizeof(emg_ctx) + sizeof(emg_timer_holder), std::nothrow);
  if (!mem) return set_error(EMG_ERR_NOMEM, "host allocation failed");
  std::memset(mem, 0, sizeof(emg_ctx));
  emg_ctx *c = static_cast<emg_ctx *>(mem);
  new (reinterpret_cast<emg_timer_holder *>(c + 1)) emg_timer_holder();
  c->cfg = *cfg;
  int rc = hip_check(hipGetDevice(&c->device), "hipGetDevice");
  if (!rc) rc = scratch_address(c->device, &c->scratch);
  if (rc) {
    emg_destroy(c);
    return rc;
  }
  rc = hip_check(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking), "stream create");
  if (rc) {
    emg_destroy(c);
    return rc;
  }
  c->own_stream = true;
  io_open(c);
  c->g.nx = cfg->n[0];
  c->g.ny = cfg->n[1];
  c->g.nz = cfg->n[2];
  c->g.slx = (double)cfg->n[0];
  c->g.sly = (double)cfg->n[1];
  c->g.slz = (double)cfg->n[2];
  for (int b = 0; (1 << b) < cfg->n[0]; b++) c->g.cbx = b + 1;
  for (int b = 0; (1 << b) < cfg->n[1]; b++) c->g.cby = b + 1;
  c->ncell = (int64_t)cfg->n[0] * cfg->n[1] * cfg->n[2];
  c->sp.nspec = cfg->nspec;
  int64_t off = 0;
  for (int s = 0; s < cfg->nspec; s++) {
    c->sp.off[s] = off;
    c->sp.cnt[s] = 0;
    c->sp.q[s] = cfg->q[s];
    c->sp.qm[s] = cfg->qm[s];
    off += cfg->capacity[s];
  }
  c->sp.off[cfg->nspec] = off;
  c->cap_total = off;
  int nsp = cfg->nspec;
  if ((rc = dalloc(c, &c->dflag, 2, "flag")) ||
      (rc = dalloc(c, (double **)&c->face, (size_t)(face_len(c->g) * nsp), "upper-face charge"))) {
    emg_destroy(c);
    return rc;
  }
  // the flag, and after it the sums that reduction kernels hand to the host
  if (hipHostMalloc((void **)&c->hflag, sizeof(double) * (1 + 3 * EMG_MAX_SPECIES),
                    hipHostMallocDefault) != hipSuccess) {
    c->hflag = nullptr;
    emg_destroy(c);
    return set_error(EMG_ERR_NOMEM, "pinned flag");
  }
  c->hsum = reinterpret_cast<double *>(c->hflag) + 1;
  launch_zero(c->dflag, 2 * sizeof(int), c->stream);
  if (cfg->precision == EMG_PLAIN_FP64) {
    int64_t nn = (int64_t)(cfg->n[0] + 1) * (cfg->n[1] + 1) * (cfg->n[2] + 1);
    if ((rc = alloc_state64(c, c->s64, c->cap_total)) || (rc = dalloc(c, &c->node64, 8 * nn, "nodal E/B")) ||
        (rc = dalloc(c, &c->rho64, c->ncell * nsp, "rho")) ||
        (rc = dalloc(c, &c->j64, 3 * c->ncell * nsp, "current")) ||
        (rc = dalloc(c, &c->ke_part, energy64_part_need(nsp), "energy partials"))) {
      emg_destroy(c);
      return rc;
    }
  } else {
    if ((rc = fx_alloc(c, c->cap_total)) || (rc = dalloc(c, &c->node32, 8 * c->ncell, "nodal E/B")) ||
        (rc = dalloc(c, &c->rhofx, c->ncell * nsp, "rho")) ||
        (rc = dalloc(c, &c->jfx, 3 * c->ncell * nsp, "current"))) {
      emg_destroy(c);
      return rc;
    }
  }
  rc = hip_check(hipStreamSynchronize(c->stream), "create");
  if (rc) {
    emg_destroy(c);
    return rc;
  }
  *out = c;
  return EMG_OK;
}

int emg_destroy(emg_ctx *c) {
  if (!c) return EMG_OK;
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  free_state64(c->s64);
  free_state64(c->t64);
  dfree(c->lam);
  for (int k = 0; k < kStateSlots; k++) free_state64(c->slot[k]);
  dfree(c->adj_e);
  dfree(c->adj_g);
  dfree(c->adj_sum);
  dfree(c->bins.count);
  dfree(c->bins.start);
  dfree(c->bins.rec);
  FxBuckets &B = c->fx;
  for (int k = 0; k < 2; k++) {
    dfree(B.st[k].cell);
    dfree(B.st[k].fx);
    dfree(B.st[k].fy);
    dfree(B.st[k].fz);
    dfree(B.st[k].vx);
    dfree(B.st[k].vy);
    dfree(B.st[k].vz);
    dfree(B.st[k].pid);
    dfree(B.start[k]);
    dfree(B.count[k]);
    dfree(B.spill[k]);
    dfree(B.nst[k]);
    dfree(B.cap[k]);
    dfree(B.ob[k]);
    dfree(B.pre[k]);
  }
  dfree(B.stay);
  dfree(B.extra);
  dfree(B.hist);
  dfree(B.cursor);
  dfree(B.shist[0]);
  dfree(B.shist[1]);
  dfree(B.plan_word);
  dfree(B.plan_ticket);
  dfree(B.scur);
  dfree(B.spre);
  dfree(B.spl);
  dfree(c->eb_dev);
  dfree(c->fe_buf);
  dfree(c->sort_rec);
  es_solver_free(c);
  dfree(c->bk_dev);
  dfree(c->node64);
  dfree(c->node32);
  dfree(c->rho64);
  dfree(c->rhofx);
  dfree(c->j64);
  dfree(c->jfx);
  dfree(c->ke_part);
  dfree(c->face);
  dfree(c->runs[0]);
  dfree(c->runs[1]);
  dfree(c->run_base);
  dfree(c->sort_count);
  dfree(c->sort_start);
  dfree(c->scan_tmp);
  dfree(c->dflag);
  if (c->hflag) (void)hipHostFree(c->hflag);
  io_close(c);
  TimerState *t = tstate(c);
  for (EvPair &p : t->pending) t->free_pairs.push_back(p);
  for (EvPair &p : t->free_pairs) {
    (void)hipEventDestroy(p.a);
    (void)hipEventDestroy(p.b);
  }
  for (int k = 0; k < kTNum; k++)
    if (t->is_open[k]) {
      (void)hipEventDestroy(t->open[k].a);
      (void)hipEventDestroy(t->open[k].b);
    }
  if (c->stream && c->own_stream) (void)hipStreamDestroy(c->stream);
  reinterpret_cast<emg_timer_holder *>(c + 1)->~emg_timer_holder();
  ::operator delete(c);
  return EMG_OK;
}

int emg_set_stream(emg_ctx *c, void *stream) {
  CTX_CHECK(c);
  int rc = hip_check(hipStreamSynchronize(c->stream), "stream synchronize");
  if (rc) return rc;
  if (c->own_stream && stream) {
    (void)hipStreamDestroy(c->stream);
    c->own_stream = false;
  }
  if (stream) {
    c->stream = (hipStream_t)stream;
  } else if (!c->own_stream) {
    rc = hip_check(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking), "stream create");
    if (rc) return rc;
    c->own_stream = true;
  }
  return es_solver_stream(c);
}

int emg_synchronize(emg_ctx *c) {
  CTX_CHECK(c);
  int rc = hip_check(hipGetLastError(), "kernel launch");
  if (rc) return rc;
  return read_flags(c);
}

int emg_upload_particles(emg_ctx *c, const emg_particle *pbuf, const int64_t *counts, int32_t nspec) {
  CTX_CHECK(c);
  if (nspec != c->sp.nspec) return set_error(EMG_ERR_ARG, "nspec differs from the context");
  if (!counts) return set_error(EMG_ERR_ARG, "null counts");
  int64_t total = 0;
  for (int s = 0; s < nspec; s++) {
    if (counts[s] < 0) return set_error(EMG_ERR_ARG, "negative count");
    total += counts[s];
  }
  if (total > 0 && !pbuf) return set_error(EMG_ERR_ARG, "null pbuf");
  State64 tgt = c->s64;
  State64 tmp{};
  const SpeciesTab before = c->sp;
  std::atomic<bool> touched{false};  // records of the new state have been sent
  *c->hflag = 0;
  // the records (with `living`, those of them), cnt[s] of species s, into tgt
  auto send = [&](const int64_t *cnt, const LivingRecords *living) {
    int64_t first[EMG_MAX_SPECIES + 1] = {0};
    for (int s = 0; s < nspec; s++) first[s + 1] = first[s] + cnt[s];
    const int need_pid0 = c->cfg.precision == EMG_FP32_FIXED && !c->cfg.track_pid ? 1 : 0;
    for (int s = 0; s < nspec; s++) c->sp.cnt[s] = cnt[s];
    launch_zero(c->dflag + 1, sizeof(int), c->stream);
    const IoFn use = [&](size_t off, size_t len, void *slot) {
      const int64_t at = off / sizeof(emg_particle), m0 = living ? living->before(at) : at,
                    m1 = m0 + len / sizeof(emg_particle);
      touched = true;
      for (int s = 0; s < nspec; s++) {
        const int64_t a = std::max(m0, first[s]), b = std::min(m1, first[s + 1]);
        if (a < b)
          hipLaunchKernelGGL(k_split, dim3((unsigned)((b - a + kBlock - 1) / kBlock)), dim3(kBlock),
                             0, c->stream, static_cast<emg_particle *>(slot) + (a - m0), b - a, tgt,
                             c->sp.off[s] + (a - first[s]), c->g, c->dflag, need_pid0,
                             c->dflag + 1);
      }
      return hip_check(hipGetLastError(), "upload split");
    };
    IoCopy copy;
    if (living)
      copy = [&](size_t off, size_t len, void *slot) {
        return living->copy(off / sizeof(emg_particle), len / sizeof(emg_particle),
                            static_cast<emg_particle *>(slot));
      };
    return io_write(c, pbuf, sizeof(emg_particle) * total, sizeof(emg_particle), use, copy);
  };
  bool fits = true;
  for (int s = 0; s < nspec; s++) fits = fits && counts[s] <= c->cfg.capacity[s];
  int rc = EMG_OK;
  bool dead = !fits;  // more records than room: only the living have to fit
  int64_t sent = total;
  if (c->cfg.precision == EMG_FP32_FIXED) {
    if ((rc = alloc_state64(c, tmp, std::max<int64_t>(c->cap_total, 1)))) return rc;
    tgt = tmp;
  }
  if (fits) {
    rc = send(counts, nullptr);
    if (!rc) {
      rc = read_flags(c);
      dead = rc != EMG_OK && *c->hflag == kFlagDead;  // (and no other error)
    }
  }
  if (dead) {
    // transbound: keep nid >= 0 in order
    LivingRecords living;
    int64_t kept[EMG_MAX_SPECIES] = {0};
    rc = living.count(c, pbuf, total);
    sent = 0;
    for (int64_t s = 0, m = 0; s < nspec && !rc; m += counts[s], s++) {
      kept[s] = living.before(m + counts[s]) - living.before(m);
      sent += kept[s];
      if (kept[s] > c->cfg.capacity[s])
        rc = set_error(EMG_ERR_CAPACITY, "species count exceeds the context capacity");
    }
    if (!rc) rc = send(kept, &living);
    if (!rc) rc = read_flags(c);
  }
  if (rc && !touched && *c->hflag == 0) {  // nothing has been sent: the old state stands
    free_state64(tmp);
    c->sp = before;
    return rc;
  }
  if (!rc && c->cfg.precision == EMG_FP32_FIXED) {
    rc = fx_from64(c, tmp);
    if (!rc) rc = read_flags(c);
  }
  free_state64(tmp);
  if (rc) {
    for (int s = 0; s < nspec; s++) c->sp.cnt[s] = 0;
    c->have_particles = false;
    return rc;
  }
  c->have_particles = true;
  // most neighbours in the order share a tile: the blocks' windows catch them
  c->ordered = (int64_t)c->hflag[1] * kNearSample * 2 > sent;
  c->pushes_since_sort = c->cfg.sort_every;  // unsorted: sort before the first push
  c->moves_after_sort = emg::kUnsorted;
  c->runs_valid = false;
  c->rho_valid = false;
  c->faces_valid = false;
  c->j_valid = false;
  c->ke_valid = false;
  return EMG_OK;
}

int emg_particle_counts(emg_ctx *c, int64_t *counts) {
  CTX_CHECK(c);
  if (!counts) return set_error(EMG_ERR_ARG, "null counts");
  for (int s = 0; s < c->sp.nspec; s++) counts[s] = c->sp.cnt[s];
  return EMG_OK;
}

int emg_download_particles(emg_ctx *c, emg_particle *pbuf, int64_t *counts) {
  CTX_CHECK(c);
  int rc = read_flags(c);
  if (rc) return rc;
  int64_t total = 0;
  for (int s = 0; s < c->sp.nspec; s++) total += c->sp.cnt[s];
  if (counts)
    for (int s = 0; s < c->sp.nspec; s++) counts[s] = c->sp.cnt[s];
  if (total == 0) return EMG_OK;
  if (!pbuf) return set_error(EMG_ERR_ARG, "null pbuf");
  State64 src = c->s64;
  State64 tmp{};
  if (c->cfg.precision == EMG_FP32_FIXED) {
    if ((rc = alloc_state64(c, tmp, c->cap_total))) return rc;
    rc = fx_to64(c, tmp);
    if (rc) {
      free_state64(tmp);
      return rc;
    }
    src = tmp;
  }
  int64_t first[EMG_MAX_SPECIES + 1] = {0};
  for (int s = 0; s < c->sp.nspec; s++) first[s + 1] = first[s] + c->sp.cnt[s];
  rc = io_read(c, pbuf, sizeof(emg_particle) * total, sizeof(emg_particle),
               [&](size_t off, size_t len, void *slot) {
                 const int64_t m0 = off / sizeof(emg_particle), m1 = m0 + len / sizeof(emg_particle);
                 for (int s = 0; s < c->sp.nspec; s++) {
                   const int64_t a = std::max(m0, first[s]), b = std::min(m1, first[s + 1]);
                   if (a < b)
                     hipLaunchKernelGGL(k_join, dim3((unsigned)((b - a + kBlock - 1) / kBlock)),
                                        dim3(kBlock), 0, c->stream, src,
                                        c->sp.off[s] + (a - first[s]), b - a, s + 1,
                                        static_cast<emg_particle *>(slot) + (a - m0));
                 }
                 return hip_check(hipGetLastError(), "download join");
               });
  free_state64(tmp);
  return rc;
}

int emg_set_fields(emg_ctx *c, const double *eb, const int32_t lo[3], const int32_t hi[3]) {
  CTX_CHECK(c);
  if (!eb || !lo || !hi) return set_error(EMG_ERR_ARG, "null argument");
  int n[3] = {c->g.nx, c->g.ny, c->g.nz};
  int elo[3], ext[3];
  for (int d = 0; d < 3; d++) {
    if (lo[d] > -1 || hi[d] < n[d])
      return set_error(EMG_ERR_ARG, "eb bounds must cover -1..n on every axis");
    elo[d] = lo[d];
    ext[d] = hi[d] - lo[d] + 1;
  }
  const size_t bytes = sizeof(double) * 6 * (size_t)ext[0] * ext[1] * ext[2];
  int rc = hip_check(hipStreamSynchronize(c->stream), "stream synchronize");
  if (rc) return rc;
  if (bytes > c->eb_dev_bytes) {
    dfree(c->eb_dev);
    c->eb_dev = nullptr;
    c->eb_dev_bytes = 0;
    if ((rc = dalloc(c, &c->eb_dev, bytes / sizeof(double), "eb"))) return rc;
    c->eb_dev_bytes = bytes;
  }
  for (int d = 0; d < 3; d++) {
    c->eb_lo[d] = elo[d];
    c->eb_ext[d] = ext[d];
  }
  const size_t unit = 6 * sizeof(double);
  rc = io_write(c, eb, bytes, unit, [&](size_t off, size_t len, void *slot) {
    launch_eb_split(c, (const double *)slot, (int64_t)(off / unit), (int64_t)(len / unit));
    return hip_check(hipGetLastError(), "eb upload");
  });
  if (rc) return rc;
  launch_relocate64(c);
  c->fields_set = true;
  c->nodes_stale = false;
  return hip_check(hipGetLastError(), "relocate launch");
}

// ---- device-resident fields: the Yee update on the uploaded eb
static int need_eb(emg_ctx *c) {
  if (!c->fields_set || !c->eb_dev) return set_error(EMG_ERR_STATE, "emg_set_fields has not been called");
  return EMG_OK;
}

int emg_bfield(emg_ctx *c) {
  CTX_CHECK(c);
  int rc = need_eb(c);
  if (rc) return rc;
  launch_bfield(c);
  c->nodes_b_valid = false;
  c->b_recorded = c->b_recorded || capturing(c);
  c->nodes_stale = true;
  return hip_check(hipGetLastError(), "bfield launch");
}

int emg_efield(emg_ctx *c, double tcs, double dlt) {
  CTX_CHECK(c);
  int rc = need_eb(c);
  if (rc) return rc;
  if (!c->j_valid) return set_error(EMG_ERR_STATE, "no current deposited (call emg_push_em first)");
  launch_efield(c, tcs, dlt);
  c->nodes_stale = true;
  return hip_check(hipGetLastError(), "efield launch");
}

int emg_grdcrt(emg_ctx *c) {
  CTX_CHECK(c);
  int rc = need_eb(c);
  if (rc) return rc;
  launch_relocate64(c);
  c->nodes_stale = false;
  return hip_check(hipGetLastError(), "relocate launch");
}

int emg_get_fields(emg_ctx *c, double *eb, const int32_t lo[3], const int32_t hi[3]) {
  CTX_CHECK(c);
  int rc = need_eb(c);
  if (rc) return rc;
  if (!eb || !lo || !hi) return set_error(EMG_ERR_ARG, "null argument");
  for (int d = 0; d < 3; d++)
    if (lo[d] < c->eb_lo[d] || hi[d] > c->eb_lo[d] + c->eb_ext[d] - 1 || hi[d] < lo[d])
      return set_error(EMG_ERR_ARG, "eb bounds outside the uploaded array");
  const int l[3] = {lo[0], lo[1], lo[2]};
  const int ext[3] = {hi[0] - lo[0] + 1, hi[1] - lo[1] + 1, hi[2] - lo[2] + 1};
  const size_t count = (size_t)6 * ext[0] * ext[1] * ext[2], unit = 6 * sizeof(double);
  return io_read(c, eb, sizeof(double) * count, unit, [&](size_t off, size_t len, void *slot) {
    launch_eb_box(c, l, ext, (int64_t)(off / unit), (int64_t)(len / unit), (double *)slot);
    return hip_check(hipGetLastError(), "eb read-out");
  });
}

int emg_solve_es(emg_ctx *c, double rhobk) {
  CTX_CHECK(c);
  if (!c->rho_valid) return set_error(EMG_ERR_STATE, "rho is not deposited for the current positions");
  if (!c->eb_dev) {  // no eb uploaded: eb(6, -1:n+1)^3 with B = 0
    int n[3] = {c->g.nx, c->g.ny, c->g.nz};
    size_t count = 6;
    for (int d = 0; d < 3; d++) {
      c->eb_lo[d] = -1;
      c->eb_ext[d] = n[d] + 3;
      count *= (size_t)c->eb_ext[d];
    }
    int rc = dalloc(c, &c->eb_dev, count, "eb");
    if (rc) return rc;
    c->eb_dev_bytes = count * sizeof(double);
    launch_zero(c->eb_dev, c->eb_dev_bytes, c->stream);
    c->nodes_b_valid = false;
  }
  int rc = solve_es(c, rhobk);
  if (rc) return rc;
  c->fields_set = true;
  c->nodes_stale = false;
  return EMG_OK;
}

int emg_set_background(emg_ctx *c, const double *rhobk) {
  CTX_CHECK(c);
  if (!rhobk) {
    dfree(c->bk_dev);
    c->bk_dev = nullptr;
    return EMG_OK;
  }
  int rc;
  if (!c->bk_dev && (rc = dalloc(c, &c->bk_dev, (size_t)c->ncell, "background charge"))) return rc;
  rc = hip_check(hipMemcpyAsync(c->bk_dev, rhobk, sizeof(double) * c->ncell,
                                hipMemcpyHostToDevice, c->stream),
                 "background copy");
  if (!rc) rc = hip_check(hipStreamSynchronize(c->stream), "background copy");
  return rc;
}

int emg_get_potential(emg_ctx *c, double *phi) {
  CTX_CHECK(c);
  if (!phi) return set_error(EMG_ERR_ARG, "null argument");
  return read_potential(c, phi);
}

// wait for a reduction that left its sums in hsum and the flags in hflag
static int read_sums(emg_ctx *c) {
  int rc = hip_check(hipGetLastError(), "reduction launch");
  if (!rc) rc = hip_check(hipStreamSynchronize(c->stream), "stream synchronize");
  return rc ? rc : flags_error(c);
}

int emg_field_energy(emg_ctx *c, double cs, double *engeb) {
  CTX_CHECK(c);
  int rc = need_eb(c);
  if (rc) return rc;
  if (!engeb) return set_error(EMG_ERR_ARG, "null argument");
  if (!c->fe_buf && (rc = dalloc(c, &c->fe_buf, (size_t)field_energy_part_need(), "field energy")))
    return rc;
  launch_field_energy(c, cs, c->fe_buf, c->hsum);
  if ((rc = read_sums(c))) return rc;
  engeb[0] = c->hsum[0];
  engeb[1] = c->hsum[1];
  return EMG_OK;
}

static int need_particles(emg_ctx *c) {
  if (!c->have_particles) return set_error(EMG_ERR_STATE, "no particles uploaded");
  return EMG_OK;
}

static int need_fields(emg_ctx *c) {
  if (!c->fields_set) return set_error(EMG_ERR_STATE, "emg_set_fields has not been called");
  if (c->nodes_stale)
    return set_error(EMG_ERR_STATE, "eb changed on the device since the last relocation: call emg_grdcrt");
  return EMG_OK;
}

// PLAIN_FP64 with sort_every > 0: the cell sort that is due before a push.
// With `carry` (a push that can move the particles into the new order
// itself) a re-sort close to the last sort only counts the cells here and
// *carry is set: the caller launches its push with the re-sort and then
// calls sort64_commit.  which: the run table of the launch that follows.
static int sort_if_due(emg_ctx *c, int which, bool *carry = nullptr) {
  if (carry) *carry = false;
  if (c->cfg.precision != EMG_PLAIN_FP64 || c->cfg.sort_every <= 0) return EMG_OK;
  if (c->pushes_since_sort < c->cfg.sort_every) {
    c->pushes_since_sort++;
    return EMG_OK;
  }
  int rc;
  if (carry && emg::sort64_fusable(c)) {
    rc = emg::sort64_rank(c, which);
    if (!rc) *carry = true;
  } else {
    rc = sort64(c, true);
  }
  if (!rc) c->pushes_since_sort = 1;
  return rc;
}

// a call that moves the particles (and deposits their charge) is recorded
static void note_recorded(emg_ctx *c, bool deposits) {
  if (!capturing(c)) return;
  c->push_recorded = true;
  c->move_recorded = c->move_recorded || !deposits;
}

int emg_positn(emg_ctx *c, int32_t ustep) {
  CTX_CHECK(c);
  int rc = need_particles(c);
  if (rc) return rc;
  if (ustep < 0) return set_error(EMG_ERR_ARG, "ustep must be >= 0");
  note_recorded(c, false);
  if ((rc = sort_if_due(c, 0))) return rc;
  if (c->cfg.precision == EMG_PLAIN_FP64) {
    launch_positn64(c, ustep);
    if (c->moves_after_sort < emg::kUnsorted) c->moves_after_sort++;
  } else {
    launch_fx_step(c, ustep, false, false, false);
  }
  c->rho_valid = false;
  c->faces_valid = false;
  c->j_valid = false;
  return hip_check(hipGetLastError(), "positn launch");
}

int emg_push_es(emg_ctx *c, int32_t ustep) {
  CTX_CHECK(c);
  int rc = need_particles(c);
  if (!rc) rc = need_fields(c);
  if (rc) return rc;
  if (ustep < 0) return set_error(EMG_ERR_ARG, "ustep must be >= 0");
  note_recorded(c, true);
  bool carry;
  if ((rc = sort_if_due(c, 0, &carry))) return rc;
  if (c->cfg.precision == EMG_PLAIN_FP64) {
    if (!carry && (rc = sort64_runs(c, 0))) return rc;
    launch_push_es64(c, ustep, carry);  // push + charge at the new positions
    if (carry) rc = emg::sort64_commit(c);
    if (c->moves_after_sort < emg::kUnsorted) c->moves_after_sort++;
    c->rho_valid = true;
    c->faces_valid = false;
    c->ke_valid = false;
  } else {
    launch_fx_step(c, ustep, true, true, false);
    c->rho_valid = true;
    c->faces_valid = false;
    c->ke_valid = true;  // fused partials of the new velocities
  }
  c->j_valid = false;
  if (rc) return rc;
  return hip_check(hipGetLastError(), "push launch");
}

int emg_deposit_rho(emg_ctx *c, int32_t func) {
  CTX_CHECK(c);
  int rc = need_particles(c);
  if (rc) return rc;
  if (func < 0 || func > 2) return set_error(EMG_ERR_ARG, "func must be 0, 1 or 2");
  // a push deposits at its new positions itself (in a capture, the last call is
  // the last one of a replay too)
  if (!c->rho_valid || (c->move_recorded && !capturing(c))) {
    if (c->cfg.precision == EMG_PLAIN_FP64) {
      if ((rc = sort64_runs(c, 0))) return rc;
      launch_deposit64(c);
    } else {
      launch_fx_deposit(c);
    }
    c->rho_valid = true;
    c->faces_valid = false;
  }
  return hip_check(hipGetLastError(), "deposit launch");
}

// Read a grid array back: in chunks through the pinned slots, or (stage, of
// stage_cap doubles) whole through a device array with one copy.
static int read_grid(emg_ctx *c, double *host, const int32_t lo[3], const int32_t hi[3], int comps,
                     int species, bool current, double *stage = nullptr, int64_t stage_cap = 0) {
  if (!host || !lo || !hi) return set_error(EMG_ERR_ARG, "null argument");
  int l[3], h[3];
  int64_t points = 1;
  for (int d = 0; d < 3; d++) {
    if (hi[d] < lo[d]) return set_error(EMG_ERR_ARG, "hi < lo");
    l[d] = lo[d];
    h[d] = hi[d];
    points *= (int64_t)(hi[d] - lo[d] + 1);
  }
  if (stage && points * comps > stage_cap)
    return set_error(EMG_ERR_CAPACITY, "the read-out exceeds the library's static staging "
                                       "array (2^24 values, 128 MiB): read it with emg_get_rho");
  const bool ghosts = !current && prepare_read_rho(c, l, h);
  auto launch = [&](int64_t o0, int64_t n, double *dst) {
    if (current)
      launch_read_current(c, species, dst, l, h, o0, n);
    else
      launch_read_rho(c, species, ghosts, dst, l, h, o0, n);
    return hip_check(hipGetLastError(), "read-out");
  };
  const size_t unit = sizeof(double) * comps;
  if (!stage)
    return io_read(c, host, unit * points, unit, [&](size_t off, size_t len, void *slot) {
      return launch((int64_t)(off / unit), (int64_t)(len / unit), static_cast<double *>(slot));
    });
  int rc = launch(0, points, stage);
  if (!rc) rc = read_flags(c);
  if (!rc)
    rc = hip_check(hipMemcpyAsync(host, stage, unit * points, hipMemcpyDeviceToHost, c->stream),
                   "read-out copy");
  if (!rc) rc = hip_check(hipStreamSynchronize(c->stream), "read-out copy");
  return rc;
}

int emg_get_rho(emg_ctx *c, double *rho, const int32_t lo[3], const int32_t hi[3]) {
  CTX_CHECK(c);
  if (!c->rho_valid) return set_error(EMG_ERR_STATE, "rho is not deposited for the current positions");
  return read_grid(c, rho, lo, hi, 1, -1, false);
}

int emg_get_rho_noalloc(emg_ctx *c, double *rho, const int32_t lo[3], const int32_t hi[3]) {
  CTX_CHECK(c);
  if (!c->rho_valid) return set_error(EMG_ERR_STATE, "rho is not deposited for the current positions");
  if (!c->scratch) return set_error(EMG_ERR_STATE, "no scratch address for this device");
  return read_grid(c, rho, lo, hi, 1, -1, false, c->scratch, kScratchDoubles);
}

int emg_get_rhodg(emg_ctx *c, int32_t is, double *rho, const int32_t lo[3], const int32_t hi[3]) {
  CTX_CHECK(c);
  if (is < 0 || is >= c->sp.nspec) return set_error(EMG_ERR_ARG, "species out of range");
  if (!c->rho_valid) return set_error(EMG_ERR_STATE, "rho is not deposited for the current positions");
  return read_grid(c, rho, lo, hi, 1, is, false);
}

int emg_energy(emg_ctx *c, double *engk) {
  CTX_CHECK(c);
  if (!engk) return set_error(EMG_ERR_ARG, "null argument");
  int rc = need_particles(c);
  if (rc) return rc;
  if (c->cfg.precision == EMG_PLAIN_FP64)
    launch_energy64(c);
  else if (c->ke_valid)
    fx_energy_from_push(c);
  else
    launch_fx_energy(c);
  if ((rc = read_sums(c))) return rc;
  const double *sums = c->hsum;
  double vol = c->g.slx * c->g.sly * c->g.slz;
  for (int s = 0; s < c->sp.nspec; s++)
    for (int d = 0; d < 3; d++) engk[3 * s + d] = 0.0 + 0.5 * c->cfg.rm[s] * sums[3 * s + d] / vol;
  return EMG_OK;
}

int emg_push_em(emg_ctx *c, int32_t ustep) {
  CTX_CHECK(c);
  int rc = need_particles(c);
  if (!rc) rc = need_fields(c);
  if (rc) return rc;
  if (ustep < 1) return set_error(EMG_ERR_ARG, "ustep must be >= 1");
  note_recorded(c, false);
  bool carry;
  if ((rc = sort_if_due(c, 1, &carry))) return rc;
  if (c->cfg.precision == EMG_PLAIN_FP64) {
    if (!carry && (rc = sort64_runs(c, 1))) return rc;
    launch_push_em64(c, ustep, carry);
    if (carry) rc = emg::sort64_commit(c);
    if (c->moves_after_sort < emg::kUnsorted) c->moves_after_sort++;
    c->ke_valid = false;
  } else {
    launch_fx_step(c, ustep, true, false, true);
    c->ke_valid = true;  // fused partials of the new velocities
  }
  c->j_valid = true;
  c->rho_valid = false;
  c->faces_valid = false;
  if (rc) return rc;
  return hip_check(hipGetLastError(), "push_em launch");
}

int emg_get_current(emg_ctx *c, double *aj, const int32_t lo[3], const int32_t hi[3]) {
  CTX_CHECK(c);
  if (!c->j_valid) return set_error(EMG_ERR_STATE, "no current deposited");
  return read_grid(c, aj, lo, hi, 3, -1, true);
}

int emg_get_ajdg(emg_ctx *c, int32_t is, double *aj, const int32_t lo[3], const int32_t hi[3]) {
  CTX_CHECK(c);
  if (!c->j_valid) return set_error(EMG_ERR_STATE, "no current deposited");
  if (is < 0 || is >= c->sp.nspec) return set_error(EMG_ERR_ARG, "species index");
  return read_grid(c, aj, lo, hi, 3, is, true);
}

// ---- adjoint window (FP64 form)
static int need_fp64(emg_ctx *c) {
  if (c->cfg.precision != EMG_PLAIN_FP64)
    return set_error(EMG_ERR_UNSUPPORTED, "the adjoint window runs in EMG_PLAIN_FP64 contexts");
  return EMG_OK;
}

static int copy_state(const State64 &src, const State64 &dst, int64_t n, hipStream_t st) {
  const void *from[7] = {src.x, src.y, src.z, src.vx, src.vy, src.vz, src.pid};
  void *to[7] = {dst.x, dst.y, dst.z, dst.vx, dst.vy, dst.vz, dst.pid};
  for (int q = 0; q < 7; q++) {
    size_t bytes = (q < 6 ? sizeof(double) : sizeof(int32_t)) * (size_t)n;
    int rc = hip_check(hipMemcpyAsync(to[q], from[q], bytes, hipMemcpyDeviceToDevice, st),
                       "state copy");
    if (rc) return rc;
  }
  return EMG_OK;
}

// the adjoint arrays and the step's bins, so that only the window's first call
// allocates and a step can be recorded after any other call of it
static int need_adjoint(emg_ctx *c) {
  int rc = need_fp64(c);
  if (rc) return rc;
  if (c->adj_sum) return bins_alloc(c);  // the last one: then all are there
  if ((!c->lam && (rc = dalloc(c, &c->lam, 8 * (size_t)c->cap_total, "particle adjoints"))) ||
      (!c->adj_e && (rc = dalloc(c, &c->adj_e, 3 * c->ncell, "adjoint field"))) ||
      (!c->adj_g && (rc = dalloc(c, &c->adj_g, c->ncell, "adjoint density"))) ||
      (rc = dalloc(c, &c->adj_sum, (size_t)adj_vsum_need(), "adjoint sums")))
    return rc;
  launch_zero(c->lam, 8 * sizeof(double) * c->cap_total, c->stream);
  launch_zero(c->adj_e, sizeof(double) * 3 * c->ncell, c->stream);
  if ((rc = hip_check(hipGetLastError(), "adjoint allocation"))) return rc;
  return bins_alloc(c);
}

int emg_state_save(emg_ctx *c, int32_t slot) {
  CTX_CHECK(c);
  int rc = need_fp64(c);
  if (!rc) rc = need_particles(c);
  if (rc) return rc;
  if (slot < 0 || slot >= kStateSlots) return set_error(EMG_ERR_ARG, "slot must be 0..63");
  if (!c->slot[slot].x && (rc = alloc_state64(c, c->slot[slot], c->cap_total))) return rc;
  for (int s = 0; s < c->sp.nspec; s++) c->slot_cnt[slot][s] = c->sp.cnt[s];
  c->slot_ordered[slot] = c->ordered || c->runs_valid;
  return copy_state(c->s64, c->slot[slot], c->cap_total, c->stream);
}

int emg_state_load(emg_ctx *c, int32_t slot) {
  CTX_CHECK(c);
  int rc = need_fp64(c);
  if (rc) return rc;
  if (slot < 0 || slot >= kStateSlots || !c->slot[slot].x)
    return set_error(EMG_ERR_ARG, "slot holds no saved state");
  for (int s = 0; s < c->sp.nspec; s++) c->sp.cnt[s] = c->slot_cnt[slot][s];
  c->have_particles = true;
  c->ordered = c->slot_ordered[slot];
  c->moves_after_sort = emg::kUnsorted;
  c->runs_valid = false;
  c->rho_valid = c->j_valid = c->ke_valid = false;
  c->faces_valid = false;
  return copy_state(c->slot[slot], c->s64, c->cap_total, c->stream);
}

int emg_adj_reset(emg_ctx *c) {
  CTX_CHECK(c);
  int rc = need_adjoint(c);
  if (rc) return rc;
  launch_zero(c->lam, 8 * sizeof(double) * c->cap_total, c->stream);
  return hip_check(hipGetLastError(), "adjoint reset");
}

int emg_adj_step(emg_ctx *c, int32_t ustep) {
  CTX_CHECK(c);
  int rc = need_adjoint(c);
  if (!rc) rc = need_particles(c);
  if (!rc) rc = need_fields(c);
  if (rc) return rc;
  if (ustep < 0) return set_error(EMG_ERR_ARG, "ustep must be >= 0");
  launch_adj_step64(c, ustep);
  return hip_check(hipGetLastError(), "adjoint step launch");
}

int emg_adj_get_field(emg_ctx *c, double *lam_e) {
  CTX_CHECK(c);
  if (!lam_e) return set_error(EMG_ERR_ARG, "null argument");
  int rc = need_adjoint(c);
  if (rc) return rc;
  return io_read_array(c, lam_e, c->adj_e, sizeof(double) * 3 * c->ncell);
}

int emg_adj_add_density(emg_ctx *c, const double *g, const double *qfac) {
  CTX_CHECK(c);
  if (!g || !qfac) return set_error(EMG_ERR_ARG, "null argument");
  int rc = need_adjoint(c);
  if (!rc) rc = need_particles(c);
  if (rc) return rc;
  if ((rc = hip_check(hipMemcpyAsync(c->adj_g, g, sizeof(double) * c->ncell, hipMemcpyHostToDevice,
                                     c->stream), "adjoint density upload")))
    return rc;
  launch_adj_density64(c, qfac);
  // the host buffers may be reused once this returns
  return hip_check(hipStreamSynchronize(c->stream), "adjoint density");
}

int emg_adj_velocity_sums(emg_ctx *c, double *out) {
  CTX_CHECK(c);
  if (!out) return set_error(EMG_ERR_ARG, "null argument");
  int rc = need_adjoint(c);
  if (!rc) rc = need_particles(c);
  if (rc) return rc;
  launch_adj_vsum(c, c->adj_sum, c->hsum);
  if ((rc = read_sums(c))) return rc;
  for (int k = 0; k < 3 * c->sp.nspec; k++) out[k] = c->hsum[k];
  return EMG_OK;
}

int emg_sort(emg_ctx *c) {
  CTX_CHECK(c);
  int rc = need_particles(c);
  if (rc) return rc;
  if (c->cfg.precision == EMG_PLAIN_FP64) {
    rc = sort64(c, false);
    for (int k = 0; k < 2 && !rc; k++) rc = sort64_runs(c, k);
    if (!rc) c->pushes_since_sort = 0;
  } else {
    rc = fx_rebucket(c);
  }
  return rc;
}

int emg_init_device(emg_ctx *c, const emg_device_species *spec, int32_t nspec, uint64_t seed) {
  CTX_CHECK(c);
  if (!spec || nspec != c->sp.nspec) return set_error(EMG_ERR_ARG, "species table");
  for (int s = 0; s < nspec; s++) {
    if (spec[s].count < 0 || spec[s].count > c->cfg.capacity[s])
      return set_error(EMG_ERR_CAPACITY, "species count exceeds the context capacity");
  }
  int rc;
  State64 tmp{};
  if (c->cfg.precision != EMG_PLAIN_FP64 && (rc = alloc_state64(c, tmp, c->cap_total))) return rc;
  for (int s = 0; s < nspec; s++) c->sp.cnt[s] = spec[s].count;
  if (c->cfg.precision == EMG_PLAIN_FP64) {
    rc = init_device_into(c, c->s64, spec, nspec, seed);
  } else {
    rc = init_device_into(c, tmp, spec, nspec, seed);
    if (!rc) rc = fx_from64(c, tmp);
    if (!rc) rc = hip_check(hipStreamSynchronize(c->stream), "init");
    free_state64(tmp);
  }
  if (!rc) rc = read_flags(c);
  if (rc) {
    for (int s = 0; s < nspec; s++) c->sp.cnt[s] = 0;
    return rc;
  }
  c->have_particles = true;
  c->ordered = false;
  c->pushes_since_sort = c->cfg.sort_every;  // unsorted: sort before the first push
  c->moves_after_sort = emg::kUnsorted;
  c->runs_valid = false;
  c->rho_valid = false;
  c->faces_valid = false;
  c->j_valid = false;
  c->ke_valid = false;
  return EMG_OK;
}

int emg_enable_timing(emg_ctx *c, int32_t on) {
  CTX_CHECK(c);
  if (!on) timer_flush(c);
  c->timing = on != 0;
  return EMG_OK;
}

int emg_kernel_stats(emg_ctx *c, int32_t which, double *total_ms, int64_t *launches) {
  CTX_CHECK(c);
  if (which < 0 || which >= kTNum) return set_error(EMG_ERR_ARG, "kernel kind");
  timer_flush(c);
  if (total_ms) *total_ms = c->timers[which].total_ms;
  if (launches) *launches = c->timers[which].launches;
  return EMG_OK;
}

int emg_reset_kernel_stats(emg_ctx *c) {
  CTX_CHECK(c);
  timer_flush(c);
  for (int k = 0; k < kTNum; k++) {
    c->timers[k].total_ms = 0.0;
    c->timers[k].launches = 0;
    c->timers[k].last_ms = 0.0;
  }
  return EMG_OK;
}

}  // extern "C"
