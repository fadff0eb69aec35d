// The HIP calls that libemgpu.so makes, for tests of its host logic without a
// GPU: device memory is host memory (counted, and limited or made to fail on
// request), a kernel launch only enters the kernel's name in a log, streams and
// events do nothing.  Loaded with RTLD_GLOBAL before the library, it takes the
// place of the HIP and hipFFT runtimes there.
#include <cxxabi.h>

#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {
std::mutex mu;
std::map<char *, size_t> live, dead;      // device allocations; freed ones (kept)
struct Kernel {
  std::string name;
  std::vector<bool> pointer;              // its parameters
};
std::map<const void *, Kernel> kernels;   // by host stub
std::string launches;
size_t used = 0, peak = 0, limit = SIZE_MAX;
long fail_in = -1, fail_times = 0;        // this allocation from now fails, and so many in all
int bad_frees = 0, bad_copies = 0, bad_args = 0, mallocs = 0, capturing = 0, last_error = 0;
int flags[2] = {0, 0};                    // what the next k_flag reports
std::map<int64_t, int> split;             // pid of the record that k_split puts where
struct Dim3 {
  uint32_t x, y, z;
};
thread_local struct {
  Dim3 g, b;
  size_t shm;
  void *stream;
} config;
int fail(int e) { return last_error = e; }
bool inside(const std::map<char *, size_t> &m, char *p, size_t &left) {
  auto it = m.upper_bound(p);
  if (it == m.begin()) return false;
  --it;
  left = p < it->first + it->second ? it->first + it->second - p : 0;
  return left > 0;
}
// [p, p + n) within one allocation, or in none, freed ones included (host memory)
bool within(const void *v, size_t n) {
  size_t left;
  if (inside(dead, (char *)v, left)) return false;
  return !inside(live, (char *)v, left) || n <= left;
}
void note(const std::string &what) { launches += what + "\n"; }
}  // namespace

#define API extern "C" __attribute__((visibility("default")))

// ---- what a test sets and reads
API void fake_log_clear() { std::lock_guard<std::mutex> l(mu); launches.clear(); }
API const char *fake_log() { return launches.c_str(); }
API void fake_limit(size_t bytes) { limit = bytes; }
API void fake_fail_in(long n, long times) { fail_in = n; fail_times = times; }
API size_t fake_used() { return used; }
API size_t fake_peak(int reset) { const size_t p = peak; if (reset) peak = used; return p; }
API int fake_mallocs() { return mallocs; }
API int fake_bad_frees() { return bad_frees; }
API int fake_bad_copies() { return bad_copies; }
API int fake_bad_args() { return bad_args; }  // kernels given freed memory
API void fake_capture(int on) { capturing = on; }
API void fake_flags(int a, int b) { flags[0] = a; flags[1] = b; }

API int64_t fake_split(int64_t *slot, int *pid, int64_t n) {  // and start anew
  std::lock_guard<std::mutex> l(mu);
  int64_t k = 0;
  for (auto &e : split)
    if (k < n) {
      slot[k] = e.first;
      pid[k++] = e.second;
    }
  k = (int64_t)split.size();
  split.clear();
  return k;
}

// ---- memory
API int hipMalloc(void **p, size_t n) {
  std::lock_guard<std::mutex> l(mu);
  mallocs++;
  if (capturing) return fail(900);  // not while a stream is captured
  if (fail_in > 0 && fail_times > 0 && --fail_in == 0) {
    fail_in = 1;
    fail_times--;
    return fail(2);
  }
  if (n > limit || used > limit - n) return fail(2);
  char *q = (char *)std::malloc(n ? n : 1);
  if (!q) return fail(2);
  live[q] = n;
  used += n;
  peak = used > peak ? used : peak;
  *p = q;
  return 0;
}
API int hipFree(void *p) {
  std::lock_guard<std::mutex> l(mu);
  if (!p) return 0;
  auto it = live.find((char *)p);
  if (it == live.end()) {
    bad_frees++;
    return fail(1);
  }
  used -= it->second;
  dead[it->first] = it->second;
  live.erase(it);
  return 0;
}
API int hipHostMalloc(void **p, size_t n, unsigned) { *p = std::calloc(n, 1); return *p ? 0 : 2; }
API int hipHostFree(void *p) { std::free(p); return 0; }
API int hipMemcpy(void *d, const void *s, size_t n, int) {
  std::lock_guard<std::mutex> l(mu);
  if (!within(d, n) || !within(s, n)) bad_copies++;
  else std::memcpy(d, s, n);
  return 0;
}
API int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *) { return hipMemcpy(d, s, n, k); }
API int hipGetSymbolAddress(void **p, const void *) {
  static char *mem = (char *)std::malloc(size_t(128) << 20);
  *p = mem;
  return 0;
}

// ---- launches
API int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t shm, void *stream) {
  config = {g, b, shm, stream};
  return 0;
}
API int __hipPopCallConfiguration(Dim3 *g, Dim3 *b, size_t *shm, void **stream) {
  *g = config.g;
  *b = config.b;
  *shm = config.shm;
  *stream = config.stream;
  return 0;
}
API int hipLaunchKernel(const void *f, Dim3, Dim3, void **args, size_t, void *) {
  std::lock_guard<std::mutex> l(mu);
  const Kernel &k = kernels[f];
  for (size_t i = 0; i < k.pointer.size(); i++)
    if (k.pointer[i] && !within(*(void **)args[i], 1)) bad_args++;
  if (k.name == "k_flag") {
    int *h = *(int **)args[1];
    h[0] = flags[0];
    h[1] = flags[1];
    flags[0] = flags[1] = 0;
  }
  if (k.name == "k_split") {
    const char *rec = *(char **)args[0];
    for (int64_t i = 0; i < *(int64_t *)args[1]; i++)
      std::memcpy(&split[*(int64_t *)args[3] + i], rec + 64 * i + 48, 4);
  }
  note(k.name);
  return 0;
}
API void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
API void __hipUnregisterFatBinary(void **) {}
API void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
API void __hipRegisterFunction(void **, const void *host, char *, const char *dev, unsigned, void *,
                               void *, void *, void *, int *) {
  int st = 0;
  char *d = abi::__cxa_demangle(dev, nullptr, nullptr, &st);
  std::string s = st == 0 && d ? d : dev;
  std::free(d);
  // "void emg::(anonymous namespace)::k_x<8, true>(args)" -> "k_x<8, true>"
  const size_t at = s.find("k_");
  s = at == std::string::npos ? s : s.substr(at);
  Kernel k;
  int depth = 0;
  for (size_t i = 0; i < s.size(); i++) {
    const bool top = depth == (k.name.empty() ? 0 : 1);
    if (k.name.empty() && top && s[i] == '(') {
      k.name = s.substr(0, i);
    } else if (!k.name.empty() && top && (s[i] == ',' || s[i] == ')')) {
      k.pointer.push_back(s[i - 1] == '*');
    }
    depth += s[i] == '<' || s[i] == '(' ? 1 : (s[i] == '>' || s[i] == ')' ? -1 : 0);
  }
  kernels[host] = k;
}

// ---- the rest
API int hipGetDevice(int *d) { *d = 0; return 0; }
API int hipSetDevice(int) { return 0; }
API int hipGetLastError() { const int e = last_error; last_error = 0; return e; }
API const char *hipGetErrorString(int) { return "fake"; }
API int hipStreamCreateWithFlags(void **s, unsigned) { *s = std::malloc(1); return 0; }
API int hipStreamDestroy(void *s) { std::free(s); return 0; }
API int hipStreamSynchronize(void *) { return 0; }
API int hipStreamIsCapturing(void *, int *st) { *st = capturing; return 0; }
API int hipEventCreate(void **e) { *e = std::malloc(1); return 0; }
API int hipEventCreateWithFlags(void **e, unsigned) { return hipEventCreate(e); }
API int hipEventDestroy(void *e) { std::free(e); return 0; }
API int hipEventRecord(void *, void *) { return 0; }
API int hipEventSynchronize(void *) { return 0; }
API int hipEventElapsedTime(float *ms, void *, void *) { *ms = 0.f; return 0; }
API int hipFuncSetAttribute(const void *, int, int) { return 0; }
API int hipfftPlan3d(void **p, int, int, int, int) { static char h[64]; static int k; *p = &h[k++ % 64]; note("hipfftPlan3d"); return 0; }
API int hipfftSetStream(void *p, void *s) {
  char t[64];
  std::snprintf(t, sizeof t, "hipfftSetStream %p", s);
  note(t);
  (void)p;
  return 0;
}
API int hipfftExecD2Z(void *, void *, void *) { note("hipfftExecD2Z"); return 0; }
API int hipfftExecZ2D(void *, void *, void *) { note("hipfftExecZ2D"); return 0; }
API int hipfftDestroy(void *) { return 0; }
