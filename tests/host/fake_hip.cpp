// A HIP runtime without a device: memory is host memory, launches are noted
// and not run.  Loaded (RTLD_GLOBAL) before libedge_amd.so, it lets the host
// code of the library run on the CPU, so that tests can see which kernels a
// call launches on which stream with which buffers, and what it does when an
// allocation fails.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <utility>

namespace {
std::recursive_mutex lock_;
std::map<const void*, std::string> kernels_;
std::map<void*, size_t> live_;
std::string log_;
int fail_after_ = -1;         // allocations until one fails (0: the next), -1: none does
size_t largest_ = 1ull << 36; // a larger allocation fails
int setup_flags_ = 0;         // what the flux solver set-up kernel reports
int mode_ = 0;                // the thread's capture mode (2: relaxed)
void* capturing_ = nullptr;   // a stream that its owner captures
int last_ = 0;
uintptr_t next_ = 0x1000;

constexpr int kOom = 2;
struct Config {
  unsigned g[3], b[3];
  size_t shared;
  void* stream;
} config_;

void note(const std::string& s) {
  std::lock_guard<std::recursive_mutex> l(lock_);
  log_ += s + "\n";
}
std::string hex(const void* p) {
  char b[32];
  snprintf(b, sizeof b, "%llx", (unsigned long long)(uintptr_t)p);
  return b;
}
int fresh(void** p) {
  std::lock_guard<std::recursive_mutex> l(lock_);
  *p = (void*)(next_ += 16);
  return 0;
}
}  // namespace

struct Dim3 {
  unsigned x, y, z;
};

extern "C" {
// for the tests
const char* fake_log() { return log_.c_str(); }
void fake_clear() { log_.clear(); }
int fake_fail_after(int n) {  // and what was left of the count (below 0: it has failed, or was not set)
  std::swap(n, fail_after_);
  return n;
}
void fake_setup_flags(int f) { setup_flags_ = f; }
void fake_capturing(void* st) { capturing_ = st; }
size_t fake_live() { return live_.size(); }
size_t fake_bytes() {
  size_t n = 0;
  for (const auto& a : live_) n += a.second;
  return n;
}
size_t fake_size(void* p) { return live_.count(p) ? live_[p] : 0; }

// the runtime
void** __hipRegisterFatBinary(const void*) {
  static void* h;
  return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  kernels_[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t shared, void* st) {
  config_ = {{g.x, g.y, g.z}, {b.x, b.y, b.z}, shared, st};
  return 0;
}
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* shared, void** st) {
  *g = {config_.g[0], config_.g[1], config_.g[2]};
  *b = {config_.b[0], config_.b[1], config_.b[2]};
  *shared = config_.shared;
  *st = config_.stream;
  return 0;
}
int hipLaunchKernel(const void* f, Dim3 g, Dim3, void** args, size_t, void* st) {
  const std::string name = kernels_[f];
  auto ptr = [&](int i) { return *(void**)args[i]; };
  std::string s = "launch " + name + " stream=" + hex(st) + " grid=" + std::to_string(g.x);
  if (name.find("k_sparse") != std::string::npos) {  // (SolverDev, SpDev, first, n, dt, dofs, t_int, proj_in)
    void** x = (void**)args[1];                      // phys, rot, proj, ...
    s += " phys=" + hex(x[0]) + " rot=" + hex(x[1]) + " proj=" + hex(x[2]) + " proj_in=" + hex(ptr(7));
  }
  if (name.find("k_flux_solvers") != std::string::npos) *(int*)ptr(18) |= setup_flags_;
  note(s);
  return 0;
}
int hipMalloc(void** p, size_t n) {
  std::lock_guard<std::recursive_mutex> l(lock_);
  if (capturing_ && mode_ != 2) {
    note("allocation that ends a capture");
    return last_ = kOom;
  }
  if (n > largest_ || (fail_after_ >= 0 && fail_after_-- == 0)) {
    *p = nullptr;
    return last_ = kOom;
  }
  *p = calloc(n ? n : 1, 1);
  live_[*p] = n;
  return 0;
}
int hipFree(void* p) {
  std::lock_guard<std::recursive_mutex> l(lock_);
  if (p && !live_.erase(p)) note("free of unknown memory");
  free(p);
  return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int) {
  memcpy(d, s, n);
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) {
  memcpy(d, s, n);
  return 0;
}
int hipMemset(void* d, int v, size_t n) {
  memset(d, v, n);
  return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void*) {
  memset(d, v, n);
  return 0;
}
int hipGetLastError() {
  const int e = last_;
  last_ = 0;
  return e;
}
const char* hipGetErrorString(int) { return "error of the fake runtime"; }
int hipDeviceSynchronize() { return 0; }
int hipFuncSetAttribute(const void*, int, int) { return 0; }
int hipGetDevice(int* d) { return *d = 0; }
int hipGetSymbolAddress(void** p, const void* s) {
  *p = const_cast<void*>(s);
  return 0;
}
int hipEventCreate(void** e) { return fresh(e); }
int hipEventCreateWithFlags(void** e, unsigned) { return fresh(e); }
int hipEventDestroy(void*) { return 0; }
int hipEventElapsedTime(float* t, void*, void*) {
  *t = 1.f;
  return 0;
}
int hipEventRecord(void* e, void* st) {
  note("record " + hex(e) + " stream=" + hex(st));
  return 0;
}
int hipEventSynchronize(void*) { return 0; }
int hipStreamWaitEvent(void* st, void* e, unsigned) {
  note("wait " + hex(e) + " stream=" + hex(st));
  return 0;
}
int hipStreamCreateWithFlags(void** s, unsigned) { return fresh(s); }
int hipStreamDestroy(void*) { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamIsCapturing(void* st, int* c) {
  *c = st && st == capturing_;
  return 0;
}
int hipThreadExchangeStreamCaptureMode(int* m) {
  std::swap(*m, mode_);
  return 0;
}
int hipStreamBeginCapture(void* st, int) {
  if (st == capturing_) return last_ = 401;  // (already being captured)
  note("begin stream=" + hex(st));
  return 0;
}
int hipStreamEndCapture(void* st, void** g) {
  note("end stream=" + hex(st));
  return fresh(g);
}
int hipGraphInstantiate(void** e, void*, void*, char*, size_t) { return fresh(e); }
int hipGraphLaunch(void* e, void* st) {
  note("graph " + hex(e) + " stream=" + hex(st));
  return 0;
}
int hipGraphDestroy(void*) { return 0; }
int hipGraphExecDestroy(void*) { return 0; }
}
