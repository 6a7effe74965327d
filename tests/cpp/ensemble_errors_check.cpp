// The ensemble solve's error paths on the CPU: libodehip's host code linked against a HIP
// runtime that runs nothing and fails one chosen call.  Whatever call fails, no work may
// be left in flight on the one-workgroup solves' stream that the next call's work is not
// ordered behind: it would still write buffers which that call sets up again.
//
// Every operation on a stream is a number.  Waiting for a stream or an event completes the
// stream's operations up to there, and with them those of other streams that it waited for.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

#include "odehip.h"

namespace {

struct Stream {
  long issued = 0, done = 0;
  std::map<Stream*, long> waited;  // other stream -> its operation this one waits for
};
struct Event {
  Stream* stream = nullptr;
  long at = 0;
  std::map<Stream*, long> waited;
};
std::vector<Stream*> streams;
long calls = 0, fail_at = -1;
const char* failed = "";

bool fails(const char* what) {
  if (++calls != fail_at) return false;
  failed = what;
  return true;
}
#define CALL \
  if (fails(__func__)) return hipErrorUnknown

Stream* of(hipStream_t s) { return reinterpret_cast<Stream*>(s); }
Event* of(hipEvent_t e) { return reinterpret_cast<Event*>(e); }
void issue(hipStream_t s) {
  if (s) ++of(s)->issued;
}
void complete(Stream* s, long at, const std::map<Stream*, long>& waited) {
  if (s && at > s->done) s->done = at;
  for (const auto& [o, n] : waited)
    if (n > o->done) complete(o, n, {});
}
void* zeroed(size_t n) { return std::calloc(n ? n : 1, 1); }

}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n) { CALL; *p = zeroed(n); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { CALL; *p = zeroed(n); return hipSuccess; }
hipError_t hipFree(void* p) { CALL; std::free(p); return hipSuccess; }
hipError_t hipHostFree(void* p) { CALL; std::free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  CALL;
  std::memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
  CALL;
  std::memmove(d, s, n);
  issue(st);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t st) {
  CALL;
  std::memset(d, v, n);
  issue(st);
  return hipSuccess;
}
hipError_t hipMemcpyToSymbol(const void*, const void*, size_t, size_t, hipMemcpyKind) {
  CALL;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { CALL; *p = zeroed(1 << 20); return hipSuccess; }
hipError_t hipSetDevice(int) { CALL; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { CALL; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "made to fail"; }
hipError_t hipDeviceSynchronize() {
  CALL;
  for (Stream* s : streams) s->done = s->issued;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  CALL;
  streams.push_back(new Stream());
  *s = reinterpret_cast<hipStream_t>(streams.back());
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  CALL;
  if (s) complete(of(s), of(s)->issued, of(s)->waited);
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  CALL;
  if (s && of(e)->stream) {
    long& n = of(s)->waited[of(e)->stream];
    if (of(e)->at > n) n = of(e)->at;
  }
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { CALL; return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  CALL;
  *g = reinterpret_cast<hipGraph_t>(zeroed(8));
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  CALL;
  *e = reinterpret_cast<hipGraphExec_t>(zeroed(8));
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) { CALL; issue(s); return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { std::free(g); return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { std::free(e); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { CALL; *e = reinterpret_cast<hipEvent_t>(new Event()); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { CALL; *e = reinterpret_cast<hipEvent_t>(new Event()); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { delete of(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  CALL;
  of(e)->stream = of(s);
  of(e)->at = s ? of(s)->issued : 0;
  of(e)->waited = s ? of(s)->waited : std::map<Stream*, long>{};
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) { CALL; complete(of(e)->stream, of(e)->at, of(e)->waited); return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t e) { CALL; complete(of(e)->stream, of(e)->at, of(e)->waited); return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { CALL; *ms = 1.0f; return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t s) {
  CALL;
  issue(s);
  return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t);
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*);
static dim3 grid_, block_;
static size_t shared_;
static hipStream_t stream_;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s) {
  grid_ = g;
  block_ = b;
  shared_ = m;
  stream_ = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
  *g = grid_;
  *b = block_;
  *m = shared_;
  *s = stream_;
  return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*,
                           void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
}

// Fails the k-th HIP call of a solve, for every k it makes; returns the number of
// violations.
int main() {
  const int sizes[] = {16, 100, 300, 700, 40};
  size_t nv = 0;
  for (int n : sizes) nv += 6 * static_cast<size_t>(n);
  int bad = 0;
  long tried = 0;
  for (int rounds = 1; rounds >= 0; --rounds) {
    const int n_sys = rounds ? 5 : 2;  // with lockstep rounds beside, and without
    for (long k = 1;; ++k) {
      fail_at = -1;
      streams.clear();
      odehip_context* ctx = nullptr;
      if (odehip_create(0, &ctx) != ODEHIP_OK) return 100;
      double* x = static_cast<double*>(zeroed(nv * sizeof(double)));
      odehip_ensemble_options o{};
      o.tf = 1.0;
      o.atol = o.rtol = 1e-6;
      o.tile_config = ODEHIP_ENS_TILE_AUTO;
      auto solve = [&] {
        return odehip_ensemble_solve(ctx, ODEHIP_TABLEAU_DOPRI5, n_sys, sizes,
                                     ODEHIP_NBODY_FAST, 1e-2, nullptr, &o, x, x, nullptr,
                                     nullptr);
      };
      calls = 0;
      fail_at = k;
      failed = "";
      const int rc = solve();
      const bool hit = *failed != 0;
      // the context's stream comes first; what it waits for is ordered before any
      // later work on it
      Stream* own = streams[0];
      for (Stream* s : streams) {
        if (s == own) continue;
        const auto w = own->waited.find(s);
        const long ordered = w == own->waited.end() ? 0 : w->second;
        if (s->issued > s->done && s->issued > ordered) {
          std::printf("call %ld (%s) failed, rc %d: %ld operations left in flight\n", k, failed,
                      rc, s->issued - std::max(s->done, ordered));
          ++bad;
        }
      }
      // (after the arena's allocation has failed, too, the next call finds what it needs)
      fail_at = -1;
      calls = 0;
      if (hit && solve() != ODEHIP_OK) {
        std::printf("call %ld (%s) failed: so does the next solve\n", k, failed);
        ++bad;
      }
      odehip_destroy(ctx);
      std::free(x);
      if (!hit) break;
      ++tried;
      if (k > 100000) return 101;
    }
  }
  std::printf("%ld failing calls tried, %d violations\n", tried, bad);
  return bad ? 1 : 0;
}
