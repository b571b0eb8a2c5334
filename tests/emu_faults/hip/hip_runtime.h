// The HIP emulation of tests/emu/hip with failures and stream order: any host
// call or launch can be made to fail, allocations can be limited, and every
// stream knows which work of the other streams it follows (through events and
// synchronisations), so that a test can ask what a failed call left behind.
#pragma once
#include "../../emu/hip/hip_runtime.h"
#include <map>

namespace hipfault {

using Clock = std::map<const void *, long>;          // stream -> its launches that are followed

inline std::map<const void *, Clock> g_seen;         // of each stream; its own entry counts its launches
inline std::map<const void *, Clock> g_event;
inline Clock g_host;                                 // what the host has waited for
inline long g_fail_at = 0, g_calls = 0, g_launches = 0;
inline size_t g_limit = 0;                           // bytes of one allocation, 0: none
inline hipError_t g_last = hipSuccess;

inline bool fails()
{
   g_calls++;
   if (g_fail_at == 0 || g_calls != g_fail_at) return false;
   g_last = hipErrorInvalidValue;
   return true;
}

inline void merge(Clock &to, const Clock &from)
{
   for (const auto &e : from) { long &v = to[e.first]; if (v < e.second) v = e.second; }
}

inline hipError_t malloc_(void **p, size_t n)
{
   if (g_limit && n > g_limit) { *p = nullptr; return g_last = hipErrorMemoryAllocation; }
   return fails() ? g_last : (hipMalloc)(p, n);
}
template<class T> inline hipError_t malloc_(T **p, size_t n) { return malloc_((void **)p, n); }

inline hipError_t memcpy_(void *d, const void *s, size_t n, hipMemcpyKind k) { return fails() ? g_last : (hipMemcpy)(d, s, n, k); }

inline hipError_t record(hipEvent_t e, hipStream_t s = nullptr)
{
   if (fails()) return g_last;
   g_event[e] = g_seen[s];
   return hipSuccess;
}

inline hipError_t wait(hipStream_t s, hipEvent_t e, unsigned = 0)
{
   if (fails()) return g_last;
   merge(g_seen[s], g_event[e]);
   return hipSuccess;
}

inline hipError_t sync(hipStream_t s)
{
   merge(g_host, g_seen[s]);
   return hipSuccess;
}

inline hipError_t last_error()
{
   const hipError_t e = g_last;
   g_last = hipSuccess;
   return e;
}

// a launch: false if it fails
inline bool launched(hipStream_t s)
{
   if (fails()) return false;
   g_launches++;
   merge(g_seen[s], g_host);
   g_seen[s][s]++;
   return true;
}

} // namespace hipfault

extern "C" {
// the n-th call from now fails (0: none does)
inline __attribute__((used)) void hipfault_arm(long n) { hipfault::g_fail_at = n; hipfault::g_calls = 0; hipfault::g_last = hipSuccess; }
inline __attribute__((used)) long hipfault_calls() { return hipfault::g_calls; }
inline __attribute__((used)) long hipfault_launches() { return hipfault::g_launches; }
inline __attribute__((used)) void hipfault_limit(size_t bytes) { hipfault::g_limit = bytes; }
// streams with launches that neither stream s nor the host follows
inline __attribute__((used)) int hipfault_unfollowed(hipStream_t s)
{
   using namespace hipfault;
   Clock have = g_seen[s];
   merge(have, g_host);
   int n = 0;
   for (auto &e : g_seen) if (e.first != s && e.second[e.first] > have[e.first]) n++;
   return n;
}
}

#undef hipLaunchKernelGGL
#define hipLaunchKernelGGL(kern, grid, block, shm, stream, ...)                                       \
   do {                                                                                               \
      if (::hipfault::launched(stream)) ::hipemu::launch(kern, dim3(grid), dim3(block), (size_t)(shm), __VA_ARGS__); \
   } while (0)
#define hipMalloc(p, n) ::hipfault::malloc_(p, n)
#define hipMemcpy(d, s, n, k) ::hipfault::memcpy_(d, s, n, k)
#define hipEventRecord(...) ::hipfault::record(__VA_ARGS__)
#define hipStreamWaitEvent(...) ::hipfault::wait(__VA_ARGS__)
#define hipStreamSynchronize(s) ::hipfault::sync(s)
#define hipGetLastError() ::hipfault::last_error()
