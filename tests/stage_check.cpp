// Host transfers (fib_stage.h) on the CPU: HIP's memory calls are stand-ins,
// operator new fails at the k-th request.  Prints "ok" when every transfer
// either moved its arrays bit for bit or returned an error, and threw nothing.
#include <cstdio>
#include <cstdlib>
#include <functional>

#include "../fib_md_amd/csrc/fib_stage.h"

static std::atomic<long> left{-1};  // requests until one fails (-1: none does)
static std::atomic<int> hip_left{-1};
void *operator new(size_t n) {
  if (left >= 0 && left-- == 0) throw std::bad_alloc();
  if (void *p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

static hipError_t hip(hipError_t e) {
  return hip_left >= 0 && hip_left-- == 0 ? e : hipSuccess;
}
extern "C" {
hipError_t hipMalloc(void **p, size_t n) { *p = std::malloc(n); return hipSuccess; }
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = std::malloc(n); return hipSuccess; }
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)std::malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return hipErrorInvalidValue; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hip(hipErrorUnknown);
}
}

static bool transfer(size_t n, std::atomic<int> *hip_fail, long fail_at, bool &failed) {
  std::vector<unsigned char> a(3 * n), b(3 * n), c(n);
  for (size_t k = 0; k < a.size(); ++k) a[k] = (unsigned char)(k * 7 + k / 251);
  for (size_t k = 0; k < c.size(); ++k) c[k] = (unsigned char)(k * 5 + 1);
  Stage st;
  st.fit(n / 8);
  Parts P, Q;
  const size_t oa = P.add(3 * n, a.data()), oz = P.add(3 * n, nullptr), oc = P.add(n, c.data());
  (void)oz;
  std::vector<unsigned char> c2(n);
  Q.add(3 * n, b.data());
  Q.add(n, c2.data());
  bool ok = st.reserve(P.used) == hipSuccess;
  if (hip_fail) *hip_fail = (int)fail_at; else left = fail_at;
  const hipError_t up = st.copy(true, P, nullptr);
  const bool whole = up != hipSuccess || (!std::memcmp(st.dev + oa, a.data(), 3 * n) &&
                                          !std::memcmp(st.dev + oc, c.data(), n));
  const hipError_t back = up != hipSuccess ? up : st.copy(false, Q, nullptr);
  failed = up != hipSuccess || back != hipSuccess;
  left = -1;
  hip_left = -1;
  if (up == hipSuccess && back == hipSuccess)
    ok = ok && !std::memcmp(a.data(), b.data(), 3 * n) && !std::memcmp(c.data(), c2.data(), n);
  st.release();
  return ok && whole;
}

int main() {
  int failures = 0;
  // one copy, one chunk each, several chunks per lane
  for (size_t n : {(size_t)8, (size_t)4096, (size_t)600000, (size_t)1500001, (size_t)6000000})
    for (int by_hip = 0; by_hip < 2; ++by_hip)
      for (long k = -1; k < 40; ++k) {
        bool failed = false;
        try {
          if (!transfer(n, by_hip ? &hip_left : nullptr, k, failed)) {
            std::printf("wrong data: %zu bytes, request %ld\n", n, k);
            return 1;
          }
        } catch (...) {
          std::printf("thrown: %zu bytes, request %ld\n", n, k);
          return 1;
        }
        if (k < 0 && failed) return std::printf("failed without cause: %zu\n", n), 1;
        failures += failed;
      }
  std::printf("ok, %d transfers failed\n", failures);
  return failures > 0 ? 0 : 1;
}
