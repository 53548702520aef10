// fib_set_impact (fib_runtime.cpp) on the CPU, with copies to the device that
// fail: the device's record is the host's after every call that succeeds.
#include <cstdio>
#include <cstdlib>

#include "../fib_md_amd/csrc/fib_runtime.cpp"

static int fail_copy = 0, fail_sync = 0, copies = 0;
extern "C" {
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  if (fail_copy) return hipErrorUnknown;
  ++copies;
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return fail_sync ? hipErrorUnknown : hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "made to fail"; }
}

#define WANT(x) \
  if (!(x)) return std::printf("line %d: %s\n", __LINE__, #x), 1

int main() {
  static fib_handle h;  // (not destroyed: no device)
  h.inst.resize(3);
  static DInst dev[3];
  std::memset((void *)h.inst.data(), 0, sizeof(dev));
  std::memset((void *)dev, 0, sizeof(dev));
  h.d.I = dev;
  WANT(fib_set_impact(&h, 1, 0) == FIB_OK && copies == 0);  // as it was
  WANT(fib_set_impact(&h, 1, 2) == FIB_OK && dev[1].impact == 2 && copies == 1);
  WANT(fib_set_impact(&h, 1, 2) == FIB_OK && copies == 1);
  fail_copy = 1;
  WANT(fib_set_impact(&h, 1, 3) == FIB_ERR_HIP && dev[1].impact == 2);
  WANT(fib_set_impact(&h, 2, 5) == FIB_ERR_HIP);
  fail_copy = 0;
  WANT(fib_set_impact(&h, 1, 3) == FIB_OK && dev[1].impact == 3);  // the same again
  WANT(dev[2].impact == 5 || fib_set_impact(&h, 2, 5) == FIB_OK);
  WANT(dev[2].impact == 5);
  fail_sync = 1;
  WANT(fib_set_impact(&h, 0, 4) == FIB_ERR_HIP);
  dev[0].impact = 9;  // whatever the copy left
  fail_sync = 0;
  WANT(fib_set_impact(&h, 0, 4) == FIB_OK && dev[0].impact == 4 && dev[1].impact == 3);
  const int c = copies;
  WANT(fib_set_impact(&h, 0, 4) == FIB_OK && copies == c);
  WANT(fib_set_impact(&h, 0, -1) == FIB_ERR_ARG && fib_set_impact(&h, 3, 1) == FIB_ERR_ARG);
  std::printf("ok\n");
  std::fflush(stdout);
  std::_Exit(0);
}
