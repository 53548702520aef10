// fib_arena_force (fib_runtime.cpp) on the CPU: configurations that do not fit
// the arena are refused before anything is launched (no kernel is linked here:
// a launch would end the program).
#include <cstdio>
#include <cstdlib>

#include "../fib_md_amd/csrc/fib_runtime.cpp"

namespace fibk {
size_t bsum_len(int nbucket) { return (size_t)nbucket / 2048 + 3; }
}

#define WANT(x) \
  if (!(x)) return std::printf("line %d: %s\n", __LINE__, #x), 1

int main() {
  fib_params p;
  fib_default_params(&p);
  const double a = 1.1 * 1.8 * 2.0951e-10;
  double X[6] = {}, F[6], u = 0;
  int32_t at[2] = {1, 1};
  static char byte;  // (never written)
  const size_t arena = (size_t)64 << 20;
  // one of the cell arrays, or both, or a per-atom array does not fit; what
  // follows it would
  const double boxes[][3] = {{600.5, 600.5, 600.5}, {400.5, 400.5, 100.5}, {260.5, 260.5, 260.5}};
  for (int prec : {FIB_PREC_FP64, FIB_PREC_MIXED})
    for (auto &b : boxes) {
      const double lb[3] = {b[0] * a, b[1] * a, b[2] * a};
      const int32_t rc = fib_arena_force(&p, prec, 2, 2, 0, lb, 0, X, at, F, &u, &byte, arena, 1 << 20, nullptr);
      WANT(rc == FIB_ERR_ARG);
      WANT(std::string(fib_last_error(nullptr)).find("arena") != std::string::npos);
    }
  const double lb[3] = {10.5 * a, 10.5 * a, 10.5 * a};
  for (size_t bytes : {(size_t)0, (size_t)100, (size_t)4096, (size_t)100000})
    WANT(fib_arena_force(&p, FIB_PREC_MIXED, 2, 2, 0, lb, 0, X, at, F, &u, &byte, bytes, 1 << 20, nullptr) == FIB_ERR_ARG);
  std::printf("ok\n");
  return 0;
}
