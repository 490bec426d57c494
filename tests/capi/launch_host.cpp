// Host check of the evaluation's block size (stormm_amd/csrc/mm_device.h): whatever size a caller
// asks for, a launch uses whole wavefronts, at least the threads that stage_load needs for the
// largest unit and at most what the kernel is compiled for, and sizes that fit as they are stay.
#include <climits>
#include <cstdio>
#include <cstring>

#include <hip/hip_runtime.h>

#include "../../stormm_amd/csrc/mm_device.h"

using namespace stormm_amd;

static int failures = 0;

template <typename T, bool HEAVY> static void check(const char *kernel) {
  constexpr int limit = EvalBlockLimit<T, HEAVY>::value;
  const int asked[] = {1, 63, 64, 127, 128, 192, 255, 256, 257, 300, 384, 512, 513, 700, 768,
                       1000, 1024, 1025, 4096, INT_MAX};
  for (int a : asked) {
    for (int blocks : {1, 256, 257, 5000}) {
      for (int maxa : {16, 128, 336, 512}) {
        MMKit k;
        std::memset(&k, 0, sizeof(k));
        k.block = a;
        k.cus = 256;
        k.maxa = maxa;
        const int b = eval_block<T, HEAVY>(k, blocks);
        const bool whole = (b % 64 == 0) && b >= kMinEvalBlock && b <= limit;
        const bool kept = !(a % 64 == 0 && a >= kMinEvalBlock && a <= limit) || b == a;
        if ((!whole || !kept) && failures++ < 10) {
          std::printf("MISMATCH %s: %d threads asked for, %d used\n", kernel, a, b);
        }
      }
    }
  }
}

int main() {
  check<float, false>("single precision");
  check<double, false>("double precision");
  check<double, true>("double precision, clash-damped forces");
  std::printf(failures == 0 ? "launch ok\n" : "launch FAILED\n");
  return failures == 0 ? 0 : 1;
}
