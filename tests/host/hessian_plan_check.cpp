// Properties of plan::hessian_plan over grids of shapes: every tile gets at
// least one split, the partial tiles fit the room they are given, no split of
// a finer tail is empty, and no tile gets fewer splits than asked for.
#include <cinttypes>
#include <cstdio>

#include "../../distributed_gptq_amd/csrc/plan.hpp"

using namespace gptq;

static int failed = 0;
#define CHECK(cond, n, K)                                                             \
  do {                                                                                \
    if (!(cond)) {                                                                    \
      ++failed;                                                                       \
      std::printf("%s: n=%" PRId64 " K=%" PRId64 "\n", #cond, int64_t(n), int64_t(K)); \
    }                                                                                 \
  } while (0)

int main() {
  const int64_t Ks[] = {8, 64, 256, 264, 752, 768, 1024, 2048, 3072, 4096, 4104, 5120, 6152, 8192, 11008, 11272, 13824,
                        14336, 28672, 65536, 1 << 20};
  const int64_t ns[] = {1, 31, 32, 100, 511, 512, 1023, 1024, 2048, 4097, 8229, 10277, 16384, 27685, 28709, 32768, 44038,
                        65536, 262144, 1 << 24, INT64_MAX};
  for (int64_t K : Ks)
    for (int64_t n : ns) {
      const int64_t nt = plan::hessian_tiles(K);
      const int S = plan::choose_splits(n, nt);
      CHECK(plan::hessian_room(nt, S) >= S && plan::hessian_room(nt, S) <= 64, n, K);
      for (int cap = S; cap >= 1; cap = cap / 2)
        for (int room = cap; room <= plan::hessian_room(nt, cap); ++room) {
          const plan::HessPlan p = plan::hessian_plan(n, nt, cap, room);
          const int64_t tail = nt - p.whole;
          CHECK(p.s1 == cap && p.whole >= 1 && p.whole <= nt && p.s2 >= 1 && p.s2 <= 64, n, K);
          // (one split: the first tiles have no partials)
          const int64_t parts = (p.s1 == 1 ? 0 : p.s1 * p.whole) + p.s2 * tail;
          CHECK(parts <= static_cast<int64_t>(room) * nt, n, K);
          CHECK(tail == 0 || p.s2 >= p.s1, n, K);
          CHECK(tail == 0 || p.s2 == p.s1 || n / p.s2 >= 512, n, K);
          const int64_t per = ((n / p.s2 + (n % p.s2 != 0)) + 31) / 32 * 32;  // a tail split's tokens
          CHECK(tail == 0 || p.s2 == p.s1 || (p.s2 - 1) * per < n, n, K);
        }
    }
  const plan::HessPlan none = plan::hessian_plan(0, 10, 3, 3);
  CHECK(none.s1 == 3 && none.whole == 10, 0, 0);
  std::printf("%d check(s) failed\n", failed);
  return failed != 0;
}
