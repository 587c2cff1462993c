// Host check of balanced_xchunk: the choice against a look at every chunk
// count, and the host time of a call on grids of few tiles and many planes.
// Prints "OK <case>" per case; exits non-zero at a violation.
#include <chrono>
#include <cstdio>

#include "evx_stencil_tiles.hpp"

using namespace evx;

// Every chunk count up to 64, and on to eight resident rounds.
static int every_count(int64_t nx, int64_t tiles, int64_t resident, int warm) {
  int best = (int)nx;
  double best_cost = 1e300;
  for (int64_t n = 1; n <= nx; ++n) {
    const int64_t xc = (nx + n - 1) / n, used = (nx + xc - 1) / xc;
    const double cost = (double)((tiles * used + resident - 1) / resident) * (double)(xc + warm);
    if (cost < best_cost) {
      best_cost = cost;
      best = (int)xc;
    }
    if (n > 64 && tiles * n > 8 * resident) break;
  }
  return best;
}

int main() {
  int bad = 0;
  long looked = 0;
  for (int64_t resident : {256, 512, 1024, 1280, 2048})
    for (int warm : {3, 4, 6})
      for (int64_t nx : {1, 2, 3, 5, 31, 32, 33, 64, 65, 66, 67, 96, 100, 128, 201, 300, 512, 1000, 4000, 4096, 65537})
        for (int64_t tiles = 1; tiles < 6000; tiles += 1 + tiles / 7) {
          ++looked;
          const int got = balanced_xchunk(nx, tiles, resident, warm), want = every_count(nx, tiles, resident, warm);
          if (got != want && bad++ < 5)
            std::fprintf(stderr, "FAIL nx %lld tiles %lld resident %lld warm %d: %d, not %d\n", (long long)nx,
                         (long long)tiles, (long long)resident, warm, got, want);
        }
  std::printf("%s same choice in %ld cases\n", bad ? "FAILED" : "OK", looked);
  // a launch on the GPU takes about 10 us: the choice has to be a small part of that
  for (int64_t nx : {4096, 65536, 1000000}) {
    volatile int sink = 0;
    double best = 1e9;
    for (int rep = 0; rep < 5; ++rep) {
      const auto t0 = std::chrono::steady_clock::now();
      for (int i = 0; i < 200; ++i) sink = sink + balanced_xchunk(nx, 1 + (i & 1), 1024, 3);
      const double us = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count() / 200 * 1e6;
      if (us < best) best = us;
    }
    const bool ok = best < 5.0;
    bad += !ok;
    std::printf("%s %lld planes: %.2f us a call\n", ok ? "OK" : "FAILED", (long long)nx, best);
  }
  return bad != 0;
}
