// Host emulation of the index arithmetic of the explicit right-hand sides
// (evx_explicit.hip): every block, thread and plane, with the kernels' own tile
// and chunk helpers.  Global and LDS accesses stay inside, every point is written
// once, and float64 grids of few rows do not leave most of a tile's threads
// without a point.  Prints "OK <case>" per case; exits non-zero at a violation.
#include <cstdio>
#include <vector>

#include "evx_explicit.hpp"
#include "evx_fft_engine.hpp"

using namespace evx;

#define CHECK(cond, ...)                                          \
  do {                                                            \
    if (!(cond)) {                                                \
      std::fprintf(stderr, "FAIL (%s): ", #cond);                 \
      std::fprintf(stderr, __VA_ARGS__);                          \
      std::fprintf(stderr, "\n");                                 \
      return false;                                               \
    }                                                             \
  } while (0)

template <typename X>
static bool emulate(const Dims& d, const Bc& bc, int64_t resident, double* busy) {
  TileGrid tg;
  const unsigned blocks = x_tiles<X>(d, d.c, resident, &tg);
  const int64_t plane = d.ny * d.nz;
  std::vector<uint8_t> written((size_t)(d.c * d.vol()), 0);
  int64_t threads = 0, working = 0;
  for (unsigned b = 0; b < blocks; ++b) {
    const TileOrigin o = tile_origin<X::BY, X::TZ>(tg, d, xcd_tile(b, blocks));
    CHECK(o.ch >= 0 && o.ch < d.c && o.x0 >= 0 && o.x0 < o.x1 && o.x1 <= d.nx, "tile of block %u", b);
    for (int64_t x = o.x0 - 1; x <= o.x1; ++x) {  // planes loaded, wrapped by one period at most
      const int64_t w = x < 0 ? x + d.nx : x >= d.nx ? x - d.nx : x;
      CHECK(w >= 0 && w < d.nx, "plane %lld", (long long)x);
    }
    for (int tid = 0; tid < NT; ++tid) {
      for (int k = 0; k < X::NPT; ++k) {
        const int i = tid + k * NT < X::PLANE - 1 ? tid + k * NT : X::PLANE - 1;
        uint8_t f;
        const uint32_t off = X::source(i, o.y0, o.z0, d, bc, &f);
        CHECK(off < (uint64_t)plane, "load %u of thread %d, block %u", off, tid, b);
        CHECK(!(f & 12) || bc.kind[1] != EVX_BC_PERIODIC, "y ghost rule on a periodic axis");
        const bool last_ok = tid + (X::NPT - 1) * NT < X::PLANE;
        if (k < X::NPT - 1 || last_ok) CHECK(tid + k * NT < X::PLANE, "LDS store of thread %d", tid);
      }
      const int tz = tid % X::TZ, r0 = tid / X::TZ * X::PY, at = (r0 + 1) * X::W + tz + 1;
      CHECK(at - X::W - 1 >= 0 && at + X::PY * X::W + 1 < X::PLANE, "LDS reads of thread %d", tid);
      const int64_t gz = o.z0 + tz, gy0 = o.y0 + r0;
      const int rows = gz < d.nz ? (int)(gy0 + X::PY <= d.ny ? X::PY : d.ny - gy0) : 0;
      ++threads;
      working += rows > 0;
      for (int64_t x = o.x0; x < o.x1; ++x)
        for (int q = 0; q < X::PY; ++q)
          if (q < rows) {
            const int64_t at_out = o.ch * d.vol() + x * plane + (uint32_t)(gy0 * d.nz + gz) + q * (uint32_t)d.nz;
            CHECK(at_out < d.c * d.vol() && !written[at_out], "store %lld", (long long)at_out);
            written[at_out] = 1;
          }
    }
  }
  for (size_t i = 0; i < written.size(); ++i) CHECK(written[i], "point %zu never written", i);
  *busy = (double)working / (double)threads;
  return true;
}

int main() {
  int bad = 0;
  const Dims shapes[] = {{1, 1, 1, 1},   {2, 3, 1, 700},  {1, 2, 8, 33},  {1, 5, 8, 64},   {1, 4, 9, 100},
                         {1, 3, 16, 64}, {1, 3, 17, 65},  {1, 7, 24, 63}, {3, 9, 40, 129}, {1, 2, 41, 40},
                         {1, 40, 8, 32}, {1, 300, 1, 1},  {1, 6, 48, 96}, {1, 33, 34, 35}, {1, 5, 7, 2000}};
  const int kinds[][3] = {{EVX_BC_PERIODIC, EVX_BC_PERIODIC, EVX_BC_PERIODIC},
                          {EVX_BC_NEUMANN, EVX_BC_DIRICHLET, EVX_BC_PERIODIC},
                          {EVX_BC_DIRICHLET, EVX_BC_PERIODIC, EVX_BC_NEUMANN}};
  for (const Dims& d : shapes)
    for (int64_t resident : {1, 7, 1280}) {
      bool ok = true;
      double busy[2] = {0.0, 0.0};
      for (const auto& k : kinds) {
        Bc bc{};
        for (int a = 0; a < 3; ++a) bc.kind[a] = k[a];
        ok = ok && !flat_tiles<float>(d) && emulate<XTile<float, false>>(d, bc, resident, &busy[0]);
        ok = ok && (flat_tiles<double>(d) ? emulate<XTile<double, true>>(d, bc, resident, &busy[1])
                                          : emulate<XTile<double, false>>(d, bc, resident, &busy[1]));
      }
      // of up to eight rows in wide tiles a row of threads without a point is one in eight
      if (d.ny <= 8 && d.nz >= 700) ok = ok && busy[1] >= 0.8 * (double)((d.ny + 1) / 2) / 4.0;
      bad += !ok;
      std::printf("%s (%lld,%lld,%lld,%lld) resident %lld: threads with points %.2f, %.2f\n", ok ? "OK" : "FAILED",
                  (long long)d.c, (long long)d.nx, (long long)d.ny, (long long)d.nz, (long long)resident, busy[0],
                  busy[1]);
    }
  return bad != 0;
}
