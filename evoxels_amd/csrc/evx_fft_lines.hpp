// Transforms of line lengths without a size-specialised kernel: a Stockham
// engine whose radices are chosen at plan time and whose butterflies are
// compile-time (2-10 and, in float32, 12, 15 and 16 in registers; the primes
// 11-31 by the symmetric form below).
//
// A line of n points is worked on by tpl threads; in the pass of radix R a
// thread owns up to line_span<T>(R) whole butterflies i = tl + s*tpl (i < m =
// n/R), reads elements i + r*m and writes (i - i mod p)*R + i mod p + r*p, p
// the product of the radices before.  The first pass reads its line from
// global memory and the last one writes it back, so LDS holds one copy of the
// lines and carries only the exchanges between passes (read, barrier,
// write).  What bounds these kernels is the same HBM stream as the
// size-specialised ones; few, large radices keep the exchanges and the
// twiddle products down (350 = 10*7*5).  Index division by p is a multiply by
// a precomputed reciprocal, and each pass reads its own twiddle table, so that
// consecutive butterflies read consecutive entries.
//
// Measured on a 300x270x350 float32 step (MI355X), before (every pass a loop
// over run-time radix 2/3/4/5/8 passes in LDS, element-major lines, integer
// divisions per element): z R2C 469 -> 57 us, y 272 / 217 -> 57 / 48, x 300 ->
// 88, z C2R 597 -> 86; the step 1950 -> 416 us.  The size-specialised kernels
// stay for their lengths: 256^3 float32 186 us against 215 with these,
// 100^3 float64 61 against 73, 32^3 float32 29 against 39.
#pragma once
#include "evx_common.hpp"
#include "evx_fft_tiles.hpp"

#include <vector>

namespace evx {

// -------------------------------------------------------------------- plan --
constexpr int LINE_MAXPASS = 8;

// Butterflies a thread holds in one pass: two where they fit the registers
// of four wavefronts per SIMD.
__host__ __device__ constexpr int line_span(int R, bool f64) { return f64 ? (R <= 5 ? 2 : 1) : (R <= 10 ? 2 : 1); }

struct LinePass {
  int R, m, p;     // radix, butterflies n/R, product of the radices before
  int tw, rt;      // table offsets: w_{pR}^(rk) at tw + (r-1)*p + k; for prime R > 10, w_R^j at rt + j
  uint32_t magic;  // i / p = umulhi(i, magic) for i < 65536 (p > 1)
};

struct LinePlan {
  int n, npass, tpl, tab;  // points, passes, threads per line, table entries
  int big;                 // a prime radix above 10 is among the passes
  LinePass ps[LINE_MAXPASS];
};

// Cost of a radix per point: the exchange plus the butterfly's operations.
inline double line_radix_cost(int R) {
  switch (R) {
    case 2: return 17;
    case 3: return 20;
    case 4: return 19;
    case 5: return 23;
    case 6: return 22;
    case 7: return 28;
    case 8: return 22;
    case 9: return 26;
    case 10: return 26;
    case 12: return 26;
    case 15: return 30;
    case 16: return 27;
    default: return 22 + 1.5 * R;
  }
}

inline void line_search(int n, int from, bool f64, std::vector<int>& cur, double cost, std::vector<int>& best,
                        double& best_cost) {
  if (n == 1) {
    if (cost < best_cost) {
      best_cost = cost;
      best = cur;
    }
    return;
  }
  static const int radices[] = {31, 29, 23, 19, 17, 16, 15, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};
  if ((int)cur.size() == LINE_MAXPASS) return;
  for (int i = from; i < (int)(sizeof(radices) / sizeof(radices[0])); ++i) {
    const int R = radices[i];
    if (n % R || (f64 && (R == 12 || R == 15 || R == 16))) continue;
    cur.push_back(R);
    line_search(n / R, i, f64, cur, cost + line_radix_cost(R), best, best_cost);
    cur.pop_back();
  }
}

// The passes of an n-point line (prime factors up to 31), largest radix
// first: the first pass has no twiddles.  False if no plan of at most
// LINE_MAXPASS passes exists.
inline bool line_make_plan(int n, bool f64, LinePlan* out) {
  std::vector<int> cur, best;
  double bc = 1e300;
  line_search(n, 0, f64, cur, 0.0, best, bc);
  if (bc >= 1e300) return false;
  while (best.size() < 2) best.push_back(1);  // at least one exchange: a first and a last pass
  LinePlan& P = *out;
  P.n = n;
  P.npass = (int)best.size();
  P.tpl = 1;
  P.tab = 0;
  P.big = 0;
  int p = 1;
  for (int s = 0; s < P.npass; ++s) {
    const int R = best[s];
    LinePass& q = P.ps[s];
    q.R = R;
    q.m = n / R;
    q.p = p;
    q.magic = p > 1 ? (uint32_t)((uint64_t(1) << 32) / (uint32_t)p + 1) : 0u;
    q.tw = P.tab;
    if (p > 1) P.tab += (R - 1) * p;
    q.rt = P.tab;
    if (R > 10 && R != 12 && R != 15 && R != 16) {
      P.big = 1;
      P.tab += R;
    }
    const int span = line_span(R, f64), t = (q.m + span - 1) / span;
    if (t > P.tpl) P.tpl = t;
    p *= R;
  }
  return true;
}

// Fills the table of a plan: w(j, n) = exp(-2 pi i j / n).
template <typename T, typename W>
void line_fill_table(const LinePlan& P, cpx<T>* tab, W&& w) {
  for (int s = 0; s < P.npass; ++s) {
    const LinePass& q = P.ps[s];
    if (q.p > 1)
      for (int r = 1; r < q.R; ++r)
        for (int k = 0; k < q.p; ++k) tab[q.tw + (r - 1) * q.p + k] = w((int64_t)r * k, q.p * q.R);
    if (q.R > 10 && q.R != 12 && q.R != 15 && q.R != 16)
      for (int j = 0; j < q.R; ++j) tab[q.rt + j] = w(j, q.R);
  }
}

// ------------------------------------------------------------------ launch --
struct LineGeom {
  int lines;    // strided: lines per block (a power of two); z: line pairs per block
  int sh;       // log2(lines) / pad shift of a z line
  int ls;       // z: LDS elements per line
  int threads;
  size_t lds;
};

constexpr size_t LINE_LDS = 80 * 1024;  // two blocks per CU
// Threads per block the kernels are compiled for: the prime radices in
// float64 need the registers of two wavefronts per SIMD.
__host__ __device__ constexpr int line_max_threads(bool f64, bool big) { return f64 && big ? 512 : 1024; }

// Wavefronts per SIMD asked of the compiler: as many (up to `most`) as each
// kernel's registers allow without spilling (but for two registers of the
// float32 x sweep with prime radices).
__host__ __device__ constexpr int line_min_waves(bool f64, bool big, int most = 6) {
  return big ? (f64 ? 2 : 4) : f64 && most > 5 ? 5 : most;
}

// Strided sweeps: bricks of 128 bytes of adjacent lines (more for short
// lines, so that a block has 256 threads, as long as the launch keeps a
// thousand blocks), fewer where a brick would exceed the LDS.
template <typename T>
inline LineGeom line_strided_geom(const LinePlan& P, int64_t nlines) {
  constexpr size_t el = sizeof(cpx<T>);
  const size_t tab = el * P.tab;
  const int maxt = line_max_threads(sizeof(T) == 8, P.big != 0);
  int sh = sizeof(T) == 8 ? 3 : 4;
  auto lds = [&](int s) { return tab + el * ((size_t)P.n << s); };
  while ((P.tpl << sh) < 256 && sh < 6 && lds(sh + 1) <= 40 * 1024 && (nlines >> (sh + 1)) >= 1024) ++sh;
  while (sh > 0 && (lds(sh) > LINE_LDS || (P.tpl << sh) > maxt)) --sh;
  LineGeom g;
  g.sh = sh;
  g.lines = 1 << sh;
  g.ls = 0;
  g.threads = ((P.tpl << sh) + 63) / 64 * 64;
  g.lds = lds(sh);
  return g;
}

// z sweeps: line pairs per block for about 256 threads in whole wavefronts,
// fewer on small grids so that the launch keeps a thousand blocks.
template <typename T>
inline LineGeom line_z_geom(const LinePlan& P, int64_t npairs) {
  constexpr size_t el = sizeof(cpx<T>);
  const size_t tab = el * P.tab;
  const int slots = 2 * (P.n / 2 + 1);  // the C2R stages both half spectra of a pair
  LineGeom g;
  g.sh = 4;
  g.ls = slots + (slots - 1) / 16;
  if (tab + el * g.ls > LINE_LDS) {
    g.sh = 30;  // no padding
    g.ls = slots;
  }
  int lp = 256 / P.tpl;
  if (lp < 1) lp = 1;
  while (lp > 1 && tab + el * g.ls * lp > 40 * 1024) --lp;
  while (lp > 1 && npairs / lp < 1024) --lp;
  // the pair count of [lp/2, lp] that fills its wavefronts best
  int pick = lp;
  double fill = 0.0;
  for (int c = lp; c >= 1 && 2 * c >= lp; --c) {
    const double f = (double)(c * P.tpl) / ((c * P.tpl + 63) / 64 * 64);
    if (f > fill + 0.02) {
      fill = f;
      pick = c;
    }
  }
  g.lines = pick;
  g.threads = (pick * P.tpl + 63) / 64 * 64;
  g.lds = tab + el * g.ls * (size_t)pick;
  return g;
}

// Launches (instantiated per type in evx_fft_lines_f32.hip / _f64.hip): z R2C and
// C2R of nlines lines, and the strided sweep of MODE 0 (forward), 1 (inverse)
// or 2 (forward * multiplier * inverse).  tab: the plan's table on the device.
template <typename T>
int line_run_z_r2c(const LinePlan& P, const void* tab, const void* x, void* spec, int64_t nlines, int64_t pitch,
                   hipStream_t s);
template <typename T>
int line_run_z_c2r(const LinePlan& P, const void* tab, const void* spec, void* out, const void* base, double scale,
                   int64_t nlines, int64_t pitch, hipStream_t s);
template <typename T>
int line_run_strided(int mode, const LinePlan& P, const void* tab, void* spec, int64_t nlines, const LineMap& lm,
                     const Prefac& pf, hipStream_t s);

}  // namespace evx
