// Host emulation of the index arithmetic of the semi-implicit step's and its
// adjoint's kernels, for every block, thread, plane and pass, with the
// geometry helpers that the kernels and their launches use:
//   * the periodic Cahn-Hilliard tile (evx_stencil_tiles.hpp), its plane ring included;
//   * the whole-plane z/y sweeps (evx_fft_planes.hpp);
//   * the runtime-radix line kernels (evx_fft_lines.hpp);
//   * the adjoint's streaming and separate kernels (evx_adjoint.hpp).
// Every global and LDS access must lie inside its allocation and every output
// must be written exactly once.  Prints "OK <case>" per case; exits non-zero at
// a violation.
#include <cstdio>
#include <vector>

#include "evx_adjoint.hpp"
#include "evx_fft_lines.hpp"
#include "evx_fft_planes.hpp"
#include "evx_stencil_tiles.hpp"

using namespace evx;

#define CHECK(cond, ...)                         \
  do {                                           \
    if (!(cond)) {                               \
      std::fprintf(stderr, "FAIL (%s): ", #cond); \
      std::fprintf(stderr, __VA_ARGS__);         \
      std::fprintf(stderr, "\n");                \
      return false;                              \
    }                                            \
  } while (0)

// ------------------------------------------------------- periodic CH tile --
template <typename T, int TZ, int PY>
static bool ch_launch(const Dims& d, int64_t resident, int64_t xa, int64_t xb, std::vector<uint8_t>& written) {
  using P = ChPer<T, TZ, PY>;
  using Loader = PeriodicLoader<T, 2, P::CR, P::CW, true>;
  constexpr int BY = P::BY, CW = P::CW, MW = P::MW, CS = P::CR * CW, MS = P::MR * MW;
  CHECK(sizeof(T) * (size_t)(P::NC * CS + P::NM * MS) <= P::LDS_BYTES && P::LDS_BYTES <= 160 * 1024, "LDS");
  TileGrid tg;
  unsigned base = 0;
  const unsigned blocks = ch_periodic_grid<P>(d, resident, xa, xb, &tg, &base);
  const bool is_short = tg.xc <= CH_SHORT;
  const int64_t plane_bytes = d.ny * d.nz * (int64_t)sizeof(T);
  auto in_c = [&](int at) { return at >= 0 && at < CS; };
  auto in_m = [&](int at) { return at >= 0 && at < MS; };
  for (unsigned b = 0; b < blocks; ++b) {
    const TileOrigin o = tile_origin<BY, TZ>(tg, d, base + xcd_tile(b, blocks));
    CHECK(o.ch >= 0 && o.ch < d.c && o.x0 >= 0 && o.x0 < o.x1 && o.x1 <= d.nx, "tile of block %u", b);
    const int nxp = (int)(o.x1 - o.x0), nx = (int)d.nx;
    // the plane walk and the ring: which plane every slot holds (block-uniform)
    int xw = (int)o.x0 - 2;
    while (xw < 0) xw += nx;
    std::vector<int> fetched;  // plane of the p-th fetch
    auto fetch = [&]() {
      fetched.push_back(xw);
      xw = xw + 1 == nx ? 0 : xw + 1;
    };
    const int pre = is_short ? CH_SHORT + 4 : 6;
    std::vector<int> w(pre, -1);
    for (int p = 0; p < pre; ++p)
      if (p < 5 || p <= nxp + 3) {
        w[p] = p;
        fetch();
      }
    int slot[4] = {0, 1, 2, 3};  // fetch number held: plane x0 - 2 + number
    slot[0] = 4;                 // after the warm-up's last commit
    for (int i = 0; i < nxp; ++i) {
      int* v = is_short ? &w[i + 5 < pre ? i + 5 : pre - 1] : &w[5];
      const int reads[3] = {(i + 2) & 3, (i + 3) & 3, i & 3};
      for (int q = 0; q < 3; ++q)
        CHECK(slot[reads[q]] == i + 2 + q, "step %d reads slot %d with plane number %d", i, reads[q], slot[reads[q]]);
      if (i + 3 <= nxp + 1) {
        const int to = (i + 1) & 3;
        CHECK(to != reads[0] && to != reads[1] && to != reads[2], "step %d writes a slot it reads", i);
        CHECK(*v == i + 5, "step %d commits plane number %d", i, *v);
        slot[to] = *v;
      }
      if (!is_short && i + 4 <= nxp + 1) {
        *v = (int)fetched.size();
        fetch();
      }
    }
    for (size_t p = 0; p < fetched.size(); ++p)
      CHECK(fetched[p] >= 0 && fetched[p] < nx && fetched[p] == (int)wrap(o.x0 - 2 + (int64_t)p, d.nx), "plane walk");
    std::vector<uint8_t> mu(MS, 0);
    for (int tid = 0; tid < NT; ++tid) {
      for (int k = 0; k < Loader::NPT; ++k) {
        const bool valid = k < Loader::NPT - 1 || tid + (Loader::NPT - 1) * NT < CS;
        if (!valid) continue;
        const uint32_t off = Loader::src_byte(tid, k, o.y0, o.z0, d);
        CHECK((int64_t)off + (int64_t)sizeof(T) <= plane_bytes, "load byte %u", off);
        CHECK(in_c(tid + k * NT), "LDS store %d", tid + k * NT);
      }
      const int tz = tid % TZ, r0 = tid / TZ * PY;
      const int oc = (r0 + 2) * CW + tz + 2, om = (r0 + 1) * MW + tz + 1;
      CHECK(in_c(oc - CW) && in_c(oc + PY * CW) && in_c(oc - 1) && in_c(oc + (PY - 1) * CW + 1), "c reads of %d", tid);
      CHECK(in_m(om - MW) && in_m(om + PY * MW) && in_m(om - 1) && in_m(om + (PY - 1) * MW + 1), "mu reads of %d", tid);
      for (int q = 0; q < PY; ++q) ++mu[om + q * MW];
      if (tid < P::NHALO) {
        int y, z;
        if (tid < 2 * TZ) {
          y = tid < TZ ? -1 : BY;
          z = tid % TZ;
        } else {
          const int h = tid - 2 * TZ;
          y = h % BY;
          z = h < BY ? -1 : TZ;
        }
        const int hc = (y + 2) * CW + z + 2, hm = (y + 1) * MW + z + 1;
        CHECK(in_c(hc - CW) && in_c(hc + CW) && in_c(hc - 1) && in_c(hc + 1) && in_m(hm), "halo of %d", tid);
        ++mu[hm];
      }
      const bool full = o.y0 + BY <= d.ny && o.z0 + TZ <= d.nz;
      const int64_t gz = o.z0 + tz;
      const uint32_t obyte = static_cast<uint32_t>(((o.y0 + r0) * d.nz + gz) * (int64_t)sizeof(T));
      const uint32_t orow = static_cast<uint32_t>(d.nz * (int64_t)sizeof(T));
      for (int64_t x = o.x0; x < o.x1; ++x)
        for (int q = 0; q < PY; ++q)
          if (full || (o.y0 + r0 + q < d.ny && gz < d.nz)) {
            const uint32_t at = obyte + q * orow;
            CHECK((int64_t)at + (int64_t)sizeof(T) <= plane_bytes, "store byte %u", at);
            const int64_t e = (o.ch * d.nx + x) * d.ny * d.nz + at / sizeof(T);
            CHECK(!written[e], "store twice at %lld", (long long)e);
            written[e] = 1;
          }
    }
    for (int r = 0; r < P::MR; ++r)
      for (int z = 0; z < MW; ++z) {
        const bool corner = (r == 0 || r == P::MR - 1) && (z == 0 || z == MW - 1);
        CHECK(mu[r * MW + z] == (corner ? 0 : 1), "mu (%d, %d) formed %d times", r, z, mu[r * MW + z]);
      }
  }
  return true;
}

template <typename T, int TZ, int PY>
static bool ch_case(const Dims& d, int64_t resident, int slabs) {
  std::vector<uint8_t> written((size_t)(d.c * d.vol()), 0);
  if (slabs == 0) {
    if (!ch_launch<T, TZ, PY>(d, resident, 0, -1, written)) return false;
  } else {
    int64_t w = (d.nx + slabs - 1) / slabs;
    w = (w + SLAB_XCHUNK - 1) / SLAB_XCHUNK * SLAB_XCHUNK;
    for (int64_t xa = 0; xa < d.nx; xa += w)
      if (!ch_launch<T, TZ, PY>(d, resident, xa, xa + w < d.nx ? xa + w : d.nx, written)) return false;
  }
  for (size_t i = 0; i < written.size(); ++i) CHECK(written[i], "point %zu never written", i);
  return true;
}

// ------------------------------------------------------------ whole planes --
template <typename T, int N>
static bool plane_case() {
  using G = PGeo<T, N>;
  constexpr int E = G::E, TPL = G::TPL, NH = G::NH, PITCH = G::PITCH, LDS = G::ROWS * PITCH;
  CHECK(G::LDS <= 160 * 1024 && G::THREADS % 64 == 0, "LDS %zu", G::LDS);
  CHECK((pass_tw_size<N>(typename PlaneSpec<N>::R{}) <= N), "pass tables");
  std::vector<int> spec(N * NH, 0), real(N * N, 0), rows(LDS, 0);
  for (int tid = 0; tid < G::THREADS; ++tid) {
    {  // z lines: a pair in its two rows, idle threads in the two spare rows
      const int pr = tid / TPL, tl = tid - pr * TPL;
      const bool mine = pr < N / 2;
      const int row = (mine ? pr : N / 2) * (2 * PITCH);
      if (G::WAVE) CHECK(tid / 64 == (pr * TPL) / 64 && (pr * TPL + TPL - 1) / 64 == tid / 64, "pair %d spans waves", pr);
      for (int q = 0; q < E; ++q) {
        const int e = tl + TPL * q;
        const int a = (mine ? pr : 0) * (2 * N) + e;
        CHECK(e < N && a + N < N * N, "z load %d", a);
        CHECK(row + line_slot(e) < LDS && line_slot(e) < 2 * PITCH, "exchange slot of %d", e);
        if (mine) {
          ++real[a];
          ++real[a + N];
        }
      }
      for (int k = tl; k < NH; k += TPL) {
        CHECK(row + PITCH + k < LDS && line_slot(k == 0 ? 0 : N - k) < 2 * PITCH, "row value %d", k);
        if (mine) {
          ++rows[row + k];
          ++rows[row + PITCH + k];
        }
      }
    }
    {  // y columns, idle threads in the spare column
      const int k = tid % NH, tl = tid / NH;
      const bool mine = tl < TPL;
      const int col = mine ? k : NH, t = mine ? tl : 0;
      CHECK(col < PITCH, "column %d", col);
      for (int q = 0; q < E; ++q) {
        const int e = t + TPL * q;
        CHECK(e < N && col + e * PITCH < LDS, "column value %d", e);
        CHECK(e * NH + k < N * NH, "spectrum %d", e * NH + k);
        if (mine) ++spec[e * NH + k];
      }
    }
  }
  for (int v : spec) CHECK(v == 1, "a spectrum value moved %d times", v);
  for (int v : real) CHECK(v == 1, "a real value moved %d times", v);
  for (int r = 0; r < N; ++r)
    for (int k = 0; k < NH; ++k) CHECK(rows[r * PITCH + k] == 1, "row %d value %d written %d times", r, k, rows[r * PITCH + k]);
  return true;
}

// ------------------------------------------------------------ line kernels --
static bool lines_case(int n, bool f64) {
  LinePlan P;
  CHECK(line_make_plan(n, f64, &P), "no plan of %d", n);
  CHECK(P.npass >= 2 && P.npass <= LINE_MAXPASS, "%d passes", P.npass);
  int64_t prod = 1;
  int tab = 0;
  for (int s = 0; s < P.npass; ++s) {
    const LinePass& q = P.ps[s];
    CHECK(q.p == prod && q.m * q.R == n, "pass %d", s);
    prod *= q.R;
    const bool prime = q.R > 10 && q.R != 12 && q.R != 15 && q.R != 16;
    const int span = line_span(q.R, f64);
    std::vector<int> wrote(n, 0), read(n, 0);
    for (int tl = 0; tl < P.tpl; ++tl) {
      auto butterfly = [&](int i, int q0, int step) -> bool {  // output pairs q0, q0 + step, ... of a prime pass
        int j = i * q.R, k = 0;
        if (q.p > 1) {
          const int quot = (int)(((uint64_t)(uint32_t)i * q.magic) >> 32);
          CHECK(quot == i / q.p, "%d / %d by the reciprocal: %d", i, q.p, quot);
          k = i - quot * q.p;
          j -= k * (q.R - 1);
          CHECK(q.tw + (q.R - 2) * q.p + k < P.tab, "twiddle");
        }
        for (int r = 0; r < q.R; ++r) {
          CHECK(i + r * q.m < n && j + r * q.p < n, "pass %d element", s);
          if (step == 0 || q0 == 0) ++read[i + r * q.m];
        }
        if (step == 0) {
          for (int r = 0; r < q.R; ++r) ++wrote[j + r * q.p];
        } else {
          if (q0 == 0) ++wrote[j];
          for (int o = q0 + 1; o <= (q.R - 1) / 2; o += step) {
            ++wrote[j + o * q.p];
            ++wrote[j + (q.R - o) * q.p];
          }
        }
        return true;
      };
      if (prime) {
        const int parts = P.tpl / q.m, part = tl / q.m;
        CHECK(parts >= 1, "a prime pass with too few threads");
        if (part < parts && !butterfly(tl - part * q.m, part, parts)) return false;
      } else {
        for (int t = 0; t < span; ++t)
          if (tl + t * P.tpl < q.m && !butterfly(tl + t * P.tpl, 0, 0)) return false;
      }
    }
    for (int e = 0; e < n; ++e) CHECK(wrote[e] == 1 && read[e] == 1, "pass %d: element %d read %d, written %d", s, e, read[e], wrote[e]);
    if (q.p > 1) {
      CHECK(q.tw == tab, "table of pass %d", s);
      tab += (q.R - 1) * q.p;
    }
    if (prime) {
      CHECK(q.rt == tab && P.big, "roots of pass %d", s);
      tab += q.R;
    }
  }
  CHECK(prod == n && tab == P.tab, "plan of %d", n);
  for (int64_t lines : {1, 2, 3, 7, 63, 1000, 5000, 200000}) {
    const LineGeom g = f64 ? line_strided_geom<double>(P, lines) : line_strided_geom<float>(P, lines);
    const size_t el = f64 ? 16 : 8;
    CHECK(g.lines == 1 << g.sh && g.threads >= P.tpl * g.lines && g.threads <= line_max_threads(f64, P.big != 0),
          "strided threads %d", g.threads);
    CHECK(g.threads % 64 == 0 && g.lds <= 160 * 1024, "strided LDS %zu", g.lds);
    CHECK(el * (P.tab + ((size_t)(n - 1) << g.sh) + g.lines) <= g.lds, "strided brick");
    CHECK(((g.threads - 1) >> g.sh) >= P.tpl - 1, "threads of a line");
    const LineGeom z = f64 ? line_z_geom<double>(P, (lines + 1) / 2) : line_z_geom<float>(P, (lines + 1) / 2);
    const int last = 2 * (n / 2 + 1) - 1;  // both half spectra of a pair
    CHECK(z.lines >= 1 && z.threads >= z.lines * P.tpl && z.threads <= line_max_threads(f64, P.big != 0),
          "z threads %d", z.threads);
    CHECK(z.lds <= 160 * 1024 && last + (last >> z.sh) < z.ls && n - 1 + ((n - 1) >> z.sh) < z.ls, "z line");
    CHECK(el * (P.tab + (size_t)z.lines * z.ls) <= z.lds, "z LDS");
    const int64_t blocks = (lines + 2 * z.lines - 1) / (2 * z.lines);
    CHECK((blocks - 1) * 2 * z.lines < lines && blocks * 2 * z.lines >= lines, "z blocks");
  }
  return true;
}

// ----------------------------------------------------------------- adjoint --
static bool adjoint_case(int32_t dtype, const Dims& d) {
  const AdjTiling t = adj_tiling(dtype, d);
  const AdjGeo a = adj_geo(d, t);
  const int rw = a.zw + 2 * AHALO, rows = a.tw + 2 * AHALO;
  CHECK(rw <= APAD && rw * rows <= AT, "tile %d x %d", a.zw, a.tw);
  CHECK(adj_lds(dtype == EVX_F32 ? 4 : 8) <= 160 * 1024, "LDS");
  const int64_t blocks = t.per_channel() * d.c;
  CHECK(a.per_channel() == t.per_channel(), "blocks");
  std::vector<uint8_t> written((size_t)(d.c * d.vol()), 0);
  const int slot_size = AT + 2 * APAD;
  for (int64_t bb = 0; bb < blocks; ++bb) {
    const int b = (int)xcd_tile((unsigned)bb, (unsigned)blocks);
    const int ch = b / a.per_channel(), blk = b - ch * a.per_channel();
    const int tz = blk % a.gz, ty = blk / a.gz % a.gy, tx = blk / (a.gz * a.gy);
    const int z0 = tz * a.zw, y0 = ty * a.tw, xa = tx * a.xl, xb = xa + a.xl < a.nx ? xa + a.xl : a.nx;
    CHECK(ch < a.c && xa < xb, "block %d", b);
    // planes loaded and slots of c, block-uniform
    int X = (int)wrap(xa - AHALO, a.nx), Xo = xa, s0 = 0, s1 = 2, s2 = 1;
    int held[3] = {-100, -100, -100};
    for (int p = xa - AHALO; p < xb + AHALO; ++p) {
      CHECK(X == (int)wrap(p, a.nx), "plane walk at %d", p);
      X = X + 1 == a.nx ? 0 : X + 1;  // also the plane loaded ahead
      CHECK(X >= 0 && X < a.nx, "plane ahead");
      held[s0] = p;
      if (p - 1 >= xa - AHALO) CHECK(held[s1] == p - 1, "slot of plane %d", p - 1);
      if (p - 2 >= xa - AHALO) CHECK(held[s2] == p - 2, "slot of plane %d", p - 2);
      const bool emit = p - AHALO >= xa;
      if (emit) CHECK(Xo == p - AHALO && Xo < a.nx, "output plane %d", Xo);
      Xo += emit;
      const int r = s2;
      s2 = s1;
      s1 = s0;
      s0 = r;
    }
    CHECK(Xo == xb, "chunk");
    for (int tid = 0; tid < AT; ++tid) {
      CHECK(tid - rw >= -APAD && tid + rw < AT + APAD, "LDS neighbours of %d", tid);
      for (int base : {0, 3, 5, 7})  // c, w, mu and Gmu planes
        CHECK(APAD + (base + (base == 0 ? 2 : 1)) * slot_size + tid + rw < 9 * slot_size, "LDS planes");
      const int yr = tid / rw, zr = tid - yr * rw, z = z0 + zr - AHALO, y = y0 + yr - AHALO;
      const bool own = zr >= AHALO && zr < rw - AHALO && yr >= AHALO && yr < rows - AHALO && z < a.nz && y < a.ny;
      const int64_t off = yr < rows ? wrap(y, a.ny) * a.nz + wrap(z, a.nz) : 0;
      CHECK(off >= 0 && off < (int64_t)a.ny * a.nz, "column of %d", tid);
      if (own) {
        CHECK(tid - rw >= 0 && tid + rw < rw * rows, "neighbours of an own column");
        for (int x = xa; x < xb; ++x) {
          const int64_t e = ((int64_t)ch * a.nx + x) * a.ny * a.nz + off;
          CHECK(!written[e], "output %lld twice", (long long)e);
          written[e] = 1;
        }
      }
    }
  }
  for (size_t i = 0; i < written.size(); ++i) CHECK(written[i], "voxel %zu never written", i);
  // the separate kernels: blocks of (VZ, VY) over every plane
  CHECK(vox_blocks(d) == (d.nz + VZ - 1) / VZ * ((d.ny + VY - 1) / VY) * d.nx, "blocks");
  for (int64_t x : {(int64_t)0, d.nx / 2, d.nx - 1})
    for (int64_t y : {(int64_t)0, d.ny / 2, d.ny - 1})
      for (int64_t z : {(int64_t)0, d.nz / 2, d.nz - 1}) {
        const int64_t plane = d.ny * d.nz, j = (x * d.ny + y) * d.nz + z;
        for (int64_t k : {j + (x == 0 ? (d.nx - 1) * plane : -plane), j + (x == d.nx - 1 ? -(d.nx - 1) * plane : plane),
                          j + (y == 0 ? (d.ny - 1) * d.nz : -d.nz), j + (y == d.ny - 1 ? -(d.ny - 1) * d.nz : d.nz),
                          j + (z == 0 ? d.nz - 1 : -1), j + (z == d.nz - 1 ? -(d.nz - 1) : 1)})
          CHECK(k >= 0 && k < d.vol(), "neighbour %lld", (long long)k);
      }
  return true;
}

int main() {
  int bad = 0;
  auto report = [&](bool ok, const char* what, const Dims& d) {
    bad += !ok;
    std::printf("%s %s (%lld,%lld,%lld,%lld)\n", ok ? "OK" : "FAILED", what, (long long)d.c, (long long)d.nx,
                (long long)d.ny, (long long)d.nz);
  };
  const Dims ch[] = {{1, 1, 1, 1},  {2, 1, 2, 3},   {1, 2, 3, 5},    {3, 3, 15, 31},  {1, 4, 16, 32}, {2, 5, 17, 33},
                     {1, 6, 16, 64}, {1, 12, 8, 512}, {1, 4, 4, 1024}, {1, 33, 34, 63}, {1, 300, 5, 6}, {1, 64, 100, 100}};
  for (const Dims& d : ch) {
    bool ok = true;
    for (int64_t resident : {1, 7, 64, 1280})
      ok = ok && ch_case<float, 32, 2>(d, resident, 0) && ch_case<float, 64, 4>(d, resident, 0) &&
           ch_case<double, 32, 2>(d, resident, 0);
    if (d.c == 1)
      for (int slabs : {1, 2, 5}) ok = ok && ch_case<float, 32, 2>(d, 1280, slabs) && ch_case<double, 32, 2>(d, 1280, slabs);
    report(ok, "periodic CH tile", d);
  }
#define X(N) report(plane_case<float, N>() && plane_case<double, N>(), "whole planes", Dims{1, 1, N, N});
  EVX_PLANE_SIZES(X)
#undef X
  int plans = 0;
  bool ok = true;
  for (int f64 = 0; f64 < 2; ++f64)
    for (int n = 1; n <= (f64 ? 2048 : 4096); ++n) {
      int rest = n;
      for (int p : {2, 3, 5, 7, 11, 13, 17, 19, 23, 29, 31})
        while (rest % p == 0) rest /= p;
      if (rest != 1) continue;
      ++plans;
      if (!lines_case(n, f64 != 0)) {
        std::fprintf(stderr, "  at %d points, float%d\n", n, f64 ? 64 : 32);
        ok = false;
      }
    }
  bad += !ok;
  std::printf("%s line plans: %d lengths\n", ok ? "OK" : "FAILED", plans);
  const Dims adj[] = {{1, 1, 1, 1},   {2, 2, 3, 1},   {1, 1, 2, 5},  {1, 4, 1, 200}, {2, 3, 8, 64}, {3, 5, 9, 65},
                      {1, 71, 7, 63}, {1, 9, 17, 130}, {1, 2, 300, 3}, {2, 300, 2, 3}, {1, 4000, 1, 7}, {1, 64, 64, 64}};
  for (const Dims& d : adj) report(adjoint_case(EVX_F32, d) && adjoint_case(EVX_F64, d), "adjoint", d);
  return bad != 0;
}
