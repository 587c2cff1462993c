// Explicit right-hand sides with their step epilogues: reaction-diffusion, the
// two-species Gray-Scott system and two-phase Allen-Cahn.
//
// Every kernel streams along x: a block owns a (BY x TZ) tile of (y, z) and an
// x-chunk, loads each x-plane of the tile (plus a one-point halo) once, and
// passes it through one of two LDS slots.  A thread owns PY rows of one
// column and reads its own column (with the rows above and below) and the
// columns at z-1 and z+1 of each plane once; the planes x-1 and x it needs
// beside the new plane x+1 stay in its registers.  So a plane takes one
// barrier and (3 PY + 2)/PY LDS reads per point (3 (PY + 2)/PY with corners)
// instead of one per neighbour.  The epilogue is compiled in, its operands are
// loaded before the arithmetic, and tiles without a Dirichlet ghost skip the
// ghost arithmetic.
//
// Ghost values never exist in HBM: out-of-grid points are resolved on load
// (periodic wrap, Neumann copy, Dirichlet 2v-u, applied x then y then z as in
// boundary_conditions.py:33-59).  Floating-point contraction is off so that
// every product and sum rounds where the reference's eager torch expression
// rounds.
#include "evx_explicit.hpp"

#pragma clang fp contract(off)

namespace evx {
namespace {

// Loads the tile's points of one x-plane into registers and writes them to
// LDS with clip and ghost rules applied.  The y/z part of every point is
// resolved once: periodic axes wrap, others clamp, which is the Neumann rule.
template <typename T, bool CLIP, typename X>
struct XLoader {
  static constexpr int NPT = X::NPT;
  uint32_t off[NPT];  // in-plane element of the source point
  uint8_t f[NPT];     // y/z ghost flags: 4/8 = y low/high, 16/32 = z low/high
  bool last_ok;       // this thread's last point lies in the tile
  bool rules;         // block-uniform: some y/z ghost of the tile is a Dirichlet one

  struct Plane {
    T v[NPT];
    int xf;  // x ghost: 1 low, 2 high, 64 values final (staggered_x)
  };

  __device__ __forceinline__ void init(int64_t y0, int64_t z0, const Dims& d, const Bc& bc, int tid) {
    const bool yd = bc.kind[1] == EVX_BC_DIRICHLET && (y0 == 0 || y0 + X::BY >= d.ny);
    const bool zd = bc.kind[2] == EVX_BC_DIRICHLET && (z0 == 0 || z0 + X::TZ >= d.nz);
    rules = yd || zd;
    last_ok = tid + (NPT - 1) * NT < X::PLANE;
#pragma unroll
    for (int k = 0; k < NPT; ++k) {
      const int i = tid + k * NT < X::PLANE - 1 ? tid + k * NT : X::PLANE - 1;
      off[k] = X::source(i, y0, z0, d, bc, &f[k]);
    }
  }

  // Plane xg in [-1, nx] of the field u.
  __device__ __forceinline__ void fetch(const T* __restrict__ u, int64_t xg, const Dims& d, const Bc& bc,
                                        Plane& p) const {
    const int64_t plane = d.ny * d.nz;
    p.xf = 0;
    if (xg < 0 || xg >= d.nx) {
      if (bc.kind[0] == EVX_BC_PERIODIC) {
        xg += xg < 0 ? d.nx : -d.nx;
      } else if (staggered_x(bc)) {
        fetch_node(u, xg < 0, d, bc, p);
        return;
      } else {
        p.xf = xg < 0 ? 1 : 2;
        xg = xg < 0 ? 0 : d.nx - 1;
      }
    }
    const T* const q = u + xg * plane;
#pragma unroll
    for (int k = 0; k < NPT; ++k) p.v[k] = q[off[k]];
  }

  // staggered_x ghost plane (boundary_conditions.py:96-121), in the order of
  // the reference's expression fac1*u1 - fac2*u2 with the factors rounded to
  // the working precision.
  __device__ void fetch_node(const T* __restrict__ u, bool low, const Dims& d, const Bc& bc, Plane& p) const {
    p.xf = 64;
    if (bc.kind[0] == EVX_BC_NODE_VALUE) {
      const T v0 = static_cast<T>(low ? bc.node_lo : bc.node_hi);
#pragma unroll
      for (int k = 0; k < NPT; ++k) p.v[k] = v0;
      return;
    }
    const int64_t plane = d.ny * d.nz;
    const T* p1 = u + (low ? 0 : d.nx - 1) * plane;
    const T* p2 = u + (low ? 1 : d.nx - 2) * plane;
    const T f1 = static_cast<T>(4.0 / 3.0), f2 = static_cast<T>(1.0 / 3.0);
#pragma unroll
    for (int k = 0; k < NPT; ++k) {
      T a = p1[off[k]], b = p2[off[k]];
      if (CLIP) {
        a = clip01(a);
        b = clip01(b);
      }
      p.v[k] = f1 * a - f2 * b;
    }
  }

  __device__ __forceinline__ void commit(T* s, const Plane& p, const Bc& bc, int tid) const {
    const bool plain = !rules && !(p.xf & 3 && bc.kind[0] == EVX_BC_DIRICHLET);  // block-uniform
#pragma unroll
    for (int k = 0; k < NPT; ++k) {
      T x = p.v[k];
      if (CLIP) x = (p.xf & 64) ? x : clip01(x);
      if (!plain && !(p.xf & 64)) {
        const int g = p.xf | f[k];
        if (g) {  // only the wavefronts that hold a ghost point
          const int8_t o[3] = {(int8_t)((g & 1) ? -1 : (g & 2) ? 1 : 0), (int8_t)((g & 4) ? -1 : (g & 8) ? 1 : 0),
                               (int8_t)((g & 16) ? -1 : (g & 32) ? 1 : 0)};
          x = apply_rules(x, o, bc);
        }
      }
      if (k < NPT - 1 || last_ok) s[tid + k * NT] = x;
    }
  }
};

// A thread's view of one plane: its column rows r0-1 .. r0+PY, and the rows
// r0-H .. of the columns at z-1, z+1 (H = 1 with corners, 0 without).
template <typename T, int H, typename X>
struct XView {
  static constexpr int PY = X::PY;
  T c[PY + 2], m[PY + 2 * H], p[PY + 2 * H];
  __device__ __forceinline__ void read(const T* s, int at) {  // at: LDS offset of the point (r0, z)
    constexpr int W = X::W;
#pragma unroll
    for (int j = 0; j < PY + 2; ++j) c[j] = s[at + (j - 1) * W];
#pragma unroll
    for (int j = 0; j < PY + 2 * H; ++j) {
      m[j] = s[at + (j - H) * W - 1];
      p[j] = s[at + (j - H) * W + 1];
    }
  }
};

// Epilogue of one output plane: operands loaded early, the result stored.
// EULER's u is the state at the point; the RK4 base defaults to it.
template <typename T, int MODE>
struct XOut {
  T* out;
  const T* u;         // the state (for a base of NULL)
  const T* base;
  const T* acc_in;
  T* acc_out;
  T c;
  __device__ __forceinline__ void load(uint32_t i, T& b, T& a) const {
    if constexpr (MODE == EVX_OUT_EULER) b = u[i];
    if constexpr (MODE >= EVX_OUT_RK4_FIRST) b = base[i];
    if constexpr (MODE >= EVX_OUT_RK4_MID) a = acc_in[i];
  }
  __device__ __forceinline__ void store(uint32_t i, T r, T b, T a) const {
    if constexpr (MODE == EVX_OUT_RHS) {
      out[i] = r;
    } else if constexpr (MODE == EVX_OUT_EULER) {
      out[i] = b + c * r;
    } else if constexpr (MODE == EVX_OUT_RK4_FIRST) {
      out[i] = b + c * r;
      acc_out[i] = r;
    } else if constexpr (MODE == EVX_OUT_RK4_MID) {
      out[i] = b + c * r;
      acc_out[i] = a + T(2) * r;
    } else {
      out[i] = b + c * (a + r);
    }
  }
  __device__ __forceinline__ void advance(int64_t plane) {
    out += plane;
    if constexpr (MODE == EVX_OUT_EULER) u += plane;
    if constexpr (MODE >= EVX_OUT_RK4_FIRST) base += plane;
    if constexpr (MODE >= EVX_OUT_RK4_MID) acc_in += plane;
    if constexpr (MODE == EVX_OUT_RK4_FIRST || MODE == EVX_OUT_RK4_MID) acc_out += plane;
  }
};

template <typename T, int MODE>
__device__ __forceinline__ XOut<T, MODE> x_out(const Epi& ep, const T* u, T* out, int64_t at) {
  const T* const b = ep.base ? static_cast<const T*>(ep.base) : u;
  return {out + at, u + at, b + at, static_cast<const T*>(ep.acc_in) + at, static_cast<T*>(ep.acc_out) + at,
          static_cast<T>(ep.coef)};
}

// Walks the planes x0 .. x1-1 with the views of three successive planes.  ROT:
// the views change roles (the loop written out three times) instead of being
// copied.  That saves the copies and costs code and registers, so it is for
// the kernels that are light enough: copied / changing roles at 256^3, us
// (MI355X): diffusion Euler float32 24.7 / 23.9, float64 47.4 / 44.4, two species
// Euler float64 114.9 / 113.7; but two species Euler float32 45.4 / 50.7,
// diffusion RK4 float32 205 / 240, two species RK4 574 / 888, Allen-Cahn Euler
// 50.0 / 52.9 and RK4 242 / 297.
template <bool ROT, typename V, typename F>
__device__ __forceinline__ void x_march(int64_t x0, int64_t x1, V& a, V& b, V& c, F&& step) {
  if constexpr (ROT) {
    for (int64_t x = x0;;) {
      step(a, b, c, x);
      if (++x == x1) break;
      step(b, c, a, x);
      if (++x == x1) break;
      step(c, a, b, x);
      if (++x == x1) break;
    }
  } else {
    for (int64_t x = x0; x < x1; ++x) {
      step(a, b, c, x);
      a = b;
      b = c;
    }
  }
}

// ---------------------------------------------------------------------------
// Reaction-diffusion (f == 0): r = D * laplace(pad_bc(u))
// (problem_definition.py:226-229, fd_stencils.py:62-75)
// ---------------------------------------------------------------------------
template <typename T, int MODE, bool FLAT>
__global__ __launch_bounds__(NT) void rd_rhs_kernel(const T* __restrict__ u, T* __restrict__ out, Dims d, Bc bc,
                                                    Geo<T> g, T D, Epi ep, TileGrid tg) {
  using X = XTile<T, FLAT>;
  using Ld = XLoader<T, false, X>;
  using View = XView<T, 0, X>;
  constexpr int PY = X::PY, W = X::W;
  __shared__ T cs[2][X::PLANE];
  const int tid = threadIdx.x, tz = tid % X::TZ, r0 = tid / X::TZ * PY;
  const TileOrigin o = tile_origin<X::BY, X::TZ>(tg, d, xcd_tile(blockIdx.x, gridDim.x));
  const int64_t x0 = o.x0, x1 = o.x1, plane = d.ny * d.nz;
  const T* const uc = u + o.ch * d.vol();
  Ld ld;
  ld.init(o.y0, o.z0, d, bc, tid);
  const int at = (r0 + 1) * W + tz + 1;
  View va, vb, vc;
  typename Ld::Plane w;
  {  // warm-up: planes x0-1 .. x0+2 in flight together
    typename Ld::Plane a, b, c;
    ld.fetch(uc, x0 - 1, d, bc, a);
    ld.fetch(uc, x0, d, bc, b);
    ld.fetch(uc, x0 + 1, d, bc, c);
    if (x0 + 2 <= x1) ld.fetch(uc, x0 + 2, d, bc, w);
    ld.commit(cs[0], a, bc, tid);
    ld.commit(cs[1], b, bc, tid);
    __syncthreads();
    va.read(cs[0], at);
    vb.read(cs[1], at);
    __syncthreads();
    ld.commit(cs[0], c, bc, tid);
    __syncthreads();
  }
  const int64_t gz = o.z0 + tz, gy0 = o.y0 + r0;
  const uint32_t i0 = (uint32_t)(gy0 * d.nz + gz), nz = (uint32_t)d.nz;
  const int rows = gz < d.nz ? (int)(gy0 + PY <= d.ny ? PY : d.ny - gy0) : 0;  // valid rows (may be <= 0)
  XOut<T, MODE> eo = x_out<T, MODE>(ep, u, out, o.ch * d.vol() + x0 * plane);
  int s = 0;  // slot of plane x+1; the other takes plane x+2
  auto step = [&](const View& vm, const View& v0, View& v1, int64_t x) {
    T eb[PY], ea[PY];
    if constexpr (MODE >= EVX_OUT_RK4_FIRST) {
#pragma unroll
      for (int q = 0; q < PY; ++q)
        if (q < rows) eo.load(i0 + q * nz, eb[q], ea[q]);
    }
    v1.read(cs[s], at);
    if (x + 2 <= x1) ld.commit(cs[s ^ 1], w, bc, tid);
    if (x + 3 <= x1) ld.fetch(uc, x + 3, d, bc, w);
#pragma unroll
    for (int q = 0; q < PY; ++q) {
      const T c0 = v0.c[q + 1];
      const T lap = lap7(c0, v1.c[q + 1], vm.c[q + 1], v0.c[q + 2], v0.c[q], v0.p[q], v0.m[q], g);
      if constexpr (MODE == EVX_OUT_EULER) eb[q] = c0;  // the state itself, without a second load
      if (q < rows) eo.store(i0 + q * nz, D * lap, eb[q], ea[q]);
    }
    eo.advance(plane);
    s ^= 1;
    __syncthreads();
  };
  x_march<(MODE < EVX_OUT_RK4_FIRST)>(x0, x1, va, vb, vc, step);
}

// ---------------------------------------------------------------------------
// Two species with the Gray-Scott interaction a*b^2
// (problem_definition.py:612-633):
//   r_a = D_a*lap(a) - a*b^2 + F*(1 - a),   r_b = D_b*lap(b) + a*b^2 - k*b.
// One block streams both species; the tile grid has no channel dimension.
// ---------------------------------------------------------------------------
template <typename T>
struct GsCoef {
  T Da, Db, feed, kill;
};

template <typename T, int MODE, bool FLAT>
__global__ __launch_bounds__(NT) void gs_rhs_kernel(const T* __restrict__ u, T* __restrict__ out, Dims d, Bc bc,
                                                    Geo<T> g, GsCoef<T> k, Epi ep, TileGrid tg) {
  using X = XTile<T, FLAT>;
  using Ld = XLoader<T, false, X>;
  using View = XView<T, 0, X>;
  constexpr int PY = X::PY, W = X::W;
  __shared__ T cs[2][2][X::PLANE];
  const int tid = threadIdx.x, tz = tid % X::TZ, r0 = tid / X::TZ * PY;
  const TileOrigin o = tile_origin<X::BY, X::TZ>(tg, d, xcd_tile(blockIdx.x, gridDim.x));
  const int64_t x0 = o.x0, x1 = o.x1, plane = d.ny * d.nz, vol = d.vol();
  Ld ld;
  ld.init(o.y0, o.z0, d, bc, tid);
  const int at = (r0 + 1) * W + tz + 1;
  struct Views {
    View v[2];
  };
  Views va, vb, vc;
  typename Ld::Plane w[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const T* const uc = u + c * vol;
    typename Ld::Plane a, b;
    ld.fetch(uc, x0 - 1, d, bc, a);
    ld.fetch(uc, x0, d, bc, b);
    ld.fetch(uc, x0 + 1, d, bc, w[c]);
    ld.commit(cs[0][c], a, bc, tid);
    ld.commit(cs[1][c], b, bc, tid);
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    va.v[c].read(cs[0][c], at);
    vb.v[c].read(cs[1][c], at);
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    ld.commit(cs[0][c], w[c], bc, tid);
    if (x0 + 2 <= x1) ld.fetch(u + c * vol, x0 + 2, d, bc, w[c]);
  }
  __syncthreads();
  const int64_t gz = o.z0 + tz, gy0 = o.y0 + r0;
  const uint32_t i0 = (uint32_t)(gy0 * d.nz + gz), nz = (uint32_t)d.nz;
  const int rows = gz < d.nz ? (int)(gy0 + PY <= d.ny ? PY : d.ny - gy0) : 0;
  XOut<T, MODE> eo[2] = {x_out<T, MODE>(ep, u, out, x0 * plane), x_out<T, MODE>(ep, u, out, vol + x0 * plane)};
  int s = 0;
  auto step = [&](const Views& vm, const Views& v0, Views& v1, int64_t x) {
    T eb[2][PY], ea[2][PY];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      if constexpr (MODE >= EVX_OUT_RK4_FIRST) {
#pragma unroll
        for (int q = 0; q < PY; ++q)
          if (q < rows) eo[c].load(i0 + q * nz, eb[c][q], ea[c][q]);
      }
      v1.v[c].read(cs[s][c], at);
      if (x + 2 <= x1) ld.commit(cs[s ^ 1][c], w[c], bc, tid);
      if (x + 3 <= x1) ld.fetch(u + c * vol, x + 3, d, bc, w[c]);
    }
#pragma unroll
    for (int q = 0; q < PY; ++q) {
      const View&a0 = v0.v[0], &b0 = v0.v[1];
      const T av = a0.c[q + 1], bv = b0.c[q + 1];
      const T la = lap7(av, v1.v[0].c[q + 1], vm.v[0].c[q + 1], a0.c[q + 2], a0.c[q], a0.p[q], a0.m[q], g);
      const T lb = lap7(bv, v1.v[1].c[q + 1], vm.v[1].c[q + 1], b0.c[q + 2], b0.c[q], b0.p[q], b0.m[q], g);
      const T inter = av * (bv * bv);
      const T ra = (k.Da * la - inter) + k.feed * (T(1) - av);
      const T rb = (k.Db * lb + inter) - k.kill * bv;
      if constexpr (MODE == EVX_OUT_EULER) {
        eb[0][q] = av;
        eb[1][q] = bv;
      }
      if (q < rows) {
        eo[0].store(i0 + q * nz, ra, eb[0][q], ea[0][q]);
        eo[1].store(i0 + q * nz, rb, eb[1][q], ea[1][q]);
      }
    }
    eo[0].advance(plane);
    eo[1].advance(plane);
    s ^= 1;
    __syncthreads();
  };
  x_march<(MODE < EVX_OUT_RK4_FIRST && sizeof(T) == 8)>(x0, x1, va, vb, vc, step);
}

// ---------------------------------------------------------------------------
// Two-phase Allen-Cahn (problem_definition.py:440-447) with the 19-point
// normal Laplacian of fd_stencils.py:77-103.  Edge ghosts are used here, so
// the x-then-y-then-z composition of the ghost rules matters.
// ---------------------------------------------------------------------------
template <typename T>
struct AcCoef {
  T s18;       // 18/eps
  T eps;       // eps
  T curv;      // curvature
  T one_m_curv;// 1-curvature
  T gab, M, force;
  T s3;        // 3/eps
  // 1/eps where eps is a power of two (the default 2 is one), else 0: the product
  // is then the quotient, bit for bit, and spares one of the two IEEE divisions
  // a point.  256^3 RK4, us, eps = 2 / eps = 3 (MI355X): float32 242 / 260, with
  // walls in y 256 / 273, float64 512 / 526.
  T inv_eps;
};

template <typename T, int MODE, bool FLAT>
__global__ __launch_bounds__(NT) void ac_rhs_kernel(const T* __restrict__ u, T* __restrict__ out, Dims d, Bc bc,
                                                    Geo<T> g, AcCoef<T> k, Epi ep, TileGrid tg) {
  using X = XTile<T, FLAT>;
  using Ld = XLoader<T, true, X>;
  using View = XView<T, 1, X>;
  constexpr int PY = X::PY, W = X::W;
  __shared__ T cs[2][X::PLANE];
  const int tid = threadIdx.x, tz = tid % X::TZ, r0 = tid / X::TZ * PY;
  const TileOrigin o = tile_origin<X::BY, X::TZ>(tg, d, xcd_tile(blockIdx.x, gridDim.x));
  const int64_t x0 = o.x0, x1 = o.x1, plane = d.ny * d.nz;
  const T* const uc = u + o.ch * d.vol();
  Ld ld;
  ld.init(o.y0, o.z0, d, bc, tid);
  const int at = (r0 + 1) * W + tz + 1;
  View va, vb, vc;
  typename Ld::Plane w;
  {
    typename Ld::Plane a, b, c;
    ld.fetch(uc, x0 - 1, d, bc, a);
    ld.fetch(uc, x0, d, bc, b);
    ld.fetch(uc, x0 + 1, d, bc, c);
    if (x0 + 2 <= x1) ld.fetch(uc, x0 + 2, d, bc, w);
    ld.commit(cs[0], a, bc, tid);
    ld.commit(cs[1], b, bc, tid);
    __syncthreads();
    va.read(cs[0], at);
    vb.read(cs[1], at);
    __syncthreads();
    ld.commit(cs[0], c, bc, tid);
    __syncthreads();
  }
  const int64_t gz = o.z0 + tz, gy0 = o.y0 + r0;
  const uint32_t i0 = (uint32_t)(gy0 * d.nz + gz), nz = (uint32_t)d.nz;
  const int rows = gz < d.nz ? (int)(gy0 + PY <= d.ny ? PY : d.ny - gy0) : 0;
  XOut<T, MODE> eo = x_out<T, MODE>(ep, u, out, o.ch * d.vol() + x0 * plane);
  int s = 0;
  auto step = [&](const View& vm, const View& v0, View& v1, int64_t x) {
    T eb[PY], ea[PY];
    if constexpr (MODE != EVX_OUT_RHS) {  // EULER adds to the unclipped state
#pragma unroll
      for (int q = 0; q < PY; ++q)
        if (q < rows) eo.load(i0 + q * nz, eb[q], ea[q]);
    }
    v1.read(cs[s], at);
    if (x + 2 <= x1) ld.commit(cs[s ^ 1], w, bc, tid);
    if (x + 3 <= x1) ld.fetch(uc, x + 3, d, bc, w);
#pragma unroll
    for (int q = 0; q < PY; ++q) {
      const int j = q + 1;
      const T phi = v0.c[j];
      const T pot = ((k.s18 * phi) * (T(1) - phi)) * (T(1) - T(2) * phi);
      const T R = v1.c[j], L = vm.c[j], Tp = v0.c[j + 1], Bm = v0.c[j - 1], F = v0.p[j], K = v0.m[j];
      const T lap = k.curv * lap7(phi, R, L, Tp, Bm, F, K, g);
      const T cxy = ((v1.c[j + 1] + vm.c[j - 1]) - vm.c[j + 1]) - v1.c[j - 1];
      const T cxz = ((v1.p[j] + vm.m[j]) - vm.p[j]) - v1.m[j];
      const T cyz = ((v0.p[j + 1] + v0.m[j - 1]) - v0.p[j - 1]) - v0.m[j + 1];
      const T nlap = k.one_m_curv * normal_lap_of(phi, R, L, Tp, Bm, F, K, cxy, cxz, cyz, g);
      const T half = pot / T(2);
      const T bulk = k.inv_eps != T(0) ? half * k.inv_eps : half / k.eps;
      const T df = k.gab * ((lap + nlap) - bulk) + ((k.s3 * phi) * (T(1) - phi)) * k.force;
      if (q < rows) eo.store(i0 + q * nz, k.M * df, eb[q], ea[q]);
    }
    eo.advance(plane);
    s ^= 1;
    __syncthreads();
  };
  x_march<false>(x0, x1, va, vb, vc, step);
}

// ---------------------------------------------------------------------------
// launches
// ---------------------------------------------------------------------------
template <typename K>
int64_t x_resident(K kernel) {
  int dev = 0, cus = 0, per = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, NT, 0) != hipSuccess || per < 1 || cus < 1)
    return 1024;
  return (int64_t)per * cus;
}

// Launches KERNEL<T, mode, tile> for the epilogue's mode; the resident round is
// queried once per instance (all devices of a process are taken to be alike).
#define EVX_X_LAUNCH(KERNEL, CHANNELS, WHAT, ...)                                                        \
  switch (ep.mode) {                                                                                     \
    EVX_X_CASE(KERNEL, EVX_OUT_RHS, CHANNELS, __VA_ARGS__)                                               \
    EVX_X_CASE(KERNEL, EVX_OUT_EULER, CHANNELS, __VA_ARGS__)                                             \
    EVX_X_CASE(KERNEL, EVX_OUT_RK4_FIRST, CHANNELS, __VA_ARGS__)                                         \
    EVX_X_CASE(KERNEL, EVX_OUT_RK4_MID, CHANNELS, __VA_ARGS__)                                           \
    EVX_X_CASE(KERNEL, EVX_OUT_RK4_LAST, CHANNELS, __VA_ARGS__)                                          \
  }                                                                                                      \
  return check_launch(WHAT);
#define EVX_X_CASE(KERNEL, MODE, CHANNELS, ...)                                                          \
  case MODE:                                                                                             \
    if (flat_tiles<T>(d)) {                                                                              \
      EVX_X_ONE(KERNEL, MODE, sizeof(T) == 8, CHANNELS, __VA_ARGS__)                                     \
    } else {                                                                                             \
      EVX_X_ONE(KERNEL, MODE, false, CHANNELS, __VA_ARGS__)                                              \
    }                                                                                                    \
    break;
#define EVX_X_ONE(KERNEL, MODE, FLAT, CHANNELS, ...)                                                     \
  static const int64_t resident = x_resident(KERNEL<T, MODE, FLAT>);                                     \
  const unsigned blocks = x_tiles<XTile<T, FLAT>>(d, CHANNELS, resident, &tg);                           \
  hipLaunchKernelGGL((KERNEL<T, MODE, FLAT>), dim3(blocks), dim3(NT), 0, s, static_cast<const T*>(u),    \
                     static_cast<T*>(out), d, bc, make_geo<T>(g), __VA_ARGS__, ep, tg);

template <typename T>
int launch_rd_t(const void* u, void* out, const Dims& d, const Bc& bc, const evx_grid* g, double D, const Epi& ep,
                hipStream_t s) {
  TileGrid tg;
  EVX_X_LAUNCH(rd_rhs_kernel, d.c, "rd_rhs_kernel", static_cast<T>(D))
}

template <typename T>
int launch_gs_t(const void* u, void* out, const Dims& dims, const Bc& bc, const evx_grid* g, double Da, double Db,
                double feed, double kill, const Epi& ep, hipStream_t s) {
  TileGrid tg;
  Dims d = dims;
  d.c = 1;  // one block covers both species of its tile
  const GsCoef<T> k{static_cast<T>(Da), static_cast<T>(Db), static_cast<T>(feed), static_cast<T>(kill)};
  EVX_X_LAUNCH(gs_rhs_kernel, 1, "gs_rhs_kernel", k)
}

template <typename T>
int launch_ac_t(const void* u, void* out, const Dims& d, const Bc& bc, const evx_grid* g, double eps, double gab,
                double M, double force, double curv, const Epi& ep, hipStream_t s) {
  TileGrid tg;
  const T e = static_cast<T>(eps);
  int ex = 0;
  // x / 2^n is x * 2^-n exactly
  const bool pow2 = std::isfinite(e) && std::frexp(std::fabs(e), &ex) == T(0.5) && ex > -100 && ex < 100;
  const AcCoef<T> k{static_cast<T>(18.0 / eps), e, static_cast<T>(curv), static_cast<T>(1.0 - curv),
                    static_cast<T>(gab), static_cast<T>(M), static_cast<T>(force), static_cast<T>(3.0 / eps),
                    pow2 ? T(1) / e : T(0)};
  EVX_X_LAUNCH(ac_rhs_kernel, d.c, "ac_rhs_kernel", k)
}

}  // namespace

int launch_rd(int32_t dtype, const void* u, void* out, const Dims& d, const Bc& bc, const evx_grid* g, double D,
              const Epi& ep, hipStream_t s) {
  return dtype == EVX_F32 ? launch_rd_t<float>(u, out, d, bc, g, D, ep, s)
                          : launch_rd_t<double>(u, out, d, bc, g, D, ep, s);
}

int launch_gs(int32_t dtype, const void* u, void* out, const Dims& d, const Bc& bc, const evx_grid* g, double Da,
              double Db, double feed, double kill, const Epi& ep, hipStream_t s) {
  return dtype == EVX_F32 ? launch_gs_t<float>(u, out, d, bc, g, Da, Db, feed, kill, ep, s)
                          : launch_gs_t<double>(u, out, d, bc, g, Da, Db, feed, kill, ep, s);
}

int launch_ac(int32_t dtype, const void* u, void* out, const Dims& d, const Bc& bc, const evx_grid* g, double eps,
              double gab, double M, double force, double curv, const Epi& ep, hipStream_t s) {
  return dtype == EVX_F32 ? launch_ac_t<float>(u, out, d, bc, g, eps, gab, M, force, curv, ep, s)
                          : launch_ac_t<double>(u, out, d, bc, g, eps, gab, M, force, curv, ep, s);
}

}  // namespace evx
