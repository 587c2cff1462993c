// Tile machinery of the 2.5-D streaming stencils and the Cahn-Hilliard
// right-hand-side tile body, shared by the one-grid kernels and the batched
// (many-grid) kernels.
#pragma once
#include "evx_ch_math.hpp"
#include "evx_common.hpp"
#include "evx_fft_engine.hpp"

#include <type_traits>

namespace evx {

constexpr int BZ = 64;   // threads (and tile width) along z
constexpr int NTY = 4;   // thread rows along y
constexpr int NT = BZ * NTY;

template <typename T>
struct TileCfg;
template <>
struct TileCfg<float> { static constexpr int PY = 4; };   // BY = 16
template <>
struct TileCfg<double> { static constexpr int PY = 2; };  // BY = 8

struct Epi {
  int mode;
  double coef;
  const void* base;
  const void* acc_in;
  void* acc_out;
};

// Writes the fused output for right-hand side value r at flat index i.
template <typename T>
__device__ __forceinline__ void epilogue(const Epi& ep, const T* __restrict__ u,
                                         T* __restrict__ out, int64_t i, T r) {
#pragma clang fp contract(off)
  const T c = static_cast<T>(ep.coef);
  switch (ep.mode) {
    case EVX_OUT_RHS:
      out[i] = r;
      break;
    case EVX_OUT_EULER:
      out[i] = u[i] + c * r;
      break;
    case EVX_OUT_RK4_FIRST: {
      const T* b = ep.base ? static_cast<const T*>(ep.base) : u;
      out[i] = b[i] + c * r;
      static_cast<T*>(ep.acc_out)[i] = r;
      break;
    }
    case EVX_OUT_RK4_MID: {
      const T* b = ep.base ? static_cast<const T*>(ep.base) : u;
      const T a = static_cast<const T*>(ep.acc_in)[i];
      out[i] = b[i] + c * r;
      static_cast<T*>(ep.acc_out)[i] = a + T(2) * r;
      break;
    }
    default: {  // EVX_OUT_RK4_LAST
      const T* b = ep.base ? static_cast<const T*>(ep.base) : u;
      const T a = static_cast<const T*>(ep.acc_in)[i];
      out[i] = b[i] + c * (a + r);
      break;
    }
  }
}

template <typename T>
__host__ Geo<T> make_geo(const evx_grid* g) {
  return make_geo_from<T>(g->div_dx, g->div_dx2);
}

// Register-staged loader of one x-plane tile [y0-H, y0+BY+H) x [z0-H, z0+BZ+H).
// init() resolves, once per block, the y/z part of every element this thread
// loads: periodic axes wrap, non-periodic ones clamp and remember the ghost
// rule.  fetch() then only resolves the (uniform) x index of the plane and
// issues one load per element; commit() applies clip and the ghost rules and
// writes the element to LDS slot tid + k*NT of the plane.  (The multiphase kernel
// takes the offsets and flags of init() alone.)
template <typename T, int H, int ROWS, int W, bool CLIP>
struct PlaneLoader {
  static constexpr int NPT = (ROWS * W + NT - 1) / NT;
  int off[NPT];      // in-plane offset y*nz + z of the source point, -1 if unused
  uint8_t yzf[NPT];  // y/z ghost flags: 4/8 = y low/high, 16/32 = z low/high
  T v[NPT];
  uint8_t xf;        // x ghost flag of the fetched plane: 1 = low, 2 = high

  __device__ __forceinline__ void init(int64_t y0, int64_t z0, const Dims& d, const Bc& bc, int tid) {
#pragma unroll
    for (int k = 0; k < NPT; ++k) {
      const int i = tid + k * NT;
      off[k] = -1;
      yzf[k] = 0;
      if (i < ROWS * W) {
        int64_t gy = y0 - H + i / W, gz = z0 - H + i % W;
        uint8_t f = 0;
        if (gy < 0 || gy >= d.ny) {
          if (bc.kind[1] == EVX_BC_PERIODIC) gy = wrap_near(gy, d.ny);
          else { f |= gy < 0 ? 4 : 8; gy = gy < 0 ? 0 : d.ny - 1; }
        }
        if (gz < 0 || gz >= d.nz) {
          if (bc.kind[2] == EVX_BC_PERIODIC) gz = wrap_near(gz, d.nz);
          else { f |= gz < 0 ? 16 : 32; gz = gz < 0 ? 0 : d.nz - 1; }
        }
        off[k] = (int)(gy * d.nz + gz);
        yzf[k] = f;
      }
    }
  }

  __device__ __forceinline__ void fetch(const T* __restrict__ uc, int64_t xg, const Dims& d, const Bc& bc) {
    xf = 0;
    if (xg < 0 || xg >= d.nx) {
      if (bc.kind[0] == EVX_BC_PERIODIC) xg = wrap_near(xg, d.nx);
      else { xf = xg < 0 ? 1 : 2; xg = xg < 0 ? 0 : d.nx - 1; }
    }
    const T* pl = uc + xg * (d.ny * d.nz);
#pragma unroll
    for (int k = 0; k < NPT; ++k)
      if (off[k] >= 0) v[k] = pl[off[k]];
  }

  __device__ __forceinline__ void commit(T* flat, const Bc& bc, int tid) const {
#pragma unroll
    for (int k = 0; k < NPT; ++k) {
      if (off[k] >= 0) {
        T x = CLIP ? clip01(v[k]) : v[k];
        const int f = xf | yzf[k];
        if (f) {
          const int8_t o[3] = {(int8_t)((f & 1) ? -1 : (f & 2) ? 1 : 0), (int8_t)((f & 4) ? -1 : (f & 8) ? 1 : 0),
                               (int8_t)((f & 16) ? -1 : (f & 32) ? 1 : 0)};
          x = apply_rules(x, o, bc);
        }
        flat[tid + k * NT] = x;
      }
    }
  }
};

// Source points of the fully periodic tiles (the semi-implicit path): every
// coordinate wraps, so there are no ghost rules.  They are kept as 32-bit byte
// offsets from the plane base, which lets the loads use a scalar base address
// plus a 32-bit vector offset (no 64-bit address arithmetic per element).
// Requires ny*nz*sizeof(T) < 2^32.
template <typename T, int H, int ROWS, int W, bool CLIP>
struct PeriodicLoader {
  static constexpr int NPT = (ROWS * W + NT - 1) / NT;
  uint32_t boff[NPT];
  bool last_ok;  // whether this thread's last element lies in the tile

  // Byte offset in its x-plane of the tile point this thread loads as
  // element k (clamped to the tile's last point past the end).
  __host__ __device__ static uint32_t src_byte(int tid, int k, int64_t y0, int64_t z0, const Dims& d) {
    const int i = tid + k * NT < ROWS * W - 1 ? tid + k * NT : ROWS * W - 1;
    const int64_t gy = wrap_near(y0 - H + i / W, d.ny), gz = wrap_near(z0 - H + i % W, d.nz);
    return static_cast<uint32_t>((gy * d.nz + gz) * (int64_t)sizeof(T));
  }

  __device__ __forceinline__ void init(int64_t y0, int64_t z0, const Dims& d, int tid) {
    last_ok = tid + (NPT - 1) * NT < ROWS * W;
#pragma unroll
    for (int k = 0; k < NPT; ++k) boff[k] = src_byte(tid, k, y0, z0, d);
  }

  __device__ __forceinline__ bool valid(int k) const { return k < NPT - 1 || last_ok; }
};

// Ring slot of a plane at small relative index rel >= -3 (32-bit, constant modulus).
template <int NS>
__device__ __forceinline__ int ring(int64_t rel) { return (int)((unsigned)((int)rel + 3 * NS) % NS); }

// Flat launch: tiles ordered z-tile fastest, then y-tile, then x-chunk and
// channel; xcd_tile() gives each XCD a contiguous range so y/z halos of
// neighbouring tiles are shared through one L2.
struct TileGrid {
  int ntz, nty, nxc, xc;
};

struct TileOrigin {
  int64_t z0, y0, x0, x1, ch;
};

template <int BY, int TZ = BZ>
__host__ __device__ __forceinline__ TileOrigin tile_origin(const TileGrid& tg, const Dims& d, unsigned t) {
  TileOrigin o;
  o.z0 = (int64_t)(t % tg.ntz) * TZ;
  t /= tg.ntz;
  o.y0 = (int64_t)(t % tg.nty) * BY;
  t /= tg.nty;
  o.x0 = (int64_t)(t % tg.nxc) * tg.xc;
  o.ch = t / tg.nxc;
  o.x1 = o.x0 + (int64_t)tg.xc < d.nx ? o.x0 + (int64_t)tg.xc : d.nx;
  return o;
}

__host__ inline int pick_xchunk(const Dims& d, int64_t tiles_yz, int64_t target = 2048) {
  // About `target` blocks (a few per CU of the 256), but at least 4 planes
  // per block so the warm-up planes stay a bounded fraction of the work.
  // The minimum only binds for grids of a few tens of MB, which the
  // last-level cache holds; there a lower minimum means more blocks and
  // shorter per-block chains (100^3 float64 CH step: 0.0743 ms/step with at
  // least 8 planes, 0.0712 with 4, 0.0708 with 2; MI355X).
  int64_t chunks = (target + tiles_yz * d.c - 1) / (tiles_yz * d.c);
  if (chunks < 1) chunks = 1;
  int64_t xc = (d.nx + chunks - 1) / chunks;
  if (xc < 4) xc = 4;
  if (xc > d.nx) xc = d.nx;
  return (int)xc;
}

// Tile grid of a streaming stencil launch of about `target` blocks; returns
// the block count (tiles over z, y, x-chunks and channels).
template <typename T>
__host__ inline unsigned stencil_tiles(const Dims& d, TileGrid* tg, int64_t target) {
  constexpr int BY = NTY * TileCfg<T>::PY;
  const int64_t ty = (d.ny + BY - 1) / BY, tzn = (d.nz + BZ - 1) / BZ;
  tg->xc = pick_xchunk(d, ty * tzn, target);
  const int64_t nxc = (d.nx + tg->xc - 1) / tg->xc;
  tg->ntz = (int)tzn;
  tg->nty = (int)ty;
  tg->nxc = (int)nxc;
  return (unsigned)(tzn * ty * nxc * d.c);
}

// ---------------------------------------------------------------------------
// Cahn-Hilliard (problem_definition.py:328-371):
//   c = clip(u,0,1); mu = ((18/eps*c)*(1-c))*(1-2c) - (2eps)*lap(cB)
//   r = D * sum_axes grad_face( (cf*(1-cf)) * grad_face(muB) )
// mu lives in an LDS plane ring with a one-voxel (y,z) halo, c in one with a
// two-voxel halo.  mu ghosts (non-periodic faces) are the BC rule applied to
// mu at the adjacent interior voxel, as pad_bc(mu) does.
// ---------------------------------------------------------------------------
// Thread (ty, tz) owns PY consecutive rows r0 = ty*PY .. r0+PY-1 of column tz.
// Per output plane it evaluates mu for its own rows (sharing the column loads
// between rows) while threads 0..H-1 evaluate the one-voxel mu halo with the
// full ghost logic; the flux through the face between two own rows is
// computed once, and the flux through the x face x+1/2 is carried in a
// register to the next plane.  The c ring holds 4 planes (x-1..x+2, the
// slot of x-1 being refilled with x+3 during the output of plane x), the mu
// ring 2 (x, x+1); plane x+4 is fetched into registers during the output of
// plane x.
template <typename T>
struct ChTile {
  static constexpr int PY = TileCfg<T>::PY, BY = NTY * PY;
  static constexpr int CW = BZ + 4, CR = BY + 4, NC = 4;
  static constexpr int MW = BZ + 2, MR = BY + 2, NM = 2;
  static constexpr size_t LDS_BYTES = sizeof(T) * (NC * CR * CW + NM * MR * MW);
};

// One (y,z) tile x x-chunk of the CH right-hand side.  tid = flat thread index
// in a 256-thread block, tile = flat tile index (see tile_origin), smem =
// ChTile<T>::LDS_BYTES of LDS.
template <typename T>
__device__ __forceinline__ void ch_rhs_tile(const T* __restrict__ u, T* __restrict__ out, const Dims& d,
                                            const Bc& bc, const Geo<T>& g, ChCoef<T> k, const Epi& ep,
                                            const TileGrid& tg, unsigned tile, int tid, unsigned char* smem) {
#pragma clang fp contract(off)
  using Op = Ops<true>;
  using TC = ChTile<T>;
  constexpr int PY = TC::PY, BY = TC::BY;
  constexpr int CW = TC::CW, CR = TC::CR, NC = TC::NC;
  constexpr int MW = TC::MW, MR = TC::MR, NM = TC::NM;
  constexpr int HALO = 2 * MW + 2 * BY;  // mu halo points: rows -1, BY and columns -1, BZ
  T(*cs)[CR][CW] = reinterpret_cast<T(*)[CR][CW]>(smem);
  T(*ms)[MR][MW] = reinterpret_cast<T(*)[MR][MW]>(smem + sizeof(T) * NC * CR * CW);
  const int tz = tid % BZ, ty = tid / BZ;
  const TileOrigin o = tile_origin<BY>(tg, d, tile);
  const int64_t z0 = o.z0, y0 = o.y0, x0 = o.x0, x1 = o.x1;
  const T* uc = u + o.ch * d.vol();
  T* oc = out + o.ch * d.vol();
  const bool xper = bc.kind[0] == EVX_BC_PERIODIC;
  const bool yper = bc.kind[1] == EVX_BC_PERIODIC, zper = bc.kind[2] == EVX_BC_PERIODIC;
  const int r0 = ty * PY;
  const int64_t gz = z0 + tz;

  // mu at tile point (yy, zz) of x-plane xm with every ghost rule applied.
  auto mu_general = [&](int64_t xm, int yy, int zz) -> T {
    int8_t oo[3] = {0, 0, 0};
    int64_t xs = xm;
    if (!xper && xm < 0) { oo[0] = -1; xs = 0; }
    if (!xper && xm >= d.nx) { oo[0] = 1; xs = d.nx - 1; }
    const T(*Cm)[CW] = cs[ring<NC>(xs - 1 - x0 + 2)];
    const T(*C0)[CW] = cs[ring<NC>(xs - x0 + 2)];
    const T(*Cp)[CW] = cs[ring<NC>(xs + 1 - x0 + 2)];
    const int64_t gy = y0 + yy, gzz = z0 + zz;
    int a = yy + 2, b = zz + 2;
    if (!yper && (gy < 0 || gy >= d.ny)) {
      oo[1] = gy < 0 ? -1 : 1;
      a += gy < 0 ? 1 : -1;
    }
    if (!zper && (gzz < 0 || gzz >= d.nz)) {
      oo[2] = gzz < 0 ? -1 : 1;
      b += gzz < 0 ? 1 : -1;
    }
    T m = Op::mu(C0[a][b], Cp[a][b], Cm[a][b], C0[a + 1][b], C0[a - 1][b], C0[a][b + 1], C0[a][b - 1], g, k);
    if (oo[0] | oo[1] | oo[2]) m = apply_rules(m, oo, bc);
    return m;
  };

  // Tiles that cut a non-periodic y/z boundary evaluate every mu point with
  // the ghost logic; all other tiles only their halo.
  const bool tile_partial = (!yper && y0 + BY > d.ny) || (!zper && z0 + BZ > d.nz);
  // This thread's point of the one-voxel mu halo (rows -1, BY and columns -1,
  // BZ, corners excluded), resolved once: c coordinates (ha, hb) of the source
  // point and its y/z ghost flags.
  constexpr int NHALO = 2 * MW + 2 * BY - 4;
  int hy = 0, hz = 0, ha = 0, hb = 0;
  int8_t hoy = 0, hoz = 0;
  if (tid < NHALO) {
    int h = tid;
    if (h < 2 * (MW - 2)) {
      hy = h < MW - 2 ? -1 : BY;
      hz = h < MW - 2 ? h : h - (MW - 2);
    } else {
      h -= 2 * (MW - 2);
      hy = h % BY;
      hz = h < BY ? -1 : BZ;
    }
    ha = hy + 2;
    hb = hz + 2;
    const int64_t gy = y0 + hy, gzz = z0 + hz;
    if (!yper && (gy < 0 || gy >= d.ny)) { hoy = gy < 0 ? -1 : 1; ha += gy < 0 ? 1 : -1; }
    if (!zper && (gzz < 0 || gzz >= d.nz)) { hoz = gzz < 0 ? -1 : 1; hb += gzz < 0 ? 1 : -1; }
  }

  auto compute_mu = [&](int64_t xm) {
    T(*M)[MW] = ms[ring<NM>(xm - x0 + 1)];
    const bool general = tile_partial || (!xper && (xm < 0 || xm >= d.nx));
    if (!general) {
      const T(*Cm)[CW] = cs[ring<NC>(xm - 1 - x0 + 2)];
      const T(*C0)[CW] = cs[ring<NC>(xm - x0 + 2)];
      const T(*Cp)[CW] = cs[ring<NC>(xm + 1 - x0 + 2)];
      T col[PY + 2];
#pragma unroll
      for (int j = 0; j < PY + 2; ++j) col[j] = C0[r0 + j + 1][tz + 2];
#pragma unroll
      for (int q = 0; q < PY; ++q) {
        const int a = r0 + q + 2, b = tz + 2;
        M[r0 + q + 1][tz + 1] =
            Op::mu(col[q + 1], Cp[a][b], Cm[a][b], col[q + 2], col[q], C0[a][b + 1], C0[a][b - 1], g, k);
      }
      if (tid < NHALO) {
        T m = Op::mu(C0[ha][hb], Cp[ha][hb], Cm[ha][hb], C0[ha + 1][hb], C0[ha - 1][hb], C0[ha][hb + 1],
                     C0[ha][hb - 1], g, k);
        if (hoy | hoz) {
          const int8_t oo[3] = {0, hoy, hoz};
          m = apply_rules(m, oo, bc);
        }
        M[hy + 1][hz + 1] = m;
      }
    } else {
      for (int p = tid; p < BY * BZ + NHALO; p += NT) {
        int yy, zz;
        if (p < BY * BZ) {
          yy = p / BZ;
          zz = p % BZ;
        } else {
          int h = p - BY * BZ;
          if (h < 2 * (MW - 2)) {
            yy = h < MW - 2 ? -1 : BY;
            zz = h < MW - 2 ? h : h - (MW - 2);
          } else {
            h -= 2 * (MW - 2);
            yy = h % BY;
            zz = h < BY ? -1 : BZ;
          }
        }
        M[yy + 1][zz + 1] = mu_general(xm, yy, zz);
      }
    }
  };

  PlaneLoader<T, 2, CR, CW, true> pl;
  auto pl_fetch = [&](int64_t xg) { pl.fetch(uc, xg, d, bc); };
  auto pl_commit = [&](int slot) { pl.commit(&cs[slot][0][0], bc, tid); };
  pl.init(y0, z0, d, bc, tid);
  const int b = tz + 2, bm = tz + 1;
  // Warm-up: planes x0-2 .. x0+1, mu(x0-1) and mu(x0), and the flux through
  // the x face x0-1/2 (afterwards carried in registers, so neither c(x-1)
  // nor mu(x-1) is read again and the rings hold 4 c planes and 2 mu planes).
  for (int64_t xg = x0 - 2; xg <= x0 + 1; ++xg) {
    pl_fetch(xg);
    pl_commit(ring<NC>(xg - x0 + 2));
  }
  if (x0 + 2 <= x1 + 1) pl_fetch(x0 + 2);
  __syncthreads();
  compute_mu(x0 - 1);
  compute_mu(x0);
  __syncthreads();
  T carry[PY];  // flux through the x face x-1/2 of each own row
  {
    const T(*Cm)[CW] = cs[ring<NC>(-1 + 2)];
    const T(*C0)[CW] = cs[ring<NC>(0 + 2)];
    const T(*Mm)[MW] = ms[ring<NM>(-1 + 1)];
    const T(*M0)[MW] = ms[ring<NM>(0 + 1)];
#pragma unroll
    for (int q = 0; q < PY; ++q)
      carry[q] = Op::flux(Cm[r0 + q + 2][b], C0[r0 + q + 2][b], Mm[r0 + q + 1][bm], M0[r0 + q + 1][bm], g.idx);
  }
  // plane x0+2 goes to the slot of x0-2 (last read by mu(x0-1))
  if (x0 + 2 <= x1 + 1) pl_commit(ring<NC>(4));
  if (x0 + 3 <= x1 + 1) pl_fetch(x0 + 3);
  __syncthreads();  // mu(x0+1) below reuses the slot of mu(x0-1) read above
  const int64_t plane = d.ny * d.nz;
  for (int64_t x = x0; x < x1; ++x) {
    // mu(x+1) from c(x), c(x+1), c(x+2), into the slot of mu(x-1)
    compute_mu(x + 1);
    __syncthreads();
    const T(*C0)[CW] = cs[ring<NC>(x - x0 + 2)];
    const T(*Cp)[CW] = cs[ring<NC>(x + 1 - x0 + 2)];
    const T(*M0)[MW] = ms[ring<NM>(x - x0 + 1)];
    const T(*Mp)[MW] = ms[ring<NM>(x + 1 - x0 + 1)];
    T cc[PY + 2], mc[PY + 2], fy[PY + 1];
#pragma unroll
    for (int j = 0; j < PY + 2; ++j) {
      cc[j] = C0[r0 + j + 1][b];
      mc[j] = M0[r0 + j][bm];
    }
#pragma unroll
    for (int j = 0; j <= PY; ++j) fy[j] = Op::flux(cc[j], cc[j + 1], mc[j], mc[j + 1], g.idy);
#pragma unroll
    for (int q = 0; q < PY; ++q) {
      const int a = r0 + q + 2, am = r0 + q + 1;
      const T c0 = cc[q + 1], m0 = mc[q + 1];
      const T fxp = Op::flux(c0, Cp[a][b], m0, Mp[am][bm], g.idx);
      const T fzm = Op::flux(C0[a][b - 1], c0, M0[am][bm - 1], m0, g.idz);
      const T fzp = Op::flux(c0, C0[a][b + 1], m0, M0[am][bm + 1], g.idz);
      const T r = Op::div(carry[q], fxp, fy[q], fy[q + 1], fzm, fzp, g, k.D);
      carry[q] = fxp;
      const int64_t gy = y0 + r0 + q;
      if (gy < d.ny && gz < d.nz) epilogue(ep, uc, oc, x * plane + gy * d.nz + gz, r);
    }
    // plane x+3 (fetched one iteration ago) goes to the slot of c(x-1), which
    // neither the output above nor mu(x+1) reads; it feeds mu(x+2)
    if (x + 3 <= x1 + 1) pl_commit(ring<NC>(x + 3 - x0 + 2));
    if (x + 4 <= x1 + 1) pl_fetch(x + 4);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// The same right-hand side on a fully periodic grid, written plainly (the
// semi-implicit path): no ghost logic, contracted algebra.  A block owns a
// (BY x TZ) tile of (y, z) and an x-chunk; thread (ty, tz) owns PY rows of one
// column and keeps c(x), c(x+1), c(x+2), mu(x), mu(x+1) and the flux through
// the face x-1/2 of its points in registers, so only y and z neighbours come
// from LDS (a ring of four c planes and two mu planes) and a plane takes one
// barrier: plane x+3 is written to the fourth slot and mu(x+1) to the second
// while c(x), c(x+1), c(x+2) and mu(x) are read.
//
// The planes of the warm-up are fetched together (one memory latency instead
// of one per plane); SHORT, for chunks of at most CH_SHORT planes, fetches
// every plane of the chunk that way.
//
// Bound by vector issue on large grids (64 vector instructions per point and
// plane with 16 x 32 tiles, 57 with 16 x 64) and by the chain of planes on
// small ones.  MI355X, us, before (two barriers a plane, neighbours of both
// fields from LDS) -> now: 32^3 float32 12.4 -> 5.2, 100^3 float64 13.8 -> 11,
// 4 x 96^3 float64 36 -> 21, 300x270x350 float32 92 -> 62, 400^3 float64
// 394 -> 267, 512^3 float32 282 -> 262.
// ---------------------------------------------------------------------------
constexpr int CH_SHORT = 4;

template <typename T, int TZ_, int PY_>
struct ChPer {
  static constexpr int TZ = TZ_, NR = NT / TZ;  // tile width, thread rows
  static constexpr int PY = PY_, BY = NR * PY;
  static constexpr int CW = TZ + 4, CR = BY + 4, NC = 4;
  static constexpr int MW = TZ + 2, MR = BY + 2, NM = 2;
  static constexpr int NHALO = 2 * TZ + 2 * BY;  // mu points on rows -1, BY and columns -1, TZ
  static constexpr size_t LDS_BYTES = sizeof(T) * (NC * CR * CW + NM * MR * MW);
  static_assert(NHALO <= NT, "one mu halo point per thread");
};

constexpr int SLAB_XCHUNK = 16;  // planes a chunk of slab launches

// Tile of the periodic float32 right-hand side: 16 x 64 points on large grids
// whose z length wastes no more of a 64-wide tile than of a 32-wide one, else
// 16 x 32 (MI355X, us, 64 / 32 wide: 512^3 265 / 305, 16 x 128^3 81 / 86,
// 256^3 36.4 / 36.4, 200^3 30.2 / 27.1, 300x270x350 64.7 / 63.7, 32^3 9.0 / 7.0).
// Float64 tiles are 16 x 32 (400^3 285 / 257, 4 x 96^3 26 / 22).
__host__ inline bool ch_wide_tile(const Dims& d) {
  return (d.nz + 63) / 64 * 2 == (d.nz + 31) / 32 && d.c * d.vol() >= (int64_t(1) << 24);
}

// Tile grid of the periodic kernel with tile P over the whole field (xb < 0), or
// over the x-slab [xa, xb) of a one-channel field at tile-chunk granularity:
// the launch then starts at tile `base`.
template <typename P>
__host__ inline unsigned ch_periodic_grid(const Dims& d, int64_t resident, int64_t xa, int64_t xb, TileGrid* tg,
                                          unsigned* base) {
  tg->ntz = (int)((d.nz + P::TZ - 1) / P::TZ);
  tg->nty = (int)((d.ny + P::BY - 1) / P::BY);
  const int64_t per_chunk = (int64_t)tg->ntz * tg->nty;
  tg->xc = xb >= 0 ? SLAB_XCHUNK : (int)balanced_xchunk(d.nx, per_chunk * d.c, resident, 4);
  tg->nxc = (int)((d.nx + tg->xc - 1) / tg->xc);
  *base = 0;
  if (xb < 0) return (unsigned)(per_chunk * tg->nxc * d.c);
  const int64_t ca = xa / tg->xc, cb = (xb + tg->xc - 1) / tg->xc;
  *base = (unsigned)(ca * per_chunk);
  return (unsigned)((cb - ca) * per_chunk);
}

template <typename T, int TZ, int PYT, bool SHORT>
__device__ __forceinline__ void ch_periodic_tile(const T* __restrict__ u, T* __restrict__ out, const Dims& d,
                                                 const Geo<T>& g, ChCoef<T> k, const TileGrid& tg,
                                                 const double* __restrict__ chan, unsigned tile, int tid,
                                                 unsigned char* smem) {
  using P = ChPer<T, TZ, PYT>;
  using Op = Ops<false>;
  constexpr int PY = P::PY, BY = P::BY, CW = P::CW, MW = P::MW;
  constexpr int CS = P::CR * CW, MS = P::MR * MW;
  using Loader = PeriodicLoader<T, 2, P::CR, CW, true>;
  constexpr int NPT = Loader::NPT;
  T* const cs = reinterpret_cast<T*>(smem);
  T* const ms = cs + P::NC * CS;
  const int tz = tid % TZ, r0 = tid / TZ * PY;
  const TileOrigin o = tile_origin<BY, TZ>(tg, d, tile);
  const int64_t x0 = o.x0;
  const int nxp = (int)(o.x1 - x0);  // planes of the chunk
  const T* const uc = u + o.ch * d.vol();
  if (chan) {  // per-channel (eps, D), rounded as the host rounds the scalars
    const double e = chan[2 * o.ch], dd = chan[2 * o.ch + 1];
    k = ChCoef<T>{static_cast<T>(18.0 / e), static_cast<T>(2.0 * e), static_cast<T>(dd)};
  }
  const ChW<T> W = ch_weights(g, k);
  const int oc = (r0 + 2) * CW + tz + 2, om = (r0 + 1) * MW + tz + 1;
  // this thread's mu halo point: offset of its c point in a c plane and of itself in a mu plane
  int hc = 0, hm = 0;
  const bool halo = tid < P::NHALO;
  if (halo) {
    int y, z;
    if (tid < 2 * TZ) {
      y = tid < TZ ? -1 : BY;
      z = tid % TZ;
    } else {
      const int h = tid - 2 * TZ;
      y = h % BY;
      z = h < BY ? -1 : TZ;
    }
    hc = (y + 2) * CW + z + 2;
    hm = (y + 1) * MW + z + 1;
  }
  Loader pl;
  pl.init(o.y0, o.z0, d, tid);
  // fetch() loads the planes x0-2, x0-1, ... in turn: the wrapped index is
  // advanced by a compare (a modulo per plane is a 64-bit division)
  const int nx = (int)d.nx;
  int xw = (int)x0 - 2;
  while (xw < 0) xw += nx;
  auto fetch = [&](T(&v)[NPT]) {
    const char* p = reinterpret_cast<const char*>(uc + (int64_t)xw * (d.ny * d.nz));
#pragma unroll
    for (int q = 0; q < NPT; ++q)
      if (pl.valid(q)) v[q] = *reinterpret_cast<const T*>(p + pl.boff[q]);
    xw = xw + 1 == nx ? 0 : xw + 1;
  };
  auto commit = [&](int slot, const T(&v)[NPT]) {
    T* const c = cs + slot * CS;
#pragma unroll
    for (int q = 0; q < NPT; ++q)
      if (pl.valid(q)) c[tid + q * NT] = clip01(v[q]);
  };
  // mu of the own points of plane slot C with x neighbours xm, xp
  auto mu_own = [&](const T* C, const T(&c)[PY], const T(&xm)[PY], const T(&xp)[PY], T(&m)[PY]) {
    const T lo = C[oc - CW], hi = C[oc + PY * CW];
#pragma unroll
    for (int q = 0; q < PY; ++q)
      m[q] = mu_w(c[q], xp[q], xm[q], q + 1 < PY ? c[q + 1 < PY ? q + 1 : q] : hi, q > 0 ? c[q > 0 ? q - 1 : q] : lo,
                  C[oc + q * CW + 1], C[oc + q * CW - 1], W);
  };
  auto mu_halo = [&](const T* Cm, const T* C, const T* Cp, T* M) {
    if (halo)
      M[hm] = mu_w(C[hc], Cp[hc], Cm[hc], C[hc + CW], C[hc - CW], C[hc + 1], C[hc - 1], W);
  };

  // warm-up: planes x0-2 .. x0+3 (SHORT: to the chunk's last) in flight together
  constexpr int PRE = SHORT ? CH_SHORT + 4 : 6;
  T w[PRE][NPT];
#pragma unroll
  for (int p = 0; p < PRE; ++p)
    if (p < 5 || p <= nxp + 3) fetch(w[p]);
#pragma unroll
  for (int p = 0; p < 4; ++p) commit(p, w[p]);
  __syncthreads();
  T c0[PY], c1[PY], m0[PY], carry[PY];
  {
    T a[PY], b[PY], mp[PY];
#pragma unroll
    for (int q = 0; q < PY; ++q) {
      a[q] = cs[oc + q * CW];
      b[q] = cs[CS + oc + q * CW];
      c0[q] = cs[2 * CS + oc + q * CW];
      c1[q] = cs[3 * CS + oc + q * CW];
    }
    mu_own(cs + CS, b, a, c0, mp);
    mu_own(cs + 2 * CS, c0, b, c1, m0);
#pragma unroll
    for (int q = 0; q < PY; ++q) {
      ms[om + q * MW] = m0[q];
      carry[q] = Op::flux_q(T(1) - b[q], c0[q], mp[q], m0[q]);
    }
    mu_halo(cs + CS, cs + 2 * CS, cs + 3 * CS, ms);
  }
  __syncthreads();  // every read of plane x0-2 is done
  commit(0, w[4]);
  __syncthreads();

  const int64_t plane = d.ny * d.nz;
  const bool full = o.y0 + BY <= d.ny && o.z0 + TZ <= d.nz;
  const int64_t gz = o.z0 + tz;
  const uint32_t obyte = static_cast<uint32_t>(((o.y0 + r0) * d.nz + gz) * (int64_t)sizeof(T));
  const uint32_t orow = static_cast<uint32_t>(d.nz * (int64_t)sizeof(T));
  T* ox = out + o.ch * d.vol() + x0 * plane;
  // output plane x0 + i; c(x0+i+3) is in v on entry (if the chunk needs it)
  auto step = [&](int i, T(&v)[NPT]) {
    const T* const C0 = cs + ((i + 2) & 3) * CS;
    const T* const C1 = cs + ((i + 3) & 3) * CS;
    const T* const C2 = cs + (i & 3) * CS;
    const T* const M0 = ms + (i & 1) * MS;
    T* const M1 = ms + ((i + 1) & 1) * MS;
    if (i + 3 <= nxp + 1) commit((i + 1) & 3, v);
    if (!SHORT && i + 4 <= nxp + 1) fetch(v);
    T c2[PY], m1[PY];
#pragma unroll
    for (int q = 0; q < PY; ++q) c2[q] = C2[oc + q * CW];
    mu_own(C1, c1, c0, c2, m1);
#pragma unroll
    for (int q = 0; q < PY; ++q) M1[om + q * MW] = m1[q];
    mu_halo(C0, C1, C2, M1);
    T fy[PY + 1];
    {
      const T cl = C0[oc - CW], ch = C0[oc + PY * CW], ml = M0[om - MW], mh = M0[om + PY * MW];
      fy[0] = Op::flux_q(T(1) - cl, c0[0], ml, m0[0]);
#pragma unroll
      for (int q = 1; q < PY; ++q) fy[q] = Op::flux_q(T(1) - c0[q - 1], c0[q], m0[q - 1], m0[q]);
      fy[PY] = Op::flux_q(T(1) - c0[PY - 1], ch, m0[PY - 1], mh);
    }
#pragma unroll
    for (int q = 0; q < PY; ++q) {
      const T q0 = T(1) - c0[q];
      const T fxp = Op::flux_q(q0, c1[q], m0[q], m1[q]);
      const T fzm = Op::flux_q(q0, C0[oc + q * CW - 1], M0[om + q * MW - 1], m0[q]);
      const T fzp = Op::flux_q(q0, C0[oc + q * CW + 1], m0[q], M0[om + q * MW + 1]);
      const T r = div_w(carry[q], fxp, fy[q], fy[q + 1], fzm, fzp, W);
      carry[q] = fxp;
      if (full || (o.y0 + r0 + q < d.ny && gz < d.nz))
        *reinterpret_cast<T*>(reinterpret_cast<char*>(ox) + (obyte + q * orow)) = r;
    }
#pragma unroll
    for (int q = 0; q < PY; ++q) {
      c0[q] = c1[q];
      c1[q] = c2[q];
      m0[q] = m1[q];
    }
    ox += plane;
    __syncthreads();
  };
  if constexpr (SHORT) {
#pragma unroll
    for (int i = 0; i < CH_SHORT; ++i)
      if (i < nxp) step(i, w[i + 5 < PRE ? i + 5 : PRE - 1]);
  } else {
    for (int i = 0; i < nxp; ++i) step(i, w[5]);
  }
}

}  // namespace evx
