// Tiles and launches of the explicit right-hand sides (evx_explicit.hip) and the
// normal Laplacian they share with the padded operators.
#pragma once
#include "evx_stencil_tiles.hpp"

#include <cmath>

namespace evx {

// 19-point normal Laplacian (fd_stencils.py:77-103) from the point C, its x
// neighbours R, L, its y neighbours Tp, Bm, its z neighbours F, K and the
// mixed differences cxy, cxz, cyz of the twelve edge points.
template <typename T>
__device__ __forceinline__ T normal_lap_of(T C, T R, T L, T Tp, T Bm, T F, T K, T cxy, T cxz, T cyz,
                                           const Geo<T>& g) {
#pragma clang fp contract(off)
  const T gx = (T(0.5) * (R - L)) * g.idx;
  const T gy = (T(0.5) * (Tp - Bm)) * g.idy;
  const T gz = (T(0.5) * (F - K)) * g.idz;
  const T t1 = ((gx * gx) * ((R - T(2) * C) + L)) * g.idx2;
  const T t2 = ((gy * gy) * ((Tp - T(2) * C) + Bm)) * g.idy2;
  const T t3 = ((gz * gz) * ((F - T(2) * C) + K)) * g.idz2;
  const T t4 = ((((T(0.5) * gx) * gy) * cxy) * g.idx) * g.idy;
  const T t5 = ((((T(0.5) * gx) * gz) * cxz) * g.idx) * g.idz;
  const T t6 = ((((T(0.5) * gy) * gz) * cyz) * g.idy) * g.idz;
  const T num = ((((t1 + t2) + t3) + t4) + t5) + t6;
  T n2 = ((gx * gx) + (gy * gy)) + (gz * gz);
  if (n2 <= static_cast<T>(1e-7)) n2 = T(1);
  return num / n2;
}

// Tiles of 16 x 64 points in float32, 16 x 32 in float64, and for thin float64
// grids 8 x 64 (FLAT, see flat_tiles).
template <typename T, bool FLAT>
struct XTile {
  static constexpr int TZ = sizeof(T) == 4 || FLAT ? 64 : 32, PY = sizeof(T) == 4 ? 4 : 2;
  static constexpr int BY = NT / TZ * PY, W = TZ + 2, ROWS = BY + 2, PLANE = ROWS * W;
  static constexpr int NPT = (PLANE + NT - 1) / NT;

  // In-plane element that holds point i of the tile at (y0, z0) or of its halo
  // of one; flags: the ghost rules it takes, 4/8 = y low/high, 16/32 = z low/high.
  __host__ __device__ static uint32_t source(int i, int64_t y0, int64_t z0, const Dims& d, const Bc& bc,
                                             uint8_t* flags) {
    int64_t gy = y0 - 1 + i / W, gz = z0 - 1 + i % W;
    uint8_t g = 0;
    if (gy < 0 || gy >= d.ny) {
      if (bc.kind[1] == EVX_BC_PERIODIC) gy = wrap_near(gy, d.ny);
      else { g |= gy < 0 ? 4 : 8; gy = gy < 0 ? 0 : d.ny - 1; }
    }
    if (gz < 0 || gz >= d.nz) {
      if (bc.kind[2] == EVX_BC_PERIODIC) gz = wrap_near(gz, d.nz);
      else { g |= gz < 0 ? 16 : 32; gz = gz < 0 ? 0 : d.nz - 1; }
    }
    *flags = g;
    return (uint32_t)(gy * d.nz + gz);
  }
};

// Float64 tiles of 8 x 64 points for one, three or five groups of eight rows, of
// which 16 x 32 tiles leave a half, a quarter or a sixth of the threads
// without a point; more rows gain nothing (201 x 183 x 219 Allen-Cahn 47.4 us
// with 16 x 32, 51.8 with 8 x 64).  Up to 32 columns a 16 x 32 tile has no more
// idle threads than the other.  16 x 32 / 8 x 64, us (MI355X): diffusion Euler
// 3 x 1 x 100000 14.8 / 9.4, with walls 22.3 / 13.8, 500 x 8 x 500 11.7 / 9.2,
// 1302 x 24 x 64 with walls 13.8 / 10.4, 500 x 40 x 500 28.9 / 26.8;
// Allen-Cahn 2857 x 1 x 700 78.9 / 41.9; two species 2000 x 2 x 500 51.2 / 29.7.
template <typename T>
__host__ inline bool flat_tiles(const Dims& d) {
  return sizeof(T) == 8 && d.ny <= 40 && (d.ny + 7) / 8 % 2 == 1 && d.nz > 32;
}

// Tile grid of a launch over `channels` channels: chunks for whole resident
// rounds (balanced_xchunk), the warm-up counted as three planes.
template <typename X>
__host__ inline unsigned x_tiles(const Dims& d, int64_t channels, int64_t resident, TileGrid* tg) {
  tg->ntz = (int)((d.nz + X::TZ - 1) / X::TZ);
  tg->nty = (int)((d.ny + X::BY - 1) / X::BY);
  const int64_t per = (int64_t)tg->ntz * tg->nty * channels;
  tg->xc = (int)balanced_xchunk(d.nx, per, resident, 3);
  tg->nxc = (int)((d.nx + tg->xc - 1) / tg->xc);
  return (unsigned)(per * tg->nxc);
}

int launch_rd(int32_t dtype, const void* u, void* out, const Dims& d, const Bc& bc, const evx_grid* g, double D,
              const Epi& ep, hipStream_t s);
int launch_gs(int32_t dtype, const void* u, void* out, const Dims& d, const Bc& bc, const evx_grid* g, double Da,
              double Db, double feed, double kill, const Epi& ep, hipStream_t s);
int launch_ac(int32_t dtype, const void* u, void* out, const Dims& d, const Bc& bc, const evx_grid* g, double eps,
              double gab, double M, double force, double curv, const Epi& ep, hipStream_t s);

}  // namespace evx
