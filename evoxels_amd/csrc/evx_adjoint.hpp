// Geometry of the Cahn-Hilliard adjoint's kernels (evx_adjoint.hip): tiles and
// chunks of the streaming one, blocks of the separate ones, and the rule
// between them.
#pragma once
#include <algorithm>

#include "evx_common.hpp"

namespace evx {

constexpr int AT = 1024;  // threads of a block: the columns of its tile, halo included
constexpr int AHALO = 3;           // out(j) reads u, w and mu up to 3, 2 and 2 voxels away
constexpr int AZW = 64;            // longest z extent of a tile
constexpr int APAD = AZW + 2 * AHALO;

// Tiles of zw x tw columns (z, y) that march xl planes along x.
struct AdjGeo {
  int nx, ny, nz, c;
  int zw, tw, xl;
  int gz, gy, gx;  // tiles along z and y, chunks along x
  __host__ __device__ int per_channel() const { return gz * gy * gx; }
};

constexpr size_t adj_lds(size_t es) { return 9 * (size_t)(AT + 2 * APAD) * es; }

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Equal tiles of up to AZW voxels along z (short rows cost more than the halo they
// save: 32 wide at 16 x 128^3 280 instead of 271 us) and as many rows as the
// block's threads hold; along x the chunk that minimises rounds of blocks times planes a block
// marches (its chunk and the 2*AHALO planes that it shares with its neighbours).  Up to 64
// chunks, or a block on every CU: with 64, 4000 x 12 x 60 marched 63 planes
// in 128 blocks (float32 66.4 us, float64 94.0; 42.3 and 58.4 with 256 blocks);
// chunks for two blocks a CU on such grids are slower again (256 x 256 x 1
// float32 25.5 us instead of 18.3; MI355X).
// In 64 bits: the workspace query answers for any extents, also those of which
// adj_check refuses the launch.
struct AdjTiling {
  int64_t zw, tw, xl, gz, gy, gx;
  int64_t per_channel() const { return gz * gy * gx; }
};

inline AdjTiling adj_tiling(int32_t dtype, const Dims& d) {
  AdjTiling a;
  a.zw = ceil_div(d.nz, ceil_div(d.nz, AZW));
  a.gz = ceil_div(d.nz, a.zw);
  a.tw = ceil_div(d.ny, ceil_div(d.ny, AT / (a.zw + 2 * AHALO) - 2 * AHALO));
  a.gy = ceil_div(d.ny, a.tw);
  const int64_t tiles = a.gz * a.gy * d.c;
  a.xl = balanced_xchunk(d.nx, tiles, dtype == EVX_F32 ? 512 : 256, 2 * AHALO, std::max<int64_t>(64, 256 / tiles));
  a.gx = ceil_div(d.nx, a.xl);
  return a;
}

inline AdjGeo adj_geo(const Dims& d, const AdjTiling& t) {
  return {(int)d.nx, (int)d.ny, (int)d.nz, (int)d.c, (int)t.zw, (int)t.tw, (int)t.xl, (int)t.gz, (int)t.gy, (int)t.gx};
}

constexpr int VZ = 64, VY = 4, VT = VZ * VY;  // a block of the separate kernels: a voxel a thread

inline int64_t vox_blocks(const Dims& d) { return ceil_div(d.nz, VZ) * ceil_div(d.ny, VY) * d.nx; }  // a channel's

// Whether the three kernels take less time than adj_stream: asked of grids of
// up to eight planes or rows only (small thick ones are even, 64^3 float32
// 25.7 / 25.1 us, and adj_stream has half the launches).  Estimates in
// microseconds: a CU works its streaming blocks off one after another, 0.70 us
// a plane and 2.8 to start in float32 (1.25 and 5 in float64), and every block
// marches its chunk and six planes more; the three kernels take 2.3 ns a block
// and 4 ps a voxel (2.6 and 10).  Over 614 calls of 4 thousand to 8 million
// voxels and 1 to 16 channels, run both ways (MI355X), they choose within 0.4 %
// of the better one in the mean, 13 % at worst.  The three win on one or two
// planes or rows: streaming / separate, 1 x 1024^2 float32 80 / 30 us and 8
// channels of it 529 / 115, 8 channels of 2 x 512^2 151 / 64, 16 channels of
// 4000 x 1 x 4 float64 321 / 140; but 3 x 200^2 float32 19 / 26.
inline bool adj_separate(int32_t dtype, const Dims& d, const AdjTiling& t) {
  if ((d.nx > 8 && d.ny > 8) || ceil_div(d.ny, VY) > 65535) return false;  // the latter: the launch's grid
  const double rounds = (double)ceil_div(t.per_channel() * d.c, 256), planes = (double)(t.xl + 2 * AHALO);
  const double blocks = (double)vox_blocks(d) * (double)d.c, voxels = (double)d.vol() * (double)d.c;
  const double stream = dtype == EVX_F32 ? 10 + rounds * (0.70 * planes + 2.8) : 5 + rounds * (1.25 * planes + 5);
  const double apart = dtype == EVX_F32 ? 18 + 2.3e-3 * blocks + 4e-6 * voxels : 20 + 2.6e-3 * blocks + 1e-5 * voxels;
  return apart < stream;
}

}  // namespace evx
