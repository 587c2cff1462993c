// Launches of the explicit right-hand sides (evx_explicit.hip) and the normal
// Laplacian they share with the padded operators.
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

int launch_rd(int32_t dtype, const void* u, void* out, const Dims& d, const Bc& bc, const evx_grid* g, double D,
              const Epi& ep, hipStream_t s);
int launch_gs(int32_t dtype, const void* u, void* out, const Dims& d, const Bc& bc, const evx_grid* g, double Da,
              double Db, double feed, double kill, const Epi& ep, hipStream_t s);
int launch_ac(int32_t dtype, const void* u, void* out, const Dims& d, const Bc& bc, const evx_grid* g, double eps,
              double gab, double M, double force, double curv, const Epi& ep, hipStream_t s);

}  // namespace evx
