// Reverse mode of the periodic Cahn-Hilliard right-hand side
// (CahnHilliard.rhs, problem_definition.py:328-371):
//
//   c = clip(u, 0, 1)
//   mu_j = f(c_j) - kappa * lap(c)_j,          f = 18/eps c(1-c)(1-2c), kappa = 2 eps
//   F at the face between lo and hi along axis a:
//        F = m(cf) * (mu_hi - mu_lo) * id_a,    cf = (c_lo + c_hi)/2, m = cf (1 - cf)
//   r_j = D * sum_a id_a (F_{j+a/2} - F_{j-a/2})
//
// Given w = dJ/dr, the transpose is evaluated face by face:
//   GF  = dJ/dF      = D id_a (w_lo - w_hi)
//   H   = dJ/dg      = GF * m(cf)                 (g = (mu_hi - mu_lo) id_a)
//   Kf  = dJ/dcf     = GF * g * (1 - 2 cf)
//   Gmu_j = dJ/dmu_j = sum_a id_a (H_{j-a/2} - H_{j+a/2})
//   dJ/dc_j = f'(c_j) Gmu_j - kappa lap(Gmu)_j + 1/2 sum_faces(j) Kf
// (the periodic 7-point Laplacian is symmetric), and dJ/du_j = dJ/dc_j where
// 0 <= u_j <= 1 (torch.clip's backward), else 0.  Parameter gradients:
//   dJ/dD   = sum over faces F * GF / D
//   dJ/deps = sum_j Gmu_j * (-f(c_j)/eps - 2 lap(c)_j)
//
// One streaming kernel evaluates all of it: mu, the faces, Gmu and the output of
// successive planes follow each other through registers and LDS, so each field
// crosses memory once (adj_stream).  Thin grids, on which its tiles would be
// mostly halo, take three kernels with mu, Gmu and a pointwise part in memory.
// Every block writes its partial parameter sums to its own slot and a last
// kernel folds them in a fixed order, so results are deterministic.
#include "evx_adjoint.hpp"
#include "evx_ch_math.hpp"
#include "evx_common.hpp"
#include "evx_fft_engine.hpp"
#include "evx_sum.hpp"

namespace evx {
namespace {

template <typename T>
struct AdjCoef {
  T s18, kappa, s18e, D;  // 18/eps, 2 eps, 18/eps^2
  T ax, ay, az;           // id_a^2 / 4
};

template <typename T>
__device__ __forceinline__ AdjCoef<T> adj_coef(const double* chan, double eps, double D, int c, const Geo<T>& g) {
  if (chan) {
    eps = chan[2 * c];
    D = chan[2 * c + 1];
  }
  auto face = [&](T id) { return static_cast<T>(0.25 * static_cast<double>(id) * static_cast<double>(id)); };
  return {static_cast<T>(18.0 / eps), static_cast<T>(2.0 * eps), static_cast<T>(18.0 / (eps * eps)),
          static_cast<T>(D), face(g.idx), face(g.idy), face(g.idz)};
}

// One face, scaled: with s = c_lo + c_hi, 4 m = s (2 - s) and 1 - 2 cf = 1 - s;
// h = id H / D and k = Kf / (4 D); h * (mu_hi - mu_lo) = F * GF / D.
template <typename T>
struct AdjFace {
  T h, k, dm;
};
template <typename T>
__device__ __forceinline__ AdjFace<T> adj_face(T cl, T ch, T ml, T mh, T wl, T wh, T a) {
  const T s = cl + ch, t = a * (wl - wh), dm = mh - ml;
  return {t * (s * (T(2) - s)), (t * dm) * (T(1) - s), dm};
}

__device__ __forceinline__ int wrap(int i, int n) {
  i %= n;
  return i < 0 ? i + n : i;
}

// grad = base + J^T w, plane by plane.  A thread owns one column (y, z) of the
// tile or of its halo of three; while plane p of u and w arrives it forms
//   mu(p-1), Gmu(p-2) and the pointwise part P(p-2), out(p-3)
// from its own registers along x and from LDS in the plane.  Every LDS plane
// is read one iteration after it was written, so one barrier orders an iteration.
// The face (p-2, p-1) is evaluated once and carried.
//
// Bound: vector issue (about 130 operations a column and plane; 1024 columns
// hold 64 x 8 outputs, so each is done about twice) and, for float64, its one block a
// CU.  Three kernels with mu, Gmu and P in memory between them moved 17 fields;
// this moves 5 and the halos.  One call at 16 x 128^3 float32 596 -> 264 us,
// float64 1021 -> 425, 4 x 96^3 float64 129 -> 60, 256^3 float32 398 -> 128,
// 8 x 32^3 float32 41 -> 27 (MI355X).  One column a thread: two columns of
// 512 threads took 303 and 554 us at 16 x 128^3 (102 registers, half the
// wavefronts), two of 832 threads 313.  u and base of the output's plane are
// read where they are used: loaded with the next plane they cost registers
// (271 us).  float32 is held to 64 registers, two blocks a CU.
template <typename T, bool STEP>
__global__ __launch_bounds__(AT, sizeof(T) == 4 ? 8 : 4) void adj_stream(
    const T* __restrict__ u, const T* __restrict__ w, const T* base, T* out, const T* __restrict__ u1, double dt,
    double* __restrict__ part, AdjGeo d, Geo<T> g, const double* __restrict__ chan, double eps, double D) {
  constexpr int SLOT = AT + 2 * APAD;  // a row of padding on both sides: neighbours of halo columns stay inside
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* const lds = reinterpret_cast<T*>(smem_raw) + APAD;
  T* const cs = lds;              // three planes of c
  T* const ws = lds + 3 * SLOT;   // two each of w, mu and Gmu
  T* const ms = lds + 5 * SLOT;
  T* const gs = lds + 7 * SLOT;

  const int tid = threadIdx.x;
  const int b = (int)xcd_tile(blockIdx.x, gridDim.x);
  const int ch = b / d.per_channel();
  const int blk = b - ch * d.per_channel();
  const int tz = blk % d.gz, ty = blk / d.gz % d.gy, tx = blk / (d.gz * d.gy);
  const int z0 = tz * d.zw, y0 = ty * d.tw, xa = tx * d.xl, xb = min(xa + d.xl, d.nx);
  const int rw = d.zw + 2 * AHALO, rows = d.tw + 2 * AHALO;
  const AdjCoef<T> k = adj_coef<T>(chan, eps, D, ch, g);
  const int plane = d.ny * d.nz;
  const int64_t cb = (int64_t)ch * d.nx * plane;

  const int yr = tid / rw, zr = tid - yr * rw;
  const int z = z0 + zr - AHALO, y = y0 + yr - AHALO;
  const bool own = zr >= AHALO && zr < rw - AHALO && yr >= AHALO && yr < rows - AHALO && z < d.nz && y < d.ny;
  const int off = yr < rows ? wrap(y, d.ny) * d.nz + wrap(z, d.nz) : 0;

  // c and w of planes p, p-1, p-2; mu of p-2; Gmu of p-3, p-4; P of p-3;
  // dmu/deps of p-2; the face (p-3, p-2)
  T c0, c1, c2, w0, w1, w2, w3, m2, g3, g4, p3, de, hx, kx, un, wn;
  double acc[3] = {0.0, 0.0, 0.0};  // dJ/dD; dJ/deps; (w - dt base)(u1 - u)
  int X = wrap(xa - AHALO, d.nx), Xo = xa;
  c0 = c1 = w0 = w1 = w2 = m2 = g3 = g4 = p3 = de = hx = kx = T(0);
  const int64_t at = cb + (int64_t)X * plane;
  un = u[at + off];
  wn = w[at + off];
  int s0 = 0, s1 = 2 * SLOT, s2 = SLOT;  // slots of c(p), c(p-1), c(p-2)
  for (int p = xa - AHALO; p < xb + AHALO; ++p) {
    const bool emit = p - AHALO >= xa, sums = p - 2 >= xa && p - 2 < xb;
    const int even = (p & 1) * SLOT, odd = SLOT - even;  // slots of planes p, p-2 and of p-1, p-3
    X = X + 1 == d.nx ? 0 : X + 1;
    const int64_t at = cb + (int64_t)X * plane, ato = cb + (int64_t)Xo * plane;
    c2 = c1;
    c1 = c0;
    c0 = clip01(un);
    w3 = w2;
    w2 = w1;
    w1 = w0;
    w0 = wn;
    un = u[at + off];
    wn = w[at + off];
    cs[s0 + tid] = c0;
    ws[odd + tid] = w1;
    // mu(p-1)
    const T* const ca = cs + s1 + tid;
    const T lap1 = Ops<false>::lap7(c1, c0, c2, ca[rw], ca[-rw], ca[1], ca[-1], g);
    const T f1 = (c1 * (T(1) - c1)) * (T(1) - T(2) * c1);
    const T m1 = k.s18 * f1 - k.kappa * lap1;
    const T de1 = -(k.s18e * f1) - T(2) * lap1;  // dmu/deps
    ms[odd + tid] = m1;
    // faces of plane p-2
    const T* const cc = cs + s2 + tid;
    const T* const wc = ws + even + tid;
    const T* const mc = ms + even + tid;
    const T cj = c2, wj = w2, mj = m2;
    const AdjFace<T> x1 = adj_face(cj, c1, mj, m1, wj, w1, k.ax);
    const AdjFace<T> ya = adj_face(cc[-rw], cj, mc[-rw], mj, wc[-rw], wj, k.ay);
    const AdjFace<T> yb = adj_face(cj, cc[rw], mj, mc[rw], wj, wc[rw], k.ay);
    const AdjFace<T> za = adj_face(cc[-1], cj, mc[-1], mj, wc[-1], wj, k.az);
    const AdjFace<T> zb = adj_face(cj, cc[1], mj, mc[1], wj, wc[1], k.az);
    const T gm = k.D * (((hx - x1.h) + (ya.h - yb.h)) + (za.h - zb.h));
    const T ks = (T(2) * k.D) * (((kx + x1.k) + (ya.k + yb.k)) + (za.k + zb.k));
    const T pw = (k.s18 * ((T(1) - T(6) * cj) + T(6) * cj * cj)) * gm + ks;
    hx = x1.h;
    kx = x1.k;
    gs[even + tid] = gm;
    if (sums && own) {
      acc[0] += static_cast<double>((x1.h * x1.dm + yb.h * yb.dm) + zb.h * zb.dm);
      acc[1] += static_cast<double>(gm) * static_cast<double>(de);
    }
    // out(p-3)
    T uo = T(0), bo = T(0), u1o = T(0);
    if (emit && own) {
      uo = u[ato + off];
      if (base) bo = base[ato + off];
      if (STEP) u1o = u1[ato + off];
    }
    const T* const gc = gs + odd + tid;
    const T lapg = Ops<false>::lap7(g3, gm, g4, gc[rw], gc[-rw], gc[1], gc[-1], g);
    if (emit && own) {
      const T gu = (uo >= T(0) && uo <= T(1)) ? p3 - k.kappa * lapg : T(0);
      out[ato + off] = bo + gu;
      if (STEP)
        acc[2] += static_cast<double>(w3 - static_cast<T>(dt) * bo) * static_cast<double>(u1o - uo);
    }
    m2 = m1;
    de = de1;
    g4 = g3;
    g3 = gm;
    p3 = pw;
    Xo += emit ? 1 : 0;
    const int t = s2;
    s2 = s1;
    s1 = s0;
    s0 = t;
    __syncthreads();
  }

  __shared__ SumPair red[3][AT / 64];
#pragma unroll
  for (int v = 0; v < 3; ++v) {
    const SumPair sp = wave_sum(SumPair{acc[v], 0.0});
    if ((tid & 63) == 0) red[v][tid >> 6] = sp;
  }
  __syncthreads();
  if (tid < 3) {
    SumPair sp = red[tid][0];
    for (int i = 1; i < AT / 64; ++i) sp = sum_merge(sp, red[tid][i]);
    part[3 * (int64_t)b + tid] = sp.s + sp.c;
  }
}

// ---------------------------------------------------------------------------
// The same in three kernels with mu, Gmu and the pointwise part P in memory: mu;
// Gmu, P and the parameter sums; the output with lap(Gmu).  A voxel per
// thread and no halo, so nothing is evaluated twice: taken where adj_stream's
// tiles and chunks would be mostly halo (adj_separate).
// ---------------------------------------------------------------------------
struct AdjDims {
  int nx, ny, nz, c;
  int gx, gy;  // blocks along z and y per plane
};

template <typename T>
struct VoxCoef {
  T s18, kappa, D, eps;
};
template <typename T>
__device__ __forceinline__ VoxCoef<T> vox_coef(const double* chan, double eps, double D, int c) {
  if (chan) {
    eps = chan[2 * c];
    D = chan[2 * c + 1];
  }
  return {static_cast<T>(18.0 / eps), static_cast<T>(2.0 * eps), static_cast<T>(D), static_cast<T>(eps)};
}

// Offsets of a voxel and its six periodic neighbours inside one channel.
struct Nb7 {
  int64_t base;  // channel offset
  int j, xm, xp, ym, yp, zm, zp;
  bool valid;
  int c, blk;  // channel, block index inside the channel
};

__device__ __forceinline__ Nb7 neighbours(const AdjDims& d) {
  Nb7 n;
  const int z = blockIdx.x * VZ + threadIdx.x;
  const int y = blockIdx.y * VY + threadIdx.y;
  const int zc = blockIdx.z;  // = c * nx + x
  const int c = zc / d.nx, x = zc - (zc / d.nx) * d.nx;
  n.c = c;
  n.blk = (x * d.gy + (int)blockIdx.y) * d.gx + (int)blockIdx.x;
  n.valid = z < d.nz && y < d.ny;
  const int zz = n.valid ? z : 0, yy = n.valid ? y : 0;
  const int plane = d.ny * d.nz;
  n.base = (int64_t)c * d.nx * plane;
  n.j = (x * d.ny + yy) * d.nz + zz;
  n.xm = n.j + (x == 0 ? (d.nx - 1) * plane : -plane);
  n.xp = n.j + (x == d.nx - 1 ? -(d.nx - 1) * plane : plane);
  n.ym = n.j + (yy == 0 ? (d.ny - 1) * d.nz : -d.nz);
  n.yp = n.j + (yy == d.ny - 1 ? -(d.ny - 1) * d.nz : d.nz);
  n.zm = n.j + (zz == 0 ? d.nz - 1 : -1);
  n.zp = n.j + (zz == d.nz - 1 ? -(d.nz - 1) : 1);
  return n;
}

template <typename T>
__device__ __forceinline__ T f_hom(T c, T s18) {
  return ((s18 * c) * (T(1) - c)) * (T(1) - T(2) * c);
}

// Deterministic block sum of NV doubles per thread; thread 0 gets the totals.
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV]) {
  __shared__ double red[VT / 64][NV];
#pragma unroll
  for (int k = 0; k < NV; ++k)
    for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_down(v[k], off, 64);
  const int tid = threadIdx.y * VZ + threadIdx.x, wid = tid >> 6;
  if ((tid & 63) == 0)
#pragma unroll
    for (int k = 0; k < NV; ++k) red[wid][k] = v[k];
  __syncthreads();
  if (tid == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      double s = 0.0;
      for (int w = 0; w < VT / 64; ++w) s += red[w][k];
      v[k] = s;
    }
  }
}

// mu = f(c) - kappa*lap(c), c = clip(u).
template <typename T>
__global__ __launch_bounds__(VT) void adj_mu_kernel(const T* __restrict__ u, T* __restrict__ mu, AdjDims d,
                                                    Geo<T> g, const double* __restrict__ chan, double eps,
                                                    double D) {
  const Nb7 n = neighbours(d);
  if (!n.valid) return;
  const VoxCoef<T> k = vox_coef<T>(chan, eps, D, n.c);
  const T* uc = u + n.base;
  const T c = clip01(uc[n.j]);
  const T lap = Ops<false>::lap7(c, clip01(uc[n.xp]), clip01(uc[n.xm]), clip01(uc[n.yp]), clip01(uc[n.ym]),
                                 clip01(uc[n.zp]), clip01(uc[n.zm]), g);
  mu[n.base + n.j] = f_hom(c, k.s18) - k.kappa * lap;
}

// Gmu and P = f'(c) Gmu + 1/2 sum Kf; partial parameter sums (dD, deps).
template <typename T>
__global__ __launch_bounds__(VT) void adj_faces_kernel(const T* __restrict__ u, const T* __restrict__ w,
                                                       const T* __restrict__ mu, T* __restrict__ gmu,
                                                       T* __restrict__ pw, double* __restrict__ part, AdjDims d,
                                                       Geo<T> g, const double* __restrict__ chan, double eps,
                                                       double D, int nblk) {
  const Nb7 n = neighbours(d);
  const VoxCoef<T> k = vox_coef<T>(chan, eps, D, n.c);
  double acc[2] = {0.0, 0.0};  // dJ/dD, dJ/deps
  if (n.valid) {
    const T* uc = u + n.base;
    const T* wc = w + n.base;
    const T* mc = mu + n.base;
    const T cj = clip01(uc[n.j]), wj = wc[n.j], mj = mc[n.j];
    const int lo[3] = {n.xm, n.ym, n.zm}, hi[3] = {n.xp, n.yp, n.zp};
    const T id[3] = {g.idx, g.idy, g.idz};
    T cn[3][2];
    T gm = T(0), ks = T(0), dd = T(0);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const T cl = clip01(uc[lo[a]]), ch = clip01(uc[hi[a]]);
      cn[a][0] = cl;
      cn[a][1] = ch;
      // face (j-a, j)
      T cf = T(0.5) * (cl + cj);
      T m = cf * (T(1) - cf);
      T gg = (mj - mc[lo[a]]) * id[a];
      T gf = k.D * id[a] * (wc[lo[a]] - wj);
      const T hm = gf * m;
      ks += gf * gg * (T(1) - T(2) * cf);
      // face (j, j+a)
      cf = T(0.5) * (cj + ch);
      m = cf * (T(1) - cf);
      gg = (mc[hi[a]] - mj) * id[a];
      const T wd = wj - wc[hi[a]];
      gf = k.D * id[a] * wd;
      const T hp = gf * m;
      ks += gf * gg * (T(1) - T(2) * cf);
      dd += (m * gg) * (id[a] * wd);
      gm += id[a] * (hm - hp);
    }
    const T fp = k.s18 * ((T(1) - T(6) * cj) + T(6) * cj * cj);
    gmu[n.base + n.j] = gm;
    pw[n.base + n.j] = fp * gm + T(0.5) * ks;
    const T lapc = Ops<false>::lap7(cj, cn[0][1], cn[0][0], cn[1][1], cn[1][0], cn[2][1], cn[2][0], g);
    const T dmu_deps = -f_hom(cj, k.s18) / k.eps - T(2) * lapc;
    acc[0] = static_cast<double>(dd);
    acc[1] = static_cast<double>(gm) * static_cast<double>(dmu_deps);
  }
  block_sum<2>(acc);
  if (threadIdx.x == 0 && threadIdx.y == 0) {
    double* p = part + 3 * ((int64_t)n.c * nblk + n.blk);
    p[0] = acc[0];
    p[1] = acc[1];
  }
}

// out = base + mask(u) * (P - kappa lap(Gmu)); with u1 != NULL also the
// partial of sum (w - dt*base) * (u1 - u) for the prefactor gradient.
template <typename T>
__global__ __launch_bounds__(VT) void adj_out_kernel(const T* __restrict__ u, const T* __restrict__ gmu,
                                                     const T* __restrict__ pw, const T* base, T* out,
                                                     const T* __restrict__ w, const T* __restrict__ u1,
                                                     double dt, double* __restrict__ part, AdjDims d, Geo<T> g,
                                                     const double* __restrict__ chan, double eps, double D,
                                                     int nblk) {
  const Nb7 n = neighbours(d);
  const VoxCoef<T> k = vox_coef<T>(chan, eps, D, n.c);
  double acc[1] = {0.0};
  if (n.valid) {
    const T* gc = gmu + n.base;
    const int64_t i = n.base + n.j;
    const T uj = u[i];
    const T lapg = Ops<false>::lap7(gc[n.j], gc[n.xp], gc[n.xm], gc[n.yp], gc[n.ym], gc[n.zp], gc[n.zm], g);
    const T gu = (uj >= T(0) && uj <= T(1)) ? pw[i] - k.kappa * lapg : T(0);
    const T b = base ? base[i] : T(0);
    out[i] = b + gu;
    if (u1) acc[0] = static_cast<double>(w[i] - static_cast<T>(dt) * b) * static_cast<double>(u1[i] - uj);
  }
  if (u1) {
    block_sum<1>(acc);
    if (threadIdx.x == 0 && threadIdx.y == 0) part[3 * ((int64_t)n.c * nblk + n.blk) + 2] = acc[0];
  }
}

// Per channel: fold the block partials (compensated, fixed order) and add the
// gradients to dparams = {dJ/deps, dJ/dD}.  With step the prefactor
// term S/(dt*theta) is added as well.  W wavefronts a sum.
template <int W>
__global__ __launch_bounds__(192 * W) void adj_final_kernel(const double* __restrict__ part, int nblk, int step,
                                                            double* dparams, const double* __restrict__ chan,
                                                            double eps, double D, double dt) {
  const int c = blockIdx.x, v = threadIdx.x / (64 * W), lane = threadIdx.x % (64 * W);
  __shared__ SumPair wsum[3 * W];
  __shared__ double tot[3];
  SumPair s{0.0, 0.0};
  for (int b = lane; b < nblk; b += 64 * W) s = sum_merge(s, SumPair{part[3 * ((int64_t)c * nblk + b) + v], 0.0});
  s = wave_sum(s);
  if ((lane & 63) == 0) wsum[threadIdx.x >> 6] = s;
  __syncthreads();
  if (lane == 0) {
    s = wsum[v * W];
    for (int w = 1; w < W; ++w) s = sum_merge(s, wsum[v * W + w]);
    tot[v] = s.s + s.c;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (chan) {
      eps = chan[2 * c];
      D = chan[2 * c + 1];
    }
    double g_d = tot[0], g_e = tot[1];
    if (step) {
      g_e += tot[2] / (dt * eps);
      g_d += tot[2] / (dt * D);
    }
    dparams[2 * c] += g_e;
    dparams[2 * c + 1] += g_d;
  }
}

size_t align_up(size_t v) { return (v + 255) & ~size_t(255); }

int adj_check(const Dims& d) {
  if (d.nx * d.c > 65535) return fail(EVX_ERR_UNSUPPORTED, "adjoint kernels need channels*nx <= 65535");
  if (d.vol() >= (int64_t(1) << 31)) return fail(EVX_ERR_UNSUPPORTED, "adjoint kernels need nx*ny*nz < 2^31");
  return EVX_OK;
}

template <typename T>
int adj_launch(const void* u, const void* w, const void* base, void* grad, double* dparams, const AdjGeo& a,
               const Geo<T>& g, double eps, double D, const double* chan, const void* u1, double dt, double* part,
               hipStream_t s) {
  const dim3 grid((unsigned)((int64_t)a.per_channel() * a.c));
  const T *ut = static_cast<const T*>(u), *wt = static_cast<const T*>(w), *bt = static_cast<const T*>(base),
          *vt = static_cast<const T*>(u1);
  if (u1)
    hipLaunchKernelGGL((adj_stream<T, true>), grid, dim3(AT), adj_lds(sizeof(T)), s, ut, wt, bt,
                       static_cast<T*>(grad), vt, dt, part, a, g, chan, eps, D);
  else
    hipLaunchKernelGGL((adj_stream<T, false>), grid, dim3(AT), adj_lds(sizeof(T)), s, ut, wt, bt,
                       static_cast<T*>(grad), vt, dt, part, a, g, chan, eps, D);
  EVX_TRY(check_launch("adj_stream"));
  hipLaunchKernelGGL(adj_final_kernel<1>, dim3(a.c), dim3(192), 0, s, part, a.per_channel(), u1 ? 1 : 0, dparams, chan,
                     eps, D, dt);
  return check_launch("adj_final_kernel");
}

template <typename T>
int adj_launch_separate(const void* u, const void* w, const void* base, void* grad, double* dparams, const Dims& d,
                        const Geo<T>& g, double eps, double D, const double* chan, const void* u1, double dt, void* ws,
                        hipStream_t s) {
  const AdjDims a{(int)d.nx, (int)d.ny, (int)d.nz, (int)d.c, (int)ceil_div(d.nz, VZ), (int)ceil_div(d.ny, VY)};
  const size_t field = align_up((size_t)d.c * d.vol() * sizeof(T));
  char* const p = static_cast<char*>(ws);
  T *mu = reinterpret_cast<T*>(p), *gmu = reinterpret_cast<T*>(p + field), *pw = reinterpret_cast<T*>(p + 2 * field);
  double* const part = reinterpret_cast<double*>(p + 3 * field);
  const int nblk = (int)vox_blocks(d);
  const dim3 grid(a.gx, a.gy, a.nx * a.c), block(VZ, VY);
  const T *ut = static_cast<const T*>(u), *wt = static_cast<const T*>(w), *bt = static_cast<const T*>(base),
          *vt = static_cast<const T*>(u1);
  hipLaunchKernelGGL(adj_mu_kernel<T>, grid, block, 0, s, ut, mu, a, g, chan, eps, D);
  EVX_TRY(check_launch("adj_mu_kernel"));
  hipLaunchKernelGGL(adj_faces_kernel<T>, grid, block, 0, s, ut, wt, mu, gmu, pw, part, a, g, chan, eps, D, nblk);
  EVX_TRY(check_launch("adj_faces_kernel"));
  hipLaunchKernelGGL(adj_out_kernel<T>, grid, block, 0, s, ut, gmu, pw, bt, static_cast<T*>(grad), wt, vt, dt, part, a,
                     g, chan, eps, D, nblk);
  EVX_TRY(check_launch("adj_out_kernel"));
  hipLaunchKernelGGL(adj_final_kernel<4>, dim3(a.c), dim3(768), 0, s, part, nblk, u1 ? 1 : 0, dparams, chan, eps, D,
                     dt);
  return check_launch("adj_final_kernel");
}

}  // namespace

// Workspace: the blocks' partial sums, after three fields where the kernels are separate.
size_t ch_rhs_vjp_ws_bytes(int32_t dtype, const Dims& d) {
  const AdjTiling t = adj_tiling(dtype, d);
  if (adj_separate(dtype, d, t))
    return 3 * align_up((size_t)d.c * d.vol() * (dtype == EVX_F32 ? 4 : 8)) +
           align_up((size_t)d.c * (size_t)vox_blocks(d) * 3 * sizeof(double));
  return align_up((size_t)d.c * (size_t)t.per_channel() * 3 * sizeof(double));
}

// dparams += ...; grad = base + J^T w.  With u1 != NULL (semi-implicit step)
// the prefactor term is added with S = sum (w - dt*base)(u1 - u).
int ch_rhs_vjp_launch(int32_t dtype, const void* u, const void* w, const void* base, void* grad,
                      double* dparams, const Dims& d, const double dd[3], const double dd2[3], double eps,
                      double D, const double* chan, const void* u1, double dt, void* ws, hipStream_t s) {
  EVX_TRY(adj_check(d));
  evx_grid eg{d.c, d.nx, d.ny, d.nz, {dd[0], dd[1], dd[2]}, {dd2[0], dd2[1], dd2[2]}};
  const Geo<float> gf = make_geo_from<float>(eg.div_dx, eg.div_dx2);
  const Geo<double> gd = make_geo_from<double>(eg.div_dx, eg.div_dx2);
  const AdjTiling t = adj_tiling(dtype, d);
  if (adj_separate(dtype, d, t))
    return dtype == EVX_F32
               ? adj_launch_separate<float>(u, w, base, grad, dparams, d, gf, eps, D, chan, u1, dt, ws, s)
               : adj_launch_separate<double>(u, w, base, grad, dparams, d, gd, eps, D, chan, u1, dt, ws, s);
  const AdjGeo a = adj_geo(d, t);
  double* part = static_cast<double*>(ws);
  return dtype == EVX_F32 ? adj_launch<float>(u, w, base, grad, dparams, a, gf, eps, D, chan, u1, dt, part, s)
                          : adj_launch<double>(u, w, base, grad, dparams, a, gd, eps, D, chan, u1, dt, part, s);
}

}  // namespace evx

using namespace evx;

extern "C" int evx_ch_rhs_vjp_workspace_bytes(int32_t dtype, const evx_grid* g, size_t* bytes) {
  if (!g || !bytes) return fail(EVX_ERR_INVALID, "null argument");
  if (dtype != EVX_F32 && dtype != EVX_F64) return fail(EVX_ERR_INVALID, "dtype must be EVX_F32 or EVX_F64");
  Dims d;
  EVX_TRY(make_dims(g, &d));
  *bytes = ch_rhs_vjp_ws_bytes(dtype, d);
  return EVX_OK;
}

extern "C" int evx_ch_rhs_vjp(int32_t dtype, const void* u, const void* w, const void* base, void* grad_u,
                              double* dparams, const evx_grid* g, double eps, double D, const double* chan_params,
                              void* workspace, void* stream) {
  if (!u || !w || !grad_u || !dparams || !g || !workspace) return fail(EVX_ERR_INVALID, "null argument");
  if (dtype != EVX_F32 && dtype != EVX_F64) return fail(EVX_ERR_INVALID, "dtype must be EVX_F32 or EVX_F64");
  if (!chan_params && !(eps != 0.0)) return fail(EVX_ERR_INVALID, "eps must be nonzero");
  if (grad_u == u || grad_u == w) return fail(EVX_ERR_INVALID, "grad_u must not alias u or w");
  Dims d;
  EVX_TRY(make_dims(g, &d));
  return ch_rhs_vjp_launch(dtype, u, w, base, grad_u, dparams, d, g->div_dx, g->div_dx2, eps, D, chan_params,
                           nullptr, 0.0, workspace, static_cast<hipStream_t>(stream));
}
