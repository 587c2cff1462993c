// Device code of the runtime-radix line transforms (evx_fft_lines.hpp) and
// their launches, compiled once per type.
#pragma once
#include "evx_fft_engine.hpp"
#include "evx_fft_lines.hpp"

namespace evx {

// ------------------------------------------------------------------ passes --
// Line accessors: element e = i + rm of the thread's line, rm block-uniform.
template <typename T>
struct LineGlobal {  // strided line in global memory
  cpx<T>* base;
  int64_t es;
  static constexpr bool LDS = false, BASE = false;
  __device__ __forceinline__ cpx<T> load(int i, int rm) const { return base[(int64_t)i * es + (int64_t)rm * es]; }
  __device__ __forceinline__ void store(int i, int rm, cpx<T> v) const { base[(int64_t)i * es + (int64_t)rm * es] = v; }
};

// As LineGlobal with the upper half of the line (n = 2h) read as the mirror
// image of the stored lower half (sign +-1) and not stored.
template <typename T>
struct LineMirror {
  cpx<T>* base;
  int64_t es;
  int n, h;
  T sign;
  static constexpr bool LDS = false, BASE = false;
  __device__ __forceinline__ cpx<T> load(int i, int rm) const {
    const int e = i + rm;
    const cpx<T> v = base[(int64_t)(e < h ? e : n - 1 - e) * es];
    return e < h ? v : cpx<T>{sign * v.x, sign * v.y};
  }
  __device__ __forceinline__ void store(int i, int rm, cpx<T> v) const {
    if (i + rm < h) base[(int64_t)(i + rm) * es] = v;
  }
};

template <typename T>
struct LineBrick {  // brick of 2^sh lines in LDS, elements 2^sh apart
  cpx<T>* base;
  int sh;
  static constexpr bool LDS = true, BASE = false;
  __device__ __forceinline__ cpx<T> load(int i, int rm) const { return base[(i << sh) + (rm << sh)]; }
  __device__ __forceinline__ void store(int i, int rm, cpx<T> v) const { base[(i << sh) + (rm << sh)] = v; }
};

// Contiguous line in LDS with one pad element after every 2^psh.
template <typename T>
struct LinePadded {
  cpx<T>* base;
  int psh;
  static constexpr bool LDS = true, BASE = false;
  __device__ __forceinline__ cpx<T>* at(int e) const { return base + e + (e >> psh); }
  __device__ __forceinline__ cpx<T> load(int i, int rm) const { return *at(i + rm); }
  __device__ __forceinline__ void store(int i, int rm, cpx<T> v) const { *at(i + rm) = v; }
};

// Element `rm` elements after a block-uniform base plus a lane's 32-bit byte
// offset: the base stays in scalar registers, a load takes one address
// register and no address arithmetic.
template <typename T>
__device__ __forceinline__ T* at_offset(T* base, int rm, uint32_t off) {
  using B = typename std::conditional<std::is_const<T>::value, const char, char>::type;
  return reinterpret_cast<T*>(reinterpret_cast<B*>(base + rm) + off);
}

// Source of the z R2C: a pair of real lines as one complex line.  x is the
// block's first line, l the pair's first element from it.
template <typename T>
struct LinePair {
  const T* x;
  uint32_t l;
  int n;
  bool has_b;
  static constexpr bool LDS = false, BASE = false;
  __device__ __forceinline__ cpx<T> load(int i, int rm) const {
    const uint32_t off = (l + (uint32_t)i) * (uint32_t)sizeof(T);
    return {*at_offset(x, rm, off), has_b ? *at_offset(x, n + rm, off) : T(0)};
  }
};

// Source of the z C2R: Z[e] = A[e] + i B[e] from the staged half spectra.
template <typename T>
struct LineHermitian {
  LinePadded<T> l;
  int n, nh;
  static constexpr bool LDS = true, BASE = false;
  __device__ __forceinline__ cpx<T> load(int i, int rm) const {
    const int e = i + rm, k = e < nh ? e : n - e;
    const T s = e < nh ? T(1) : T(-1);
    const cpx<T> A = *l.at(k), B = *l.at(nh + k);
    return {A.x - s * B.y, s * A.y + B.x};
  }
};

// Destination of the z C2R: the pair's real lines, added to their base.  The
// base values of a butterfly are read before its arithmetic: out may alias
// base, so a read after the first store would wait for it.
template <typename T>
struct LineOut {
  T* out;         // the block's first line
  const T* base;  // the same of the base, or NULL
  uint32_t l;     // the pair's first element
  T scale;
  int n;
  bool has_b;
  static constexpr bool LDS = false, BASE = true;
  __device__ __forceinline__ cpx<T> load_base(int i, int rm) const {
    if (!base) return cpx<T>{T(0), T(0)};
    const uint32_t off = (l + (uint32_t)i) * (uint32_t)sizeof(T);
    return {*at_offset(base, rm, off), has_b ? *at_offset(base, n + rm, off) : T(0)};
  }
  __device__ __forceinline__ void store(int i, int rm, cpx<T> v, cpx<T> bv) const {
    const uint32_t off = (l + (uint32_t)i) * (uint32_t)sizeof(T);
    *at_offset(out, rm, off) = bv.x + scale * v.x;
    if (has_b) *at_offset(out, n + rm, off) = bv.y + scale * v.y;
  }
};

// LDS destination of the last forward pass of an x sweep.
template <typename T>
struct LineMult {  // stores v times the spectral multiplier of its x frequency
  LineBrick<T> l;
  const Prefac& pf;
  PrefacLine pl;
  float ssc;
  int jy, jz;
  int64_t ch;
  static constexpr bool LDS = true, BASE = false;
  __device__ __forceinline__ void store(int i, int rm, cpx<T> v) const {
    const int jx = i + rm;
    T f;
    if (pf.etd) f = static_cast<T>(etd1_f32(jx, jy, jz, pf, ssc)) * static_cast<T>(pf.scale);
    else if (pf.exact) f = static_cast<T>(prefac_f64(jx, jy, jz, pf, ch) * pf.scale);
    else f = static_cast<T>(prefac_f32_line<false>(jx, pl, pf)) * static_cast<T>(pf.scale);
    l.store(i, rm, cscale(v, f));
  }
};

// One pass of radix R.  A source in LDS is synchronised before it is read
// and, when the pass writes LDS again, after.
template <typename T, bool INV, int R, typename Src, typename Dst>
__device__ __forceinline__ void line_pass_r(const LinePass ps, int tl, int tpl, bool active, const cpx<T>* tw,
                                            const Src& src, const Dst& dst) {
  constexpr int S = line_span(R, sizeof(T) == 8);
  const int m = ps.m, p = ps.p;
  if constexpr (Src::LDS) __syncthreads();
  cpx<T> x[S][R];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int i = tl + s * tpl;
    if (active && i < m) {
#pragma unroll
      for (int r = 0; r < R; ++r) x[s][r] = src.load(i, r * m);
    }
  }
  if constexpr (Src::LDS && Dst::LDS) __syncthreads();
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int i = tl + s * tpl;
    if (active && i < m) {
      int j = i * R;
      if (p > 1) {
        const int k = i - (int)__umulhi((uint32_t)i, ps.magic) * p;
        j -= k * (R - 1);
#pragma unroll
        for (int r = 1; r < R; ++r) {
          const cpx<T> w = tw[ps.tw + (r - 1) * p + k];
          x[s][r] = INV ? cmulc(x[s][r], w) : cmul(x[s][r], w);
        }
      }
      if constexpr (Dst::BASE) {
        cpx<T> bv[R];
#pragma unroll
        for (int r = 0; r < R; ++r) bv[r] = dst.load_base(j, r * p);
        dft_any<T, INV, R>(x[s]);
#pragma unroll
        for (int r = 0; r < R; ++r) dst.store(j, r * p, x[s][r], bv[r]);
      } else {
        dft_any<T, INV, R>(x[s]);
#pragma unroll
        for (int r = 0; r < R; ++r) dst.store(j, r * p, x[s][r]);
      }
    }
  }
}

// Prime radix R > 10 through a_r = x_r + x_{R-r}, b_r = x_r - x_{R-r}: outputs
// q and R - q share sum_r a_r cos(2 pi rq/R) and sum_r b_r sin(2 pi rq/R).  The
// outputs are formed one pair at a time (a loop, not unrolled) with the
// coefficients read from the table.  The pass has few butterflies (n/R of a
// line's tpl threads), so the threads left over share their output pairs:
// thread tl takes butterfly tl mod m and every parts-th pair.  One serial chain
// of R(R-1)/2 products a butterfly bounded the sweep: a float64 step of
// 40 x 33 x 31 took 54.8 us with one thread a butterfly and takes 34.5, one of
// 69 x 92 x 115 110.7 and 93 (MI355X).
template <typename T, bool INV, int R, typename Src, typename Dst>
__device__ __forceinline__ void line_pass_prime(const LinePass ps, int tl, int tpl, bool active, const cpx<T>* tw,
                                                const Src& src, const Dst& dst) {
  constexpr int H = (R - 1) / 2;
  const int m = ps.m, p = ps.p;
  const int parts = tpl / m, part = tl / m, i = tl - part * m;
  const bool mine = active && part < parts;
  __syncthreads();  // the source lines, or in a first pass the table
  cpx<T> x[R];
  if (mine) {
#pragma unroll
    for (int r = 0; r < R; ++r) x[r] = src.load(i, r * m);
  }
  if constexpr (Src::LDS && Dst::LDS) __syncthreads();
  if (mine) {
    int j = i * R;
    if (p > 1) {
      const int k = i - (int)__umulhi((uint32_t)i, ps.magic) * p;
      j -= k * (R - 1);
#pragma unroll
      for (int r = 1; r < R; ++r) {
        const cpx<T> w = tw[ps.tw + (r - 1) * p + k];
        x[r] = INV ? cmulc(x[r], w) : cmul(x[r], w);
      }
    }
    cpx<T> sum = x[0];
#pragma unroll
    for (int r = 1; r <= H; ++r) {
      const cpx<T> a = cadd(x[r], x[R - r]), b = csub(x[r], x[R - r]);
      x[r] = a;
      x[R - r] = b;
      sum = cadd(sum, a);
    }
    cpx<T> b0, b1;  // base values of the next output pair
    if constexpr (Dst::BASE) {
      const cpx<T> bs = dst.load_base(j, 0);
      const int q0 = part < H ? part + 1 : H;
      b0 = dst.load_base(j, q0 * p);
      b1 = dst.load_base(j, (R - q0) * p);
      if (part == 0) dst.store(j, 0, sum, bs);
    } else {
      if (part == 0) dst.store(j, 0, sum);
    }
    const cpx<T>* const rt = tw + ps.rt;
#pragma unroll 1
    for (int q = part + 1; q <= H; q += parts) {
      cpx<T> u = x[0], v = {T(0), T(0)};
      int e = 0;
#pragma unroll
      for (int r = 1; r <= H; ++r) {
        e += q;
        if (e >= R) e -= R;
        const cpx<T> w = rt[e];  // (cos, -sin)
        u.x += w.x * x[r].x;
        u.y += w.x * x[r].y;
        v.x -= w.y * x[R - r].x;
        v.y -= w.y * x[R - r].y;
      }
      v = mul_mi<T, INV>(v);
      if constexpr (Dst::BASE) {
        const cpx<T> c0 = b0, c1 = b1;
        const int qn = q + parts <= H ? q + parts : q;
        b0 = dst.load_base(j, qn * p);
        b1 = dst.load_base(j, (R - qn) * p);
        dst.store(j, q * p, cadd(u, v), c0);
        dst.store(j, (R - q) * p, csub(u, v), c1);
      } else {
        dst.store(j, q * p, cadd(u, v));
        dst.store(j, (R - q) * p, csub(u, v));
      }
    }
  }
}

template <typename T, bool INV, bool BIG, typename Src, typename Dst>
__device__ __forceinline__ void line_pass(const LinePass ps, int tl, int tpl, bool active, const cpx<T>* tw,
                                          const Src& src, const Dst& dst) {
  switch (ps.R) {
#define X(RR) \
  case RR: line_pass_r<T, INV, RR>(ps, tl, tpl, active, tw, src, dst); return;
    X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10)
    default: break;
  }
  if constexpr (sizeof(T) == 4) {
    switch (ps.R) {
      X(12) X(15) X(16)
#undef X
      default: break;
    }
  }
  if constexpr (BIG) {
    switch (ps.R) {
#define X(RR) \
  case RR: line_pass_prime<T, INV, RR>(ps, tl, tpl, active, tw, src, dst); return;
      X(11) X(13) X(17) X(19) X(23) X(29) X(31)
#undef X
      default: break;
    }
  }
}

// All passes of a line from src through the LDS line lds to dst.
template <typename T, bool INV, bool BIG, typename Src, typename L, typename Dst>
__device__ __forceinline__ void line_transform(const LinePlan& P, int tl, bool active, const cpx<T>* tw,
                                               const Src& src, const L& lds, const Dst& dst) {
  line_pass<T, INV, BIG>(P.ps[0], tl, P.tpl, active, tw, src, lds);
  for (int s = 1; s < P.npass - 1; ++s) line_pass<T, INV, BIG>(P.ps[s], tl, P.tpl, active, tw, lds, lds);
  line_pass<T, INV, BIG>(P.ps[P.npass - 1], tl, P.tpl, active, tw, lds, dst);
}

// ----------------------------------------------------------------- kernels --
template <typename T>
__device__ __forceinline__ cpx<T>* line_table(unsigned char* smem, const cpx<T>* __restrict__ tab, int n) {
  cpx<T>* tw = reinterpret_cast<cpx<T>*>(smem);
  for (int i = threadIdx.x; i < n; i += blockDim.x) tw[i] = tab[i];
  return tw;
}

// z R2C: real lines (2q, 2q+1) as one complex line; the half spectra of the
// pair are untangled from the transformed line in LDS.
template <typename T, bool BIG>
__global__ __launch_bounds__(line_max_threads(sizeof(T) == 8, BIG), line_min_waves(sizeof(T) == 8, BIG)) void line_z_r2c(
    const T* __restrict__ x, cpx<T>* __restrict__ spec, int64_t nlines, int64_t pitch, LinePlan P, LineGeom g,
    const cpx<T>* __restrict__ tab) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cpx<T>* const tw = line_table(smem_raw, tab, P.tab);
  const int n = P.n, nh = n / 2 + 1, tid = threadIdx.x;
  const int pr = tid / P.tpl, tl = tid - pr * P.tpl;
  const int64_t la = ((int64_t)blockIdx.x * g.lines + pr) * 2;
  const bool active = pr < g.lines && la < nlines, has_b = la + 1 < nlines;
  const LinePadded<T> lds{tw + P.tab + (pr < g.lines ? pr : 0) * g.ls, g.sh};
  const LinePair<T> src{x + (int64_t)blockIdx.x * g.lines * 2 * n, (uint32_t)pr * 2u * (uint32_t)n, n, has_b};
  line_transform<T, false, BIG>(P, tl, active, tw, src, lds, lds);
  __syncthreads();
  if (active) {
    cpx<T>* const sa = spec + la * pitch;
    for (int k = tl; k < nh; k += P.tpl) {
      const cpx<T> Z = *lds.at(k), Zc = *lds.at(k == 0 ? 0 : n - k);
      sa[k] = cpx<T>{(Z.x + Zc.x) * T(0.5), (Z.y - Zc.y) * T(0.5)};
      if (has_b) sa[pitch + k] = cpx<T>{(Z.y + Zc.y) * T(0.5), (Zc.x - Z.x) * T(0.5)};
    }
  }
}

// z C2R: out = base + scale * irfft(spec) per line (base may be NULL, out may
// alias base).  The half spectra A, B of a pair are staged in the pair's LDS
// line (A[k] at slot k, B[k] at slot nh + k); the first pass reads
// Z[e] = A[e] + i B[e] of their Hermitian extensions.
template <typename T, bool BIG>
__global__ __launch_bounds__(line_max_threads(sizeof(T) == 8, BIG), line_min_waves(sizeof(T) == 8, BIG, 4)) void line_z_c2r(
    const cpx<T>* __restrict__ spec, T* out, const T* base, T scale, int64_t nlines, int64_t pitch, LinePlan P,
    LineGeom g, const cpx<T>* __restrict__ tab) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cpx<T>* const tw = line_table(smem_raw, tab, P.tab);
  const int n = P.n, nh = n / 2 + 1, tid = threadIdx.x;
  const int pr = tid / P.tpl, tl = tid - pr * P.tpl;
  const int64_t la = ((int64_t)blockIdx.x * g.lines + pr) * 2;
  const bool active = pr < g.lines && la < nlines, has_b = la + 1 < nlines;
  const LinePadded<T> lds{tw + P.tab + (pr < g.lines ? pr : 0) * g.ls, g.sh};
  if (active) {
    const cpx<T>* const sa = spec + la * pitch;
    for (int k = tl; k < nh; k += P.tpl) {
      cpx<T> A = sa[k], B = has_b ? sa[pitch + k] : cpx<T>{T(0), T(0)};
      if (k == 0 || 2 * k == n) A.y = B.y = T(0);  // C2R ignores Im of the DC and Nyquist bins
      *lds.at(k) = A;
      *lds.at(nh + k) = B;
    }
  }
  const int64_t first = (int64_t)blockIdx.x * g.lines * 2 * n;
  const LineOut<T> dst{out + first, base ? base + first : nullptr, (uint32_t)pr * 2u * (uint32_t)n, scale, n, has_b};
  line_transform<T, true, BIG>(P, tl, active, tw, LineHermitian<T>{lds, n, nh}, lds, dst);
}

// y / x sweep of a brick of adjacent lines.  MODE 0: forward, 1: inverse,
// 2: forward * multiplier * inverse (x axis; semi-implicit, exact-symbol or
// exponential multiplier), the product formed as the forward transform's last
// pass writes LDS.
template <typename T, int MODE, bool BIG>
__global__ __launch_bounds__(line_max_threads(sizeof(T) == 8, BIG), line_min_waves(sizeof(T) == 8, BIG, MODE == 2 ? 5 : 6)) void line_strided(
    cpx<T>* spec, int64_t nlines, LineMap lm, LinePlan P, LineGeom g, const cpx<T>* __restrict__ tab, Prefac pf) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cpx<T>* const tw = line_table(smem_raw, tab, P.tab);
  const int tid = threadIdx.x, t = tid & (g.lines - 1), tl = tid >> g.sh;
  const int64_t L = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * g.lines + t;
  const bool active = L < nlines && tl < P.tpl;
  int64_t outer, k, o, gg;
  if (nlines < (int64_t(1) << 31) && lm.nh < (int64_t(1) << 31) && lm.G < (int64_t(1) << 31)) {  // 32-bit division
    const uint32_t l = active ? (uint32_t)L : 0u, q = l / (uint32_t)lm.nh, h = q / (uint32_t)lm.G;
    outer = q;
    k = l - q * (uint32_t)lm.nh;
    gg = h;
    o = q - h * (uint32_t)lm.G;
  } else {
    const int64_t l = active ? L : 0;
    outer = l / lm.nh;
    k = l - outer * lm.nh;
    gg = outer / lm.G;
    o = outer - gg * lm.G;
  }
  cpx<T>* const line = spec + gg * lm.GM + o * lm.OM + k;
  const LineBrick<T> lds{tw + P.tab + t, g.sh};
  const LineGlobal<T> io{line, lm.es};
  if constexpr (MODE < 2) {
    line_transform<T, MODE == 1, BIG>(P, tl, active, tw, io, lds, io);
  } else {
    const float ssc = symbol_scalar(pf, gg);
    const LineMult<T> mul{lds, pf, prefac_line((int)o, (int)k, pf, ssc), ssc, (int)o, (int)k, gg};
    if (lm.mirror) {
      const LineMirror<T> mio{line, lm.es, P.n, P.n / 2, lm.mirror == 2 ? T(-1) : T(1)};
      line_transform<T, false, BIG>(P, tl, active, tw, mio, lds, mul);
      line_transform<T, true, BIG>(P, tl, active, tw, lds, lds, mio);
    } else {
      line_transform<T, false, BIG>(P, tl, active, tw, io, lds, mul);
      line_transform<T, true, BIG>(P, tl, active, tw, lds, lds, io);
    }
  }
}

// ---------------------------------------------------------------- launches --
template <typename T>
int line_run_z_r2c(const LinePlan& P, const void* tab, const void* x, void* spec, int64_t nlines, int64_t pitch,
                   hipStream_t s) {
  const LineGeom g = line_z_geom<T>(P, (nlines + 1) / 2);
  const int64_t blocks = (nlines + 2 * g.lines - 1) / (2 * g.lines);
  auto kernel = P.big ? line_z_r2c<T, true> : line_z_r2c<T, false>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(g.threads), g.lds, s, static_cast<const T*>(x),
                     static_cast<cpx<T>*>(spec), nlines, pitch, P, g, static_cast<const cpx<T>*>(tab));
  return check_launch("line_z_r2c");
}

template <typename T>
int line_run_z_c2r(const LinePlan& P, const void* tab, const void* spec, void* out, const void* base, double scale,
                   int64_t nlines, int64_t pitch, hipStream_t s) {
  const LineGeom g = line_z_geom<T>(P, (nlines + 1) / 2);
  const int64_t blocks = (nlines + 2 * g.lines - 1) / (2 * g.lines);
  auto kernel = P.big ? line_z_c2r<T, true> : line_z_c2r<T, false>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(g.threads), g.lds, s, static_cast<const cpx<T>*>(spec),
                     static_cast<T*>(out), static_cast<const T*>(base), static_cast<T>(scale), nlines, pitch, P, g,
                     static_cast<const cpx<T>*>(tab));
  return check_launch("line_z_c2r");
}

template <typename T>
int line_run_strided(int mode, const LinePlan& P, const void* tab, void* spec, int64_t nlines, const LineMap& lm,
                     const Prefac& pf, hipStream_t s) {
  const LineGeom g = line_strided_geom<T>(P, nlines);
  const int64_t blocks = (nlines + g.lines - 1) / g.lines;
  auto kernel = mode == 0   ? (P.big ? line_strided<T, 0, true> : line_strided<T, 0, false>)
                : mode == 1 ? (P.big ? line_strided<T, 1, true> : line_strided<T, 1, false>)
                            : (P.big ? line_strided<T, 2, true> : line_strided<T, 2, false>);
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(g.threads), g.lds, s, static_cast<cpx<T>*>(spec), nlines,
                     lm, P, g, static_cast<const cpx<T>*>(tab), pf);
  return check_launch("line_strided");
}

#define EVX_LINE_INSTANTIATE(T)                                                                                      \
  template int line_run_z_r2c<T>(const LinePlan&, const void*, const void*, void*, int64_t, int64_t, hipStream_t);   \
  template int line_run_z_c2r<T>(const LinePlan&, const void*, const void*, void*, const void*, double, int64_t,     \
                                 int64_t, hipStream_t);                                                              \
  template int line_run_strided<T>(int, const LinePlan&, const void*, void*, int64_t, const LineMap&, const Prefac&, \
                                   hipStream_t);

}  // namespace evx
