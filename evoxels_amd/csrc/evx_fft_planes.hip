// Whole-plane z and y sweeps of N x N planes (see evx_fft_planes.hpp).
//
// A block holds one plane: N rows of half spectra, PITCH complex values apart.
// In the z phase TPL threads transform a pair of real lines inside the pair's
// two LDS rows (the exchange line of N + N/16 slots fits two rows); in the y
// phase TPL threads transform a column.  The values a thread holds are those of
// the register engine (E per thread), so a plane takes one round of threads.
//
// Bound: below about 32 MB of state a launch and a plane's latency (the two
// sweeps of 32^3 float32 take 3.5 and 4.5 us, hardly more than empty launches), so
// two launches instead of four are the gain; above it memory, where a plane
// sweep reads and writes once (zy 55.8 us for 16 x 128^3 float32, 4.8 TB/s)
// and the pair of sweeps it replaces twice (51.0 + 71.9).
//
// Few passes of high radix: each pass costs two barriers of the whole block
// and a trip through LDS, and one plane's block is alone on its CU at the
// large sizes.  100 as 10*10 instead of 2*5*2*5 took 100^3 float64's pair of
// sweeps from 34.6 to 27.0 us; 96 as 6*4*4 instead of 3*4*4*2 and 128 as 16*8
// instead of 2*8*8 took 96^3 float32's step from 35 to 31.7 and
// 128^3 float32's from 45.8 to 42.2 (MI355X).
//
// plane_inv of 128 points in float64 is held to 168 registers by its 9
// wavefronts and spills 28 of them (116 bytes of scratch a lane): the state's
// values wait in registers during the transform.
#include "evx_fft_planes.hpp"

namespace evx {
namespace {

template <typename T, int PITCH>
struct ColLay {  // column of the LDS plane
  static constexpr bool SPLIT = false, WAVE = false;
  cpx<T>* base;
  __device__ __forceinline__ cpx<T>* at(int e) const { return base + e * PITCH; }
  template <int TPL>
  __device__ __forceinline__ cpx<T>* at_q(int tl, int q) const { return at(tl) + q * (TPL * PITCH); }
};

template <typename T, int N>
__global__ __launch_bounds__((PGeo<T, N>::THREADS)) void plane_fwd(const T* __restrict__ x, cpx<T>* __restrict__ spec,
                                                                const cpx<T>* __restrict__ twg) {
  using G = PGeo<T, N>;
  constexpr int E = G::E, TPL = G::TPL, NH = G::NH, PITCH = G::PITCH;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  cpx<T>* const tw = reinterpret_cast<cpx<T>*>(smem_raw);
  cpx<T>* const lds = tw + N;
  const int tid = threadIdx.x;
  const int64_t plane = xcd_tile(blockIdx.x, gridDim.x);
  using Rx = typename PlaneSpec<N>::R;
  static_assert(pass_tw_size<N>(Rx{}) <= N, "pass tables fit the twiddle region");
  {
    const int pr = tid / TPL, tl = tid - (tid / TPL) * TPL;
    const bool mine = pr < N / 2;
    const T* const a = x + plane * (N * N) + (mine ? pr : 0) * (2 * N);
    cpx<T> v[E];
#pragma unroll
    for (int q = 0; q < E; ++q) v[q] = cpx<T>{a[tl + TPL * q], a[N + tl + TPL * q]};
    pass_tw_fill<T, N>(tw, twg, tid, G::THREADS, Rx{});
    __syncthreads();  // twiddles
    cpx<T>* const row = lds + (mine ? pr : N / 2) * (2 * PITCH);
    const LineLay<T, G::LINE, G::WAVE> lay{row};
    fft_regs_pt<T, N, TPL, false>(v, lay, tl, tw, Rx{});
    xsync<G::WAVE>();
#pragma unroll
    for (int q = 0; q < E; ++q) *lay.template at_q<TPL>(tl, q) = v[q];
    xsync<G::WAVE>();
    // the pair's half spectra through registers into its two rows
    constexpr int H = (NH + TPL - 1) / TPL;
    cpx<T> z[H];
#pragma unroll
    for (int q = 0; q < H; ++q) {
      const int k = tl + TPL * q;
      if (k < NH) z[q] = *lay.at(k == 0 ? 0 : N - k);
    }
    xsync<G::WAVE>();
#pragma unroll
    for (int q = 0; q < H; ++q) {
      const int k = tl + TPL * q;
      if (k < NH) {
        const cpx<T> Z = v[q], Zc = z[q];
        row[k] = cpx<T>{(Z.x + Zc.x) * T(0.5), (Z.y - Zc.y) * T(0.5)};
        row[PITCH + k] = cpx<T>{(Z.y + Zc.y) * T(0.5), (Zc.x - Z.x) * T(0.5)};
      }
    }
  }
  __syncthreads();
  const int k = tid % NH, tl = tid / NH;  // threads past the last column's share work on the spare column
  const bool mine = tl < TPL;
  const ColLay<T, PITCH> lay{lds + (mine ? k : NH)};
  const int t = mine ? tl : 0;
  cpx<T> v[E];
#pragma unroll
  for (int q = 0; q < E; ++q) v[q] = *lay.template at_q<TPL>(t, q);
  fft_regs_pt<T, N, TPL, false>(v, lay, t, tw, Rx{});
  if (mine) {
    cpx<T>* const sp = spec + plane * (N * NH) + tl * NH + k;
#pragma unroll
    for (int q = 0; q < E; ++q) sp[q * (TPL * NH)] = v[q];
  }
}

template <typename T, int N>
__global__ __launch_bounds__((PGeo<T, N>::THREADS)) void plane_inv(const cpx<T>* __restrict__ spec, T* out, const T* base,
                                                                T scale, const cpx<T>* __restrict__ twg,
                                                                SumRec* __restrict__ rec) {
  using G = PGeo<T, N>;
  constexpr int E = G::E, TPL = G::TPL, NH = G::NH, PITCH = G::PITCH;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ SumPair wsum[16];
  __shared__ int wflag[16];
  cpx<T>* const tw = reinterpret_cast<cpx<T>*>(smem_raw);
  cpx<T>* const lds = tw + N;
  const int tid = threadIdx.x;
  const int64_t plane = xcd_tile(blockIdx.x, gridDim.x);
  using Rx = typename PlaneSpec<N>::R;
  {
    const int k = tid % NH, tl = tid / NH;
    const bool mine = tl < TPL;
    const int t = mine ? tl : 0;
    const cpx<T>* const sp = spec + plane * (N * NH) + t * NH + k;
    cpx<T> v[E];
#pragma unroll
    for (int q = 0; q < E; ++q) v[q] = sp[q * (TPL * NH)];
    pass_tw_fill<T, N>(tw, twg, tid, G::THREADS, Rx{});
    __syncthreads();  // twiddles
    const ColLay<T, PITCH> lay{lds + (mine ? k : NH)};
    fft_regs_pt<T, N, TPL, true>(v, lay, t, tw, Rx{});
    __syncthreads();  // the last exchange reads are done
#pragma unroll
    for (int q = 0; q < E; ++q) *lay.template at_q<TPL>(t, q) = v[q];
  }
  const int pr = tid / TPL, tl = tid - (tid / TPL) * TPL;
  const bool mine = pr < N / 2;
  const int64_t first = plane * (N * N) + (mine ? pr : 0) * (2 * N);
  cpx<T> bv[E];  // the state added to the update, in flight during the transform
#pragma unroll
  for (int q = 0; q < E; ++q)
    bv[q] = base ? cpx<T>{base[first + tl + TPL * q], base[first + N + tl + TPL * q]} : cpx<T>{T(0), T(0)};
  __syncthreads();  // the plane's rows are in LDS
  cpx<T>* const row = lds + (mine ? pr : N / 2) * (2 * PITCH);
  cpx<T> v[E];
  // Z[k] = A[k] + i B[k] of the Hermitian extensions; the DC and Nyquist terms are real
#pragma unroll
  for (int q = 0; q < E; ++q) {
    const int k = tl + TPL * q, j = k <= N / 2 ? k : N - k;
    const cpx<T> a = row[j], b = row[PITCH + j];
    if (j == 0 || j == N / 2) v[q] = cpx<T>{a.x, b.x};
    else v[q] = k < N / 2 ? cpx<T>{a.x - b.y, a.y + b.x} : cpx<T>{a.x + b.y, b.x - a.y};
  }
  const LineLay<T, G::LINE, G::WAVE> lay{row};
  fft_regs_pt<T, N, TPL, true>(v, lay, tl, tw, Rx{});
  double acc = 0.0;
  bool nan = false, inf = false;
  if (mine) {
    T* const o = out + first;
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const T a = bv[q].x + scale * v[q].x, b = bv[q].y + scale * v[q].y;
      o[tl + TPL * q] = a;
      o[N + tl + TPL * q] = b;
      if (rec) {
        acc += static_cast<double>(a);
        acc += static_cast<double>(b);
        nan = nan || a != a || b != b;
        inf = inf || __builtin_isinf(a) || __builtin_isinf(b);
      }
    }
  }
  if (rec) {  // uniform
    const SumPair s = wave_sum(SumPair{acc, 0.0});
    const int f = (__any(nan) ? 1 : 0) | (__any(inf) ? 2 : 0);
    if ((tid & 63) == 0) {
      wsum[tid >> 6] = s;
      wflag[tid >> 6] = f;
    }
    __syncthreads();
    if (tid == 0) {
      SumPair b = wsum[0];
      int e = wflag[0];
      for (int i = 1; i < G::THREADS / 64; ++i) {
        b = sum_merge(b, wsum[i]);
        e |= wflag[i];
      }
      rec[plane] = SumRec{b.s, b.c, e & 1, (e >> 1) & 1, {0, 0}};
    }
  }
}

}  // namespace

bool plane_sweeps_apply(int dtype, const Dims& d) {
  if (d.ny != d.nz) return false;
  if (dtype == EVX_F64 && d.ny == 128 && d.c * d.nx < 48) return false;
  switch (d.ny) {
#define X(N) case N:
    EVX_PLANE_SIZES(X)
#undef X
    return true;
    default:
      return false;
  }
}

template <typename T>
int plane_run_fwd(int n, const void* twg, const T* x, cpx<T>* spec, int64_t nplanes, hipStream_t s) {
  switch (n) {
#define X(N)                                                                                                       \
  case N:                                                                                                          \
    hipLaunchKernelGGL((plane_fwd<T, N>), dim3((unsigned)nplanes), dim3(PGeo<T, N>::THREADS), (PGeo<T, N>::LDS), s, x, \
                       spec, static_cast<const cpx<T>*>(twg));                                                     \
    break;
    EVX_PLANE_SIZES(X)
#undef X
    default:
      return fail(EVX_ERR_UNSUPPORTED, "no plane sweep of %d points", n);
  }
  return check_launch("plane_fwd");
}

template <typename T>
int plane_run_inv(int n, const void* twg, const cpx<T>* spec, T* out, const T* base, double scale, int64_t nplanes,
                  SumRec* rec, hipStream_t s) {
  switch (n) {
#define X(N)                                                                                                        \
  case N:                                                                                                           \
    hipLaunchKernelGGL((plane_inv<T, N>), dim3((unsigned)nplanes), dim3(PGeo<T, N>::THREADS), (PGeo<T, N>::LDS), s,     \
                       spec, out, base, static_cast<T>(scale), static_cast<const cpx<T>*>(twg), rec);                \
    break;
    EVX_PLANE_SIZES(X)
#undef X
    default:
      return fail(EVX_ERR_UNSUPPORTED, "no plane sweep of %d points", n);
  }
  return check_launch("plane_inv");
}

template int plane_run_fwd<float>(int, const void*, const float*, cpx<float>*, int64_t, hipStream_t);
template int plane_run_fwd<double>(int, const void*, const double*, cpx<double>*, int64_t, hipStream_t);
template int plane_run_inv<float>(int, const void*, const cpx<float>*, float*, const float*, double, int64_t, SumRec*,
                                  hipStream_t);
template int plane_run_inv<double>(int, const void*, const cpx<double>*, double*, const double*, double, int64_t,
                                   SumRec*, hipStream_t);

}  // namespace evx
