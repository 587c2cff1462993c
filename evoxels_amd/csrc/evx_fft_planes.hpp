// Whole-plane sweeps (evx_fft_planes.hip): z R2C and forward y, or inverse y and
// z C2R, of an x-plane of N x N points in one block, with the half-spectrum plane in
// LDS, so that the spectrum crosses memory once instead of three times.
#pragma once
#include "evx_common.hpp"
#include "evx_fft_engine.hpp"
#include "evx_fft_tiles.hpp"
#include "evx_sum.hpp"

namespace evx {

// Radices and values per thread of a plane's lines.
template <int N> struct PlaneSpec;
template <> struct PlaneSpec<32>  { using R = Rad<4, 8>;    static constexpr int E = 8; };
template <> struct PlaneSpec<48>  { using R = Rad<12, 4>;   static constexpr int E = 12; };
template <> struct PlaneSpec<64>  { using R = Rad<8, 8>;    static constexpr int E = 8; };
template <> struct PlaneSpec<96>  { using R = Rad<6, 4, 4>; static constexpr int E = 12; };
template <> struct PlaneSpec<100> { using R = Rad<10, 10>;  static constexpr int E = 10; };
template <> struct PlaneSpec<128> { using R = Rad<16, 8>;   static constexpr int E = 16; };
#define EVX_PLANE_SIZES(X) X(32) X(48) X(64) X(96) X(100) X(128)

#define X(N)                                                                                            \
  static_assert(rad_product(PlaneSpec<N>::R{}) == N && rad_divides<PlaneSpec<N>::E>(PlaneSpec<N>::R{}), \
                "radix plan of size " #N);
EVX_PLANE_SIZES(X)
#undef X

template <typename T, int N>
struct PGeo {
  static constexpr int E = PlaneSpec<N>::E, TPL = N / E, NH = N / 2 + 1;
  static constexpr int LINE = N + N / 16;  // padded exchange line (line_slot)
  // rows hold NH values, one spare column for idle threads and half an exchange line
  static constexpr int PITCH = NH + 1 > (LINE + 1) / 2 ? NH + 1 : (LINE + 1) / 2;
  static constexpr int ROWS = N + 2;  // two spare rows for idle threads
  static constexpr int THREADS = (NH * TPL + 63) / 64 * 64;
  static constexpr bool WAVE = 64 % TPL == 0;  // a pair's threads share a wavefront
  static constexpr size_t LDS = sizeof(cpx<T>) * (N + (size_t)ROWS * PITCH);
  static_assert(N / 2 * TPL <= THREADS && THREADS <= 1024, "one round of threads");
};


// Whether the steps of a grid run their z and y sweeps plane by plane: ny = nz,
// one of the lengths whose plane fits LDS in both types (128 takes 143 of
// 160 KB in float64) and whose N/2 line pairs give a block a plane's work in
// one round of threads.  Separate sweeps against planes, the semi-implicit
// step (MI355X, microseconds): 32^3 float32 27.2 / 19.6, 8 x 48^3 float64
// 45.4 / 28.5, 96^3 float32 40.7 / 31.7, 100^3 float64 50.7 / 42.4,
// 128^3 float32 50.9 / 42.2, 4 x 128^3 float64 163.4 / 139.2, 16 x 128^3
// float32 368.5 / 286.7.  8 and 16 keep separate sweeps: a plane of them
// leaves most of a block idle.  A float64 plane of 128 takes a whole CU and 35 us
// for both sweeps however few there are, so it needs 48 of them: separate sweeps
// / planes of n x 128^2 float64 take 28.9 / 33.2 us at n = 16, 33.6 / 34.5 at 32,
// 38.4 / 35.2 at 64, 52.9 / 38.9 at 128.  The others win from the first plane on
// (8 x 96^2 float64 36.7 / 26.8, 16 x 128^2 float32 27.7 / 22.6).
bool plane_sweeps_apply(int dtype, const Dims& d);

// Planes 0 .. nplanes-1 of N x N points; twg: the N roots of unity.  With rec, the
// inverse writes rec[plane]: the compensated float64 sum of its outputs and
// their NaN / Inf flags.
template <typename T>
int plane_run_fwd(int n, const void* twg, const T* x, cpx<T>* spec, int64_t nplanes, hipStream_t s);
template <typename T>
int plane_run_inv(int n, const void* twg, const cpx<T>* spec, T* out, const T* base, double scale, int64_t nplanes,
                  SumRec* rec, hipStream_t s);

}  // namespace evx
