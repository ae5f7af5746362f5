/*
 * gp_common.h -- device layout constants and helpers shared by the step kernels.
 */
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gpk {

constexpr int kYOff = 61; /* element offset of y = 0 inside a row: y = 3 lands on a 64-element boundary */

/* halo index maps of the two fields (0 phi, 1 mu): source x/y of allocated x/y = 0,1,2, m+3, m+4, m+5 */
struct Maps {
  int32_t sx[2][6], sy[2][6];
  int32_t hx[6], hy[6];
};

/* An interior cell is copied to every halo cell whose proxy it is (apply_boundary_conditions as a scatter):
 * X in {x} u {halo x with source x}, Y likewise, all (X, Y) but (x, y). */
template <typename R>
__device__ __forceinline__ void write_images(R *__restrict__ base, int ncomp, const R *vals, int f, const Maps &mp,
                                             int64_t x, int64_t y, int64_t fs, int64_t ps) {
  int64_t X[3], Y[3];
  int nx = 1, ny = 1;
  X[0] = x;
  Y[0] = y;
  for (int k = 0; k < 6; k++) {
    if (mp.sx[f][k] == x && nx < 3) X[nx++] = mp.hx[k];
    if (mp.sy[f][k] == y && ny < 3) Y[ny++] = mp.hy[k];
  }
  for (int i = 0; i < nx; i++)
    for (int j = 0; j < ny; j++) {
      if (i == 0 && j == 0) continue;
      const int64_t c = X[i] * ps + Y[j] + kYOff;
      for (int a = 0; a < ncomp; a++) base[a * fs + c] = vals[a];
    }
}

/* Wavefront sums over the 64 lanes, returned to every lane. DPP steps keep the data in the
 * VALU (no LDS round trips): quad_perm [1,0,3,2] and [2,3,0,1], row_half_mirror and row_mirror reduce each
 * 16-lane row; row_bcast:15 (rows 1, 3) and row_bcast:31 (rows 2, 3) combine the rows, leaving the result in
 * lane 63. Lanes that a masked step does not write receive the operation's identity. */
namespace dpp {
constexpr int kQuad1032 = 0xB1, kQuad2301 = 0x4E, kRowHalfMirror = 0x141, kRowMirror = 0x140, kRowBcast15 = 0x142,
              kRowBcast31 = 0x143;
template <int CTRL, int ROWMASK>
__device__ __forceinline__ double mov(double v, double identity) {
  const long long b = __double_as_longlong(v), id = __double_as_longlong(identity);
  const int lo = __builtin_amdgcn_update_dpp((int)(id & 0xffffffffll), (int)(b & 0xffffffffll), CTRL, ROWMASK, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(id >> 32), (int)(b >> 32), CTRL, ROWMASK, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double lane63(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), 63), hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
template <int CTRL, int ROWMASK>
__device__ __forceinline__ int mov(int v, int identity) {
  return __builtin_amdgcn_update_dpp(identity, v, CTRL, ROWMASK, 0xf, false);
}
__device__ __forceinline__ int lane63(int v) { return __builtin_amdgcn_readlane(v, 63); }
template <class T, class Op>
__device__ __forceinline__ T reduce(T v, T identity, Op op) {
  v = op(v, mov<kQuad1032, 0xf>(v, identity));
  v = op(v, mov<kQuad2301, 0xf>(v, identity));
  v = op(v, mov<kRowHalfMirror, 0xf>(v, identity));
  v = op(v, mov<kRowMirror, 0xf>(v, identity));
  v = op(v, mov<kRowBcast15, 0xa>(v, identity));
  v = op(v, mov<kRowBcast31, 0xc>(v, identity));
  return lane63(v);
}
}  // namespace dpp

__device__ __forceinline__ double wave_sum(double v) {
  return dpp::reduce<double>(v, 0.0, [](double a, double b) { return a + b; });
}
__device__ __forceinline__ int wave_sum(int v) {
  return dpp::reduce<int>(v, 0, [](int a, int b) { return a + b; });
}

/* Many wavefront reductions at once. Reduced one by one, M values take M times six steps of two registers; here the
 * first step (v_permlane32_swap) halves the lanes and packs two values into one register, the second
 * (v_permlane16_swap) two of those, and the four steps within a row of 16 lanes then work on four values at a time:
 * 16 statistics take about 130 instructions instead of 650, and leave with one store each for the extrema and the sums.
 * out[j] holds value 4 j + row_value(lane) of v in every lane of a row. op must not care about the order. */
__device__ __forceinline__ int row_value(int lane) { return ((lane >> 5) & 1) | ((lane >> 3) & 2); }
namespace dpp {
template <int HALF>
__device__ __forceinline__ void swap_words(unsigned &a, unsigned &b) {
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  u2 r;
  if constexpr (HALF == 32) r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  else r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r.x;
  b = r.y;
}
/* HALF 32: a's upper half of the lanes against b's lower half; 16: a's odd rows against b's even rows */
template <int HALF>
__device__ __forceinline__ void swap(double &a, double &b) {
  const uint64_t x = (uint64_t)__double_as_longlong(a), y = (uint64_t)__double_as_longlong(b);
  unsigned al = (unsigned)x, ah = (unsigned)(x >> 32), bl = (unsigned)y, bh = (unsigned)(y >> 32);
  swap_words<HALF>(al, bl);
  swap_words<HALF>(ah, bh);
  a = __longlong_as_double((long long)(((uint64_t)ah << 32) | al));
  b = __longlong_as_double((long long)(((uint64_t)bh << 32) | bl));
}
template <int HALF>
__device__ __forceinline__ void swap(float &a, float &b) {
  unsigned x = __float_as_uint(a), y = __float_as_uint(b);
  swap_words<HALF>(x, y);
  a = __uint_as_float(x);
  b = __uint_as_float(y);
}
/* v of another lane of the row (every lane has a source in these patterns) */
template <int CTRL>
__device__ __forceinline__ double row_mov(double v) {
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)b, CTRL, 0xf, 0xf, true);
  const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
template <int CTRL>
__device__ __forceinline__ float row_mov(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
}  // namespace dpp
template <int M, typename T, class Op>
__device__ __forceinline__ void wave_reduce(const T (&v)[M], T (&out)[(M + 3) / 4], Op op) {
  constexpr int H = (M + 1) / 2, Q = (M + 3) / 4;
  T u[2 * Q];
#pragma unroll
  for (int j = 0; j < H; j++) {
    T a = v[2 * j], b = v[2 * j + 1 < M ? 2 * j + 1 : 2 * j];
    dpp::swap<32>(a, b);
    u[j] = op(a, b);
  }
  if (H < 2 * Q) u[2 * Q - 1] = u[H - 1];
#pragma unroll
  for (int j = 0; j < Q; j++) {
    T a = u[2 * j], b = u[2 * j + 1];
    dpp::swap<16>(a, b);
    T t = op(a, b);
    t = op(t, dpp::row_mov<dpp::kQuad1032>(t));
    t = op(t, dpp::row_mov<dpp::kQuad2301>(t));
    t = op(t, dpp::row_mov<dpp::kRowHalfMirror>(t));
    out[j] = op(t, dpp::row_mov<dpp::kRowMirror>(t));
  }
}
/* extrema of values that are not signalling NaNs (results of arithmetic): fmax without the quieting of its operands. The two
 * wait states stand for the ones a lane-crossing read of a just-written register needs, which the compiler counts for its
 * own instructions only. */
__device__ __forceinline__ double max_val(double a, double b) {
#if defined(__AMDGCN__)
  double r;
  asm("v_max_f64 %0, %1, %2\n\ts_nop 1" : "=v"(r) : "v"(a), "v"(b));
  return r;
#else
  return fmax(a, b);
#endif
}
__device__ __forceinline__ float max_val(float a, float b) {
#if defined(__AMDGCN__)
  float r;
  asm("v_max_f32 %0, %1, %2\n\ts_nop 1" : "=v"(r) : "v"(a), "v"(b));
  return r;
#else
  return fmaxf(a, b);
#endif
}
/* The statistics of a wavefront's lanes (layout of stats_init: extrema of phi and mu first, then the sums), reduced:
 * put(i, value) is called once for every statistic i, by one lane each. Extrema reduce in the statistics' own precision
 * (exact; a minimum as the maximum of the negated values), sums in FP64. PHI_SUMS_ZERO: the squared phi increments are
 * +0 on every lane, and so are their sums. more: unless NULL, second sums of the lane's squared mu increments. */
template <int N, int NC, bool PHI_SUMS_ZERO, int NSA, typename R, class F>
__device__ __forceinline__ void stats_reduce(const R (&st)[NSA], int lane, F put, const R *more = nullptr) {
  constexpr int ME = 2 * N + 2 * NC, S0 = PHI_SUMS_ZERO ? 3 * N + 2 * NC : ME, MS = NSA - S0;
  constexpr int QE = (ME + 3) / 4, QS = (MS + 3) / 4;
  const auto is_min = [](int i) { return (i >= N && i < 2 * N) || i >= 2 * N + NC; };
  R e[ME], te[QE];
  double v[MS], ts[QS];
#pragma unroll
  for (int i = 0; i < ME; i++) e[i] = is_min(i) ? -st[i] : st[i];
#pragma unroll
  for (int i = 0; i < MS; i++) v[i] = (double)st[S0 + i];
  if (more) {
#pragma unroll
    for (int k = 0; k < NC; k++) v[3 * N + 2 * NC - S0 + k] += (double)more[k];
  }
  wave_reduce(e, te, [](R a, R b) { return max_val(a, b); });
  wave_reduce(v, ts, [](double a, double b) { return a + b; });
  /* lane q of a row stores its j = q value, so that each group leaves in one store */
  const int q = lane & 15, i = 4 * q + row_value(lane);
  R x = te[0];
  double y = ts[0];
#pragma unroll
  for (int j = 1; j < QE; j++) x = q == j ? te[j] : x;
#pragma unroll
  for (int j = 1; j < QS; j++) y = q == j ? ts[j] : y;
  if (i < ME) put(i, (double)(is_min(i) ? -x : x));
  if (i < MS) put(S0 + i, y);
  if (PHI_SUMS_ZERO && i < N) put(ME + i, 0.0);
}

}  // namespace gpk
