/*
 * gp_pack.h -- states between the host's layout (halo-inclusive FP64 planes, rows_x x rows_y, y fastest) and the device
 * planes (row pitch ps, kYOff leading elements, the stored precision).
 *
 * The host's rows cross the bus as they are and the kernels here lay them out, encode or decode them: on the host that
 * was a copy of the state, a second one in the device layout and a conversion per element, single-threaded, three to ten
 * times the transfer (4096^2 compensated, 671 MB: 337 ms up and 220 ms down). The kernels are memory-bound and take a few
 * hundred microseconds of such a state. Planes are whole rows one after another on both sides (fs = rows_x ps), so a run of
 * rows may cross planes: row g of a field is row g mod rows_x of component g / rows_x.
 */
#pragma once

#include "gp_common.h"
#include "gp_model.h"

namespace gpk {

/* how a field's values are stored */
enum PackForm { PACK_F64, PACK_F32, PACK_DF, PACK_C32 };

/* rows [row0, row0 + nrows) of a field from src (their values, ry a row) into the planes d0 and, unless it is NULL, d1 (the
 * second state buffer); PACK_DF / PACK_C32 with the second parts in l0 and l1. The pitch's padding is set to zero. */
template <int FORM>
__global__ __launch_bounds__(256) void k_pack(const double *__restrict__ src, void *__restrict__ d0, void *__restrict__ d1,
                                              void *__restrict__ l0, void *__restrict__ l1, int64_t row0, int64_t nrows,
                                              int64_t ry, int64_t ps) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x, y = e - kYOff;
  if (e >= ps) return;
  for (int64_t r = blockIdx.y; r < nrows; r += gridDim.y) {
    const double v = y >= 0 && y < ry ? src[r * ry + y] : 0.0;
    const int64_t o = (row0 + r) * ps + e;
    if constexpr (FORM == PACK_F64) {
      ((double *)d0)[o] = v;
      if (d1) ((double *)d1)[o] = v;
    } else if constexpr (FORM == PACK_F32) {
      ((float *)d0)[o] = (float)v;
      if (d1) ((float *)d1)[o] = (float)v;
    } else if constexpr (FORM == PACK_DF) {
      float hi, lo;
      df_encode(v, hi, lo);
      ((float *)d0)[o] = hi;
      ((float *)l0)[o] = lo;
      if (d1) {
        ((float *)d1)[o] = hi;
        ((float *)l1)[o] = lo;
      }
    } else {
      float hi;
      int8_t q;
      c32_encode(v, hi, q);
      ((float *)d0)[o] = hi;
      ((int8_t *)l0)[o] = q;
      if (d1) {
        ((float *)d1)[o] = hi;
        ((int8_t *)l1)[o] = q;
      }
    }
  }
}

/* rows [row0, row0 + nrows) of a field into dst (ry values a row), decoded */
template <int FORM>
__global__ __launch_bounds__(256) void k_unpack(double *__restrict__ dst, const void *__restrict__ s,
                                                const void *__restrict__ l, int64_t row0, int64_t nrows, int64_t ry,
                                                int64_t ps) {
  const int64_t y = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (y >= ry) return;
  for (int64_t r = blockIdx.y; r < nrows; r += gridDim.y) {
    const int64_t o = (row0 + r) * ps + y + kYOff;
    double v;
    if constexpr (FORM == PACK_F64) v = ((const double *)s)[o];
    else if constexpr (FORM == PACK_F32) v = (double)((const float *)s)[o];
    else if constexpr (FORM == PACK_DF) v = df_decode(((const float *)s)[o], ((const float *)l)[o]);
    else v = c32_decode(((const float *)s)[o], ((const int8_t *)l)[o]);
    dst[r * ry + y] = v;
  }
}

/* The boundary copies of an uploaded field f: halo rows from the rows of the maps, then halo columns over every row, as
 * one gather, since every source lies in the interior. One thread per halo cell (the six halo rows over the full width,
 * then the six halo cells of each interior row), blockIdx.y the component. */
template <typename T>
__global__ __launch_bounds__(256) void k_pack_halo(T *__restrict__ d0, T *__restrict__ d1, Maps maps, int f, int64_t fs,
                                                   int64_t ps, int64_t mx, int64_t my) {
  const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x, ry = my + 6, nrow = 6 * ry;
  if (j >= nrow + 6 * mx) return;
  int64_t X, Y;
  if (j < nrow) {
    const uint32_t r = (uint32_t)j / (uint32_t)ry;
    X = r < 3u ? (int64_t)r : mx + r;
    Y = j - r * ry;
  } else {
    const uint32_t k = (uint32_t)(j - nrow), row = k / 6u, q = k - 6u * row;
    Y = q < 3u ? (int64_t)q : my + q;
    X = 3 + (int64_t)row;
  }
  int64_t sx = X, sy = Y;
#pragma unroll
  for (int k = 0; k < 6; k++) {
    sx = maps.hx[k] == X ? maps.sx[f][k] : sx;
    sy = maps.hy[k] == Y ? maps.sy[f][k] : sy;
  }
  const int64_t o = blockIdx.y * fs + X * ps + Y + kYOff, s = blockIdx.y * fs + sx * ps + sy + kYOff;
  d0[o] = d0[s];
  if (d1) d1[o] = d1[s];
}

}  // namespace gpk
