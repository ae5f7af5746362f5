/*
 * gp_cells.h -- the update part of the step as a pair of cell-classified kernels (the default path).
 *
 * Every interior cell is either a bulk cell or an interface cell. A bulk cell's radius-2 diamond of phase codes
 * (the 13 cells within Manhattan distance 2) is purely one phase b: then it and its four neighbours are not
 * delta-phi candidates (delta-phi exactly 0), every anti-trapping current on its faces returns +0, every mobility
 * it reads is Mpure[b], and its update is the pure-phase arithmetic of phase b. Every other interior cell is an
 * interface cell.
 *
 * k_cbulk updates the bulk cells of a tile (124-cell y-strip x SEG x-rows, one wavefront, two adjacent cells per
 * lane): it streams the mu rows through a ring of registers and forms, per cell, the same operations in the same order
 * as the pure-phase step and k_bulk, so the results are bit-identical. A tile whose staged codes are all one phase
 * takes that phase as a scalar. The other tiles classify their cells with one bit per row in each lane and run
 * the row loop once per phase that has bulk cells. phi of a bulk cell is e_b; when the output buffer already holds e_b
 * there (the cell was purely b two states back) it is not rewritten.
 * k_cbulk also appends the interface cells and the delta-phi candidates of its tile to two global lists (one atomic
 * per mixed tile);
 * k_ilist runs the general per-cell update (gp_model.h: jat_x, jat_y, mu_update -- bit-identical to the
 * reference by construction) on the listed cells in a grid-stride loop, so that every lane of every wavefront
 * works on an interface cell (a march row has about one in five) and no wavefront holds more than its share.
 * Every interior cell is written by exactly one of the two. They read the phase codes of the current state and
 * write those of the new one (a second buffer). The halo of the new state is filled along the way (halo_cell).
 */
#pragma once

#include "gp_march.h"

namespace gpk {

constexpr int kCellOut = 124;  /* output cells of a k_cbulk strip: 64 lanes x 2 cells less two on either side */
constexpr int kCellSegMax = 16; /* longest x-segment of k_cbulk (instantiated for 16 and kCellSegMin rows) */
constexpr int kCellSegMin = 4;
/* Tiles from which k_cbulk takes the long segments: about one wavefront per SIMD. Below it the rows of a tile in turn are
 * the step's critical path; above it the short segments' doubled prologue costs more than it hides. Measured with
 * statistics, ternary n^2, short / long segments in us (long tiles):
 *            1024 (576)    1280 (880)    1408 (1056)   1600 (1300)   2048 (2176)   2560 (3360)
 *   FP32     18.5 / 23.3   24.2 / 24.9   27.3 / 27.2   32.5 / 29.2   41.7 / 35.4   59.4 / 45.3
 *   FP32C    20.3 / 27.7   26.9 / 29.4   30.5 / 33.1   33.6 / 35.5   43.9 / 43.4   61.9 / 58.0
 *   FP64     24.1 / 36.2   31.9 / 37.4   32.8 / 41.7   37.9 / 46.5   48.6 / 62.3   68.3 / 83.9
 * The line is FP32's. FP32C's would lie at about 2000 tiles, and FP64 (161-175 registers with long segments, 140-158 with
 * short ones) does not reach its own by 2560^2. */
constexpr int kCellFill = 1024;
constexpr int kPadOut = 60, kPadSeg = 16; /* tiles of the statistics' padding rows (pad_stats) */

/* a wave-uniform value read as a scalar: a per-lane choice among such values then stays a register select */
__device__ __forceinline__ float scalar_val(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

/* FP32 bulk cells take the closed form through Model::Kbulk; FP64 keeps the reference's operations (bit-exact) */
template <typename R>
constexpr bool kLeanBulk = sizeof(R) < sizeof(double);

/* The pure-phase update of one cell from mu of the cell, m1, and of its neighbours m0 (x-1), m2 (x+1), muu (y-1) and
 * mud (y+1): the new mu and its increment.
 * FP32: the closed form dmu = K . lap(mu), K = Kbulk of the cell's phase (equal in exact arithmetic to the flux
 * divergence through Mpure followed by Mu_lin; the anti-trapping divergence is a signed zero). The second differences
 * are formed from first differences, so their rounding is relative to the increment, as in the flux form. */
template <int NC>
__device__ __forceinline__ void bulk_update_lean(const Model<float> &m, const float (*K)[NC], const float *m0,
                                                 const float *m1, const float *m2, const float *mud, const float *muu,
                                                 float *munew, float *deltamu) {
  float lap[NC];
#pragma unroll
  for (int l = 0; l < NC; l++) {
    const float gx = (m2[l] - m1[l]) - (m1[l] - m0[l]);
    const float gy = (mud[l] - m1[l]) - (m1[l] - muu[l]);
    lap[l] = __builtin_fmaf(gx, m.lap_x, gy * m.lap_y);
  }
#pragma unroll
  for (int k = 0; k < NC; k++) {
    float s = K[k][0] * lap[0];
#pragma unroll
    for (int l = 1; l < NC; l++) s = __builtin_fmaf(K[k][l], lap[l], s);
    deltamu[k] = s;
    munew[k] = m1[k] + s;
  }
}
/* FP64: the reference's operations, phase b wave-uniform (its coefficients are scalars) */
template <int N, int NC, typename R, bool P2>
__device__ __forceinline__ void bulk_update_ref(const Model<R> &m, int b, const R *m0, const R *m1, const R *m2,
                                                const R *mud, const R *muu, R divjat0, R *munew, R *deltamu) {
  using Vw = View<R, P2, false, kFastOf<R>>;
  R c_new[NC];
#pragma unroll
  for (int k = 0; k < NC; k++) {
    R divflux = R(0.0);
#pragma unroll
    for (int l = 0; l < NC; l++) {
      const R Mb = m.Mpure[b][k][l];
      const R Fb = Mb * divx<Vw>(m, (m1[l] - m0[l]));
      const R Ff = Mb * divx<Vw>(m, (m2[l] - m1[l]));
      const R Fy = Mb * divy<Vw>(m, (mud[l] - m1[l]));
      const R Fyl = Mb * divy<Vw>(m, (m1[l] - muu[l])); /* = Fy of the cell below, bit for bit */
      divflux += divx<Vw>(m, (Ff - Fb));
      divflux += divy<Vw>(m, (Fy - Fyl));
    }
    c_new[k] = c_mu<NC>(m, m1, b, k) + m.dt * (divflux)-divjat0;
  }
#pragma unroll
  for (int k = 0; k < NC; k++) {
    munew[k] = Mu<NC>(m, c_new, b, k);
    deltamu[k] = munew[k] - m1[k];
  }
}

/* the mu statistics of one bulk cell: delta-phi is 0 and phi = e_b, so the squared increments of phi add +0 to sums
 * that start at +0 and e_b is finite; the extrema of phi follow from the phases seen (bulk_seen_fold). sum: where the
 * squared increments of mu add up (st + 3 N + 2 NC, or a lane's second sums) */
template <int N, int NC, typename R, int NSA>
__device__ __forceinline__ void bulk_stats(R (&st)[NSA], R *sum, const R *munew, const R *deltamu) {
#pragma unroll
  for (int k = 0; k < NC; k++) {
    st[2 * N + k] = fmax(st[2 * N + k], munew[k]);
    st[2 * N + NC + k] = fmin(st[2 * N + NC + k], munew[k]);
    sum[k] += deltamu[k] * deltamu[k];
    if (!isfinite(munew[k])) st[NSA - 1] += R(1.0);
  }
}

/* the phi extrema of a lane's bulk cells of the phases in `seen` (bit b: a cell equal to e_b) into st: over such
 * cells phi_a is 1 where b = a and 0 elsewhere */
template <int N, typename R, int NSA>
__device__ __forceinline__ void bulk_seen_fold(R (&st)[NSA], unsigned seen) {
#pragma unroll
  for (int a = 0; a < N; a++) {
    const bool own = (seen >> a) & 1u, other = (seen & ~(1u << a)) != 0u;
    if (own) st[a] = fmax(st[a], R(1.0));
    else if (other) st[a] = fmax(st[a], R(0.0));
    if (other) st[N + a] = fmin(st[N + a], R(0.0));
    else if (own) st[N + a] = fmin(st[N + a], R(1.0));
  }
}

/* mu rows in flight ahead of the row after the current one; kCellRing = depth + 2 register slots hold rows x-1, x,
 * x+1 and those in flight, and divides the tile's rows */
constexpr int kCellDepth = 2;
constexpr int kCellRing = kCellDepth + 2;
static_assert(kCellSegMin % kCellRing == 0 && kCellSegMax % kCellRing == 0 && kCellSegMax + 4 <= 32,
              "a tile is whole turns of the ring, and its staged rows fit one 32-bit mask");

/* k_cbulk keeps its row offsets in 32 bits. The largest it forms is the refill offset of the last tile: row
 * x + D + 1 for a row x <= xb + RG - 1 of the unrolled ring (rows past xb run on clamped rows), i.e. below
 * (xb + RG + D + 1) ps with xb <= mesh_x + 2, before it is clamped to row xb + 1; the in-row offset adds less than
 * ps. A grid takes the cells path only when all of these fit: (rows_x + kCellSlack) * ps <= INT32_MAX. */
constexpr int kCellSlack = 32;
static_assert(kCellRing + kCellDepth + 1 <= kCellSlack - 4, "the cells path's 32-bit offset bound needs a larger slack");
__host__ __device__ constexpr bool cells_fit(int64_t rows_x, int64_t ps) {
  return (rows_x + kCellSlack) * ps <= (int64_t)0x7fffffff;
}

/* Append to the two lists of a step: counts holds their lengths (interface cells, delta-phi candidates) as one 64-bit
 * word, so that a wavefront reserves its entries in both with one atomic. */
__device__ __forceinline__ uint64_t list_reserve(int *counts, int ni, int nc) {
  return atomicAdd((unsigned long long *)counts, (unsigned long long)ni | ((unsigned long long)nc << 32));
}

/* Delta-phi candidates on the ring x or y in {2, mesh+3} around the interior (k_cbulk's tiles list the interior
 * ones): ring cell i (one per thread of k_cbulk's extra blocks), appended to the same list. */
__device__ __forceinline__ void dring_cell(int64_t i, const int8_t *__restrict__ codes, int32_t *__restrict__ clist,
                                           int *counts, int64_t ps, int64_t mx, int64_t my) {
  const int lane = threadIdx.x & 63;
  const int64_t nxr = my + 2, nyr = mx; /* rows x = 2, mx+3 over y in [2, my+3]; columns y = 2, my+3 over x in [3, mx+2] */
  int64_t x = -1, y = -1;
  if (i < 2 * nxr) {
    x = (i < nxr) ? 2 : mx + 3;
    y = 2 + (i < nxr ? i : i - nxr);
  } else if (i < 2 * nxr + 2 * nyr) {
    const int64_t k = i - 2 * nxr;
    y = (k < nyr) ? 2 : my + 3;
    x = 3 + (k < nyr ? k : k - nyr);
  }
  bool cand = false;
  const int64_t c = x * ps + y + kYOff;
  if (x >= 0) {
    const int8_t k0 = codes[c], k1 = codes[c - ps], k2 = codes[c + ps], k3 = codes[c - 1], k4 = codes[c + 1];
    cand = (k0 < 0) | (k1 != k0) | (k2 != k0) | (k3 != k0) | (k4 != k0);
  }
  const uint64_t mask = __ballot(cand);
  if (!mask) return;
  const int leader = __ffsll((long long)mask) - 1;
  int base = 0;
  if (lane == leader) base = (int)(list_reserve(counts, 0, __popcll(mask)) >> 32);
  base = __shfl(base, leader);
  if (cand) clist[base + __popcll(mask & ((1ull << lane) - 1ull))] = (int32_t)c;
}

/* Element i of a row at the wave-uniform address p: a scalar base plus an unsigned 32-bit byte offset per lane, the
 * addressing mode of the global instructions. The base goes through an empty asm so that the compiler keeps that form: left
 * to itself it adds the lane's offset first and holds a 64-bit vector address per plane. */
template <typename T, typename E>
__device__ __forceinline__ T row_ld(const E *p, unsigned i) {
#if defined(__AMDGCN__)
  uint64_t b = (uint64_t)p;
  asm("" : "+s"(b));
  return *(const __attribute__((address_space(1))) T *)(b + (uint64_t)(i * (unsigned)sizeof(E)));
#else
  return *(const T *)(p + i);
#endif
}
template <typename T, typename E>
__device__ __forceinline__ void row_st(E *p, unsigned i, T v) {
#if defined(__AMDGCN__)
  uint64_t b = (uint64_t)p;
  asm("" : "+s"(b));
  *(__attribute__((address_space(1))) T *)(b + (uint64_t)(i * (unsigned)sizeof(E))) = v;
#else
  *(T *)(p + i) = v;
#endif
}

/* two adjacent cells of a row, the first (x) at an even element offset */
template <typename R>
struct PairOf;
template <>
struct PairOf<float> {
  typedef float type __attribute__((ext_vector_type(2)));
};
template <>
struct PairOf<double> {
  typedef double type __attribute__((ext_vector_type(2)));
};
template <typename R>
using Pair = typename PairOf<R>::type;
/* their phase codes, zero-extended: the first in the low byte, the second in the high one */
__device__ __forceinline__ unsigned code_pair(const int8_t *row, unsigned i) { return row_ld<uint16_t>(row, i); }

/* Row classes of a lane's two columns over the staged rows, one bit per row (bit r: staged row r): bulk cells of every
 * phase, and cells whose five-point codes are uniform (no delta-phi candidate). Vertical neighbours are shifts of
 * the column's mask, horizontal ones the other column of the lane or a DPP move of the neighbour lane's masks: about
 * 25 VALU instructions per phase for all rows of the tile, where the code-by-code test reads 13 codes per cell. */
template <int N>
struct TileMasks {
  uint32_t be[N], bo[N]; /* bulk cells of phase b in the first / second column */
  uint32_t ue, uo;       /* cells with uniform five-point codes */
};
template <int N, int ROWS>
__device__ __forceinline__ TileMasks<N> tile_masks(const unsigned (&cv)[ROWS]) {
  TileMasks<N> t;
  t.ue = t.uo = 0u;
#pragma unroll
  for (int b = 0; b < N; b++) {
    uint32_t e = 0u, o = 0u;
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
      e |= ((cv[r] & 0xffu) == (unsigned)b ? 1u : 0u) << r;
      o |= ((cv[r] >> 8) == (unsigned)b ? 1u : 0u) << r;
    }
    const uint32_t el = (uint32_t)lane_up((int)e), er = (uint32_t)lane_dn((int)e);
    const uint32_t ol = (uint32_t)lane_up((int)o), or_ = (uint32_t)lane_dn((int)o);
    auto v1 = [](uint32_t c) { return c & (c << 1) & (c >> 1); };
    const uint32_t e1 = v1(e), o1 = v1(o);
    t.be[b] = e1 & (e << 2) & (e >> 2) & o1 & v1(ol) & el & er;
    t.bo[b] = o1 & (o << 2) & (o >> 2) & e1 & v1(er) & ol & or_;
    t.ue |= e1 & o & ol;
    t.uo |= o1 & e & er;
  }
  return t;
}

/* The statistics of the padding rows: a known defect that is kept. The reported extrema and sums of squared increments of
 * mu include, on a grid whose rows are not a multiple of four, up to three rows past mesh+2 for the tiles of kPadOut cells
 * by kPadSeg rows at the grid's end whose cells and neighbours are all of one phase: the updates of row mesh+3 with itself
 * as the row above (and, after the first, below). They came from a step whose uniform tiles ran their padding rows into
 * the statistics, belong to no cell and can make rel_change_mu a few percent too large (gp_stats); without them the
 * figure of every such run would change. One wavefront per strip s; returns its partials through st. */
template <int N, int NC, typename R, bool P2, bool C, int NSA>
__device__ __forceinline__ void pad_stats(const Model<R> &m, const R *__restrict__ mu, const int8_t *__restrict__ mlo,
                                          const int8_t *__restrict__ codes, int s, int64_t fs, int64_t ps, int64_t mx,
                                          int64_t my, R divjat0, R (&st)[NSA]) {
  const int lane = threadIdx.x & 63;
  const int64_t y = 3 + (int64_t)s * kPadOut - 2 + lane, ry = my + 6, c0 = (y < ry - 1 ? y : ry - 1) + kYOff;
  const int64_t xb = mx + 2, xa = 3 + (mx - 1) / kPadSeg * kPadSeg;
  const int b = codes[(xa - 2) * ps + c0];
  bool same = b >= 0;
  for (int64_t x = xa - 1; x <= xb + 2; x++) same = same & (codes[x * ps + c0] == b);
  const int b0 = __builtin_amdgcn_readfirstlane(b);
  if (!__all(same && b == b0)) return;
  R m0[NC], m1[NC], up[NC], dn[NC], mn[NC], dm[NC];
#pragma unroll
  for (int k = 0; k < NC; k++) {
    m0[k] = mu[k * fs + xb * ps + c0];
    m1[k] = mu[k * fs + (xb + 1) * ps + c0];
    up[k] = lane_up(m1[k]);
    dn[k] = lane_dn(m1[k]);
  }
  const bool out = lane >= 2 && lane <= 61 && y <= my + 2;
  for (int64_t i = mx % 4; i < 4; i++) {
    if constexpr (kLeanBulk<R>) {
      R K[NC][NC];
#pragma unroll
      for (int k = 0; k < NC; k++)
#pragma unroll
        for (int l = 0; l < NC; l++) K[k][l] = m.Kbulk[b0][k][l];
      bulk_update_lean<NC>(m, K, m0, m1, m1, dn, up, mn, dm);
    } else {
      bulk_update_ref<N, NC, R, P2>(m, b0, m0, m1, m1, dn, up, divjat0, mn, dm);
    }
#pragma unroll
    for (int k = 0; k < NC; k++) {
      if constexpr (C) {
        float hn;
        int8_t qn;
        c32_encode(c32_decode((float)m1[k], mlo[k * fs + (xb + 1) * ps + c0]) + (double)dm[k], hn, qn);
        mn[k] = (R)hn;
      }
      m0[k] = m1[k];
    }
    if (out) bulk_stats<N, NC>(st, st + 3 * N + 2 * NC, mn, dm);
  }
}

/* Two cells per lane and no LDS: a wavefront has 512 B (FP32) or 1 KiB (FP64) per load in flight, neighbouring lanes meet by
 * one DPP move per two cells, and a strip re-reads 4 of 128 columns where one cell per lane re-reads 4 of 64. Bound by
 * VALU issue and memory together: 4096^2 compensated with statistics 118 us a step over a run (137 with one cell per
 * lane, codes in LDS), about 480 MB; FP32 2047 x 1801 30 us (45). FP64 at that size gains nothing: 190 us (193), although
 * it moves 9% less (670 MB): 175 registers leave two wavefronts per SIMD. On small grids it is one tile's latency:
 * 48 x 40 ternary FP64 13 us with 4-row segments (39 with 16-row ones and the cell-by-cell test), 200^2 binary 9 (30). */
template <int N, int NC, typename R, bool P2, bool STATS, int SEG, bool C = false>
__global__ __launch_bounds__(256) void k_cbulk(const Model<R> *__restrict__ mp, const R *__restrict__ mu, const int8_t *__restrict__ codes_in,
             R *__restrict__ phi_o, R *__restrict__ mu_o, int8_t *__restrict__ codes_out,
             double *__restrict__ partials, int64_t pstride, int64_t fs, int64_t ps, int64_t mx, int64_t my,
             int nstrips, int nwaves, int keep, const int8_t *__restrict__ tin, int8_t *__restrict__ tout,
             int32_t *__restrict__ ilist, int32_t *__restrict__ clist, int *counts, int *counts_next, int *mcount_next, int tile_blocks,
             int ring_blocks, const int8_t *__restrict__ mlo, float *__restrict__ plo_o, int8_t *__restrict__ mlo_o) {
  using Vw = View<R, P2, false, kFastOf<R>>;
  constexpr int NS = 3 * N + 3 * NC + 1;
  constexpr int NSA = STATS ? NS : 1;
  constexpr int RG = kCellRing, D = kCellDepth, ROWS = SEG + 4;
  const Model<R> &m = *mp;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const R zj = R(0.0) * m.jat_fac; /* (j - j_prev) * jat_fac with both currents +0 */
  R divjat0 = divx<Vw>(m, zj);
  divjat0 += divy<Vw>(m, zj);
  if ((int)blockIdx.x >= tile_blocks) {
    /* the blocks past the tiles list the delta-phi candidates of the ring x or y in {2, mesh+3} around the
     * interior (one thread per ring cell; the tiles list the interior ones), then fold the padding rows */
    const int q = (int)blockIdx.x - tile_blocks;
    if (q < ring_blocks) {
      dring_cell((int64_t)q * 256 + threadIdx.x, codes_in, clist, counts, ps, mx, my);
    } else if constexpr (STATS) {
      const int s = (q - ring_blocks) * 4 + wv, npad = (int)((my + kPadOut - 1) / kPadOut);
      if (s >= npad) return;
      R st[NSA];
      stats_init<N, NC>(st);
      pad_stats<N, NC, R, P2, C>(m, mu, mlo, codes_in, s, fs, ps, mx, my, divjat0, st);
      stats_partials<N, NC, true>(st, partials, pstride, nwaves + s, nwaves + npad, lane);
    }
    return;
  }
  /* the next step's list lengths start at zero (the kernels that read them last ran before this one) */
  if (blockIdx.x == 0 && threadIdx.x < 2) counts_next[threadIdx.x] = 0;
  if (blockIdx.x == 0 && threadIdx.x == 2) *mcount_next = 0;
  /* blocks go round the eight XCDs in turn: each XCD takes a contiguous run of tiles, so that the lines and rows two
   * neighbouring tiles share meet in one L2 */
  const int chunk = tile_blocks >> 3, bid = (int)blockIdx.x;
  const int tblk = bid < 8 * chunk ? (bid & 7) * chunk + (bid >> 3) : bid;
  const int w = tblk * 4 + wv; /* wave-uniform: the tile's rows and the row loop are scalar */
  if (w >= nwaves) return;
  const int strip = w % nstrips, seg = w / nstrips;
  const int xa = 3 + seg * SEG, nrow = min(SEG, (int)mx + 3 - xa), xb = xa + nrow - 1;
  /* the lane's cells y (an even element offset) and y + 1; lanes past the grid read its last pair */
  const int y = 1 + strip * kCellOut + 2 * lane, ry = (int)my + 6;
  const int yl = min(y, (ry - 3) | 1);
  const bool inner = lane >= 1 && lane <= 62;
  const bool oe = inner && y <= (int)my + 2, oo = inner && y + 1 <= (int)my + 2;
  /* addresses: a scalar row offset and an unsigned in-row offset per lane, so that a plane costs no vector registers */
  const int pso = (int)ps, xlast = (xb + 1) * pso;
  const unsigned c0i = (unsigned)(yl + kYOff), cyi = (unsigned)(y + kYOff);

  R st[NSA];
  if constexpr (STATS) stats_init<N, NC>(st);
  /* FP32: no sum of squared increments adds more than 16 terms before it is widened, so in long segments the second
   * column has sums of its own (one sum for both doubled the rounding of rel_change_mu: 0.8e-9 off at 4096^2) */
  constexpr bool TWO_SUMS = kLeanBulk<R> && 2 * SEG > 16;
  R odd[NC];
#pragma unroll
  for (int k = 0; k < NC; k++) odd[k] = R(0.0);
  unsigned seen = 0u; /* phases of the lane's bulk cells (their phi extrema, folded at the end) */

  /* mu rows in a ring of kCellRing register slots, row r in slot (r - xa) mod kCellRing, so that no slot is
   * ever copied: the row being updated reads rows x-1, x, x+1 where they were loaded, and the slot of x-1 then
   * takes row x + kCellDepth + 1. The phase codes of the output buffers (which tell whether phi is already e_b
   * there) ride the same ring in the mixed tiles. A loaded value is first read kCellDepth rows after its load, and
   * no wait in between covers a newer load (the counter of outstanding memory operations is in order). */
  Pair<R> ring[RG][NC];
  uint16_t qring[RG][NC]; /* compensated mode: the mu extensions of the ring's rows */
  unsigned kc[RG];
  auto load_row = [&](int slot, int off) {
#pragma unroll
    for (int k = 0; k < NC; k++) ring[slot][k] = row_ld<Pair<R>>(mu + (k * fs + off), c0i);
    if constexpr (C) {
#pragma unroll
      for (int k = 0; k < NC; k++) qring[slot][k] = row_ld<uint16_t>(mlo + (k * fs + off), c0i);
    }
  };
  /* the tile's first loads all issue before the first wait: its phase codes (rows xa-2 .. xa+SEG+1, clamped to xb+2)
   * and the first mu rows of the ring (rows past the tile's end are clamped to its last row + 1) */
  unsigned cv[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; r++) cv[r] = code_pair(codes_in + (int64_t)(min(xa - 2 + r, xb + 2) * pso), c0i);
#pragma unroll
  for (int d = -1; d <= D; d++) load_row((d + RG) % RG, min((xa + d) * pso, xlast));
  /* a full tile whose staged codes are all one phase tb has only bulk cells of that phase */
  int tb = -1;
  if (nrow == SEG && (strip + 1) * kCellOut <= (int)my) {
    unsigned diff = 0u;
#pragma unroll
    for (int r = 1; r < ROWS; r++) diff |= cv[r] ^ cv[0];
    const unsigned u0 = __builtin_amdgcn_readfirstlane(cv[0]);
    if (__all(diff == 0u && cv[0] == u0) && (u0 >> 8) == (u0 & 0xffu) && !(u0 & 0x80u)) tb = (int)(u0 & 0xffu);
  }
  /* tile flags: the phase of a uniform tile of the current state for the next step, whose output buffers hold this
   * state; the previous step's flag says the same of this step's output buffers */
  const bool kept_tile = keep && tb >= 0 && tin[w] == tb;
  if (lane == 0) tout[w] = (int8_t)tb;

  /* The rows of the tile, instantiated twice so that the uniform form is a loop of its own: every lane of it computes
   * and folds the mu statistics, only the inner ones write. t: the mixed form's bulk cells, bit r + 2 for row xa + r.
   * In FP32 a mixed row is one pass with each cell's coefficients selected by its phase; in FP64, whose update takes
   * seven times the coefficients, it is one pass per phase that has bulk cells in the row. */
  auto rows = [&](auto uniform, const TileMasks<N> &t) {
    constexpr bool UNI = decltype(uniform)::value;
    int xoff = xa * pso;
    for (int x0 = 0; x0 < nrow; x0 += RG) {
#pragma unroll
      for (int j = 0; j < RG; j++) {
        const int64_t xo = xoff;
        R e0[NC], e1[NC], e2[NC], o0[NC], o1[NC], o2[NC], ol[NC], er[NC];
#pragma unroll
        for (int k = 0; k < NC; k++) {
          const Pair<R> q0 = ring[(j + RG - 1) % RG][k], q1 = ring[j][k], q2 = ring[(j + 1) % RG][k];
          e0[k] = q0.x;
          o0[k] = q0.y;
          e1[k] = q1.x;
          o1[k] = q1.y;
          e2[k] = q2.x;
          o2[k] = q2.y;
          ol[k] = lane_up(o1[k]);
          er[k] = lane_dn(e1[k]);
        }
        /* the cells' new mu (and extensions), phi = e_b where the output buffer does not hold it already, statistics */
        auto finish = [&](bool se, bool so, int be, int bo, R *ne, R *de, R *no, R *dn) {
          uint16_t qn[NC];
          if constexpr (C) {
            /* compensated mode: the increment is added to the decoded value (hi plus its extension) and the sum is
             * re-encoded, so the bits of the increment below the FP32 part are kept */
#pragma unroll
            for (int k = 0; k < NC; k++) {
              const unsigned q = qring[j][k];
              float he, ho;
              int8_t ne8, no8;
              c32_encode(c32_decode((float)e1[k], (int8_t)(q & 0xffu)) + (double)de[k], he, ne8);
              c32_encode(c32_decode((float)o1[k], (int8_t)(q >> 8)) + (double)dn[k], ho, no8);
              ne[k] = (R)he;
              no[k] = (R)ho;
              qn[k] = (uint16_t)((unsigned)(uint8_t)ne8 | ((unsigned)(uint8_t)no8 << 8));
            }
          }
          if (se && so) {
#pragma unroll
            for (int k = 0; k < NC; k++) row_st<Pair<R>>(mu_o + (k * fs + xo), cyi, Pair<R>{ne[k], no[k]});
            if constexpr (C) {
#pragma unroll
              for (int k = 0; k < NC; k++) row_st<uint16_t>(mlo_o + (k * fs + xo), cyi, qn[k]);
            }
          } else if (!UNI && (se || so)) {
            const unsigned c1 = se ? cyi : cyi + 1u;
#pragma unroll
            for (int k = 0; k < NC; k++) row_st<R>(mu_o + (k * fs + xo), c1, se ? ne[k] : no[k]);
            if constexpr (C) {
#pragma unroll
              for (int k = 0; k < NC; k++)
                row_st<int8_t>(mlo_o + (k * fs + xo), c1, (int8_t)(se ? qn[k] & 0xffu : qn[k] >> 8));
            }
          }
          if (UNI) {
            if (!kept_tile && inner) {
#pragma unroll
              for (int a = 0; a < N; a++) {
                const R p = a == be ? R(1.0) : R(0.0);
                row_st<Pair<R>>(phi_o + (a * fs + xo), cyi, Pair<R>{p, p});
                if constexpr (C) row_st<Pair<float>>(plo_o + (a * fs + xo), cyi, Pair<float>{0.0f, 0.0f});
              }
              row_st<uint16_t>(codes_out + xo, cyi, (uint16_t)(be * 0x101));
            }
          } else {
            if (se && !(keep && (kc[j] & 0xffu) == (unsigned)be)) {
#pragma unroll
              for (int a = 0; a < N; a++) {
                row_st<R>(phi_o + (a * fs + xo), cyi, a == be ? R(1.0) : R(0.0));
                if constexpr (C) row_st<float>(plo_o + (a * fs + xo), cyi, 0.0f);
              }
              row_st<int8_t>(codes_out + xo, cyi, (int8_t)be);
            }
            if (so && !(keep && (kc[j] >> 8) == (unsigned)bo)) {
#pragma unroll
              for (int a = 0; a < N; a++) {
                row_st<R>(phi_o + (a * fs + xo), cyi + 1u, a == bo ? R(1.0) : R(0.0));
                if constexpr (C) row_st<float>(plo_o + (a * fs + xo), cyi + 1u, 0.0f);
              }
              row_st<int8_t>(codes_out + xo, cyi + 1u, (int8_t)bo);
            }
          }
          if (STATS) {
            if (UNI || se) bulk_stats<N, NC>(st, st + 3 * N + 2 * NC, ne, de);
            if (UNI || so) bulk_stats<N, NC>(st, TWO_SUMS ? odd : st + 3 * N + 2 * NC, no, dn);
          }
        };
        R ne[NC], no[NC], de[NC], dn[NC];
        if constexpr (kLeanBulk<R>) {
          R Ke[NC][NC], Ko[NC][NC];
          bool se = UNI && inner, so = se;
          int be = UNI ? tb : 0, bo = be;
#pragma unroll
          for (int a = 0; a < N; a++) {
            const bool ea = (t.be[a] >> (x0 + j + 2)) & 1u, oa = (t.bo[a] >> (x0 + j + 2)) & 1u;
            if (!UNI) {
              se = se || ea;
              so = so || oa;
              be = ea ? a : be;
              bo = oa ? a : bo;
            }
#pragma unroll
            for (int k = 0; k < NC; k++)
#pragma unroll
              for (int l = 0; l < NC; l++) {
                const R kk = UNI ? m.Kbulk[tb][k][l] : scalar_val(m.Kbulk[a][k][l]);
                Ke[k][l] = UNI || a == 0 || ea ? kk : Ke[k][l];
                Ko[k][l] = UNI || a == 0 || oa ? kk : Ko[k][l];
              }
            if (UNI) break;
          }
          if (UNI || __any(se || so)) {
            bulk_update_lean<NC>(m, Ke, e0, e1, e2, o1, ol, ne, de);
            bulk_update_lean<NC>(m, Ko, o0, o1, o2, er, e1, no, dn);
            finish(se, so, be, bo, ne, de, no, dn);
          }
        } else {
#pragma unroll
          for (int a = 0; a < (UNI ? 1 : N); a++) {
            const bool se = UNI ? inner : (t.be[a] >> (x0 + j + 2)) & 1u;
            const bool so = UNI ? inner : (t.bo[a] >> (x0 + j + 2)) & 1u;
            if (UNI || __any(se || so)) {
              const int b = UNI ? tb : a;
              bulk_update_ref<N, NC, R, P2>(m, b, e0, e1, e2, o1, ol, divjat0, ne, de);
              bulk_update_ref<N, NC, R, P2>(m, b, o0, o1, o2, er, e1, divjat0, no, dn);
              finish(se, so, b, b, ne, de, no, dn);
            }
          }
        }
        /* refill: row x + D + 1 into the slot of row x - 1, the output codes of row x + D */
        const int xn = min(xoff + (D + 1) * pso, xlast);
        load_row((j + RG - 1) % RG, xn);
        if (!UNI) kc[(j + D) % RG] = code_pair(codes_out + (xn - pso), c0i);
        xoff += pso;
        /* the rows stay apart: interleaved, the four rows of a turn would take twice the registers */
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  if (tb >= 0) {
    /* the prologue's loads complete here, once per tile: the loop's first row then waits on nothing, and the
     * wait counts inside the loop follow from the loop body alone (vmcnt 0, expcnt and lgkmcnt unconstrained) */
    __builtin_amdgcn_s_waitcnt(0x0f70);
    rows(std::true_type{}, TileMasks<N>{});
    if (STATS) {
      if (!inner) {
        stats_init<N, NC>(st);
#pragma unroll
        for (int k = 0; k < NC; k++) odd[k] = R(0.0);
      } else {
        seen = 1u << tb;
      }
    }
  } else {
#pragma unroll
    for (int d = 0; d < D; d++) kc[d] = code_pair(codes_out + min((xa + d) * pso, xlast - pso), c0i);
    TileMasks<N> t = tile_masks<N>(cv);
    const uint32_t live = ((1u << nrow) - 1u) << 2;
    const uint32_t le = oe ? live : 0u, lo = oo ? live : 0u;
    uint32_t ie = le, io = lo;
#pragma unroll
    for (int b = 0; b < N; b++) {
      t.be[b] &= le;
      t.bo[b] &= lo;
      ie &= ~t.be[b];
      io &= ~t.bo[b];
      if (t.be[b] | t.bo[b]) seen |= 1u << b;
    }
    const uint32_t ce = le & ~t.ue, co = lo & ~t.uo;
    /* reserve the tile's list entries (the atomic's latency passes under the row loop) */
    const int cnt = wave_sum((int)((__popc(ie) + __popc(io)) | ((__popc(ce) + __popc(co)) << 16)));
    uint64_t base = 0;
    if (cnt && lane == 0) base = list_reserve(counts, cnt & 0xffff, cnt >> 16);
    rows(std::false_type{}, t);
    /* the lists, row by row: a wavefront of the list kernels then gathers neighbouring cells of a row */
    if (cnt) {
      int bi = __builtin_amdgcn_readfirstlane((int)(base & 0xffffffffull));
      int bc = __builtin_amdgcn_readfirstlane((int)(base >> 32));
      int cell = xa * pso + (int)cyi;
      auto emit = [&](int32_t *list, int &at, uint32_t e, uint32_t o, int r) {
        const bool pe = (e >> r) & 1u, po = (o >> r) & 1u;
        const uint64_t be = __ballot(pe), bo = __ballot(po);
        if (!(be | bo)) return;
        const uint64_t lt = (1ull << lane) - 1ull;
        const int pos = at + __popcll(be & lt) + __popcll(bo & lt);
        if (pe) list[pos] = cell;
        if (po) list[pos + (pe ? 1 : 0)] = cell + 1;
        at += __popcll(be) + __popcll(bo);
      };
      for (int r = 2; r < nrow + 2; r++, cell += pso) {
        emit(ilist, bi, ie, io, r);
        emit(clist, bc, ce, co, r);
      }
    }
  }
  if constexpr (STATS) {
    bulk_seen_fold<N>(st, seen);
    stats_partials<N, NC, true>(st, partials, pstride, w, nwaves, lane, TWO_SUMS ? odd : nullptr);
  }
}

/* The halo of the new state: each halo cell takes the value of its proxy, as write_images scatters it
 * (apply_boundary_conditions as a gather). Halo row X = hx[k] has the proxy row sx[f][k] when that is an interior row and
 * at most one k' < k shares it (write_images takes the first two images of a row); an interior row is its own (likewise
 * for columns). Field group f = 0 holds phi, its low parts and the phase codes, f = 1 mu and its extensions. A halo cell
 * without a proxy is left as it is.
 * No launch of its own: k_cbulk has written the bulk cells when the delta-phi launch runs, so extra blocks of that launch
 * copy the halo cells whose proxy is a bulk cell and list the others, and k_ilist updates a listed proxy once more with
 * the halo cell as its target (the separate pass was 4 to 10 us a step, nearly all of it launch and memory latency; images
 * scattered by the lane that updates the proxy lengthened every k_ilist by 4 us: 1024^2 FP64 12.3 -> 16.5). */
__device__ __forceinline__ int64_t halo_source(const int32_t *src, const int32_t *h, int64_t X, int64_t lo,
                                               int64_t hi) {
  if (X >= lo && X <= hi) return X;
  int64_t s = -1;
#pragma unroll
  for (int k = 0; k < 6; k++) {
    int before = 0;
#pragma unroll
    for (int j = 0; j < k; j++) before += src[j] == src[k];
    if (h[k] == X && src[k] >= lo && src[k] <= hi && before < 2) s = src[k];
  }
  return s;
}

/* the phase of a bulk cell at offset s (its radius-2 diamond is purely that phase), else -1 */
__device__ __forceinline__ int bulk_code(const int8_t *__restrict__ codes, int64_t s, int64_t ps) {
  const int b = codes[s];
  bool same = b >= 0;
#pragma unroll
  for (int di = -2; di <= 2; di++)
#pragma unroll
    for (int dj = -2; dj <= 2; dj++)
      if ((di < 0 ? -di : di) + (dj < 0 ? -dj : dj) <= 2) same = same & (codes[s + di * ps + dj] == b);
  return same ? b : -1;
}

/* the output buffers of a step (plo, mlo: compensated mode) */
template <typename R>
struct NewState {
  R *phi, *mu;
  int8_t *codes;
  float *plo;
  int8_t *mlo;
};

/* An image in k_ilist's second list: the proxy's offset, the halo cell's, and the field groups to write there (bit 0: phi
 * and codes, bit 1: mu). Offsets have 31 bits (cells_fit). */
__device__ __forceinline__ uint64_t image_entry(int64_t src, int64_t dst, unsigned groups) {
  return (uint64_t)src | ((uint64_t)dst << 31) | ((uint64_t)groups << 62);
}
/* item i of k_ilist: cell c and target dst, groups and whether it counts in the statistics; i < n: listed cells */
struct IfaceItem {
  int64_t c, dst;
  unsigned groups;
  bool own;
  __device__ __forceinline__ IfaceItem(int i, int n, const int32_t *__restrict__ ilist, const uint64_t *__restrict__ mlist) {
    own = i < n;
    if (own) {
      c = dst = ilist[i];
      groups = 3u;
    } else {
      const uint64_t e = mlist[i - n];
      c = (int64_t)(e & 0x7fffffffu);
      dst = (int64_t)((e >> 31) & 0x7fffffffu);
      groups = (unsigned)(e >> 62);
    }
  }
};

/* halo cell j (the six halo rows over the full width, then the six halo cells of each interior row): copied where the
 * proxy is a bulk cell of the step from codes_in, listed where it is an interface cell */
template <int N, int NC, typename R, bool C>
__device__ __forceinline__ void halo_cell(int64_t j, const int8_t *__restrict__ codes_in, const NewState<R> &o,
                                          uint64_t *__restrict__ mlist, int *mcount, const Maps &maps, int64_t fs,
                                          int64_t ps, int64_t mx, int64_t my) {
  const int64_t ry = my + 6, nrow = 6 * ry, ncol = 6 * mx;
  if (j >= nrow + ncol) return;
  /* the index arithmetic in 32 bits (the halo has fewer than 2^31 cells; 64-bit division is a long sequence) */
  int64_t X, Y;
  if (j < nrow) {
    const uint32_t iu = (uint32_t)j, ryu = (uint32_t)ry, r = iu / ryu;
    X = r < 3u ? (int64_t)r : mx + r;
    Y = iu - r * ryu;
  } else {
    /* six consecutive threads take the six halo cells of one interior row (two runs of three adjacent elements) */
    const uint32_t k = (uint32_t)(j - nrow), row = k / 6u, q = k - 6u * row;
    Y = q < 3u ? (int64_t)q : my + q;
    X = 3 + (int64_t)row;
  }
  const int64_t c = X * ps + Y + kYOff;
  int64_t s[2];
  int b[2];
#pragma unroll
  for (int f = 0; f < 2; f++) {
    const int64_t sx = halo_source(maps.sx[f], maps.hx, X, 3, mx + 2);
    const int64_t sy = halo_source(maps.sy[f], maps.hy, Y, 3, my + 2);
    s[f] = sx < 0 || sy < 0 ? -1 : sx * ps + sy + kYOff;
    b[f] = s[f] < 0 ? -1 : bulk_code(codes_in, s[f], ps);
  }
  if (b[0] >= 0) {
    o.codes[c] = (int8_t)b[0];
#pragma unroll
    for (int a = 0; a < N; a++) {
      o.phi[a * fs + c] = a == b[0] ? R(1.0) : R(0.0);
      if constexpr (C) o.plo[a * fs + c] = 0.0f;
    }
  }
  if (b[1] >= 0) {
#pragma unroll
    for (int k = 0; k < NC; k++) {
      o.mu[k * fs + c] = o.mu[k * fs + s[1]];
      if constexpr (C) o.mlo[k * fs + c] = o.mlo[k * fs + s[1]];
    }
  }
  /* interface proxies: one entry, or one per field group where the groups' proxies differ */
  const bool i0 = s[0] >= 0 && b[0] < 0, i1 = s[1] >= 0 && b[1] < 0, one = i0 && i1 && s[0] == s[1];
  const int n = one ? 1 : (int)i0 + (int)i1;
  if (n) {
    const int at = atomicAdd(mcount, n);
    if (one) {
      mlist[at] = image_entry(s[0], c, 3);
    } else {
      if (i0) mlist[at] = image_entry(s[0], c, 1);
      if (i1) mlist[at + (i0 ? 1 : 0)] = image_entry(s[1], c, 2);
    }
  }
}

/* number of halo cells halo_cell covers */
__host__ __device__ constexpr int64_t halo_cells(int64_t mx, int64_t my) { return 6 * (my + 6) + 6 * mx; }

/* blocks of the halo pass at the front of a delta-phi launch */
__host__ __device__ constexpr unsigned halo_blocks(int64_t mx, int64_t my) {
  return (unsigned)((halo_cells(mx, my) + 255) / 256);
}

/* Fold the partials of a step's wavefronts into the cumulative statistics: one block per statistic, each reading its
 * contiguous row of partials (statistic-major layout) in a fixed order, so the result is deterministic. */
template <int N, int NC, int THREADS>
__device__ __forceinline__ void stats_fold_block(const double *__restrict__ partials, int64_t stride, int64_t nparts,
                                                 double *__restrict__ cum, int i) {
  constexpr int NS = 3 * N + 3 * NC + 1;
  __shared__ double red[THREADS];
  if (i >= NS) return;
  const bool mx = (i < N || (i >= 2 * N && i < 2 * N + NC));
  const bool mn = !mx && i < 2 * N + 2 * NC;
  double r = mx ? -INFINITY : mn ? INFINITY : 0.0;
  const double *row = partials + (int64_t)i * stride;
  /* a thread folds its partials in index order; the loads of eight of them are issued before the first is used */
  int64_t b = threadIdx.x;
  for (; b + 7 * THREADS < nparts; b += 8 * THREADS) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) v[u] = row[b + u * THREADS];
#pragma unroll
    for (int u = 0; u < 8; u++) r = mx ? fmax(r, v[u]) : mn ? fmin(r, v[u]) : r + v[u];
  }
  for (; b < nparts; b += THREADS) {
    const double v = row[b];
    r = mx ? fmax(r, v) : mn ? fmin(r, v) : r + v;
  }
  red[threadIdx.x] = r;
  __syncthreads();
  for (int s = THREADS / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) {
      double o = red[threadIdx.x + s];
      red[threadIdx.x] = mx ? fmax(red[threadIdx.x], o) : mn ? fmin(red[threadIdx.x], o) : red[threadIdx.x] + o;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    double v = red[0];
    if (mx) cum[i] = fmax(cum[i], v);
    else if (mn) cum[i] = fmin(cum[i], v);
    else if (i < NS - 1) cum[i] = v;
    else cum[i] += v;
  }
}

/* What rides in the delta-phi launch of a step, in blocks before those of the list: the fold of the previous step's
 * statistics (nfold blocks; its partials lie in the half of the buffer that this step does not write), and the halo of the
 * new state (nhalo blocks). Launches of their own for the two were 4 to 10 us a step. */
template <typename R>
struct StepExtras {
  int nfold, nhalo;
  const double *partials;
  int64_t pstride;
  double *cum;
  const int8_t *codes_in;
  NewState<R> o;
  uint64_t *mlist;
  int *mcount;
  Maps maps;
  int64_t mx, my;
};
/* true when the calling block was one of the extras */
template <int N, int NC, typename R, bool C>
__device__ __forceinline__ bool step_extras(const StepExtras<R> &e, int64_t fs, int64_t ps) {
  const int b = (int)blockIdx.x;
  if (b >= e.nfold + e.nhalo) return false;
  if (b < e.nfold) stats_fold_block<N, NC, 256>(e.partials, e.pstride, e.pstride, e.cum, b);
  else halo_cell<N, NC, R, C>((int64_t)(b - e.nfold) * 256 + threadIdx.x, e.codes_in, e.o, e.mlist, e.mcount, e.maps, fs, ps, e.mx,
                              e.my);
  return true;
}

/* The delta-phi launch of a step: the extras, then the candidates (k_dlist's loop). */
template <int N, int NC, typename R, bool P2>
__global__ __launch_bounds__(256) void k_dlist_step(const Model<R> *__restrict__ mp, const R *__restrict__ phi,
                                                    const R *__restrict__ mu, R *__restrict__ dphi, int64_t fs, int64_t ps,
                                                    const int32_t *__restrict__ clist, const int *__restrict__ ccount,
                                                    StepExtras<R> ex) {
  if (step_extras<N, NC, R, false>(ex, fs, ps)) return;
  const int nex = ex.nfold + ex.nhalo, n = *ccount, stride = ((int)gridDim.x - nex) * 256;
  for (int i = ((int)blockIdx.x - nex) * 256 + (int)threadIdx.x; i < n; i += stride)
    dphi_cell<N, NC, R, P2>(*mp, phi, mu, dphi, fs, ps, clist[i]);
}

/* The general update of the interface cells listed by k_cbulk (any order), then of the images (IfaceItem): a grid-stride
 * loop of full wavefronts. Each cell gathers its stencil from memory in one batch: phi on the 3x3 neighbourhood, mu and
 * delta-phi on the 5-point one, and the phase codes of its radius-2 diamond, which decide which of the five
 * delta-phi values are k_dphi's (candidates) and which are exactly 0. Statistics: one partial per wavefront of the
 * grid (the grid is fixed, the order of the cells within it is not). */
template <int N, int NC, typename R, bool P2, bool STATS>
__global__ __launch_bounds__(256, 2) void k_ilist(const Model<R> *__restrict__ mp, const R *__restrict__ phi,
                                               const R *__restrict__ mu, const R *__restrict__ dphi,
                                               const int8_t *__restrict__ codes_in, R *__restrict__ phi_o,
                                               R *__restrict__ mu_o, int8_t *__restrict__ codes_out,
                                               double *__restrict__ partials, int64_t pstride, int64_t fs,
                                               int64_t ps, const int32_t *__restrict__ ilist,
                                               const int *__restrict__ icount,
                                               const uint64_t *__restrict__ mlist, const int *__restrict__ mcount) {
  constexpr int NS = 3 * N + 3 * NC + 1;
  constexpr int NSA = STATS ? NS : 1;
  const Model<R> &m = *mp;
  const int lane = threadIdx.x & 63;
  const int w = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int nw = gridDim.x * 4;
  R st[NSA];
  if constexpr (STATS) stats_init<N, NC>(st);
  const int n = *icount, ntot = n + *mcount;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < ntot; i += gridDim.x * blockDim.x) {
    const IfaceItem it(i, n, ilist, mlist);
    const int64_t c = it.c;
    const int y = (int)((uint32_t)c % (uint32_t)ps) - kYOff;
    /* codes of the diamond: slot (di, dj) for |di| + |dj| <= 2 */
    int8_t cd[5][5];
#pragma unroll
    for (int di = -2; di <= 2; di++)
#pragma unroll
      for (int dj = -2; dj <= 2; dj++)
        if ((di < 0 ? -di : di) + (dj < 0 ? -dj : dj) <= 2) cd[di + 2][dj + 2] = codes_in[c + di * ps + dj];
    RegStore<N, NC, R> rs;
    const int oi[5] = {0, 1, -1, 0, 0}, oj[5] = {0, 0, 0, 1, -1};
#pragma unroll
    for (int a = 0; a < N; a++)
#pragma unroll
      for (int di = 0; di < 3; di++)
#pragma unroll
        for (int dj = 0; dj < 3; dj++) rs.p[a][di][dj] = phi[a * fs + c + (di - 1) * ps + (dj - 1)];
#pragma unroll
    for (int o = 0; o < 5; o++) {
      const int64_t co = c + oi[o] * ps + oj[o];
#pragma unroll
      for (int k = 0; k < NC; k++) rs.u[k][o] = mu[k * fs + co];
      const int r = oi[o] + 2, q = oj[o] + 2;
      const int8_t k0 = cd[r][q];
      const bool cand = k0 < 0 || cd[r - 1][q] != k0 || cd[r + 1][q] != k0 || cd[r][q - 1] != k0 || cd[r][q + 1] != k0;
#pragma unroll
      for (int a = 0; a < N; a++) {
        const R v = dphi[a * fs + co];
        rs.d[a][o] = cand ? v : R(0.0);
      }
    }
    const RegView<N, NC, R, P2, kFastOf<R>> v{&rs, 0, 0};
    R jx0[NC], jxb[NC], jy0[NC], jyl[NC], d[N], pn[N], mn[NC], dm[NC];
    if constexpr (kBySolids<R>) {
      jat_faces<N, NC>(m, v, y, jx0, jxb, jy0, jyl);
    } else {
      jat_x<N, NC>(m, v, 0, 0, jx0);
      jat_x<N, NC>(m, v, -1, 0, jxb);
      jat_y<N, NC>(m, v, 0, 0, y, jy0);
      jat_y<N, NC>(m, v, 0, -1, y - 1, jyl);
    }
#pragma unroll
    for (int a = 0; a < N; a++) d[a] = v.dp(a, 0, 0);
    mu_update<N, NC>(m, v, false, d, jx0, jxb, jy0, jyl, pn, mn, dm);
    if (it.groups & 1u) {
#pragma unroll
      for (int a = 0; a < N; a++) phi_o[a * fs + it.dst] = pn[a];
      codes_out[it.dst] = (int8_t)pure_phase<N>(pn);
    }
    if (it.groups & 2u) {
#pragma unroll
      for (int k = 0; k < NC; k++) mu_o[k * fs + it.dst] = mn[k];
    }
    if constexpr (STATS)
      if (it.own) stats_add<N, NC>(st, pn, d, mn, dm);
  }
  if constexpr (STATS) stats_partials<N, NC>(st, partials, pstride, w, nw, lane);
}

}  // namespace gpk
