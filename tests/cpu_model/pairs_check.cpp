// Host build of gp_pairs.h against gp_model.h, one random cell at a time: delta-phi (phi_delta_pairs / phi_delta) and
// the face currents (jat_faces / jat_x, jat_y) of the same register stencil and model.
#include <cmath>

#include "gp_pairs.h"
#include "gp_reverse.h"

using namespace gpk;

template <int N, int NC, typename R, bool P2, bool FAST>
static int compare(const gp_params *p, const double *in, double *out) {
  Model<R> m;
  if (make_model(p, &m)) return -1;
  if (P2 && !m.pow2) return -3;
  RegStore<N, NC, R> rs;
  for (int a = 0; a < N; a++)
    for (int i = 0; i < 9; i++) rs.p[a][i / 3][i % 3] = (R)*in++;
  for (int k = 0; k < NC; k++)
    for (int o = 0; o < 5; o++) rs.u[k][o] = (R)*in++;
  for (int a = 0; a < N; a++)
    for (int o = 0; o < 5; o++) rs.d[a][o] = (R)*in++;
  const int64_t y = (int64_t)*in;
  const RegView<N, NC, R, P2, FAST> v{&rs, 0, 0};
  R d0[N], d1[N], j0[4][NC], j1[4][NC];
  phi_delta<N, NC>(m, v, false, d0);
  phi_delta_pairs<N, NC>(m, v, d1);
  jat_x<N, NC>(m, v, 0, 0, j0[0]);
  jat_x<N, NC>(m, v, -1, 0, j0[1]);
  jat_y<N, NC>(m, v, 0, 0, y, j0[2]);
  jat_y<N, NC>(m, v, 0, -1, y - 1, j0[3]);
  jat_faces<N, NC>(m, v, y, j1[0], j1[1], j1[2], j1[3]);
  for (int a = 0; a < N; a++) {
    *out++ = (double)d0[a];
    *out++ = (double)d1[a];
  }
  for (int f = 0; f < 4; f++)
    for (int k = 0; k < NC; k++) {
      *out++ = (double)j0[f][k];
      *out++ = (double)j1[f][k];
    }
  return 2 * (N + 4 * NC);
}

template <int N, int NC>
static int pick_form(const gp_params *p, int form, const double *in, double *out) {
  switch (form) {
    case 0: return compare<N, NC, double, false, false>(p, in, out);
    case 1: return compare<N, NC, double, true, false>(p, in, out);
    case 2: return compare<N, NC, double, true, true>(p, in, out);
    case 3: return compare<N, NC, float, true, true>(p, in, out);
  }
  return -2;
}

// form 0: FP64, 1: FP64 with power-of-two spacings, 2: the compensated mode's FP64, 3: FP32. Returns the number of values
// written to out: (full loops, by pairs) for delta-phi of every phase, then for the four currents of every mu field.
extern "C" int pairs_check(const gp_params *p, int form, const double *in, double *out) {
  const int N = p->nphases, NC = p->ncomp - 1;
  if (N == 2 && NC == 1) return pick_form<2, 1>(p, form, in, out);
  if (N == 3 && NC == 2) return pick_form<3, 2>(p, form, in, out);
  if (N == 4 && NC == 2) return pick_form<4, 2>(p, form, in, out);
  if (N == 3 && NC == 3) return pick_form<3, 3>(p, form, in, out);
  return -2;
}

// Stage P transposed, of the same cell: the adjoint gout[N] follows the cell's values in `in`. Writes (full loops, by pairs)
// of the stencil adjoint, the mu adjoint and theta; returns the number of values.
template <int N, int NC>
static int compare_vjp(const gp_params *p, const double *in, double *out) {
  Model<double> m;
  if (make_model(p, &m)) return -1;
  RegStore<N, NC, double> rs;
  for (int a = 0; a < N; a++)
    for (int i = 0; i < 9; i++) rs.p[a][i / 3][i % 3] = *in++;
  for (int k = 0; k < NC; k++)
    for (int o = 0; o < 5; o++) rs.u[k][o] = *in++;
  in += 5 * N + 1;
  const RegView<N, NC, double, false> v{&rs, 0, 0};
  RevAcc<N, NC> r, q;
  r.clear();
  q.clear();
  phi_delta_vjp<N, NC>(m, v, in, r);
  phi_delta_vjp_pairs<N, NC>(m, v, in, q, [&](int a, int i, int j, double x) { q.ph(a, i, j) += x; });
  int n = 0;
  auto put = [&](double x, double y) {
    out[n++] = x;
    out[n++] = y;
  };
  for (int a = 0; a < N; a++)
    for (int i = 0; i < 9; i++) put(r.p[a][i / 3][i % 3], q.p[a][i / 3][i % 3]);
  for (int k = 0; k < NC; k++) put(r.u[k][0], q.u[k][0]);
  for (int t = 0; t < kThetaN<N, NC>; t++) put(r.th[t], q.th[t]);
  return n;
}
extern "C" int pairs_check_vjp(const gp_params *p, const double *in, double *out) {
  const int N = p->nphases, NC = p->ncomp - 1;
  if (N == 2 && NC == 1) return compare_vjp<2, 1>(p, in, out);
  if (N == 3 && NC == 2) return compare_vjp<3, 2>(p, in, out);
  if (N == 4 && NC == 2) return compare_vjp<4, 2>(p, in, out);
  if (N == 3 && NC == 3) return compare_vjp<3, 3>(p, in, out);
  return -2;
}
