/*
 * gp_pairs.h -- the step's two interface evaluations by the phases that are present: delta-phi of a cell from its
 * unordered phase pairs (phi_delta_pairs) and its four anti-trapping face currents from its solids (jat_faces).
 *
 * gp_model.h states both as loops over all ordered phase pairs and all solids. Nearly every interface cell holds two
 * phases: the terms of a phase that is zero on the cell's whole 3x3 stencil are zeros, and the terms of (b, a) are those
 * of (a, b) with the sign turned, since q_ba = -q_ab exactly. The functions here visit, per lane, only the pairs and
 * solids that are present, in the order of the full loops, and add the same rounded terms to the same sums, so the
 * results equal gp_model.h's bit for bit (zeros may differ in sign). A lane picks the fields of its pair with register
 * selects; a wavefront runs as many turns as its busiest lane has pairs (one or two along an interface, against six
 * ordered pairs of three phases and twelve of four), and the code holds one pair's arithmetic instead of all.
 * The list kernels are bound by this arithmetic (FP64 issue at two wavefronts per SIMD on large grids, one wavefront's chain
 * of instructions on small ones). delta-phi, full loops -> pairs: 4096^2 compensated, 0.8 M candidates, 115 -> 55 us;
 * four phases 391 x 523 FP64 32.9 -> 12.6 us; 1024^2 ternary FP64 21.0 -> 10.6 us. The update with its currents
 * (k_ilist): 1024^2 16.5 -> 14.2 us, four phases 19.8 -> 17.1 us.
 *
 * A stencil with a non-finite value keeps every pair and solid, so that a non-finite state spreads as in the full loops.
 * Coefficients that differ between (a, b) and (b, a), or are not finite, keep the ordered pairs (Model::pairs_sym).
 */
#pragma once

#include "gp_model.h"

namespace gpk {

/* Where the list kernels take these forms. In FP32 the device build rounds a quotient or square root to 1-2.5 ulp, or
 * correctly where the compiler has hoisted it out of its condition (qdiv), so another form of the loops has other last
 * bits, which a thousand steps carry to 3e-4 of a ternary state. delta-phi with power-of-two spacings holds the same
 * quotients in both forms and changes no bit; the others keep the full loops in FP32. */
template <typename R, bool P2>
constexpr bool kByPairs = sizeof(R) == sizeof(double) || P2;
template <typename R>
constexpr bool kBySolids = sizeof(R) == sizeof(double);

/* v(i) by register selects, i < COUNT varying from lane to lane (an indexed register array would live in memory, and so
 * would one read in the arms of the select: the compiler selects the address then) */
template <int COUNT, typename F>
GP_HD auto pick(int i, F v) -> decltype(v(0)) {
  auto r = v(0);
#pragma unroll
  for (int j = 1; j < COUNT; j++) {
    const auto x = v(j);
    r = i == j ? x : r;
  }
  return r;
}

/* bit a for every phase of the first COUNT that is not zero on the whole 3x3 stencil; all of them when a value among
 * them is not finite (the sum of magnitudes is zero, or finite, exactly when every term is) */
template <int COUNT, typename R, class V>
GP_HD unsigned phases_present(const V &v) {
  unsigned mask = 0u;
  bool finite = true;
#pragma unroll
  for (int a = 0; a < COUNT; a++) {
    R s = R(0.0);
#pragma unroll
    for (int i = -1; i <= 1; i++)
#pragma unroll
      for (int j = -1; j <= 1; j++) s += fabs(v.ph(a, i, j));
    mask |= s != R(0.0) ? 1u << a : 0u;
    finite = finite && s < R(INFINITY);
  }
  return finite ? mask : (1u << COUNT) - 1u;
}

template <typename R>
struct PairCoef {
  R gamma, dab, rot[2][2], rot_inv[2][2];
};

/* One face of the pair (phases 0 and 1 of v): the x-face between offsets (i,j) and (i+1,j) (DIR 0) or the y-face between
 * (i,j) and (i,j+1) (DIR 1). sa, sb the face averages, f1 = a_c^2 (s_a grad_n phi_b - s_b grad_n phi_a),
 * f2 = a_c |q|^2 (R^-1 d a_c/dq)_n; both change sign with the order of the pair. */
template <int DIR, typename R, class V>
GP_HD void pair_face(const Model<R> &m, const PairCoef<R> &k, const V &v, int i, int j, R &sa, R &sb, R &f1, R &f2) {
  R r[2];
  if constexpr (DIR == 0) {
    sa = sx(m, v, 0, i, j);
    sb = sx(m, v, 1, i, j);
    r[0] = (sa * gx(m, v, 1, i, j) - sb * gx(m, v, 0, i, j));
    r[1] = R(0.5) * (sa * (cy(m, v, 1, i, j) + cy(m, v, 1, i + 1, j)) - sb * (cy(m, v, 0, i, j) + cy(m, v, 0, i + 1, j)));
  } else {
    sa = sy(m, v, 0, i, j);
    sb = sy(m, v, 1, i, j);
    r[0] = R(0.5) * (sa * (cx(m, v, 1, i, j) + cx(m, v, 1, i, j + 1)) - sb * (cx(m, v, 0, i, j) + cx(m, v, 0, i, j + 1)));
    r[1] = (sa * gy(m, v, 1, i, j) - sb * gy(m, v, 0, i, j));
  }
  f1 = r[DIR];
  f2 = R(0.0);
  if (m.fn_aniso) {
    R q[2], ac, d[2], di[2];
    rot2(k.rot, r, q);
    if constexpr (V::kFast) {
      aniso_ac_dadq_fast(k.dab, q, ac, d);
    } else {
      ac = aniso_ac(k.dab, q);
      aniso_dadq(k.dab, q, d);
    }
    f1 = ac * ac * r[DIR];
    rot2(k.rot_inv, d, di);
    f2 = ac * qnorm2(q) * di[DIR];
  }
}

/* the pairs to visit, bit a N + b: a < b with both present and `on` set for one of them, or (coefficients that are not
 * symmetric) every ordered pair of an `on` phase a */
template <int N, typename R, class V>
GP_HD unsigned pairs_to_visit(const Model<R> &m, const V &v, unsigned on) {
  const bool sym = m.pairs_sym != 0;
  const unsigned present = sym ? phases_present<N, R>(v) : (1u << N) - 1u;
  unsigned todo = 0u;
#pragma unroll
  for (int a = 0; a < N; a++)
#pragma unroll
    for (int b = 0; b < N; b++) {
      if (b == a) continue;
      const bool both = (present >> a) & (present >> b) & 1u;
      const bool ona = (on >> a) & 1u, onb = (on >> b) & 1u;
      if (a < b ? both && (ona || (sym && onb)) : !sym && ona) todo |= 1u << (a * N + b);
    }
  return todo;
}

/* the stencils of phases a and b of v as phases 0 and 1 */
template <int N, typename R, class V>
GP_HD void pair_stencil(const V &v, int a, int b, RegStore<2, 0, R> &rs) {
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int j = 0; j < 3; j++) {
      rs.p[0][i][j] = pick<N>(a, [&](int c) { return v.ph(c, i - 1, j - 1); });
      rs.p[1][i][j] = pick<N>(b, [&](int c) { return v.ph(c, i - 1, j - 1); });
    }
}

/* the coefficients of pair p = a N + b */
template <int N, typename R>
GP_HD PairCoef<R> pair_coef(const Model<R> &m, int p) {
  PairCoef<R> k;
  auto load = [&](auto coef) {
    k.gamma = coef([&](int i, int j) { return m.gamma[i][j]; });
    if (!m.fn_aniso) return;
    k.dab = coef([&](int i, int j) { return m.dab[i][j]; });
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
      for (int c = 0; c < 2; c++) {
        k.rot[r][c] = coef([&](int i, int j) { return m.rot[i][j][r][c]; });
        k.rot_inv[r][c] = coef([&](int i, int j) { return m.rot_inv[i][j][r][c]; });
      }
  };
  if (m.pairs_sym) {
    /* wave-uniform coefficients of the pairs i < j, picked per lane */
    load([&](auto f) {
      R r = f(0, 1);
#pragma unroll
      for (int i = 0; i < N; i++)
#pragma unroll
        for (int j = i + 1; j < N; j++) {
          const R x = f(i, j);
          r = p == i * N + j ? x : r;
        }
      return r;
    });
  } else {
    load([&](auto f) { return f(p / N, p % N); });
  }
  return k;
}

/* delta-phi of the centre cell before the simplex projection, with phi, its Laplacians, psi and the active phases (those of
 * nonzero Laplacian; none: out is zero and psi is not formed). V: a RegView. */
template <int N, int NC, typename R, class V>
GP_HD unsigned phi_rates_pairs(const Model<R> &m, const V &v, R *phi, R *divphi, R *psi, R *out) {
  unsigned active = 0u;
#pragma unroll
  for (int a = 0; a < N; a++) {
    phi[a] = v.ph(a, 0, 0);
    divphi[a] = divx<V>(m, (gx(m, v, a, 0, 0) - gx(m, v, a, -1, 0)));
    divphi[a] += divy<V>(m, (gy(m, v, a, 0, 0) - gy(m, v, a, 0, -1)));
    active |= fabs(divphi[a]) > R(0.0) ? 1u << a : 0u;
    out[a] = R(0.0);
  }
  if (!active) return 0u; /* no lambda, no tau */
  const bool sym = m.pairs_sym != 0;
  unsigned todo = pairs_to_visit<N>(m, v, active);
  R A1[N], A2[N], D1[N], D2[N];
#pragma unroll
  for (int a = 0; a < N; a++) A1[a] = A2[a] = D1[a] = D2[a] = R(0.0);
  while (todo) {
    const int p = __builtin_ctz(todo), a = p / N, b = p % N;
    todo &= todo - 1u;
    RegStore<2, 0, R> rs;
    pair_stencil<N>(v, a, b, rs);
    const PairCoef<R> k = pair_coef<N>(m, p);
    const RegView<2, 0, R, V::kPow2, V::kFast> w{&rs, 0, 0};
    /* the centre term dA/dphi: x1 + x2 of phase a, y1 + y2 of phase b */
    R x1, x2 = R(0.0), y1, y2 = R(0.0);
    {
      const R pa = w.ph(0, 0, 0), pb = w.ph(1, 0, 0);
      const R ga[2] = {cx(m, w, 0, 0, 0), cy(m, w, 0, 0, 0)}, gb[2] = {cx(m, w, 1, 0, 0), cy(m, w, 1, 0, 0)};
      const R r[2] = {pa * gb[0] - pb * ga[0], pa * gb[1] - pb * ga[1]};
      if (m.fn_aniso) {
        R q[2], d[2], ac, ta[2], tb[2];
        rot2(k.rot, r, q);
        if constexpr (V::kFast) {
          aniso_ac_dadq_fast(k.dab, q, ac, d);
        } else {
          aniso_dadq(k.dab, q, d);
          ac = aniso_ac(k.dab, q);
        }
        rot2(k.rot, ga, ta);
        rot2(k.rot, gb, tb);
        const R g1 = k.gamma * (ac * ac), g2 = k.gamma * ac * qnorm2(q);
        x1 = (q[0] * tb[0] + q[1] * tb[1]) * g1;
        y1 = -((q[0] * ta[0] + q[1] * ta[1]) * g1);
        x2 = (d[0] * tb[0] + d[1] * tb[1]) * g2;
        y2 = -((d[0] * ta[0] + d[1] * ta[1]) * g2);
      } else {
        x1 = (r[0] * gb[0] + r[1] * gb[1]) * k.gamma;
        y1 = -((r[0] * ga[0] + r[1] * ga[1]) * k.gamma);
      }
    }
    /* the divergence term: its faces, then phase a with weights -s_b and phase b with s_a */
    R saF, sbF, f1F, f2F, saB, sbB, f1B, f2B, saR, sbR, f1R, f2R, saL, sbL, f1L, f2L;
    pair_face<0>(m, k, w, 0, 0, saF, sbF, f1F, f2F);
    pair_face<0>(m, k, w, -1, 0, saB, sbB, f1B, f2B);
    pair_face<1>(m, k, w, 0, 0, saR, sbR, f1R, f2R);
    pair_face<1>(m, k, w, 0, -1, saL, sbL, f1L, f2L);
    R u1 = divx<V>(m, (f1F * (-sbF) - f1B * (-sbB)));
    u1 += divy<V>(m, (f1R * (-sbR) - f1L * (-sbL)));
    R w1 = divx<V>(m, (f1F * saF - f1B * saB));
    w1 += divy<V>(m, (f1R * saR - f1L * saL));
    u1 *= k.gamma;
    w1 *= k.gamma;
    R u2 = R(0.0), w2 = R(0.0);
    if (m.fn_aniso) {
      u2 = divx<V>(m, (f2F * (-sbF) - f2B * (-sbB)));
      u2 += divy<V>(m, (f2R * (-sbR) - f2L * (-sbL)));
      w2 = divx<V>(m, (f2F * saF - f2B * saB));
      w2 += divy<V>(m, (f2R * saR - f2L * saL));
      u2 *= k.gamma;
      w2 *= k.gamma;
    }
#pragma unroll
    for (int c = 0; c < N; c++) {
      const bool ia = c == a, ib = sym && c == b;
      A1[c] += ia ? x1 : ib ? y1 : R(0.0);
      A2[c] += ia ? x2 : ib ? y2 : R(0.0);
      D1[c] += ia ? u1 : ib ? w1 : R(0.0);
      D2[c] += ia ? u2 : ib ? w2 : R(0.0);
    }
  }
  R mu[NC > 0 ? NC : 1];
#pragma unroll
  for (int k = 0; k < NC; k++) mu[k] = v.m(k, 0, 0);
  psi_all<N, NC>(m, mu, psi);
  R lambda[N], sum_lambda = R(0.0);
  int count = 0;
#pragma unroll
  for (int a = 0; a < N; a++) {
    lambda[a] = R(0.0);
    if ((active >> a) & 1u) {
      const R dA = R(2.0) * (A1[a] + A2[a]), dD = R(2.0) * (D1[a] + D2[a]) + R(0.0);
      R dp = R(0.0);
#pragma unroll
      for (int b = 0; b < N; b++) dp += psi[b] * dhphi<N>(phi, b, a);
      lambda[a] = m.eps * (-dA + dD) - m.inv_eps * dwdphi<N>(m, phi, divphi, a, false) - dp;
      sum_lambda += lambda[a];
      count++;
    }
  }
  if (count) sum_lambda = qdiv(sum_lambda, R(count));
  const R den = tau_of<N>(m, phi) * m.eps;
#pragma unroll
  for (int a = 0; a < N; a++) out[a] = (active >> a) & 1u ? qdiv(m.dt * (lambda[a] - sum_lambda), den) : R(0.0);
  return active;
}

/* delta-phi of the centre cell: phi_delta (not its smoothing form; the projection clamps a negative phi of an inactive
 * phase too). V: a RegView. */
template <int N, int NC, typename R, class V>
GP_HD void phi_delta_pairs(const Model<R> &m, const V &v, R *out) {
  R phi[N], divphi[N], psi[N];
  phi_rates_pairs<N, NC>(m, v, phi, divphi, psi, out);
  project_simplex<N>(phi, divphi, out);
}

/* s_obst of solid a (varying per lane) from the phases of a point: the other phases, in ascending order, are picked for
 * the pair sum of hphi */
template <int N, typename R>
GP_HD R s_obst_of(int a, const R *phi) {
  const R p = pick<N - 1>(a, [&](int c) { return phi[c]; });
  if (!(p * (R(1.0) - p) > R(0.0))) return R(0.0);
  R o[N - 1], s1 = R(0.0);
#pragma unroll
  for (int i = 0; i < N - 1; i++) {
    const R lo = phi[i], hi = phi[i + 1];
    o[i] = i < a ? lo : hi;
  }
#pragma unroll
  for (int b = 0; b < N - 1; b++)
#pragma unroll
    for (int c = b + 1; c < N - 1; c++) s1 += o[b] * o[c];
  s1 *= R(2.0) * p;
  const R h = R(3.0) * p * p - R(2.0) * p * p * p + s1;
  return qdiv(p * (R(1.0) - h), (qsqrt(p * (R(1.0) - p))));
}

/* The four face currents of the centre cell: jat_x(0,0), jat_x(-1,0), jat_y(0,0), jat_y(0,-1). V: a RegView;
 * y: allocated y of the centre. */
template <int N, int NC, typename R, class V>
GP_HD void jat_faces(const Model<R> &m, const V &v, int64_t y, R *jx0, R *jxb, R *jy0, R *jyl) {
  constexpr int L = N - 1;
  constexpr int oi[5] = {0, 1, -1, 0, 0}, oj[5] = {0, 0, 0, 1, -1};
  R j[4][NC];
#pragma unroll
  for (int f = 0; f < 4; f++)
#pragma unroll
    for (int k = 0; k < NC; k++) j[f][k] = R(0.0);
  /* face f lies between the centre and point f + 1; it carries a current when delta-phi of a solid moves on either side */
  bool moves[5], on[4], some = false;
#pragma unroll
  for (int o = 0; o < 5; o++) {
    moves[o] = false;
#pragma unroll
    for (int a = 0; a < L; a++) moves[o] = moves[o] || v.dp(a, oi[o], oj[o]) != R(0.0);
  }
#pragma unroll
  for (int f = 0; f < 4; f++) {
    on[f] = moves[0] || moves[f + 1];
    if (f >= 2) {
      const int64_t yf = f == 2 ? y : y - 1;
      on[f] = on[f] && !(yf == 0 || yf == m.jat_skip_row);
    }
    some = some || on[f];
  }
  unsigned todo = some ? phases_present<L, R>(v) : 0u;
  /* normal (n) and tangential (t) gradient of phase view w's field 0 on face f */
  auto grad = [&](const auto &w, int c, int f, R &n, R &t) {
    const int i = f == 1 ? -1 : 0, jj = f == 3 ? -1 : 0;
    if (f < 2) {
      t = R(0.5) * (cy(m, w, c, i, jj) + cy(m, w, c, i + 1, jj));
      n = gx(m, w, c, i, jj);
    } else {
      t = R(0.5) * (cx(m, w, c, i, jj) + cx(m, w, c, i, jj + 1));
      n = gy(m, w, c, i, jj);
    }
  };
  R nL[4], tL[4], gL[4], cl[5][NC];
  if (todo) {
#pragma unroll
    for (int f = 0; f < 4; f++) {
      grad(v, L, f, nL[f], tL[f]);
      gL[f] = qsqrt(tL[f] * tL[f] + nL[f] * nL[f]);
    }
#pragma unroll
    for (int o = 0; o < 5; o++) {
      R mu[NC];
#pragma unroll
      for (int k = 0; k < NC; k++) mu[k] = v.m(k, oi[o], oj[o]);
#pragma unroll
      for (int k = 0; k < NC; k++) cl[o][k] = c_mu<NC>(m, mu, L, k);
    }
  }
  while (todo) {
    const int a = __builtin_ctz(todo);
    todo &= todo - 1u;
    RegStore<1, 0, R> rs;
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
      for (int c = 0; c < 3; c++) rs.p[0][r][c] = pick<L>(a, [&](int q) { return v.ph(q, r - 1, c - 1); });
    const RegView<1, 0, R, V::kPow2, V::kFast> w{&rs, 0, 0};
    R cmu[NC][NC], bmu[NC], dr[NC];
#pragma unroll
    for (int k = 0; k < NC; k++) {
      bmu[k] = pick<L>(a, [&](int q) { return m.Bmu[q][k]; });
      dr[k] = pick<L>(a, [&](int q) { return m.dratio[q][k]; });
#pragma unroll
      for (int l = 0; l < NC; l++) cmu[k][l] = pick<L>(a, [&](int q) { return m.cmu[q][k][l]; });
    }
    /* per point: s (obstacle potential) times the composition step, times delta-phi of the solid */
    R e[5][NC];
#pragma unroll
    for (int o = 0; o < 5; o++) {
      R mu[NC], s = R(0.0);
#pragma unroll
      for (int k = 0; k < NC; k++) mu[k] = v.m(k, oi[o], oj[o]);
      if (m.fn_w == 1) {
        R ph[N];
#pragma unroll
        for (int c = 0; c < N; c++) ph[c] = v.ph(c, oi[o], oj[o]);
        s = s_obst_of<N>(a, ph);
      }
      const R d = pick<L>(a, [&](int q) { return v.dp(q, oi[o], oj[o]); });
#pragma unroll
      for (int k = 0; k < NC; k++) {
        R cs = R(0.0);
#pragma unroll
        for (int l = 0; l < NC; l++) cs += cmu[k][l] * (mu[l] - bmu[l]);
        e[o][k] = m.fn_w == 1 ? s * (cl[o][k] - cs) * d : (cl[o][k] - cs) * d;
      }
    }
    const R half = m.fn_w == 2 ? m.jat_well : R(0.5);
#pragma unroll
    for (int f = 0; f < 4; f++) {
      R n, t;
      grad(w, 0, f, n, t);
      const R ng = qsqrt(t * t + n * n);
      if (!(ng != R(0.0)) || !on[f]) continue;
      /* the projection on the liquid's normal, its terms in the order of the normal component first */
      R sp = n * nL[f];
      sp += t * tL[f];
      if (gL[f] > R(0.0)) sp = qdiv(sp, (gL[f] * ng));
#pragma unroll
      for (int k = 0; k < NC; k++)
        j[f][k] += qdiv(dr[k] * fabs(sp) * half * (e[f + 1][k] + e[0][k]) * n, ng);
    }
  }
#pragma unroll
  for (int k = 0; k < NC; k++) {
    jx0[k] = j[0][k];
    jxb[k] = j[1][k];
    jy0[k] = j[2][k];
    jyl[k] = j[3][k];
  }
}

}  // namespace gpk
