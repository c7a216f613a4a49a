// Group solvers of the spring chains for the methods beside DOPRI5: RK4, Euler,
// the embedded family and DOP853 with G lanes per system and C masses per lane
// (GroupCommon in de_spring_solvers.h), every vector in registers.
//
// They run the operations of the one-lane solvers (VecFixed, VecErk, VecDop853)
// component by component, so their results are those solvers' bits: RK4 and
// Euler have no norm, the embedded family's is a maximum (which has no order),
// and the sums that do have an order -- DOP853's two error sums, the initial
// step's norms and the stiffness test -- are added in the reference's component
// order from LDS (ordered2).
//
// Bound: FP64 VALU, and below a few thousand systems the serial chain of the
// longest solve.  One lane per system streams about 7 (RK4) to 26 (DOP853)
// state vectors through memory in every step, each lane of a wave at its own
// addresses: 727 ms for 8192 chains of 4 to 256 masses over 500 RK4 steps
// against 1.74 ms here, and 536 ms against 0.98 ms for 4099 chains with DOP853
// at rtol 1e-8 over t in [0, 10].
#pragma once

#include "de_erk_lane.h"
#include "de_spring_solvers.h"

namespace de {

#if defined(__HIP_DEVICE_COMPILE__) || defined(__HIPCC__)
// Orders the LDS accesses of one wavefront (the hardware keeps them in order;
// this keeps the compiler from moving them).
DE_DEV void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Two sums over the state's components in the order x_0 .. x_{N-1}, v_0 ..
// v_{N-1}, each added one component after the other from 0 (the reference's
// loops), with both results on every lane of the group.  The terms go to LDS
// in component order; even lanes then add the first sum's and odd lanes the
// second's, so a step of the two serial chains is one addition per wavefront.
// The terms are squares: starting from 0 or from the first term is the same.
// The rows are 4 banks apart so that the two broadcast reads of a group do not
// meet on a bank.
template <int G, int C>
DE_DEV void ordered2(int l, int nm, const double* ax, const double* av, const double* bx,
                     const double* bv, double* sa, double* sb) {
  constexpr int kRow = 2 * G * C + 2;
  __shared__ __align__(16) double buf[kGroupBlock / G][2][kRow];
  double* rows = &buf[threadIdx.x / G][0][0];
  wave_lds_fence();  // the readers of the last call are done
#pragma unroll
  for (int q = 0; q < C; ++q) {
    const int j = l * C + q;
    if (j < nm) {
      rows[j] = ax[q];
      rows[nm + j] = av[q];
      rows[kRow + j] = bx[q];
      rows[kRow + nm + j] = bv[q];
    }
  }
  wave_lds_fence();
  const double2* row = (const double2*)(rows + (l & 1) * kRow);
  double s = 0.0;
#pragma unroll 4
  for (int e = 0; e < nm; ++e) {  // 2 nm components
    const double2 w = row[e];
    s = s + w.x;
    s = s + w.y;
  }
  constexpr int kEven = 0xA0, kOdd = 0xF5;  // quad_perm [0,0,2,2] and [1,1,3,3]
  *sa = dpp_double<kEven>(s);
  *sb = dpp_double<kOdd>(s);
}

// The automatic initial step of order ORDER (h_init.rs:45-135), the operations
// of VecCommon::h_init.
template <int ORDER, int G, int C>
DE_DEV double group_h_init(const SpringArgs& A, const GroupCommon<G, C, false>& S) {
  const OdeArgs& a = A.o;
  double f0x[C], f0v[C], skx[C], skv[C], ax[C], av[C], bx[C], bv[C], f1x[C], f1v[C];
  S.rhs(S.x, S.v, f0x, f0v);
#pragma unroll
  for (int q = 0; q < C; ++q) {
    const int j = S.l * C + q;
    const bool real = j < S.nm;
    skx[q] = real ? S.at(a, j) + S.rt(a, j) * fabs(S.x[q]) : 1.0;
    skv[q] = real ? S.at(a, S.nm + j) + S.rt(a, S.nm + j) * fabs(S.v[q]) : 1.0;
    const double u = f0x[q] / skx[q], u2 = f0v[q] / skv[q];
    const double w = S.x[q] / skx[q], w2 = S.v[q] / skv[q];
    ax[q] = u * u;
    av[q] = u2 * u2;
    bx[q] = w * w;
    bv[q] = w2 * w2;
  }
  double dnf, dny, der2;
  ordered2<G, C>(S.l, S.nm, ax, av, bx, bv, &dnf, &dny);
  double hh = (dnf <= 1.0e-10 || dny <= 1.0e-10) ? 1.0e-6 : sqrt(dny / dnf) * 0.01;
  hh = fmin(hh, a.h_max);
  hh *= S.dir;
#pragma unroll
  for (int q = 0; q < C; ++q) {
    ax[q] = S.x[q] + hh * f0x[q];
    av[q] = S.v[q] + hh * f0v[q];
  }
  S.rhs(ax, av, f1x, f1v);
#pragma unroll
  for (int q = 0; q < C; ++q) {
    const double d = (f1x[q] - f0x[q]) / skx[q], d2 = (f1v[q] - f0v[q]) / skv[q];
    ax[q] = d * d;
    av[q] = d2 * d2;
  }
  ordered2<G, C>(S.l, S.nm, ax, av, ax, av, &der2, &dny);
  der2 = sqrt(der2) / fabs(hh);
  const double der12 = fmax(sqrt(dnf), der2);
  const double h1 = der12 <= 1.0e-15 ? fabs(hh) * 1.0e-3
                                     : DE_CTRL_POW(0.01 / der12, 1.0 / (double)ORDER);
  const double interval = fabs(S.tf - S.t);
  hh = fmin(fmax(fmin(fmin(fabs(hh) * 100.0, h1), a.h_max), a.h_min), interval);
  return hh * S.dir;
}

// Maximum of a non-negative value over the group's lanes, on every lane.
template <int G>
DE_DEV double gmax(double m) {
  if constexpr (G >= 2) m = fmax(m, dpp_double<kDppQuadSwap1>(m));
  if constexpr (G >= 4) m = fmax(m, dpp_double<kDppQuadSwap2>(m));
  if constexpr (G >= 8) m = fmax(m, dpp_double<kDppHalfMirror>(m));
  if constexpr (G >= 16) m = fmax(m, dpp_double<kDppMirror>(m));
  double a, b;
  if constexpr (G >= 32) {
    swap_pair<16>(m, &a, &b);
    m = fmax(a, b);
  }
  if constexpr (G >= 64) {
    swap_pair<32>(m, &a, &b);
    m = fmax(a, b);
  }
  return m;
}

// The cubic Hermite interpolant on [tp, tn] (cubic_hermite_interpolate,
// src/interpolate.rs:40-60): its four weights, then per component the sum in
// the reference's order.
struct HermiteWeights {
  double h00, w10, h01, w11;
  DE_DEV void at(double te, double tp, double tn) {
    const double hh = tn - tp;
    const double s = (te - tp) / hh;
    const double s2 = s * s;
    const double s3 = s2 * s;
    h00 = 2.0 * s3 - 3.0 * s2 + 1.0;
    const double h10 = s3 - 2.0 * s2 + s;
    h01 = -2.0 * s3 + 3.0 * s2;
    const double h11 = s3 - s2;
    w10 = h10 * hh;
    w11 = h11 * hh;
  }
};

// -------------------------------------------------------------- GroupFixed --
// RK4 / Euler (the operations of VecFixed).
template <int STAGES, int G, int C>
struct GroupFixed : GroupCommon<G, C, false> {
  static constexpr bool OUT = false;
  DE_GROUP_MEMBERS
  int64_t acc;  // steps taken; evals = 1 + STAGES acc

  DE_DEV void finish(const SpringArgs& A, int32_t st) const {
    write(A, st, acc, 0, st == kBadInput ? 0 : 1 + STAGES * acc);
  }

  DE_DEV bool init(const SpringArgs& A, int64_t s, int lane_in_group) {
    const OdeArgs& a = A.o;
    const double t0 = setup(A, s, lane_in_group);
    acc = 0;
    bool ok = dir == 1.0 || dir == -1.0;
    double h0 = a.h0;
    if (h0 == 0.0) h0 = fabs(tf - t0) / 100.0;
    ok = ok && validate_step_size(h0, a.h_min, a.h_max, t0, tf);
    if (!ok) {
      finish(A, kBadInput);
      return false;
    }
    h = h0;
    rhs(x, v, k0x, k0v);
    output_start(A);
    return true;
  }

  DE_DEV bool advance(const SpringArgs& A) {
    const OdeArgs& a = A.o;
    if ((t + h - tf) * dir > 0.0) {
      const double hn = tf - t;
      if (fabs(hn) < kTenEps) {
        finish(A, kComplete);
        return true;
      }
      h = hn;
    }
    if (acc >= a.max_steps) {
      finish(A, kMaxSteps);
      return true;
    }
    double nx[C], nv[C], dnx[C], dnv[C];
    if constexpr (STAGES == 4) {
      double k1x[C], k1v[C], k2x[C], k2v[C], k3x[C], k3v[C], sx[C], sv[C];
      const double hh = 0.5 * h;
#pragma unroll
      for (int q = 0; q < C; ++q) {
        sx[q] = x[q] + hh * k0x[q];
        sv[q] = v[q] + hh * k0v[q];
      }
      rhs(sx, sv, k1x, k1v);
#pragma unroll
      for (int q = 0; q < C; ++q) {
        sx[q] = x[q] + hh * k1x[q];
        sv[q] = v[q] + hh * k1v[q];
      }
      rhs(sx, sv, k2x, k2v);
      const double h1 = 1.0 * h;
#pragma unroll
      for (int q = 0; q < C; ++q) {
        sx[q] = x[q] + h1 * k2x[q];
        sv[q] = v[q] + h1 * k2v[q];
      }
      rhs(sx, sv, k3x, k3v);
      const double b0h = (1.0 / 6.0) * h, b1h = (1.0 / 3.0) * h;
#pragma unroll
      for (int q = 0; q < C; ++q) {
        nx[q] = (((x[q] + b0h * k0x[q]) + b1h * k1x[q]) + b1h * k2x[q]) + b0h * k3x[q];
        nv[q] = (((v[q] + b0h * k0v[q]) + b1h * k1v[q]) + b1h * k2v[q]) + b0h * k3v[q];
      }
    } else {
      const double b0h = 1.0 * h;
#pragma unroll
      for (int q = 0; q < C; ++q) {
        nx[q] = x[q] + b0h * k0x[q];
        nv[q] = v[q] + b0h * k0v[q];
      }
    }
    const double tp = t;
    t += h;
    rhs(nx, nv, dnx, dnv);
    acc += 1;
    int32_t sol = -1;
    if (a.n_eval > 0) {
      const double tc = t;
      auto interp = [&](double te, double* ox, double* ov) {
        if (te < tp || te > tc) return false;
        HermiteWeights w;
        w.at(te, tp, tc);
#pragma unroll
        for (int q = 0; q < C; ++q) {
          ox[q] = ((w.h00 * x[q] + w.w10 * k0x[q]) + w.h01 * nx[q]) + w.w11 * dnx[q];
          ov[q] = ((w.h00 * v[q] + w.w10 * k0v[q]) + w.h01 * nv[q]) + w.w11 * dnv[q];
        }
        return true;
      };
      if (!emit(A, t, tp, nx, nv, interp)) sol = kOutOfBounds;
    }
#pragma unroll
    for (int q = 0; q < C; ++q) {
      x[q] = nx[q];
      v[q] = nv[q];
      k0x[q] = dnx[q];
      k0v[q] = dnv[q];
    }
    if (sol >= 0) {
      finish(A, sol);
      return true;
    }
    if (fabs(tf - t) <= kTenEps) {
      finish(A, kComplete);
      return true;
    }
    return false;
  }
};

// ---------------------------------------------------------------- GroupErk --
// The embedded family (the operations of VecErk, the coefficients read at
// compile-time indices as in ErkLane).  Zero coefficients and the masks of
// stages that are not finite: see de_erk_lane.h.
template <class Tab, int G, int C>
struct GroupErk : GroupCommon<G, C, false> {
  static constexpr bool OUT = false;
  DE_GROUP_MEMBERS
  static constexpr int S = Tab::S, I = Tab::I, O = Tab::O;
  static constexpr bool kBi = Tab::kBi, kFsal = Tab::kFsal;
  static constexpr uint32_t kZeroStages = erk_zero_stages<Tab>(kBi ? I : S, kBi);
  static constexpr int kAccEvals = (kFsal ? 0 : 1) + (kBi ? I - S : 0);
  int64_t acc, rej;
  int32_t base_ev, stiff;
  bool rejected_last;

  // The stages of one attempt and each component's non-finite masks.
  struct Stages {
    double kx[kBi ? I : S][C], kv[kBi ? I : S][C];
    uint32_t badx[C], badv[C];
    DE_DEV void mark(int r, uint32_t bit) {
#pragma unroll
      for (int q = 0; q < C; ++q) {
        badx[q] |= isfinite(kx[r][q]) ? 0u : bit;
        badv[q] |= isfinite(kv[r][q]) ? 0u : bit;
      }
    }
  };

  DE_DEV void finish(const SpringArgs& A, int32_t st) const {
    write(A, st, acc, rej,
          st == kBadInput ? 0 : base_ev + (int64_t)(S - 1) * (acc + rej) + (int64_t)kAccEvals * acc);
  }

  DE_DEV bool init(const SpringArgs& A, int64_t s, int lane_in_group) {
    const OdeArgs& a = A.o;
    const double t0 = setup(A, s, lane_in_group);
    acc = rej = 0;
    base_ev = 1;
    bool ok = dir == 1.0 || dir == -1.0;
    double h0 = a.h0;
    if (ok && h0 == 0.0) {
      h0 = group_h_init<O, G, C>(A, *this);
      base_ev = 5;
    }
    ok = ok && validate_step_size(h0, a.h_min, a.h_max, t0, tf);
    if (!ok) {
      finish(A, kBadInput);
      return false;
    }
    h = h0;
    rhs(x, v, k0x, k0v);
    h_prev = 0.0;
    stiff = 0;
    rejected_last = false;
    output_start(A);
    return true;
  }

  template <int R, int J>
  DE_DEV static void stage_term(const Stages& K, double hh, double* sx, double* sv) {
    constexpr double c = Tab::A[R][J];
    if constexpr (c != 0.0) {
      const double ah = c * hh;
#pragma unroll
      for (int q = 0; q < C; ++q) {
        sx[q] = sx[q] + ah * K.kx[J][q];
        sv[q] = sv[q] + ah * K.kv[J][q];
      }
    }
  }
  template <int R, int... J>
  DE_DEV static void stage_terms(std::integer_sequence<int, J...>, const Stages& K, double hh,
                                 double* sx, double* sv) {
    (stage_term<R, J>(K, hh, sx, sv), ...);
  }
  template <int R, int END>
  DE_DEV void stages(Stages& K, double hh) const {
    if constexpr (R < END) {
      double sx[C], sv[C];
#pragma unroll
      for (int q = 0; q < C; ++q) {
        sx[q] = x[q];
        sv[q] = v[q];
      }
      stage_terms<R>(std::make_integer_sequence<int, R>{}, K, hh, sx, sv);
      constexpr uint32_t z = erk_zero_mask(Tab::A[R], R);
      if constexpr (z != 0) {
#pragma unroll
        for (int q = 0; q < C; ++q) {
          sx[q] = (K.badx[q] & z) ? as_f64(kNaNBits) : sx[q];
          sv[q] = (K.badv[q] & z) ? as_f64(kNaNBits) : sv[q];
        }
      }
      rhs(sx, sv, K.kx[R], K.kv[R]);
      if constexpr ((kZeroStages >> R) & 1u) K.mark(R, 1u << R);
      stages<R + 1, END>(K, hh);
    }
  }

  template <int SEL, int J>
  DE_DEV static void weight_term(const Stages& K, double hh, int q, double& wx, double& wv) {
    constexpr double w = SEL ? Tab::BH[J] : Tab::B[J];
    if constexpr (w != 0.0) {
      const double wh = w * hh;
      wx = wx + wh * K.kx[J][q];
      wv = wv + wh * K.kv[J][q];
    }
  }
  template <int SEL, int... J>
  DE_DEV static void weight_terms(std::integer_sequence<int, J...>, const Stages& K, double hh,
                                  int q, double& wx, double& wv) {
    (weight_term<SEL, J>(K, hh, q, wx, wv), ...);
  }
  template <int SEL>
  DE_DEV void weighted(const Stages& K, int q, double* wx, double* wv) const {
    double rx = x[q], rv = v[q];
    weight_terms<SEL>(std::make_integer_sequence<int, S>{}, K, h, q, rx, rv);
    constexpr uint32_t z = erk_zero_mask(SEL ? Tab::BH : Tab::B, S);
    if constexpr (z != 0) {
      rx = (K.badx[q] & z) ? as_f64(kNaNBits) : rx;
      rv = (K.badv[q] & z) ? as_f64(kNaNBits) : rv;
    }
    *wx = rx;
    *wv = rv;
  }

  // One interpolation row: q(s) by Horner, then + (q h_prev) k[r].
  template <int R, int... P>
  DE_DEV static double bi_horner(std::integer_sequence<int, P...>, double s) {
    double qv = Tab::BI[R][O - 1];
    ((qv = qv * s + bi_coef<R, O - 2 - P>()), ...);
    return qv * s;
  }
  template <int R, int J>
  DE_DEV static double bi_coef() {
    constexpr double c = Tab::BI[R][J];
    return c;
  }
  template <int R>
  DE_DEV static void bi_term(const Stages& K, double s, double hp, bool all, double* ox,
                             double* ov) {
    constexpr bool zero = (erk_zero_bi_rows<Tab>() >> R) & 1u;
    if (zero && !all) return;
    const double wq = bi_horner<R>(std::make_integer_sequence<int, O - 1>{}, s) * hp;
#pragma unroll
    for (int q = 0; q < C; ++q) {
      ox[q] = ox[q] + wq * K.kx[R][q];
      ov[q] = ov[q] + wq * K.kv[R][q];
    }
  }
  template <int... R>
  DE_DEV static void bi_terms(std::integer_sequence<int, R...>, const Stages& K, double s,
                              double hp, bool all, double* ox, double* ov) {
    (bi_term<R>(K, s, hp, all, ox, ov), ...);
  }

  DE_DEV bool advance(const SpringArgs& A) {
    const OdeArgs& a = A.o;
    if ((t + h - tf) * dir > 0.0) {
      const double hn = tf - t;
      if (fabs(hn) < kTenEps) {
        finish(A, kComplete);
        return true;
      }
      h = hn;
    }
    if (fabs(h) < fabs(h_prev) * 1e-14) {
      finish(A, kStepSize);
      return true;
    }
    if (acc + rej >= a.max_steps) {
      finish(A, kMaxSteps);
      return true;
    }
    Stages K;
    const uint32_t hbad = isfinite(h) ? 0u : ~0u;
#pragma unroll
    for (int q = 0; q < C; ++q) {
      K.kx[0][q] = k0x[q];
      K.kv[0][q] = k0v[q];
      K.badx[q] = K.badv[q] = hbad;
    }
    if constexpr (kZeroStages & 1u) K.mark(0, 1u);
    stages<1, S>(K, h);
    double nx[C], nv[C];
    double m = 0.0;
#pragma unroll
    for (int q = 0; q < C; ++q) {
      double lx, lv;
      weighted<0>(K, q, &nx[q], &nv[q]);
      weighted<1>(K, q, &lx, &lv);
      const int j = l * C + q;
      if (j < nm) {
        const double ex = nx[q] + (-1.0) * lx, ev = nv[q] + (-1.0) * lv;
        const double skx = at(a, j) + rt(a, j) * fmax(fabs(x[q]), fabs(nx[q]));
        const double skv = at(a, nm + j) + rt(a, nm + j) * fmax(fabs(v[q]), fabs(nv[q]));
        m = fmax(m, fabs(ex / skx));
        m = fmax(m, fabs(ev / skv));
      }
    }
    m = gmax<G>(m);
    double scale = a.safety * DE_CTRL_POW(m, -(1.0 / (double)O));
    scale = fmin(fmax(scale, a.min_scale), a.max_scale);
    const bool accept = m <= 1.0;
    const int32_t stiff_next = accept ? (rejected_last ? 0 : stiff) : stiff + 1;
    const bool stop = !accept && (int64_t)stiff_next >= a.max_rejects;
    const double t_new = t + h;
    int32_t sol = -1;
    if (accept) {
      double dnx[C], dnv[C];
      if constexpr (kFsal) {
#pragma unroll
        for (int q = 0; q < C; ++q) {
          dnx[q] = K.kx[S - 1][q];
          dnv[q] = K.kv[S - 1][q];
        }
      } else {
        rhs(nx, nv, dnx, dnv);
      }
      // The interpolant is built when the next t_eval point is not past the
      // new time.
      if (teval_due(a, t_new)) {
        const double tp = t, hp = h;
        bool fin = true;
        if constexpr (kBi) {
          stages<S, I>(K, h);
          constexpr uint32_t zr = erk_zero_bi_rows<Tab>();
          if constexpr (zr != 0) {
            uint32_t any = 0;
#pragma unroll
            for (int q = 0; q < C; ++q) any |= K.badx[q] | K.badv[q];
            // Over the whole state, as the one-lane solver.
            fin = gmax<G>((any & zr) ? 1.0 : 0.0) == 0.0;
          }
        }
        auto interp = [&](double te, double* ox, double* ov) {
          if (te < tp || te > t_new) return false;
          if constexpr (kBi) {
            const double s = (te - tp) / hp;
            const bool all = !fin || !isfinite(s) || !isfinite(hp);
#pragma unroll
            for (int q = 0; q < C; ++q) {
              ox[q] = x[q];
              ov[q] = v[q];
            }
            bi_terms(std::make_integer_sequence<int, I>{}, K, s, hp, all, ox, ov);
          } else {
            HermiteWeights w;
            w.at(te, tp, t_new);
#pragma unroll
            for (int q = 0; q < C; ++q) {
              ox[q] = (((0.0 + w.h00 * x[q]) + w.w10 * K.kx[0][q]) + w.h01 * nx[q]) + w.w11 * dnx[q];
              ov[q] = (((0.0 + w.h00 * v[q]) + w.w10 * K.kv[0][q]) + w.h01 * nv[q]) + w.w11 * dnv[q];
            }
          }
          return true;
        };
        if (!emit(A, t_new, tp, nx, nv, interp)) sol = kOutOfBounds;
      }
      h_prev = h;
      t = t_new;
#pragma unroll
      for (int q = 0; q < C; ++q) {
        x[q] = nx[q];
        v[q] = nv[q];
        k0x[q] = dnx[q];
        k0v[q] = dnv[q];
      }
    }
    scale = accept && rejected_last ? fmin(scale, 1.0) : scale;
    rejected_last = !accept;
    stiff = stiff_next;
    acc += accept ? 1 : 0;
    rej += (accept || stop) ? 0 : 1;
    h = constrain_step_size(h * scale, a.h_min, a.h_max);
    if (stop) {
      finish(A, kStiffness);
      return true;
    }
    if (sol >= 0) {
      finish(A, sol);
      return true;
    }
    if (accept && fabs(tf - t) <= kTenEps) {
      finish(A, kComplete);
      return true;
    }
    return false;
  }
};

// ------------------------------------------------------------- GroupDop853 --
// DOP853 (the operations of VecDop853).
template <int G, int C>
struct GroupDop853 : GroupCommon<G, C, false> {
  static constexpr bool OUT = false;
  DE_GROUP_MEMBERS
  int64_t acc, rej, steps;
  int32_t base_ev, stiff, nonstiff, countdown;
  bool rejected_last;

  DE_DEV void finish(const SpringArgs& A, int32_t st) const {
    write(A, st, acc, rej, st == kBadInput ? 0 : base_ev + 15 * acc + 11 * rej);
  }

  DE_DEV bool init(const SpringArgs& A, int64_t s, int lane_in_group) {
    const OdeArgs& a = A.o;
    const double t0 = setup(A, s, lane_in_group);
    acc = rej = steps = 0;
    bool ok = dir == 1.0 || dir == -1.0;
    double h0 = a.h0;
    base_ev = 1;
    if (ok && h0 == 0.0) {
      h0 = group_h_init<8, G, C>(A, *this);
      base_ev = 3;
    }
    ok = ok && validate_step_size(h0, a.h_min, a.h_max, t0, tf);
    if (!ok) {
      finish(A, kBadInput);
      return false;
    }
    h = h0;
    rhs(x, v, k0x, k0v);
    h_prev = 0.0;
    stiff = nonstiff = 0;
    countdown = 100;
    rejected_last = false;
    output_start(A);
    return true;
  }

  struct Stages {
    double kx[16][C], kv[16][C];
  };

  template <int R, int J>
  DE_DEV static void stage_term(const Stages& K, double hh, double* sx, double* sv) {
    constexpr double c = d8::A[R][J];
    if constexpr (c != 0.0) {
      const double ah = c * hh;
#pragma unroll
      for (int q = 0; q < C; ++q) {
        sx[q] = sx[q] + ah * K.kx[J][q];
        sv[q] = sv[q] + ah * K.kv[J][q];
      }
    }
  }
  template <int R, int... J>
  DE_DEV static void stage_terms(std::integer_sequence<int, J...>, const Stages& K, double hh,
                                 double* sx, double* sv) {
    (stage_term<R, J>(K, hh, sx, sv), ...);
  }
  // Stages R .. END-1; (sx, sv) ends as the last stage's input.
  template <int R, int END>
  DE_DEV void stages(Stages& K, double hh, double* sx, double* sv) const {
    if constexpr (R < END) {
#pragma unroll
      for (int q = 0; q < C; ++q) {
        sx[q] = x[q];
        sv[q] = v[q];
      }
      stage_terms<R>(std::make_integer_sequence<int, R>{}, K, hh, sx, sv);
      rhs(sx, sv, K.kx[R], K.kv[R]);
      stages<R + 1, END>(K, hh, sx, sv);
    }
  }

  // sum_j w[j] k[j] from the first nonzero weight, W naming the weights.
  struct WB {
    static constexpr double at(int j) { return d8::B[j]; }
  };
  struct WE {
    static constexpr double at(int j) { return d8::ER[j]; }
  };
  template <int R>
  struct WI {
    static constexpr double at(int j) { return d8::BI[R][j]; }
  };
  template <class W, int J>
  static constexpr bool first_term() {
    for (int j = 0; j < J; ++j)
      if (W::at(j) != 0.0) return false;
    return true;
  }
  template <class W, int J>
  DE_DEV static void comb_term(const Stages& K, int q, double& sx, double& sv) {
    constexpr double w = W::at(J);
    if constexpr (w != 0.0) {
      if constexpr (first_term<W, J>()) {
        sx = w * K.kx[J][q];
        sv = w * K.kv[J][q];
      } else {
        sx = sx + w * K.kx[J][q];
        sv = sv + w * K.kv[J][q];
      }
    }
  }
  template <class W, int... J>
  DE_DEV static void comb(std::integer_sequence<int, J...>, const Stages& K, int q, double& sx,
                          double& sv) {
    (comb_term<W, J>(K, q, sx, sv), ...);
  }
  template <int J>
  DE_DEV static void bh_term(const Stages& K, int q, double& sx, double& sv) {
    constexpr double w = d8::BH[J];
    if constexpr (w != 0.0) {
      sx = sx + (-w) * K.kx[J][q];
      sv = sv + (-w) * K.kv[J][q];
    }
  }
  template <int... J>
  DE_DEV static void bh_terms(std::integer_sequence<int, J...>, const Stages& K, int q,
                              double& sx, double& sv) {
    (bh_term<J>(K, q, sx, sv), ...);
  }

  DE_DEV bool advance(const SpringArgs& A) {
    const OdeArgs& a = A.o;
    if ((t + h - tf) * dir > 0.0) {
      const double hn = tf - t;
      if (fabs(hn) < kTenEps) {
        finish(A, kComplete);
        return true;
      }
      h = hn;
    }
    if (fabs(h) < fabs(h_prev) * 1e-14) {
      finish(A, kStepSize);
      return true;
    }
    if (steps >= a.max_steps) {
      finish(A, kMaxSteps);
      return true;
    }
    steps += 1;
    countdown -= 1;
    const bool stiff_check = countdown == 0;
    if (stiff_check) countdown = 100;
    using Twelve = std::make_integer_sequence<int, 12>;
    Stages K;
#pragma unroll
    for (int q = 0; q < C; ++q) {
      K.kx[0][q] = k0x[q];
      K.kv[0][q] = k0v[q];
    }
    double sx[C], sv[C];  // the stage-11 input
    stages<1, 12>(K, h, sx, sv);
    double segx[C], segv[C], nx[C], nv[C], ex[C], ev[C], e2x[C], e2v[C];
#pragma unroll
    for (int q = 0; q < C; ++q) {
      comb<WB>(Twelve{}, K, q, segx[q], segv[q]);
      nx[q] = x[q] + h * segx[q];
      nv[q] = v[q] + h * segv[q];
      double esx = 0.0, esv = 0.0, e2sx = segx[q], e2sv = segv[q];
      comb<WE>(Twelve{}, K, q, esx, esv);
      bh_terms(Twelve{}, K, q, e2sx, e2sv);
      const int j = l * C + q;
      const bool real = j < nm;
      const double skx =
          real ? at(a, j) + rt(a, j) * fmax(fabs(x[q]), fabs(nx[q])) : 1.0;
      const double skv =
          real ? at(a, nm + j) + rt(a, nm + j) * fmax(fabs(v[q]), fabs(nv[q])) : 1.0;
      esx = esx / skx;
      e2sx = e2sx / skx;
      esv = esv / skv;
      e2sv = e2sv / skv;
      ex[q] = esx * esx;
      ev[q] = esv * esv;
      e2x[q] = e2sx * e2sx;
      e2v[q] = e2sv * e2sv;
    }
    double err, err2;
    ordered2<G, C>(l, nm, ex, ev, e2x, e2v, &err, &err2);
    double deno = err + 0.01 * err2;
    if (deno <= 0.0) deno = 1.0;
    err = fabs(h) * err * sqrt(1.0 / (deno * (double)(2 * nm)));
    double scale = a.safety * DE_CTRL_POW(err, -0.125);
    scale = fmin(fmax(scale, a.min_scale), a.max_scale);
    if (err <= 1.0) {
      const double t_new = t + h;
      rhs(nx, nv, K.kx[12], K.kv[12]);  // f(t_new, y_new), the 13th stage of the dense output
      if (stiff_check) {
        double ux[C], uv[C], wx[C], wv[C];
#pragma unroll
        for (int q = 0; q < C; ++q) {
          ux[q] = segx[q] - K.kx[11][q];
          uv[q] = segv[q] - K.kv[11][q];
          wx[q] = K.kx[12][q] - sx[q];
          wv[q] = K.kv[12][q] - sv[q];
          ux[q] *= ux[q];
          uv[q] *= uv[q];
          wx[q] *= wx[q];
          wv[q] *= wv[q];
        }
        double stdnum, stden;
        ordered2<G, C>(l, nm, ux, uv, wx, wv, &stdnum, &stden);
        if (stden > 0.0) {
          if (stiff_exceeds(h, stdnum, stden)) {
            nonstiff = 0;
            stiff += 1;
            if (stiff == 15) {
              finish(A, kStiffness);
              return true;
            }
          }
        } else {
          nonstiff += 1;
          if (nonstiff == 6) stiff = 0;
        }
      }
      int32_t sol = -1;
      // The interpolant (three more stages and seven coefficient vectors) is
      // built when the next t_eval point is not past the new time.
      if (teval_due(a, t_new)) {
        double c1x[C], c1v[C], c2x[C], c2v[C], c3x[C], c3v[C], cx[4][C], cv[4][C];
#pragma unroll
        for (int q = 0; q < C; ++q) {
          const double dx = nx[q] + (-1.0) * x[q], dv = nv[q] + (-1.0) * v[q];
          const double bx = h * k0x[q] + (-1.0) * dx, bv = h * k0v[q] + (-1.0) * dv;
          c1x[q] = dx;
          c1v[q] = dv;
          c2x[q] = bx;
          c2v[q] = bv;
          c3x[q] = (dx + (-h) * K.kx[12][q]) + (-1.0) * bx;
          c3v[q] = (dv + (-h) * K.kv[12][q]) + (-1.0) * bv;
        }
        double tx[C], tv[C];
        stages<13, 16>(K, h, tx, tv);
        using Sixteen = std::make_integer_sequence<int, 16>;
#pragma unroll
        for (int q = 0; q < C; ++q) {
          double rx = 0.0, rv = 0.0;
          comb<WI<4>>(Sixteen{}, K, q, rx, rv);
          cx[0][q] = rx * h;
          cv[0][q] = rv * h;
          comb<WI<5>>(Sixteen{}, K, q, rx, rv);
          cx[1][q] = rx * h;
          cv[1][q] = rv * h;
          comb<WI<6>>(Sixteen{}, K, q, rx, rv);
          cx[2][q] = rx * h;
          cv[2][q] = rv * h;
          comb<WI<7>>(Sixteen{}, K, q, rx, rv);
          cx[3][q] = rx * h;
          cv[3][q] = rv * h;
        }
        const double tp = t, hp = h;
        auto horner = [](double c7, double c6, double c5, double c4, double c3, double c2,
                         double c1, double y, double s, double s1) {
          double r = c7;
          r = r * s1 + c6;
          r = r * s + c5;
          r = r * s1 + c4;
          r = r * s1 + c3;
          r = r * s + c2;
          r = r * s1 + c1;
          return y + s * r;
        };
        auto interp = [&](double te, double* ox, double* ov) {
          if (te < tp || te > t_new) return false;
          const double s = (te - tp) / hp;
          const double s1 = 1.0 - s;
#pragma unroll
          for (int q = 0; q < C; ++q) {
            ox[q] = horner(cx[3][q], cx[2][q], cx[1][q], cx[0][q], c3x[q], c2x[q], c1x[q], x[q],
                           s, s1);
            ov[q] = horner(cv[3][q], cv[2][q], cv[1][q], cv[0][q], c3v[q], c2v[q], c1v[q], v[q],
                           s, s1);
          }
          return true;
        };
        if (!emit(A, t_new, tp, nx, nv, interp)) sol = kOutOfBounds;
      }
      h_prev = h;
      t = t_new;
#pragma unroll
      for (int q = 0; q < C; ++q) {
        x[q] = nx[q];
        v[q] = nv[q];
        k0x[q] = K.kx[12][q];
        k0v[q] = K.kv[12][q];
      }
      if (rejected_last) {
        rejected_last = false;
        scale = fmin(scale, 1.0);
      }
      acc += 1;
      h = constrain_step_size(h * scale, a.h_min, a.h_max);
      if (sol >= 0) {
        finish(A, sol);
        return true;
      }
      if (fabs(tf - t) <= kTenEps) {
        finish(A, kComplete);
        return true;
      }
    } else {
      rejected_last = true;
      rej += 1;
      h = constrain_step_size(h * scale, a.h_min, a.h_max);
    }
    return false;
  }
};

// Waves per SIMD of a solver that keeps `vectors` state vectors: the largest
// whose register budget (512 / waves) holds them with about 70 registers of
// scalars and addresses.
constexpr int group_waves(int vectors, int c) {
  const int regs = 4 * vectors * c + 70;
  return regs <= 128 ? 4 : (regs <= 168 ? 3 : (regs <= 256 ? 2 : 1));
}

template <class Solver, int WAVES>
__global__ __launch_bounds__(kGroupBlock) __attribute__((amdgpu_waves_per_eu(WAVES))) void
spring_method_kernel(SpringArgs A) {
  spring_group_loop<Solver>(A);
}
#endif

}  // namespace de
