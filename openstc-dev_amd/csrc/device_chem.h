// Per-point finite-rate chemistry, mixture transport and the point-implicit
// solve, FP64, templated on the species count so every per-lane array has a
// compile-time size and stays in registers.
#pragma once

#include "device_common.h"

namespace ostc {

__host__ __device__ constexpr double kPatmD() { return 101325.0; }

// A T^b exp(-Ea / T) as A exp(b ln T - Ea / T): one exponential per rate,
// with ln T and 1 / T (lt, it) computed once per cell
__device__ inline double d_arrhenius(double lt, double it, double A, double b, double Ea) {
  return A * exp(b * lt - Ea * it);
}

// x^n for the small integer exponents of stoichiometric coefficients and
// reaction orders, as products (x^0 = 1, x^1 = x and x^2 = x*x exactly as a
// correctly rounded pow gives them; x^3 and negative orders within one or
// two roundings); any other exponent goes to pow.  The exponent is uniform
// across a wavefront (it belongs to the reaction), so the switch is a
// scalar branch.
__device__ inline double d_ipow(double x, int n) {
  switch (n) {
    case 0: return 1.0;
    case 1: return x;
    case 2: return x * x;
    case 3: return x * x * x;
    case -1: return 1.0 / x;
    case -2: return 1.0 / (x * x);
    default: return pow(x, (double)n);
  }
}

// FiniteRateChem.cu:65-149 for reaction r: kf (Arrhenius + duplicate, third
// body, Lindemann, Troe) and kb = kf / Kc (or the REV set, 0 if irreversible).
template <int NS>
__device__ inline void d_rate(MechK m, int r, double t, double lt, double it, const double *c,
                              const double *g, double temp_t, double &kf, double &kb) {
  const auto &R = m->reac[r];
  const int type = R.type;
  double k = d_arrhenius(lt, it, R.A, R.b, R.Ea);
  if (type == 3) k += d_arrhenius(lt, it, R.A2, R.b2, R.Ea2);
  if (type > 3) {
    double cc = 0;
#pragma unroll
    for (int l = 0; l < NS; ++l) cc += c[l] * m->third_body_coeff[r * NS + l];
    if (type == 4) {
      k *= cc;
    } else {
      const double klow = d_arrhenius(lt, it, R.A2, R.b2, R.Ea2);
      const double khigh = k;
      const double pr = klow * cc / khigh;
      double F = 1.0;
      if (type > 5) {
        double fc = (1 - R.alpha) * exp(-t * R.t3_inv) + R.alpha * exp(-t * R.t1_inv);
        if (type == 7) fc += exp(-R.t2 / t);
        const double lfc = log10(fc);
        const double c2 = -0.4 - 0.67 * lfc;
        const double nn = 0.75 - 1.27 * lfc;
        const double lpr = log10(pr);
        const double tempo = (lpr + c2) / (nn - 0.14 * (lpr + c2));
        const double pp = lfc / (1.0 + tempo * tempo);
        F = exp(2.302585092994046 * pp);  // 10^pp
      }
      k = khigh * pr / (1.0 + pr) * F;
    }
  }
  kf = k;
  if (type == 0) {
    kb = 0;
  } else if (type == 2) {
    kb = d_arrhenius(lt, it, R.A2, R.b2, R.Ea2);
  } else {
    double dg = 0;
#pragma unroll
    for (int l = 0; l < NS; ++l) dg += g[l] * (m->stoi_b[r * NS + l] - m->stoi_f[r * NS + l]);
    const double kc = d_ipow(temp_t, R.order) * exp(-dg);
    kb = k / kc;
  }
}

// Source and Jacobian of the chemistry batch in two passes over the
// reactions: the first computes omega and parks the rates of
// progress q1, q2 of reaction r at q[2r * stride], q[(2r + 1) * stride]
// (LDS, one column per thread), the second accumulates the Jacobian from
// them.  Keeping the 81 Jacobian sums out of the first pass (where the
// concentrations, free energies and creation / destruction sums are live)
// keeps the kernel in registers.
template <int NS>
__device__ inline void d_chem_rates(MechK m, double rho, double t, const double *Y, double *omega,
                                    double *q, int stride) {
  double c[NS], g[NS];
#pragma unroll
  for (int l = 0; l < NS; ++l) c[l] = d_div(rho * Y[l], m->mw[l], m->mw_inv[l]) * 1e-3;
  const double temp_t = (kPatmD() / kRuD * 1e-3) / t;
  const double lt = log(t), it = 1.0 / t;
#pragma unroll
  for (int l = 0; l < NS; ++l) {
    if (l % 3 == 0) m = fresh(m);
    g[l] = d_species_gibbs(m, l, t, lt, it);
  }
  const int nr = m->n_reac;
  double creation[NS], destr[NS];
#pragma unroll
  for (int l = 0; l < NS; ++l) {
    creation[l] = 0;
    destr[l] = 0;
  }
  for (int r = 0; r < nr; ++r) {
    double kf, kb;
    d_rate<NS>(m, r, t, lt, it, c, g, temp_t, kf, kb);
    double q1 = 1.0, q2 = 1.0;
#pragma unroll
    for (int l = 0; l < NS; ++l) {
      q1 *= d_ipow(c[l], m->stoi_f[r * NS + l]);
      q2 *= d_ipow(c[l], m->stoi_b[r * NS + l]);
    }
    q1 *= kf;
    q2 = m->reac[r].type != 0 ? q2 * kb : 0.0;
    q[2 * r * stride] = q1;
    q[(2 * r + 1) * stride] = q2;
#pragma unroll
    for (int l = 0; l < NS; ++l) {
      const int nf = m->stoi_f[r * NS + l], nb = m->stoi_b[r * NS + l];
      creation[l] += q2 * nf + q1 * nb;
      destr[l] += q1 * nf + q2 * nb;
    }
  }
#pragma unroll
  for (int l = 0; l < NS; ++l) omega[l] = creation[l] * (m->mw[l] * 1e+3) - destr[l] * (m->mw[l] * 1e+3);
}

// A = I - dt J with the EPI Jacobian J from the parked rates of progress
template <int NS>
__device__ inline void d_epi_matrix(MechK m, double rho, const double *Y, double dt,
                                    const double *q, int stride, double *A) {
#pragma unroll
  for (int a = 0; a < NS * NS; ++a) A[a] = 0;
  const int nr = m->n_reac;
  for (int r = 0; r < nr; ++r) {
    const double q1 = q[2 * r * stride], q2 = q[(2 * r + 1) * stride];
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      const double dn = m->stoi_f[r * NS + n] * q1 - m->stoi_b[r * NS + n] * q2;
#pragma unroll
      for (int a = 0; a < NS; ++a) A[a * NS + n] += (m->stoi_b[r * NS + a] - m->stoi_f[r * NS + a]) * dn;
    }
  }
#pragma unroll
  for (int n = 0; n < NS; ++n) {
    const bool on = Y[n] > 1e-25;
#pragma unroll
    for (int a = 0; a < NS; ++a) {
      const double J = on ? m->mw[a] * (A[a * NS + n] / (rho * Y[n])) * 1e+3 : 0.0;
      A[a * NS + n] = (a == n ? 1.0 : 0.0) - dt * J;
    }
  }
}

// FiniteRateChem.cu:7-149 (+ 151-217 and 219-232): one pass over the
// reactions giving omega [kg/m3/s] and, per WANT, nothing else (kOmega), the
// sums S_an = sum_r (nu_b - nu_f)_a (nu_f q1 - nu_b q2)_n of the
// exact-point-implicit Jacobian (kJacobian, row-major NA x NA, see
// d_jacobian_entry), or the destruction rates (kDestruction).  q1, q2 are the
// rates of progress: kf (Arrhenius + duplicate, third body, Lindemann, Troe)
// and kb = kf / Kc (or the REV set, 0 if irreversible) times the
// concentrations.
//
// NA: leading species that take part in reactions (NS, or NS - 1 when the
// last one is inert: its row and column of the Jacobian are zero).
// col: this thread's column (stride ld) of kinetics_slots(NS, WANT) pairs of
// shared memory: concentration and g / RT of every species, (1, 0) for a
// missing molecule, and with kJacobian and kDestruction the creation and
// destruction sums.  A reaction addresses its species there by wave-uniform
// index; only its owner reads a column, so there is no barrier.
//
// What bounds it: one wavefront is a long serial chain (about 40 exponentials),
// so the time goes with its instructions and with how many wavefronts share a
// SIMD.  Multiplying all NS powers of every reaction through scalar switches,
// with integer coefficients converted in the loop, took 13,100 vector and
// 6,200 scalar instructions per wavefront (9 species, 19 reactions, with the
// solve) at one wavefront per SIMD and 40 % of the cycles in waits.  Indexed
// species, coefficients read as double scalar operands and sums kept out of
// registers leave 2 wavefronts per SIMD with the Jacobian, 4 without.
enum Kinetics { kOmega, kJacobian, kDestruction };

__host__ __device__ constexpr int kinetics_slots(int ns, int want) { return want == kOmega ? ns + 1 : 2 * ns + 2; }

template <int NS, int NA, int WANT>
__device__ inline void d_kinetics(MechK m, double rho, double t, const double *Y, double2 *col, int ld, double *omega,
                                  double *out) {
  const double lt = log(t), it = 1.0 / t;
  double2 *sum = col + (NS + 1) * ld;  // (creation, destruction) of every species, one unused
#pragma unroll
  for (int l = 0; l < NS; ++l) {
    m = fresh(m);
    const double c = d_div(rho * Y[l], m->mw[l], m->mw_inv[l]) * 1e-3;
    col[l * ld] = double2{c, d_species_gibbs(m, l, t, lt, it)};
    if constexpr (WANT != kOmega) sum[l * ld] = double2{0.0, 0.0};
  }
  col[NS * ld] = double2{1.0, 0.0};
  const double p0 = (kPatmD() / kRuD * 1e-3) / t;  // concentration at p_atm and T
  if constexpr (WANT == kOmega) {
#pragma unroll
    for (int a = 0; a < NA; ++a) omega[a] = 0;
  }
  if constexpr (WANT == kJacobian) {
#pragma unroll
    for (int a = 0; a < NA * NA; ++a) out[a] = 0;
  }
  const int nr = m->n_reac;
  for (int r = 0; r < nr; ++r) {
    const auto &R = m->reac[r];
    double q1 = col[R.f0 * ld].x * col[R.f1 * ld].x, q2 = col[R.b0 * ld].x * col[R.b1 * ld].x;
    double dg = col[R.g[0] * ld].y * R.gc[0];
#pragma unroll
    for (int i = 1; i < 4; ++i) dg = fma(col[R.g[i] * ld].y, R.gc[i], dg);
    const bool more = R.more != 0;
    if (more) {
      q1 = q2 = 1.0;
      dg = 0;
#pragma unroll 1
      for (int l = 0; l < NS; ++l) {
        const int nf = m->stoi_f[r * NS + l], nb = m->stoi_b[r * NS + l];
        const double2 x = col[l * ld];
        q1 *= d_ipow(x.x, nf);
        q2 *= d_ipow(x.x, nb);
        dg += x.y * (nb - nf);
      }
    }
    const int type = R.type;
    double k = d_arrhenius(lt, it, R.A, R.b, R.Ea);
    if (type == 3) k += d_arrhenius(lt, it, R.A2, R.b2, R.Ea2);
    if (type > 3) {
      double cc = 0;
#pragma unroll
      for (int l = 0; l < NS; ++l) cc = fma(col[l * ld].x, m->third_body_coeff[r * NS + l], cc);
      if (type == 4) {
        k *= cc;
      } else {
        const double pr = d_arrhenius(lt, it, R.A2, R.b2, R.Ea2) * cc / k;
        double F = 1.0;
        if (type > 5) {
          double fc = (1 - R.alpha) * exp(-t * R.t3_inv) + R.alpha * exp(-t * R.t1_inv);
          if (type == 7) fc += exp(-R.t2 * it);
          const double lfc = log10(fc);
          const double lpr = log10(pr) + (-0.4 - 0.67 * lfc);
          const double tempo = lpr / ((0.75 - 1.27 * lfc) - 0.14 * lpr);
          F = exp(2.302585092994046 * (lfc / (1.0 + tempo * tempo)));
        }
        k = k * pr / (1.0 + pr) * F;
      }
    }
    q1 *= k;
    if (type == 0) {
      q2 = 0;
    } else if (type == 2) {
      q2 *= d_arrhenius(lt, it, R.A2, R.b2, R.Ea2);
    } else {
      const int order = R.order;
      double kc = exp(-dg);
      if (order == 1)
        kc *= p0;
      else if (order != 0)
        kc *= d_ipow(p0, order);
      q2 *= k / kc;
    }
    if constexpr (WANT == kOmega) {
      const double net = q1 - q2;
#pragma unroll
      for (int a = 0; a < NA; ++a) omega[a] = fma((double)m->nu[r * NS + a], net, omega[a]);
    } else if (more) {
#pragma unroll 1
      for (int l = 0; l < NS; ++l) {
        const double nf = m->nu_f[r * NS + l], nb = m->nu_b[r * NS + l];
        double2 s = sum[l * ld];
        s.x += q2 * nf + q1 * nb;
        s.y += q1 * nf + q2 * nb;
        sum[l * ld] = s;
      }
    } else {
      // a species of the net list stands on one side: forward (gc < 0) or backward
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        double2 *s = sum + R.g[i] * ld;
        const double c = R.gc[i], qc = c < 0 ? q2 : q1, qd = c < 0 ? q1 : q2;
        double2 v = *s;
        v.x = fma(fabs(c), qc, v.x);
        v.y = fma(fabs(c), qd, v.y);
        *s = v;
      }
    }
    if constexpr (WANT == kJacobian) {
      MechK mn = m;
#pragma unroll
      for (int n = 0; n < NA; ++n) {
        if (n % 4 == 0) mn = fresh(mn);
        const double dn = mn->nu_f[r * NS + n] * q1 - mn->nu_b[r * NS + n] * q2;
#pragma unroll
        for (int a = 0; a < NA; ++a) out[a * NA + n] = fma((double)m->nu[r * NS + a], dn, out[a * NA + n]);
      }
    }
  }
#pragma unroll
  for (int a = 0; a < NA; ++a) {
    if constexpr (WANT == kOmega) {
      omega[a] *= m->mw[a] * 1e+3;
    } else {
      const double2 s = sum[a * ld];
      omega[a] = (s.x - s.y) * (m->mw[a] * 1e+3);
      if constexpr (WANT == kDestruction) out[a] = s.y * (m->mw[a] * 1e+3);
    }
  }
}

// d omega_a / d(rho Y_n) from the sum S_an: W_a 1e3 S_an / (rho Y_n), 0 where
// species n is absent.  ry, iry: rho Y_n and its reciprocal.
__device__ inline double d_jacobian_entry(double s, bool on, double ry, double iry, double mw) {
  return on ? mw * d_div(s, ry, iry) * 1e+3 : 0.0;
}

// FiniteRateChem.cu:364-418 solve_chem_system: Crout-style LU with row
// pivoting (first maximum wins), then substitution; rhs overwritten.
template <int N>
__device__ inline void d_lu_solve(double *A, double *b) {
  int piv[N];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    // the running maximum is kept in a register (comparing against
    // A[ik][n] would index A dynamically and push it to scratch memory)
    int ik = n;
    double best = 0;
#pragma unroll
    for (int r = n; r < N; ++r) {
#pragma unroll
      for (int t = 0; t < n; ++t) A[r * N + n] -= A[r * N + t] * A[t * N + n];
      const double v = fabs(A[r * N + n]);
      if (r == n) {
        best = v;
      } else if (v > best) {
        best = v;
        ik = r;
      }
    }
    piv[n] = ik;
    // row swap n <-> ik as selects on static indices (a branch around the
    // swap keeps A out of registers)
#pragma unroll
    for (int r = n + 1; r < N; ++r) {
      const bool sw = r == ik;
#pragma unroll
      for (int t = 0; t < N; ++t) {
        const double x = A[r * N + t], y = A[n * N + t];
        A[r * N + t] = sw ? y : x;
        A[n * N + t] = sw ? x : y;
      }
    }
#pragma unroll
    for (int p = n + 1; p < N; ++p)
#pragma unroll
      for (int t = 0; t < n; ++t) A[n * N + p] -= A[n * N + t] * A[t * N + p];
#pragma unroll
    for (int r = n + 1; r < N; ++r) A[r * N + n] /= A[n * N + n];
  }
#pragma unroll
  for (int r = 0; r < N; ++r) {
#pragma unroll
    for (int q = r + 1; q < N; ++q) {
      const bool sw = q == piv[r];
      const double x = b[q], y = b[r];
      b[q] = sw ? y : x;
      b[r] = sw ? x : y;
    }
  }
#pragma unroll
  for (int r = 1; r < N; ++r)
#pragma unroll
    for (int t = 0; t < r; ++t) b[r] -= A[r * N + t] * b[t];
  b[N - 1] /= A[N * N - 1];
#pragma unroll
  for (int r = N - 2; r >= 0; --r) {
#pragma unroll
    for (int t = r + 1; t < N; ++t) b[r] -= A[r * N + t] * b[t];
    b[r] /= A[r * N + r];
  }
}

// Transport.cu:6-38 species viscosities of Chapman-Enskog form,
// vis = vis_coeff sqrt(T) / (1.147 T*^-0.145 + (T* + 0.5)^-2), T* = T / (eps/kb),
// with T*^-0.145 = exp(-0.145 (log T + log(kb/eps))); also sqrt(vis) and
// 1 / sqrt(vis), so that Wilke's sqrt(vis_a / vis_b) is a product
template <int NS>
__device__ inline void species_viscosities(MechK m, double t, double *vis, double *sv,
                                           double *isv) {
  const double st = sqrt(t), lt = log(t);
#pragma unroll
  for (int l = 0; l < NS; ++l) {
    const double x5 = t * m->LJ_potent_inv[l] + 0.5;
    const double ci = 1.147 * exp(-0.145 * (lt + m->log_LJ_potent_inv[l])) + rcp(x5 * x5);
    vis[l] = m->vis_coeff[l] * st * rcp(ci);
    sv[l] = sqrt(vis[l]);
    isv[l] = rcp(sv[l]);
  }
}

// Transport.cu:113-140 compute_viscosity: Wilke's rule alone, at the mean
// molecular weight mw_total of composition Y
template <int NS>
__device__ inline double d_viscosity(MechK m, double t, double mw_total, const double *Y) {
  double X[NS], vis[NS], sv[NS], isv[NS];
  species_viscosities<NS>(m, t, vis, sv, isv);
#pragma unroll
  for (int l = 0; l < NS; ++l) X[l] = Y[l] * mw_total * m->mw_inv[l];
  double mu = 0;
#pragma unroll
  for (int a = 0; a < NS; ++a) {
    double vt = 0;
#pragma unroll
    for (int b = 0; b < NS; ++b) {
      double pf = 1.0;
      if (a != b) {
        const double num = 1 + sv[a] * isv[b] * m->WjDivWi_to_One4th[a * NS + b];
        pf = num * num * m->sqrt_WiDivWjPl1Mul8[a * NS + b];
      }
      vt += pf * X[b];
    }
    mu += vis[a] * X[a] / vt;
  }
  return mu;
}

// Transport.cu:40-110 compute_transport_property.  The 36 pairs' collision
// integrals and diffusivities, the 9 species' viscosities and Wilke's sums
// would be 136 divisions; they are reciprocals within an ulp (rcp) and one
// division (k_properties<9>: 512x256 cells 38 -> 32 us, 1.18 M cells 191 -> 166).
template <int NS>
__device__ inline void d_transport(MechK m, double t, double p, double rho, const double *Y,
                                   const double *cp, double &mu, double &lam, double *rhoD) {
  double mwi = 0;
#pragma unroll
  for (int l = 0; l < NS; ++l) mwi += Y[l] * m->mw_inv[l];
  const double mw_total = 1 / mwi;
  double X[NS], vis[NS], sv[NS], isv[NS];
  const double st = sqrt(t);
  species_viscosities<NS>(m, t, vis, sv, isv);
#pragma unroll
  for (int l = 0; l < NS; ++l) X[l] = Y[l] * mw_total * m->mw_inv[l];
  double viscosity = 0, conductivity = 0;
#pragma unroll
  for (int a = 0; a < NS; ++a) {
    double vt = 0;
#pragma unroll
    for (int b = 0; b < NS; ++b) {
      double pf = 1.0;
      if (a != b) {
        const double num = 1 + sv[a] * isv[b] * m->WjDivWi_to_One4th[a * NS + b];
        pf = num * num * m->sqrt_WiDivWjPl1Mul8[a * NS + b];
      }
      vt += pf * X[b];
    }
    const double ct = 1.065 * vt - 0.065 * X[a];
    viscosity += vis[a] * X[a] * rcp(vt);
    const double la = vis[a] * (cp[a] + 1.25 * kRuD * m->mw_inv[a]);
    conductivity += la * X[a] * rcp(ct);
  }
  mu = viscosity;
  lam = conductivity;
  const double it32p = p / (t * st), lt = log(t);
  // reciprocal binary diffusivities 1 / D_ab of the NS (NS - 1) / 2 pairs,
  // each once: T*^-0.145 = exp(-0.145 (log T + log k_ab))
  double idij[NS * (NS - 1) / 2 > 0 ? NS * (NS - 1) / 2 : 1];
#pragma unroll
  for (int a = 0; a < NS; ++a)
#pragma unroll
    for (int b = a + 1; b < NS; ++b) {
      const double tr = t * m->kb_over_eps_jk[a * NS + b];
      const double od = exp(-0.145 * (lt + m->log_kb_over_eps_jk[a * NS + b])) + rcp((tr + 0.5) * (tr + 0.5));
      idij[a * NS - a * (a + 1) / 2 + (b - a - 1)] = od * (m->inv_binary_diffusivity[a * NS + b] * it32p);
    }
#pragma unroll
  for (int l = 0; l < NS; ++l) {
    double num = 0, den = 0;
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      if (l != n) {
        const int a = l < n ? l : n, b = l < n ? n : l;
        num += (X[n] + 1e-12) * m->mw[n];
        den += (X[n] + 1e-12) * idij[a * NS - a * (a + 1) / 2 + (b - a - 1)];
      }
    }
    rhoD[l] = rho * num * mwi * rcp(den);
  }
}

}  // namespace ostc
