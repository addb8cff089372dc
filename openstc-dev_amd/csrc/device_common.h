// Device-side data views and per-point physics shared by the gfx950
// kernels.  All state is FP64 in HBM (reference DZone layout); the flux
// arithmetic is templated on its working precision.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ostc {

constexpr int kMS = 20;   // species capacity of the device tables
constexpr int kMR = 50;   // reaction capacity of the device tables

// DParameter.cuh:13-92 content, fixed capacity, row-major packed with the
// live n_spec / n_reac.  Lives in device memory; kernels read it with
// wave-uniform addresses.
struct DMech {
  // One reaction as the kinetics loop reads it: rate constants (1 / T3 and
  // 1 / T1 of Troe's form), the species of the first two molecules of each
  // side (n_spec: no such molecule), and the net coefficients nu_b - nu_f of
  // the species that have one, ascending (g[i] with coefficient gc[i]).
  // more: a side has further molecules or a species stands on both sides;
  // stoi_f and stoi_b are walked instead.
  struct Reac {
    double A, b, Ea, A2, b2, Ea2, alpha, t3_inv, t1_inv, t2, gc[4];
    int type, order, more, f0, f1, b0, b1, g[4], pad;
  };
  int n_spec, n_reac;
  double mw[kMS], mw_inv[kMS], t_low[kMS], t_mid[kMS], hi[kMS * 7], lo[kMS * 7];
  // below t_low: cp / R stays cp(t_low) and h / R = h_ext + cp_ext T
  double cp_ext[kMS], h_ext[kMS];
  double g_ext[kMS];  // g / RT there, its value at t_low
  // the different t_low and t_mid of all species, ascending: between two of
  // them every species keeps its branch
  int n_brk;
  double brk[2 * kMS];
  double LJ_potent_inv[kMS], vis_coeff[kMS];
  double WjDivWi_to_One4th[kMS * kMS], sqrt_WiDivWjPl1Mul8[kMS * kMS];
  double inv_binary_diffusivity[kMS * kMS], kb_over_eps_jk[kMS * kMS];  // 1 / D_ab at T = p = 1 and T* = T k_ab
  Reac reac[kMR];
  int stoi_f[kMR * kMS], stoi_b[kMR * kMS];
  // per reaction (rows of n_spec): forward and backward coefficients,
  // nu_b - nu_f, third-body efficiencies
  double nu_f[kMR * kMS], nu_b[kMR * kMS], nu[kMR * kMS], third_body_coeff[kMR * kMS];
  // logarithms of LJ_potent_inv and kb_over_eps_jk: the collision-integral
  // powers T*^-0.145 become exp(-0.145 (log T + log k))
  double log_LJ_potent_inv[kMS], log_kb_over_eps_jk[kMS * kMS];
  // R_u / W_l, rounded as the quotient itself (so h_l, cp_l equal the
  // divided forms bit for bit)
  double r_mw[kMS];
};

// Scheme switches and constants (the scalar part of DParameter).
struct DParams {
  int mx, my, mz, g, dim;
  int nv, ns, nsc, nt;  // n_var, species, scalars (species + turbulence), turbulence scalars (0 or 2)
  int mix, reaction, chemSrcMethod;
  int inviscid_scheme, reconstruction, limiter, viscous, inviscid_type, gradP;
  double cfl, Pr, Sc, Prt, Sct;
  double efix;  // Roe entropy-fix factor
  int turb_implicit, compress;  // SST: implicit source diagonal; compressibility correction 0-3
  int nr;                       // reactions of the mechanism (0 without chemistry)
  int last_inert;               // the last species takes part in no reaction
  int jface;                    // HLLC / LF face vector (J0 m0 + J1 m1) / 2 (conservative metrics)
};

// (a, b, c) of linear index t over an a-fastest na x nb x nc box, in 32-bit
// unsigned arithmetic: block point counts stay below 2^32 (checked when the
// blocks are built), and 64-bit division is a long instruction sequence
__device__ inline void unflatten3(int64_t t, int na, int nb, int &a, int &b, int &c) {
  const uint32_t u = (uint32_t)t, ua = (uint32_t)na, ub = (uint32_t)nb;
  const uint32_t r = u / ua;
  a = (int)(u - r * ua);
  c = (int)(r / ub);
  b = (int)(r - (uint32_t)c * ub);
}

// Raw device pointers of one block (DZone, Field.h:13-71).  bv/sv/cv/qn and
// the property arrays use the ngg-ghosted layout; dq/dt_local/bv_last use
// the ghost-free layout.  metric is 9 component-major arrays
// (index (r*3+c)*sz + p  =  d xi_r / d x_c).
struct ZoneView {
  int mx, my, mz, g;
  int64_t d2, d1, sz;      // ghosted
  int64_t e2, e1, sz0;     // ghost-free
  double *bv, *sv, *cv, *qn;
  double *vel, *acoustic, *mach, *mul, *cond, *rhoD, *gam, *cp;
  const double *jac, *metric;
  double *dq, *dt_local, *bv_last, *chem_jac;
  double *inv_sr;          // steady path: inviscid spectral radii, 3 x ghost-free (null otherwise)
  double *dq0, *dqk;       // DPLUR work arrays, n_var x ghost-free (null otherwise)
  double *dplur_h;         // DPLUR, mixtures: species enthalpies and mixture total enthalpy of each
                           // interior point, (n_spec + 1) x ghost-free (null otherwise)
  double *mut, *tcond;     // SST: turbulent viscosity and conductivity (ghosted; null when laminar)
  double *wdist;           // SST: wall distance (ghosted)
  double *turb_jac;        // SST: source Jacobian diagonal of k and omega, 2 x ghost-free

  __host__ __device__ int64_t at(int i, int j, int k) const {
    return (int64_t)(k + g) * d1 + (int64_t)(j + g) * d2 + (i + g);
  }
  __host__ __device__ int64_t at0(int i, int j, int k) const { return (int64_t)k * e1 + (int64_t)j * e2 + i; }
};

constexpr double kRuD = 8314.462618;
constexpr double kGam = 1.4;
constexpr double kMwAirD = 28.9647;

// ---------------------------------------------------------------- thermo
// Thermo.cu:5-79.  Below t_low: h extrapolated with cp(t_low), cp and g/RT
// frozen at t_low.
//
// The tables are read through a pointer into the constant address space, so
// every load is a scalar one (uniform address, never aliased by the kernel's
// stores), and each species takes its temperature branch by selecting the
// value, not the coefficients: a coefficient pointer chosen per lane made
// each evaluation 6 or 7 vector loads per species behind divergent branches,
// some 700 of the 980 vector loads of a 9-species AWENO face.  With the
// branch-free forms, the mixture polynomial below and products with 1 / W_l
// in place of quotients: 512x256 mixing layer 2.69 -> 1.71 ms per RK3 step,
// 192x96x64 channel 12.5 -> 8.6 ms per pseudo-iteration; the laminar 9-species
// AWENO sweeps no longer use scratch memory (with SST they use 76 to 148 B per
// lane).
typedef const __attribute__((address_space(4))) DMech *MechK;
__device__ inline MechK mech_k(const DMech *m) { return (MechK)m; }

// Any table read at wave-uniform addresses that no kernel writes, the same way
template <typename T>
__device__ inline const __attribute__((address_space(4))) T *uniform_table(const T *p) {
  return (const __attribute__((address_space(4))) T *)p;
}

// The mechanism pointer made opaque to the optimiser: a property evaluation
// given fresh(m) loads its coefficients where it uses them (scalar-cache
// hits) instead of sharing loads hoisted once and held in registers for the
// rest of the kernel (the flux sweeps evaluate the properties at many
// temperatures per face).
__device__ inline MechK fresh(MechK m) {
  asm volatile("" : "+s"(m));
  return m;
}

// a / b for a finite a and a normal quotient, with rb = 1 / b correctly
// rounded: the residual of a * rb is exact in a fused multiply-add, and adding
// its share back rounds to the quotient itself (Markstein 1990), so the result
// is the one a division gives, in 3 operations instead of 11.
__device__ inline double d_div(double a, double b, double rb) {
  const double q = a * rb;
  return fma(fma(-b, q, a), rb, q);
}

// c ? a : b with both sides evaluated: left to itself the compiler turns a
// choice between two polynomials into divergent branches that load their
// coefficients inside, one scalar-load latency each
__device__ inline double d_select(bool c, double a, double b) {
  asm("" : "+v"(a), "+v"(b));
  return c ? a : b;
}

// 1 / x for finite, normal x: the hardware estimate refined by two
// Newton-Raphson steps r <- r + r (1 - x r), each squaring the relative
// error, so the result is within an ulp of 1 / x, in 5 operations where a
// division takes 11.  A quotient a * rcp(b) then differs from a / b by rounding
// only; shared denominators are inverted once.
__device__ inline double rcp(double x) {
  double r = __builtin_amdgcn_rcp(x);
  double e = fma(-x, r, 1.0);
  r = fma(r, e, r);
  e = fma(-x, r, 1.0);
  return fma(r, e, r);
}
__device__ inline float rcp(float x) { return __builtin_amdgcn_rcpf(x); }

// T and the weights of a0 .. a4 in h / R = a0 T + a1 T^2 / 2 + .. + a4 T^5 / 5 + a5
struct TPow {
  double t, t2, t3, t4, p2, p3, p4, p5;
  __device__ explicit TPow(double T) : t(T) {
    t2 = t * t;
    t3 = t2 * t;
    t4 = t3 * t;
    p2 = 0.5 * t2;
    p3 = t3 * (1.0 / 3);
    p4 = 0.25 * t4;
    p5 = 0.2 * (t4 * t);
  }
};

// h_l of species l at T
__device__ inline double d_species_h(MechK m, int l, const TPow &q) {
  const auto *a = &m->lo[l * 7];
  const auto *b = &m->hi[l * 7];
  const double hl = fma(a[4], q.p5, fma(a[3], q.p4, fma(a[2], q.p3, fma(a[1], q.p2, fma(a[0], q.t, a[5])))));
  const double hh = fma(b[4], q.p5, fma(b[3], q.p4, fma(b[2], q.p3, fma(b[1], q.p2, fma(b[0], q.t, b[5])))));
  const double he = fma(m->cp_ext[l], q.t, m->h_ext[l]);
  const double h = q.t < m->t_mid[l] ? hl : hh;
  return (q.t < m->t_low[l] ? he : h) * m->r_mw[l];
}

// cp_l of species l at T
__device__ inline double d_species_cp(MechK m, int l, const TPow &q) {
  const auto *a = &m->lo[l * 7];
  const auto *b = &m->hi[l * 7];
  const double cl = fma(a[4], q.t4, fma(a[3], q.t3, fma(a[2], q.t2, fma(a[1], q.t, a[0]))));
  const double ch = fma(b[4], q.t4, fma(b[3], q.t3, fma(b[2], q.t2, fma(b[1], q.t, b[0]))));
  const double c = q.t < m->t_mid[l] ? cl : ch;
  return (q.t < m->t_low[l] ? (double)m->cp_ext[l] : c) * m->r_mw[l];
}

template <int NS>
__device__ inline void d_enthalpy(double t, MechK m, double *h) {
  const TPow q(t);
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    if (i % 4 == 0) m = fresh(m);
    h[i] = d_species_h(m, i, q);
  }
}

template <int NS>
__device__ inline void d_enthalpy_cp(double t, MechK m, double *h, double *cp) {
  const TPow q(t);
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    if (i % 3 == 0) m = fresh(m);
    h[i] = d_species_h(m, i, q);
    cp[i] = d_species_cp(m, i, q);
  }
}

template <int NS>
__device__ inline void d_cp(double t, MechK m, double *cp) {
  const TPow q(t);
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    if (i % 4 == 0) m = fresh(m);
    cp[i] = d_species_cp(m, i, q);
  }
}

// g_l / RT of species l at T (lt = ln T, it = 1 / T), frozen at t_low below it
__device__ inline double d_species_gibbs(MechK m, int l, double t, double lt, double it) {
  const double t2 = t * t, t3 = t2 * t, t4 = t3 * t;
  auto poly = [&](double c0, double c1, double c2, double c3, double c4, double c5, double c6) {
    return c0 * (1.0 - lt) - 0.5 * c1 * t - d_div(c2 * t2, 6.0, 1 / 6.0) - d_div(c3 * t3, 12.0, 1 / 12.0) -
           c4 * t4 * 0.05 + c5 * it - c6;
  };
  const auto *a = &m->lo[l * 7];
  const auto *b = &m->hi[l * 7];
  const double gl = poly(a[0], a[1], a[2], a[3], a[4], a[5], a[6]);
  const double gh = poly(b[0], b[1], b[2], b[3], b[4], b[5], b[6]);
  return d_select(t < m->t_low[l], m->g_ext[l], d_select(t < m->t_mid[l], gl, gh));
}

// sum_l w_l h_l(T) and sum_l w_l cp_l(T) as one polynomial in T, its
// coefficients the weighted sums of the species': each species adds its own
// branch at T, so the polynomial is exact on [ta, tb), the interval between
// two branch points around T.  One construction costs about one evaluation
// of all species; a Newton iteration then costs ten multiply-adds instead of
// twenty per species.
struct MixPoly {
  double a0, a1, a2, a3, a4, a5, ta, tb;

  // fresh: the coefficients are loaded for two species at a time.  It orders
  // the loads among themselves and not the arithmetic behind them, so in the
  // sweeps most of a species' set still waits in vector-register lanes (1,036
  // spilled scalar registers in the 9-species AWENO j-sweep)
  template <int NS>
  __device__ inline void build(MechK m, const double *w, double t) {
    a0 = a1 = a2 = a3 = a4 = a5 = 0;
#pragma unroll
    for (int l = 0; l < NS; ++l) {
      if (l % 2 == 0) m = fresh(m);
      const double x = w[l] * m->r_mw[l];
      const bool cold = t < m->t_low[l], low = t < m->t_mid[l];
      const double xl = low && !cold ? x : 0.0, xh = low || cold ? 0.0 : x, xe = cold ? x : 0.0;
      const auto *a = &m->lo[l * 7];
      const auto *b = &m->hi[l * 7];
      a0 = fma(xl, a[0], fma(xh, b[0], fma(xe, m->cp_ext[l], a0)));
      a1 = fma(xl, a[1], fma(xh, b[1], a1));
      a2 = fma(xl, a[2], fma(xh, b[2], a2));
      a3 = fma(xl, a[3], fma(xh, b[3], a3));
      a4 = fma(xl, a[4], fma(xh, b[4], a4));
      a5 = fma(xl, a[5], fma(xh, b[5], fma(xe, m->h_ext[l], a5)));
    }
    ta = -1e300;
    tb = 1e300;
    const int nb = m->n_brk;
    for (int i = 0; i < nb; ++i) {
      const double b = m->brk[i];
      const bool above = t >= b;
      ta = above ? b : ta;
      tb = !above && b < tb ? b : tb;
    }
  }
  __device__ inline bool holds(double t) const { return t >= ta && t < tb; }
  __device__ inline double cp(double t) const { return fma(t, fma(t, fma(t, fma(t, a4, a3), a2), a1), a0); }
  __device__ inline double h(double t) const {
    return fma(t, fma(t, fma(t, fma(t, fma(t, 0.2 * a4, 0.25 * a3), (1.0 / 3) * a2), 0.5 * a1), a0), a5);
  }
};

// Transport.cu:6-9
// (T / 273)^1.5 as x sqrt(x): the same power within an ulp, without the
// log / exp of a general pow
__device__ inline double d_sutherland(double t) {
  const double x = t / 273;
  return 1.716e-5 * (x * sqrt(x)) * (273 + 111) / (t + 111);
}

// FieldOperation.cu:3-39: Newton on e(T) from the warm start; tolerance
// |1 - T1/T| <= 1e-3, at most 1000 iterations.
template <int NS>
__device__ inline double d_temperature(MechK m, double rho, double rhoE, double u, double v, double w, const double *Y,
                                       double t, double &p) {
  double mwi = 0;
#pragma unroll
  for (int l = 0; l < NS; ++l) mwi += Y[l] * m->mw_inv[l];
  const double gas = kRuD * mwi;
  const double e = rhoE / rho - 0.5 * (u * u + v * v + w * w);
  MixPoly q;
  q.ta = q.tb = 0;  // built in the loop
  double err = 1;
  int iter = 0;
  while (err > 1e-3 && iter++ < 1000) {
    if (!q.holds(t)) q.build<NS>(m, Y, t);
    const double et = q.h(t) - gas * t;
    const double cv = q.cp(t) - gas;
    const double t1 = t - (et - e) / cv;
    err = fabs(1 - t1 / t);
    t = t1;
  }
  p = rho * t * gas;
  return t;
}

// TimeAdvanceFunc.cuh:50-100: the CFL time step of the cell at point p
// (interior index q): the inviscid spectral radii of the three directions
// plus the viscous radius.  The inviscid radii are kept per direction when
// the zone stores them (z.inv_sr, for DPLUR).  a, gamma, mul: sound speed,
// specific-heat ratio and viscosity of the point.  One definition for the
// stand-alone pass and for the kernels that compute it on the way.
__device__ inline double cell_dt(const ZoneView &z, const DParams &P, int64_t p, int64_t q, double a, double gamma,
                                 double mul) {
  double mm[9];
#pragma unroll
  for (int c = 0; c < 9; ++c) mm[c] = z.metric[c * z.sz + p];
  const double gxi = sqrt(mm[0] * mm[0] + mm[1] * mm[1] + mm[2] * mm[2]);
  const double geta = sqrt(mm[3] * mm[3] + mm[4] * mm[4] + mm[5] * mm[5]);
  const double gzeta = sqrt(mm[6] * mm[6] + mm[7] * mm[7] + mm[8] * mm[8]);
  const double u = z.bv[z.sz + p], v = z.bv[2 * z.sz + p], w = z.bv[3 * z.sz + p];
  const double U = u * mm[0] + v * mm[1] + w * mm[2];
  const double V = u * mm[3] + v * mm[4] + w * mm[5];
  const double W = u * mm[6] + v * mm[7] + w * mm[8];
  const double r0 = fabs(U) + a * gxi, r1 = fabs(V) + a * geta;
  const double r2 = P.dim == 3 ? fabs(W) + a * gzeta : 0.0;
  const double sri = r0 + r1 + r2;
  if (z.inv_sr) {
    z.inv_sr[q] = r0;
    z.inv_sr[z.sz0 + q] = r1;
    z.inv_sr[2 * z.sz0 + q] = r2;
  }
  const double c1 = fmax(gamma, 4.0 / 3.0) / z.bv[p];
  double c2 = mul / P.Pr;
  if (z.mut) c2 += z.mut[p] / P.Prt;
  double srv = gxi * gxi + geta * geta;
  if (P.dim == 3) srv += gzeta * gzeta;
  srv *= c1 * c2;
  return P.cfl / (sri + srv);
}

// the same with the stored properties of the point
template <int MIX>
__device__ inline double cell_dt(const ZoneView &z, const DParams &P, int64_t p, int64_t q) {
  return cell_dt(z, P, p, q, z.acoustic[p], MIX ? z.gam[p] : kGam, z.mul[p]);
}

}  // namespace ostc
