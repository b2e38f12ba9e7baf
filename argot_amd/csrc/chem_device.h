// Device-side primordial chemistry of one cell (gfx950): the HI/HII,
// HeI/HeII/HeIII and electron network with photoionization, integrated
// together with radiative heating and cooling, as the reference's GPU
// chemistry does it (src/step_reaction.cu:402-733, src/step_heatcool.cu:19-181,
// src/heatcool_rate.cu:10-74, src/cooling_rate.cu, src/reaction_rate.cu:33-212)
// for its flag set here: helium on, H2 off, __HEATCOOL__ and __CASE_B__ on.
//
// Every float/double promotion of the reference's expressions is written
// out, and the file is compiled without contraction or fast-math, so each
// rounding sits where the C source puts it.  The transcendental functions
// (exp, log, log10, pow) are the device library's double routines; they may
// differ from a host libm in the last bit, which is the only source of
// difference from a host restatement of the same code.
#pragma once
#include <hip/hip_runtime.h>
#include <float.h>
#include <stdint.h>

#include "argot_internal.h"

namespace argot {

namespace chem {

constexpr double kKtoEV = 8.61623e-5;    // K_to_eV, chemistry.h:10
constexpr double kXH = 0.755;            // XHYDROGEN, chemistry.h:23
constexpr double kYHe = 0.245;           // YHELIUM, chemistry.h:24
constexpr double kTiny = 1.0e-31;        // TINY, step_reaction.cu:11
constexpr double kDtFactor = 0.1;        // step_reaction.cu:400
constexpr double kSqrtFact = 1.0488088481;   // sqrt(1.1), step_heatcool.cu:14

// One cell's chemical state, struct prim_chem (13 floats).
struct State {
  float wmol, felec, fHI, fHII, fHeI, fHeII, fHeIII;
  float GammaHI, HeatHI, GammaHeI, GammaHeII, HeatHeI, HeatHeII;
};

// The reference's MIN/MAX macros (run_param.h:238-242), NaN behaviour included.
template <typename T>
__device__ __forceinline__ T min_of(T a, T b) { return a > b ? b : a; }
template <typename T>
__device__ __forceinline__ T max_of(T a, T b) { return a > b ? a : b; }

// 1/((1+x_e) X + Y/4), the WMOL macro of chemistry.h:69 (double).
__device__ __forceinline__ double mean_mass_inv(const State& c) {
  return 1.0 / ((1.0 + (double)c.felec) * kXH + 0.25 * kYHe);
}

// ---------------------------------------------------------------- rates ---

// The fits below are products of powers and exponentials of the temperature.
// Every power is formed as exp(p ln T + const) from one logarithm per
// temperature, and powers whose bases differ by a constant factor share an
// exponential.  What bounds the chemistry is the length of this arithmetic:
// a cell's sub-steps are a serial chain, and the cells next to a source need
// thousands of them.  pow() in double keeps a double-double logarithm, about
// 5 times the instructions of exp(); the fits' relative error grows from
// 1e-16 to a few 1e-15, far below the float the coefficients are rounded to.

// c0 + c1 L + c2 L^2 + ... with the powers of L formed by repeated
// multiplication and the terms added left to right (the collisional
// ionization fits of reaction_rate.cu; the signs live in the coefficients).
template <int N>
__device__ __forceinline__ double poly_left(const double (&c)[N], double L) {
  double s = c[0];
  double p = L;
  s = s + c[1] * p;
#pragma unroll
  for (int i = 2; i < N; i++) {
    p = p * L;
    s = s + c[i] * p;
  }
  return s;
}

// ln(lam T) for lam_HII = 2 * 157807 K / T and lam_HeIII = 2 * 631515 K / T
// of the case-B fits a lam^p / (1 + (lam/b)^q)^r (Hui & Gnedin 1997).
constexpr double kLnLamHII = 12.662275226919286;
constexpr double kLnLamHeIII = 14.049024154019651;

// The six rate coefficients at one temperature, each rounded to float as
// the reference stores them (float K_01 ... K_06).
struct KSet {
  float k1, k2, k3, k4, k5, k6;
};

// k01, k03, k05 (collisional ionization), reaction_rate.cu:33-62,108-136,
// 167-192; k02, k06 (case-B recombination, Hui & Gnedin 1997), :98-103,
// 200-203; k04, :152-164.
__device__ inline KSet rate_coefficients(float T) {
  constexpr double c1[9] = {-32.71396786375,      13.53655609057,     -5.739328757388,
                            1.563154982022,       -0.2877056004391,   0.03482559773736999,
                            -0.00263197617559,    0.0001119543953861, -2.039149852002e-6};
  constexpr double c3[9] = {-44.09864886561001, 23.91596563469,      -10.75323019821,
                            3.058038757198,     -0.5685118909884001, 0.06795391233790001,
                            -0.005009056101857001, 0.0002067236157507, -3.649161410833e-6};
  constexpr double c5[9] = {-68.71040990212001, 43.93347632635,      -18.48066993568,
                            4.701626486759002,  -0.7692466334492,    0.08113042097303,
                            -0.005324020628287001, 0.0001975705312221, -3.165581065665e-6};
  // ln(K_to_eV), ln(2.740)
  constexpr double kLnKtoEV = -9.359277830950614, kLnB = 1.007957920399979;
  const double t = (double)T;
  const double tev = t * kKtoEV;
  const double L = log(tev);
  KSet K;
  K.k1 = (float)exp(poly_left(c1, L));
  K.k3 = 0.0f;
  K.k5 = 0.0f;
  if (tev > 0.8) {
    K.k3 = (float)exp(poly_left(c3, L));
    K.k5 = (float)exp(poly_left(c5, L));
  }
  const double l2 = (kLnLamHII + kLnKtoEV) - L;     // ln lam_HII
  const double l6 = (kLnLamHeIII + kLnKtoEV) - L;   // ln lam_HeIII
  const double x2 = exp(0.407 * (l2 - kLnB));
  constexpr double kX6 = 1.7584044112379005;        // (631515/157807)^0.407
  const double x6 = x2 * kX6;
  K.k2 = (float)(2.753e-14 * exp(1.5 * l2 - 2.242 * log(1.0 + x2)));
  K.k6 = (float)(1.3765e-14 * exp(1.5 * l6 - 2.242 * log(1.0 + x6)));
  if (t > 500.3) {
    constexpr double kLnLamHeII = 13.254566388120152;
    K.k4 = (float)(1.26e-14 * exp(0.75 * ((kLnLamHeII + kLnKtoEV) - L)));
  } else {
    constexpr double kLog10e = 0.43429448190325182765;
    K.k4 = (float)((1.12e-10 - 2.1e-11 * ((L - kLnKtoEV) * kLog10e)) / sqrt(t));
  }
  return K;
}

// ------------------------------------------------------------- cooling ---

// What heat - cool of one cell depends on besides the temperature, formed
// once per energy update.
struct CoolTerms {
  double heat;                          // photoheating [erg cm^-3 s^-1]
  double hii, heii, heiii, hi, hei;     // ion densities times n_e
  double ions;                          // (n_HII + n_HeII + n_HeIII) n_e
  double ne;
  double compt, tcmb;                   // Compton: compt * (T - tcmb) * n_e
  double scale;                         // to code units: convfact / dens
};

__device__ __forceinline__ CoolTerms cool_terms(const State& c, float zred, double nH,
                                                double helium_fact, double scale) {
  CoolTerms k;
  const double nHe = nH * helium_fact;
  const double nHI = nH * (double)c.fHI, nHII = nH * (double)c.fHII;
  const double nHeI = nHe * (double)c.fHeI, nHeII = nHe * (double)c.fHeII;
  const double nHeIII = nHe * (double)c.fHeIII;
  k.ne = nH * (double)c.felec;
  k.heat = (double)c.HeatHI * nHI;
  k.heat += (double)c.HeatHeI * nHeI + (double)c.HeatHeII * nHeII;
  k.hi = nHI * k.ne;
  k.hii = nHII * k.ne;
  k.hei = nHeI * k.ne;
  k.heii = nHeII * k.ne;
  k.heiii = nHeIII * k.ne;
  k.ions = k.hii + (k.heii + k.heiii);
  const double z1 = 1.0 + (double)zred;
  k.compt = 5.406e-36 * (z1 * z1 * z1 * z1);
  k.tcmb = 2.73 * z1;
  k.scale = scale;
  return k;
}

// heat - cool of one cell in code units, calc_heatcool_rate_dev
// (heatcool_rate.cu:10-74) with cooling_rate.cu's case-B functions:
// recombination creh2 / crehe2 / crexihe2 / crehe3, collisional ionization
// cioh1 / ciohe1 / ciohe2 and excitation cexh1 / cexhe1 / cexhe2,
// bremsstrahlung with its Gaunt factor, Compton cooling off the CMB.
// cexhe1 carries another factor n_e, which the reference gives it
// ((cexhe1 n_e n_HeI + ...) n_e).  3 logarithms and 12 exponentials.
__device__ __forceinline__ double heatcool_rate(const CoolTerms& k, double T) {
  constexpr double kLnB = 0.8109302162163288;    // ln 2.25
  constexpr double kX3 = 1.6844137772424854;      // (631515/157807)^0.376
  constexpr double kLog10e = 0.43429448190325182765;
  const double L = log(T);
  const double it5 = 1.0e5 / T;                   // 1 / (T/1e5)
  const double sq = sqrt(T);
  const double sq5 = sq * 0.0031622776601683794;  // sqrt(T/1e5)
  const double l1 = kLnLamHII - L, l3 = kLnLamHeIII - L;
  const double x1 = exp(0.376 * (l1 - kLnB));
  const double x3 = x1 * kX3;
  const double a = 3.435e-30 * T;
  const double creh2 = a * exp(1.97 * l1 - 3.72 * log(1.0 + x1));
  const double crehe3 = a * exp(1.97 * l3 - 3.72 * log(1.0 + x3));
  // pow(T, 0.35) and pow(T/1e3, 0.15), either side of 980 K
  const bool cold = T < 980.0;
  const double crehe2 = (cold ? 1.7e-26 : 1.9e-25) *
                        exp(cold ? 0.35 * L : 0.15 * (L - 6.907755278982137));
  // exp(-4.7/t5) as the fifth power of exp(-0.94/t5)
  const double y = exp(-0.94 * it5);
  const double y2 = y * y;
  const double rsq = 1.0 / (T * sq * (1.0 + sq5));  // one division for T^-1.5 and 1/(1+sqrt(T5))
  const double t15 = rsq * (1.0 + sq5);
  const double r5 = rsq * (T * sq);
  const double crexihe2 = 1.24e-13 * t15 * (y2 * y2 * y) * (1.0 + 0.3 * y);
  const double cioh1 = exp(-1.578091 * it5), ciohe1 = exp(-2.853354 * it5);
  const double ciohe2 = exp(-6.31515 * it5), cexh1 = exp(-1.18348 * it5);
  const double cexhe1 = exp(-0.1687 * L - 0.13179 * it5);
  const double cexhe2 = exp(-0.397 * L - 4.73638 * it5);
  const double lg = 5.5 - L * kLog10e;
  const double gaunt = 1.1 + 0.34 * exp(-lg * lg * (1.0 / 3.0));
  const double brems = 1.42e-27 * gaunt * sq;
  const double col = (k.hi * (1.27e-21 * sq * cioh1 + 7.5e-19 * cexh1) +
                      k.hei * (9.38e-22 * sq * ciohe1 + 9.1e-27 * cexhe1 * k.ne) +
                      k.heii * (4.95e-22 * sq * ciohe2 + 5.54e-17 * cexhe2)) * r5;
  const double cool = creh2 * k.hii + crehe3 * k.heiii + (crehe2 + crexihe2) * k.heii + col +
                      brems * k.ions + k.compt * (T - k.tcmb) * k.ne;
  return (k.heat - cool) * k.scale;
}

// ------------------------------------------------------ heating/cooling ---

// Implicit energy update over dtime (code units): bracket the root of
// F(u) = u - u_old - dt Lambda((u_old + u)/2) and bisect it to 1e-5
// (advance_heatcool_dev, step_heatcool.cu:19-181).  Returns the bisection
// count.
//
// The result is the bisection's last midpoint, so the bisection itself is
// replayed; but a midpoint's sign needs no evaluation where it is known from
// the root's place.  Two secant steps from the bracket's own two evaluations
// place the root to 1e-9 of u (F is close to linear over the bracket's 10%),
// and a midpoint is evaluated only when it falls inside that margin: about 4
// evaluations of Lambda per update instead of 16.  The midpoints and their
// order are the bisection's, so the result is too, as long as F rises through
// the bracket.  Where that is not plain (a slope of the secants below 0.3 or
// changing by more than a factor 1.6, the recombination fits' break at 980 K
// inside the bracket, a value that is no number) every midpoint is evaluated.
// With the fits above, a 128^3 mesh over 100 kyr (8.0e6 sub-steps, the longest
// cell's chain setting the time) took 12.4 ms instead of 100 ms, with the same
// bits in every cell.
__device__ inline int advance_heatcool(float dens_cell, float* uene, const State& c,
                                       const ChemParams& p, float dtime) {
  const double dens = (double)(dens_cell * p.anow3i);
  const double uene_min = (double)p.uene_min, uene_max = (double)p.uene_max;

  const double uene_in = (double)*uene;
  double uene_old = uene_in;
  if (uene_old < uene_min) {
    uene_old = uene_min;
  } else if (uene_old > uene_max) {
    uene_old = uene_max;
  }
  const float wmol = (float)mean_mass_inv(c);
  const double nH = dens * p.denstonh;
  const CoolTerms k = cool_terms(c, p.znow, nH, p.helium_fact, p.convfact / dens);
  auto temp = [&](double u) { return u * p.uenetok * (double)wmol; };
  const double dt = (double)dtime;
  const double h0 = heatcool_rate(k, temp(uene_in));
  // Heating brackets upwards, cooling downwards; one loop for both, so that
  // the lanes of a wavefront evaluate together.
  const bool heating = h0 > 0.0;
  double uene_up = min_of(uene_old * kSqrtFact, uene_max);
  double uene_lo = max_of(uene_old / kSqrtFact, uene_min);
  double h1, end;
  for (;;) {
    end = heating ? uene_up : uene_lo;
    h1 = heatcool_rate(k, temp(end));
    const double f = end - uene_old - h1 * dt;
    if (!(heating ? f < 0.0 : f > 0.0)) break;
    uene_up = heating ? uene_up * 1.1 : uene_up / 1.1;
    uene_lo = heating ? uene_lo * 1.1 : uene_lo / 1.1;
    if (heating ? uene_up > uene_max : uene_lo < uene_min) break;
  }
  auto residual = [&](double u) {
    return u - uene_old - heatcool_rate(k, temp(0.5 * (uene_old + u))) * dt;
  };
  // F(u) <= 0 is known for u <= below, F(u) > 0 for u >= above
  double below = -DBL_MAX, above = DBL_MAX;
  {
    const double m = (h1 - h0) / (end - uene_in);
    double s = 1.0 - 0.5 * dt * m;
    const double r0 = uene_old + dt * (h0 + m * (uene_old - uene_in)) / s;
    const bool smooth = s > 0.3 && s < 1.0e6 && r0 > 0.5 * uene_lo && r0 < 2.0 * uene_up &&
                        !(temp(0.5 * (uene_old + uene_lo)) < 980.0 &&
                          temp(0.5 * (uene_old + uene_up)) >= 980.0);
    if (smooth) {
      double f = residual(r0), r = r0;
      for (int it = 0; it < 4; it++) {
        const double rn = r - f / s;
        const double fn = residual(rn);
        // (points closer than rounding lets F be told apart keep the slope)
        const double sn = fabs(rn - r) > 1.0e-11 * r0 ? (fn - f) / (rn - r) : s;
        if (!(sn > 0.6 * s && sn < 1.6 * s)) break;
        s = sn;
        r = rn;
        f = fn;
        const double step = f / s;
        const double tol = fabs(step) + 1.0e-12 * r;
        if (tol < 1.0e-9 * r) {
          below = r - step - tol;
          above = r - step + tol;
          break;
        }
      }
    }
  }
  int iter = 0;
  double uene_new;
  do {
    uene_new = 0.5 * (uene_up + uene_lo);
    bool positive = uene_new >= above;
    if (!positive && !(uene_new <= below)) {
      positive = residual(uene_new) > 0.0;
    }
    if (positive)
      uene_up = uene_new;
    else
      uene_lo = uene_new;
    iter++;
  } while ((uene_up - uene_lo) > 1.0e-5 * uene_new && iter < 32);
  *uene = (float)uene_new;
  return iter;
}

// ---------------------------------------------------------- network step ---

// Number densities of one cell [cm^-3], each rounded to float as the
// reference's float locals hold them.
struct Dens {
  float nH, nHe, nHI, nHII, nHeI, nHeII, nHeIII, ne;
};

__device__ __forceinline__ float expansion_inv3(float anow) {
  return 1.0f / (anow * anow * anow);
}

__device__ __forceinline__ Dens number_densities(float dens, const State& c, const ChemParams& p) {
  Dens n;
  n.nH = (float)((double)dens * p.denstonh * (double)expansion_inv3(p.anow));
  n.nHI = n.nH * c.fHI;
  n.nHII = n.nH * c.fHII;
  n.nHe = (float)((double)n.nH * p.helium_fact);
  n.nHeI = n.nHe * c.fHeI;
  n.nHeII = n.nHe * c.fHeII;
  n.nHeIII = n.nHe * c.fHeIII;
  n.ne = n.nH * c.felec;
  return n;
}

// Temperature of specific energy u (float, as the reference's float T).
__device__ __forceinline__ float temperature(float u, const State& c, const ChemParams& p) {
  return (float)((double)u * p.uenetok * mean_mass_inv(c));
}

// Safe time step [s] from the electron and HI source/sink balance,
// calc_dtime_dev (step_reaction.cu:18-196).  uene is the mesh's current
// specific energy; K holds the coefficients at its temperature.
__device__ inline float safe_dtime(const Dens& n, const State& c, const KSet& K) {
  const float GHI = c.GammaHI;
  const double GHeI = (double)c.GammaHeI, GHeII = (double)c.GammaHeII;
  double elec_p = (double)(K.k1 * n.nHI * n.ne + GHI * n.nHI);
  double elec_m = (double)(K.k2 * n.nHII * n.ne);
  elec_p += (double)(K.k3 * n.nHeI * n.ne + K.k5 * n.nHeII * n.ne) + GHeI * (double)n.nHeI +
            GHeII * (double)n.nHeII;
  elec_m += (double)(K.k4 * n.nHeII * n.ne + K.k6 * n.nHeIII * n.ne);
  const double hi_p = (double)(K.k2 * n.nHII * n.ne);
  const double hi_m = (double)(K.k1 * n.nHI * n.ne + GHI * n.nHI);
  const double eps = (double)1.e-20f;
  const double dt_elec = (double)n.ne / (fabs(elec_p - elec_m) + eps);
  const double dt_hi = (double)n.nHI / (fabs(hi_p - hi_m) + eps);
  double dt = 0.1 * dt_elec + 0.00001 * dt_hi;
  dt = max_of(dt, 1.0);   // shortest step: 1 s
  return (float)dt;
}

// Implicit (backward-Euler) update of one density: (s dt + n)/(1 + a dt)
// with float source s and sink a, double dt, rounded to float.
__device__ __forceinline__ float implicit_update(float n, float s, float a, double dt) {
  return (float)(((double)s * dt + (double)n) / (1.0 + (double)a * dt));
}


// The reaction network and the heating/cooling integrated together over
// dtime (code units), advance_reaction_and_heatcool_dev
// (step_reaction.cu:402-733), split into its set-up (cell_begin) and its
// sub-steps (cell_substep, while cell_more) so that a kernel can interleave
// cells.  c enters as prev_chem (with the cell's photoionization and
// heating rates) and leaves as the updated state; uene enters as prev_uene.
// mesh_uene is the mesh's current specific energy, which the reference reads
// for the first temperature and for every safe-step estimate.
struct CellRun {
  State c;
  float dens, mesh_uene, uene;
  float nH, nHe, nHI, nHII, nHeI, nHeII, nHeIII, ne;
  float GHI;
  double GHeI, GHeII;
  KSet K;
  double dtime_p, dtime_safe, elapsed;
  int nsub, niter;
};

__device__ inline void cell_begin(CellRun& r, const ChemParams& p, float dtime) {
  r.nsub = r.niter = 0;
  r.dtime_p = (double)dtime * p.tunit;
  const Dens n = number_densities(r.dens, r.c, p);
  r.nH = n.nH;
  r.nHe = n.nHe;
  r.nHI = n.nHI;
  r.nHII = n.nHII;
  r.nHeI = n.nHeI;
  r.nHeII = n.nHeII;
  r.nHeIII = n.nHeIII;
  r.ne = n.ne;
  r.GHI = r.c.GammaHI;
  r.GHeI = (double)r.c.GammaHeI;
  r.GHeII = (double)r.c.GammaHeII;
  r.K = rate_coefficients(temperature(r.mesh_uene, r.c, p));
  // calc_dtime reads the same cell state and temperature here: same K.
  r.dtime_safe = kDtFactor * (double)safe_dtime(n, r.c, r.K);
  if (r.dtime_p < r.dtime_safe) r.dtime_safe = r.dtime_p;
  r.elapsed = 0.0;
}

// The reference sub-steps until the elapsed time reaches dtime.  Two
// guards stop a cell earlier, where the reference would run for an
// unbounded time: a state that has turned NaN (e.g. an infinite rate in a
// cell that holds a source) makes every later safe step the 1-second floor,
// and a cell is given at most kMaxSubsteps sub-steps.  Both are counted
// (cell_stopped).
constexpr int kMaxSubsteps = 1000000;

__device__ __forceinline__ bool cell_nan(const CellRun& r) {
  return !(r.c.felec == r.c.felec) || !(r.uene == r.uene);
}

__device__ __forceinline__ bool cell_more(const CellRun& r) {
  return r.elapsed < r.dtime_p && r.nsub < kMaxSubsteps && !cell_nan(r);
}

// Did a guard, not the elapsed time, end this cell?
__device__ __forceinline__ bool cell_stopped(const CellRun& r) {
  return r.elapsed < r.dtime_p;
}

__device__ inline void cell_substep(CellRun& r, const ChemParams& p) {
  State& c = r.c;
  const KSet& K = r.K;
  if (r.elapsed + r.dtime_safe > r.dtime_p) r.dtime_safe = r.dtime_p - r.elapsed;
  r.elapsed += r.dtime_safe;
  r.nsub++;
  const double dts = r.dtime_safe;
  float nHI = r.nHI, nHII = r.nHII, nHeI = r.nHeI, nHeII = r.nHeII, nHeIII = r.nHeIII;
  float ne = r.ne;
  const float GHI = r.GHI;
  const double GHeI = r.GHeI, GHeII = r.GHeII;

  nHI = implicit_update(nHI, K.k2 * nHII * ne, K.k1 * ne + GHI, dts);
  nHII = implicit_update(nHII, K.k1 * nHI * ne + GHI * nHI, K.k2 * ne, dts);
  nHeI = implicit_update(nHeI, K.k4 * nHeII * ne, (float)((double)(K.k3 * ne) + GHeI), dts);
  nHeII = implicit_update(
      nHeII, (float)((double)((K.k3 * nHeI + K.k6 * nHeIII) * ne) + GHeI * (double)nHeI),
      (float)((double)((K.k4 + K.k5) * ne) + GHeII), dts);
  nHeIII = implicit_update(nHeIII, (float)((double)(K.k5 * nHeII * ne) + GHeII * (double)nHeII),
                           K.k6 * ne, dts);
  {
    float s = K.k1 * nHI * ne + GHI * nHI;
    float a = K.k2 * nHII;
    s = (float)((double)s + ((double)(K.k3 * nHeI * ne + K.k5 * nHeII * ne) +
                             GHeI * (double)nHeI + GHeII * (double)nHeII));
    a = a + (K.k4 * nHeII + K.k6 * nHeIII);
    ne = implicit_update(ne, s, a, dts);
  }

  // fractions, renormalised per element; electrons from the ions
  c.fHI = nHI / r.nH;
  c.fHII = nHII / r.nH;
  float cf = 1.0f / (c.fHI + c.fHII);
  c.fHI *= cf;
  c.fHII *= cf;
  const double nHe_t = (double)r.nHe + kTiny;
  c.fHeI = (float)((double)nHeI / nHe_t);
  c.fHeII = (float)((double)nHeII / nHe_t);
  c.fHeIII = (float)((double)nHeIII / nHe_t);
  cf = (float)(1.0 / ((double)(c.fHeI + c.fHeII + c.fHeIII) + kTiny));
  c.fHeI *= cf;
  c.fHeII *= cf;
  c.fHeIII *= cf;
  c.felec = c.fHII;
  c.felec = (float)((double)c.felec +
                    (p.helium_fact * ((double)c.fHeII + 2.0 * (double)c.fHeIII) + kTiny));

  r.dtime_safe = dts / p.tunit;
  r.niter += advance_heatcool(r.dens, &r.uene, c, p, (float)r.dtime_safe);

  // densities, temperature and coefficients for the next sub-step
  const Dens n = number_densities(r.dens, c, p);
  r.nHI = n.nHI;
  r.nHII = n.nHII;
  r.nHeI = n.nHeI;
  r.nHeII = n.nHeII;
  r.nHeIII = n.nHeIII;
  r.ne = n.ne;
  const float T = temperature(r.uene, c, p);
  r.K = rate_coefficients(T);
  // calc_dtime takes the temperature of the mesh's (unchanged) energy;
  // its coefficients equal K only when the two temperatures agree.
  const float Tm = temperature(r.mesh_uene, c, p);
  const KSet Km = Tm == T ? r.K : rate_coefficients(Tm);
  r.dtime_safe = kDtFactor * (double)safe_dtime(n, c, Km);
}

// Relative change of the HI photoionization rate and of the electron
// fraction between two states, diff_chem (chemistry.cu:271-287).
__device__ __forceinline__ float chem_change(const State& a, const State& b) {
  const float dH = (float)((double)fabsf(a.GammaHI - b.GammaHI) / ((double)a.GammaHI + 1.0e-30));
  const float de = (float)((double)fabsf(a.felec - b.felec) / ((double)a.felec + 1.0e-30));
  return max_of(dH, de);
}

// Relative change of the specific energy, diff_uene (chemistry.cu:289-295).
__device__ __forceinline__ float uene_change(float u1, float u2) {
  return (float)((double)fabsf(u1 - u2) / ((double)max_of(u1, u2) + 1.0e-30));
}

}  // namespace chem
}  // namespace argot
