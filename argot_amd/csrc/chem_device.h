// Device-side primordial chemistry of one cell (gfx950): the HI/HII,
// HeI/HeII/HeIII and electron network with photoionization, integrated
// together with radiative heating and cooling, as the reference's GPU
// chemistry does it (src/step_reaction.cu:402-733, src/step_heatcool.cu:19-181,
// src/heatcool_rate.cu:10-74, src/cooling_rate.cu, src/reaction_rate.cu:33-212)
// for its flag set here: helium on, H2 off, __HEATCOOL__ and __CASE_B__ on.
//
// Every float/double promotion of the reference's expressions is written
// out, and the file is compiled without contraction or fast-math, so each
// rounding sits where the C source puts it.  Two things differ from a host
// restatement of the same code, both far below the floats that the results are
// rounded to: the transcendental functions are the device library's double
// routines, which may differ from a host libm in the last bit, and the powers
// of the fits are formed from one logarithm (below), to a few 1e-15.
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

// A cell's arithmetic is done by one lane, or by the 16 lanes of a DPP row
// together: a cell beside a source takes thousands of sub-steps one after the
// other, and when only such cells are left, what counts is how long one
// sub-step takes.  The fits are then spread over the row, a fit or a term of
// the cooling sum per lane, and everything else is done by all 16 lanes alike.
// Both ways form each term with the same operations and add the terms in the
// same tree, so a cell's result does not depend on which it went through.

// Sum over the row, in every lane: ((t0 + t1) + (t2 + t3)) + ... as tree_sum.
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
  union { double d; int i[2]; } a, b;
  a.d = v;
  b.i[0] = __builtin_amdgcn_mov_dpp(a.i[0], CTRL, 0xf, 0xf, true);
  b.i[1] = __builtin_amdgcn_mov_dpp(a.i[1], CTRL, 0xf, 0xf, true);
  return v + b.d;
}
__device__ __forceinline__ double row_sum(double v) {
  v = dpp_add<0xb1>(v);    // quad_perm [1,0,3,2]
  v = dpp_add<0x4e>(v);    // quad_perm [2,3,0,1]
  v = dpp_add<0x141>(v);   // row_half_mirror: the other quad of the half row
  return dpp_add<0x140>(v);   // row_mirror: the other half
}
__device__ __forceinline__ double tree_sum(const double (&t)[16]) {
  const double a = ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
  const double b = ((t[8] + t[9]) + (t[10] + t[11])) + ((t[12] + t[13]) + (t[14] + t[15]));
  return a + b;
}
// Value of lane `from` of each row, in all its lanes.
template <int FROM>
__device__ __forceinline__ float row_pick(float v) {
  return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x10 | (FROM << 5)));
}

constexpr double kLnKtoEV = -9.359277830950614;   // ln(K_to_eV)
constexpr double kLnB274 = 1.0079579203999789;    // ln(2.740)
constexpr double kLnLamHeII = 13.254566388120152;
constexpr double kX6 = 1.7584044112379005;        // (631515/157807)^0.407
constexpr double kLog10e = 0.43429448190325182765;

// Fits of k01, k03, k05 (collisional ionization), reaction_rate.cu:33-62,
// 108-136, 167-192, by powers of ln(T in eV).
constexpr double kIon1[9] = {-32.71396786375,      13.53655609057,     -5.739328757388,
                             1.563154982022,       -0.2877056004391,   0.03482559773736999,
                             -0.00263197617559,    0.0001119543953861, -2.039149852002e-6};
constexpr double kIon3[9] = {-44.09864886561001, 23.91596563469,      -10.75323019821,
                             3.058038757198,     -0.5685118909884001, 0.06795391233790001,
                             -0.005009056101857001, 0.0002067236157507, -3.649161410833e-6};
constexpr double kIon5[9] = {-68.71040990212001, 43.93347632635,      -18.48066993568,
                             4.701626486759002,  -0.7692466334492,    0.08113042097303,
                             -0.005324020628287001, 0.0001975705312221, -3.165581065665e-6};

// k02, k06 (case-B recombination, Hui & Gnedin 1997), :98-103,200-203; k04,
// :152-164.
__device__ inline KSet rate_coefficients(float T) {
  const double t = (double)T;
  const double tev = t * kKtoEV;
  const double L = log(tev);
  KSet K;
  K.k1 = (float)exp(poly_left(kIon1, L));
  K.k3 = 0.0f;
  K.k5 = 0.0f;
  if (tev > 0.8) {
    K.k3 = (float)exp(poly_left(kIon3, L));
    K.k5 = (float)exp(poly_left(kIon5, L));
  }
  const double l2 = (kLnLamHII + kLnKtoEV) - L;     // ln lam_HII
  const double l6 = (kLnLamHeIII + kLnKtoEV) - L;   // ln lam_HeIII
  const double x2 = exp(0.407 * (l2 - kLnB274));
  const double x6 = x2 * kX6;
  K.k2 = (float)(2.753e-14 * exp(1.5 * l2 - 2.242 * log(1.0 + x2)));
  K.k6 = (float)(1.3765e-14 * exp(1.5 * l6 - 2.242 * log(1.0 + x6)));
  if (t > 500.3)
    K.k4 = (float)(1.26e-14 * exp(0.75 * ((kLnLamHeII + kLnKtoEV) - L)));
  else
    K.k4 = (float)((1.12e-10 - 2.1e-11 * ((L - kLnKtoEV) * kLog10e)) / sqrt(t));
  return K;
}

// ------------------------------------------------------------- cooling ---

// Terms of the cooling sum, each w * exp(p ln T + q 1e5/T + r z) with w the
// densities times a constant (times 1/(1 + sqrt(T/1e5)) for 5 to 10), and
// z = ln(1 + x) for the two Hui & Gnedin fits, (5.5 - log10 T)^2 for the Gaunt
// factor: calc_heatcool_rate_dev (heatcool_rate.cu:10-74) with
// cooling_rate.cu's case-B functions.
//   0 creh2, 1 crehe3, 2 crehe2 (two branches at 980 K), 3 and 4 crexihe2,
//   5 cioh1, 6 ciohe1, 7 ciohe2, 8 cexh1, 9 cexhe1, 10 cexhe2,
//   11 and 12 bremsstrahlung (constant part and Gaunt factor)
constexpr int kTerms = 13;
constexpr double kTermP[kTerms] = {-0.97, -0.97, 0.15, -1.5, -1.5, 0.5, 0.5,
                                   0.5,   0.0,   -0.1687, -0.397, 0.5, 0.5};
constexpr double kTermQ[kTerms] = {0.0,       0.0,      0.0,      -4.7,     -5.64, -1.578091, -2.853354,
                                   -6.31515, -1.18348, -0.13179, -4.73638, 0.0,   0.0};
constexpr double kColdP = 0.35;              // term 2 below 980 K
constexpr double kColdW = 1.7e-26;
// constants of w: creh2 and crehe3 hold lam^1.97 without its temperature
constexpr double kTermW[kTerms] = {
    3.435e-30 * 68129912473.377426, 3.435e-30 * 1046610102391.0461,
    1.9e-25 * 0.35481338923357547, 1.24e-13, 1.24e-13 * 0.3, 1.27e-21, 9.38e-22, 4.95e-22,
    7.5e-19, 9.1e-27, 5.54e-17, 1.42e-27 * 1.1, 1.42e-27 * 0.34};
constexpr double kRecR = -3.72, kGauntR = -1.0 / 3.0;
constexpr double kLnB225 = 0.8109302162163288;    // ln 2.25
constexpr double kX3 = 1.6844137772424854;        // (631515/157807)^0.376

// Constants of a lane of a row: its term of the cooling sum (lanes beyond have
// weight 0) and its fit among two sets of rate coefficients (lanes 0 to 5: k1,
// k2, k3, k4, k5, k6 at one temperature, 8 to 13 at another).
struct RowLane {
  int sub;
  double p, pc, q, r, x;     // cooling term (pc: below 980 K)
  double ion[9];             // collisional ionization fit
  double lam, xk, kw;        // Hui & Gnedin fit; constant factor
};

__device__ inline RowLane row_lane() {
  RowLane r;
  r.sub = threadIdx.x & 15;
  r.p = r.pc = r.q = r.r = r.x = 0.0;
#pragma unroll
  for (int i = 0; i < kTerms; i++)
    if (r.sub == i) {
      r.p = kTermP[i];
      r.pc = i == 2 ? kColdP : kTermP[i];
      r.q = kTermQ[i];
      r.r = i < 2 ? kRecR : i == 12 ? kGauntR : 0.0;
      r.x = i == 0 ? 1.0 : i == 1 ? kX3 : 0.0;
    }
  const int f = r.sub & 7;
#pragma unroll
  for (int i = 0; i < 9; i++) r.ion[i] = f == 0 ? kIon1[i] : f == 2 ? kIon3[i] : kIon5[i];
  r.lam = f == 1 ? kLnLamHII + kLnKtoEV : f == 5 ? kLnLamHeIII + kLnKtoEV : kLnLamHeII + kLnKtoEV;
  r.xk = f == 5 ? kX6 : 1.0;
  r.kw = f == 1 ? 2.753e-14 : f == 5 ? 1.3765e-14 : f == 3 ? 1.26e-14 : 1.0;
  return r;
}

// Rate coefficients at two temperatures, by the row.
__device__ inline void row_coefficients(const RowLane& r, float T0, float T1, KSet* K0, KSet* K1) {
  const int f = r.sub & 7;
  const double t = (double)(r.sub < 8 ? T0 : T1);
  const double tev = t * kKtoEV;
  const double L = log(tev);
  const double l2 = (kLnLamHII + kLnKtoEV) - L;
  const double l = r.lam - L;
  const double x2 = exp(0.407 * (l2 - kLnB274));
  const bool rec = f == 1 || f == 5;
  const double arg = rec ? 1.5 * l - 2.242 * log(1.0 + x2 * r.xk)
                         : f == 3 ? 0.75 * l : poly_left(r.ion, L);
  float v = (float)(r.kw * exp(arg));
  if ((f == 2 || f == 4) && !(tev > 0.8)) v = 0.0f;
  if (f == 3 && !(t > 500.3))
    v = (float)((1.12e-10 - 2.1e-11 * ((L - kLnKtoEV) * kLog10e)) / sqrt(t));
  *K0 = KSet{row_pick<0>(v), row_pick<1>(v), row_pick<2>(v),
             row_pick<3>(v), row_pick<4>(v), row_pick<5>(v)};
  *K1 = KSet{row_pick<8>(v), row_pick<9>(v), row_pick<10>(v),
             row_pick<11>(v), row_pick<12>(v), row_pick<13>(v)};
}

// What heat - cool of one cell depends on besides the temperature, formed
// once per energy update.  w: the terms' weights (a row's lane: its own), wc:
// term 2's below 980 K.
struct CoolCell {
  double heat;              // photoheating [erg cm^-3 s^-1]
  double compt, tcmb;       // Compton cooling: compt (T - tcmb)
  double scale;             // to code units: convfact / dens
};
struct CoolTerms : CoolCell {
  double w[kTerms], wc;
};
struct CoolRow : CoolCell {
  const RowLane& r;
  double w, wc;
};

__device__ __forceinline__ void cool_cell(const State& c, float zred, double nH,
                                          double helium_fact, double scale, CoolCell* k,
                                          double (&n)[6]) {
  const double nHe = nH * helium_fact;
  const double nHI = nH * (double)c.fHI, nHII = nH * (double)c.fHII;
  const double nHeI = nHe * (double)c.fHeI, nHeII = nHe * (double)c.fHeII;
  const double nHeIII = nHe * (double)c.fHeIII;
  const double ne = nH * (double)c.felec;
  k->heat = (double)c.HeatHI * nHI;
  k->heat += (double)c.HeatHeI * nHeI + (double)c.HeatHeII * nHeII;
  const double z1 = 1.0 + (double)zred;
  k->compt = 5.406e-36 * (z1 * z1 * z1 * z1) * ne;
  k->tcmb = 2.73 * z1;
  k->scale = scale;
  // densities times n_e: HI, HII, HeI, HeII, HeIII, and n_HeI n_e^2 (the
  // reference gives cexhe1 another n_e)
  n[0] = nHI * ne;
  n[1] = nHII * ne;
  n[2] = nHeI * ne;
  n[3] = nHeII * ne;
  n[4] = nHeIII * ne;
  n[5] = n[2] * ne;
}

__device__ __forceinline__ CoolTerms cool_terms(const State& c, float zred, double nH,
                                                double helium_fact, double scale) {
  CoolTerms k;
  double n[6];
  cool_cell(c, zred, nH, helium_fact, scale, &k, n);
  const double ions = n[1] + (n[3] + n[4]);
  const double d[kTerms] = {n[1], n[4], n[3], n[3], n[3], n[0], n[2],
                            n[3], n[0], n[5], n[3], ions, ions};
#pragma unroll
  for (int i = 0; i < kTerms; i++) k.w[i] = kTermW[i] * d[i];
  k.wc = kColdW * n[3];
  return k;
}

__device__ __forceinline__ CoolRow cool_terms(const State& c, float zred, double nH,
                                              double helium_fact, double scale,
                                              const RowLane& r) {
  CoolRow k{{}, r, 0.0, 0.0};
  double n[6];
  cool_cell(c, zred, nH, helium_fact, scale, &k, n);
  const double ions = n[1] + (n[3] + n[4]);
  const double d[kTerms] = {n[1], n[4], n[3], n[3], n[3], n[0], n[2],
                            n[3], n[0], n[5], n[3], ions, ions};
#pragma unroll
  for (int i = 0; i < kTerms; i++)
    if (r.sub == i) k.w = kTermW[i] * d[i];
  k.wc = r.sub == 2 ? kColdW * n[3] : k.w;
  return k;
}

// heat - cool of one cell in code units.
__device__ __forceinline__ double heatcool_rate(const CoolTerms& k, double T) {
  const double L = log(T);
  const double it5 = 1.0e5 / T;
  const double r5 = 1.0 / (1.0 + sqrt(T) * 3.1622776601683794e-3);   // 1/(1 + sqrt(T/1e5))
  const double x = exp(0.376 * ((kLnLamHII - L) - kLnB225));
  const double lg = 5.5 - L * kLog10e;
  const bool cold = T < 980.0;
  double t[16];
#pragma unroll
  for (int i = 0; i < kTerms; i++) {
    double arg = (i == 2 && cold ? kColdP : kTermP[i]) * L;
    if (kTermQ[i] != 0.0) arg = arg + kTermQ[i] * it5;
    if (i < 2) arg = arg + kRecR * log(1.0 + (i == 0 ? x : x * kX3));
    if (i == 12) arg = arg + kGauntR * (lg * lg);
    t[i] = (i == 2 && cold ? k.wc : k.w[i]) * exp(arg);
    if (i >= 5 && i <= 10) t[i] = t[i] * r5;
  }
  for (int i = kTerms; i < 16; i++) t[i] = 0.0;
  const double cool = tree_sum(t) + k.compt * (T - k.tcmb);
  return (k.heat - cool) * k.scale;
}

__device__ __forceinline__ double heatcool_rate(const CoolRow& k, double T) {
  const RowLane& r = k.r;
  const double L = log(T);
  const double it5 = 1.0e5 / T;
  const double r5 = 1.0 / (1.0 + sqrt(T) * 3.1622776601683794e-3);
  const double x = exp(0.376 * ((kLnLamHII - L) - kLnB225));
  const double lg = 5.5 - L * kLog10e;
  const bool cold = T < 980.0;
  // (a lane without a factor multiplies by 0 or 1: exact)
  const double z = r.sub == 12 ? lg * lg : log(1.0 + x * r.x);
  const double arg = ((cold ? r.pc : r.p) * L + r.q * it5) + r.r * z;
  double t = (cold ? k.wc : k.w) * exp(arg);
  t = t * (r.sub >= 5 && r.sub <= 10 ? r5 : 1.0);
  const double cool = row_sum(t) + k.compt * (T - k.tcmb);
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
//
// row: the lane's constants when a row does the cell, nothing otherwise.
template <typename... Row>
__device__ inline int advance_heatcool(float dens_cell, float* uene, const State& c,
                                       const ChemParams& p, float dtime, const Row&... row) {
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
  const auto k = cool_terms(c, p.znow, nH, p.helium_fact, p.convfact / dens, row...);
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

// A cell between two sub-steps: what differs from its prev_chem record and the
// mesh, and its progress.
struct CellPaused {
  double dtime_safe, elapsed;
  int cell, nsub, niter;
  float uene;
  float felec, fHI, fHII, fHeI, fHeII, fHeIII;
};

__device__ __forceinline__ CellPaused cell_pause(const CellRun& r, int cell) {
  const State& c = r.c;
  return {r.dtime_safe, r.elapsed, cell,   r.nsub,  r.niter,  r.uene,
          c.felec,      c.fHI,     c.fHII, c.fHeI, c.fHeII, c.fHeIII};
}

// r holds the cell's dens, mesh_uene and prev_chem; continues from s (after
// at least one sub-step: the densities and coefficients follow from the state).
__device__ inline void cell_resume(CellRun& r, const CellPaused& s, const ChemParams& p,
                                   float dtime) {
  r.nsub = s.nsub;
  r.niter = s.niter;
  r.uene = s.uene;
  r.c.felec = s.felec;
  r.c.fHI = s.fHI;
  r.c.fHII = s.fHII;
  r.c.fHeI = s.fHeI;
  r.c.fHeII = s.fHeII;
  r.c.fHeIII = s.fHeIII;
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
  r.K = rate_coefficients(temperature(r.uene, r.c, p));
  r.dtime_safe = s.dtime_safe;
  r.elapsed = s.elapsed;
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

template <typename... Row>
__device__ inline void cell_substep(CellRun& r, const ChemParams& p, const Row&... row) {
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
  r.niter += advance_heatcool(r.dens, &r.uene, c, p, (float)r.dtime_safe, row...);

  // densities, temperature and coefficients for the next sub-step
  const Dens n = number_densities(r.dens, c, p);
  r.nHI = n.nHI;
  r.nHII = n.nHII;
  r.nHeI = n.nHeI;
  r.nHeII = n.nHeII;
  r.nHeIII = n.nHeIII;
  r.ne = n.ne;
  const float T = temperature(r.uene, c, p);
  // calc_dtime takes the temperature of the mesh's (unchanged) energy;
  // its coefficients equal K only when the two temperatures agree.
  const float Tm = temperature(r.mesh_uene, c, p);
  KSet Km;
  if constexpr (sizeof...(Row) == 0) {
    r.K = rate_coefficients(T);
    Km = Tm == T ? r.K : rate_coefficients(Tm);
  } else {
    row_coefficients(row..., T, Tm, &r.K, &Km);
  }
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
