// Quadrature form of the frequency integral.
//
// A ray's rates are sums over the 256 bins of spectrum times cross-section
// times f(k), where f, the attenuated and cell-averaged exponential of the
// optical depths, is smooth between the species' edges.  Within each of the
// three bin ranges f is determined to FP32 rounding by its values at a few
// nodes (the Gauss nodes of the discrete polynomials over the range's bins),
// and the sum over bins becomes a sum over nodes with the weights
//   W_j = sum_k S_k sigma_s(k) L_j(k),   L_j the Lagrange polynomials of the nodes,
// formed once per spectrum.  The rule is exact for every f that is a
// polynomial of lower degree than the number of nodes, whatever the
// spectrum, and close to twice that degree for a smooth one.  44 nodes take
// the place of 256 bins: the bin loop was half of the step's arithmetic.
//
// How thick a ray the rule serves is found out for every spectrum and each of
// the three ranges by itself: a range's error against the sum over its own bins
// is evaluated in full on test columns (mixes of the species that absorb in it,
// at rising scales), and its limit is the largest scale up to which every rate
// of every column stays within kRuleTol.  A ray takes the nodes in the ranges
// within whose limits it lies and the bins in the others.  All terms are
// positive, so no rate's relative error exceeds the worst range's, however much
// the other species take away.  (The total over the ranges says little about
// the first: where HI is thick, most of what is left lies in the other two, but
// not for a ray whose helium absorbs those.  Judged by the total, a 5e4 K
// blackbody with one bin 30% up had a limit of 136 at the HI edge; rays of 71
// whose helium is thick too had errors of 1e-4 within it.  It is 16 now.  A ray
// that is thick in HI alone is told by its sums: kRuleShare.)
// Between the test columns the error was at most 2e-7, on 36000 spectra drawn
// with lines, steps, noise, waves, cut-offs and second temperatures.
// A 1e5 K blackbody passes to optical depth 104 at the HI edge, 75 at the HeI
// edge and 21 at the HeII edge, a 3e4 K one to 104, 32 and 8.
// Measured with the bin loops as the other side: the step on 256^3 cells and 4096
// sources 147 -> 111 ms, on 72 x 58 x 87 cells and 250 sources 13.0 -> 6.5 ms;
// errors against 64-bit rates 0.7e-7 to 1e-7 by nodes and 2.3e-7 by bins (64^3,
// uniform); 10, 12 and 16 nodes serve only half as thick rays at that error, and
// nodes of the continuous Legendre polynomials a fifth.
#include "rate_rule.h"

#include <math.h>
#include <string.h>

#include <algorithm>

namespace argot {
namespace {

// Polynomials orthonormal over the n points t_i = (2i + 1 - n)/n with weight
// 1/n, by their three-term recurrence.
struct Gram {
  int n, m;                       // points, degrees 0 .. m - 1 (and the m-th up to scale)
  std::vector<double> t, b;       // points; recurrence coefficients (the points are symmetric)
  std::vector<double> p;          // [m][n] values at the points
  Gram(int n_, int m_) : n(n_), m(m_), t(n_), b(m_ + 1, 0.0), p((size_t)m_ * n_) {
    for (int i = 0; i < n; i++) t[i] = (2.0 * i + 1.0 - n) / n;
    std::vector<double> q(n);
    for (int i = 0; i < n; i++) p[i] = 1.0;
    for (int d = 0; d < m; d++) {
      const double* p1 = &p[(size_t)d * n];
      double s = 0.0;
      for (int i = 0; i < n; i++) {
        q[i] = t[i] * p1[i] - (d > 0 ? b[d] * p1[i - n] : 0.0);
        s += q[i] * q[i] / n;
      }
      b[d + 1] = sqrt(s);
      if (d + 1 < m)
        for (int i = 0; i < n; i++) p[(size_t)(d + 1) * n + i] = q[i] / b[d + 1];
    }
  }
  // values of degrees 0 .. m - 1 at x into v; returns the m-th (unscaled)
  double at(double x, double* v) const {
    double p0 = 0.0, p1 = 1.0;
    for (int d = 0; d < m; d++) {
      if (v) v[d] = p1;
      const double q = x * p1 - b[d] * p0;
      p0 = p1;
      p1 = d + 1 < m ? q / b[d + 1] : q;
    }
    return p1;
  }
  // the m roots of the m-th polynomial: sign changes on a fine grid, bisected
  std::vector<double> roots() const {
    std::vector<double> r;
    const int grid = 1024;   // the closest roots are 0.01 apart
    double x0 = -1.0, f0 = at(x0, nullptr);
    for (int g = 1; g <= grid; g++) {
      const double x1 = -1.0 + 2.0 * g / grid, f1 = at(x1, nullptr);
      if (f0 == 0.0) {
        r.push_back(x0);
      } else if ((f0 < 0.0) != (f1 < 0.0) && f1 != 0.0) {
        double a = x0, c = x1;
        for (int it = 0; it < 60; it++) {
          const double mid = 0.5 * (a + c);
          if ((at(mid, nullptr) < 0.0) == (f0 < 0.0)) a = mid; else c = mid;
        }
        r.push_back(0.5 * (a + c));
      }
      x0 = x1;
      f0 = f1;
    }
    return r;
  }
};

// Mixes of the species on which the ranges are tried, by optical depth at the
// range's first bin.
constexpr double kMix[3][6][3] = {
    {{1.0, 0.0, 0.0}},
    {{1.0, 0.0, 0.0}, {0.0, 1.0, 0.0}, {1.0, 1.0, 0.0}, {1.0, 0.25, 0.0}},
    {{1.0, 0.0, 0.0}, {0.0, 1.0, 0.0}, {0.0, 0.0, 1.0}, {1.0, 1.0, 1.0}, {1.0, 0.3, 0.1},
     {0.1, 1.0, 0.3}}};

}  // namespace

void build_rate_rule(const float* sig, const float* hsig, int ngrid, int k1, int k2, RateRule* r) {
  const int nn[3] = {kRuleN1, kRuleN2, kRuleN3};
  const int first[4] = {0, k1, k2, ngrid};
  const int fit[3] = {11, 11, 13};   // terms of the fits to ln sigma
  r->usable = false;
  for (int g = 0; g < 4; g++) r->start[g] = first[g];
  r->node.assign(3 * kRuleNodes, 0.0);
  r->sig.assign(3 * kRuleNodes, 0.0f);
  r->dsig.assign(3 * kRuleNodes, 0.0f);
  r->lag.assign((size_t)ngrid * kRuleN3, 0.0);
  r->rate.assign((size_t)6 * ngrid, 0.0f);
  r->test.clear();
  memset(r->edge, 0, sizeof r->edge);
  memset(r->end, 0, sizeof r->end);
  for (int g = 0; g < 3; g++)
    if (first[g + 1] - first[g] < nn[g]) return;
  // a species of range g has a positive cross-section in every bin of it
  for (int s = 0; s < 3; s++)
    for (int k = first[s]; k < ngrid; k++)
      if (!(sig[s * ngrid + k] > 0.0f) || !(sig[s * ngrid + k] < 1.0e-10f)) return;

  std::vector<double>& nodes = r->node;
  std::vector<double>& lag = r->lag;
  for (int g = 0, o = 0; g < 3; o += nn[g], g++) {
    const int a = first[g], n = first[g + 1] - a, m = nn[g];
    const Gram gram(n, m);
    const std::vector<double> y = gram.roots();
    if ((int)y.size() != m) return;
    std::vector<double> v(m);
    for (int j = 0; j < m; j++) {
      // Gauss nodes: L_j(x) = w_j sum_d p_d(x) p_d(y_j), 1/w_j = sum_d p_d(y_j)^2
      gram.at(y[j], v.data());
      double sum = 0.0;
      for (int d = 0; d < m; d++) sum += v[d] * v[d];
      for (int i = 0; i < n; i++) {
        double l = 0.0;
        for (int d = 0; d < m; d++) l += gram.p[(size_t)d * n + i] * v[d];
        lag[(size_t)(a + i) * kRuleN3 + j] = l / sum;
      }
    }
    // The cross-sections at the nodes, from least-squares fits to ln sigma
    // (the tables hold floats: a fit averages their rounding out).
    const Gram smooth(n, std::min(fit[g], n));
    std::vector<double> u(smooth.m);
    for (int s = 0; s <= g; s++) {
      std::vector<double> c(smooth.m, 0.0);
      for (int d = 0; d < smooth.m; d++)
        for (int i = 0; i < n; i++)
          c[d] += log((double)sig[s * ngrid + a + i]) * smooth.p[(size_t)d * n + i] / n;
      for (int j = 0; j < m; j++) {
        smooth.at(y[j], u.data());
        double l = 0.0;
        for (int d = 0; d < smooth.m; d++) l += c[d] * u[d];
        nodes[s * kRuleNodes + o + j] = exp(l);
      }
    }
  }
  // (A node's differences are those to the last bin of its own range: the sums
  // come from there, and the optical depths that FP32 rounds are small there.)
  for (int s = 0; s < 3; s++)
    for (int g = 0, o = 0; g < 3; o += nn[g], g++)
      for (int j = o; j < o + nn[g]; j++) {
        const double v = nodes[s * kRuleNodes + j];
        r->sig[s * kRuleNodes + j] = (float)v;
        r->dsig[s * kRuleNodes + j] =
            s <= g ? (float)(v - (double)sig[s * ngrid + first[g + 1] - 1]) : 0.0f;
      }
  r->end[0] = sig[k1 - 1];
  r->end[1] = sig[k2 - 1];
  r->end[2] = sig[ngrid + k2 - 1];
  for (int s = 0; s < 3; s++)
    for (int k = 0; k < ngrid; k++) {
      r->rate[(size_t)(2 * s) * ngrid + k] = sig[s * ngrid + k] * (float)kRuleScale;
      r->rate[(size_t)(2 * s + 1) * ngrid + k] = hsig[s * ngrid + k] * (float)kRuleScale;
    }
  for (int g = 0; g < 3; g++)
    for (int s = 0; s < 3; s++)
      r->edge[g][s] = (float)((double)sig[s * ngrid + first[g]] / kRuleEdge[g]);
  // Test columns.  f is taken at zero cell depth: a cell of depth d averages it
  // over columns t to t + d, so its relative error is at most the largest there.
  for (int g = 0, o = 0; g < 3; o += nn[g], g++) {
    const int a = first[g], n = first[g + 1] - a, ncol = rule_columns(g);
    const size_t at = r->test.size();
    r->test.resize(at + (size_t)n * ncol * 2, 0.0f);
    for (int c = 0; c < ncol; c++) {
      const int level = c / kRuleMixes[g];   // 0: the reversed ones
      const double* mix = kMix[g][c % kRuleMixes[g]];
      const double scale = (level > 0 ? (double)kRuleLevel[g][level - 1] : -(double)kRuleNegative) *
                           kRuleEdge[g] / (mix[0] + mix[1] + mix[2]);
      double col[3] = {0.0, 0.0, 0.0};
      for (int s = 0; s <= g; s++) col[s] = scale * mix[s] / (double)sig[s * ngrid + a];
      double shift = 0.0;   // the smallest optical depth: f is at most 1
      for (int i = 0; i < n; i++) {
        double tau = 0.0;
        for (int s = 0; s <= g; s++) tau += col[s] * (double)sig[s * ngrid + a + i];
        if (i == 0 || tau < shift) shift = tau;
      }
      double fn[kRuleN3];
      for (int j = 0; j < nn[g]; j++) {
        double tau = 0.0;
        for (int s = 0; s <= g; s++) tau += col[s] * nodes[s * kRuleNodes + o + j];
        fn[j] = exp(shift - tau);
      }
      for (int i = 0; i < n; i++) {
        double tau = 0.0, q = 0.0;
        for (int s = 0; s <= g; s++) tau += col[s] * (double)sig[s * ngrid + a + i];
        const double f = exp(shift - tau);
        for (int j = 0; j < nn[g]; j++) q += lag[(size_t)(a + i) * kRuleN3 + j] * fn[j];
        float* t = &r->test[at + ((size_t)i * ncol + c) * 2];
        t[0] = (float)f;
        t[1] = (float)(q - f);
      }
    }
  }
  r->usable = true;
}

void project_spectra_host(const RateRule& r, const float* spec, int nspec, int ngrid,
                          float* weight, float* limit) {
  // (an unusable rule has no bins to project and fails every spectrum)
  const int nn[3] = {kRuleN1, kRuleN2, kRuleN3};
  for (int u = 0; u < nspec; u++) {
    const float* sp = spec + (size_t)u * ngrid;
    float* w = weight + (size_t)u * kRuleWeights;
    const float* m = r.test.data();
    for (int g = 0; g < 3; g++) {
      const int a = r.start[g], n = r.usable ? r.start[g + 1] - a : 0, ncol = rule_columns(g);
      for (int i = 0; i < 2 * (g + 1); i++)
        for (int j = 0; j < nn[g]; j++) {
          double v = 0.0;
          for (int k = a; k < a + n; k++)
            v += (double)sp[k] *
                 ((double)r.rate[(size_t)i * ngrid + k] * r.lag[(size_t)k * kRuleN3 + j]);
          *w++ = (float)v;
        }
      unsigned fail = r.usable ? 0u : 1u, loose = fail;
      for (int t = 0; r.usable && t < rule_tests(g); t++) {
        const int c = t / (2 * (g + 1)), i = t % (2 * (g + 1));
        float sum = 0.0f, err = 0.0f;
        for (int k = 0; k < n; k++) {
          const float v = sp[a + k] * r.rate[(size_t)i * ngrid + a + k];
          sum = fmaf(v, m[((size_t)k * ncol + c) * 2], sum);
          err = fmaf(v, m[((size_t)k * ncol + c) * 2 + 1], err);
        }
        const unsigned level = 1u << (c / kRuleMixes[g]);
        if (!(fabsf(err) <= kRuleTol * sum)) fail |= level;
        if (!(fabsf(err) <= kRuleLoose * sum)) loose |= level;
      }
      limit[(size_t)u * kRuleLimits + g] = rule_limit(g, fail);
      if (g == 0) limit[(size_t)u * kRuleLimits + 3] = rule_limit(3, loose);
      m += (size_t)n * ncol * 2;
    }
  }
}

}  // namespace argot
