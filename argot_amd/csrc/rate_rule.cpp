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
// How thick a ray the rule serves is found out for every spectrum: its
// error against the sum over bins is evaluated in full on test columns
// (mixes of the species at rising scales), and the spectrum's limit is the
// largest scale up to which every rate of every column stays within
// kRuleTol.  A steep or spiky spectrum gets a low limit or none; rays beyond
// it take the sum over bins.  A 1e5 K blackbody passes to optical depth 240 at the
// HI edge (24 where all species absorb), a 3e4 K one to 80 (8).
// Measured with the bin loops as the other side: the step on 256^3 cells and 4096
// sources 147 -> 111 ms, on 72 x 58 x 87 cells and 250 sources 13.0 -> 6.5 ms,
// with the same error against 64-bit rates (2.6e-7 and 8.4e-6 of the mesh's
// rates); 10, 12 and 16 nodes serve only half as thick rays at that error, and
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

// exp(-x) averaged over nothing but the column itself: the tests take f at
// zero cell depth.  A cell of depth d averages f over columns t to t + d, so
// its relative error is at most the largest among them.
double attenuate(double x) { return exp(-x); }

}  // namespace

void build_rate_rule(const float* sig, const float* hsig, int ngrid, int k1, int k2, RateRule* r) {
  const int nn[3] = {kRuleN1, kRuleN2, kRuleN3};
  const int first[4] = {0, k1, k2, ngrid};
  const int fit[3] = {11, 11, 13};   // terms of the fits to ln sigma
  r->usable = false;
  for (int g = 0; g < 4; g++) r->start[g] = first[g];
  r->sig.assign(3 * kRuleNodes, 0.0f);
  r->dsig.assign(3 * kRuleNodes, 0.0f);
  r->project.assign((size_t)ngrid * kRuleW3, 0.0);
  r->test.assign((size_t)ngrid * kRuleTests * 2, 0.0f);
  memset(r->edge, 0, sizeof r->edge);
  for (int g = 0; g < 3; g++)
    if (first[g + 1] - first[g] < nn[g]) return;
  // a species of range g has a positive cross-section in every bin of it
  for (int s = 0; s < 3; s++)
    for (int k = first[s]; k < ngrid; k++)
      if (!(sig[s * ngrid + k] > 0.0f) || !(sig[s * ngrid + k] < 1.0e-10f)) return;

  std::vector<double> nodes(3 * kRuleNodes, 0.0);   // sigma_s at the nodes
  std::vector<double> lag((size_t)ngrid * kRuleN3, 0.0);   // L_j(k) of bin k's range
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
  double last[3];
  for (int s = 0; s < 3; s++) last[s] = (double)sig[s * ngrid + ngrid - 1];
  for (int s = 0; s < 3; s++)
    for (int j = 0; j < kRuleNodes; j++) {
      r->sig[s * kRuleNodes + j] = (float)nodes[s * kRuleNodes + j];
      // (a species absent at the node enters through the range's constant)
      r->dsig[s * kRuleNodes + j] =
          nodes[s * kRuleNodes + j] > 0.0 ? (float)(nodes[s * kRuleNodes + j] - last[s]) : 0.0f;
    }
  // Bin k's share in the weights of its range.
  for (int g = 0; g < 3; g++)
    for (int k = first[g]; k < first[g + 1]; k++)
      for (int s = 0; s <= g; s++)
        for (int h = 0; h < 2; h++) {
          const double c = (double)(h ? hsig : sig)[s * ngrid + k] * kRuleScale;
          for (int j = 0; j < nn[g]; j++)
            r->project[(size_t)k * kRuleW3 + (2 * s + h) * nn[g] + j] =
                c * lag[(size_t)k * kRuleN3 + j];
        }
  // Test columns.
  const double mix[kRuleMixes][3] = {
      {1.0, 0.0, 0.0}, {0.0, 1.0, 0.0}, {0.0, 0.0, 1.0}, {1.0, 1.0, 1.0}, {1.0, 0.08, 0.01}};
  for (int g = 0; g < 3; g++)
    for (int s = 0; s < 3; s++)
      r->edge[g][s] = (float)((double)sig[s * ngrid + first[g]] / kRuleEdge[g]);
  for (int c = 0; c < kRuleColumns; c++) {
    const int level = c / kRuleMixes;   // kRuleLevels: the reversed ones
    double n[3], top = 0.0;
    for (int s = 0; s < 3; s++) n[s] = mix[c % kRuleMixes][s] / (double)sig[s * ngrid + first[s]];
    for (int g = 0; g < 3; g++) {
      double e = 0.0;
      for (int s = 0; s < 3; s++) e += n[s] * (double)sig[s * ngrid + first[g]] / kRuleEdge[g];
      top = std::max(top, e);
    }
    const double scale = (level < kRuleLevels ? (double)kRuleLevel[level] : -(double)kRuleNegative) / top;
    for (int s = 0; s < 3; s++) n[s] *= scale;
    double shift = 0.0;   // the smallest optical depth: f is at most 1
    for (int k = 0; k < ngrid; k++) {
      double tau = 0.0;
      for (int s = 0; s < 3; s++) tau += n[s] * (double)sig[s * ngrid + k];
      if (k == 0 || tau < shift) shift = tau;
    }
    double fn[kRuleNodes];
    for (int j = 0; j < kRuleNodes; j++) {
      double tau = 0.0;
      for (int s = 0; s < 3; s++) tau += n[s] * nodes[s * kRuleNodes + j];
      fn[j] = attenuate(tau - shift);
    }
    for (int g = 0, o = 0; g < 3; o += nn[g], g++)
      for (int k = first[g]; k < first[g + 1]; k++) {
        double tau = 0.0, q = 0.0;
        for (int s = 0; s < 3; s++) tau += n[s] * (double)sig[s * ngrid + k];
        const double f = attenuate(tau - shift);
        for (int j = 0; j < nn[g]; j++) q += lag[(size_t)k * kRuleN3 + j] * fn[o + j];
        for (int s = 0; s <= g; s++)
          for (int h = 0; h < 2; h++) {
            const double w = (double)(h ? hsig : sig)[s * ngrid + k] * kRuleScale;
            float* t = &r->test[((size_t)k * kRuleTests + 6 * c + 2 * s + h) * 2];
            t[0] = (float)(w * f);
            t[1] = (float)(w * (q - f));
          }
      }
  }
  r->usable = true;
}

void project_spectra_host(const RateRule& r, const float* spec, int nspec, int ngrid,
                          float* weight, float* limit) {
  // (an unusable rule has no bins to project and fails every spectrum)
  const int rows[4] = {0, kRuleW1, kRuleW1 + kRuleW2, kRuleWeights};
  for (int u = 0; u < nspec; u++) {
    const float* sp = spec + (size_t)u * ngrid;
    for (int g = 0; g < 3; g++)
      for (int o = rows[g]; o < rows[g + 1]; o++) {
        double w = 0.0;
        for (int k = r.start[g]; r.usable && k < r.start[g + 1]; k++)
          w += (double)sp[k] * r.project[(size_t)k * kRuleW3 + (o - rows[g])];
        weight[(size_t)u * kRuleWeights + o] = (float)w;
      }
    unsigned fail = r.usable ? 0u : 1u;
    for (int t = 0; t < kRuleTests; t++) {
      float sum = 0.0f, err = 0.0f;
      for (int k = 0; k < ngrid; k++) {
        const float* m = &r.test[((size_t)k * kRuleTests + t) * 2];
        sum += sp[k] * m[0];
        err += sp[k] * m[1];
      }
      if (!(fabsf(err) <= kRuleTol * sum)) {
        const int level = t / 6 / kRuleMixes;
        fail |= 1u << (level < kRuleLevels ? level : 0);
      }
    }
    int pass = 0;
    while (pass < kRuleLevels && !(fail >> pass & 1u)) pass++;
    limit[u] = pass > 0 ? kRuleLevel[pass - 1] : 0.0f;
  }
}

}  // namespace argot
