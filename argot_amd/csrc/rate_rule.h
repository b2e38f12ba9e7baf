// Quadrature form of the frequency integral (see rate_rule.cpp).
#pragma once
#include <vector>

#include "argot_internal.h"

namespace argot {

// Nodes in the three bin ranges (HI alone; HI and HeI; all three species),
// each a multiple of 4.
constexpr int kRuleN1 = 12, kRuleN2 = 12, kRuleN3 = 20;
constexpr int kRuleNodes = kRuleN1 + kRuleN2 + kRuleN3;
// Weights of one spectrum: the rows G_HI, H_HI | G_HI, H_HI, G_HeI, H_HeI |
// G_HI, H_HI, G_HeI, H_HeI, G_HeII, H_HeII over the nodes of each range.
constexpr int kRuleW1 = 2 * kRuleN1, kRuleW2 = 4 * kRuleN2, kRuleW3 = 6 * kRuleN3;
constexpr int kRuleWeights = kRuleW1 + kRuleW2 + kRuleW3;
// Test columns a spectrum is tried on in each range: mixes of the range's
// species at rising scales, and at kRuleNegative with the sign reversed.  Between
// two scales an error can be larger than at both (a line's, mostly: five times
// with steps of 0.3 in the first range, which has one mix and so many scales).
constexpr int kRuleLevels[3] = {19, 9, 9}, kRuleMixes[3] = {1, 4, 6};
constexpr float kRuleLevel[3][19] = {
    {0.05f, 0.1f, 0.15f, 0.2f, 0.25f, 0.3f, 0.35f, 0.4f, 0.475f, 0.55f, 0.625f, 0.7f, 0.85f, 1.0f,
     1.15f, 1.3f, 1.7f, 2.3f, 3.0f},
    {0.2f, 0.4f, 0.7f, 1.0f, 1.3f, 1.7f, 2.3f, 2.7f, 3.0f},
    {0.2f, 0.4f, 0.7f, 1.0f, 1.3f, 1.7f, 2.3f, 2.7f, 3.0f}};
constexpr int rule_columns(int g) { return kRuleMixes[g] * (kRuleLevels[g] + 1); }
// Tests of a range: a rate (two of each species) on a column.
constexpr int rule_tests(int g) { return 2 * (g + 1) * rule_columns(g); }
constexpr int kRuleTests = rule_tests(0) + rule_tests(1) + rule_tests(2);
constexpr float kRuleNegative = 0.05f;   // scale of the columns of reversed sign
constexpr float kRuleTol = 1.0e-7f;     // relative error allowed on every test column
// Where HI is so thick that the first range leaves next to nothing of the whole,
// its nodes need not be that good: with at most kRuleLoose on the test columns (and
// five times that between them) they serve rays of whose sums the first range
// holds at most kRuleShare.
constexpr float kRuleLoose = 1.0e-2f;
constexpr double kRuleShare = 2.0e-6;
// Limits of a spectrum: by range at kRuleTol, and the first range's at kRuleLoose,
// for which its last three scales are (too far apart for the other).
constexpr int kRuleLimits = 4;   // (16 B: read at once)
constexpr int kRuleTopLevel[kRuleLimits] = {kRuleLevels[0] - 3, kRuleLevels[1], kRuleLevels[2],
                                            kRuleLevels[0]};
// Optical depths at the lower edges of the three ranges that scale 1 means.
constexpr double kRuleEdge[3] = {80.0, 25.0, 8.0};
// The weights carry the cross-sections times this power of two.
constexpr int kRuleExponent = 60;
constexpr double kRuleScale = 1152921504606846976.0;   // 2^60

struct RateRule {
  bool usable = false;              // the tables have three ranges long enough
  int start[4] = {0, 0, 0, 0};      // first bin of each range, and the bin count
  std::vector<double> node;         // [3 * kRuleNodes] sigma_s at the nodes, by species
  std::vector<float> sig, dsig;     // the same in FP32, and sigma_s - sigma_s(last bin of the range)
  std::vector<double> lag;          // [ngrid][kRuleN3]: the Lagrange polynomials of bin k's range
  std::vector<float> rate;          // [6][ngrid]: sigma_s and sigma_s (nu - nu_s), times kRuleScale
  std::vector<float> test;          // by range: [bins][rule_columns][2], f at bin k on each test
                                    // column and the nodes' error there
  float edge[3][3] = {};            // sigma_s at the first bin of each range / kRuleEdge
  float end[3] = {};                // sigma_HI at the last bin of the first range; sigma_HI and
                                    // sigma_HeI at the last bin of the second
};

// Rule for frequency tables in the layouts of RateTables (species-major sig
// and hsig, last-bin differences dsig); k1, k2: first bins of the second and
// third range.
void build_rate_rule(const float* sig, const float* hsig, int ngrid, int k1, int k2, RateRule* r);

// The i-th limit of a spectrum: the largest scale up to which no test has failed
// (bit 0 of fail: the reversed columns, bit l: level l - 1), 0 for none.
#ifdef __HIPCC__
__host__ __device__
#endif
inline float rule_limit(int i, unsigned fail) {
  float lim = 0.0f;
  for (int l = 0; l < kRuleTopLevel[i] && (fail & ((4u << l) - 1u)) == 0u; l++)
    lim = kRuleLevel[i % 3][l];
  return lim;
}

// Weights [nspec][kRuleWeights] and limits [nspec][kRuleLimits] of spectra
// spec[nspec][ngrid] on the host, as project_spectra_kernel forms them.
void project_spectra_host(const RateRule& r, const float* spec, int nspec, int ngrid,
                          float* weight, float* limit);

}  // namespace argot
