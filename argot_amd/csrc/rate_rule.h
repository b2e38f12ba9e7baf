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
// Test columns a spectrum is tried on: kRuleMixes mixes of the species at
// kRuleLevels scales, and with the sign of the smallest scale reversed.
constexpr int kRuleLevels = 6, kRuleMixes = 5;
constexpr int kRuleColumns = (kRuleLevels + 1) * kRuleMixes;
constexpr int kRuleTests = 6 * kRuleColumns;
constexpr float kRuleLevel[kRuleLevels] = {0.2f, 0.4f, 0.7f, 1.0f, 1.7f, 3.0f};
constexpr float kRuleNegative = 0.05f;   // scale of the columns of reversed sign
constexpr float kRuleTol = 1.0e-7f;     // relative error allowed on every test column
// Optical depths at the lower edges of the three ranges that scale 1 means.
constexpr double kRuleEdge[3] = {80.0, 25.0, 8.0};
// The weights carry the cross-sections times this power of two.
constexpr double kRuleScale = 1152921504606846976.0;   // 2^60

struct RateRule {
  bool usable = false;              // the tables have three ranges long enough
  int start[4] = {0, 0, 0, 0};      // first bin of each range, and the bin count
  std::vector<float> sig, dsig;     // [3 * kRuleNodes] sigma_s, sigma_s - sigma_s(last), by species
  std::vector<double> project;      // [ngrid][kRuleW3]: bin k's share in its range's weights
  std::vector<float> test;          // [ngrid][kRuleTests][2]: bin k's share in the full sum and
                                    // in the quadrature's error of each test column and rate
  float edge[3][3] = {};            // sigma_s at the first bin of each range / kRuleEdge
};

// Rule for frequency tables in the layouts of RateTables (species-major sig
// and hsig, last-bin differences dsig); k1, k2: first bins of the second and
// third range.
void build_rate_rule(const float* sig, const float* hsig, int ngrid, int k1, int k2, RateRule* r);

// Weights [nspec][kRuleWeights] and limits [nspec] of spectra
// spec[nspec][ngrid] on the host, as project_spectra_kernel forms them.
void project_spectra_host(const RateRule& r, const float* spec, int nspec, int ngrid,
                          float* weight, float* limit);

}  // namespace argot
