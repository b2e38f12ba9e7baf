// Launch interface of kernels.hip (host side of libargot_hip.so).
#pragma once
#include <hip/hip_runtime.h>

#include "argot_internal.h"
#include "surrogate.h"

namespace argot {

struct FusedArgs {
  GridDev grid;
  TreeDev tree;
  RateTables rates;
  const float4* nf;            // per-cell (nHI, nHeI, nHeII, 0)
  unsigned char* mesh;         // AoS fluid_mesh (reads fractions, adds rates)
  StepCounters* ctr;
  RayRecord* rec;              // capture mode only
  int64_t rec_cap;
  SurrDev surr;                // rate surrogate (surrogate launches only)
  int tile_bits[3];            // target tile of a wavefront: 2^bx x 2^by x 2^bz = 64 cells
};

hipError_t launch_pack_fields(const void* mesh, int64_t ncell, double helium_fact, float4* nf,
                              hipStream_t s);
hipError_t launch_zero_rates(void* mesh, int64_t ncell, hipStream_t s);
// launch_pack_fields and launch_zero_rates in one pass, and the counters to zero.
hipError_t launch_begin_step(void* mesh, int64_t ncell, double helium_fact, float4* nf,
                             StepCounters* ctr, hipStream_t s);
hipError_t launch_add_rates(void* mesh, const float* rate, int64_t ncell, hipStream_t s);
// rate[6c + k] := prev_chem rate k of cell c, and back
hipError_t launch_get_rates(const void* mesh, float* rate, int64_t ncell, hipStream_t s);
hipError_t launch_set_rates(void* mesh, const float* rate, int64_t ncell, hipStream_t s);
// wide: address the cell fields in 64 bits even when the mesh has fewer
// than 2^28 cells (meshes with more always are).
hipError_t launch_walk_segments(const GridDev& g, const float4* nf, void* seg, int64_t nseg,
                                int kahan, int wide, hipStream_t s);
// The same walk with the densities formed from the AoS mesh records at each
// crossing (no packed-field buffer; identical optical depths).
hipError_t launch_walk_segments_mesh(const GridDev& g, const void* mesh, double helium_fact,
                                     void* seg, int64_t nseg, int kahan, hipStream_t s);
// The quadrature rule on the device (rate_rule.h).
struct RuleDev {
  int usable;
  int start[4];
  const double* lag;       // [ngrid][kRuleN3]
  const float* rate;       // [6][ngrid]
  const float* test;       // by range: [bins][rule_columns][2]
};
// Quadrature weights [nspec * kRuleWeights] and limits [nspec * kRuleLimits] of spectra
// [nspec * ngrid].
hipError_t launch_project_spectra(const RuleDev& rule, const float* spec, int nspec, int ngrid,
                                  float* weight, float* limit, hipStream_t s);
// The distinct spectra of a calc_photoion_rate_cuda call.
struct CallSpectra {
  const float* spec32;     // [nspec * ngrid] scaled by 1/scale
  const double* spec64;    // [nspec * ngrid] as given
  const double* scale;     // [nspec] the spectrum's maximum
  const float* weight;     // quadrature weights of spec32, and
  const float* limit;      // the thickest rays they serve
};
// calc_photoion_rate_cuda: ntarget targets, each with its consecutive rays
// (rays[first .. first + count)), rates added to the mesh's prev_chem.
hipError_t launch_target_rates(const GridDev& g, const RateTables& rt, void* mesh,
                              const CallTarget* tg, int64_t ntarget, const CallRay* rays,
                              const CallSpectra& sp, hipStream_t s);
// smooth_photoion_rate on one rank; tmp_in: 6*ncell floats; tmp_out: null, or
// 6*ncell floats that get the smoothed rates as six planes too.
hipError_t launch_smooth_rates(void* mesh, int nx, int ny, int nz, float* tmp_in, float* tmp_out,
                               hipStream_t s);
hipError_t launch_copy_probe(const float4* src, float4* dst, int64_t n, int nblock,
                             hipStream_t s);
hipError_t launch_fused_step(const FusedArgs& a, int kahan, int capture, int surr, int wide,
                             int nblock, hipStream_t s);

// Chemistry (chemistry.hip).  Each launch first resets *ctr on the stream.
// queue_blocks > 0: the persistent cell-queue kernel on that many blocks;
// 0: one cell per thread.  paused: kPausedCells * kPausedBytes bytes.
constexpr int kPausedCells = 16384, kPausedBytes = 56;
hipError_t launch_chem_step(void* mesh, int64_t ncell, const ChemParams& p, float dtime,
                            ChemCounters* ctr, void* paused, int queue_blocks, int min_refill,
                            hipStream_t s);
hipError_t launch_chem_dtime(const void* mesh, int64_t ncell, const ChemParams& p,
                             ChemCounters* ctr, hipStream_t s);
hipError_t launch_chem_update(void* mesh, int64_t ncell, hipStream_t s);

}  // namespace argot
