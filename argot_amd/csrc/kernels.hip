// HIP kernels of the point-source radiation step for gfx950 (MI355X).
//
//   pack_fields         AoS fluid_mesh -> per-cell FP32 (nHI, nHeI, nHeII)
//   zero_rates          prev_chem rates := 0         (zero_out_photoion_rate)
//   add_rates           prev_chem rates += table     (merge_photoion_data)
//   walk_segments       optical depth of a segment list (calc_optical_depth)
//   target_rates        per-target rates and sums of a ray list (calc_photoion_rate)
//   fused_step          tree walk + segment + optical depth + rates + per-cell
//                       sum for 4x4x4 target tiles, one wavefront per tile
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>

#include "argot_device.h"
#include "argot_internal.h"
#include "kernels.h"
#include "rate_rule.h"

namespace argot {

// Offsets inside struct fluid_mesh (156 B, include/argot_hip.h).
constexpr int kMeshStride = 156;
constexpr int kOffDens = 0;
constexpr int kOffFHI = 52;
constexpr int kOffFHeI = 60;
constexpr int kOffFHeII = 64;
constexpr int kOffRates = 124;   // prev_chem.GammaHI .. HeatHeII (6 floats)

__device__ __forceinline__ const float* mesh_f(const unsigned char* mesh, int64_t c, int off) {
  return reinterpret_cast<const float*>(mesh + c * kMeshStride + off);
}
__device__ __forceinline__ float* mesh_fw(unsigned char* mesh, int64_t c, int off) {
  return reinterpret_cast<float*>(mesh + c * kMeshStride + off);
}

// calc_optical_depth.c:150-156: nHI = dens*fHI, nHe = dens*HELIUM_FACT in
// double rounded to float, nHeI = nHe*fHeI, all FP32.
__device__ __forceinline__ float4 form_fields(const unsigned char* __restrict__ mesh, int64_t c,
                                              double helium_fact) {
  const float nH = *mesh_f(mesh, c, kOffDens);
  const float nHI = nH * *mesh_f(mesh, c, kOffFHI);
  const float nHe = (float)((double)nH * helium_fact);
  const float nHeI = nHe * *mesh_f(mesh, c, kOffFHeI);
  const float nHeII = nHe * *mesh_f(mesh, c, kOffFHeII);
  return make_float4(nHI, nHeI, nHeII, 0.0f);
}

__global__ void pack_fields_kernel(const unsigned char* __restrict__ mesh, int64_t ncell,
                                   double helium_fact, float4* __restrict__ nf) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  nf[c] = form_fields(mesh, c, helium_fact);
}

// Per-cell densities formed from the AoS mesh records at each crossing, with
// pack_fields_kernel's arithmetic (so the optical depths are the packed
// walk's bits): the walk of a call that has no packed-field buffer.
struct MeshFields {
  const unsigned char* __restrict__ mesh;
  double helium_fact;
  static constexpr uint32_t kScale = 1u;
  static constexpr bool kChecked = false;
  __device__ __forceinline__ float4 operator()(uint32_t idx) const {
    return form_fields(mesh, (int64_t)idx, helium_fact);
  }
};

__global__ void zero_rates_kernel(unsigned char* __restrict__ mesh, int64_t ncell) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  float* r = mesh_fw(mesh, c, kOffRates);
#pragma unroll
  for (int k = 0; k < 6; k++) r[k] = 0.0f;
}

// What a step begins with, in one pass over the records: the packed fields, the
// rates to zero, the counters of the fused kernel.  256^3: 1.04 ms (5.1 TB/s
// over the records read and written) instead of 0.53 and 0.85 in two passes;
// 64^3: 14 us instead of 29 in three launches.
__global__ void begin_step_kernel(unsigned char* __restrict__ mesh, int64_t ncell,
                                  double helium_fact, float4* __restrict__ nf,
                                  StepCounters* __restrict__ ctr) {
  if (blockIdx.x == 0) {
    const int i = threadIdx.x;
    if (i < kNumQueues) ctr->queue[i] = StepCounters::Queue{0, 0, 0, 0, 0, 0, 0};
    if (i == 0) {
      ctr->nrecord = 0;
      ctr->noverflow = 0;
    }
  }
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  nf[c] = form_fields(mesh, c, helium_fact);
  float* r = mesh_fw(mesh, c, kOffRates);
#pragma unroll
  for (int k = 0; k < 6; k++) r[k] = 0.0f;
}

__global__ void add_rates_kernel(unsigned char* __restrict__ mesh, const float* __restrict__ rate,
                                 int64_t ncell) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  float* r = mesh_fw(mesh, c, kOffRates);
#pragma unroll
  for (int k = 0; k < 6; k++) r[k] = r[k] + rate[6 * c + k];
}

// The six rates of every cell between the mesh and a photoion_rate table
// (24 B per cell, the prev_chem rates in the same order):
// recv_photoion_data_kernel / send_photoion_data_kernel of
// src/recv_photoion_data.cu and src/send_photoion_data.cu.
__global__ void get_rates_kernel(const unsigned char* __restrict__ mesh, int64_t ncell,
                                 float* __restrict__ rate) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  const float* r = mesh_f(mesh, c, kOffRates);
#pragma unroll
  for (int k = 0; k < 6; k++) rate[6 * c + k] = r[k];
}

__global__ void set_rates_kernel(unsigned char* __restrict__ mesh, const float* __restrict__ rate,
                                 int64_t ncell) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  float* r = mesh_fw(mesh, c, kOffRates);
#pragma unroll
  for (int k = 0; k < 6; k++) r[k] = rate[6 * c + k];
}

// ray_segment records (56 B): start @16, end @28, tau @40.  A block takes
// 256 consecutive segments and hands them to its lanes in order of their
// estimated crossing count (counting sort in LDS), so that the lanes of a
// wavefront walk segments of similar length; each segment's result does not
// depend on which lane walks it.
// walk(g, s, e, kahan, out) walks one segment: WalkPacked or WalkMesh.
constexpr int kWalkBlock = 256;

// Cap of the float form for a wavefront's segments.  A segment that ends outside
// the box leaves it before its end cell, and the float form would find that out
// late and hand it to the other; its wavefront takes the other form at once (2% of
// such segments: 0.82 ms for 2^19 of them without that, 0.72 by the other form
// alone).  Otherwise the segments cross at most one face more per axis than the
// cells between their ends; a cap that is too small only costs a second walk.
__device__ inline int segment_passes(const GridDev& g, Vec3f s, Vec3f e) {
  const bool inside = e.x >= g.xmin && e.x <= g.xmax && e.y >= g.ymin && e.y <= g.ymax &&
                      e.z >= g.zmin && e.z <= g.zmax;
  if (__any(!inside)) return 0;
  const float est = fabsf(e.x - s.x) * g.rdx + fabsf(e.y - s.y) * g.rdy + fabsf(e.z - s.z) * g.rdz;
  const int most = box_passes(g);
  int cap = 8;   // (crossings in pairs, and three faces more)
  while (cap < most && __any(!(est + 3.0f < 2.0f * (float)cap))) cap *= 2;
  return min(cap, most);
}

// The walk over packed densities (see walk_segment).
template <bool NARROW, bool POW2, bool FLOAT>
struct WalkPacked {
  // Wavefronts per SIMD.  The float form is bound by the gathers' cache lines:
  // more wavefronts push one another's out (8 Mi segments on 256^3: 4, 5 and 8
  // take 2.68, 2.85 and 3.0 ms).
  static constexpr int kWaves = FLOAT ? 4 : 8;
  const float4* nf;
  __device__ __forceinline__ void operator()(const GridDev& g, Vec3f s, Vec3f e, bool kahan,
                                             WalkOut* w) const {
    const RayDir dir = ray_dir(e.x - s.x, e.y - s.y, e.z - s.z);
    const int passes = FLOAT ? segment_passes(g, s, e) : 0;
    if (kahan)
      walk_segment<true, false, NARROW, POW2, FLOAT>(g, nf, dir, s, e, passes, w);
    else
      walk_segment<false, false, NARROW, POW2, FLOAT>(g, nf, dir, s, e, passes, w);
  }
};

// The walk over the mesh records.
template <bool POW2>
struct WalkMesh {
  static constexpr int kWaves = 8;
  MeshFields f;
  __device__ __forceinline__ void operator()(const GridDev& g, Vec3f s, Vec3f e, bool kahan,
                                             WalkOut* w) const {
    if (kahan)
      walk_segment_with<true, false, POW2>(g, f, s, e, w);
    else
      walk_segment_with<false, false, POW2>(g, f, s, e, w);
  }
};

template <typename Walk>
__global__ __launch_bounds__(kWalkBlock)
    __attribute__((amdgpu_waves_per_eu(Walk::kWaves, Walk::kWaves))) void walk_segments_kernel(
    GridDev g, Walk walk, unsigned char* __restrict__ seg, int64_t nseg, int kahan) {
  __shared__ unsigned bucket_lds[64];
  __shared__ unsigned perm_lds[kWalkBlock];
  const int t = threadIdx.x;
  const int64_t base = (int64_t)blockIdx.x * kWalkBlock;
  if (t < 64) bucket_lds[t] = 0;
  __syncthreads();
  unsigned b = 0;
  if (base + t < nseg) {
    const float* r = reinterpret_cast<const float*>(seg + (base + t) * 56);
    const float est = fabsf(r[7] - r[4]) / g.dx + fabsf(r[8] - r[5]) / g.dy +
                      fabsf(r[9] - r[6]) / g.dz;
    b = est < 504.0f ? (unsigned)est >> 3 : 63u;   // buckets of 8 crossings
  }
  const unsigned pos = atomicAdd(&bucket_lds[b], 1u);
  __syncthreads();
  if (t < 64) {   // exclusive prefix sum of the 64 bucket sizes (one wavefront)
    const unsigned v = bucket_lds[t];
    unsigned incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const unsigned u = __shfl_up(incl, d, 64);
      if (t >= d) incl += u;
    }
    bucket_lds[t] = incl - v;
  }
  __syncthreads();
  perm_lds[bucket_lds[b] + pos] = (unsigned)t;
  __syncthreads();
  const int64_t i = base + perm_lds[t];
  if (i >= nseg) return;
  float* rec = reinterpret_cast<float*>(seg + i * 56);
  const Vec3f s{rec[4], rec[5], rec[6]};
  const Vec3f e{rec[7], rec[8], rec[9]};
  WalkOut w;
  walk(g, s, e, kahan != 0, &w);
  rec[10] = w.tau[0];
  rec[11] = w.tau[1];
  rec[12] = w.tau[2];
}

// Bins [k0, k1) of the FP32 frequency loop with NS active species (the
// species s >= NS have sigma_s = 0 in these bins, so their optical depth
// enters only through the constant cst).  Tables are read with scalar loads
// (wave-uniform bin index); sums run in FP32 over 32 bins, then in FP64.
constexpr float kLog2e = 1.4426950408889634f;

// sinh(y)/y for 0 <= y <= 2.5 from yl = -log2(e) y: a degree-4 polynomial
// in u = y^2 (minimax relative error over u in [0, 6.25]: 3.3e-7 before
// rounding, 4.4e-7 after FP32 evaluation), evaluated in yl^2 with
// coefficient k scaled by log2(e)^(-2k).
constexpr double kL2 = 1.4426950408889634 * 1.4426950408889634;
constexpr float kSh0 = (float)1.0000003313e+00;
constexpr float kSh1 = (float)(1.6666356469e-01 / kL2);
constexpr float kSh2 = (float)(8.3377321051e-03 / (kL2 * kL2));
constexpr float kSh3 = (float)(1.9630612284e-04 / (kL2 * kL2 * kL2));
constexpr float kSh4 = (float)(3.1551783390e-06 / (kL2 * kL2 * kL2 * kL2));
// The polynomial's range: in-cell optical depth 2y <= kThinMax, i.e.
// yl >= kYlThin.
constexpr double kThinMax = 5.0;
constexpr float kYlThin = (float)(-0.5 * kThinMax * 1.4426950408889634);
__device__ __forceinline__ float sinhc_l(float yl) {
  const float u = yl * yl;
  float p = __builtin_fmaf(u, kSh4, kSh3);
  p = __builtin_fmaf(u, p, kSh2);
  p = __builtin_fmaf(u, p, kSh1);
  return __builtin_fmaf(u, p, kSh0);
}
// The same of degree 5 for the quadrature's nodes (minimax relative error
// 3.3e-9).  44 nodes average their roundings less than 256 bins do; with this
// the errors of their rates against 64 bits are still well below the bins': root
// mean square 0.7e-7 to 1.4e-7 over spectra and columns within the limits, 2.7e-7
// to 4.4e-7 by bins, where the other polynomial's 3.3e-7 at y = 0 dominates.
constexpr float kTh0 = (float)9.9999999673e-01;
constexpr float kTh1 = (float)(1.6666670980e-01 / kL2);
constexpr float kTh2 = (float)(8.3332447187e-03 / (kL2 * kL2));
constexpr float kTh3 = (float)(1.9847749592e-04 / (kL2 * kL2 * kL2));
constexpr float kTh4 = (float)(2.7347502032e-06 / (kL2 * kL2 * kL2 * kL2));
constexpr float kTh5 = (float)(2.8118837888e-08 / (kL2 * kL2 * kL2 * kL2 * kL2));
__device__ __forceinline__ float sinhc5_l(float yl) {
  const float u = yl * yl;
  float p = __builtin_fmaf(u, kTh5, kTh4);
  p = __builtin_fmaf(u, p, kTh3);
  p = __builtin_fmaf(u, p, kTh2);
  p = __builtin_fmaf(u, p, kTh1);
  return __builtin_fmaf(u, p, kTh0);
}

// Bins [k0, k1) of a ray whose in-cell optical depth is at most kThinMax in
// every bin: exp(-tau) (1 - exp(-dtau)) / dtau = exp(-(tau + y)) sinh(y)/y with
// y = dtau/2, one exponential per bin.  dl holds the ray's in-cell weights
// times -log2(e)/2, so that their sum with the cross sections is
// yl = -log2(e) y and 2^(yl - log2(e) tau) = exp(-(tau + y)).  FOLD (bins
// where cst = 0): nl holds the column densities times -log2(e), and the
// exponent is summed onto yl directly, one instruction fewer per bin.
template <int NS, bool FOLD, typename SpecF>
__device__ __forceinline__ void rate_bins_thin(const RateTables& rt, int k0, int k1, float cst,
                                               const float n[3], const float nl[3],
                                               const float dl[3], SpecF spec, double G[3],
                                               double H[3]) {
  const int ng = rt.ngrid;
  for (int c = k0; c < k1; c += 32) {
    float g[NS], h[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) g[s] = h[s] = 0.0f;
    const int ce = min(c + 32, k1);
#pragma unroll 4
    for (int k = c; k < ce; k++) {
      float sg[NS], hs[NS];
      float yl = 0.0f, z;
#pragma unroll
      for (int s = 0; s < NS; s++) {
        sg[s] = ldc(rt.sig + s * ng + k);
        hs[s] = ldc(rt.hsig + s * ng + k);
        yl = __builtin_fmaf(dl[s], sg[s], yl);
      }
      if constexpr (FOLD) {
        z = yl;
#pragma unroll
        for (int s = 0; s < NS; s++) z = __builtin_fmaf(nl[s], ldc(rt.dsig + s * ng + k), z);
      } else {
        float tau = cst;
#pragma unroll
        for (int s = 0; s < NS; s++) tau = __builtin_fmaf(n[s], ldc(rt.dsig + s * ng + k), tau);
        z = __builtin_fmaf(tau, -kLog2e, yl);
      }
      const float e = __builtin_amdgcn_exp2f(z);
      const float b = spec(k) * e * sinhc_l(yl);
#pragma unroll
      for (int s = 0; s < NS; s++) {
        g[s] = __builtin_fmaf(sg[s], b, g[s]);
        h[s] = __builtin_fmaf(hs[s], b, h[s]);
      }
    }
#pragma unroll
    for (int s = 0; s < NS; s++) {
      G[s] += g[s];
      H[s] += h[s];
    }
  }
}

// Bins [k0, k1) for a wavefront in which some lane's ray has an in-cell
// optical depth above kThinMax.  A lane flagged thin computes exactly what
// rate_bins_thin computes (the same operations in the same order), so a
// cell's rates do not depend on which rays share its wavefront.  The other
// lanes take, bin by bin, the same thin form where yl >= kYlThin, and
// otherwise exp(-tau) (1 - exp(-2y)) / (2y) with the optical depth tau
// summed on its own (no cancellation: exp(-2y) <= exp(-kThinMax)).
template <int NS, bool FOLD, typename SpecF>
__device__ __forceinline__ void rate_bins_mixed(const RateTables& rt, int k0, int k1, float cst,
                                                const float n[3], const float nl[3],
                                                const float dl[3], bool thin, SpecF spec,
                                                double G[3], double H[3]) {
  constexpr float kHalfLog2eN = -0.5f * kLog2e;  // 1/(2y) = kHalfLog2eN / yl
  const int ng = rt.ngrid;
  for (int c = k0; c < k1; c += 32) {
    float g[NS], h[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) g[s] = h[s] = 0.0f;
    const int ce = min(c + 32, k1);
#pragma unroll 2
    for (int k = c; k < ce; k++) {
      float sg[NS], hs[NS], ds[NS];
      float yl = 0.0f, z, tau = cst;
#pragma unroll
      for (int s = 0; s < NS; s++) {
        sg[s] = ldc(rt.sig + s * ng + k);
        hs[s] = ldc(rt.hsig + s * ng + k);
        ds[s] = ldc(rt.dsig + s * ng + k);
        yl = __builtin_fmaf(dl[s], sg[s], yl);
      }
#pragma unroll
      for (int s = 0; s < NS; s++) tau = __builtin_fmaf(n[s], ds[s], tau);
      if constexpr (FOLD) {
        z = yl;
#pragma unroll
        for (int s = 0; s < NS; s++) z = __builtin_fmaf(nl[s], ds[s], z);
      } else {
        z = __builtin_fmaf(tau, -kLog2e, yl);
      }
      const float sk = spec(k);
      const float bt = sk * __builtin_amdgcn_exp2f(z) * sinhc_l(yl);
      const float e1 = __builtin_amdgcn_exp2f(tau * -kLog2e);
      const float om = 1.0f - __builtin_amdgcn_exp2f(yl + yl);
      const float bk = sk * e1 * om * (__builtin_amdgcn_rcpf(yl) * kHalfLog2eN);
      const float b = (thin || yl >= kYlThin) ? bt : bk;
#pragma unroll
      for (int s = 0; s < NS; s++) {
        g[s] = __builtin_fmaf(sg[s], b, g[s]);
        h[s] = __builtin_fmaf(hs[s], b, h[s]);
      }
    }
#pragma unroll
    for (int s = 0; s < NS; s++) {
      G[s] += g[s];
      H[s] += h[s];
    }
  }
}

typedef float F4 __attribute__((ext_vector_type(4)));

// Nodes [o, o + N) of the quadrature form for one bin range with NS active
// species: the same f as the bin loops above (thin form, and in MIXED
// wavefronts the direct form by lane and node), at the range's nodes, summed
// with the spectrum's weight rows G_s, H_s into g, h.  w(i): the i-th four
// weights of the range.  The optical depths are those beyond the depth at the range's last
// bin, whose attenuation the caller puts in: the sums come from there, and what FP32
// rounds off an optical depth is relative to its size.  (Taken beyond the depth
// at the last bin of all, a ray of 100 at the HI edge has 25 at the end of the
// first range and its rates errors of 2e-6, as large as the bin loops'.)
template <int NS, int N, bool MIXED, typename WeightF>
__device__ __forceinline__ void rate_nodes(const RateTables& rt, int o, const float nl[3],
                                           const float dl[3], bool thin, WeightF w, float g[NS],
                                           float h[NS]) {
  constexpr float kHalfLog2eN = -0.5f * kLog2e;
#pragma unroll
  for (int s = 0; s < NS; s++) g[s] = h[s] = 0.0f;
#pragma unroll 1
  for (int j = 0; j < N; j += 4) {
    F4 sg[NS], ds[NS], wg[NS], wh[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
      sg[s] = ldc(reinterpret_cast<const F4*>(rt.qsig + s * kRuleNodes + o + j));
      ds[s] = ldc(reinterpret_cast<const F4*>(rt.qdsig + s * kRuleNodes + o + j));
      wg[s] = w((2 * s * N + j) / 4);
      wh[s] = w(((2 * s + 1) * N + j) / 4);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      float yl = 0.0f;
#pragma unroll
      for (int s = 0; s < NS; s++) yl = __builtin_fmaf(dl[s], sg[s][i], yl);
      float z = yl;
#pragma unroll
      for (int s = 0; s < NS; s++) z = __builtin_fmaf(nl[s], ds[s][i], z);
      float f = __builtin_amdgcn_exp2f(z) * sinhc5_l(yl);
      if constexpr (MIXED) {
        float zt = 0.0f;
#pragma unroll
        for (int s = 0; s < NS; s++) zt = __builtin_fmaf(nl[s], ds[s][i], zt);
        const float om = 1.0f - __builtin_amdgcn_exp2f(yl + yl);
        const float fk =
            __builtin_amdgcn_exp2f(zt) * om * (__builtin_amdgcn_rcpf(yl) * kHalfLog2eN);
        f = (thin || yl >= kYlThin) ? f : fk;
      }
#pragma unroll
      for (int s = 0; s < NS; s++) {
        g[s] = __builtin_fmaf(wg[s][i], f, g[s]);
        h[s] = __builtin_fmaf(wh[s][i], f, h[s]);
      }
    }
  }
}

// exp(x) 2^e as 2^n 2^f, n = floor(x log2 e) and f in [0, 1): the FP32
// exponential of f (relative error about 1e-7) times an exact power of two, in
// FP64 range.  The library exponential's polynomial would hold a dozen FP64
// constants in registers across the kernel, which the register budget spills.
// (fast_rate_ok bounds x above.)
__device__ __forceinline__ double exp_scaled(double x, int e) {
  constexpr double kLog2eD = 1.4426950408889634;
  const double xl = x * kLog2eD;
  const double fl = fmax(floor(xl), -2000.0);
  return ldexp((double)__builtin_amdgcn_exp2f((float)(xl - fl)), (int)fl + e);
}

// One range of the frequency integral: by N nodes from node o on, or bin by bin.
// unit: the nodes' unit in that of G, H.  loose: the nodes serve only if their sums
// are at most kRuleShare of G[0], H[0] (else they are dropped for the bins).
template <int NS, int N, bool FOLD, typename SpecF, typename WeightF>
__device__ __forceinline__ void rate_range(const RateTables& rt, bool nodes, bool loose,
                                           bool all_thin, int k0, int k1, int o, double unit,
                                           float cst, const float n[3], const float nl[3],
                                           const float dl[3], bool thin, SpecF spec, WeightF w,
                                           double G[3], double H[3]) {
  if (nodes) {
    float g[NS], h[NS];
    if (all_thin)
      rate_nodes<NS, N, false>(rt, o, nl, dl, thin, w, g, h);
    else
      rate_nodes<NS, N, true>(rt, o, nl, dl, thin, w, g, h);
    const double g0 = (double)g[0] * unit, h0 = (double)h[0] * unit;
    if (NS == 1 && loose && !(g0 <= kRuleShare * G[0] && h0 <= kRuleShare * H[0])) {
      nodes = false;
    } else {
      G[0] += g0;
      H[0] += h0;
#pragma unroll
      for (int s = 1; s < NS; s++) {
        G[s] = __builtin_fma((double)g[s], unit, G[s]);
        H[s] = __builtin_fma((double)h[s], unit, H[s]);
      }
    }
  }
  if (!nodes) {
    if (all_thin)
      rate_bins_thin<NS, FOLD>(rt, k0, k1, cst, n, nl, dl, spec, G, H);
    else
      rate_bins_mixed<NS, FOLD>(rt, k0, k1, cst, n, nl, dl, thin, spec, G, H);
  }
}

// FP32 frequency integral (photon-conserving form, calc_photoion_rate.c:327-386
// regrouped): with B_k = N_k exp(-tau_k) (1 - exp(-dtau_k)) / dtau_k,
//   Gamma_s = r_s d_s sum_k sigma_s(k) B_k,  Heat_s = r_s d_s sum_k hsig_s(k) B_k.
// The optical depth is shifted by its last-bin value tsh (folded back in
// FP64): tau_k - tsh = sum_s N_s (sigma_s(k) - sigma_s(last)).  Bins below
// the HeI and HeII edges skip the absent species.
// In a range within whose limit of its spectrum it lies a ray takes the sums as
// quadratures over the range's nodes (rate_rule.cpp), in any other bin by bin;
// which one depends on the ray alone, not on its wavefront.  limit: the
// spectrum's (kRuleLimits).
template <typename SpecF, typename WeightF>
__device__ inline void rate_loop_f32(const RateTables& rt, const RayRate& rr, double scale,
                                     F4 limit, SpecF spec, WeightF weight, double out[6]) {
  const double sh2 = rr.t[2] * rt.cs_last[2];
  const double sh1 = __builtin_fma(rr.t[1], rt.cs_last[1], sh2);
  const double tsh = __builtin_fma(rr.t[0], rt.cs_last[0], sh1);
  const float n[3] = {(float)rr.t[0], (float)rr.t[1], (float)rr.t[2]};
  const float c1 = (float)-sh1;
  const float c2 = (float)-sh2;
  // Scale of the ray against the rule's test columns in each range, from its
  // columns at the far side of the cell (and, where the half-cell shift made
  // one negative, its negative part).
  bool nodes[3], loose = false;   // loose: the first range's nodes, for a small share
  {
    float tf[3], tn[3];
#pragma unroll
    for (int s = 0; s < 3; s++) {
      tf[s] = fmaxf(n[s], n[s] + (float)rr.d[s]);
      tn[s] = fmaxf(-n[s], 0.0f);
    }
#pragma unroll
    for (int g = 0; g < 3; g++) {
      float e = 0.0f, m = 0.0f;
#pragma unroll
      for (int s = 0; s <= g; s++) {
        e = __builtin_fmaf(fabsf(tf[s]), rt.edge[3 * g + s], e);
        m = __builtin_fmaf(tn[s], rt.edge[3 * g + s], m);
      }
      const float top = limit[g];
      nodes[g] = e <= top && m <= kRuleNegative && top > 0.0f;
      if (g == 0) loose = !nodes[0] && e <= limit[3] && m <= kRuleNegative && limit[3] > 0.0f;
    }
  }
  // per-ray prefactors first (same operations as after the loop), so that
  // only they, not the ray's FP64 quantities, stay live through the bins
  const double pre = scale * exp_scaled(-tsh, 0);
  const double p0 = 1.0 / rr.v[0] * rr.d[0] * pre;
  const double p1 = 1.0 / rr.v[1] * rr.d[1] * pre;
  const double p2 = 1.0 / rr.v[2] * rr.d[2] * pre;
  double G[3] = {0, 0, 0}, H[3] = {0, 0, 0};
  // largest in-cell optical depth of this ray over the bins.  A wavefront
  // whose rays are all thin runs the thin loop; one with a thicker ray runs
  // the combined loop, in which a thin lane does the thin loop's operations
  // exactly, so a cell's rates do not depend on which rays share its
  // wavefront (tile shape, grid size).
  const double dmax = rr.d[0] * rt.cs_max[0] + rr.d[1] * rt.cs_max[1] + rr.d[2] * rt.cs_max[2];
  constexpr double kHalfLog2e = 0.5 * 1.4426950408889634;
  constexpr double kLog2eD = 1.4426950408889634;
  const float dl[3] = {(float)(rr.d[0] * -kHalfLog2e), (float)(rr.d[1] * -kHalfLog2e),
                       (float)(rr.d[2] * -kHalfLog2e)};
  const float nl[3] = {(float)(rr.t[0] * -kLog2eD), (float)(rr.t[1] * -kLog2eD),
                       (float)(rr.t[2] * -kLog2eD)};
  const bool thin = dmax <= kThinMax;
  const bool all_thin = __all(thin);
  // (the sums are in units of exp(-tsh), the nodes' weights in those of kRuleScale)
  const double unit1 = exp_scaled(tsh - rr.t[0] * rt.end[0], -kRuleExponent);
  const double unit2 = exp_scaled(
      tsh - __builtin_fma(rr.t[0], rt.end[1], rr.t[1] * rt.end[2]), -kRuleExponent);
  rate_range<3, kRuleN3, true>(rt, nodes[2], false, all_thin, rt.k_he2, rt.ngrid, kRuleN1 + kRuleN2,
                               1.0 / kRuleScale, 0.0f, n, nl, dl, thin, spec,
                               [&](int i) { return weight((kRuleW1 + kRuleW2) / 4 + i); }, G, H);
  rate_range<2, kRuleN2, false>(rt, nodes[1], false, all_thin, rt.k_he1, rt.k_he2, kRuleN1, unit2,
                                c2, n, nl, dl, thin, spec,
                                [&](int i) { return weight(kRuleW1 / 4 + i); }, G, H);
  rate_range<1, kRuleN1, false>(rt, nodes[0] || loose, loose, all_thin, 0, rt.k_he1, 0, unit1, c1,
                                n, nl, dl, thin, spec, weight, G, H);
  out[0] = p0 * G[0];
  out[1] = p0 * H[0] * kHnuL;
  out[2] = p1 * G[1];
  out[3] = p2 * G[2];
  out[4] = p1 * H[1] * kHnuL;
  out[5] = p2 * H[2] * kHnuL;
}

// Quadrature weights and limits of nspec spectra (rows of ngrid floats,
// scaled to their maximum): a thread per weight (192) and per test (560), a
// wavefront's all of one range, so that its loop has uniform bounds and eight of
// its loads in flight: the chain of loads over the 153 bins of the last range is
// what a launch on few spectra takes (23 us on the tree of 16 sources; with bounds
// that differ between lanes, and loads waited for one by one, 50).  A block takes NB
// spectra, so that each entry it reads of the rule's tables serves NB of them.
// first thread of each kind: weights by range, then tests by range
constexpr int wave_up(int n) { return (n + 63) & ~63; }
constexpr int kAtW2 = wave_up(kRuleW1), kAtW3 = kAtW2 + wave_up(kRuleW2),
              kAtT1 = kAtW3 + wave_up(kRuleW3), kAtT2 = kAtT1 + wave_up(rule_tests(0)),
              kAtT3 = kAtT2 + wave_up(rule_tests(1)),
              kProjectThreads = kAtT3 + wave_up(rule_tests(2));
static_assert(kProjectThreads <= 1024, "one block");
template <int NB>
__global__ __launch_bounds__(kProjectThreads) void project_spectra_kernel(
    RuleDev rule, const float* __restrict__ spec, int nspec, int ngrid,
    float* __restrict__ weight, float* __restrict__ limit) {
  __shared__ float sp[kNgridMax][NB];
  __shared__ float rate[6][kNgridMax + 1];   // (rows in different banks)
  __shared__ unsigned fail[kRuleLimits * NB];
  const int t = threadIdx.x;
  const int u0 = blockIdx.x * NB;
  for (int i = t; i < NB * ngrid; i += kProjectThreads) {
    const int j = i / ngrid, k = i % ngrid;
    sp[k][j] = u0 + j < nspec ? spec[(int64_t)(u0 + j) * ngrid + k] : 0.0f;
  }
  if (rule.usable)
    for (int i = t; i < 6 * ngrid; i += kProjectThreads) rate[i / ngrid][i % ngrid] = rule.rate[i];
  if (t < kRuleLimits * NB) fail[t] = 0u;
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(t) & ~63;   // its first thread
  if (wave < kAtT1) {
    const int g = wave < kAtW2 ? 0 : wave < kAtW3 ? 1 : 2;
    const int o = t - (g == 0 ? 0 : g == 1 ? kAtW2 : kAtW3);
    const int nn = g == 0 ? kRuleN1 : g == 1 ? kRuleN2 : kRuleN3;
    const int row = min(o / nn, 2 * g + 1), node = o % nn;   // (lanes beyond the rows: the last)
    const double* __restrict__ lag = rule.lag + node;
    double w[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) w[j] = 0.0;
    const int first = rule.start[g], last = rule.start[g + 1];
    constexpr int kAhead = NB > 4 ? 2 : 8;   // (more spill where a block holds many sums)
    for (int k0 = first; k0 < last; k0 += kAhead) {
      double l[kAhead];
#pragma unroll
      for (int i = 0; i < kAhead; i++) l[i] = lag[min(k0 + i, last - 1) * kRuleN3];
      __builtin_amdgcn_sched_barrier(0);   // (the loads go out together)
#pragma unroll
      for (int i = 0; i < kAhead; i++) {
        const int k = min(k0 + i, last - 1);
        const double m = k0 + i < last ? (double)rate[row][k] * l[i] : 0.0;
#pragma unroll
        for (int j = 0; j < NB; j++) w[j] += (double)sp[k][j] * m;
      }
    }
    const int at = g == 0 ? 0 : g == 1 ? kRuleW1 : kRuleW1 + kRuleW2;
#pragma unroll
    for (int j = 0; j < NB; j++)
      if (u0 + j < nspec && o < 2 * (g + 1) * nn)
        weight[(int64_t)(u0 + j) * kRuleWeights + at + o] = (float)w[j];
  } else if (rule.usable) {
    const int g = wave < kAtT2 ? 0 : wave < kAtT3 ? 1 : 2;
    const int q = t - (g == 0 ? kAtT1 : g == 1 ? kAtT2 : kAtT3);
    const int ncol = g == 2 ? rule_columns(2) : g == 1 ? rule_columns(1) : rule_columns(0);
    const int mixes = g == 2 ? kRuleMixes[2] : g == 1 ? kRuleMixes[1] : kRuleMixes[0];
    const int c = min(q / (2 * (g + 1)), ncol - 1);   // (lanes beyond the tests repeat one)
    const int row = q % (2 * (g + 1));
    const int first = rule.start[g], last = rule.start[g + 1];
    const float2* __restrict__ f =
        reinterpret_cast<const float2*>(rule.test) + c +
        (g > 0 ? (rule.start[1] - rule.start[0]) * rule_columns(0) : 0) +
        (g > 1 ? (rule.start[2] - rule.start[1]) * rule_columns(1) : 0);
    float sum[NB], err[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) sum[j] = err[j] = 0.0f;
#pragma unroll 8
    for (int k = first; k < last; k++) {
      const float2 m = f[(k - first) * ncol];
      const float r = rate[row][k];
#pragma unroll
      for (int j = 0; j < NB; j++) {
        const float v = sp[k][j] * r;
        sum[j] = __builtin_fmaf(v, m.x, sum[j]);
        err[j] = __builtin_fmaf(v, m.y, err[j]);
      }
    }
    const int level = c / mixes;
#pragma unroll
    for (int j = 0; j < NB; j++) {
      if (!(fabsf(err[j]) <= kRuleTol * sum[j])) atomicOr(&fail[kRuleLimits * j + g], 1u << level);
      if (g == 0 && !(fabsf(err[j]) <= kRuleLoose * sum[j]))
        atomicOr(&fail[kRuleLimits * j + 3], 1u << level);
    }
  }
  __syncthreads();
  if (t < kRuleLimits * NB && u0 + t / kRuleLimits < nspec) {
    const unsigned f = rule.usable ? fail[t] : 1u;
    const int i = t % kRuleLimits;
    const float lim[kRuleLimits] = {rule_limit(0, f), rule_limit(1, f), rule_limit(2, f),
                                    rule_limit(3, f)};
    limit[(int64_t)kRuleLimits * u0 + t] =
        i == 0 ? lim[0] : i == 1 ? lim[1] : i == 2 ? lim[2] : lim[3];
  }
}

// Lower bound of the shifted bin optical depth and upper bound of the
// in-cell optical depth decide whether the FP32 loop is safe.
__device__ __forceinline__ bool fast_rate_ok(const RateTables& rt, const RayRate& rr) {
  double lo = 0.0, dmax = 0.0;
  bool finite = true;
  for (int s = 0; s < 3; s++) {
    lo += rr.t[s] >= 0.0 ? -rr.t[s] * rt.cs_last[s] : rr.t[s] * rt.cs_span[s];
    dmax += rr.d[s] * rt.cs_max[s];
    finite = finite && fabs(rr.t[s]) < 1.0e36 && rr.d[s] < 1.0e36;
  }
  return finite && lo > -60.0 && dmax < 1.0e30;
}

__device__ __forceinline__ int wave_min(int v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = min(v, __shfl_xor(v, off, 64));
  return __builtin_amdgcn_readfirstlane(v);
}

// Orders the LDS accesses of the lanes of a wavefront before and after it (a
// block of one wavefront needs no barrier: its LDS accesses are in order).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// ARGOT_WAVES_PER_EU (build option, 4 by default) caps the register budget of
// the fused and the per-call rate kernels so that this many wavefronts fit per
// SIMD.  Their issue and the gathers' cache lines bound them, so registers
// (spills are instructions) count for more than wavefronts: on 256^3 cells and
// 4096 sources 3, 4, 5 and 6 wavefronts take 84, 81, 87 and 90 ms, on 128^3 and
// 1024 with Kahan sums 27.0, 28.0, 30.6 and 32.1, on 72 x 58 x 87 and 250 4.2, 4.3,
// 4.8 and 5.3 (each with the grid that fills it).
#if defined(ARGOT_WAVES_PER_EU) && ARGOT_WAVES_PER_EU > 0
#define ARGOT_OCCUPANCY __attribute__((amdgpu_waves_per_eu(ARGOT_WAVES_PER_EU)))
#else
#define ARGOT_OCCUPANCY
#endif

// calc_photoion_rate_cuda (calc_photoion_rate_cuda.cu:92-216 with the
// per-target merge of calc_photoion_rate.c:403-425): one lane per target
// cell.  A target's rays are consecutive in the caller's order and its lane
// sums their rates in FP64 in that order, then adds the sum to the cell
// once: no atomics, no per-ray buffer.  Each ray names one of the call's
// distinct spectra (rays from one source or tree node share it), whose
// quadrature weights (768 B) its lane reads in 16-B loads: every lane takes
// its next ray at each pass, whichever spectra the wavefront's rays have.
// Each ray's arithmetic is the fused kernel's, so a ray list taken from the
// fused step gives its bits.
__global__ __launch_bounds__(64) ARGOT_OCCUPANCY void target_rates_kernel(
    GridDev g, RateTables rt, unsigned char* __restrict__ mesh, const CallTarget* __restrict__ tg,
    int64_t ntarget, const CallRay* __restrict__ rays, CallSpectra sp) {
  const int lane = threadIdx.x;
  const int64_t t = (int64_t)blockIdx.x * 64 + lane;
  const bool valid = t < ntarget;
  CallTarget T{0, 0, 0, {0, 0, 0}};
  if (valid) T = tg[t];
  float dens = 0.0f, fHI = 0.0f, fHeI = 0.0f, fHeII = 0.0f;
  if (valid) {
    dens = *mesh_f(mesh, T.cell, kOffDens);
    fHI = *mesh_f(mesh, T.cell, kOffFHI);
    fHeI = *mesh_f(mesh, T.cell, kOffFHeI);
    fHeII = *mesh_f(mesh, T.cell, kOffFHeII);
  }
  const Vec3f tgt{cell_centre(g.gxmin, T.g[0], g.dx), cell_centre(g.gymin, T.g[1], g.dy),
                  cell_centre(g.gzmin, T.g[2], g.dz)};
  int64_t r = T.first;
  const int64_t rend = T.first + T.count;
  double acc[6] = {0, 0, 0, 0, 0, 0};
  const int ng = rt.ngrid;
  while (__any(r < rend)) {
    const bool more = r < rend;
    bool wide = false;   // FP32 cannot serve this ray
    int u = 0;
    RayRate rr;
    double res[6];
    if (more) {
      const CallRay R = rays[r];
      u = R.spec;
      const Vec3f src{R.src[0], R.src[1], R.src[2]};
      const Vec3f d{tgt.x - src.x, tgt.y - src.y, tgt.z - src.z};
      const Chord chord = ray_chord(g, ray_dir(d.x, d.y, d.z), d.x, d.y, d.z);
      ray_rate_setup(g, chord, R.tau, dens, fHI, fHeI, fHeII, &rr);
      wide = !fast_rate_ok(rt, rr);
    }
    rate_f64_wave(rt, rr, wide,
                  [&](int owner, int k) {
                    return sp.spec64[(int64_t)__shfl(u, owner, 64) * ng + k];
                  },
                  res);
    if (more && !wide) {
      const float* s32 = sp.spec32 + (int64_t)u * ng;
      const F4* w = reinterpret_cast<const F4*>(sp.weight + (int64_t)u * kRuleWeights);
      const F4 limit = reinterpret_cast<const F4*>(sp.limit)[u];
      rate_loop_f32(rt, rr, sp.scale[u], limit, [&](int k) { return s32[k]; },
                    [&](int i) { return w[i]; }, res);
    }
    if (more) {
#pragma unroll
      for (int k = 0; k < 6; k++) acc[k] += res[k];
      r++;
    }
  }
  if (valid && T.count > 0) {
    float* o = mesh_fw(mesh, T.cell, kOffRates);
#pragma unroll
    for (int k = 0; k < 6; k++) o[k] = (float)((double)o[k] + acc[k]);
  }
}

// Every third bit of v (bits 0, 3, 6, ...) packed together: one axis of a
// Morton index.
__device__ __forceinline__ uint32_t compact3(uint32_t v) {
  v &= 0x09249249u;
  v = (v ^ (v >> 2)) & 0x030c30c3u;
  v = (v ^ (v >> 4)) & 0x0300f00fu;
  v = (v ^ (v >> 8)) & 0xff0000ffu;
  v = (v ^ (v >> 16)) & 0x000003ffu;
  return v;
}

// Next tile for this wavefront: its own XCD's queue first (blocks are
// dispatched round-robin over the 8 XCDs), then the others in turn.  A queue
// that a plain load shows to be drained is passed over without an atomic
// (the counters only grow): at the end of a launch every wavefront looks at
// every queue, and 6144 wavefronts' atomics on 8 words of one cache line took
// 0.6 ms, half of a 16^3 mesh's step.
__device__ __forceinline__ int64_t next_tile(StepCounters* ctr, int64_t ntile, int* q, int* tried) {
  while (*tried < kNumQueues) {
    const int64_t lo = ntile * (*q) / kNumQueues;
    const int64_t hi = ntile * (*q + 1) / kNumQueues;
    int* const next = &ctr->queue[*q].next;
    int t = 0;
    if (threadIdx.x == 0) {
      t = __hip_atomic_load(next, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (lo + t < hi) t = atomicAdd(next, 1);
    }
    t = __shfl(t, 0, 64);
    if (lo + t < hi) return lo + t;
    *q = (*q + 1) % kNumQueues;
    (*tried)++;
  }
  return -1;
}


// 2-point Gauss-Legendre nodes on [0, 1].
constexpr double kGl1 = 0.21132486540518711775, kGl2 = 0.78867513459481288225;

// Can the network serve this ray?  Its node's spectrum must have the
// trained shape (q > 0), the in-cell optical depth must be small enough
// for the 2-point rule, and both nodes of the in-cell path (threshold
// optical depths (t_s + x d_s) sig_th_s) must lie below the hull's upper
// edge and in trusted cells.  Below the lower edge the kernels are flat
// (relative change < 1e-5), so inputs are clamped there.
__device__ inline bool surr_inputs(const SurrDev& S, const RateTables& rt, const RayRate& rr,
                                   double q, float xa[3], float xb[3]) {
  if (!(q > 0.0)) return false;
  bool ok = true;
  double dmax = 0.0;
  int ca[3], cb[3];
#pragma unroll
  for (int s = 0; s < 3; s++) {
    const double t = rr.t[s], d = rr.d[s];
    ok = ok && t >= 0.0 && d >= 0.0;
    dmax += d * rt.cs_max[s];
    const double ta = (t + kGl1 * d) * (double)S.sig_th[s];
    const double tb = (t + kGl2 * d) * (double)S.sig_th[s];
    ok = ok && tb <= S.tau_hi;
    xa[s] = __log10f((float)fmax(ta, S.tau_lo));
    xb[s] = __log10f((float)fmax(tb, S.tau_lo));
    ca[s] = min(S.trust_n - 1, max(0, (int)((xa[s] - S.lo) * S.inv_cell)));
    cb[s] = min(S.trust_n - 1, max(0, (int)((xb[s] - S.lo) * S.inv_cell)));
  }
  ok = ok && dmax <= (double)S.dtau_max;
  if (!ok) return false;
  const int n = S.trust_n;
  return S.trust[(ca[0] * n + ca[1]) * n + ca[2]] && S.trust[(cb[0] * n + cb[1]) * n + cb[2]];
}

// 10^y in FP64 from an FP32 exponent (kernels reach 1e-90, below FP32).
__device__ __forceinline__ double exp10_wide(float y) {
  const double t = (double)y * 3.3219280948873623479;   // log2(10)
  const double n = floor(t);
  return ldexp((double)exp2f((float)(t - n)), (int)n);
}

// Rates of a ray from the network: Gamma_s = r_s d_s q <F_s>, Heat_s =
// r_s d_s q <G_s> hplanck nu_L, with <.> the 2-point mean over the in-cell
// path (the photon-conserving cell average of exp(-tau)).
__device__ inline void surr_rates(const RayRate& rr, double q, const float ya[kNout],
                                  const float yb[kNout], double res[6]) {
  double m[kNout];
#pragma unroll
  for (int o = 0; o < kNout; o++) m[o] = 0.5 * (exp10_wide(ya[o]) + exp10_wide(yb[o]));
  const double p0 = rr.d[0] / rr.v[0] * q, p1 = rr.d[1] / rr.v[1] * q, p2 = rr.d[2] / rr.v[2] * q;
  res[0] = p0 * m[0];
  res[1] = p0 * m[3] * kHnuL;
  res[2] = p1 * m[1];
  res[3] = p2 * m[2];
  res[4] = p1 * m[4] * kHnuL;
  res[5] = p2 * m[5] * kHnuL;
}

template <bool KAHAN, bool CAPTURE, bool SURR, bool NARROW, bool POW2, bool FLOAT>
__global__ __launch_bounds__(64) ARGOT_OCCUPANCY void fused_step_kernel(FusedArgs a) {
  const GridDev& g = a.grid;
  const TreeDev& tr = a.tree;
  const RateTables& rt = a.rates;
  const int lane = threadIdx.x;
  const int bx = a.tile_bits[0], by = a.tile_bits[1], bz = a.tile_bits[2];
  const int TX = 1 << bx, TY = 1 << by, TZ = 1 << bz;
  const int ntx = (g.nx + TX - 1) / TX, nty = (g.ny + TY - 1) / TY, ntz = (g.nz + TZ - 1) / TZ;
  const int64_t ntile = (int64_t)ntx * nty * ntz;
  // Tiles are handed out in Morton (Z-curve) order over the smallest
  // power-of-two cube of tiles that holds the mesh, whose places outside
  // the mesh are skipped: each XCD's queue is then an octant of that cube,
  // and the wavefronts running at one time on an XCD hold a compact block
  // of targets whose rays cross the same cells, so that more of their
  // gathers hit the XCD's L2 (1.08x on the 256^3 / 4096-source step).
  // A mesh whose cube would be more than 8 times its tile count keeps the
  // linear order.
  int mbits = 0;
  while ((1 << mbits) < max(ntx, max(nty, ntz))) mbits++;
  const int64_t ncube = (int64_t)1 << (3 * mbits);
  const bool morton = mbits <= 10 && ncube <= 8 * ntile;
  const int64_t nqueue_tiles = morton ? ncube : ntile;
  int q = blockIdx.x % kNumQueues, tried = 0;
  // Each lane's counts: rays, crossings, FP64 fallbacks and, the same in every
  // lane, visits and visits with a ray (over a launch they fit in 32 bits).  They
  // are in LDS, where adding to them takes no register: as variables they were
  // spilled, and read and written back at every visit through the texture path,
  // which bounds the kernel (16 cycles of it an 8-B access; with 64-bit visits 3%
  // of the launch).  (The surrogate variant has no room for the visits' in LDS.)
  constexpr int kCounts = SURR ? 3 : 5;
  __shared__ unsigned int count_lds[kCounts][64];
  unsigned int my_surr = 0, my_visit = 0, my_emit_iter = 0;
  const auto count = [&](int i, unsigned int by) {
    (void)__hip_atomic_fetch_add(&count_lds[i][lane], by, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_WAVEFRONT);
  };
#pragma unroll
  for (int i = 0; i < kCounts; i++) count_lds[i][lane] = 0u;
  // The targets' per-cell FP64 sums, centres, and densities and fractions live
  // in LDS between rays, by the target's place in the tile: the walk and the
  // frequency loop have the registers to themselves, and a ray can be worked
  // by any lane.
  __shared__ double acc_lds[6][64];
  // (the surrogate variant passes centres between lanes and reads the
  // target's fields from the mesh at each ray instead, so that with the
  // network's LDS it still fits 16 wavefronts per CU)
  __shared__ float4 tgt_lds[SURR ? 1 : 64];
  __shared__ float4 cell_lds[SURR ? 1 : 64];
  float* lds = nullptr;
  if constexpr (SURR) {
    __shared__ float surr_lds[kMlpLds];
    lds = surr_lds;
  }

  for (;;) {
    const int64_t t = next_tile(a.ctr, nqueue_tiles, &q, &tried);
    if (t < 0) break;
    int tx, ty, tz;
    if (morton) {
      tx = (int)compact3((uint32_t)t >> 2);
      ty = (int)compact3((uint32_t)t >> 1);
      tz = (int)compact3((uint32_t)t);
      if (tx >= ntx || ty >= nty || tz >= ntz) continue;   // outside the mesh
    } else {
      tz = (int)(t % ntz);
      ty = (int)((t / ntz) % nty);
      tx = (int)(t / ((int64_t)ntz * nty));
    }
    // The lane's own target: it follows the tree for it and adds its sums to
    // the mesh at the end.
    const int ix = tx * TX + ((lane >> (by + bz)) & (TX - 1));
    const int iy = ty * TY + ((lane >> bz) & (TY - 1));
    const int iz = tz * TZ + (lane & (TZ - 1));
    const bool valid = ix < g.nx && iy < g.ny && iz < g.nz;
    const int64_t cell = (int64_t)iz + (int64_t)g.nz * ((int64_t)iy + (int64_t)g.ny * ix);
    float4 mine;
    {
      float4 f = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (valid)
        f = make_float4(*mesh_f(a.mesh, cell, kOffDens), *mesh_f(a.mesh, cell, kOffFHI),
                        *mesh_f(a.mesh, cell, kOffFHeI), *mesh_f(a.mesh, cell, kOffFHeII));
      mine = make_float4(cell_centre(g.gxmin, ix + g.ox, g.dx),
                         cell_centre(g.gymin, iy + g.oy, g.dy),
                         cell_centre(g.gzmin, iz + g.oz, g.dz), 0.0f);
      if constexpr (!SURR) {
        cell_lds[lane] = f;
        tgt_lds[lane] = mine;
      }
#pragma unroll
      for (int k = 0; k < 6; k++) acc_lds[k][lane] = 0.0;
    }
    wave_sync();
    const auto centre_of = [&](int t) {
      if constexpr (SURR)
        return make_float4(__shfl(mine.x, t, 64), __shfl(mine.y, t, 64), __shfl(mine.z, t, 64),
                           0.0f);
      else
        return tgt_lds[t];
    };
    // A place in the tile, to pick the axis that rays from a node run along.
    const float4 far = centre_of(63);
    const auto target_cell = [&](int t) {
      const int jx = tx * TX + (t >> (by + bz)), jy = ty * TY + ((t >> bz) & (TY - 1)),
                jz = tz * TZ + (t & (TZ - 1));
      return (int64_t)jz + (int64_t)g.nz * ((int64_t)jy + (int64_t)g.ny * jx);
    };
    int p = valid ? 0 : tr.nnode;
    int seq = 0;
    for (;;) {
      const int u = wave_min(p);
      if (u >= tr.nnode) break;
      const float cx = tr.node_cm[4 * u + 0], cy = tr.node_cm[4 * u + 1],
                  cz = tr.node_cm[4 * u + 2], len2 = tr.node_cm[4 * u + 3];
      const NodeLink ln = tr.link[u];
      const bool here = (p == u);
      // setup_light_ray_to (setup_light_ray_tree.c:346-354), FP32
      const float4 own = SURR ? mine : tgt_lds[lane];
      const float ddx = own.x - cx, ddy = own.y - cy, ddz = own.z - cz;
      const float r2 = ddx * ddx + ddy * ddy + ddz * ddz;
      const bool accept = r2 * g.theta_sq > len2;
      const bool leaf = ln.n <= 1;
      const bool emit = here && (accept || ln.n == 1);
      if (here) p = (accept || leaf || ln.first < 0) ? ln.skip : ln.first;
      if constexpr (SURR)
        my_visit++;
      else
        count(3, 1u);
      const unsigned long long emitting = __ballot(emit);
      if (emitting == 0) continue;
      if constexpr (SURR)
        my_emit_iter++;
      else
        count(4, 1u);
      // Which target's ray each lane works: targets that follow one another
      // along the axis the rays run along mostly (from the node to the tile)
      // go to neighbouring lanes.  Their rays share most of their cells, and
      // the vector memory path serves a 12-B gather four neighbouring lanes at
      // a time, a cycle for each cache line the four touch: 24.6 lines a gather
      // instead of 28.2 with lanes in mesh order (counted on 256^3 and 4096
      // clumped sources; 1.5% of the time: issue bounds the kernel as much).  Bricks of
      // 2 x 2 x 2 cells would touch a few less, but their alternating strides cost
      // registers, and what they spilled cost 30%.
      const float ax = fabsf(far.x - cx), ay = fabsf(far.y - cy), az = fabsf(far.z - cz);
      int t = lane;
      if (ax > ay && ax > az)
        t = ((lane & (TX - 1)) << (by + bz)) | (lane >> bx);
      else if (ay > az)
        t = ((lane >> (by + bz)) << (by + bz)) | ((lane & (TY - 1)) << bz) |
            ((lane >> by) & (TZ - 1));
      const bool work = (emitting >> t) & 1ull;
      const bool node = (__ballot(accept) >> t) & 1ull;   // the ray comes from the node's centre
      const float4 tc = centre_of(t);
      const Vec3f tgt{tc.x, tc.y, tc.z};
      Vec3f src{0.0f, 0.0f, 0.0f}, st{0.0f, 0.0f, 0.0f};
      WalkOut w{};
      RayRate rr;      // (of working lanes; no other lane's is used)
      double res[6];
      if (work) {
        if (node) {
          src = Vec3f{cx, cy, cz};
        } else {
          src = Vec3f{tr.src_pos[4 * ln.src + 0], tr.src_pos[4 * ln.src + 1],
                      tr.src_pos[4 * ln.src + 2]};
        }
        // a ray the reference refuses (calc_ray_segment.c:212) is counted
        // where it happens, on the path of sources outside the box
        segment_start(g, src, tgt, &st, &a.ctr->noverflow);
        const Vec3f d{tgt.x - src.x, tgt.y - src.y, tgt.z - src.z};
        RayDir along = ray_dir(d.x, d.y, d.z);
        // (formed here, so that two numbers are kept through the walk)
        const Chord chord = ray_chord(g, along, d.x, d.y, d.z);
        // from the segment's start: the source, if inside the box
        if (st.x != src.x || st.y != src.y || st.z != src.z)
          along = ray_dir(tgt.x - st.x, tgt.y - st.y, tgt.z - st.z);
        walk_segment<KAHAN, CAPTURE, NARROW, POW2, FLOAT>(g, a.nf, along, st, tgt, box_passes(g),
                                                          &w);
        float4 f;
        if constexpr (SURR) {
          const int64_t tcell = target_cell(t);
          f = make_float4(*mesh_f(a.mesh, tcell, kOffDens), *mesh_f(a.mesh, tcell, kOffFHI),
                          *mesh_f(a.mesh, tcell, kOffFHeI), *mesh_f(a.mesh, tcell, kOffFHeII));
        } else {
          f = cell_lds[t];
        }
        ray_rate_setup(g, chord, w.tau, f.x, f.y, f.z, f.w, &rr);
      }
      bool exact = work;
      if constexpr (SURR) {
        // The network runs on the whole wavefront (MFMA) and serves the
        // visit only when every emitting lane can use it; otherwise every
        // lane takes the exact integral below: a visit that ran both would
        // pay for both.
        const double qn = a.surr.node_q[u];
        float xa[3] = {0.0f, 0.0f, 0.0f}, xb[3] = {0.0f, 0.0f, 0.0f};
        const bool use = work && surr_inputs(a.surr, rt, rr, qn, xa, xb);
        if (__ballot(use) == __ballot(work)) {
          float ya[kNout], yb[kNout];
          mlp_forward(a.surr.net, xa[0], xa[1], xa[2], ya, lds);
          mlp_forward(a.surr.net, xb[0], xb[1], xb[2], yb, lds);
          if (use) {
            surr_rates(rr, qn, ya, yb, res);
            exact = false;
            my_surr++;
          }
        }
      }
      const float* sp = tr.spec + (int64_t)u * rt.ngrid;
      const double sc = ldc(tr.spec_scale + u);
      const bool wide = exact && !fast_rate_ok(rt, rr);   // FP32 cannot serve this ray
      // the node spectrum as spec * spec_scale (within 6e-8 of the double
      // sums; this loop serves the rays FP32 cannot).  It comes first, so that
      // the ray's FP64 quantities need not outlive the FP32 loop.
      rate_f64_wave(rt, rr, wide, [&](int, int k) { return (double)sp[k] * sc; }, res);
      if (wide) count(2, 1u);
      if (exact && !wide) {
        const F4* wt = reinterpret_cast<const F4*>(tr.weight + (int64_t)u * kRuleWeights);
        rate_loop_f32(rt, rr, sc, ldc(reinterpret_cast<const F4*>(tr.limit) + u),
                      [&](int k) { return ldc(sp + k); },
                      [&](int i) { return ldc(wt + i); }, res);
      }
      const int nth = CAPTURE ? __shfl(seq, t, 64) : 0;
      if (work) {
#pragma unroll
        for (int k = 0; k < 6; k++) acc_lds[k][t] += res[k];
        count(0, 1u);
        count(1, (unsigned int)w.ncross);
        if (CAPTURE) {
          const unsigned long long slot = atomicAdd(&a.ctr->nrecord, 1ull);
          if (slot < (unsigned long long)a.rec_cap) {
            RayRecord& R = a.rec[slot];
            R.target = target_cell(t);
            R.seq = nth;
            R.kind = node ? 0 : 1;
            R.id = node ? u : ln.src;
            R.ncross = w.ncross;
            R.start[0] = st.x; R.start[1] = st.y; R.start[2] = st.z;
            R.src[0] = src.x; R.src[1] = src.y; R.src[2] = src.z;
            R.tau[0] = w.tau[0]; R.tau[1] = w.tau[1]; R.tau[2] = w.tau[2];
            R.surrogate = exact ? 0.0f : 1.0f;
            R.hash = w.hash;
            for (int k = 0; k < 6; k++) R.rate[k] = res[k];
          }
        }
      }
      if (CAPTURE && emit) seq++;
      wave_sync();   // the sums of this visit before another lane's
    }
    if (valid) {
      float* r = mesh_fw(a.mesh, cell, kOffRates);
#pragma unroll
      for (int k = 0; k < 6; k++) r[k] = (float)((double)r[k] + acc_lds[k][lane]);
    }
  }
  if constexpr (!SURR) {
    my_visit = count_lds[3][lane];
    my_emit_iter = count_lds[4][lane];
  }
  const unsigned long long sr = wave_sum((unsigned long long)count_lds[0][lane]),
                           sc = wave_sum((unsigned long long)count_lds[1][lane]),
                           sf = wave_sum((unsigned long long)count_lds[2][lane]),
                           ss = wave_sum((unsigned long long)my_surr);
  if (lane == 0 && my_visit) {
    StepCounters::Queue& c = a.ctr->queue[blockIdx.x % kNumQueues];
    atomicAdd(&c.nray, sr);
    atomicAdd(&c.ncross, sc);
    if (sf) atomicAdd(&c.nfallback, sf);
    if (SURR && ss) atomicAdd(&c.nsurrogate, ss);
    atomicAdd(&c.nvisit, (unsigned long long)my_visit);
    atomicAdd(&c.nemit_iter, (unsigned long long)my_emit_iter);
  }
}

// smooth_photoion_rate (smooth_photoion_rate.c:1058-1090) on one rank.
// The six prev_chem rates go to SoA planes; each plane is smoothed by the
// 27-point stencil (central weight 30, 1/56; ghost cells are the nearest
// interior cell) and the results go straight back into prev_chem.  The floor is
// passing over the records twice, whose rates lie in nearly every one of the
// mesh's cache lines.  128^3: 65 us for the gather (5 TB/s) and 77 for the
// rest, against 65 + 90 + 69 with a scatter pass of its own and a thread per
// plane and cell.
__global__ void gather_rates_kernel(const unsigned char* __restrict__ mesh, int64_t ncell,
                                    float* __restrict__ soa) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  const float* r = mesh_f(mesh, c, kOffRates);
#pragma unroll
  for (int k = 0; k < 6; k++) soa[k * ncell + c] = r[k];
}

// Blocks of consecutive (y, z) cells; a thread takes kSmoothX cells along x,
// whose stencils share rows (108 loads a cell instead of 162).  A call on 128^3
// cells takes 150, 144 and 146 us with 1, 2 and 4 cells a thread, on 16^3 20,
// 20 and 22, where 4 are too long a chain.
// out: the smoothed planes too, when the caller wants them (else null).
constexpr int kSmoothX = 2;
__global__ __launch_bounds__(256) void smooth_rates_kernel(int nx, int ny, int nz, int x0,
                                                           const float* __restrict__ in,
                                                           unsigned char* __restrict__ mesh,
                                                           float* __restrict__ out) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  const int iy = (int)(i / (unsigned)nz), iz = (int)(i % (unsigned)nz);
  const int ix = x0 + (int)blockIdx.y * kSmoothX;
  if (iy >= ny) return;
  const int64_t plane = (int64_t)ny * nz, ncell = plane * nx;
  int64_t place[9];   // (iy + dy, iz + dz) in a plane, ghosts clamped
#pragma unroll
  for (int q = 0; q < 9; q++) {
    const int jy = min(max(iy + q / 3 - 1, 0), ny - 1), jz = min(max(iz + q % 3 - 1, 0), nz - 1);
    place[q] = (int64_t)jy * nz + jz;
  }
  float smoothed[6][kSmoothX];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    const float* p = in + (int64_t)k * ncell;
    float v[kSmoothX + 2][9];
#pragma unroll
    for (int x = 0; x < kSmoothX + 2; x++)
#pragma unroll
      for (int q = 0; q < 9; q++)
        v[x][q] = p[(int64_t)min(max(ix + x - 1, 0), nx - 1) * plane + place[q]];
#pragma unroll
    for (int x = 0; x < kSmoothX; x++) {
      // C evaluation order of the reference's sum: thirteen float additions,
      // then the double central term, then double additions
      float s = v[x][0];
#pragma unroll
      for (int term = 1; term < 13; term++) s = s + v[x + term / 9][term % 9];
      double d = (double)s + 30.0 * (double)v[x + 1][4];
#pragma unroll
      for (int term = 14; term < 27; term++) d = d + (double)v[x + term / 9][term % 9];
      smoothed[k][x] = (float)((1.0 / (30.0 + 26.0)) * d);
    }
  }
  // a record's stores side by side: spread over the six planes they miss one
  // another in the cache
#pragma unroll
  for (int x = 0; x < kSmoothX; x++) {
    if (ix + x >= nx) break;
    const int64_t c = (int64_t)(ix + x) * plane + place[4];
    float* const r = mesh_fw(mesh, c, kOffRates);
#pragma unroll
    for (int k = 0; k < 6; k++) r[k] = smoothed[k][x];
    if (out)
#pragma unroll
      for (int k = 0; k < 6; k++) out[(int64_t)k * ncell + c] = smoothed[k][x];
  }
}

hipError_t launch_smooth_rates(void* mesh, int nx, int ny, int nz, float* tmp_in, float* tmp_out,
                               hipStream_t s) {
  const int64_t ncell = (int64_t)nx * ny * nz;
  gather_rates_kernel<<<(unsigned)((ncell + 255) / 256), 256, 0, s>>>(
      static_cast<const unsigned char*>(mesh), ncell, tmp_in);
  // a plane's cells number below 2^31: the mesh of 2^31 cells would not fit the device
  const unsigned blocks = (unsigned)(((int64_t)ny * nz + 255) / 256);
  constexpr int most = 65535 * kSmoothX;   // (the grid's second extent)
  for (int x0 = 0; x0 < nx; x0 += most)
    smooth_rates_kernel<<<dim3(blocks, (unsigned)((std::min(nx - x0, most) + kSmoothX - 1) / kSmoothX)),
                          256, 0, s>>>(nx, ny, nz, x0, tmp_in,
                                       static_cast<unsigned char*>(mesh), tmp_out);
  return hipGetLastError();
}

// Plain device-to-device copy (16 B per thread per iteration, grid-stride):
// the bandwidth probe whose byte count calibrates the HBM counters.
__global__ void copy_probe_kernel(const float4* __restrict__ src, float4* __restrict__ dst,
                                  int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    dst[i] = src[i];
}

hipError_t launch_copy_probe(const float4* src, float4* dst, int64_t n, int nblock,
                             hipStream_t s) {
  copy_probe_kernel<<<nblock, 256, 0, s>>>(src, dst, n);
  return hipGetLastError();
}

// ------------------------------------------------------------------------
// Launch wrappers (host side).

static inline unsigned nblocks(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

hipError_t launch_pack_fields(const void* mesh, int64_t ncell, double helium_fact, float4* nf,
                              hipStream_t s) {
  pack_fields_kernel<<<nblocks(ncell, 256), 256, 0, s>>>(
      static_cast<const unsigned char*>(mesh), ncell, helium_fact, nf);
  return hipGetLastError();
}

hipError_t launch_zero_rates(void* mesh, int64_t ncell, hipStream_t s) {
  zero_rates_kernel<<<nblocks(ncell, 256), 256, 0, s>>>(static_cast<unsigned char*>(mesh), ncell);
  return hipGetLastError();
}

hipError_t launch_begin_step(void* mesh, int64_t ncell, double helium_fact, float4* nf,
                             StepCounters* ctr, hipStream_t s) {
  static_assert(kNumQueues <= 256, "one block clears the queues");
  begin_step_kernel<<<nblocks(ncell, 256), 256, 0, s>>>(static_cast<unsigned char*>(mesh), ncell,
                                                        helium_fact, nf, ctr);
  return hipGetLastError();
}

hipError_t launch_add_rates(void* mesh, const float* rate, int64_t ncell, hipStream_t s) {
  add_rates_kernel<<<nblocks(ncell, 256), 256, 0, s>>>(static_cast<unsigned char*>(mesh), rate,
                                                        ncell);
  return hipGetLastError();
}

// Can the walk keep face positions instead of face counters?  Every cell
// size must be a power of two (then an integer face counter below 2^24
// times it is exact) and every mesh size below 2^23 (so that n + 1/2 is
// exact too).
static bool pow2_cells(const GridDev& g) {
  const float d[3] = {g.dx, g.dy, g.dz};
  const int n[3] = {g.nx, g.ny, g.nz};
  for (int k = 0; k < 3; k++) {
    int e = 0;
    if (!(d[k] >= FLT_MIN) || !(d[k] <= 1.0e30f) || std::frexp(d[k], &e) != 0.5f) return false;
    if (n[k] < 1 || n[k] >= (1 << 23)) return false;
  }
  return true;
}

// How the walk takes a mesh: its float form up to 2^24 cells (byte offsets of
// 16-B records are exact in FP32 up to there) where the cell sizes leave its
// FP32 quotients room, 32-bit offsets below 2^28 cells, and 64-bit addresses
// and face counters otherwise (and always when wide is set).
enum class WalkForm { kFloat, kNarrow, kWide };
static WalkForm walk_form(const GridDev& g, int wide) {
  const int64_t ncell = (int64_t)g.nx * g.ny * g.nz;
  if (wide || ncell >= kNarrowCells) return WalkForm::kWide;
  for (float h : {g.dx, g.dy, g.dz})
    if (!(h > 1.0e-12f && h < 1.0e6f)) return WalkForm::kNarrow;
  return ncell <= kFloatCells ? WalkForm::kFloat : WalkForm::kNarrow;
}

template <typename Walk>
static void launch_walk(const GridDev& g, const Walk& w, void* seg, int64_t nseg, int kahan,
                        hipStream_t s) {
  walk_segments_kernel<<<nblocks(nseg, kWalkBlock), kWalkBlock, 0, s>>>(
      g, w, static_cast<unsigned char*>(seg), nseg, kahan);
}

hipError_t launch_walk_segments(const GridDev& g, const float4* nf, void* seg, int64_t nseg,
                                int kahan, int wide, hipStream_t s) {
  if (nseg <= 0) return hipSuccess;
  const bool pow2 = pow2_cells(g);
  switch (walk_form(g, wide)) {
    case WalkForm::kFloat:
      if (pow2)
        launch_walk(g, WalkPacked<true, true, true>{nf}, seg, nseg, kahan, s);
      else
        launch_walk(g, WalkPacked<true, false, true>{nf}, seg, nseg, kahan, s);
      break;
    case WalkForm::kNarrow:
      if (pow2)
        launch_walk(g, WalkPacked<true, true, false>{nf}, seg, nseg, kahan, s);
      else
        launch_walk(g, WalkPacked<true, false, false>{nf}, seg, nseg, kahan, s);
      break;
    case WalkForm::kWide:
      launch_walk(g, WalkPacked<false, false, false>{nf}, seg, nseg, kahan, s);
  }
  return hipGetLastError();
}

hipError_t launch_walk_segments_mesh(const GridDev& g, const void* mesh, double helium_fact,
                                     void* seg, int64_t nseg, int kahan, hipStream_t s) {
  if (nseg <= 0) return hipSuccess;
  const MeshFields f{static_cast<const unsigned char*>(mesh), helium_fact};
  if (pow2_cells(g))
    launch_walk(g, WalkMesh<true>{f}, seg, nseg, kahan, s);
  else
    launch_walk(g, WalkMesh<false>{f}, seg, nseg, kahan, s);
  return hipGetLastError();
}

hipError_t launch_target_rates(const GridDev& g, const RateTables& rt, void* mesh,
                              const CallTarget* tg, int64_t ntarget, const CallRay* rays,
                              const CallSpectra& sp, hipStream_t s) {
  if (ntarget <= 0) return hipSuccess;
  target_rates_kernel<<<nblocks(ntarget, 64), 64, 0, s>>>(
      g, rt, static_cast<unsigned char*>(mesh), tg, ntarget, rays, sp);
  return hipGetLastError();
}

// 16 spectra to a block where that still gives every CU a block; few spectra
// spread out, 4 to a block, so that the launch is short.
hipError_t launch_project_spectra(const RuleDev& rule, const float* spec, int nspec, int ngrid,
                                  float* weight, float* limit, hipStream_t s) {
  if (nspec <= 0) return hipSuccess;
  if (nspec >= 16 * 256)
    project_spectra_kernel<16><<<nblocks(nspec, 16), kProjectThreads, 0, s>>>(
        rule, spec, nspec, ngrid, weight, limit);
  else
    project_spectra_kernel<4><<<nblocks(nspec, 4), kProjectThreads, 0, s>>>(
        rule, spec, nspec, ngrid, weight, limit);
  return hipGetLastError();
}

hipError_t launch_get_rates(const void* mesh, float* rate, int64_t ncell, hipStream_t s) {
  if (ncell <= 0) return hipSuccess;
  get_rates_kernel<<<nblocks(ncell, 256), 256, 0, s>>>(static_cast<const unsigned char*>(mesh),
                                                      ncell, rate);
  return hipGetLastError();
}

hipError_t launch_set_rates(void* mesh, const float* rate, int64_t ncell, hipStream_t s) {
  if (ncell <= 0) return hipSuccess;
  set_rates_kernel<<<nblocks(ncell, 256), 256, 0, s>>>(static_cast<unsigned char*>(mesh), rate,
                                                      ncell);
  return hipGetLastError();
}

template <bool SURR, bool NARROW, bool POW2, bool FLOAT>
static void launch_fused(const FusedArgs& a, int kahan, int capture, int nblock, hipStream_t s) {
  if (capture) {
    if (kahan)
      fused_step_kernel<true, true, SURR, NARROW, POW2, FLOAT><<<nblock, 64, 0, s>>>(a);
    else
      fused_step_kernel<false, true, SURR, NARROW, POW2, FLOAT><<<nblock, 64, 0, s>>>(a);
  } else {
    if (kahan)
      fused_step_kernel<true, false, SURR, NARROW, POW2, FLOAT><<<nblock, 64, 0, s>>>(a);
    else
      fused_step_kernel<false, false, SURR, NARROW, POW2, FLOAT><<<nblock, 64, 0, s>>>(a);
  }
}

template <bool SURR>
static void launch_fused_form(const FusedArgs& a, int kahan, int capture, int wide, int nblock,
                              hipStream_t s) {
  const bool pow2 = pow2_cells(a.grid);
  switch (walk_form(a.grid, wide)) {
    case WalkForm::kFloat:
      if (pow2)
        launch_fused<SURR, true, true, true>(a, kahan, capture, nblock, s);
      else
        launch_fused<SURR, true, false, true>(a, kahan, capture, nblock, s);
      break;
    case WalkForm::kNarrow:
      if (pow2)
        launch_fused<SURR, true, true, false>(a, kahan, capture, nblock, s);
      else
        launch_fused<SURR, true, false, false>(a, kahan, capture, nblock, s);
      break;
    case WalkForm::kWide:
      launch_fused<SURR, false, false, false>(a, kahan, capture, nblock, s);
  }
}

// nblock: the persistent grid; a mesh of fewer tiles gets a block per tile
// (one wavefront each), since any more would only look for work.
hipError_t launch_fused_step(const FusedArgs& a, int kahan, int capture, int surr, int wide,
                             int nblock, hipStream_t s) {
  int64_t ntile = 1;
  const int n[3] = {a.grid.nx, a.grid.ny, a.grid.nz};
  for (int d = 0; d < 3; d++)
    ntile *= (n[d] + (1 << a.tile_bits[d]) - 1) >> a.tile_bits[d];
  nblock = (int)std::min<int64_t>(nblock, std::max<int64_t>(ntile, 1));
  if (surr)
    launch_fused_form<true>(a, kahan, capture, wide, nblock, s);
  else
    launch_fused_form<false>(a, kahan, capture, wide, nblock, s);
  return hipGetLastError();
}

}  // namespace argot
