// ART diffuse-photon transfer on one MI355X (one rank): parallel rays for
// every HEALPix direction sweep the box, carrying three band intensities
// through the cells (emission and absorption per crossing), and the
// per-cell band intensities and path lengths become photoionization and
// heating rates, averaged over directions.
//
// Reference: src/diffuse_photon/ (calc_diffuse_photon_radiation.c:38-120,
// ray_tracing.c:60-394, calc_rmesh_data.c:37-117, calc_GH_tot.c:171-246,
// set_angle.c, set_start_pos.c, set_step_func_factor.c), with __HELIUM__
// on, __HELIUM_BB__ off and __USE_ATOMIC__ off.
//
// GPU layout: directions run in batches; each direction of a batch owns a
// float4 accumulator slice {length, I1, I2, I3} over the mesh.  Within a ray
// group no two rays touch the same cell (their start points are two cells
// apart and a ray moves at most one cell sideways per layer of its dominant
// axis), so the accumulators need no atomics and the sums keep the reference's
// group order.  A block sweeps one direction's rays through the box layer by
// layer with the layer's accumulators in LDS (art_sweep_kernel); where its
// bounds do not hold, a launch per ray group adds to the slices in memory
// (art_trace_kernel).  Per-cell rates then accumulate over the batch's
// directions in the reference's (sorted) direction order.
#include <hip/hip_runtime.h>
#include <math.h>
#include <string.h>

#include <algorithm>
#include <chrono>
#include <vector>

#include "argot_device.h"
#include "argot_hip.h"
#include "surrogate.h"

namespace argot {
namespace {

constexpr double kTinyArt = 1.0e-31;
constexpr double kPiArt = 3.1415926535897932384626433;   // constants.h:22
constexpr double kHplanck = 6.626e-27;                   // constants.h:16
constexpr double kKtoeV = 8.61623e-5;                    // chemistry.h:10
constexpr double kEVtoErg = 1.6022e-12;                  // chemistry.h:12
constexpr double kNuLeV = 13.6;                          // chemistry.h:15
constexpr double kXH = 0.755, kYHe = 0.245;              // chemistry.h:23-24

// diffuse_photon.h:48-75 (band cross-section and integral ratios)
constexpr double kRcHI2 = 1.9529766579e-01, kRcHI3 = 1.9513732355e-02;
constexpr double kRcHeI3 = 2.6858709594e-01;
constexpr double kRjHI2 = 1.128855608262e-01, kRjHI3 = 5.288790581895e-03;
constexpr double kRjHeI3 = 1.2404369898e-01;
constexpr double kRhHI2 = 3.1154224364e+00, kRhHI3 = 5.2452188546e-01;
constexpr double kRhHeI3 = 8.7872474963e+00;

// fluid_mesh offsets (156 B): dens @0, prev_chem @96 {wmol, felec, fHI,
// fHII, fHeI, fHeII, fHeIII, GammaHI, HeatHI, GammaHeI, GammaHeII, HeatHeI,
// HeatHeII}, prev_uene @148.
constexpr int kStride = 156;
constexpr int kPrevChem = 96;
constexpr int kPrevUene = 148;

struct ArtDir {
  float ovr[3];
  int base;
  double rcp[3];   // 1 / (double)ovr: exact FP32 quotient dx/ovr via div_by
  float rcpf[3];   // 1 / ovr in FP32: the same quotient via div_exact
  int order;       // the batch's direction that this place of the launch sweeps
};

// A cell's absorption coefficients and source functions (3 bands).
struct ArtMedium {
  float k0, k1, k2, s0, s1, s2;
};

struct ArtGrid {
  int nx, ny, nz;
  int64_t ncell;
  float xmin, ymin, zmin, xmax, ymax, zmax, dx, dy, dz;
  double lunit;
};

// ----------------------------------------------------------------------
// Position of index i along an axis of even length n with the even indices
// first: the rays of one group start two cells apart across the entry face,
// so with this order neighbouring lanes touch neighbouring records.
__device__ __forceinline__ int art_split(int i, int n) { return (i & 1) * (n >> 1) + (i >> 1); }

// Cell index of the layout a direction's slices use: z fastest (split) for
// directions whose dominant axis is x or y; y fastest (split) for z-dominant
// ones (base 0, 1), whose neighbouring rays are two cells apart in y.
__device__ __forceinline__ int64_t art_index(bool zdom, int nx, int ny, int nz, int ix, int iy,
                                             int iz) {
  return zdom ? (int64_t)art_split(iy, ny) + (int64_t)ny * ((int64_t)ix + (int64_t)nx * iz)
              : (int64_t)art_split(iz, nz) + (int64_t)nz * ((int64_t)iy + (int64_t)ny * ix);
}


// Per-cell absorption and source function (calc_rmesh_data.c:37-117).

__device__ inline double k02_A(double t) {
  const double l1 = log(t * kKtoeV), l2 = l1 * l1, l3 = l2 * l1, l4 = l3 * l1, l5 = l4 * l1,
               l6 = l5 * l1, l7 = l6 * l1, l8 = l7 * l1, l9 = l8 * l1;
  return exp(-28.61303380689232 - 0.7241125657826851 * l1 - 0.02026044731984691 * l2 -
             0.002380861877349834 * l3 - 0.0003212605213188796 * l4 -
             0.00001421502914054107 * l5 + 4.989108920299513e-6 * l6 +
             5.755614137575758e-7 * l7 - 1.856767039775261e-8 * l8 -
             3.071135243196595e-9 * l9);
}
__device__ inline double k02_B(double t) {
  const double lambda = 2.0 * 157807.0 / t;
  return 2.753e-14 * pow(lambda, 1.5) / pow(1.0 + pow(lambda / 2.740, 0.407), 2.242);
}
__device__ inline double k04_A(double t) {
  const double tev = t * kKtoeV;
  if (tev > 0.8)
    return 1.54e-9 * (1. + 0.3 / exp(8.099328789667 / tev)) /
               (exp(40.49664394833662 / tev) * pow(tev, 1.5)) +
           3.92e-13 / pow(tev, 0.6353);
  return 3.92e-13 / pow(tev, 0.6353);
}
__device__ inline double k04_B(double t) {
  if (t > 500.3) return 1.26e-14 * pow(2.0 * 285335.0 / t, 0.75);
  return (1.12e-10 - 2.1e-11 * log10(t)) / sqrt(t);
}
__device__ inline double k06_A(double t) {
  return 3.36e-10 / sqrt(t) / pow((t / 1.e3), 0.2) / (1.0 + pow((t / 1.e6), 0.7));
}
__device__ inline double k06_B(double t) {
  const double lambda = 2.0 * 631515.0 / t;
  return 1.3765e-14 * pow(lambda, 1.5) / pow(1.0 + pow(lambda / 2.740, 0.407), 2.242);
}

__global__ void art_rmesh_kernel(const unsigned char* __restrict__ mesh, int nx, int ny, int nz,
                                 double denstonh, double uenetok, double helium_fact,
                                 float csHI, float csHeI, float csHeII,
                                 ArtMedium* __restrict__ med, ArtMedium* __restrict__ medT) {
  const int64_t ncell = (int64_t)nx * ny * nz;
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  const unsigned char* m = mesh + c * kStride;
  const float* ch = reinterpret_cast<const float*>(m + kPrevChem);
  const float dens = *reinterpret_cast<const float*>(m);
  const float uene = *reinterpret_cast<const float*>(m + kPrevUene);
  const float wmol = (float)(1.0 / ((1.0 + ch[1]) * kXH + 0.25 * kYHe));
  float temper = (float)((double)uene * uenetok * (double)wmol);
  if (temper < 1.0f) temper = 1.0f;
  const double nH = (double)dens * denstonh;
  const double nHI = (double)ch[2] * nH, nHII = (double)ch[3] * nH;
  double ne = nHII;
  const double nHeI = (double)ch[4] * helium_fact * nH;
  const double nHeII = (double)ch[5] * helium_fact * nH;
  const double nHeIII = (double)ch[6] * helium_fact * nH;
  ne += nHeII + 2.0e0 * nHeIII;
  const double aHI = (double)csHI * nHI;
  const double aHeI = (double)csHeI * nHeI, aHeII = (double)csHeII * nHeII;
  ArtMedium r;
  r.k0 = (float)(aHI + kTinyArt);
  r.k1 = (float)(aHI * kRcHI2 + aHeI + kTinyArt);
  r.k2 = (float)(aHI * kRcHI3 + aHeI * kRcHeI3 + aHeII + kTinyArt);
  const double t = temper;
  r.s0 = (float)((k02_A(t) - k02_B(t)) * ne * nHII * kNuLeV * 1.0 * kEVtoErg / (4.0 * kPiArt) /
                (double)r.k0);
  r.s1 = (float)((k04_A(t) - k04_B(t)) * ne * nHeII * kNuLeV * 1.8125 * kEVtoErg /
                (4.0 * kPiArt) / (double)r.k1);
  r.s2 = (float)((k06_A(t) - k06_B(t)) * ne * nHeIII * kNuLeV * 4.0 * kEVtoErg / (4.0 * kPiArt) /
                (double)r.k2);
  // the record in both trace layouts
  const int ix = (int)(c / ((int64_t)ny * nz));
  const int iy = (int)((c / nz) % ny);
  const int iz = (int)(c % nz);
  const int64_t cm = art_index(false, nx, ny, nz, ix, iy, iz);
  const int64_t cT = art_index(true, nx, ny, nz, ix, iy, iz);
  med[cm] = r;
  medT[cT] = r;
}


// ----------------------------------------------------------------------
// Ray tracing (ray_tracing.c:60-394 on one rank).

struct TraceArgs {
  ArtGrid g;
  const ArtDir* dirs;     // the batch's directions
  int ndir;
  int group;              // ray group 0..3 (set_boundary_ray's parity classes)
  int nray_max;           // rays per group and direction (largest face / 4)
  const ArtMedium* med;
  const ArtMedium* medT;  // the same, y-fastest layout (z-dominant directions)
  float4* acc;            // [ndir][ncell] {length, I1, I2, I3}, in the direction's layout
  unsigned long long* ncross;
};

// One band of calc_intensity.  F64: as the reference, exp and expm1 in
// double on the float optical depth, rounded to float.  Otherwise FP32:
// exp(-tau) from the hardware exponential (a few ulp), 1 - exp(-tau) from
// its Taylor series below 0.25 (truncation < 2e-9 relative) so that thin
// cells keep full relative precision.
template <bool F64>
__device__ __forceinline__ void band(float tau, float src, float& Icell, float& Iin) {
  float etau, etaum1;
  if (F64) {
    etau = (float)exp(-(double)tau);
    etaum1 = (float)(-expm1(-(double)tau));
  } else {
    etau = __expf(-tau);
    float p = __builtin_fmaf(tau, -1.0f / 5040, 1.0f / 720);
    p = __builtin_fmaf(tau, p, -1.0f / 120);
    p = __builtin_fmaf(tau, p, 1.0f / 24);
    p = __builtin_fmaf(tau, p, -1.0f / 6);
    p = __builtin_fmaf(tau, p, 1.0f / 2);
    p = __builtin_fmaf(tau, p, -1.0f);
    const float series = -tau * p;   // tau - tau^2/2 + ... + tau^7/5040
    etaum1 = tau < 0.25f ? series : 1.0f - etau;
  }
  Icell += Iin * etaum1;
  Iin = Iin * etau + src * etaum1;
}

template <bool F64>
__global__ __launch_bounds__(256) void art_trace_kernel(TraceArgs a) {
  const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int d = (int)(gid / a.nray_max);
  const int r = (int)(gid % a.nray_max);
  unsigned long long nc = 0;
  if (d < a.ndir) {
    const ArtGrid& g = a.g;
    const ArtDir dir = a.dirs[d];
    const int base = dir.base;
    const int da = a.group >> 1, db = a.group & 1;
    int i = 0, j = 0, k = 0, nface = 0;
    if (base <= 1) {
      nface = g.nx * g.ny / 4;
      i = 2 * (r / (g.ny >> 1)) + da;
      j = 2 * (r % (g.ny >> 1)) + db;
      k = base == 0 ? 0 : g.nz - 1;
    } else if (base <= 3) {
      nface = g.ny * g.nz / 4;
      j = 2 * (r / (g.nz >> 1)) + da;
      k = 2 * (r % (g.nz >> 1)) + db;
      i = base == 2 ? 0 : g.nx - 1;
    } else {
      // neighbouring threads take rays two cells apart in z (the fastest
      // axis of the mesh), so that their accesses share cache lines
      nface = g.nz * g.nx / 4;
      i = 2 * (r / (g.nz >> 1)) + db;
      k = 2 * (r % (g.nz >> 1)) + da;
      j = base == 4 ? 0 : g.ny - 1;
    }
    if (r < nface) {
      // set_position (set_start_pos.c:195-229)
      double sx = (double)g.xmin + (double)(i + 0.521212345) * (double)g.dx;
      double sy = (double)g.ymin + (double)(j + 0.508512345) * (double)g.dy;
      double sz = (double)g.zmin + (double)(k + 0.468287655) * (double)g.dz;
      if (base == 0) sz = g.zmin;
      if (base == 1) sz = g.zmax;
      if (base == 2) sx = g.xmin;
      if (base == 3) sx = g.xmax;
      if (base == 4) sy = g.ymin;
      if (base == 5) sy = g.ymax;
      float x = (float)sx, y = (float)sy, z = (float)sz;
      const float xovr = dir.ovr[0], yovr = dir.ovr[1], zovr = dir.ovr[2];
      const int xs = xovr > 0.0f ? 1 : 0, xn = xovr > 0.0f ? 1 : -1;
      const int ys = yovr > 0.0f ? 1 : 0, yn = yovr > 0.0f ? 1 : -1;
      const int zs = zovr > 0.0f ? 1 : 0, zn = zovr > 0.0f ? 1 : -1;
      int ix = (int)((x - g.xmin) / g.dx);
      int iy = (int)((y - g.ymin) / g.dy);
      int iz = (int)((z - g.zmin) / g.dz);
      if (xovr < 0.0f && ix == g.nx) --ix;
      if (yovr < 0.0f && iy == g.ny) --iy;
      if (zovr < 0.0f && iz == g.nz) --iz;
      auto out = [&]() {
        return ix >= g.nx || iy >= g.ny || iz >= g.nz || ix < 0 || iy < 0 || iz < 0;
      };
      float I0 = 0.0f, I1 = 0.0f, I2 = 0.0f;
      const bool zdom = base <= 1;
      float4* __restrict__ acc = a.acc + (int64_t)d * g.ncell;
      const ArtMedium* __restrict__ med = zdom ? a.medT : a.med;
      auto cell = [&]() { return art_index(zdom, g.nx, g.ny, g.nz, ix, iy, iz); };
      bool live = !out();
      int64_t pos = 0;
      ArtMedium m{};
      float4 ac{};
      if (live) {
        pos = cell();
        m = med[pos];
        ac = acc[pos];
      }
      // Each pass: the crossing's geometry and the next cell (with the
      // side-face wrap) first, the next cell's loads issued, then the
      // current cell's intensities (the geometry never reads the medium).
      while (live) {
        const float ddx = g.dx * (float)(xs + ix) - (x - g.xmin);
        const float ddy = g.dy * (float)(ys + iy) - (y - g.ymin);
        const float ddz = g.dz * (float)(zs + iz) - (z - g.zmin);
        float rdx = div_by(ddx, dir.rcp[0]);
        float rdy = div_by(ddy, dir.rcp[1]);
        float rdz = div_by(ddz, dir.rcp[2]);
        if (rdx < 0.0f) rdx = 0.0f;
        if (rdy < 0.0f) rdy = 0.0f;
        if (rdz < 0.0f) rdz = 0.0f;
        float rmin = fminf(fminf(rdx, rdy), rdz);
        x += rmin * xovr;
        y += rmin * yovr;
        z += rmin * zovr;
        if (rdx == rmin) ix += xn;
        if (rdy == rmin) iy += yn;
        if (rdz == rmin) iz += zn;
        rmin = (float)((double)rmin * g.lunit);
        // next cell: far face ends the ray; a side face wraps it to the
        // opposite face, whose intensity restarts at zero after this
        // cell's update (ray_cycle + reset_I on one rank)
        bool wrapped = false, cont = true;
        if (out()) {
          const bool far = base <= 1 ? (iz >= g.nz || iz < 0)
                                     : (base <= 3 ? (ix >= g.nx || ix < 0) : (iy >= g.ny || iy < 0));
          if (far) {
            cont = false;
          } else {
            auto wrap_x = [&]() {
              if (ix >= g.nx) { ix = 0; x = g.xmin; wrapped = true; }
              else if (ix < 0) { ix = g.nx - 1; x = g.xmax; wrapped = true; }
            };
            auto wrap_y = [&]() {
              if (iy >= g.ny) { iy = 0; y = g.ymin; wrapped = true; }
              else if (iy < 0) { iy = g.ny - 1; y = g.ymax; wrapped = true; }
            };
            auto wrap_z = [&]() {
              if (iz >= g.nz) { iz = 0; z = g.zmin; wrapped = true; }
              else if (iz < 0) { iz = g.nz - 1; z = g.zmax; wrapped = true; }
            };
            if (base <= 1) { wrap_x(); wrap_y(); }
            else if (base <= 3) { wrap_y(); wrap_z(); }
            else { wrap_z(); wrap_x(); }
            cont = !out();
          }
        }
        int64_t npos = pos;
        ArtMedium nm = m;
        float4 nac = ac;
        if (cont) {
          // another ray of this group never touches these cells, and this
          // ray never returns to one: the early read of acc is safe
          npos = cell();
          nm = med[npos];
          nac = acc[npos];
        }
        ac.x += rmin;
        band<F64>(m.k0 * rmin, m.s0, ac.y, I0);
        band<F64>(m.k1 * rmin, m.s1, ac.z, I1);
        band<F64>(m.k2 * rmin, m.s2, ac.w, I2);
        acc[pos] = ac;
        nc++;
        if (wrapped) I0 = I1 = I2 = 0.0f;
        pos = npos;
        m = nm;
        ac = nac;
        live = cont;
      }
    }
  }
  // crossings of the wavefront, one atomic per wavefront
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) nc += __shfl_xor(nc, off, 64);
  if ((threadIdx.x & 63) == 0 && nc) atomicAdd(a.ncross, nc);
}

// The same rays swept layer by layer (along the direction's dominant axis D;
// A and B are the other two, B the fast one of the layout).
//
// A launch per ray group reads and writes a record of the slice per crossing,
// after a pass that clears it: at 128^3 and 768 directions some 170 GB, which
// bound the trace (31.3 ms of 37 with the clearing, at 5 TB/s).  Here a
// block takes one tile of a direction's layers, its accumulators stay in LDS
// while the four groups pass through the layer one after the other, and the
// slice is written once: 26 GB, and 15.5 to 16.5 ms with everything below.
// What bounds it now is the memory again: 13 GB of medium (each direction reads
// it once; nearly nothing is shared between directions) and 8.6 GB of slices
// for 256 directions, 4.1 TB/s of the 4.75 that a copy reaches.  Blocks of 512
// threads leave two to a compute unit at 115 registers, so that one runs while
// the other meets a barrier (1024 threads and one block: 5% slower; 640 threads
// and 96 registers spill: 36 ms a pass instead of 21).
//
// Tiles: all rays of a direction are translates of one another, so a tile of
// cells that moves from layer to layer by the direction's own shift meets the
// rays of its own start cells and of two more on the side they come from, which
// two tiles trace: with p the ray's place at the layer's entry and a shift of
// floor(p - 1/4), a ray of slope up to 1 touches the cells 0 to 2 from its start
// cell plus the shift, also where rounding moved it by 0.2 cells (sweep_applies;
// the mirror image for slopes below 0).  Tiles part a
// layer's cells exactly; a crossing outside the block's tile adds nothing.  An
// axis that fits goes whole: no halo, and the rays' wrap stays in the tile.
// A thread carries four rays, one of each group, the same place in the pairs
// of cells.
struct SweepOri {
  int axA, axB, axD;            // 0 x, 1 y, 2 z
  int nA, nB, nD;
  uint32_t mA, mD;              // cell index: split(B) + nB * (mA * A + mD * D)
  int rA, rB, tA, tB;           // cells of a tile along A and B, tiles
  int hA, hB;                   // halo rays: 0 (whole axis) or 2
  int pA, pB;                   // pairs of rays of a full tile along A and B
  int swap;                     // group bit 0 belongs to A (else to B)
  float mnA, mxA, mnB, mxB, mnD, mxD, cell;
  double centreA, centreB;      // start fractions of set_position
  const ArtMedium* med;
};

struct SweepArgs {
  double lunit;
  const ArtDir* dirs;
  int64_t ncell;
  int tiles;                    // largest tile count of the three orientations
  float4* acc;
  unsigned long long* ncross;
  SweepOri ori[3];              // by base / 2: z, x, y dominant
};

struct SweepRay {
  float a, b, d;       // position
  float i0, i1, i2;    // band intensities
  int ia, ib;          // cell (the layer is the block's)
};

// One crossing: path length, place in the tile and flags, the cell's record,
// its medium.
constexpr uint32_t kStepMine = 1u << 30, kStepWrap = 1u << 31, kStepSlot = kStepMine - 1;
struct SweepStep {
  float rmin;
  uint32_t at, pos;
  ArtMedium m;
};
// Crossings of a layer that are planned ahead.  A fifth of a ray's layers have a
// third one; it is taken by itself, as are those that rounding could add (three
// planned ahead: 3% slower).
constexpr int kSweepSteps = 2;

typedef float art_f4 __attribute__((ext_vector_type(4)));

// A barrier for what the block shares in LDS only: __syncthreads also waits for
// every wave's loads of the medium and stores of the slice.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <bool F64, bool WHOLE_B>
__global__ __launch_bounds__(512, 4) void art_sweep_kernel(SweepArgs args) {
  extern __shared__ float4 cells[];   // [lenA][lenB], B split
  __shared__ unsigned total;
  const int dn = args.dirs[blockIdx.x / args.tiles].order, tile = (int)(blockIdx.x % args.tiles);
  const ArtDir* const __restrict__ dir = args.dirs + dn;
  const SweepOri* const __restrict__ po = args.ori + (dir->base >> 1);
  const SweepOri& o = *po;
  if (tile >= o.tA * o.tB) return;
  const int nA = o.nA, nB = o.nB, nD = o.nD;
  const uint32_t mA = o.mA;
  const int a0 = (tile / o.tB) * o.rA, b0 = (tile % o.tB) * o.rB;
  const int lenA = min(o.rA, nA - a0), lenB = min(o.rB, nB - b0);
  const float mnA = o.mnA, mnB = o.mnB, mnD = o.mnD, mxA = o.mxA, mxB = o.mxB;
  const float cell = o.cell;
  const float ovA = dir->ovr[o.axA], ovB = dir->ovr[o.axB], ovD = dir->ovr[o.axD];
  const float rcA = dir->rcpf[o.axA], rcB = dir->rcpf[o.axB], rcD = dir->rcpf[o.axD];
  const int sA = ovA > 0.0f ? 1 : 0, stA = ovA > 0.0f ? 1 : -1;
  const int sB = ovB > 0.0f ? 1 : 0, stB = ovB > 0.0f ? 1 : -1;
  const int sD = ovD > 0.0f ? 1 : 0;
  const ArtMedium* __restrict__ med = o.med;
  float4* __restrict__ acc = args.acc + (int64_t)dn * args.ncell;
  const int nthread = blockDim.x, tid = threadIdx.x;
  for (int q = tid; q < lenA * lenB; q += nthread) cells[q] = make_float4(0.f, 0.f, 0.f, 0.f);
  if (tid == 0) total = 0;

  // the thread's four rays (set_position, set_start_pos.c:195-229)
  const int pa = tid / o.pB, pb = tid % o.pB;
  SweepRay ray[4];
  bool live[4];
  unsigned nc = 0;
  unsigned own = 0;   // rays that start in this tile: their crossings count here
#pragma unroll
  for (int grp = 0; grp < 4; grp++) {
    const int da = grp >> 1, db = grp & 1;
    const int la = 2 * pa + (o.swap ? db : da) - (sA ? o.hA : 0),
              lb = 2 * pb + (o.swap ? da : db) - (sB ? o.hB : 0);
    live[grp] = la < lenA + (sA ? 0 : o.hA) && lb < lenB + (sB ? 0 : o.hB);
    if (la >= 0 && la < lenA && lb >= 0 && lb < lenB) own |= 1u << grp;
    SweepRay& r = ray[grp];
    r = SweepRay{};
    r.ia = a0 + la;
    r.ib = b0 + lb;
    r.ia += r.ia < 0 ? nA : (r.ia >= nA ? -nA : 0);
    r.ib += r.ib < 0 ? nB : (r.ib >= nB ? -nB : 0);
    r.a = (float)((double)mnA + (double)(r.ia + o.centreA) * (double)cell);
    r.b = (float)((double)mnB + (double)(r.ib + o.centreB) * (double)cell);
    r.d = sD ? mnD : o.mxD;
  }
  // A layer: the face that ends it, its first row, the tile's first cell in it
  // (start cell plus the rays' shift).
  struct Layer {
    float face;
    uint32_t row;
    int a, b;
  };
  const double slA = (double)ovA / fabs((double)ovD), slB = (double)ovB / fabs((double)ovD);
  auto at_layer = [&](int layer) {
    const int iD = sD ? layer : nD - 1 - layer;
    Layer l{cell * (float)(sD + iD), o.mD * (uint32_t)iD, 0, 0};
    auto start = [&](int first, double centre, double slope, int n) {
      int v = first + (int)floor(centre + layer * slope + (slope > 0.0 ? -0.25 : 0.25)) % n;
      v += v < 0 ? n : (v >= n ? -n : 0);
      return __builtin_amdgcn_readfirstlane(v);
    };
    if (o.tA > 1) l.a = start(a0, o.centreA, slA, nA);
    if (o.tB > 1) l.b = start(b0, o.centreB, slB, nB);
    return l;
  };
  // One crossing's geometry, and the ray goes on to the next cell.
  auto cross = [&](SweepRay& r, const Layer& l, SweepStep& st, bool& leave) {
    const uint32_t sb = (uint32_t)art_split(r.ib, nB);
    st.pos = __umul24(__umul24(mA, r.ia) + l.row, nB) + sb;
    int ja = r.ia - l.a;   // place in the tile
    ja += ja < 0 ? nA : 0;
    if (WHOLE_B) {
      st.at = ja < lenA ? kStepMine | (__umul24(ja, nB) + sb) : 0u;
    } else {
      int jb = r.ib - l.b;
      jb += jb < 0 ? nB : 0;
      st.at = ja < lenA && jb < lenB
                  ? kStepMine | (uint32_t)(__umul24(ja, lenB) + art_split(jb, lenB))
                  : 0u;
    }
    const float ddA = cell * (float)(sA + r.ia) - (r.a - mnA);
    const float ddB = cell * (float)(sB + r.ib) - (r.b - mnB);
    const float ddD = l.face - (r.d - mnD);
    const float rdA = fmaxf(div_exact(ddA, ovA, rcA), 0.0f);
    const float rdB = fmaxf(div_exact(ddB, ovB, rcB), 0.0f);
    const float rdD = fmaxf(div_exact(ddD, ovD, rcD), 0.0f);
    const float rmin = fminf(fminf(rdA, rdB), rdD);
    r.a += rmin * ovA;
    r.b += rmin * ovB;
    r.d += rmin * ovD;
    if (rdA == rmin) r.ia += stA;
    if (rdB == rmin) r.ib += stB;
    leave = rdD == rmin;
    st.rmin = (float)((double)rmin * args.lunit);
    // a side face wraps the ray to the opposite one, where its intensity
    // restarts at zero after this cell's update (ray_cycle + reset_I)
    const bool offA = (unsigned)r.ia >= (unsigned)nA, offB = (unsigned)r.ib >= (unsigned)nB;
    if (offA || offB) {
      if (offA) {
        r.a = r.ia < 0 ? mxA : mnA;
        r.ia = r.ia < 0 ? nA - 1 : 0;
      }
      if (offB) {
        r.b = r.ib < 0 ? mxB : mnB;
        r.ib = r.ib < 0 ? nB - 1 : 0;
      }
      st.at |= kStepWrap;
    }
  };
  auto absorb = [&](SweepRay& r, const SweepStep& st) {
    float4* const slot = &cells[st.at & kStepSlot];
    float4 ac = *slot;
    ac.x += st.rmin;
    band<F64>(st.m.k0 * st.rmin, st.m.s0, ac.y, r.i0);
    band<F64>(st.m.k1 * st.rmin, st.m.s1, ac.z, r.i1);
    band<F64>(st.m.k2 * st.rmin, st.m.s2, ac.w, r.i2);
    if (st.at & kStepMine) *slot = ac;
    if (st.at & kStepWrap) r.i0 = r.i1 = r.i2 = 0.0f;
  };
  // Every ray's crossings of a layer are planned one phase ahead of the phase
  // that absorbs them (the geometry never reads the medium), and their media
  // loaded between the two, so that a load's latency falls on the next phase's
  // planning: 6.4 ms per 256 directions of 128^3, against 7.0 with each cell's
  // medium loaded when the ray reaches it.
  SweepStep step[2][kSweepSteps];
  bool act[2][kSweepSteps], more[2];
  auto plan = [&](SweepRay& r, bool on, const Layer& l, int buf, bool mine) {
    unsigned n = 0;
#pragma unroll
    for (int m = 0; m < kSweepSteps; m++) {
      act[buf][m] = on;
      if (on) {
        bool leave;
        cross(r, l, step[buf][m], leave);
        on = !leave;
        n++;
      }
    }
    more[buf] = on;
    nc += mine ? n : 0u;
  };
  auto load = [&](int buf) {
#pragma unroll
    for (int m = 0; m < kSweepSteps; m++)
      if (act[buf][m]) step[buf][m].m = med[step[buf][m].pos];
  };
  // the thread's first slot of the layer and the step to its next ones
  const int qa = tid / lenB, qs = tid % lenB, stepa = nthread / lenB, steps = nthread % lenB;
  Layer now = at_layer(0);
  plan(ray[0], live[0], now, 0, own & 1u);
  load(0);
  __syncthreads();
  for (int layer = 0; layer < nD; layer++) {
    const bool last = layer == nD - 1;
    const Layer next = at_layer(last ? layer : layer + 1);
#pragma unroll
    for (int grp = 0; grp < 4; grp++) {
      const int cur = grp & 1, nxt = cur ^ 1;
      SweepRay& r = ray[grp];
      if (grp < 3)
        plan(ray[grp + 1], live[grp + 1], now, nxt, (own >> (grp + 1)) & 1u);
      else
        plan(ray[0], live[0] && !last, next, nxt, own & 1u);
#pragma unroll
      for (int m = 0; m < kSweepSteps; m++)
        if (act[cur][m]) absorb(r, step[cur][m]);
      for (bool on = more[cur]; on;) {
        SweepStep st;
        bool leave;
        cross(r, now, st, leave);
        st.m = med[st.pos];
        absorb(r, st);
        nc += (own >> grp) & 1u;
        on = !leave;
      }
      load(nxt);
      lds_barrier();
    }
    // the layer's tile to the slice, and clear
    for (int q = tid, qA = qa, qS = qs; q < lenA * lenB; q += nthread) {
      const float4 v = cells[q];
      cells[q] = make_float4(0.f, 0.f, 0.f, 0.f);
      const int h = lenB >> 1;
      int gA = now.a + qA, gB = now.b + (qS < h ? 2 * qS : 2 * (qS - h) + 1);
      gA -= gA >= nA ? nA : 0;
      gB -= gB >= nB ? nB : 0;
      const uint32_t pos =
          __umul24(__umul24(mA, gA) + now.row, nB) + (uint32_t)art_split(gB, nB);
      __builtin_nontemporal_store((art_f4){v.x, v.y, v.z, v.w},
                                  reinterpret_cast<art_f4*>(acc + pos));
      qA += stepa;
      qS += steps;
      if (qS >= lenB) { qS -= lenB; qA++; }
    }
    now = next;
    lds_barrier();
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) nc += __shfl_xor(nc, off, 64);
  if ((tid & 63) == 0) atomicAdd(&total, nc);
  __syncthreads();
  if (tid == 0 && total) atomicAdd(args.ncross, (unsigned long long)total);
}

__global__ void art_fill_kernel(float4* __restrict__ p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

// ----------------------------------------------------------------------
// calc_GH_tot for the batch's directions in order: gh[k][c] (FP32, 6
// outputs GHI, HHI, GHeI, HHeI, GHeII, HHeII); optionally Kahan-compensated
// across directions.
// One block per TILE x TILE (y, z) tile of one x plane, one thread per cell.
// The slices of x- and y-dominant directions are read in their own layout
// (z fastest); those of z-dominant directions (y fastest) go through an LDS
// tile, read along y and used along z, so that every read is a contiguous
// run.  Each cell's sums take the directions in batch order.  TILE 32 reads at
// the rate of the memory (5 TB/s).  Where its blocks would leave compute units
// without work (below two per unit), TILE 16 makes four times as many, which
// take two directions at once (one wavefront's chain of FP64 operations is
// what lasts) with the next two on their way: 32^3 with 192 directions 120 us
// instead of 197.  (Fetching ahead at 128^3 costs the wide tile a third: 2.30 ms per 256 directions instead of 1.73.)
// Grid: (ceil(ny/TILE) ceil(nz/TILE), nx), blocks of TILE^2 threads.
template <bool KAHAN, int TILE>
__global__ __launch_bounds__(TILE * TILE) void art_gh_kernel(
    const float4* __restrict__ acc, const ArtDir* __restrict__ dirs, int ndir, int nx, int ny,
    int nz, const ArtMedium* __restrict__ med, float f0, float f1, float f2, float f3, float f4,
    float f5, float* __restrict__ gh, float* __restrict__ comp) {
  constexpr int P = TILE < 32 ? 2 : 1;   // directions at once
  __shared__ float4 tile[P][TILE][TILE + 1];
  const int64_t ncell = (int64_t)nx * ny * nz;
  const int ntz = (nz + TILE - 1) / TILE;
  const int y0 = (int)(blockIdx.x / ntz) * TILE, z0 = (int)(blockIdx.x % ntz) * TILE;
  const int ix = blockIdx.y;
  const int tz = threadIdx.x % TILE, ty = threadIdx.x / TILE;
  const int iy = y0 + ty, iz = z0 + tz;
  const bool valid = iy < ny && iz < nz;
  // this cell's record in the layout of x- and y-dominant directions
  const int64_t cs = valid ? art_index(false, nx, ny, nz, ix, iy, iz) : 0;
  const int64_t c = ((int64_t)ix * ny + iy) * nz + iz;
  // the record this thread loads into the tile for z-dominant directions:
  // cell (y0 + tz, z0 + ty), read along y
  const bool tvalid = y0 + tz < ny && z0 + ty < nz;
  const int64_t ct = tvalid ? art_index(true, nx, ny, nz, ix, y0 + tz, z0 + ty) : 0;
  const ArtMedium m = valid ? med[cs] : ArtMedium{1.0f, 1.0f, 1.0f, 0.0f, 0.0f, 0.0f};
  const float3 ka = make_float3(m.k0, m.k1, m.k2), so = make_float3(m.s0, m.s1, m.s2);
  float s[6], e[6];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    s[k] = valid ? gh[k * ncell + c] : 0.0f;
    e[k] = KAHAN && valid ? comp[k * ncell + c] : 0.0f;
  }
  const double f[6] = {f0, f1, f2, f3, f4, f5};
  // Per-cell reciprocals: the float quotients I/kappa are exact through
  // div_by; the double quotients become products (within an ulp of double).
  const double rkx = 1.0 / (double)ka.x, rky = 1.0 / (double)ka.y, rkz = 1.0 / (double)ka.z;
  // source-function terms do not depend on the direction
  double sg0 = so.x;
  sg0 += (double)so.y * kRjHI2;
  sg0 += (double)so.z * kRjHI3;
  double sh0 = so.x;
  sh0 += (double)so.y * kRhHI2;
  sh0 += (double)so.z * kRhHI3;
  double sg1 = so.y;
  sg1 += (double)so.z * kRjHeI3;
  double sh1 = so.y;
  sh1 += (double)so.z * kRhHeI3;
  const double sg2 = so.z, sh2 = so.z;
  auto zdom = [&](int d) { return dirs[d].base <= 1; };   // the same for the whole block
  auto record = [&](int d) {
    if (d >= ndir) return make_float4(1.0f, 0.0f, 0.0f, 0.0f);
    return (zdom(d) ? tvalid : valid) ? acc[(int64_t)d * ncell + (zdom(d) ? ct : cs)]
                                      : make_float4(1.0f, 0.0f, 0.0f, 0.0f);
  };
  float4 ahead[P];
  if (P > 1)
#pragma unroll
    for (int p = 0; p < P; p++) ahead[p] = record(p);
  for (int d = 0; d < ndir; d += P) {
    float4 a[P];
    bool turn = false;
#pragma unroll
    for (int p = 0; p < P; p++) {
      a[p] = P > 1 ? ahead[p] : record(d);
      turn = turn || (d + p < ndir && zdom(d + p));
    }
    if (P > 1)
#pragma unroll
      for (int p = 0; p < P; p++) ahead[p] = record(d + P + p);
    if (turn) {
      lds_barrier();           // the previous tiles have been read
#pragma unroll
      for (int p = 0; p < P; p++) tile[p][ty][tz] = a[p];
      lds_barrier();
#pragma unroll
      for (int p = 0; p < P; p++)
        if (d + p < ndir && zdom(d + p)) a[p] = tile[p][tz][ty];
    }
    if (!valid) continue;
    double v[P][6];
#pragma unroll
    for (int p = 0; p < P; p++) {
      const double rl = 1.0 / (double)a[p].x;
      const double q1 = (double)div_by(a[p].y, rkx);   // I_1 / kappa_1 (float, as the reference)
      const double q2 = (double)div_by(a[p].z, rky);
      const double q3 = (double)div_by(a[p].w, rkz);
      const double z2 = (double)a[p].z * rky, w3 = (double)a[p].w * rkz;
      // HI
      double Ig = q1;
      Ig += z2 * kRjHI2;
      Ig += w3 * kRjHI3;
      double Ih = q1;
      Ih += z2 * kRhHI2;
      Ih += w3 * kRhHI3;
      v[p][0] = (Ig * rl + sg0) * f[0];
      v[p][1] = (Ih * rl + sh0) * f[1];
      // HeI
      Ig = q2;
      Ig += w3 * kRjHeI3;
      Ih = q2;
      Ih += w3 * kRhHeI3;
      v[p][2] = (Ig * rl + sg1) * f[2];
      v[p][3] = (Ih * rl + sh1) * f[3];
      // HeII
      v[p][4] = (q3 * rl + sg2) * f[4];
      v[p][5] = (q3 * rl + sh2) * f[5];
    }
#pragma unroll
    for (int p = 0; p < P; p++) {
      if (d + p >= ndir) break;
#pragma unroll
      for (int k = 0; k < 6; k++) {
        if (KAHAN) {
          const float y = (float)v[p][k] - e[k];
          const float t = s[k] + y;
          e[k] = (t - s[k]) - y;
          s[k] = t;
        } else {
          s[k] = (float)((double)s[k] + v[p][k]);
        }
      }
    }
  }
  if (!valid) return;
#pragma unroll
  for (int k = 0; k < 6; k++) {
    gh[k * ncell + c] = s[k];
    if (KAHAN) comp[k * ncell + c] = e[k];
  }
}

// calc_GH_sum: prev_chem rates += gh * (float)(1/N_ANG)
__global__ void art_gh_sum_kernel(unsigned char* __restrict__ mesh, int64_t ncell,
                                  const float* __restrict__ gh, float r_n_ang) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncell) return;
  float* r = reinterpret_cast<float*>(mesh + c * kStride + kPrevChem + 28);
  r[0] += gh[0 * ncell + c] * r_n_ang;   // GammaHI  += GHI_tot
  r[1] += gh[1 * ncell + c] * r_n_ang;   // HeatHI   += HHI_tot
  r[2] += gh[2 * ncell + c] * r_n_ang;   // GammaHeI += GHeI_tot
  r[4] += gh[3 * ncell + c] * r_n_ang;   // HeatHeI  += HHeI_tot
  r[3] += gh[4 * ncell + c] * r_n_ang;   // GammaHeII += GHeII_tot
  r[5] += gh[5 * ncell + c] * r_n_ang;   // HeatHeII += HHeII_tot
}

// ----------------------------------------------------------------------
// Host side.

int g_nside = 8;             // N_SIDE (run_param.h:159)
int g_heatcool = 1;          // __HEATCOOL__ (src/Makefile:187)
int g_batch = 0;             // directions per batch; 0: as many as 8 GiB of slices hold, <= 256
int g_kahan = 0;
int g_exp64 = 0;             // 1: exp/expm1 in FP64 as the reference
argot_diffuse_stats g_dstats{};

struct ArtCtx {
  int nside = 0;
  std::vector<ArtDir> dirs;       // sorted order
  bool sweep = false;             // sweep_directions(dirs)
  float fact[6] = {0, 0, 0, 0, 0, 0};
  hipStream_t stream = nullptr;
  hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
  ArtDir* d_dirs = nullptr;
  ArtMedium *med = nullptr, *medT = nullptr;   // [ncell]; medT: y-fastest
  float4* acc = nullptr;
  float *gh = nullptr, *comp = nullptr;
  unsigned long long* ncross = nullptr;
  int64_t ncell = 0;
  int batch = 0;
};
ArtCtx a_;

#define A_OK(expr)                                                                  \
  do {                                                                              \
    hipError_t _e = (expr);                                                         \
    if (_e != hipSuccess) {                                                         \
      (void)hipGetLastError(); /* else the next launch reports it */                \
      argot_hip_internal_set_error(_e == hipErrorOutOfMemory ? ARGOT_ERR_NOMEM      \
                                                             : ARGOT_ERR_HIP);      \
      return;                                                                       \
    }                                                                               \
  } while (0)

// Tiles of art_sweep_kernel for layers of nA x nB cells: the split with the
// fewest lanes over all tiles, of at most 512 threads a block (four rays each,
// so at most 2048 cells or 32 KiB of LDS).  Whole rows along B count for a
// tenth less, since their lanes read and write long runs and need one place
// instead of two (128^3: 6.4 ms per 256 directions with A whole, 5.7 with B
// whole).  128 x 128: 11 tiles of 12 rows, 256 x 256: 11 x 4 tiles of 24 x 64
// (both 20% more lanes than rays); up to 32 x 64 one tile.
constexpr int kSweepThreads = 512;
void sweep_tiles(SweepOri& o) {
  int64_t best = 0;
  auto axis = [](int n, int t, int& r, int& h) {   // n cells in about t tiles
    r = t == 1 ? n : ((n + t - 1) / t + 1) & ~1;
    h = r < n ? 2 : 0;
    return r == n || r + h <= n;
  };
  for (int ta = 1; ta <= o.nA; ta++) {
    int rA, hA;
    if (!axis(o.nA, ta, rA, hA)) continue;
    const int pA = (rA + hA) / 2;
    for (int tb = 1; tb <= o.nB; tb++) {
      int rB, hB;
      if (!axis(o.nB, tb, rB, hB)) continue;
      const int pB = (rB + hB) / 2;
      if ((int64_t)pA * pB > kSweepThreads) continue;
      const int cA = (o.nA + rA - 1) / rA, cB = (o.nB + rB - 1) / rB;
      const int64_t lanes = (int64_t)cA * cB * ((pA * pB + 63) & ~63) * (cB == 1 ? 9 : 10);
      if (best == 0 || lanes <= best) {   // (of equals the longest runs along B)
        best = lanes;
        o.rA = rA; o.rB = rB; o.hA = hA; o.hB = hB; o.pA = pA; o.pB = pB; o.tA = cA; o.tB = cB;
      }
      break;   // more at this ta only add halo
    }
  }
}

// Whether the sweep's bounds hold for the directions: bases that name their
// dominant axis and sign, and components (1e-31 at least, make_angles) whose
// reciprocals and remainders stay normal in FP32.
bool sweep_directions(const std::vector<ArtDir>& dirs) {
  for (const ArtDir& d : dirs) {
    if (d.base < 0 || d.base > 5) return false;
    const int ax = d.base <= 1 ? 2 : (d.base <= 3 ? 0 : 1);
    const double lead = (d.base & 1) ? -(double)d.ovr[ax] : (double)d.ovr[ax];
    if (!(lead > 0.1 && lead < 2.0)) return false;
    for (int k = 0; k < 3; k++)
      if (!(fabs((double)d.ovr[k]) <= lead * (1.0 + 1e-5) && fabs((double)d.ovr[k]) >= 9.9e-32))
        return false;
  }
  return true;
}

// The order in which a batch's directions are swept: by base, then by crossings
// a layer (1 + the slopes), most first.  Directions that go through the layers
// alike and at one pace find more of one another's medium in the L2, and the
// longest go first: 20.7 ms a pass at 128^3 instead of 21.9 in batch order.
void sweep_order(std::vector<ArtDir>& dirs, int batch) {
  auto crossings = [&](const ArtDir& d) {
    const float* o = d.ovr;
    return (fabsf(o[0]) + fabsf(o[1]) + fabsf(o[2])) /
           std::max(fabsf(o[0]), std::max(fabsf(o[1]), fabsf(o[2])));
  };
  std::vector<int> ord;
  for (size_t d0 = 0; d0 < dirs.size(); d0 += batch) {
    ord.resize(std::min<size_t>(batch, dirs.size() - d0));
    for (size_t i = 0; i < ord.size(); i++) ord[i] = (int)i;
    std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) {
      const ArtDir &p = dirs[d0 + a], &q = dirs[d0 + b];
      return p.base != q.base ? p.base < q.base : crossings(p) > crossings(q);
    });
    for (size_t i = 0; i < ord.size(); i++) dirs[d0 + i].order = ord[i];
  }
}

// Whether they hold for the box: cell indices in 32 bits, and rays that stay
// within 0.2 cells of where the tiles expect them.  What moves a ray: rounding (at
// most 3 crossings a layer, each within an ulp of the largest coordinate), and the
// part by which an axis' extent differs from its cells, once at the entry and once
// at each of up to nD/n + 1 wraps through its side faces, which put the ray back
// on the box's face.
bool sweep_applies(const ArtGrid& g) {
  const double mn[3] = {g.xmin, g.ymin, g.zmin}, mx[3] = {g.xmax, g.ymax, g.zmax};
  const double d[3] = {g.dx, g.dy, g.dz};
  const int n[3] = {g.nx, g.ny, g.nz};
  const int longest = std::max(g.nx, std::max(g.ny, g.nz));
  double big = 0.0, off = 0.0;
  for (int k = 0; k < 3; k++) {
    if (!(d[k] > 1e-12 && d[k] < 1e6)) return false;
    off = std::max(off, fabs(mx[k] - mn[k] - n[k] * d[k]) / d[k] * (2.0 + (double)longest / n[k]));
    big = std::max(big, std::max(fabs(mn[k]), fabs(mx[k])));
  }
  const double err = off + 3.0 * longest * big * 1.2e-7 / d[0];
  const int64_t rows = std::max((int64_t)g.nx * g.ny, (int64_t)g.nx * g.nz);   // 24-bit products
  return err < 0.2 && g.ncell <= ((int64_t)1 << 30) &&
         std::max(rows, (int64_t)g.ny * g.nz) < (1 << 24);
}

double now_ms() {
  return std::chrono::duration<double, std::milli>(
             std::chrono::steady_clock::now().time_since_epoch())
      .count();
}

// HEALPix ring scheme (Gorski et al. 2005, ApJ 622, 759, sec. 4): centre
// of pixel ipix as (theta, phi), the role of chealpix's pix2ang_ring.
long isqrt_l(long v) {
  long r = (long)sqrt((double)v + 0.5);
  while (r * r > v) r--;
  while ((r + 1) * (r + 1) <= v) r++;
  return r;
}

void pix2ang_ring(long nside, long ipix, double* theta, double* phi) {
  const long nl2 = 2 * nside, nl4 = 4 * nside, npix = 12 * nside * nside;
  const long ncap = nl2 * (nside - 1);
  const double fact2 = 4.0 / npix;
  double z;
  if (ipix < ncap) {
    const long iring = (1 + isqrt_l(1 + 2 * ipix)) >> 1;
    const long iphi = ipix + 1 - 2 * iring * (iring - 1);
    z = 1.0 - (double)(iring * iring) * fact2;
    *phi = ((double)iphi - 0.5) * (0.5 * kPiArt) / iring;
  } else if (ipix < npix - ncap) {
    const long ip = ipix - ncap;
    const long iring = ip / nl4 + nside;
    const long iphi = ip % nl4 + 1;
    const double fodd = ((iring + nside) & 1) ? 1.0 : 0.5;
    z = (double)(nl2 - iring) * (2.0 / (3.0 * nside));
    *phi = ((double)iphi - fodd) * kPiArt / nl2;
  } else {
    const long ip = npix - ipix;
    const long iring = (1 + isqrt_l(2 * ip - 1)) >> 1;
    const long iphi = 4 * iring + 1 - (ip - 2 * iring * (iring - 1));
    z = -1.0 + (double)(iring * iring) * fact2;
    *phi = ((double)iphi - 0.5) * (0.5 * kPiArt) / iring;
  }
  *theta = acos(z);
}

// set_angle_info + sort_angle_id (set_angle.c:12-247)
void make_angles(int nside, angle_info* out, int corner_num[8]) {
  const long npix = 12L * nside * nside;
  const double cos_pi_4 = cos(0.7853981633974483096156608458198757);
  for (int i = 0; i < 8; i++) corner_num[i] = 0;
  for (long ip = 0; ip < npix; ip++) {
    double th, ph;
    pix2ang_ring(nside, ip, &th, &ph);
    const double ct = cos(th), st = sin(th), cp = cos(ph), sp = sin(ph), tt = tan(th);
    double x = st * cp, y = st * sp, z = ct;
    if (fabs(x) < kTinyArt) x = x >= 0.0 ? kTinyArt : -kTinyArt;
    if (fabs(y) < kTinyArt) y = y >= 0.0 ? kTinyArt : -kTinyArt;
    if (fabs(z) < kTinyArt) z = z >= 0.0 ? kTinyArt : -kTinyArt;
    angle_info& a = out[ip];
    a.xovr = (float)x;
    a.yovr = (float)y;
    a.zovr = (float)z;
    const double rc = 1.0 / fabs(cp), rs = 1.0 / fabs(sp);
    int b;
    if (fabs(cp) >= cos_pi_4) {
      if (0.0 <= tt && tt <= rc) b = 0;
      else if (-rc <= tt && tt < 0.0) b = 1;
      else b = cp >= 0.0 ? 2 : 3;
    } else {
      if (0.0 <= tt && tt <= rs) b = 0;
      else if (-rs <= tt && tt < 0.0) b = 1;
      else b = sp >= 0.0 ? 4 : 5;
    }
    int cid = (cp > 0.0) ? (sp > 0.0 ? (ct > 0.0 ? 0 : 1) : (ct > 0.0 ? 2 : 3))
                         : (sp > 0.0 ? (ct > 0.0 ? 4 : 5) : (ct > 0.0 ? 6 : 7));
    a.base_id = (short)b;
    a.corner_id = (short)cid;
    corner_num[cid]++;
  }
  // sort_angle_id: bubble passes by corner, then by base within a corner
  for (long i = 0; i < npix - 1; i++)
    for (long j = npix - 1; j > i; j--)
      if (out[j - 1].corner_id > out[j].corner_id) std::swap(out[j - 1], out[j]);
  for (long i = 0; i < npix - 1; i++)
    for (long j = npix - 1; j > i; j--)
      if (out[j - 1].base_id > out[j].base_id && !(out[j - 1].corner_id < out[j].corner_id))
        std::swap(out[j - 1], out[j]);
}

double csect_HI(double nu) {
  if (nu < 1.0) return 0.0;
  const double eps = sqrt(nu - 1.0);
  return 6.3e-18 / (nu * nu * nu * nu) * exp(4.0 - 4.0 * atan(eps) / eps) /
         (1.0 - exp(-2.0 * kPiArt / eps));
}
double csect_HeI(double nu) {
  if (nu < 1.8125) return 0.0;
  return 7.83e-18 * (1.66 * pow((nu / 1.8125), -2.05) - 0.66 * pow((nu / 1.8125), -3.05));
}
double csect_HeII(double nu) {
  if (nu < 4.0) return 0.0;
  const double eps = sqrt(nu / 4.0 - 1.0);
  return 6.3e-18 * 256.0 / (nu * nu * nu * nu) * exp(4.0 - 4.0 * atan(eps) / eps) /
         (1.0 - exp(-2.0 * kPiArt / eps)) / 4.0;
}

// set_step_func_factor (set_step_func_factor.c:29-104)
void step_factors(int heatcool, step_func_factor* sf) {
  const double range = heatcool ? 0.0632353 : 0.0;
  const int nbin = heatcool ? 64 : 1;
  const double unit[3] = {1.0, 1.8125, 4.0};
  const double nuL[3] = {3.2885e15, 5.9483e15, 1.3154e16};
  double (*cs[3])(double) = {csect_HI, csect_HeI, csect_HeII};
  float* out[3] = {sf->HI, sf->HeI, sf->HeII};
  for (int s = 0; s < 3; s++) out[s][0] = out[s][1] = 0.0f;
  const double block = range / nbin;
  for (int inu = 0; inu < nbin; inu++)
    for (int s = 0; s < 3; s++) {
      double nu = unit[s] + inu * block, nu_next = unit[s] + (inu + 1) * block;
      if (nu == unit[s]) nu = unit[s] + 1e-7;
      if (nu_next == unit[s]) nu_next = unit[s] + 1e-7;
      const double c0 = 4.0e0 * kPiArt * cs[s](nu) / (kHplanck * (nu * nuL[s]));
      const double c0n = 4.0e0 * kPiArt * cs[s](nu_next) / (kHplanck * (nu_next * nuL[s]));
      const double c1 = inu == 0 ? 0.0e0 : c0 * (nu - unit[s]);
      const double c1n = c0 * (nu_next - unit[s]);
      out[s][0] += (c0 + c0n) * 0.5e0;
      out[s][1] += (c1 + c1n) * 0.5e0;
    }
  for (int s = 0; s < 3; s++) {
    out[s][0] /= nbin;
    out[s][1] /= nbin / (kHplanck * nuL[s]);
  }
}

}  // namespace
}  // namespace argot

using namespace argot;

extern "C" {

void argot_hip_set_diffuse_nside(int nside) { g_nside = nside > 0 ? nside : 8; }
void argot_hip_set_diffuse_heatcool(int on) { g_heatcool = on ? 1 : 0; }
void argot_hip_set_diffuse_batch(int ndir) { g_batch = ndir > 0 ? ndir : 0; }
void argot_hip_set_diffuse_kahan(int on) { g_kahan = on ? 1 : 0; }
void argot_hip_set_diffuse_exp64(int on) { g_exp64 = on ? 1 : 0; }
void argot_hip_diffuse_stats(struct argot_diffuse_stats* out) {
  if (out) *out = g_dstats;
}

void init_hd_param(struct host_diffuse_param* hd) {
  argot_hip_internal_clear_error();
  if (!hd) return argot_hip_internal_set_error(ARGOT_ERR_ARG);
  hd->step_fact = (struct step_func_factor*)malloc(sizeof(struct step_func_factor));
  hd->angle = (struct angle_info*)malloc(sizeof(struct angle_info) * 12 * g_nside * g_nside);
  if (!hd->step_fact || !hd->angle) argot_hip_internal_set_error(ARGOT_ERR_NOMEM);
}

void free_hd_param(struct host_diffuse_param* hd) {
  if (!hd) return;
  free(hd->step_fact);
  free(hd->angle);
  hd->step_fact = nullptr;
  hd->angle = nullptr;
}

void setup_diffuse_photon(struct host_diffuse_param* hd, struct run_param* this_run) {
  argot_hip_internal_clear_error();
  if (!hd || !hd->angle || !hd->step_fact || !this_run)
    return argot_hip_internal_set_error(ARGOT_ERR_ARG);
  make_angles(g_nside, hd->angle, hd->corner_id_num);
  step_factors(g_heatcool, hd->step_fact);
}

void init_diffuse_gpu(struct cuda_diffuse_param* cd, struct cuda_param* this_cuda,
                      struct run_param* this_run) {
  argot_hip_internal_clear_error();
  (void)this_cuda;
  if (!cd || !this_run) return argot_hip_internal_set_error(ARGOT_ERR_ARG);
  const int nx = this_run->nmesh_x_local, ny = this_run->nmesh_y_local,
            nz = this_run->nmesh_z_local;
  if (nx <= 0 || ny <= 0 || nz <= 0 || (nx | ny | nz) & 1)
    return argot_hip_internal_set_error(ARGOT_ERR_ARG);   // ray groups need even sizes
  const int64_t ncell = (int64_t)nx * ny * nz;
  const int nang = 12 * g_nside * g_nside;
  // Each direction of a batch owns one float4 slice over the mesh; more
  // directions per batch keep more rays in flight.
  int batch = g_batch;
  if (batch <= 0) {
    const int64_t fit = ((int64_t)8 << 30) / (16 * ncell);
    batch = (int)std::max<int64_t>(1, std::min<int64_t>(256, fit));
  }
  batch = std::min(batch, nang);
  if (!a_.stream) {
    A_OK(hipStreamCreate(&a_.stream));
    for (auto& e : a_.ev) A_OK(hipEventCreate(&e));
  }
  for (void* p : {(void*)a_.d_dirs, (void*)a_.med, (void*)a_.acc, (void*)a_.gh,
                  (void*)a_.comp, (void*)a_.ncross, (void*)a_.medT})
    if (p) A_OK(hipFree(p));
  a_.d_dirs = nullptr;
  a_.med = nullptr;
  a_.acc = nullptr;
  a_.medT = nullptr;
  a_.gh = a_.comp = nullptr;
  a_.ncross = nullptr;
  a_.dirs.clear();
  // The sizes are set only once every buffer exists, so that a failed
  // allocation leaves a context that every later call refuses.
  a_.ncell = 0;
  a_.batch = 0;
  A_OK(hipMalloc(&a_.d_dirs, sizeof(ArtDir) * nang));
  A_OK(hipMalloc(&a_.med, sizeof(ArtMedium) * ncell));
  A_OK(hipMalloc(&a_.medT, sizeof(ArtMedium) * ncell));
  A_OK(hipMalloc(&a_.gh, sizeof(float) * 6 * ncell));
  A_OK(hipMalloc(&a_.comp, sizeof(float) * 6 * ncell));
  A_OK(hipMalloc(&a_.ncross, sizeof(unsigned long long)));
  // The slices last: where the default batch does not fit what is left, a
  // smaller one does (the rates are the same).
  hipError_t e = hipMalloc(&a_.acc, sizeof(float4) * ncell * batch);
  while (e == hipErrorOutOfMemory && g_batch <= 0 && batch > 1) {
    (void)hipGetLastError();
    a_.acc = nullptr;
    batch = (batch + 1) / 2;
    e = hipMalloc(&a_.acc, sizeof(float4) * ncell * batch);
  }
  if (e != hipSuccess) a_.acc = nullptr;
  A_OK(e);
  a_.ncell = ncell;
  a_.batch = batch;
  a_.nside = g_nside;
  // the reference's pointers: step factors and angles live in the
  // library's context; rmesh names the accumulator slices
  cd[0].step_fact = nullptr;
  cd[0].angle = nullptr;
  cd[0].rmesh = reinterpret_cast<struct radiation_mesh*>(a_.acc);
}

void send_diffuse_data(struct host_diffuse_param* hd, struct cuda_diffuse_param* cd,
                       struct cuda_param* this_cuda) {
  argot_hip_internal_clear_error();
  (void)cd;
  (void)this_cuda;
  if (!hd || !hd->angle || !hd->step_fact) return argot_hip_internal_set_error(ARGOT_ERR_ARG);
  if (!a_.d_dirs || a_.ncell <= 0) return argot_hip_internal_set_error(ARGOT_ERR_STATE);
  const int nang = 12 * a_.nside * a_.nside;
  a_.dirs.resize(nang);
  for (int i = 0; i < nang; i++) {
    const angle_info& an = hd->angle[i];
    ArtDir& d = a_.dirs[i];
    d.ovr[0] = an.xovr;
    d.ovr[1] = an.yovr;
    d.ovr[2] = an.zovr;
    d.base = an.base_id;
    for (int k = 0; k < 3; k++) {
      d.rcp[k] = 1.0 / (double)d.ovr[k];
      d.rcpf[k] = 1.0f / d.ovr[k];
    }
  }
  sweep_order(a_.dirs, a_.batch);
  const step_func_factor* sf = hd->step_fact;
  const float f[6] = {sf->HI[0], sf->HI[1], sf->HeI[0], sf->HeI[1], sf->HeII[0], sf->HeII[1]};
  memcpy(a_.fact, f, sizeof f);
  a_.sweep = sweep_directions(a_.dirs);
  A_OK(hipMemcpy(a_.d_dirs, a_.dirs.data(), sizeof(ArtDir) * nang, hipMemcpyHostToDevice));
}

void calc_diffuse_photon_radiation(struct fluid_mesh* mesh, struct run_param* this_run,
                                   struct cuda_mem_space* cuda_mem, struct cuda_param* this_cuda,
                                   struct host_diffuse_param* hd, struct cuda_diffuse_param* cd,
                                   struct omp_param* this_omp) {
  argot_hip_internal_clear_error();
  (void)mesh;
  (void)this_cuda;
  (void)hd;
  (void)cd;
  (void)this_omp;
  const double t_start = now_ms();
  if (!this_run || !cuda_mem || !cuda_mem->mesh_dev)
    return argot_hip_internal_set_error(ARGOT_ERR_STATE);
  if (a_.dirs.empty() || !a_.d_dirs || !a_.med || !a_.acc || !a_.medT || !a_.gh || !a_.comp ||
      !a_.ncross || a_.ncell <= 0 || a_.batch <= 0)
    return argot_hip_internal_set_error(ARGOT_ERR_STATE);
  ArtGrid g;
  g.nx = this_run->nmesh_x_local;
  g.ny = this_run->nmesh_y_local;
  g.nz = this_run->nmesh_z_local;
  g.ncell = (int64_t)g.nx * g.ny * g.nz;
  if (g.ncell != a_.ncell || this_run->rank_x || this_run->rank_y || this_run->rank_z ||
      this_run->nnode_x > 1 || this_run->nnode_y > 1 || this_run->nnode_z > 1)
    return argot_hip_internal_set_error(ARGOT_ERR_ARG);
  if (this_run->delta_x != this_run->delta_y || this_run->delta_x != this_run->delta_z)
    return argot_hip_internal_set_error(ARGOT_ERR_ARG);   // the ray groups assume cubic cells
  g.xmin = this_run->xmin_local;
  g.ymin = this_run->ymin_local;
  g.zmin = this_run->zmin_local;
  g.xmax = this_run->xmax_local;
  g.ymax = this_run->ymax_local;
  g.zmax = this_run->zmax_local;
  g.dx = this_run->delta_x;
  g.dy = this_run->delta_y;
  g.dz = this_run->delta_z;
  g.lunit = this_run->lunit;
  unsigned char* dmesh = reinterpret_cast<unsigned char*>(cuda_mem->mesh_dev);
  hipStream_t st = a_.stream;
  const int64_t nc = g.ncell;
  const unsigned nb = (unsigned)((nc + 255) / 256);
  A_OK(hipEventRecord(a_.ev[0], st));
  art_rmesh_kernel<<<nb, 256, 0, st>>>(
      dmesh, g.nx, g.ny, g.nz, this_run->denstonh, this_run->uenetok,
      argot_hip_internal_helium_fact(), (float)csect_HI(1.0 + 1.0e-7),
      (float)csect_HeI(1.8125 + 1.0e-7), (float)csect_HeII(4.0 + 1.0e-7), a_.med, a_.medT);
  A_OK(hipGetLastError());
  A_OK(hipMemsetAsync(a_.gh, 0, sizeof(float) * 6 * nc, st));
  A_OK(hipMemsetAsync(a_.comp, 0, sizeof(float) * 6 * nc, st));
  A_OK(hipMemsetAsync(a_.ncross, 0, sizeof(unsigned long long), st));
  const int nang = (int)a_.dirs.size();
  const int nray_max = std::max(g.nx * g.ny, std::max(g.ny * g.nz, g.nz * g.nx)) / 4;
  float trace_ms = 0.0f, gh_ms = 0.0f;
  const bool sweep = a_.sweep && sweep_applies(g);
  SweepArgs sa{};
  unsigned sweep_threads = 0, sweep_lds = 0;
  bool sweep_whole = true;   // B whole in every orientation
  if (sweep) {
    const int n[3] = {g.nx, g.ny, g.nz};
    const float mn[3] = {g.xmin, g.ymin, g.zmin}, mx[3] = {g.xmax, g.ymax, g.zmax};
    const double centre[3] = {0.521212345, 0.508512345, 0.468287655};
    sa.lunit = g.lunit;
    sa.ncell = nc;
    sa.acc = a_.acc;
    sa.ncross = a_.ncross;
    // {A, B, D, group bit of A} for z-, x- and y-dominant directions
    const int axes[3][4] = {{0, 1, 2, 0}, {1, 2, 0, 0}, {0, 2, 1, 1}};
    for (int k = 0; k < 3; k++) {
      SweepOri& o = sa.ori[k];
      o.axA = axes[k][0];
      o.axB = axes[k][1];
      o.axD = axes[k][2];
      o.swap = axes[k][3];
      o.nA = n[o.axA];
      o.nB = n[o.axB];
      o.nD = n[o.axD];
      o.mA = k == 2 ? (uint32_t)o.nD : 1u;
      o.mD = k == 2 ? 1u : (uint32_t)o.nA;
      o.mnA = mn[o.axA];
      o.mxA = mx[o.axA];
      o.mnB = mn[o.axB];
      o.mxB = mx[o.axB];
      o.mnD = mn[o.axD];
      o.mxD = mx[o.axD];
      o.cell = g.dx;
      o.centreA = centre[o.axA];
      o.centreB = centre[o.axB];
      o.med = k == 0 ? a_.medT : a_.med;
      sweep_tiles(o);
      sa.tiles = std::max(sa.tiles, o.tA * o.tB);
      sweep_whole = sweep_whole && o.tB == 1;
      sweep_threads = std::max(sweep_threads, (unsigned)(o.pA * o.pB + 63) & ~63u);
      sweep_lds = std::max(sweep_lds, (unsigned)(sizeof(float4) * o.rA * o.rB));
    }
  }
  for (int d0 = 0; d0 < nang; d0 += a_.batch) {
    const int nd = std::min(a_.batch, nang - d0);
    A_OK(hipEventRecord(a_.ev[1], st));
    if (sweep) {
      sa.dirs = a_.d_dirs + d0;
      const unsigned nblock = (unsigned)(sa.tiles * nd);
      const auto kernel = g_exp64 ? (sweep_whole ? art_sweep_kernel<true, true>
                                                 : art_sweep_kernel<true, false>)
                                  : (sweep_whole ? art_sweep_kernel<false, true>
                                                 : art_sweep_kernel<false, false>);
      kernel<<<nblock, sweep_threads, sweep_lds, st>>>(sa);
    } else {
      const int64_t nacc = (int64_t)nd * nc;
      art_fill_kernel<<<(unsigned)((nacc + 255) / 256), 256, 0, st>>>(a_.acc, nacc);
      TraceArgs ta;
      ta.g = g;
      ta.dirs = a_.d_dirs + d0;
      ta.ndir = nd;
      ta.nray_max = nray_max;
      ta.med = a_.med;
      ta.medT = a_.medT;
      ta.acc = a_.acc;
      ta.ncross = a_.ncross;
      const int64_t nthread = (int64_t)nd * nray_max;
      for (int grp = 0; grp < 4; grp++) {
        ta.group = grp;
        if (g_exp64)
          art_trace_kernel<true><<<(unsigned)((nthread + 255) / 256), 256, 0, st>>>(ta);
        else
          art_trace_kernel<false><<<(unsigned)((nthread + 255) / 256), 256, 0, st>>>(ta);
      }
    }
    A_OK(hipGetLastError());
    A_OK(hipEventRecord(a_.ev[2], st));
    const float* f = a_.fact;
    auto sums = [&](auto kernel, int tile) {
      const dim3 grid((unsigned)(((g.ny + tile - 1) / tile) * ((g.nz + tile - 1) / tile)),
                      (unsigned)g.nx);
      kernel<<<grid, tile * tile, 0, st>>>(a_.acc, a_.d_dirs + d0, nd, g.nx, g.ny, g.nz, a_.med,
                                           f[0], f[1], f[2], f[3], f[4], f[5], a_.gh, a_.comp);
    };
    const bool wide = (int64_t)((g.ny + 31) / 32) * ((g.nz + 31) / 32) * g.nx >= 512;
    if (g_kahan)
      wide ? sums(art_gh_kernel<true, 32>, 32) : sums(art_gh_kernel<true, 16>, 16);
    else
      wide ? sums(art_gh_kernel<false, 32>, 32) : sums(art_gh_kernel<false, 16>, 16);
    A_OK(hipGetLastError());
    A_OK(hipEventRecord(a_.ev[3], st));
    A_OK(hipEventSynchronize(a_.ev[3]));
    float m0 = 0.0f, m1 = 0.0f;
    A_OK(hipEventElapsedTime(&m0, a_.ev[1], a_.ev[2]));
    A_OK(hipEventElapsedTime(&m1, a_.ev[2], a_.ev[3]));
    trace_ms += m0;
    gh_ms += m1;
  }
  const float r_n_ang = (float)(1.0e0 / nang);
  art_gh_sum_kernel<<<nb, 256, 0, st>>>(dmesh, nc, a_.gh, r_n_ang);
  A_OK(hipGetLastError());
  unsigned long long ncross = 0;
  A_OK(hipMemcpyAsync(&ncross, a_.ncross, sizeof ncross, hipMemcpyDeviceToHost, st));
  A_OK(hipStreamSynchronize(st));
  g_dstats.ndir = (uint64_t)nang;
  g_dstats.ncross = ncross;
  g_dstats.ms_trace = trace_ms;
  g_dstats.ms_gh = gh_ms;
  g_dstats.ms_total = now_ms() - t_start;
}

void free_diffuse_gpu(struct cuda_diffuse_param* cd, struct cuda_param* this_cuda) {
  (void)this_cuda;
  for (void* p : {(void*)a_.d_dirs, (void*)a_.med, (void*)a_.acc, (void*)a_.gh,
                  (void*)a_.comp, (void*)a_.ncross, (void*)a_.medT})
    if (p) (void)hipFree(p);
  a_.d_dirs = nullptr;
  a_.med = nullptr;
  a_.acc = nullptr;
  a_.medT = nullptr;
  a_.gh = a_.comp = nullptr;
  a_.ncross = nullptr;
  a_.dirs.clear();
  a_.ncell = 0;
  a_.batch = 0;
  if (cd) cd[0].rmesh = nullptr;
}

}  // extern "C"
