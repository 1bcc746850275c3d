// Strip-pipeline kernels (satt_strip.hip): geometry of the skewed layouts
// and the launch entry points used by the batched plan.
#pragma once
#include "../../include/satt.h"
#include "satt_internal.h"

namespace satt {

constexpr int kPF = 6;  // per-period skew fields: a, b, c, fun, dis_x, dis_y
constexpr int kFF = 3;  // per-item forward skew fields: T0, T0x, T0y
constexpr int kAF = 6;  // per-item adjoint skew fields: a1, a2, b1, b2, d, delta
// The FP32 strip passes address a set of up to kPF fields of one skew with
// 32-bit byte offsets: plans in mixed precision keep a skew within this.
constexpr size_t kMaxSkewElems32 = 0xFFFFFFFFull / (kPF * sizeof(float));

// Per-slot scratch of the batched path, in units of one skewed field (SE
// doubles) and one natural field (N doubles).
//   skew fields 0..11 : adjoint coefficients (a1,a2,b1,b2,d,delta) x 2 skews;
//                       the forward uses them first for T0,T0x,T0y x 2 skews
//                       (0..5), tau plus (6), tau minus (7), snapshot (8)
//   skew fields 12,13 : travel time T, plus and minus skew (forward output)
//   skew fields 14..16: Ta plus, Ta minus, snapshot (adjoint)
//   natural 0..3      : T, Ta, Td (density adjoint), delta source
// The mixed mode keeps the forward's float fields from double skew 9 (free
// until the output T skews are written).
constexpr int kSlotSkews = 17;
constexpr int kSlotNat = 4;
enum : int { kSkTauP = 6, kSkTauM = 7, kSkSnapF = 8, kSkTP = 12, kSkTM = 13,
             kSkTaP = 14, kSkTaM = 15, kSkSnapA = 16 };
enum : int { kNatT = 0, kNatTa = 1, kNatTd = 2, kNatDelta = 3 };
// The mixed mode adds 6 skewed fields per slot: the adjoint's float fields
// (coefficients k0..kN in both skews, which both its FP32 phase and its FP64
// polish read, Ta plus and minus, snapshot) from double skew 16.  Of the
// forward's FP64 fields it keeps T0 (0, 3), tau and the snapshot: its passes
// read the period fields and T0x, T0y in float.
constexpr int kSlotSkewsMixed = 23;
constexpr int kSkA32 = 16;

// Per-slot forward tables (aux): sin and cos of (xx - x0) per column, the
// frozen flags of the columns and the rows, then fun0, sin(y0), cos(y0).
inline int aux_len(int nx, int ny) { return (3 * nx + ny + 4 + 1) & ~1; }

// Doubles of one slot's scratch: its skewed fields, kSlotNat natural fields
// and the forward tables, rounded up to 256 bytes.
inline size_t slot_doubles(int nx, int ny, int slot_skews) {
  const size_t n = (size_t)slot_skews * make_skew_geom(nx, ny).skew_elems() +
                   (size_t)kSlotNat * nx * ny + (size_t)aux_len(nx, ny);
  return (n + 31) & ~(size_t)31;
}

// Sweep stages of the strip kernels; each has its own team size: the FP32
// forward, the FP64 forward (polish, or the whole FP64 solve), the FP32
// adjoint and the FP64 adjoint.
enum { kStageFwd32 = 0, kStageFwd64 = 1, kStageAdj32 = 2, kStageAdj64 = 3, kStages = 4 };

// Sizes of a launch group, for the grids of the element-wise kernels, and
// the waves per item of its strip kernels in each stage.
struct GroupDims {
  int count;        // slots
  size_t max_se;    // largest skewed field
  size_t max_n;     // largest grid
  int max_nxy;      // largest nx or ny
  int max_ny = 0, max_ns = 0;  // largest ny and strip count
  int waves[kStages] = {1, 1, 1, 1};  // waves per item (a team; at most kMaxTeam)
  int depth[kStages] = {2, 2, 2, 2};  // steps the sweeps fetch their operands ahead
};

// The deeper of the two prefetch depths the sweep kernels are built with
// (the other is two steps).  Fetching further ahead hides more memory
// latency where few waves share a SIMD, at the price of one operand set of
// registers per step.
constexpr int kDeepPrefetch = 4;

// XCDs (chiplets, each with its own L2) of the device: workgroup w of a
// launch runs on XCD w mod kXcds.
constexpr int kXcds = 8;

// Waves per item of the strip kernels: each strip of a sweep goes to one
// wave of the item's team, the next strip's wave following at least one
// strip width behind.  More waves cut an item's latency on wide grids; one
// wave per item is the throughput form when items fill the device.
constexpr int kMaxTeam = 8;
constexpr size_t kTeamLdsMax = 160 * 1024;  // a gfx950 workgroup's LDS
// one wave's two FP64 edge channels of SATT_MAX_NY rows fill it
static_assert(2 * 8 * (size_t)SATT_MAX_NY <= kTeamLdsMax, "SATT_MAX_NY exceeds the LDS");
// The largest team (<= want) of a sweep stage whose LDS (edge channels of
// the stage's value type) fits for grids up to ny rows, ns strips.
int team_waves(int want, int ny, int ns, int stage);
// Measures each sweep stage's fastest team size and prefetch depth on the
// plan's own inputs and leaves the plan set to them (satt_api.hip).
int tune_plan_shapes(satt_plan *P, satt_tune_result &r);

// T0, T0x, T0y of one cell (src/eikon_solver_2d.f90:845-857) from the
// row's sin/cos of the latitude and the column's sin/cos of the longitude
// difference: the expressions of t0_cell_s, with the same operand values.
__device__ __forceinline__ void t0_cell_tab(double sy, double cy, double sdx, double cdx,
                                            double sy0, double cy0, double fun0, double &T0,
                                            double &T0x, double &T0y) {
  const double t = sy * sy0 + cy * cy0 * cdx;
  double tc = t < 1.0 ? t : 1.0;
  tc = tc > -1.0 ? tc : -1.0;
  T0 = acos(tc) * kREarth * fun0;
  if (T0 == 0) {
    T0x = 0;
    T0y = 0;
  } else {
    const double s = sqrt(1 - t * t);
    T0x = -(1.0 / s * cy * cy0 * (-1.0) * sdx * kREarth * fun0);
    T0y = -(1.0 / s * (cy * sy0 - sy * cy0 * cdx) * kREarth * fun0);
  }
}

// Face coefficients of one interior cell (src/eikon_solver_2d.f90:1348-1370)
// from T at the 3x3 neighbourhood and the metric at the faces, and the sweep
// denominator d = (a2p-a1m)/dx + (b2p-b1m)/dy (:1392), stored as 0 where
// abs(d) < eps (:1394-1395).
__device__ __forceinline__ void adj_coef_v(double Tk, double TW, double TE, double TS, double TN,
                                           double TWS, double TWN, double TES, double TEN,
                                           double ak, double aW, double aE, double bk, double bS,
                                           double bN, double ck, double cW, double cE, double cS,
                                           double cN, double dx, double dy, double *out) {
  const double a1 = -((Tk - TW) / dx * (ak + aW) / 2) + (TN - TS + TWN - TWS) / (4 * dy) * (ck + cW) / 2;
  const double a2 = -((TE - Tk) / dx * (aE + ak) / 2) + (TEN - TES + TN - TS) / (4 * dy) * (cE + ck) / 2;
  const double b1 = -((Tk - TS) / dy * (bk + bS) / 2) + (TE - TW + TES - TWS) / (4 * dx) * (ck + cS) / 2;
  const double b2 = -((TN - Tk) / dy * (bN + bk) / 2) + (TEN - TWN + TE - TW) / (4 * dx) * (cN + ck) / 2;
  const double a1m = (a1 - fabs(a1)) / 2, a2p = (a2 + fabs(a2)) / 2;
  const double b1m = (b1 - fabs(b1)) / 2, b2p = (b2 + fabs(b2)) / 2;
  const double d = (a2p - a1m) / dx + (b2p - b1m) / dy;
  out[0] = a1; out[1] = a2; out[2] = b1; out[3] = b2;
  out[4] = fabs(d) < kAdjEps ? 0.0 : d;
}

__device__ __forceinline__ size_t skidx(int c, int r, int l, int R) {
  return ((size_t)c * R + r) * 64 + l;
}

// Position of cell (i, j) in skew sk (0 plus, 1 minus).  For 64 lanes of one
// strip and a common offset (di, dj) the positions of (i+di, j+dj) are one
// contiguous run, except for the lane that crosses into the next strip.
__device__ __forceinline__ size_t skpos(int sk, int i, int j, int R) {
  const int c = i >> 6, l = i & 63;
  const int r = sk == 0 ? j + l : j - l + 63;
  return skidx(c, r, l, R);
}

// One FP64 solve across compute units (satt_quad.hip): the forward, four lanes
// per cell, on the slot's tables and the natural-layout fields a, b, c, fun of
// pf, and the adjoint on its natural T, its receivers and a, b, c.  T or Ta,
// status and iteration count as launch_fwd_strip's and launch_adj_strip's, in
// natural layout only and without the mask.  A status of kETeamWait (a wave of
// the launch was not running) leaves the field unset.  D: the slot's
// descriptor sd on the host.  For grids that quad_fits; scratch:
// quad_scratch_bytes.  The slot's status is kOk before the launch.  quit: a
// strip that gives up at its end (for tests), or -1.
constexpr int kQuadMaxStrips = 64;  // waves of a launch: a quarter of the CUs
bool quad_fits(int nx, int ny);
size_t quad_scratch_bytes(int nx, int ny, bool adj);
void launch_fwd_quad(hipStream_t s, const SlotDesc *sd, const GroupDims &gd, const SlotDesc &D,
                     const PeriodFields &pf, void *scratch, int quit);
void launch_adj_quad(hipStream_t s, const SlotDesc *sd, const GroupDims &gd, const SlotDesc &D,
                     const PeriodFields &pf, void *scratch, int quit);

// Batched kernels over the slots of a launch group (satt_strip.hip); all
// asynchronous on `s`.  Forward: setup (per-item tables, then T0 skews and
// the tau init, one thread per element), then the sweeps: k_fwd_strip
// (FP64), or k_fwd_mixed32 (FP32 phase) followed by k_fwd_polish (FP64 to
// the reference's stop rule).
void launch_fwd_prep(hipStream_t s, const SlotDesc *sd, const GroupDims &gd);  // the tables only
void launch_fwd_setup(hipStream_t s, const SlotDesc *sd, const GroupDims &gd, bool mixed);
void launch_fwd_strip(hipStream_t s, const SlotDesc *sd, const GroupDims &gd);
void launch_fwd_mixed32(hipStream_t s, const SlotDesc *sd, const GroupDims &gd);
void launch_fwd_polish(hipStream_t s, const SlotDesc *sd, const GroupDims &gd);
// Adjoint (which 0) or density adjoint (which 1): setup (the coefficients
// without the source -- FP64 with the Ta init, and in the mixed mode the
// float set too -- then the delta source from the rhs, accumulated in
// natural layout and scattered into the coefficient fields), then the
// sweeps: k_adj_strip (FP64), or k_adj_mixed32 followed by k_adj_polish
// (one FP64 iteration).  Output Ta (which 0) or Td (which 1), masked.
void launch_adj_source(hipStream_t s, const SlotDesc *sd, const GroupDims &gd, int which,
                       bool mixed);  // the delta source only
void launch_adj_setup(hipStream_t s, const SlotDesc *sd, const GroupDims &gd, int which,
                      bool mixed);
void launch_adj_strip(hipStream_t s, const SlotDesc *sd, const GroupDims &gd, int which);
void launch_adj_mixed32(hipStream_t s, const SlotDesc *sd, const GroupDims &gd, int which);
void launch_adj_polish(hipStream_t s, const SlotDesc *sd, const GroupDims &gd, int which);
// T of every slot from natural layout into both skews, where the adjoint's
// setup reads it (a forward run writes them itself).
void launch_time_skew(hipStream_t s, const SlotDesc *sd, const GroupDims &gd);
// Each slot's own kernel Ta/svel**2 into its `kern` field (when set).
void launch_item_kernel(hipStream_t s, const SlotDesc *sd, const GroupDims &gd);
// Per-period skewed fields of one grid (out32: the same in float, or null).
void launch_period_skew(hipStream_t s, const Grid &g, const SkewGeom &sg, int np,
                        const PeriodFields &pf, double *out, float *out32);

}  // namespace satt
