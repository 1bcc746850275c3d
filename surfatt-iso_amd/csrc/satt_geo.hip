// Geographic smoothing, gradient, topographic metric and the steepest-
// descent update: the model-side steps on either side of the solver path.
//
//   gaussian_smooth_geo_2  src/shared/utils.f90:1194-1223
//   gradient_2_geo         src/shared/utils.f90:1118-1160
//   get_topo metric        src/grid.f90:114-123,137-141; dip angle src/topo.f90:123-130
//   optimize + steepest_descent  src/tomo2d.f90:203-251
//
// Smoothing.  Output cell (i,j) is sum(w*data)/sum(w) over the window
// |i'-i| <= hx, |j'-j| <= hy(j), with w = exp(-delta^2/(2 sigma^2)) and
// delta the haversine distance in degrees.  On the reference's grids (uniform
// axes from arange) a weight depends on the row pair (j, j') and the column
// offset |i'-i| only, up to the rounding of lon(i')-lon(i): the weights of a
// row pair are evaluated once per column offset, not per (cell, node), and
// the per-node work is one fused multiply-add in FP64 on register operands
// (k_smooth_geo2).  The latitude term sin((lat-lat')/2)^2 is the reference's
// per pair; the longitude term is sin(dlon_k/2)^2 with dlon_k = lon(k)-lon(0).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <type_traits>

#include "satt_internal.h"

namespace satt {
namespace {

// src/shared/shared_par.f90:11-15: pi is a default-real literal
constexpr double kGeoPi = (double)3.14159265359f;
constexpr double kGeoRadius = 6371.0;
constexpr double kGeoDeg2Rad = kGeoPi / 180.0;
constexpr double kGeoKm2Deg = 1.0 / (6371.0 * kGeoPi / 180.0);

// s2[k] = sin(dlon_k * 0.5)**2, dlon_k = (lon(k) - lon(0)) * deg2rad
__global__ void k_geo_s2(const double *lon, int nx, double *s2) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nx) return;
  const double s = sin((lon[k] - lon[0]) * kGeoDeg2Rad * 0.5);
  s2[k] = s * s;
}

// The lat-lon haversine a = sin^2(theta/2) of a window node as the exponent
// of its weight, theta^2 * kap / 4 with kap = 4 (R km2deg)^2 / (2 sigma^2).
// SMALL: theta^2 = 4 asin(sqrt(a))^2 by its power series, 4a (1 + a/3 +
// 8a^2/45 + ...), eight terms: for a <= kSmallA the next one is below 1e-18
// of the sum.  It takes 9 operations where the atan2 and the two square
// roots of the general form take about 150, which had been a quarter of the
// kernel's arithmetic at wide windows.
constexpr double kSmallA = 1.0 / 128;
template <bool SMALL>
__device__ __forceinline__ double geo_weight(double a, double kap) {
  if constexpr (SMALL) {
    double p = 512.0 / 12870;
    p = __builtin_fma(p, a, 1024.0 / 21021);
    p = __builtin_fma(p, a, 128.0 / 2079);
    p = __builtin_fma(p, a, 128.0 / 1575);
    p = __builtin_fma(p, a, 4.0 / 35);
    p = __builtin_fma(p, a, 8.0 / 45);
    p = __builtin_fma(p, a, 1.0 / 3);
    p = __builtin_fma(p, a, 1.0);
    return exp(-(kap * (a * p)));
  } else {
    const double t = atan2(sqrt(a), sqrt(1.0 - a));
    return exp(-(kap * (t * t)));
  }
}

// num[r][c] += sum over k = 0 .. n - 1, ascending, of w[k*RW + r] *
// d(c + DIR*k), for a lane's C consecutive cells c and RR output rows; d is
// the staged data row at the lane's first cell.  The cells' data slide
// through a ring of C+3 registers: per offset a lane reads one datum and RR
// weights from LDS for RR*C products.  Reads run up to C+2 elements past the
// last one used (kPadC below).
template <int RR, int RW, int C, int DIR>
__device__ __forceinline__ void smooth_side(const double *w, const double *d, int n,
                                            double (&num)[RR][C]) {
  constexpr int K = C + 3;
  const double *p = DIR > 0 ? d : d + (C - 1);
  double a[RR][C] = {}, v[K], wq[2][RR];  // wq: this offset's weights, the next one's
#pragma unroll
  for (int x = 0; x < K; ++x) v[x] = p[DIR * x];
#pragma unroll
  for (int r = 0; r < RR; ++r) wq[0][r] = w[r];
  static_assert(K % 2 == 0, "wq alternates");
  auto at = [&](int u, int k) {
    const double vn = p[DIR * (k + u + K)];
#pragma unroll
    for (int r = 0; r < RR; ++r) wq[(u + 1) & 1][r] = w[(k + u + 1) * RW + r];
#pragma unroll
    for (int r = 0; r < RR; ++r)
#pragma unroll
      for (int e = 0; e < C; ++e) {
        const int c = DIR > 0 ? e : C - 1 - e;
        a[r][c] = __builtin_fma(wq[u & 1][r], v[(u + e) % K], a[r][c]);
      }
    v[u] = vn;
  };
  int k = 0;
  for (; k + K <= n; k += K) {
#pragma unroll
    for (int u = 0; u < K; ++u) at(u, k);
  }
  const int rem = n - k;
#pragma unroll
  for (int u = 0; u < K - 1; ++u)
    if (u < rem) at(u, k);
#pragma unroll
  for (int r = 0; r < RR; ++r)
#pragma unroll
    for (int c = 0; c < C; ++c) num[r][c] = num[r][c] + a[r][c];
}

// Orders a wave's LDS accesses for the compiler (the hardware runs one wave's
// LDS instructions in order, and every wave here uses its own part of it).
__device__ __forceinline__ void lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The smoothing is sum(w*data)/sum(w): k_smooth_norm forms the denominators
// of each distinct sigma, k_smooth_geo2 the numerators and the quotients.
// Both take the window rows j' in S waves (wave j' mod S, added in wave
// order) and a row's offsets in ascending distance, one side after the other:
//   num += sum_{k>=1} w[k] d(i+k), then + sum_{k>=1} w[k] d(i-k), then + w[0] d(i)
//   den += P[min(hx, nx-1-i)],     then + P[min(hx, i)],          then + w[0]
// with P[m] the running sums of w[1..m]: on a field of ones the numerator takes the
// denominator's own operations, so that constants are kept exactly.
constexpr int kMaxSplit = 4;

// The latitude terms of a wave's window rows, 64 of them at a time, one per
// lane: cos(lat') and, for each output row, sin((lat - lat')/2)^2.
template <int RW>
struct LatTerms {
  double c1 = 0, sdl[RW] = {};
  int left = 0;
  // the terms of row jj (the wave's rows are S apart): cos(lat)cos(lat') and
  // the squared sine of every output row
  __device__ __forceinline__ void at(const GeoSmooth &P, int jj, int S, int lane,
                                     const double (&lat)[RW], const double (&cl)[RW],
                                     double (&cc)[RW], double (&sd)[RW]) {
    if (left == 0) {
      const int jl = jj + S * lane;
      const double latj = P.lat[jl < P.ny ? jl : P.ny - 1];
      c1 = cos(latj * kGeoDeg2Rad);
#pragma unroll
      for (int r = 0; r < RW; ++r) {
        const double sl = sin((lat[r] - latj) * kGeoDeg2Rad * 0.5);
        sdl[r] = sl * sl;
      }
      left = 64;
    }
    const int src = 64 - left--;
    const double cj = __shfl(c1, src, 64);
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      sd[r] = __shfl(sdl[r], src, 64);
      cc[r] = cl[r] * cj;
    }
  }
};

// kap, finite where 2 sigma^2 is not 0 (it overflows below sigma = 6e-153): the
// weight of the cell itself is then 1, as the quotient of its distance gives it.
__device__ __forceinline__ double geo_kap(double sig) {
  const double two = 2.0 * (sig * sig);
  const double kap = 4.0 * (kGeoRadius * kGeoKm2Deg) * (kGeoRadius * kGeoKm2Deg) / two;
  return two > 0.0 ? fmin(kap, 1.7976931348623157e308) : kap;
}
// the wave sw's first window row at or after n1
__device__ __forceinline__ int first_row(int n1, int sw, int S) {
  return n1 + ((sw - n1) % S + S) % S;
}

// Denominators of RN output rows, a tile of 64*kNormC columns, one sigma per
// workgroup of S waves.  A wave evaluates its window rows' weights, one lane
// per output row turns them into running sums, and every lane adds the two
// its columns need.
constexpr int kNormC = 7;
template <int RN, bool SMALL>
__global__ __launch_bounds__(64 * kMaxSplit) void k_smooth_norm(GeoSmooth P, int lds_wave) {
  extern __shared__ double lds[];
  const int lane = threadIdx.x & 63;
  const int S = blockDim.x >> 6, sw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j0 = RN * blockIdx.x, f = P.norm_field[blockIdx.y], i0 = 64 * kNormC * blockIdx.z;
  const int nx = P.nx, ny = P.ny;
  const int hx = P.hx[f], hxe = hx < nx - 1 ? hx : nx - 1;
  const int ld = (hxe + 1) | 1;  // odd: the running-sum lanes read different banks
  double *wl = lds + (size_t)sw * lds_wave;
  const double kap = geo_kap(P.sigma[f]);
  int lo[RN], hi[RN], n1 = ny, n2 = -1;
  double latr[RN], cr[RN];
#pragma unroll
  for (int r = 0; r < RN; ++r) {
    const int j = j0 + r < ny ? j0 + r : ny - 1, hy = P.hy[(size_t)f * ny + j];
    lo[r] = j - hy > 0 ? j - hy : 0;
    hi[r] = j + hy < ny - 1 ? j + hy : ny - 1;
    n1 = lo[r] < n1 ? lo[r] : n1;
    n2 = hi[r] > n2 ? hi[r] : n2;
    latr[r] = P.lat[j];
    cr[r] = cos(latr[r] * kGeoDeg2Rad);
  }
  double den[RN][kNormC] = {};
  LatTerms<RN> T;
  for (int jj = first_row(n1, sw, S); jj <= n2; jj += S) {
    double cc[RN], sd[RN], w0[RN];
    T.at(P, jj, S, lane, latr, cr, cc, sd);
    lds_order();  // the previous row's sums have been read
    for (int k = lane; k <= hxe; k += 64) {
      const double s2 = P.s2[k];
#pragma unroll
      for (int r = 0; r < RN; ++r)
        wl[r * ld + k] = geo_weight<SMALL>(__builtin_fma(s2, cc[r], sd[r]), kap);
    }
    lds_order();
#pragma unroll
    for (int r = 0; r < RN; ++r) w0[r] = wl[r * ld];
    if (lane < RN) {
      double *w = wl + lane * ld, s = 0.0;
      w[0] = 0.0;
      int k = 1;
      for (; k + 8 <= hxe + 1; k += 8) {
        double x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = w[k + u];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          s = s + x[u];
          w[k + u] = s;
        }
      }
      for (; k <= hxe; ++k) {
        s = s + w[k];
        w[k] = s;
      }
    }
    lds_order();
#pragma unroll
    for (int c = 0; c < kNormC; ++c) {
      const int q = i0 + 64 * c + lane, i = q < nx ? q : nx - 1;
      const int e = hxe < nx - 1 - i ? hxe : nx - 1 - i, w = hxe < i ? hxe : i;
#pragma unroll
      for (int r = 0; r < RN; ++r)
        if (jj >= lo[r] && jj <= hi[r])
          den[r][c] = ((den[r][c] + wl[r * ld + e]) + wl[r * ld + w]) + w0[r];
    }
  }
  __syncthreads();
  double *out = P.den + (size_t)blockIdx.y * nx * ny;
  for (int r = 0; r < RN; ++r) {
    // the waves' sums of one row at a time, through LDS
#pragma unroll
    for (int c = 0; c < kNormC; ++c) lds[(sw * kNormC + c) * 64 + lane] = den[0][c];
#pragma unroll
    for (int q = 0; q + 1 < RN; ++q)
#pragma unroll
      for (int c = 0; c < kNormC; ++c) den[q][c] = den[q + 1][c];
    __syncthreads();
    for (int c = sw; c < kNormC; c += S) {
      double b = lds[c * 64 + lane];
      for (int q = 1; q < S; ++q) b = b + lds[(q * kNormC + c) * 64 + lane];
      const int i = i0 + 64 * c + lane;
      if (i < nx && j0 + r < ny) out[(size_t)(j0 + r) * nx + i] = b;
    }
    __syncthreads();
  }
}

// Numerators and quotients.  One workgroup of S waves per (2G output rows,
// tile of C*64/G columns, field); the 64/G lanes of a group own two output
// rows, a lane C cells of each.  For each of its window rows a wave evaluates
// the weights of its output rows once, stages data row j' (0 outside the
// grid), and every lane accumulates its cells (smooth_side).
// Per offset a lane takes 2C fused multiply-adds and reads 24 bytes of LDS;
// the form before it (a thread per column of two rows) took a product and two
// sums a node and 1.5 LDS reads of 8 bytes.  With C = 7 and one group the
// reads still bound it: C = 13 and two groups halve them per node.
// MI355X, 401^2 at 0.005 degrees: smoothing of 20 kernels at sigma 0.2 8.1 ms
// and 0.2 for the denominators, against 33.6, the metric's 20 periods 6.3 and
// 1.1 ms against 29.9; at the 65 TFLOP/s that independent FP64 multiply-adds
// reach they are 4.4 and 3.2 ms.  What is left is issue: the vector units are
// busy two thirds of the cycles, a quarter of that with the weights, the
// zeroing and adding of the sums and the staging of each row, at a clock
// that falls to 1.85 GHz under it.  The window rows are split over waves because the widest of a
// call's windows are 200 times the narrowest one's work: a wave doing one
// alone ran 5 ms.
// C is odd: lanes C doubles apart then read 32 different LDS bank pairs.
constexpr size_t kLdsHalf = 80 * 1024;  // of a CU's LDS: two workgroups a CU
constexpr size_t kCus = 256;
constexpr int kPadC = 2;  // columns staged past the window on either side, in units of C
// LDS doubles of one wave: the weights, the staged row
size_t smooth_lds_doubles(int G, int C, int hxe) {
  return (size_t)2 * G * (hxe + 1) + 64 / G * C + 2 * ((size_t)hxe + (size_t)kPadC * C);
}
template <int G, int C, bool SMALL>
__global__ __launch_bounds__(64 * kMaxSplit, 2) void k_smooth_geo2(GeoSmooth P, int lds_wave) {
  static_assert(C % 2 == 1 && C >= 3, "C + 2 elements are read ahead");
  constexpr int RW = 2 * G, kLanes = 64 / G, kTile = kLanes * C;
  extern __shared__ double lds[];
  const int lane = threadIdx.x & 63, g = lane / kLanes;
  const int S = blockDim.x >> 6, sw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j0 = RW * blockIdx.x, f = P.order[blockIdx.y], i0 = kTile * blockIdx.z;
  const int nx = P.nx, ny = P.ny;
  const int hx = P.hx[f], hxe = hx < nx - 1 ? hx : nx - 1;
  const int span = hxe + kPadC * C;  // staged columns i0 - span .. i0 + kTile - 1 + span
  double *wl = lds + (size_t)sw * lds_wave, *dl = wl + (size_t)RW * (hxe + 1);
  const double *data = P.data + (P.ndata == 1 ? 0 : (size_t)f * nx * ny);
  const double kap = geo_kap(P.sigma[f]);
  int n1 = ny, n2 = -1;
  double latr[RW], cr[RW];
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    const int j = j0 + r < ny ? j0 + r : ny - 1, hy = P.hy[(size_t)f * ny + j];
    n1 = j - hy < n1 ? j - hy : n1;
    n2 = j + hy > n2 ? j + hy : n2;
    latr[r] = P.lat[j];
    cr[r] = cos(latr[r] * kGeoDeg2Rad);
  }
  n1 = n1 > 0 ? n1 : 0;
  n2 = n2 < ny - 1 ? n2 : ny - 1;
  // the window rows of the lane's two output rows
  int lo[2], hi[2];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int j = j0 + 2 * g + r, hy = j < ny ? P.hy[(size_t)f * ny + j] : 0;
    lo[r] = j < ny ? j - hy : ny;
    hi[r] = j < ny ? j + hy : -1;
  }
  for (int q = lane; q < kTile + 2 * span; q += 64) dl[q] = 0.0;
  const int c0 = i0 - span > 0 ? i0 - span : 0;
  const int c1 = i0 + kTile + span < nx ? i0 + kTile + span : nx;
  const int ic = i0 + (lane % kLanes) * C;  // the lane's first cell
  const double *dt = dl + span + (lane % kLanes) * C, *wg = wl + 2 * g;
  double num[2][C] = {};
  LatTerms<RW> T;
  for (int jj = first_row(n1, sw, S); jj <= n2; jj += S) {
    double cc[RW], sd[RW];
    T.at(P, jj, S, lane, latr, cr, cc, sd);
    lds_order();  // the previous row's weights and data have been read
    for (int k = lane; k <= hxe; k += 64) {
      const double s2 = P.s2[k];
#pragma unroll
      for (int r = 0; r < RW; ++r)
        wl[k * RW + r] = geo_weight<SMALL>(__builtin_fma(s2, cc[r], sd[r]), kap);
    }
    const double *row = data + (size_t)jj * nx;
    for (int q = c0 + lane; q < c1; q += 64) dl[q - i0 + span] = row[q];
    lds_order();
    const bool in0 = jj >= lo[0] && jj <= hi[0], in1 = jj >= lo[1] && jj <= hi[1];
    if (in0 && in1) {
      smooth_side<2, RW, C, 1>(wg + RW, dt + 1, hxe, num);
      smooth_side<2, RW, C, -1>(wg + RW, dt - 1, hxe, num);
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int c = 0; c < C; ++c) num[r][c] = __builtin_fma(wg[r], dt[c], num[r][c]);
    } else if (in0 || in1) {  // a window row of one of the two output rows
      const double *w1 = in0 ? wg : wg + 1;
      double one[1][C];
#pragma unroll
      for (int c = 0; c < C; ++c) one[0][c] = in0 ? num[0][c] : num[1][c];
      smooth_side<1, RW, C, 1>(w1 + RW, dt + 1, hxe, one);
      smooth_side<1, RW, C, -1>(w1 + RW, dt - 1, hxe, one);
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const double v = __builtin_fma(w1[0], dt[c], one[0][c]);
        num[0][c] = in0 ? v : num[0][c];
        num[1][c] = in0 ? num[1][c] : v;
      }
    }
  }
  // the waves' sums, added in wave order: [wave][2C][64] in LDS
  __syncthreads();
  if (sw > 0) {
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int c = 0; c < C; ++c)
        lds[((size_t)(sw - 1) * 2 * C + r * C + c) * 64 + lane] = num[r][c];
  }
  __syncthreads();
  if (sw > 0) return;
  double *out = P.out + (size_t)f * nx * ny;
  const double *den = P.den + (size_t)P.norm_of[f] * nx * ny;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int j = j0 + 2 * g + r;
    if (j >= ny) continue;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      double a = num[r][c];
      for (int q = 0; q < S - 1; ++q) a = a + lds[((size_t)q * 2 * C + r * C + c) * 64 + lane];
      if (ic + c < nx) out[(size_t)j * nx + ic + c] = a / den[(size_t)j * nx + ic + c];
    }
  }
}

// gradient_2_geo of field p (natural layout) at cell k; cosd of each row
// comes from the host.
__device__ __forceinline__ void grad_geo_cell(const GeoGrad &G, const double *f, int i, int j,
                                              double &tx, double &ty) {
  const int nx = G.nx, ny = G.ny;
  const size_t k = (size_t)i + (size_t)nx * j;
  const double cl = G.cosd_lat[j];
  const double gfx = i > 0 ? f[k] - f[k - 1] : 0.0;
  const double gbx = i < nx - 1 ? f[k + 1] - f[k] : 0.0;
  const double gfy = j > 0 ? f[k] - f[k - nx] : 0.0;
  const double gby = j < ny - 1 ? f[k + nx] - f[k] : 0.0;
  if (i == 0) {
    tx = gbx / (kGeoRadius * (G.lon[1] - G.lon[0]) * kGeoDeg2Rad * cl);
  } else {
    const double dxi = kGeoRadius * (G.lon[i] - G.lon[i - 1]) * kGeoDeg2Rad * cl;
    tx = i == nx - 1 ? gfx / dxi : (gfx + gbx) / (2 * dxi);
  }
  if (j == 0) {
    ty = gby / (kGeoRadius * (G.lat[1] - G.lat[0]) * kGeoDeg2Rad);
  } else {
    const double dyj = kGeoRadius * (G.lat[j] - G.lat[j - 1]) * kGeoDeg2Rad;
    ty = j == ny - 1 ? gfy / dyj : (gfy + gby) / (2 * dyj);
  }
}

// One thread per (field p fastest, cell): the period-major outputs are
// written contiguously.
__global__ void k_gradient_geo2(GeoGrad G, int nf, const double *f_nat, double *tx,
                                double *ty) {
  const size_t N = (size_t)G.nx * G.ny;
  const size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (t >= N * nf) return;
  const int p = (int)(t % nf);
  const size_t k = t / nf;
  double gx, gy;
  grad_geo_cell(G, f_nat + (size_t)p * N, (int)(k % G.nx), (int)(k / G.nx), gx, gy);
  tx[t] = gx;
  ty[t] = gy;
}

__global__ void k_topo_metric(GeoGrad G, int nf, const double *sm_nat, double *m11, double *m12,
                              double *m22, double *angle) {
  const size_t N = (size_t)G.nx * G.ny;
  const size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (t >= N * nf) return;
  const int p = (int)(t % nf);
  const size_t k = t / nf;
  double gx, gy;
  grad_geo_cell(G, sm_nat + (size_t)p * N, (int)(k % G.nx), (int)(k / G.nx), gx, gy);
  const double den = 1 + gx * gx + gy * gy;
  m11[t] = (1 + gy * gy) / den;
  m22[t] = (1 + gx * gx) / den;
  m12[t] = -(gx * gy / den);
  if (angle) angle[t] = atan(sqrt(gx * gx + gy * gy)) * (180.0 / 3.14159265358979323846);
}

__global__ void k_pm_to_nat(size_t N, int nf, const double *pm, double *nat) {
  const size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  const int p = blockIdx.y;
  if (k >= N) return;
  nat[(size_t)p * N + k] = pm[(size_t)p + (size_t)nf * k];
}

// max |v| over n values: per-block maxima, then one block over those
constexpr int kMaxBlocks = 1024;
__global__ __launch_bounds__(256) void k_absmax_part(const double *v, size_t n, double *part) {
  __shared__ double sh[256];
  double m = 0;
  for (size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x; k < n;
       k += (size_t)gridDim.x * blockDim.x) {
    const double a = fabs(v[k]);
    m = a > m ? a : m;
  }
  sh[threadIdx.x] = m;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) sh[threadIdx.x] = sh[threadIdx.x + s] > sh[threadIdx.x]
                                                    ? sh[threadIdx.x + s] : sh[threadIdx.x];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// part[nparts] = max over part[0..nparts-1], one block
__global__ __launch_bounds__(256) void k_absmax_final(double *part, int nparts) {
  __shared__ double sh[256];
  double m = 0;
  for (int b = threadIdx.x; b < nparts; b += blockDim.x) m = part[b] > m ? part[b] : m;
  sh[threadIdx.x] = m;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) sh[threadIdx.x] = sh[threadIdx.x + s] > sh[threadIdx.x]
                                                    ? sh[threadIdx.x + s] : sh[threadIdx.x];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[nparts] = sh[0];
}

// svel = svel*(1 + updatemax*gradient), gradient = ker/maxval(abs(ker))
__global__ void k_sd_update(size_t n, const double *ker, const double *mx, double updatemax,
                            double *svel) {
  const size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (k >= n) return;
  svel[k] = svel[k] * (1 + updatemax * (ker[k] / *mx));
}

// out = base*(1 + update), update = updatemax*ker/maxval(abs(ker)) with the
// product formed first, as prepare_fwd_linesearch writes it
// (src/acqui_2d.f90:179-180); out may be base
__global__ void k_ls_model(size_t n, const double *base, const double *ker, const double *mx,
                           double updatemax, double *out) {
  const size_t k = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (k >= n) return;
  out[k] = base[k] * (1 + updatemax * ker[k] / *mx);
}

dim3 flat_grid(size_t n) { return dim3((unsigned)((n + 255) / 256)); }

}  // namespace

void launch_geo_s2(hipStream_t s, const double *lon, int nx, double *s2) {
  hipLaunchKernelGGL(k_geo_s2, flat_grid((size_t)nx), dim3(256), 0, s, lon, nx, s2);
}

// The waves of a workgroup: as many as leave two workgroups a CU the LDS of
// the tile that takes the most columns (one group, C = 13).
SmoothForm smooth_form(int hx, double a) {
  int S = kMaxSplit;
  while (S > 1 && S * smooth_lds_doubles(1, 13, hx) * sizeof(double) > kLdsHalf) S >>= 1;
  return {S, a <= kSmallA};
}

namespace {

template <int RN>
void norm_launch(hipStream_t s, const GeoSmooth &P, const SmoothPart &part) {
  const int S = part.form.split;
  const size_t wave = (size_t)RN * ((part.hx_max + 1) | 1);
  const size_t lds = S * std::max(wave, (size_t)64 * kNormC) * sizeof(double);
  const dim3 grid((unsigned)((P.ny + RN - 1) / RN), (unsigned)part.norms,
                  (unsigned)((P.nx + 64 * kNormC - 1) / (64 * kNormC)));
  if (part.form.series)
    hipLaunchKernelGGL((k_smooth_norm<RN, true>), grid, dim3(64 * S), lds, s, P, (int)wave);
  else
    hipLaunchKernelGGL((k_smooth_norm<RN, false>), grid, dim3(64 * S), lds, s, P, (int)wave);
}

template <int G, int C>
void tile_launch(hipStream_t s, const GeoSmooth &P, const SmoothPart &part) {
  const int S = part.form.split;
  const size_t wave = smooth_lds_doubles(G, C, part.hx_max);
  const size_t sums = (size_t)(S - 1) * 2 * C * 64;
  const size_t lds = std::max(S * wave, sums) * sizeof(double);
  constexpr int kTile = 64 / G * C;
  const dim3 grid((unsigned)((P.ny + 2 * G - 1) / (2 * G)), (unsigned)part.fields,
                  (unsigned)((P.nx + kTile - 1) / kTile));
  if (part.form.series)
    hipLaunchKernelGGL((k_smooth_geo2<G, C, true>), grid, dim3(64 * S), lds, s, P, (int)wave);
  else
    hipLaunchKernelGGL((k_smooth_geo2<G, C, false>), grid, dim3(64 * S), lds, s, P, (int)wave);
}

int ceil_div(int a, int b) { return (a + b - 1) / b; }

// The tile of G lane groups and C columns a lane.  Where one workgroup a CU
// does, the narrowest C, in one group or two: the call is then as long as a
// workgroup, and its weights are of 2G rows.  Else the one whose columns cover
// a row with the fewest idle lanes, at equal cover the wider C and fewer groups.
// More than one group where the weights of 2G rows and the staged row leave
// two workgroups a CU.
// MI355X, numerators in us, windows of 25 / 121 columns, (2,13) is G = 2, C = 13:
//   401^2, 1 field    (1,9)  40 / 235   (2,9)  41 / 238   (2,13)  56 / 314   (4,9)  48 / 265
//   401^2, 20 fields  (1,9) 282 / 2916  (2,9) 304 / 2985  (2,13) 221 / 2186  (4,9) 305 / 2531
//   300^2, 20 fields  (1,9) 196 / 1927  (2,11) 136 / 1227 (2,13) 160 / 1456  (4,9) 218 / 1635
//   200^2, 1 field    (1,9)  33 / 213   (2,9)  37 / 222   (4,9)   46 / 255   (4,13) 59 / 333
//   200^2, 20 fields  (1,9) 129 / 1143  (2,9)  84 / 714   (4,9)  105 / 742   (4,13) 76 / 541
//   100^2, 20 fields  (1,9)  66 / 504   (2,9)  43 / 288   (4,9)   50 / 248   (4,13) 64 / 333
void part_launch(hipStream_t s, const GeoSmooth &P, const SmoothPart &part) {
  const int S = part.form.split;
  auto fits = [&](int G, int C) {
    return G == 1 || S * smooth_lds_doubles(G, C, part.hx_max) * sizeof(double) <= kLdsHalf;
  };
  int bg = 0, bc = 9;
  for (int G : {1, 2})
    if (bg == 0 && fits(G, 9) &&
        (size_t)ceil_div(P.ny, 2 * G) * part.fields * ceil_div(P.nx, 64 / G * 9) <= kCus)
      bg = G;
  if (bg == 0) {
    int cover = INT_MAX;
    for (int C : {13, 11, 9})
      for (int G : {1, 2, 4}) {
        const int tile = 64 / G * C, n = ceil_div(P.nx, tile) * tile;
        if (fits(G, C) && n < cover) {
          cover = n;
          bg = G;
          bc = C;
        }
      }
  }
  auto go = [&](auto c) {
    constexpr int C = decltype(c)::value;
    if (bg == 1)
      tile_launch<1, C>(s, P, part);
    else if (bg == 2)
      tile_launch<2, C>(s, P, part);
    else
      tile_launch<4, C>(s, P, part);
  };
  if (bc == 13)
    go(std::integral_constant<int, 13>{});
  else if (bc == 11)
    go(std::integral_constant<int, 11>{});
  else
    go(std::integral_constant<int, 9>{});
}

}  // namespace

void launch_smooth_geo2(hipStream_t s, GeoSmooth P, const SmoothPart *parts, int nparts) {
  double *den = P.den;
  for (int q = 0; q < nparts; ++q) {
    const SmoothPart &part = parts[q];
    GeoSmooth N = P;  // the sums of the part's own sigmas
    N.den = den;
    // Rows a workgroup: few where one a CU does, else four, two where the
    // weights of four leave less than two workgroups a CU.  MI355X, windows of
    // 121 columns, 4 / 2 / 1 rows: one sigma on 200^2 95 / 69 / 56 us, on 401^2
    // 98 / 70 / 89, 20 sigmas on 401^2 518 / 686 / 1135 (8 rows: 199, 202, 856).
    const size_t rows = (size_t)P.ny * part.norms * ceil_div(P.nx, 64 * kNormC);
    if (rows <= kCus)
      norm_launch<1>(s, N, part);
    else if (rows <= 2 * kCus ||
             (size_t)part.form.split * 4 * (part.hx_max + 2) * sizeof(double) > kLdsHalf)
      norm_launch<2>(s, N, part);
    else
      norm_launch<4>(s, N, part);
    part_launch(s, P, part);
    den += (size_t)part.norms * P.nx * P.ny;
    P.order += part.fields;
    P.norm_field += part.norms;
  }
}

void launch_gradient_geo2(hipStream_t s, const GeoGrad &G, int nf, const double *f_nat,
                          double *tx_pm, double *ty_pm) {
  hipLaunchKernelGGL(k_gradient_geo2, flat_grid((size_t)G.nx * G.ny * nf), dim3(256), 0, s, G,
                     nf, f_nat, tx_pm, ty_pm);
}

void launch_topo_metric(hipStream_t s, const GeoGrad &G, int nf, const double *sm_nat,
                        double *m11, double *m12, double *m22, double *angle) {
  hipLaunchKernelGGL(k_topo_metric, flat_grid((size_t)G.nx * G.ny * nf), dim3(256), 0, s, G, nf,
                     sm_nat, m11, m12, m22, angle);
}

void launch_pm_to_nat(hipStream_t s, size_t N, int nf, const double *pm, double *nat) {
  hipLaunchKernelGGL(k_pm_to_nat, dim3((unsigned)((N + 255) / 256), (unsigned)nf), dim3(256), 0,
                     s, N, nf, pm, nat);
}

int absmax_parts(size_t n) { return (int)std::min<size_t>(kMaxBlocks, (n + 255) / 256); }

const double *launch_absmax(hipStream_t s, size_t n, const double *v, double *part) {
  const int nb = absmax_parts(n);
  hipLaunchKernelGGL(k_absmax_part, dim3((unsigned)nb), dim3(256), 0, s, v, n, part);
  hipLaunchKernelGGL(k_absmax_final, dim3(1), dim3(256), 0, s, part, nb);
  return part + nb;
}

void launch_sd_update(hipStream_t s, size_t n, const double *ker, double updatemax, double *svel,
                      double *part) {
  const double *mx = launch_absmax(s, n, ker, part);
  hipLaunchKernelGGL(k_sd_update, flat_grid(n), dim3(256), 0, s, n, ker, mx, updatemax, svel);
}

void launch_ls_model(hipStream_t s, size_t n, const double *base, const double *ker,
                     const double *mx, double updatemax, double *out) {
  hipLaunchKernelGGL(k_ls_model, flat_grid(n), dim3(256), 0, s, n, base, ker, mx, updatemax, out);
}

}  // namespace satt
