// One FP64 solve across compute units: the forward with four lanes per cell,
// and the adjoint.
//
// A solve on its own is bound by the latency of its steps: a sweep is a chain
// of nx + ny anti-diagonals, and the strip kernel's wave issues every
// instruction of a cell for each of them (satt_strip.hip).  Here a wave owns a
// strip of 16 columns for the whole solve and its four rows of 16 lanes take
// one quadrant and one one-sided value of a cell each, (W,S) and W, (W,N) and
// N, (E,S) and S, (E,N) and E, of the reference's update
// (src/eikon_solver_2d.f90:910-1079).  What does not depend on tau is formed
// once per solve by the reference's expressions (k_quad_build), down to the
// reciprocals of the divisors, so that a step is one branch-free run of about
// 150 instructions with everything but tau loaded steps ahead; tau of the strip
// stays in LDS.  The values taken are the sequential loop's, bit for bit.
// The adjoint's update (:1392-1402) is too short to share: the four lanes of a
// cell do the same, on coefficients formed once per solve.
// MI355X, forward of a 401 x 343 solve (5 iterations) 24.4 -> 6.4 ms, of a 41^2
// one 1.70 -> 0.64; adjoint 8.7 -> 4.9 and 0.6 -> 0.36.
//
// Strips run on waves (workgroups) of their own and exchange edge columns
// through global memory, with no barrier.  In sweep s a strip needs, row by
// row, the upstream neighbour's facing column after s and the downstream
// neighbour's after s - 1; every strip writes both of its edge columns of
// every sweep.  A value travels as two 64-bit words of half its bits and the
// sweep's tag, each stored and loaded whole (relaxed atomics at device scope):
// a word that carries the expected tag is the value, so nothing is ordered
// by fences.  Two buffers by the sweep's parity suffice: a strip writes sweep
// s + 2 only after it has ended s + 1, which needed the neighbour's columns
// after s (downstream) or s + 1 (upstream) row by row, and the neighbour
// writes those after its last read of the columns of s.
//
// Every wait is for a wave of the same launch; all of them are resident
// together, as a launch has at most kQuadMaxStrips one-wave workgroups, unless
// other work holds the device.  A wait is bounded: past the bound the solve
// ends with kETeamWait, and the caller takes the strip kernel.  Any strip may
// be the one that gives up, in the wait for the last totals too, which the
// others may find complete: so each gives the status its own part.
#include "satt_div.h"
#include "satt_internal.h"
#include "satt_strip.h"

namespace satt {
namespace {

typedef unsigned long long u64;
constexpr int kCols = 16;      // columns of a strip
constexpr int kRec = 18;       // doubles of a lane's record of a cell (forward)
constexpr int kRecA = 8;       // of a cell's record (adjoint)
constexpr int kBatch = 8;      // rows of the edge columns fetched at once
// The step of a batch that fetches the next one's words, a load's latency
// before they are needed: a forward step takes 0.45 us, an adjoint step 0.35.
constexpr int kFetch = 5, kFetchA = 2;
constexpr int kAhead = 4;      // steps the records are loaded ahead
// Rows of tau kept past either end: a sweep runs whole batches, so its last
// step is at most ny + 21, and tau is read two steps ahead.
constexpr int kPadRows = 24;
constexpr int kQuadSpin = 1 << 20;  // polls of one wait, about a second

struct Quad {
  int nx, ny, ns;
  double *rec;    // forward [strip][row][lane][kRec], adjoint [strip][row][column][kRecA]
  double *t0;     // [row][nx]: T0, natural layout
  double *snap;   // [strip][row][kCols]
  u64 *chan;      // [parity][strip][side][row][2]
  u64 *conv;      // [parity][strip][4]: the iteration's sum and maximum
  int *stop;      // a wait ran out
  int quit;       // a strip that ends as if its last wait had run out, or -1
  double dx, dy;
};

__device__ __forceinline__ u64 word_of(unsigned tag, unsigned v) { return (u64)tag << 32 | v; }
__device__ __forceinline__ void put(u64 *p, u64 w) {
  __hip_atomic_store(p, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 get(const u64 *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned half_of(double v, int hi) {
  return hi ? (unsigned)__double2hiint(v) : (unsigned)__double2loint(v);
}
__device__ __forceinline__ double min2(double a, double b) {  // neither is NaN
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
// The value of the next column's lane within the row of 16 (FROM -1: column
// c - 1, +1: c + 1); `edge` where the strip has none.
template <int FROM>
__device__ __forceinline__ double from_column(double v, double edge) {
  constexpr int ctrl = FROM < 0 ? 0x111 : 0x101;  // row_shr:1 : row_shl:1
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(edge), __double2loint(v), ctrl, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(edge), __double2hiint(v), ctrl, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}
// The least over a cell's four lanes, in all of them.
__device__ __forceinline__ double cell_min(double v) {
  const unsigned lo = (unsigned)__double2loint(v), hi = (unsigned)__double2hiint(v);
  const auto a = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
  v = min2(__hiloint2double((int)b[0], (int)a[0]), __hiloint2double((int)b[1], (int)a[1]));
  const unsigned l2 = (unsigned)__double2loint(v), h2 = (unsigned)__double2hiint(v);
  const auto c = __builtin_amdgcn_permlane32_swap(l2, l2, false, false);
  const auto d = __builtin_amdgcn_permlane32_swap(h2, h2, false, false);
  return min2(__hiloint2double((int)d[0], (int)c[0]), __hiloint2double((int)d[1], (int)c[1]));
}

// T0 of every cell (natural layout), and the reference's 'source on the
// boundary' where a frozen cell lies there (:863-867); the item's tables are
// k_fwd_prep's.
__global__ __launch_bounds__(256) void k_quad_t0(const SlotDesc *sd, Quad Q) {
  const SlotDesc D = *sd;
  if (*D.status < 0) return;
  const int k = blockIdx.x * 256 + threadIdx.x, nx = Q.nx, ny = Q.ny;
  if (k >= nx * ny) return;
  const int i = k % nx, j = k / nx;
  const double *tail = D.aux + 3 * nx + ny;
  double t0, t0x, t0y;
  t0_cell_tab(D.g.sy[j], D.g.cy[j], D.aux[i], D.aux[nx + i], tail[1], tail[2], tail[0], t0, t0x, t0y);
  Q.t0[k] = t0;
  if (D.aux[2 * nx + i] != 0.0 && D.aux[3 * nx + j] != 0.0 &&
      (i == 0 || i == nx - 1 || j == 0 || j == ny - 1))
    *D.status = kESrcOnBoundary;
}

// The records of every cell's four lanes.  A candidate that the reference
// skips (at the grid's edge, in a frozen cell) and the columns past the grid
// get NaN in ff and dis, which no test accepts.
__global__ __launch_bounds__(256) void k_quad_build(const SlotDesc *sd, Quad Q, const double *pa,
                                                    const double *pb, const double *pc,
                                                    const double *pfun) {
  const SlotDesc D = *sd;
  if (*D.status < 0) return;
  const size_t e = blockIdx.x * (size_t)256 + threadIdx.x;
  const int nx = Q.nx, ny = Q.ny;
  if (e >= (size_t)Q.ns * ny * 64) return;
  const int lane = (int)(e & 63), q = lane >> 4, c = lane & 15;
  const int j = (int)((e >> 6) % (unsigned)ny), k = (int)((e >> 6) / (unsigned)ny);
  const int i = kCols * k + c;
  double *r = Q.rec + e * kRec;
  const double nan = __builtin_nan("");
  if (i >= nx) {
#pragma unroll
    for (int f = 0; f < kRec; ++f) r[f] = nan;
    return;
  }
  const size_t n = i + (size_t)nx * j;
  const double *tail = D.aux + 3 * nx + ny;
  double t0, t0x, t0y;
  t0_cell_tab(D.g.sy[j], D.g.cy[j], D.aux[i], D.aux[nx + i], tail[1], tail[2], tail[0], t0, t0x, t0y);
  const double ak = pa[n], bk = pb[n], ck = pc[n], fk = pfun[n];
  const double t0dx = t0 / D.g.dx, t0dy = t0 / D.g.dy;
  const bool west = q < 2, south = (q & 1) == 0;
  const bool hx = west ? i > 0 : i < nx - 1, hy = south ? j > 0 : j < ny - 1;
  const double px = west ? t0x + t0dx : t0x - t0dx, py = south ? t0y + t0dy : t0y - t0dy;
  const double ak2 = 2 * ak, bk2 = 2 * bk, ck2 = 2 * ck;
  const double A1 = ak * (px * px), B1 = bk * (py * py), C1 = ck2 * px;
  const double ea = A1 + B1 - C1 * py;
  const bool frozen = D.aux[2 * nx + i] != 0.0 && D.aux[3 * nx + j] != 0.0;
  r[0] = west ? -t0dx : t0dx;
  r[1] = south ? -t0dy : t0dy;
  r[2] = px;
  r[3] = py;
  r[4] = ak2 * px;
  r[5] = bk2 * py;
  r[6] = ak;
  r[7] = bk;
  r[8] = ck;
  r[9] = hx && hy && !frozen ? fk * fk : nan;
  r[10] = ea;
  r[11] = recip_of(2 * ea).r;
  // the lane's one-sided neighbour: W, N, S, E
  const bool isx = q == 0 || q == 3, has = (isx ? hx : hy) && !frozen;
  const bool plus = isx ? west : south;
  const double p = isx ? px : py, P = plus ? p : -p;
  const double dis = sqrt(fk * fk * ((isx ? bk : ak) / (ak * bk - ck * ck)));
  r[12] = isx ? t0dx : t0dy;
  r[13] = has ? dis : nan;
  r[14] = P;
  r[15] = recip_of(P).r;
  r[16] = has ? Q.t0[isx ? n + (west ? -1 : 1) : south ? n - nx : n + nx] : 0.0;
  r[17] = t0;
}

// The adjoint's records: a1p, a2m, b1p, b2m, delta, d and d's reciprocal; d = 0
// where the update gives 0 (:1394-1395) and on the grid's rim and past it,
// where the field stays 0.  delta: the source in the plus skew of the slot's
// coefficient fields, where k_adj_source put it.
__global__ __launch_bounds__(256) void k_quad_adj_build(const SlotDesc *sd, Quad Q,
                                                        const double *pa, const double *pb,
                                                        const double *pc) {
  const SlotDesc D = *sd;
  if (*D.status < 0) return;
  const size_t e = blockIdx.x * (size_t)256 + threadIdx.x;
  const int nx = Q.nx, ny = Q.ny;
  if (e >= (size_t)Q.ns * ny * kCols) return;
  const int c = (int)(e % kCols), j = (int)((e / kCols) % (unsigned)ny);
  const int i = kCols * (int)((e / kCols) / (unsigned)ny) + c;
  double o[5] = {0, 0, 0, 0, 0}, dl = 0;
  if (i >= 1 && i <= nx - 2 && j >= 1 && j <= ny - 2) {
    const double *T = D.T;
    const size_t n = i + (size_t)nx * j, W = n - 1, E = n + 1, S = n - nx, N = n + nx;
    adj_coef_v(T[n], T[W], T[E], T[S], T[N], T[W - nx], T[W + nx], T[E - nx], T[E + nx], pa[n],
               pa[W], pa[E], pb[n], pb[S], pb[N], pc[n], pc[W], pc[E], pc[S], pc[N], Q.dx, Q.dy, o);
    dl = D.skew[5 * D.sg.skew_elems() + skpos(0, i, j, D.sg.R)];
  }
  double *r = Q.rec + e * kRecA;
  r[0] = (o[0] + fabs(o[0])) / 2;
  r[1] = (o[1] - fabs(o[1])) / 2;
  r[2] = (o[2] + fabs(o[2])) / 2;
  r[3] = (o[3] - fabs(o[3])) / 2;
  r[4] = dl;
  r[5] = o[4];
  r[6] = o[4] == 0.0 ? 0.0 : recip_of(o[4]).r;
  r[7] = 0.0;
}

__global__ __launch_bounds__(256) void k_quad_clear(u64 *p, size_t n, int *stop) {
  const size_t k = blockIdx.x * (size_t)256 + threadIdx.x;
  if (k < n) p[k] = 0;
  if (k == 0) *stop = 0;
}

// One wave's strip.
struct Strip {
  Quad Q;
  int k, lane, q, c;
  double *tau;      // LDS: row j at tau[(j + kPadRows) * kCols]
  unsigned *edge;   // LDS: the batch's upstream and downstream values, 32 words
  int flip_x, flip_y;  // sign bit where the causality test asks for <= 0
};

// Poll until the word of every lane that needs one has its tag; false if the
// wait ran out.  p is valid in every lane.  Each round tests the word it has
// loaded, so that no load is in flight where the loop is left.
__device__ __forceinline__ bool poll(const Strip &S, const u64 *p, unsigned tag, bool need,
                                     u64 &w) {
  for (int spin = 0;; ++spin) {
    w = get(p);
    if (__all(!need || (unsigned)(w >> 32) == tag)) return true;
    if ((spin & 63) == 63 && __hip_atomic_load(S.Q.stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      return false;
    if (spin >= kQuadSpin) {
      __hip_atomic_store(S.Q.stop, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
  }
}

// One sweep of the strip, s = 1, 2, ...  MODE 1 records the snapshot, 2 sums
// and maximises |tau - snapshot|*T0 (ADJ: |Ta - snapshot|) into ss, sm.
template <int XD, int YD, int MODE, bool ADJ>
__device__ __forceinline__ bool quad_sweep(const Strip &S, unsigned s, double &ss, double &sm) {
  const Quad &Q = S.Q;
  const int ny = Q.ny, lane = S.lane, q = S.q, c = S.c;
  const int lag = XD > 0 ? c : kCols - 1 - c;
  const bool col = kCols * S.k + c < Q.nx;
  auto row_of = [&](int u) { return YD > 0 ? u : ny - 1 - u; };
  // the lane's word of a batch: lanes 0..15 the upstream neighbour's facing
  // column after this sweep, 16..31 the downstream one's after the last
  const int wi = (lane >> 1) & 7, wdn = lane >> 4;
  const int nb = wdn == 0 ? S.k - XD : S.k + XD;
  const bool has = wdn < 2 && nb >= 0 && nb < Q.ns;
  const unsigned wtag = wdn == 0 ? s + 1 : s;
  const int wside = (wdn == 0) == (XD > 0) ? 1 : 0, wpar = wdn == 0 ? (int)(s & 1) : (int)((s - 1) & 1);
  const u64 *wbase = Q.chan + (((size_t)wpar * Q.ns + (has ? nb : S.k)) * 2 + wside) * ny * 2 + (lane & 1);
  auto word_at = [&](int b, bool &need) {
    const int u = kBatch * b + wi - (wdn == 1 ? kCols - 1 : 0);
    need = has && u >= 0 && u < ny;
    return wbase + 2 * (size_t)row_of(min(max(u, 0), ny - 1));
  };
  auto fetch = [&](int b) {
    bool need;
    const u64 *p = word_at(b, need);
    return get(p);
  };
  u64 *pub = Q.chan + (((size_t)(s & 1) * Q.ns + S.k) * 2 + (c != 0)) * ny * 2 + (q & 1);
  const bool edge_lane = q < 2 && (c == 0 || c == kCols - 1);

  constexpr int kR = ADJ ? kRecA : kRec, kRowRecs = ADJ ? kCols : 64;
  const double *rec = Q.rec + ((size_t)S.k * ny * kRowRecs + (ADJ ? c : lane)) * kR;
  const Recip rdx = recip_of(Q.dx), rdy = recip_of(Q.dy);
  double *snap = Q.snap + (size_t)S.k * ny * kCols + c;
  struct Cell {
    double v[kR], snap;
  };
  auto load = [&](int t, Cell &x) {
    const unsigned j = (unsigned)min(max(row_of(t - lag), 0), ny - 1);
    const double2 *p = reinterpret_cast<const double2 *>(rec + (size_t)(j * (unsigned)(kRowRecs * kR)));
#pragma unroll
    for (int f = 0; f < kR / 2; ++f) {
      const double2 d = p[f];
      x.v[2 * f] = d.x;
      x.v[2 * f + 1] = d.y;
    }
    if (MODE == 2) x.snap = snap[(size_t)j * kCols];
  };
  double *tau = S.tau + c;
  auto tau_at = [&](int t) { return tau[(row_of(t - lag) + kPadRows) * kCols]; };
  double acc_s = 0, acc_m = 0;
  Cell cell[kBatch];
  // the first words ahead of the records, as in the loop: the wait counts
  // there hold for both
  u64 w = fetch(0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int t = 0; t < kAhead; ++t) {
    load(t, cell[t]);
    __builtin_amdgcn_sched_barrier(0);
  }
  double tprev = 0, cur = tau_at(0), nxt = tau_at(1);
  const int nbatch = (ny + kCols - 1 + kBatch - 1) / kBatch;
  for (int b = 0; b < nbatch; ++b) {
    {
      bool need;
      const u64 *p = word_at(b, need);
      // the test of the words in flight stands outside the polling loop, whose
      // own loads would make it wait for every load of the records too
      if (!__all(!need || (unsigned)(w >> 32) == wtag) && !poll(S, p, wtag, need, w)) return false;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the last batch's have been read
    if (lane < 32) S.edge[lane] = (unsigned)w;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const double *ev = reinterpret_cast<const double *>(S.edge);
#pragma unroll
    for (int o = 0; o < kBatch; ++o) {
      const int t = kBatch * b + o;
      Cell &x = cell[o];
      load(t + kAhead, cell[(o + kAhead) % kBatch]);
      if (o == (ADJ ? kFetchA : kFetch)) w = fetch(b + 1);
      const double eu = ev[o], ed = ev[kBatch + o], ahead = tau_at(t + 2);
      const int u = t - lag, j = row_of(u);
      const bool act = u >= 0 && u < ny;
      // the neighbours: new values upwind, the last sweep's downwind
      const double xu = from_column<-XD>(tprev, eu), xd = from_column<XD>(nxt, ed);
      const double tW = XD > 0 ? xu : xd, tE = XD > 0 ? xd : xu;
      const double tS = YD > 0 ? tprev : nxt, tN = YD > 0 ? nxt : tprev;
      const double *v = x.v;
      double tnew;
      if constexpr (ADJ) {
        const Recip rd{v[5], v[6]};
        const double ex = tW * v[0] - tE * v[1], ey = tS * v[2] - tN * v[3];
        tnew = quot(v[4] + (quot(ex, rdx) + quot(ey, rdy)), rd);
        // below the quotients' range; a tiny term beside a larger one does
        // not move its sum
        if (fabs(tnew) < 1e-200 && v[5] != 0)
          tnew = (v[4] + (ex / Q.dx + ey / Q.dy)) / v[5];
        tnew = v[5] == 0 ? 0.0 : tnew;
      } else {
        const double tx = q < 2 ? tW : tE, ty = (q & 1) == 0 ? tS : tN;
        const double px = v[2], py = v[3], ak = v[6], bk = v[7], ck = v[8], ck2 = 2 * ck;
        const double qx = v[0] * tx, qy = v[1] * ty;
        const double eb = v[4] * qx + v[5] * qy - ck2 * (px * qy + py * qx);
        const double ec = ak * (qx * qx) + bk * (qy * qy) - ck2 * qx * qy - v[9];
        const double delta = eb * eb - 4 * v[10] * ec;
        const Recip re{2 * v[10], v[11]};
        const double sq = root_of(delta);  // NaN below 0: no test accepts its roots
        double best = cur;
        auto take = [&](double tt) {
          const double Tx = px * tt + qx, Ty = py * tt + qy;
          const double chx = ak * Tx - ck * Ty, chy = bk * Ty - ck * Tx;
          const double gx = __hiloint2double(__double2hiint(chx) ^ S.flip_x, __double2loint(chx));
          const double gy = __hiloint2double(__double2hiint(chy) ^ S.flip_y, __double2loint(chy));
          best = gx >= 0 && gy >= 0 && tt < best ? tt : best;
        };
        take(quot(-eb + sq, re));
        take(quot(-eb - sq, re));
        {
          const double tn = q == 0 || q == 3 ? tx : ty, Qn = v[12] * tn;
          const Recip rp{v[14], v[15]};
          const double Tn = tn * v[16], lim = tn * 0.5;
          auto side = [&](double tt) {
            best = tt * v[17] >= Tn && tt > lim && tt < best ? tt : best;
          };
          side(quot(Qn + v[13], rp));
          side(quot(Qn - v[13], rp));
        }
        tnew = cell_min(best);
      }
      tau[(j + kPadRows) * kCols] = tnew;
      if (edge_lane && act) put(pub + 2 * (size_t)j, word_of(s + 1, half_of(tnew, q)));
      if (MODE == 1 && q == 0 && act) snap[(size_t)j * kCols] = cur;
      if (MODE == 2) {
        const double d = ADJ ? fabs(tnew - x.snap) : fabs(tnew - x.snap) * v[ADJ ? 0 : 17];
        if (q == 0 && act && col) {
          acc_s += d;
          acc_m = d > acc_m ? d : acc_m;
        }
      }
      tprev = tnew;
      cur = nxt;
      nxt = ahead;
    }
  }
  if (MODE == 2) {
    for (int off = 32; off > 0; off >>= 1) {
      acc_s += __shfl_xor(acc_s, off, 64);
      const double o = __shfl_xor(acc_m, off, 64);
      acc_m = o > acc_m ? o : acc_m;
    }
    ss = acc_s;
    sm = acc_m;
  }
  return true;
}

template <bool ADJ>
__global__ __launch_bounds__(64, 1) void k_quad(const SlotDesc *sd, Quad Q) {
  constexpr int kMaxIter = ADJ ? kAdjMaxIter : kFwdMaxIter;
  constexpr double kTol = ADJ ? kAdjTol : kFwdTol;
  extern __shared__ double lds[];
  const SlotDesc D = *sd;
  if (*D.status < 0) return;  // the setup failed
  Strip S;
  S.Q = Q;
  S.k = blockIdx.x;
  S.lane = threadIdx.x;
  S.q = S.lane >> 4;
  S.c = S.lane & 15;
  S.edge = reinterpret_cast<unsigned *>(lds);
  S.tau = lds + 16;
  S.flip_x = S.q < 2 ? 0 : INT_MIN;
  S.flip_y = (S.q & 1) == 0 ? 0 : INT_MIN;
  const int nx = Q.nx, ny = Q.ny, i0 = kCols * S.k;
  // tau's start (:859-872) or Ta's (:1373-1380), and the edge columns as of
  // sweep 0
  for (int e = S.lane; e < (ny + 2 * kPadRows) * kCols; e += 64) {
    const int j = e / kCols - kPadRows, i = i0 + e % kCols;
    const bool in = j >= 0 && j < ny && i < nx;
    if (ADJ)
      S.tau[e] = j > 0 && j < ny - 1 && i > 0 && i < nx - 1 ? 100.0 : 0.0;
    else
      S.tau[e] = in && D.aux[2 * nx + i] != 0.0 && D.aux[3 * nx + j] != 0.0 ? 1.0 : 10.0;
  }
  __syncthreads();
  for (int e = S.lane; e < 4 * ny; e += 64) {
    const int hi = e & 1, side = (e >> 1) & 1, j = e >> 2;
    const double v = S.tau[(j + kPadRows) * kCols + (side ? kCols - 1 : 0)];
    put(Q.chan + (((size_t)S.k * 2 + side) * ny + j) * 2 + hi, word_of(1, half_of(v, hi)));
  }
  unsigned s = 0;
  int iter = 1;
  bool conv = false, ok = true;
  for (; iter <= kMaxIter; ++iter) {
    double sum = 0, mx = 0;
    ok = quad_sweep<1, 1, 1, ADJ>(S, ++s, sum, mx) && quad_sweep<1, -1, 0, ADJ>(S, ++s, sum, mx) &&
         quad_sweep<-1, 1, 0, ADJ>(S, ++s, sum, mx) && quad_sweep<-1, -1, 2, ADJ>(S, ++s, sum, mx);
    if (!ok) break;
    // every strip's sum and maximum to every strip, added in strip order
    u64 *mine = Q.conv + ((size_t)(iter & 1) * Q.ns + S.k) * 4;
    if (S.lane < 4)
      put(mine + S.lane, word_of((unsigned)iter, half_of(S.lane < 2 ? sum : mx, S.lane & 1)));
    double tot = 0, top = 0;
    for (int k0 = 0; k0 < Q.ns && ok; k0 += 16) {  // 16 strips of four words at a time
      const int kk = min(k0 + (S.lane >> 2), Q.ns - 1);
      const u64 *p = Q.conv + ((size_t)(iter & 1) * Q.ns + kk) * 4 + (S.lane & 3);
      u64 w;
      ok = poll(S, p, (unsigned)iter, true, w);
      for (int m = 0; m < 16 && k0 + m < Q.ns; ++m) {
        const double a = __hiloint2double(__shfl((int)w, 4 * m + 1, 64), __shfl((int)w, 4 * m, 64));
        const double b = __hiloint2double(__shfl((int)w, 4 * m + 3, 64), __shfl((int)w, 4 * m + 2, 64));
        tot = tot + a;
        top = b > top ? b : top;
      }
    }
    if (!ok) break;
    const double l1 = ADJ ? tot / (double)(nx * ny) : tot / (double)nx / (double)ny;
    if (fabs(l1) < kTol && top < kTol) {
      conv = true;
      break;
    }
  }
  if (!conv) iter = kMaxIter;
  if (S.k == Q.quit) ok = false;
  __syncthreads();
  if (ok)
    for (int e = S.lane; e < ny * kCols; e += 64) {
      const int j = e / kCols, i = i0 + e % kCols;
      const size_t n = i + (size_t)nx * j;
      const double v = S.tau[e + kPadRows * kCols];
      if (i < nx) (ADJ ? D.Ta : D.T)[n] = ADJ ? v : v * Q.t0[n];
    }
  // kOk as uploaded, else the least of what the strips say: one that gave up
  // has left its columns unwritten, whatever strip 0 found
  if (S.lane == 0) {
    if (!ok)
      atomicMin(D.status, kETeamWait);
    else if (S.k == 0 && !conv)
      atomicCAS(D.status, kOk, kWMaxIter);
    if (S.k == 0) D.iters[ADJ ? 1 : 0] = iter;
  }
}

constexpr size_t quad_lds(int ny) { return (16 + (size_t)(ny + 2 * kPadRows) * kCols) * 8; }

}  // namespace

bool quad_fits(int nx, int ny) {
  return (nx + kCols - 1) / kCols <= kQuadMaxStrips && quad_lds(ny) <= kTeamLdsMax;
}

namespace {
struct QuadLayout {
  size_t rec, t0, snap, chan, conv, stop, total;
  QuadLayout(int nx, int ny, bool adj) {
    const size_t ns = (nx + kCols - 1) / kCols, n = ns * ny;
    size_t at = 0;
    auto take = [&](size_t bytes) {
      const size_t o = at;
      at = (at + bytes + 255) & ~(size_t)255;
      return o;
    };
    rec = take(n * (adj ? kCols * kRecA : 64 * kRec) * 8);
    t0 = take((size_t)nx * ny * 8);
    snap = take(n * kCols * 8);
    chan = take(n * 8 * 8);  // [2][ns][2][ny][2]
    conv = take(ns * 8 * 8);
    stop = take(4);
    total = at;
  }
};
}  // namespace

size_t quad_scratch_bytes(int nx, int ny, bool adj) { return QuadLayout(nx, ny, adj).total; }

namespace {
Quad quad_of(const SlotDesc &D, bool adj, void *scratch, int quit) {
  const QuadLayout L(D.g.nx, D.g.ny, adj);
  char *b = static_cast<char *>(scratch);
  Quad Q;
  Q.nx = D.g.nx;
  Q.ny = D.g.ny;
  Q.ns = (Q.nx + kCols - 1) / kCols;
  Q.rec = reinterpret_cast<double *>(b + L.rec);
  Q.t0 = reinterpret_cast<double *>(b + L.t0);
  Q.snap = reinterpret_cast<double *>(b + L.snap);
  Q.chan = reinterpret_cast<u64 *>(b + L.chan);
  Q.conv = reinterpret_cast<u64 *>(b + L.conv);
  Q.stop = reinterpret_cast<int *>(b + L.stop);
  Q.quit = quit;
  Q.dx = D.g.dx;
  Q.dy = D.g.dy;
  return Q;
}
// The words of the edge columns and of the totals start without a tag.
void quad_clear(hipStream_t s, const Quad &Q) {
  const size_t words = (size_t)(Q.conv - Q.chan) + 8 * (size_t)Q.ns;
  hipLaunchKernelGGL(k_quad_clear, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, s, Q.chan,
                     words, Q.stop);
}
}  // namespace

void launch_fwd_quad(hipStream_t s, const SlotDesc *sd, const GroupDims &gd, const SlotDesc &D,
                     const PeriodFields &pf, void *scratch, int quit) {
  const Quad Q = quad_of(D, false, scratch, quit);
  const size_t lanes = (size_t)Q.ns * Q.ny * 64;
  launch_fwd_prep(s, sd, gd);
  quad_clear(s, Q);
  hipLaunchKernelGGL(k_quad_t0, dim3((unsigned)((Q.nx * Q.ny + 255) / 256)), dim3(256), 0, s, sd, Q);
  hipLaunchKernelGGL(k_quad_build, dim3((unsigned)((lanes + 255) / 256)), dim3(256), 0, s, sd, Q,
                     pf.a, pf.b, pf.c, pf.fun);
  hipLaunchKernelGGL(k_quad<false>, dim3((unsigned)Q.ns), dim3(64), quad_lds(Q.ny), s, sd, Q);
}

void launch_adj_quad(hipStream_t s, const SlotDesc *sd, const GroupDims &gd, const SlotDesc &D,
                     const PeriodFields &pf, void *scratch, int quit) {
  const Quad Q = quad_of(D, true, scratch, quit);
  const size_t SE = D.sg.skew_elems(), cells = (size_t)Q.ns * Q.ny * kCols;
  launch_zero(s, D.skew + 5 * SE, SE * 8);
  launch_adj_source(s, sd, gd, 0, false);
  quad_clear(s, Q);
  hipLaunchKernelGGL(k_quad_adj_build, dim3((unsigned)((cells + 255) / 256)), dim3(256), 0, s, sd, Q,
                     pf.a, pf.b, pf.c);
  hipLaunchKernelGGL(k_quad<true>, dim3((unsigned)Q.ns), dim3(64), quad_lds(Q.ny), s, sd, Q);
}

}  // namespace satt
