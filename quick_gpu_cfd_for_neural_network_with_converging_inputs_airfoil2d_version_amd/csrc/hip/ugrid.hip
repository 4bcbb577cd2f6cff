// ugrid.hip -- batched first-order Euler solver on a shared tensor-product grid (gfx950, FP64):
// the device side of ugrid_hip.h, replacing the reference's legacy CUDA backend
// (src/euler2d_cuda.cu:153-447 kernels, :530-708 driver).
//
// Design.  The reference launches, per RK stage, separate primitive, x-flux, y-flux, collect,
// RK-combine and admissibility kernels with a host round trip per stage (flag copy) and per
// step (smax copy, dt upload).  Here one kernel per RK stage does all of it and the step
// control lives on the device:
//   * a wave owns a strip of 62 columns x `rows` rows of one case.  Lane k holds column
//     i0 - 1 + k, so lanes 0 and 63 are the strip's x halo; each lane computes the flux of the
//     face west of its cell (left state from lane k - 1 by a cross-lane shuffle) and takes its
//     east flux from lane k + 1, so every x face of the strip is evaluated once by 64 lanes at
//     a time.  The wave marches north through its rows, keeping the previous row's primitives,
//     x-residual and y-face flux in registers, so each y face is evaluated once and a cell's
//     state is read once per stage (plus one halo row per strip).  No LDS, no barriers.
//   * boundary ghosts are never materialised: a halo lane or row outside the domain reads the
//     mapped interior cell (periodic wrap, transmissive clamp, reflect mirror) and negates the
//     normal velocity for a reflection -- bit for bit the primitives of the reference's filled
//     ghost (negation is exact).
//   * the RK update, the admissibility test of the candidate and, in the last stage, the
//     candidate's wave-speed bound for the next step's dt are fused into the same pass.  A
//     one-block kernel after the last stage reduces the strips' bounds and commits or rejects the
//     trial for all cases: t += dt, step counters, buffer swap (U[cur] and the other buffer
//     alternate, so no accept copy), next dt from the bound, or dt halving and the 12-retry limit.
//   * a trial is four launches; the host replays a graph of several trials and polls the
//     control record between replays.
// The arithmetic of every formula follows the reference's GPU kernels operation for operation
// and this file is compiled without FMA contraction, so results are bitwise those of the CPU
// restatement of that backend.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <string>
#include <utility>
#include <vector>

#include "ugrid_hip.h"

namespace ugrid {

constexpr int kLanes = 64;
constexpr int kStripCells = kLanes - 2;  // columns a strip updates
constexpr int kWaves = 4;                // strips per block
constexpr int kThreads = kLanes * kWaves;
constexpr int kGhosts = 2;
constexpr int kXcds = 8;
constexpr int kMaxRetries = 12;
constexpr int kDecide = 1024;      // threads of the decision kernels that reduce the strips' partials
// Cases up to which strips store their maxima for the decision kernel instead of one 64-bit
// atomicMax per strip on the case's word: device-scope atomics on one word take about 9 ns each
// (4 cases of 400 x 311, 2184 strips: last stage 44 us, of which 20 us were its atomics).  The decision
// takes longer for it (8 cases of 1024 x 1024, 6120 strips: 5.6 -> 9.6 us of a 590 us step).  With more
// cases the words are many and the reduction's table would not fit LDS.
constexpr int kPartCases = 1024;
// Steps a first-stage pre-check tries on a cut grid (the body bench needs about six halvings a step).
constexpr int kPrechecks = 8;
enum : int { BC_PERIODIC = 0, BC_TRANSMISSIVE = 1, BC_REFLECT = 2 };
enum : int { RUNNING = -1 };
// Backward-Euler phases of a physical step (each kernel of the replayed sequence acts only in its
// phase; the one-block decision kernels move the phase).
enum : int { PH_BOUND = 0, PH_COPY = 1, PH_UPDATE = 2, PH_RETRY = 3 };
// Why a backward-Euler run stopped with 2, 3 or 4.
enum : int { WHY_NONE = 0, WHY_INITIAL = 1, WHY_PSEUDO = 2, WHY_DEFECT = 3, WHY_MAXITER = 4, WHY_DT = 5 };

// Step control of a batch (one record, device memory).
struct Control {
  double tend;
  long long maxsteps;  // steps allowed in the current run call
  long long steps;     // accepted in the current run call
  long long nsteps, nreject;
  long long events;    // decisions taken (every commit, rejection, phase change): progress
  int status;      // RUNNING, or the run's result 0 / 1 / 2 / 3 / 4 (also 0 before the first run)
  int bad;         // a stage found a nonphysical candidate cell (this trial)
  int retries;     // rejections of the current step
  int cur;         // B[cur] holds the accepted state
  int ghost_from;  // download ghosts: 0 as uploaded, 1 boundary fill of B[cur], 2 of B[cur ^ 1]
  // backward Euler
  int phase, iter, pretries, qbuf, reason;
  unsigned pre_mask;  // SSP-RK3 on a cut grid: halvings of the trial's step that the pre-check refuses
  double pseudo;   // pseudo CFL of the current physical step
  long long updates, iretries, checks;
  double initial_defect, final_defect, tolerance;
};

struct Grid {
  int nx, ny, mx, my, ncase;
  int rows;            // rows per strip
  int strips_x, strips_y, strips;
  int blocks;          // blocks that own strips (the launch is padded to a multiple of 8)
  int bc[4];
  int ausm;
  double gamma, cfl, dt_fixed;
  size_t plane;        // mx * my
  const double* dx;    // mx widths (ghosts included)
  const double* dy;    // my
  const double* rdx;   // recip() of every width
  const double* rdy;
  int plain;           // widths, gamma - 1 and AUSM+-up's reference Mach numbers are plain (see `recip`)
  const double* mco;   // ncase
  // State buffers: B[0] and B[1] alternate as accepted state and RK candidate, B[2] holds the
  // second RK stage; backward Euler rotates all three (accepted state, iterate, candidate).
  double* B[3];
  double* t;
  double* dt;          // step of the running trial
  double* dt_out;      // last accepted step
  unsigned long long* smax;  // per case: bit pattern of the largest wave-speed bound (non-negative)
  // Per strip: the largest bound (last RK stage) or scaled defect (backward Euler) of its cells, which
  // the one-block decision kernel reduces per case.  With more than kPartCases cases the strips
  // report to smax / norm by atomics instead.
  unsigned long long* part;
  int use_part;
  unsigned long long* norm;  // per case: bit pattern of the largest scaled defect (backward Euler)
  double* initial;           // per case: first defect norm of the physical step
  double pseudo0, rtol, atol;
  int maxiter;
  // Cut cells (has_cut): areas, 0 / 1 / 2 flags, apertures, wall vectors, SRD counts and
  // positions; SRD neighbourhoods as member lists, and the cells SRD rewrites with the
  // neighbourhoods each belongs to (ascending), so the sums run in one fixed order.
  int has_cut, nsmall, n_srd;
  const double* vol;
  const double* flag;
  const double* axl;
  const double* ayl;
  const double* wax;
  const double* way;
  const double* nbrcount;
  const double* smallpos;
  const double* svhat;
  const int* mem_off;
  const int* mem_idx;
  const int* srd_cell;
  const int* grp_off;
  const int* grp_idx;
  double* Qh;  // ncase x nsmall x 4 neighbourhood averages
  // One byte per plane cell for the stage kernels (so that they read the double arrays above only
  // where a value is needed): bit 0 solid (vol <= 0), bit 1 cut (flag != 0), bit 2 rewritten by
  // SRD (smallpos >= 0 or nbrcount != 1), bits 3-4 the west x face, bits 5-6 the south y face of
  // the cell: 0 aperture +0, 1 aperture equal to the full width (dy, dx; the builders store that
  // value for open faces), 2 another value (read from axl / ayl).
  const uint8_t* code;
  // The interior cut cells (plane indices, ascending): the first RK stage is tried on them alone
  // before the whole-grid pass (k_stage1_precheck).
  const int* pre_cell;
  int n_pre;
  Control* ctrl;
};

// A cell as its four faces see it: the primitives, and what both sides of every face would form
// from them again.  x and y faces exchange the roles of u and v, which no derived value notices
// (u^2 + v^2 is a commutative sum), and a reflection only negates a velocity.
//   HLLC:    a = sqrt(gamma p / r), q = sqrt(r), E = p / (gamma - 1) + r (u^2 + v^2) / 2,
//            H = (E + p) / r, e = E / r
//   AUSM+-up: a, H = E + p, e = the reciprocal of r that quotients by r share
struct Cell {
  double r, u, v, p, a, q, E, H, e;
};
struct Flux {
  double m, x, y, e;  // mass, x momentum, y momentum, energy
};

// ---------------------------------------------------------------------------------------------
// Quotients and square roots.  The kernels are bound by FP64 instruction issue, and most of it
// was IEEE division (38 a cell) and square root (10): the compiler's division is 12 instructions,
// of which seven (two range scalings, v_rcp_f64, two Newton steps) depend on the divisor alone.
// Quotients with a common divisor therefore share those (`recip`), and inside a plain range the
// scalings, which there multiply by one, are left out.  What is left are the compiler's own
// operations in its order, so the bits are those of n / d and sqrt(x); outside the plain range
// (PLAIN false) the compiler's division and square root are used.
//
// Plain (`plain_state`): density and pressure in (2^-100, 2^100), energy below 2^100, which bounds
// the velocities through p > 0; cell widths, gamma - 1 and AUSM+-up's reference Mach numbers likewise
// (Grid::plain).  Every divisor the kernels form is then a normal number in (2^-400, 2^400).  A
// numerator may be arbitrarily small where a velocity or a flux difference is (zero and rounding
// noise ahead of a wave): such quotients are formed of the numerator times 2^200 (`quot_scaled`),
// so that the remainder of the last step stays exact; the other small numerators are sums'
// negligible terms.
// ---------------------------------------------------------------------------------------------
constexpr double kPlainLow = 0x1p-100, kPlainHigh = 0x1p100;
constexpr double kScale = 0x1p200, kUnscale = 0x1p-200;

__device__ __forceinline__ double recip(double d) {
  double y = __builtin_amdgcn_rcp(d);
  y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
  return __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
}
// n / d with y = recip(d).
template <bool PLAIN>
__device__ __forceinline__ double quot(double n, double d, double y) {
  if (!PLAIN) return n / d;
  const double q = n * y;
  return __builtin_fma(__builtin_fma(-d, q, n), y, q);
}
template <bool PLAIN>
__device__ __forceinline__ double quot(double n, double d) {
  return quot<PLAIN>(n, d, PLAIN ? recip(d) : 0.0);
}
// 2^200 n / d for a numerator of any size.
__device__ __forceinline__ double quot_scaled(double n, double d, double y) { return quot<true>(n * kScale, d, y); }
template <bool PLAIN>
__device__ __forceinline__ double root(double x) {
  if (!PLAIN) return sqrt(x);
  double h = __builtin_amdgcn_rsq(x);
  double s = x * h;
  h = h * 0.5;
  const double e = __builtin_fma(-h, s, 0.5);
  s = __builtin_fma(s, e, s);
  h = __builtin_fma(h, e, h);
  s = __builtin_fma(__builtin_fma(-s, s, x), h, s);
  return __builtin_fma(__builtin_fma(-s, s, x), h, s);
}
__device__ __forceinline__ bool plain_state(double r, double p, double E) {
  return r > kPlainLow && r < kPlainHigh && p > kPlainLow && E < kPlainHigh;
}

// ---------------------------------------------------------------------------------------------
// Pointwise formulas (operation order of src/euler2d_cuda.cu:71-146, 169-205, 248-281).
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ double pressure(double r, double mu, double mv, double E, double gamma) {
  return (gamma - 1.0) * (E - 0.5 * (mu * mu + mv * mv) / r);
}

// The primitives of a cell.  `ok` (PLAIN): whether its state is plain; the quotients hold only then.
template <bool PLAIN>
__device__ __forceinline__ Cell primitives(double r, double mu, double mv, double E, double gamma, double* y,
                                           bool* ok) {
  Cell c{};
  c.r = r;
  if (PLAIN) {
    *y = recip(r);
    c.p = (gamma - 1.0) * (E - quot<true>(0.5 * (mu * mu + mv * mv), r, *y));
    *ok = plain_state(r, c.p, E);
    c.u = __builtin_copysign(quot_scaled(mu, r, *y) * kUnscale, mu);  // r > 0; 0 / r keeps its sign
    c.v = __builtin_copysign(quot_scaled(mv, r, *y) * kUnscale, mv);
  } else {
    *y = 0.0;
    c.u = mu / r;
    c.v = mv / r;
    c.p = pressure(r, mu, mv, E, gamma);
  }
  return c;
}

// The derived values of a cell; y = recip(r) (PLAIN), yg = recip(gamma - 1).
template <bool AUSM, bool PLAIN>
__device__ __forceinline__ void derive(Cell& c, double gm, double y, double yg) {
  c.a = root<PLAIN>(quot<PLAIN>(gm * c.p, c.r, y));
  const double E = quot<PLAIN>(c.p, gm - 1.0, yg) + 0.5 * c.r * (c.u * c.u + c.v * c.v);
  if (AUSM) {
    c.H = E + c.p;
    c.e = y;
  } else {
    c.q = root<PLAIN>(c.r);
    c.E = E;
    c.H = quot<PLAIN>(E + c.p, c.r, y);
    c.e = quot<PLAIN>(E, c.r, y);
  }
}

// HLLC flux in the face frame; un, ut: the normal and tangential velocity of a side.
template <bool PLAIN>
__device__ __forceinline__ void hllc(const Cell& L, double uL, double vL, const Cell& R, double uR, double vR,
                                     double gm, double f[4]) {
  const double qs = L.q + R.q, ys = PLAIN ? recip(qs) : 0.0;
  const double uT = quot<PLAIN>(L.q * uL + R.q * uR, qs, ys);
  const double vT = quot<PLAIN>(L.q * vL + R.q * vR, qs, ys);
  const double HT = quot<PLAIN>(L.q * L.H + R.q * R.H, qs, ys);
  const double aT = root<PLAIN>(fmax((gm - 1.0) * (HT - 0.5 * (uT * uT + vT * vT)), 1e-300));
  const double SL = fmin(uL - L.a, uT - aT), SR = fmax(uR + R.a, uT + aT);
  // The side that the face's flux is built on: the upwind one outside the fan, that of the
  // contact's sign inside it (where SL < 0 < SR).
  bool left = SL >= 0.0;
  const bool whole = left || SR <= 0.0;
  const double dL = SL - uL, dR = SR - uR, mL = L.r * dL, mR = R.r * dR;
  double Ss = 0.0;
  if (!whole) {
    Ss = quot<PLAIN>(R.p - L.p + L.r * uL * dL - R.r * uR * dR, mL - mR);
    left = Ss >= 0.0;
  }
  const double r = left ? L.r : R.r, u = left ? uL : uR, v = left ? vL : vR, p = left ? L.p : R.p;
  const double E = left ? L.E : R.E;
  const double mass = r * u;
  f[0] = mass;
  f[1] = mass * u + p;
  f[2] = mass * v;
  f[3] = u * (E + p);
  if (whole) return;
  // Star state of that side, then F = F_side + S_side (U* - U_side).
  const double S = left ? SL : SR, e = left ? L.e : R.e, m = left ? mL : mR;
  const double a = quot<PLAIN>(m, S - Ss);
  const double star = a * (e + (Ss - u) * (Ss + quot<PLAIN>(p, m)));
  f[0] = f[0] + S * (a - r);
  f[1] = f[1] + S * (a * Ss - mass);
  f[2] = f[2] + S * (a * v - r * v);
  f[3] = f[3] + S * (star - E);
}

// AUSM+-up split functions (Liou 2006) with the reference's constants (beta 1/8, Kp 1/4,
// Ku 3/4, sigma 1).  s is the side sign +1 / -1.
__device__ __forceinline__ double m1(double m, int s) { return 0.5 * (m + s * fabs(m)); }
__device__ __forceinline__ double m2(double m, int s) { return s * 0.25 * (m + s) * (m + s); }
__device__ __forceinline__ double m4(double m, int s) {
  if (fabs(m) >= 1.0) return m1(m, s);
  return m2(m, s) * (1.0 - s * 2.0 * m2(m, -s));
}
__device__ __forceinline__ double p5(double m, int s, double alpha) {
  if (fabs(m) >= 1.0) return 0.5 * (1.0 + s * (m > 0.0 ? 1.0 : (m < 0.0 ? -1.0 : 0.0)));
  return m2(m, s) * ((s * 2.0 - m) - s * 16.0 * alpha * m * m2(m, -s));
}

template <bool PLAIN>
__device__ __forceinline__ void ausm(const Cell& L, double uL, double vL, const Cell& R, double uR, double vR,
                                     double mco, double f[4]) {
  const double a12 = 0.5 * (L.a + R.a), ya = PLAIN ? recip(a12) : 0.0;
  const double rho12 = 0.5 * (L.r + R.r), ML = quot<PLAIN>(uL, a12, ya), MR = quot<PLAIN>(uR, a12, ya);
  const double mb2 = quot<PLAIN>(0.5 * (uL * uL + uR * uR), a12 * a12);
  const double m02 = fmin(1.0, fmax(mb2, mco * mco));
  const double m0 = root<PLAIN>(m02);
  const double fa = m0 * (2.0 - m0);
  const double alpha = 3.0 / 16.0 * (-4.0 + 5.0 * fa * fa);
  const double m12 = m4(ML, 1) + m4(MR, -1) -
                     quot<PLAIN>(quot<PLAIN>(0.25, fa) * fmax(1.0 - mb2, 0.0) * (R.p - L.p), rho12 * a12 * a12);
  const double pp = p5(ML, 1, alpha), pm = p5(MR, -1, alpha);
  const double p12 = pp * L.p + pm * R.p - 0.75 * pp * pm * (L.r + R.r) * fa * a12 * (uR - uL);
  const bool left = m12 > 0.0;
  const double r = left ? L.r : R.r, u = left ? uL : uR, v = left ? vL : vR;
  const double mdot = a12 * m12 * r;
  f[0] = mdot;
  f[1] = mdot * u + p12;
  f[2] = mdot * v;
  f[3] = quot<PLAIN>(mdot * (left ? L.H : R.H), r, left ? L.e : R.e);
}

// Flux through an x face (normal u) or a y face (normal v), returned in x / y momentum order.
template <bool XFACE, bool AUSM, bool PLAIN>
__device__ __forceinline__ Flux face_flux(double gamma, double mco, const Cell& L, const Cell& R) {
  double f[4];
  const double nL = XFACE ? L.u : L.v, tL = XFACE ? L.v : L.u;
  const double nR = XFACE ? R.u : R.v, tR = XFACE ? R.v : R.u;
  if (AUSM)
    ausm<PLAIN>(L, nL, tL, R, nR, tR, mco, f);
  else
    hllc<PLAIN>(L, nL, tL, R, nR, tR, gamma, f);
  return XFACE ? Flux{f[0], f[1], f[2], f[3]} : Flux{f[0], f[2], f[1], f[3]};
}

__device__ __forceinline__ double wave_bound(double r, double mu, double mv, double E, const Grid& g, double dx,
                                             double dy) {
  const double u = mu / r, v = mv / r;
  const double p = pressure(r, mu, mv, E, g.gamma);
  const double a = sqrt(g.gamma * p / r);
  return (fabs(u) + a) / dx + (fabs(v) + a) / dy;
}

__device__ __forceinline__ bool inadmissible(double r, double mu, double mv, double E, double gamma) {
  const double p = pressure(r, mu, mv, E, gamma);
  return !(r > 0.0) || !(p > 0.0) || !isfinite(r) || !isfinite(p);
}

// Admissibility of an RK candidate, and with WAVE its wave-speed bound: `inadmissible` and
// `wave_bound` with the quotients by r shared (pressure and sound speed see the same p).
template <bool WAVE>
__device__ __forceinline__ bool check_candidate(double r, double mu, double mv, double E, const Grid& g, double dx,
                                                double dy, double rdx, double rdy, double* bound) {
  const double y = recip(r);
  const double p = (g.gamma - 1.0) * (E - quot<true>(0.5 * (mu * mu + mv * mv), r, y));
  if (__any(!(g.plain && plain_state(r, p, E)))) {
    if (WAVE) *bound = wave_bound(r, mu, mv, E, g, dx, dy);
    return inadmissible(r, mu, mv, E, g.gamma);
  }
  if (WAVE) {  // |u| and |v| are added to the sound speed: a tiny one's last bits vanish
    const double a = root<true>(quot<true>(g.gamma * p, r, y));
    *bound = quot<true>(fabs(quot<true>(mu, r, y)) + a, dx, rdx) + quot<true>(fabs(quot<true>(mv, r, y)) + a, dy, rdy);
  }
  return false;
}

// Ghost index map of one axis (src/euler2d_cuda.cu:153-180): the interior cell a ghost copies
// and whether its normal momentum is negated.  Indices beyond the first ghost (unused lanes)
// are clamped.
__device__ __forceinline__ int map_axis(int i, int n, int lo, int hi, bool* flip) {
  if (i < 0) {
    if (lo == BC_PERIODIC) return i + n;
    if (lo == BC_REFLECT) {
      *flip = true;
      return -i - 1;
    }
    return 0;
  }
  if (i >= n) {
    if (i > n) return n - 1;
    if (hi == BC_PERIODIC) return i - n;
    if (hi == BC_REFLECT) {
      *flip = true;
      return 2 * n - 1 - i;
    }
    return n - 1;
  }
  return i;
}

__device__ __forceinline__ double shfl_up1(double x) { return __shfl_up(x, 1, kLanes); }
__device__ __forceinline__ double shfl_down1(double x) { return __shfl_down(x, 1, kLanes); }

__device__ __forceinline__ unsigned long long wave_max(unsigned long long x) {
  for (int d = kLanes / 2; d > 0; d >>= 1) {
    const unsigned long long y = __shfl_xor(x, d, kLanes);
    x = y > x ? y : x;
  }
  return x;
}

__device__ __forceinline__ double next_dt(const Grid& g, double smax_value, double t, double tend) {
  double d = g.dt_fixed > 0.0 ? g.dt_fixed : g.cfl / smax_value;
  const double remain = tend - t;
  if (remain <= 0.0)
    d = 0.0;
  else if (d > remain)
    d = remain;
  return d;
}

__device__ __forceinline__ unsigned long long load_relaxed(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Logical block of a launch: hardware dispatches consecutive blocks round-robin over the 8 XCDs;
// give each XCD a contiguous range of strips so that halo rows and columns shared by neighbours
// stay in one L2.  The launch is a multiple of 8 blocks.
__device__ __forceinline__ int logical_block() {
  const int per_xcd = gridDim.x / kXcds;
  return (blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
}

// ---------------------------------------------------------------------------------------------
// Commit of a trial (one wave, after the last stage): src/euler2d_cuda.cu:670-693.
// ---------------------------------------------------------------------------------------------
// `count` rejections in a row (one wave): each halves every positive step; the run gives up after 12
// retries or on an unusable step (which no halving mends: at the first).  True while it goes on.
__device__ bool reject(const Grid& g, int count) {
  Control* c = g.ctrl;
  const int lane = threadIdx.x % kLanes;
  int unusable = 0;
  for (int k = lane; k < g.ncase; k += kLanes) {
    const double d = g.dt[k];
    if (d < 0.0 || !isfinite(d)) unusable = 1;
  }
  unusable = __any(unusable);
  const int before = c->retries;
  const int n = unusable ? 1 : min(count, kMaxRetries + 1 - before);
  const bool on = !unusable && before + n <= kMaxRetries;
  for (int k = lane; k < g.ncase; k += kLanes) {
    double d = g.dt[k];
    for (int r = 0; r < n; ++r)
      if (d > 0.0) d *= 0.5;
    g.dt[k] = d;
    g.smax[k] = 0;
  }
  if (lane == 0) {
    c->retries = before + n;
    c->nreject += n;
    if (!on) c->status = 2;
    c->bad = 0;
    c->events += n;
  }
  return on;
}

// Maxima of the strips' partials per case, in LDS (one block, all threads).
__device__ void reduce_parts(const Grid& g, unsigned long long* s_max) {
  const int tid = threadIdx.x, lane = tid % kLanes;
  for (int k = tid; k < g.ncase; k += blockDim.x) s_max[k] = 0;
  __syncthreads();
  const int per_case = g.strips_x * g.strips_y;
  for (int first = tid - lane; first < g.strips; first += blockDim.x) {
    const int strip = first + lane;
    const bool valid = strip < g.strips;
    const unsigned long long v = valid ? g.part[strip] : 0ull;
    const int c = (valid ? strip : g.strips - 1) / per_case;
    if (__all(c == __shfl(c, 0, kLanes))) {
      const unsigned long long m = wave_max(v);
      if (lane == 0) atomicMax(&s_max[c], m);
    } else if (valid) {
      atomicMax(&s_max[c], v);
    }
  }
  __syncthreads();
}

__device__ void commit(const Grid& g, unsigned long long* s_max) {
  Control* c = g.ctrl;
  const int tid = threadIdx.x;
  if (__hip_atomic_load(&c->bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) {
    __syncthreads();  // every wave has read the flag that reject() clears
    if (tid < kLanes) reject(g, 1);
    return;
  }
  if (g.use_part) reduce_parts(g, s_max);
  // Accepted: advance the clocks of the cases that moved, then either stop (maxsteps reached,
  // or every case at tend) or choose the next step from the candidate's wave-speed bound.
  const double tend = c->tend;
  const long long steps = c->steps + 1;
  const bool maxed = steps >= c->maxsteps;
  int open = 0;
  for (int k = tid; k < g.ncase; k += blockDim.x) {
    const double d = g.dt[k];
    g.dt_out[k] = d;
    double tk = g.t[k];
    if (d > 0.0) {
      tk += d;
      g.t[k] = tk;
    }
    if (tk < tend) open = 1;
  }
  const bool any_open = __syncthreads_or(open);
  const bool next = !maxed && any_open;
  for (int k = tid; k < g.ncase; k += blockDim.x) {
    unsigned long long m = load_relaxed(&g.smax[k]);
    if (g.use_part) m = s_max[k] > m ? s_max[k] : m;
    if (next) g.dt[k] = next_dt(g, __longlong_as_double(static_cast<long long>(m)), g.t[k], tend);
    g.smax[k] = 0;
  }
  if (tid == 0) {
    c->steps = steps;
    c->cur ^= 1;
    c->nsteps += 1;
    c->retries = 0;
    c->ghost_from = next ? 1 : 2;
    if (!next) c->status = maxed ? 1 : 0;
    c->events += 1;
  }
}

// ---------------------------------------------------------------------------------------------
// One RK stage (MODE 1..3), the residual alone (MODE 0) or the backward-Euler residual with the
// defect norms (MODE 4), fused over a wave strip.
//   MODE 1: U[cur^1] = U + dt L(U)                    (in U[cur])
//   MODE 2: S2 = 3/4 U + 1/4 (U1 + dt L(U1))          (U1 in U[cur^1])
//   MODE 3: U[cur^1] = 1/3 U + 2/3 (S2 + dt L(S2)), and the candidate's wave-speed bound
//   MODE 0: R = L(in)
//   MODE 4: one pseudo update of backward Euler: per case the maximum over cells of the scaled defect
//           max_v |D| / max(1, |U|), D = dt L(Q) - (Q - U) (infinite for a non-finite defect;
//           src/euler2d_cuda.cu:331-350), and the candidate Q + omega D, omega = cfl* / (cfl* + dt
//           rate(Q)), of the cases that move, with its admissibility.  The candidate is formed before
//           k_be_decide has judged the defect and is dropped when that ends the step, so that an update
//           is two launches and reads the states once: on 8 cases of 256 x 256 59 -> 33 us against a
//           residual, a decision, a candidate and a check kernel.  A candidate that is refused is formed
//           again, with its residual, at half the pseudo CFL.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ void load_row(const double* p, size_t plane, double (&c)[4]) {
  for (int v = 0; v < 4; ++v) c[v] = p[v * plane];
}
// Bound by FP64 instruction issue (about 450 VALU instructions a cell of a row, halos included, 875 with
// every quotient a full division and both sides' sound speeds, energies and enthalpies formed at every
// face; VALU busy 75 / 66 / 68% of the three stages on 16 cases of 1024 x 1024), in stages 2 and 3 also by
// memory (4.5-4.6 TB/s, three quarters of the best copy), and by the latency of its row's loads: the next row's state is loaded while this one is evaluated, the base
// state of the row to update before the y fluxes.  That takes 124-146 VGPRs (RK stages; 146-166 on a cut
// grid), 130-173 in the pseudo update, and three waves per SIMD (168 VGPRs; the cut grid's HLLC pseudo
// update, 173, has two); four waves (128 VGPRs) spill nothing but the loads' lead: 8 cases of
// 1024 x 1024, HLLC, stages 336 / 347 / 378 us before, 218 / 276 / 294 with four waves and no
// prefetch, 202 / 230 / 244 with it.
template <int MODE, bool CUT, bool AUSM>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(CUT ? 2 : 3))) void k_stage(Grid g, const double* __restrict__ rhs_in,
                                                     double* __restrict__ rhs_out) {
  Control* ctrl = g.ctrl;
  bool skip = false;
  int cur = 0, qb = 0;
  if (MODE > 0) {
    if (__hip_atomic_load(&ctrl->status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != RUNNING) return;
    if (MODE == 4) {
      if (ctrl->phase == PH_BOUND) return;
      qb = ctrl->qbuf;
    } else {
      skip = __hip_atomic_load(&ctrl->bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
    }
    cur = ctrl->cur;
  }
  const double* base = MODE > 0 ? g.B[cur] : nullptr;
  const double* in = MODE == 0 ? rhs_in : MODE == 1 ? g.B[cur] : MODE == 2 ? g.B[cur ^ 1] : MODE == 3 ? g.B[2]
                                                                                                    : g.B[qb];
  double* out = MODE == 0 ? rhs_out : MODE == 2 ? g.B[2] : MODE == 4 ? g.B[3 - cur - qb] : g.B[cur ^ 1];
  const double pseudo = MODE == 4 ? ctrl->pseudo : 0.0;
  constexpr double A = MODE == 2 ? 0.75 : MODE == 3 ? 1.0 / 3.0 : 0.0;
  constexpr double B = MODE == 2 ? 0.25 : MODE == 3 ? 2.0 / 3.0 : 1.0;

  const int lane = threadIdx.x % kLanes;
  const int strip = __builtin_amdgcn_readfirstlane(logical_block() * kWaves + threadIdx.x / kLanes);
  bool wave_bad = false;
  unsigned long long bound = 0;
  const bool work = !skip && strip < g.strips;
  int icase = 0;
  if (work) {
    icase = strip / (g.strips_x * g.strips_y);
    const int rem = strip - icase * g.strips_x * g.strips_y;
    const int sy = rem / g.strips_x, sx = rem - sy * g.strips_x;
    const int i = sx * kStripCells - 1 + lane;
    const int j0 = sy * g.rows;
    const int jl = min(j0 + g.rows, g.ny) - 1;
    const bool owner = lane >= 1 && lane <= kStripCells && i < g.nx;
    bool flip_u = false;
    const int ic = map_axis(i, g.nx, g.bc[0], g.bc[1], &flip_u);
    const size_t plane = g.plane;
    const size_t case_base = static_cast<size_t>(icase) * 4 * plane + (ic + kGhosts);
    const double mco = g.mco[icase];
    const int iw = min(max(i, -kGhosts), g.nx + kGhosts - 1) + kGhosts;
    const double dxi = g.dx[iw], rdxi = g.rdx[iw];
    const double yg = recip(g.gamma - 1.0);
    const double dt = MODE > 0 ? g.dt[icase] : 0.0;

    Cell wprev{};
    // Whether the cells of the last three rows were evaluated by the plain quotients (bit 0: this row).
    unsigned plain = 0u;
    Flux gprev{}, xres{};  // xres: x residual of a full cell, or ae FX_e - aw FX_w of a cut cell
    double ay_prev = 1.0;  // aperture of the previous y face (cut grids)
    double ax_sum = 0.0;   // cut grids, MODE 4: apertures of the previous row's x faces
    double q0 = 0, q1 = 0, q2 = 0, q3 = 0;  // conserved state of the owned cell of the previous row
    unsigned code_prev = 0;                  // cut grids: code of the lane's cell of the previous row
    const bool in_x = i >= 0 && i <= g.nx;   // the lane's west x face is a grid face
    bool flip_v = false;
    int jc = map_axis(j0 - 1, g.ny, g.bc[2], g.bc[3], &flip_v);
    double next[4];
    load_row(in + case_base + static_cast<size_t>(jc + kGhosts) * g.mx, plane, next);
    for (int j = j0 - 1; j <= jl + 1; ++j) {
      const double c0 = next[0], c1 = next[1], c2 = next[2], c3 = next[3];
      const size_t ko = case_base + static_cast<size_t>(j - 1 + kGhosts) * g.mx;
      const int jm = jc; const bool flip_m = flip_v;
      if (j <= jl) {
        flip_v = false;
        jc = map_axis(j + 1, g.ny, g.bc[2], g.bc[3], &flip_v);
        load_row(in + case_base + static_cast<size_t>(jc + kGhosts) * g.mx, plane, next);
      }
      double base_row[4];
      if (MODE > 1 && j > j0 && owner)
        for (int v = 0; v < 4; ++v) base_row[v] = MODE == 4 ? base[ko + v * plane] : __builtin_nontemporal_load(base + ko + v * plane);
      // Cut grids: codes of the mapped cell (solid or not) and of the lane's own column at row j
      // (its faces, cut or not, rewritten by SRD or not).
      const unsigned code_m = CUT ? g.code[static_cast<size_t>(jm + kGhosts) * g.mx + ic + kGhosts] : 0u;
      const unsigned code_u = CUT && in_x ? g.code[static_cast<size_t>(j + kGhosts) * g.mx + i + kGhosts] : 0u;
      // A solid cell stands for (1, 0, 0, 1) (never a ghost's source: the body keeps clear of the sides).
      const bool solid = CUT && (code_m & 1u);
      double yr;
      bool ok;
      Cell w = primitives<true>(c0, c1, c2, c3, g.gamma, &yr, &ok);
      if (solid) w.r = 1.0, w.u = 0.0, w.v = 0.0, w.p = 1.0, yr = 1.0, ok = true;
      // (The residual alone, MODE 0, is asked for at states of any kind: always the general form.)
      const bool plain_row = MODE != 0 && g.plain && !__any(!ok);
      plain = (plain << 1 | (plain_row ? 1u : 0u)) & 7u;
      if (plain_row) {
        derive<AUSM, true>(w, g.gamma, yr, yg);
      } else {
        w = primitives<false>(c0, c1, c2, c3, g.gamma, &yr, &ok);
        if (solid) w.r = 1.0, w.u = 0.0, w.v = 0.0, w.p = 1.0;
        derive<AUSM, false>(w, g.gamma, 0.0, 0.0);
      }
      if (flip_u) w.u = -w.u;
      if (flip_m) w.v = -w.v;
      if (j >= j0) {
        // y face between rows j - 1 and j (closed faces carry no flux)
        double ay = 1.0;
        if (CUT && i >= 0 && i < g.nx) {
          const unsigned st = (code_u >> 5) & 3u;
          ay = st == 0u ? 0.0 : st == 1u ? g.dx[i + kGhosts] : g.ayl[static_cast<size_t>(j) * g.nx + i];
        }
        Flux gf{0.0, 0.0, 0.0, 0.0};
        if (!CUT || ay > 0.0)
          gf = (plain & 3u) == 3u ? face_flux<false, AUSM, true>(g.gamma, mco, wprev, w)
                                  : face_flux<false, AUSM, false>(g.gamma, mco, wprev, w);
        if (j > j0 && owner) {
          // Residual and update of the owned cell of row j - 1.
          const double dyj = g.dy[j - 1 + kGhosts], rdyj = g.rdy[j - 1 + kGhosts];
          const size_t kc = static_cast<size_t>(j - 1 + kGhosts) * g.mx + i + kGhosts;
          double r0, r1, r2, r3;
          bool fluid = true, moved = false;
          if (CUT && (code_prev & 1u)) {
            fluid = false;
            r0 = r1 = r2 = r3 = 0.0;
          } else if (!CUT || !(code_prev & 2u)) {
            if (plain == 7u) {
              r0 = __builtin_fma(-kUnscale, quot_scaled(gf.m - gprev.m, dyj, rdyj), xres.m);
              r1 = __builtin_fma(-kUnscale, quot_scaled(gf.x - gprev.x, dyj, rdyj), xres.x);
              r2 = __builtin_fma(-kUnscale, quot_scaled(gf.y - gprev.y, dyj, rdyj), xres.y);
              r3 = __builtin_fma(-kUnscale, quot_scaled(gf.e - gprev.e, dyj, rdyj), xres.e);
            } else {
              r0 = xres.m - (gf.m - gprev.m) / dyj;
              r1 = xres.x - (gf.x - gprev.x) / dyj;
              r2 = xres.y - (gf.y - gprev.y) / dyj;
              r3 = xres.e - (gf.e - gprev.e) / dyj;
            }
          } else {
            const double iv = 1.0 / g.vol[kc], pw = wprev.p;
            r0 = -iv * (xres.m + ay * gf.m - ay_prev * gprev.m);
            r1 = -iv * (xres.x + ay * gf.x - ay_prev * gprev.x);
            r2 = -iv * (xres.y + ay * gf.y - ay_prev * gprev.y);
            r3 = -iv * (xres.e + ay * gf.e - ay_prev * gprev.e);
            r1 -= iv * pw * g.wax[kc];
            r2 -= iv * pw * g.way[kc];
          }
          if (CUT && MODE == 3) moved = (code_prev & 4u) != 0u;
          if (MODE == 0) {
            out[ko] = r0;
            out[ko + plane] = r1;
            out[ko + 2 * plane] = r2;
            out[ko + 3 * plane] = r3;
          } else if (MODE == 4) {
            if (dt > 0.0 && fluid) {
              const double r[4] = {r0, r1, r2, r3}, q[4] = {q0, q1, q2, q3};
              double defect[4], norm = 0.0;
              bool finite = true;
              for (int v = 0; v < 4; ++v) {
                const double old = base_row[v];
                defect[v] = dt * r[v] - (q[v] - old);
                finite = finite && isfinite(defect[v]);
                norm = fmax(norm, fabs(defect[v]) / fmax(1.0, fabs(old)));
              }
              if (!finite) norm = HUGE_VAL;
              const unsigned long long bits = static_cast<unsigned long long>(__double_as_longlong(norm));
              bound = bits > bound ? bits : bound;
              double rate;
              if (CUT) {
                // implicit_spectral_rate of a cell of a cut grid (src/implicit2d.h:33-43)
                const double wx = g.wax[kc], wy = g.way[kc];
                const double wall = sqrt(wx * wx + wy * wy);
                rate = ((fabs(wprev.u) + wprev.a) * ax_sum + (fabs(wprev.v) + wprev.a) * (ay + ay_prev) +
                        fabs(wprev.u * wx + wprev.v * wy) + wprev.a * wall) /
                       (2.0 * g.vol[kc]);
              } else if (plain & 2u) {
                rate = quot<true>(fabs(wprev.u) + wprev.a, dxi, rdxi) + quot<true>(fabs(wprev.v) + wprev.a, dyj, rdyj);
              } else {
                rate = (fabs(wprev.u) + wprev.a) / dxi + (fabs(wprev.v) + wprev.a) / dyj;
              }
              const double omega = pseudo / (pseudo + dt * rate);
              double n[4];
              for (int v = 0; v < 4; ++v) {
                n[v] = q[v] + omega * defect[v];
                out[ko + v * plane] = n[v];
              }
              if (check_candidate<false>(n[0], n[1], n[2], n[3], g, dxi, dyj, rdxi, rdyj, nullptr)) wave_bad = true;
            }
          } else {
            double a0 = q0, a1 = q1, a2 = q2, a3 = q3;
            if (MODE > 1) {
              a0 = base_row[0], a1 = base_row[1], a2 = base_row[2], a3 = base_row[3];
            }
            const double n0 = A * a0 + B * (q0 + dt * r0);
            const double n1 = A * a1 + B * (q1 + dt * r1);
            const double n2 = A * a2 + B * (q2 + dt * r2);
            const double n3 = A * a3 + B * (q3 + dt * r3);
            out[ko] = n0;
            out[ko + plane] = n1;
            out[ko + 2 * plane] = n2;
            out[ko + 3 * plane] = n3;
            if (fluid) {
              double b = 0.0;
              if (check_candidate<MODE == 3>(n0, n1, n2, n3, g, dxi, dyj, rdxi, rdyj, &b)) wave_bad = true;
              // the next step's bound (cells that SRD rewrites report theirs after it)
              if (MODE == 3 && !moved) {
                const unsigned long long bits = static_cast<unsigned long long>(__double_as_longlong(b));
                bound = bits > bound ? bits : bound;
              }
            }
          }
        }
        gprev = gf;
        ay_prev = ay;
      }
      if (j >= j0 && j <= jl) {
        // x faces of row j: lane k evaluates the face west of its cell.
        // (Lane 0, which has no west neighbour, takes its own cell: __shfl_up returns it.)
        Cell wl{};
        wl.r = shfl_up1(w.r);
        wl.u = shfl_up1(w.u);
        wl.v = shfl_up1(w.v);
        wl.p = shfl_up1(w.p);
        wl.a = shfl_up1(w.a);
        wl.H = shfl_up1(w.H);
        wl.e = shfl_up1(w.e);
        if (!AUSM) {
          wl.q = shfl_up1(w.q);
          wl.E = shfl_up1(w.E);
        }
        double ax = 1.0;
        if (CUT && in_x) {
          const unsigned st = (code_u >> 3) & 3u;
          ax = st == 0u ? 0.0 : st == 1u ? g.dy[j + kGhosts] : g.axl[static_cast<size_t>(j) * (g.nx + 1) + i];
        }
        Flux fw{0.0, 0.0, 0.0, 0.0};
        if (!CUT || ax > 0.0)
          fw = plain_row ? face_flux<true, AUSM, true>(g.gamma, mco, wl, w)
                         : face_flux<true, AUSM, false>(g.gamma, mco, wl, w);
        const Flux fe{shfl_down1(fw.m), shfl_down1(fw.x), shfl_down1(fw.y), shfl_down1(fw.e)};
        const double ae = CUT ? shfl_down1(ax) : 1.0;
        if (CUT && MODE == 4) ax_sum = ae + ax;
        if (CUT && owner && (code_u & 2u))
          xres = Flux{ae * fe.m - ax * fw.m, ae * fe.x - ax * fw.x, ae * fe.y - ax * fw.y, ae * fe.e - ax * fw.e};
        else if (plain_row)
          xres = Flux{-kUnscale * quot_scaled(fe.m - fw.m, dxi, rdxi), -kUnscale * quot_scaled(fe.x - fw.x, dxi, rdxi),
                      -kUnscale * quot_scaled(fe.y - fw.y, dxi, rdxi), -kUnscale * quot_scaled(fe.e - fw.e, dxi, rdxi)};
        else
          xres = Flux{-(fe.m - fw.m) / dxi, -(fe.x - fw.x) / dxi, -(fe.y - fw.y) / dxi, -(fe.e - fw.e) / dxi};
      }
      wprev = w;
      q0 = c0, q1 = c1, q2 = c2, q3 = c3;
      code_prev = code_u;
    }
  }
  if (MODE == 0) return;
  if (MODE == 4) {
    if (__any(wave_bad) && lane == 0) atomicOr(&ctrl->bad, 1);
    bound = wave_max(bound);
    if (work && lane == 0) {
      if (g.use_part)
        g.part[strip] = bound;
      else if (bound)
        atomicMax(&g.norm[icase], bound);
    }
    return;
  }
  if (__any(wave_bad) && lane == 0) atomicOr(&ctrl->bad, 1);
  if (MODE == 3) {
    bound = wave_max(bound);
    if (work && lane == 0) {
      if (g.use_part)
        g.part[strip] = bound;
      else if (bound)
        atomicMax(&g.smax[icase], bound);
    }
  }
}

// recip() of the cell widths, once per session.
__global__ void k_recip(const double* dx, double* rdx, int mx, const double* dy, double* rdy, int my) {
  const size_t n = static_cast<size_t>(mx) + my;
  for (size_t k = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; k < n;
       k += static_cast<size_t>(gridDim.x) * blockDim.x) {
    if (k < static_cast<size_t>(mx))
      rdx[k] = recip(dx[k]);
    else
      rdy[k - mx] = recip(dy[k - mx]);
  }
}

// The commit of a trial, one block after the last stage (the kernel boundary orders every
// stage's flags and bounds before it; an in-kernel last-arriver commit would need device-scope
// fences, which write back and invalidate an XCD's L2 and cost more than this launch).
__global__ __launch_bounds__(kDecide) void k_commit(Grid g) {
  __shared__ unsigned long long s_max[kPartCases];
  // (The status moves only after the block's first barrier.)
  if (g.ctrl->status != RUNNING) return;
  commit(g, s_max);
}

// Wave-speed bound of every case at U[cur] (the first step of a run, src/euler2d_cuda.cu:223-237).
// Block b serves case b / per_case; each block reduces its cells to one maximum (on the bit
// patterns, as the reference's atomicMax does) and issues one atomic.
// gate >= 0: only while a run is in that backward-Euler phase.
__global__ __launch_bounds__(kThreads) void k_bound(Grid g, int per_case, int gate) {
  if (gate >= 0 && (g.ctrl->status != RUNNING || g.ctrl->phase != gate)) return;
  const int icase = blockIdx.x / per_case;
  const int part = blockIdx.x - icase * per_case;
  const double* u = g.B[g.ctrl->cur] + static_cast<size_t>(icase) * 4 * g.plane;
  const size_t inner = static_cast<size_t>(g.nx) * g.ny;
  unsigned long long best = 0;
  for (size_t q = part * static_cast<size_t>(blockDim.x) + threadIdx.x; q < inner;
       q += static_cast<size_t>(per_case) * blockDim.x) {
    const int j = static_cast<int>(q / g.nx), i = static_cast<int>(q - static_cast<size_t>(j) * g.nx);
    const size_t k = static_cast<size_t>(j + kGhosts) * g.mx + i + kGhosts;
    if (g.has_cut && g.vol[k] <= 0.0) continue;
    const double b = wave_bound(u[k], u[k + g.plane], u[k + 2 * g.plane], u[k + 3 * g.plane], g, g.dx[i + kGhosts],
                                g.dy[j + kGhosts]);
    const unsigned long long bits = static_cast<unsigned long long>(__double_as_longlong(b));
    best = bits > best ? bits : best;
  }
  best = wave_max(best);
  __shared__ unsigned long long s_best[kWaves];
  if (threadIdx.x % kLanes == 0) s_best[threadIdx.x / kLanes] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kWaves; ++w) best = s_best[w] > best ? s_best[w] : best;
    if (best) atomicMax(&g.smax[icase], best);
  }
}

// Start of a run call (src/euler2d_cuda.cu:605-619 for the first step): done / maxsteps tests
// and the first step's dt of every case.  One block.
__global__ __launch_bounds__(kThreads) void k_open(Grid g, double tend, long long maxsteps) {
  Control* c = g.ctrl;
  __shared__ int s_open;
  const int tid = threadIdx.x;
  if (tid == 0) s_open = 0;
  __syncthreads();
  for (int k = tid; k < g.ncase; k += blockDim.x)
    if (g.t[k] < tend) s_open = 1;
  __syncthreads();
  const bool run = maxsteps > 0 && s_open;
  for (int k = tid; k < g.ncase; k += blockDim.x) {
    if (run) g.dt[k] = next_dt(g, __longlong_as_double(static_cast<long long>(g.smax[k])), g.t[k], tend);
    g.smax[k] = 0;
  }
  __syncthreads();
  if (tid == 0) {
    c->tend = tend;
    c->maxsteps = maxsteps;
    c->steps = 0;
    c->retries = 0;
    c->bad = 0;
    if (maxsteps <= 0)
      c->status = 1;
    else if (!s_open)
      c->status = 0;
    else {
      c->status = RUNNING;
      c->ghost_from = 1;
    }
  }
}

// ------------------------------------------------------------------ backward Euler --
// src/euler2d_cuda.cu:370-447 with src/implicit2d.h:16-63 and src/implicit2d.cpp:37-69.  A round is
// k_bound, k_be_open, k_be_copy, which open a physical step, and kUpdates pairs of k_stage<4> and
// k_be_decide, each a pseudo update; every kernel acts only in its phase, so a round completes at
// least one phase.

// Nonphysical interior cells of B[cur] (the run's initial check).  Grid-stride over all cases.
__global__ __launch_bounds__(kThreads) void k_check_state(Grid g) {
  const double* u = g.B[g.ctrl->cur];
  const size_t inner = static_cast<size_t>(g.nx) * g.ny;
  bool bad = false;
  for (size_t q = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; q < inner * g.ncase;
       q += static_cast<size_t>(gridDim.x) * blockDim.x) {
    const size_t c = q / inner, ij = q - c * inner;
    const int j = static_cast<int>(ij / g.nx), i = static_cast<int>(ij - static_cast<size_t>(j) * g.nx);
    const size_t kc = static_cast<size_t>(j + kGhosts) * g.mx + i + kGhosts;
    if (g.has_cut && g.vol[kc] <= 0.0) continue;
    const size_t k = c * 4 * g.plane + kc;
    if (inadmissible(u[k], u[k + g.plane], u[k + 2 * g.plane], u[k + 3 * g.plane], g.gamma)) bad = true;
  }
  if (__any(bad) && threadIdx.x % kLanes == 0) atomicOr(&g.ctrl->bad, 1);
}

__global__ __launch_bounds__(kLanes) void k_be_start(Grid g, double tend, long long maxsteps) {
  Control* c = g.ctrl;
  if (threadIdx.x != 0) return;
  c->tend = tend;
  c->maxsteps = maxsteps;
  c->steps = 0;
  c->reason = WHY_NONE;
  if (c->bad) {
    c->status = 2;
    c->reason = WHY_INITIAL;
  } else {
    c->status = RUNNING;
    c->phase = PH_BOUND;
  }
  c->bad = 0;
  c->events += 1;
}

// Opening of a physical step: done / maxsteps tests, then every case's dt from its spectral
// bound (implicit2d_physical_dt: fixed or CFL step, cut to the remaining time when within
// 8 eps of it, and it must move the clock).  Cases are processed in order: those before the
// first failing one keep their new step.
__global__ __launch_bounds__(kLanes) void k_be_open(Grid g) {
  Control* c = g.ctrl;
  if (c->status != RUNNING || c->phase != PH_BOUND) return;
  const int lane = threadIdx.x;
  const double tend = c->tend;
  int open = 0;
  for (int k = lane; k < g.ncase; k += kLanes)
    if (g.t[k] < tend) open = 1;
  const bool any_open = __any(open);
  const bool maxed = c->steps >= c->maxsteps;
  int first_fail = g.ncase;
  if (any_open && !maxed) {
    for (int k = lane; k < g.ncase; k += kLanes) {
      const double t = g.t[k];
      const double remain = tend - t;
      if (remain <= 0.0) continue;
      double d = g.dt_fixed > 0.0 ? g.dt_fixed : g.cfl / __longlong_as_double(static_cast<long long>(g.smax[k]));
      if (!(d > 0.0) || !isfinite(d)) {
        first_fail = min(first_fail, k);
        continue;
      }
      const double roundoff = 8 * DBL_EPSILON * fmax(fabs(tend), fabs(t));
      if (d >= remain || remain - d <= roundoff) d = remain;
      if (!(t + d > t)) first_fail = min(first_fail, k);
    }
    for (int d = kLanes / 2; d > 0; d >>= 1) first_fail = min(first_fail, __shfl_xor(first_fail, d, kLanes));
    for (int k = lane; k < g.ncase; k += kLanes) {
      const double t = g.t[k];
      const double remain = tend - t;
      double d = 0.0;
      bool assign = true;
      if (remain > 0.0) {
        d = g.dt_fixed > 0.0 ? g.dt_fixed : g.cfl / __longlong_as_double(static_cast<long long>(g.smax[k]));
        if (!(d > 0.0) || !isfinite(d)) {
          assign = false;
        } else {
          const double roundoff = 8 * DBL_EPSILON * fmax(fabs(tend), fabs(t));
          if (d >= remain || remain - d <= roundoff) d = remain;
        }
      }
      if (assign && k <= first_fail) {
        g.dt[k] = d;
        g.dt_out[k] = d;
      }
    }
  }
  for (int k = lane; k < g.ncase; k += kLanes) g.smax[k] = 0;
  if (lane == 0) {
    if (!any_open) {
      c->status = 0;
    } else if (maxed) {
      c->status = 1;
    } else if (first_fail < g.ncase) {
      c->status = 3;
      c->reason = WHY_DT;
    } else {
      c->phase = PH_COPY;
      c->pseudo = g.pseudo0;
      c->iter = 0;
      c->pretries = 0;
      c->qbuf = c->cur == 0 ? 1 : 0;
    }
    c->events += 1;
  }
}

// Iterate and candidate start as copies of the accepted state (interior cells).
__global__ __launch_bounds__(kThreads) void k_be_copy(Grid g) {
  const Control* c = g.ctrl;
  if (c->status != RUNNING || c->phase != PH_COPY) return;
  const int cur = c->cur, qb = c->qbuf, tb = 3 - cur - qb;
  const double* u = g.B[cur];
  double* q = g.B[qb];
  double* t = g.B[tb];
  const size_t inner = static_cast<size_t>(g.nx) * g.ny;
  for (size_t e = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; e < inner * 4 * g.ncase;
       e += static_cast<size_t>(gridDim.x) * blockDim.x) {
    const size_t cv = e / inner, ij = e - cv * inner;
    const int j = static_cast<int>(ij / g.nx), i = static_cast<int>(ij - static_cast<size_t>(j) * g.nx);
    const size_t k = cv * g.plane + static_cast<size_t>(j + kGhosts) * g.mx + i + kGhosts;
    const double x = u[k];
    q[k] = x;
    t[k] = x;
  }
}

// The decision on a pseudo update.  Convergence of the iteration (implicit2d_converged): tolerance
// max(atol, rtol * the step's first norm) per case; on convergence the iterate becomes the accepted
// state and the clocks advance (implicit2d_advance_time), at the iteration limit the run ends with 4.
// Else the candidate becomes the next iterate, or, inadmissible, the pseudo CFL is halved for another
// (12 retries, then 2); a retry judges its candidate only.
__global__ __launch_bounds__(kDecide) void k_be_decide(Grid g) {
  __shared__ unsigned long long s_max[kPartCases];
  Control* c = g.ctrl;
  const int phase = c->phase;
  if (c->status != RUNNING || phase == PH_BOUND) return;
  const bool bad = c->bad != 0;
  __syncthreads();  // every wave has read the phase and the flag that the first one moves
  const bool retry = phase == PH_RETRY;
  if (g.use_part && !retry) reduce_parts(g, s_max);
  if (threadIdx.x >= kLanes) return;
  const unsigned long long* norms = g.use_part ? s_max : g.norm;
  const int lane = threadIdx.x;
  if (!retry) {
    int nonfinite = 0;
    for (int k = lane; k < g.ncase; k += kLanes)
      if (!isfinite(__longlong_as_double(static_cast<long long>(norms[k])))) nonfinite = 1;
    if (__any(nonfinite)) {
      for (int k = lane; k < g.ncase; k += kLanes) g.norm[k] = 0;
      if (lane == 0) {
        c->status = 2;
        c->reason = WHY_DEFECT;
        c->bad = 0;
        c->events += 1;
      }
      return;
    }
    const bool first = c->iter == 0;
    unsigned long long imax = 0, nmax = 0, tmax = 0;
    int open = 0;
    for (int k = lane; k < g.ncase; k += kLanes) {
      const double norm = __longlong_as_double(static_cast<long long>(norms[k]));
      if (first) g.initial[k] = norm;
      const double initial = g.initial[k];
      const double tol = fmax(g.atol, g.rtol * initial);
      const unsigned long long bi = static_cast<unsigned long long>(__double_as_longlong(initial));
      const unsigned long long bn = static_cast<unsigned long long>(__double_as_longlong(norm));
      const unsigned long long bt = static_cast<unsigned long long>(__double_as_longlong(tol));
      imax = bi > imax ? bi : imax;
      nmax = bn > nmax ? bn : nmax;
      tmax = bt > tmax ? bt : tmax;
      if (!isfinite(tol) || norm > tol) open = 1;
      g.norm[k] = 0;
    }
    imax = wave_max(imax);
    nmax = wave_max(nmax);
    tmax = wave_max(tmax);
    const bool converged = !__any(open);
    if (converged) {
      const double tend = c->tend;
      for (int k = lane; k < g.ncase; k += kLanes) {
        const double d = g.dt[k];
        if (d <= 0.0) continue;
        const double t = g.t[k];
        g.t[k] = d == tend - t ? tend : t + d;
      }
    }
    const bool limit = !converged && c->iter >= g.maxiter;
    if (lane == 0) {
      c->initial_defect = __longlong_as_double(static_cast<long long>(imax));
      c->final_defect = __longlong_as_double(static_cast<long long>(nmax));
      c->tolerance = __longlong_as_double(static_cast<long long>(tmax));
      c->checks += 1;
      c->pretries = 0;
      if (converged) {
        c->cur = c->qbuf;
        c->nsteps += 1;
        c->steps += 1;
        c->phase = PH_BOUND;
      } else if (limit) {
        c->status = 4;
        c->reason = WHY_MAXITER;
      }
    }
    if (converged || limit) {
      if (lane == 0) {
        c->bad = 0;
        c->events += 1;
      }
      return;
    }
  } else if (!g.use_part) {
    for (int k = lane; k < g.ncase; k += kLanes) g.norm[k] = 0;
  }
  if (lane != 0) return;
  c->bad = 0;
  if (bad) {
    c->iretries += 1;
    c->pretries += 1;
    if (c->pretries > kMaxRetries) {
      c->status = 2;
      c->reason = WHY_PSEUDO;
    } else {
      c->pseudo *= 0.5;
      c->phase = PH_RETRY;
    }
  } else {
    c->qbuf = 3 - c->cur - c->qbuf;
    c->updates += 1;
    c->iter += 1;
    c->phase = PH_UPDATE;
  }
  c->events += 1;
}

// ------------------------------------------------------------------------------- SRD --
// State redistribution of the stage's candidate (src/euler2d_cuda.cu:316-368, 461-468), when it is
// admissible: neighbourhood averages over the members, then every rewritten cell sums its own
// value (regular cells) and the averages of the neighbourhoods it belongs to, in ascending
// order, and divides by its count.  MODE picks the candidate buffer as the stage kernels do.
// A trial is rejected when the first stage's candidate is inadmissible in any cell (tested
// before the redistribution, src/euler2d_cuda.cu:648-651); on a cut grid that happens in the
// smallest cut cells, several times per step, until the step has been halved enough.  This
// kernel forms the first-stage candidates of every cut cell (and case) alone, with k_stage<1>'s
// formulas in its order (so the same bits: neighbours are interior, the body keeps three cells
// from every side), at the trial's step and its next halvings, and marks those steps at which one is
// inadmissible.  The residual does not depend on the step, so kPrechecks steps cost little more than
// one, and k_precheck_reject then rejects all the failing steps before the first that passes: two
// launches instead of a check and a rejection for each (8 cases of 512 x 512 with a body, about six
// halvings a step: 150 steps 51.7 -> 47.6 ms).  The decisions are those of the whole-grid pass at each
// step in turn.
template <bool AUSM>
__global__ __launch_bounds__(kThreads) void k_stage1_precheck(Grid g) {
  const Control* c = g.ctrl;
  if (__hip_atomic_load(&c->status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != RUNNING ||
      __hip_atomic_load(&c->bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)
    return;
  const double* in = g.B[c->cur];
  const size_t plane = g.plane;
  const size_t n = static_cast<size_t>(g.ncase) * g.n_pre;
  unsigned refused = 0;  // bit r: the step halved r times
  for (size_t t = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<size_t>(gridDim.x) * blockDim.x) {
    const size_t icase = t / g.n_pre;
    const int kc = g.pre_cell[t - icase * g.n_pre];
    const int jr = kc / g.mx - kGhosts, i = kc % g.mx - kGhosts;
    const double* u = in + icase * 4 * plane;
    const double mco = g.mco[icase];
    const auto cell_at = [&](int k) {
      double y;
      bool ok;
      Cell c = primitives<false>(u[k], u[k + plane], u[k + 2 * plane], u[k + 3 * plane], g.gamma, &y, &ok);
      if (g.vol[k] <= 0.0) c.r = 1.0, c.u = 0.0, c.v = 0.0, c.p = 1.0;
      derive<AUSM, false>(c, g.gamma, 0.0, 0.0);
      return c;
    };
    const Cell w = cell_at(kc);
    const double ax = g.axl[static_cast<size_t>(jr) * (g.nx + 1) + i];
    const double ae = g.axl[static_cast<size_t>(jr) * (g.nx + 1) + i + 1];
    const double as = g.ayl[static_cast<size_t>(jr) * g.nx + i];
    const double an = g.ayl[static_cast<size_t>(jr + 1) * g.nx + i];
    Flux fw{0.0, 0.0, 0.0, 0.0}, fe{0.0, 0.0, 0.0, 0.0}, gs{0.0, 0.0, 0.0, 0.0}, gn{0.0, 0.0, 0.0, 0.0};
    if (ax > 0.0) fw = face_flux<true, AUSM, false>(g.gamma, mco, cell_at(kc - 1), w);
    if (ae > 0.0) fe = face_flux<true, AUSM, false>(g.gamma, mco, w, cell_at(kc + 1));
    if (as > 0.0) gs = face_flux<false, AUSM, false>(g.gamma, mco, cell_at(kc - g.mx), w);
    if (an > 0.0) gn = face_flux<false, AUSM, false>(g.gamma, mco, w, cell_at(kc + g.mx));
    const Flux xres{ae * fe.m - ax * fw.m, ae * fe.x - ax * fw.x, ae * fe.y - ax * fw.y, ae * fe.e - ax * fw.e};
    const double iv = 1.0 / g.vol[kc], pw = w.p;
    const double r0 = -iv * (xres.m + an * gn.m - as * gs.m);
    double r1 = -iv * (xres.x + an * gn.x - as * gs.x);
    double r2 = -iv * (xres.y + an * gn.y - as * gs.y);
    const double r3 = -iv * (xres.e + an * gn.e - as * gs.e);
    r1 -= iv * pw * g.wax[kc];
    r2 -= iv * pw * g.way[kc];
    constexpr double A = 0.0, B = 1.0;  // the first stage's combination, as k_stage<1> forms it
    const double q0 = u[kc], q1 = u[kc + plane], q2 = u[kc + 2 * plane], q3 = u[kc + 3 * plane];
    double dt = g.dt[icase];
    for (int r = 0; r < kPrechecks; ++r) {
      const double n0 = A * q0 + B * (q0 + dt * r0);
      const double n1 = A * q1 + B * (q1 + dt * r1);
      const double n2 = A * q2 + B * (q2 + dt * r2);
      const double n3 = A * q3 + B * (q3 + dt * r3);
      if (inadmissible(n0, n1, n2, n3, g.gamma)) refused |= 1u << r;
      if (dt > 0.0) dt *= 0.5;
    }
  }
  unsigned any = 0;
  for (int r = 0; r < kPrechecks; ++r)
    if (__any((refused >> r & 1u) != 0u)) any |= 1u << r;
  if (any && threadIdx.x % kLanes == 0) atomicOr(&g.ctrl->pre_mask, any);
}

// Rejects (commit's rejection) the steps before the first that the pre-check passed; the last one's
// failure is left to the commit.
__global__ __launch_bounds__(kLanes) void k_precheck_reject(Grid g) {
  Control* c = g.ctrl;
  if (c->status != RUNNING) return;
  const unsigned mask = __hip_atomic_load(&c->pre_mask, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int failed = min(__builtin_ctz(~mask), kPrechecks);
  const int n = min(failed, kPrechecks - 1);
  const bool on = n == 0 || reject(g, n);
  if (threadIdx.x != 0) return;
  c->pre_mask = 0;
  if (on && failed == kPrechecks) c->bad = 1;
}

template <int MODE>
__device__ __forceinline__ double* stage_out(const Grid& g, int cur) {
  return MODE == 2 ? g.B[2] : g.B[cur ^ 1];
}

template <int MODE>
__global__ __launch_bounds__(kThreads) void k_srd_avg(Grid g) {
  const Control* c = g.ctrl;
  if (__hip_atomic_load(&c->status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != RUNNING ||
      __hip_atomic_load(&c->bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)
    return;
  const double* u = stage_out<MODE>(g, c->cur);
  const size_t n = static_cast<size_t>(g.ncase) * g.nsmall;
  for (size_t t = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; t < n;
       t += static_cast<size_t>(gridDim.x) * blockDim.x) {
    const size_t icase = t / g.nsmall;
    const int q = static_cast<int>(t - icase * g.nsmall);
    const double* uc = u + icase * 4 * g.plane;
    for (int v = 0; v < 4; ++v) {
      double sum = 0.0;
      for (int m = g.mem_off[q]; m < g.mem_off[q + 1]; ++m) {
        const int r = g.mem_idx[m];
        sum += g.vol[r] / g.nbrcount[r] * uc[v * g.plane + r];
      }
      g.Qh[t * 4 + v] = sum / g.svhat[q];
    }
  }
}

template <int MODE>
__global__ __launch_bounds__(kThreads) void k_srd_apply(Grid g) {
  Control* c = g.ctrl;
  if (__hip_atomic_load(&c->status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != RUNNING ||
      __hip_atomic_load(&c->bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)
    return;
  double* u = stage_out<MODE>(g, c->cur);
  const size_t n = static_cast<size_t>(g.ncase) * g.n_srd;
  const int lane = threadIdx.x % kLanes;
  bool bad = false;
  // Wave-uniform iterations (64 consecutive items per wave), so that the wave can reduce the
  // stage-3 bounds of one case to a single atomic.
  for (size_t base = blockIdx.x * static_cast<size_t>(blockDim.x) + (threadIdx.x - lane); base < n;
       base += static_cast<size_t>(gridDim.x) * blockDim.x) {
    const size_t t = base + lane;
    const bool valid = t < n;
    const size_t icase = valid ? t / g.n_srd : 0;
    unsigned long long bits = 0;
    if (valid) {
      const int e = static_cast<int>(t - icase * g.n_srd);
      const int k = g.srd_cell[e];
      double* uc = u + icase * 4 * g.plane;
      const double* qh = g.Qh + icase * g.nsmall * 4;
      double x[4];
      for (int v = 0; v < 4; ++v) {
        double acc = g.smallpos[k] < 0.0 ? uc[v * g.plane + k] : 0.0;
        for (int m = g.grp_off[e]; m < g.grp_off[e + 1]; ++m) acc += qh[g.grp_idx[m] * 4 + v];
        x[v] = acc / g.nbrcount[k];
        uc[v * g.plane + k] = x[v];
      }
      if (inadmissible(x[0], x[1], x[2], x[3], g.gamma)) bad = true;
      if (MODE == 3) {
        const int j = k / g.mx - kGhosts, i = k % g.mx - kGhosts;
        const double b = wave_bound(x[0], x[1], x[2], x[3], g, g.dx[i + kGhosts], g.dy[j + kGhosts]);
        bits = static_cast<unsigned long long>(__double_as_longlong(b));
      }
    }
    if (MODE == 3) {
      const size_t first = __shfl(icase, 0, kLanes);
      if (__all(!valid || icase == first)) {  // one case in the wave: one atomic
        const unsigned long long m = wave_max(bits);
        if (lane == 0 && m) atomicMax(&g.smax[first], m);
      } else if (bits) {
        atomicMax(&g.smax[icase], bits);
      }
    }
  }
  if (__any(bad) && lane == 0) atomicOr(&c->bad, 1);
}

// The two ghost layers of every plane of `out` from the interior of `in` (fill_ghosts on the device,
// for axes of at least two cells, where every ghost maps to an interior cell).  One block per plane
// and row: a row beside the interior has 2 kGhosts ghosts, a row above or below it is all ghosts.
__global__ __launch_bounds__(kThreads) void k_fill_ghosts(Grid g, const double* in, double* out) {
  const int jj = blockIdx.x, j = jj - kGhosts;
  const size_t plane = static_cast<size_t>(blockIdx.y) * g.plane;
  const int v = blockIdx.y % 4;
  const auto mapped = [](int k, int n, int lo, int hi, bool* flip) {
    if (k < 0) {
      if (lo == BC_PERIODIC) return k + n;
      *flip = lo == BC_REFLECT;
      return lo == BC_REFLECT ? -k - 1 : 0;
    }
    if (k >= n) {
      if (hi == BC_PERIODIC) return k - n;
      *flip = hi == BC_REFLECT;
      return hi == BC_REFLECT ? 2 * n - 1 - k : n - 1;
    }
    return k;
  };
  bool flip_v = false;
  const int js = mapped(j, g.ny, g.bc[2], g.bc[3], &flip_v);
  const bool inside = j >= 0 && j < g.ny;
  const int count = inside ? 2 * kGhosts : g.mx;
  for (int q = threadIdx.x; q < count; q += blockDim.x) {
    const int ii = inside && q >= kGhosts ? g.nx + q : q;
    bool flip_u = false;
    const int is = mapped(ii - kGhosts, g.nx, g.bc[0], g.bc[1], &flip_u);
    double sign = 1.0;
    if (v == 1 && flip_u) sign = -sign;
    if (v == 2 && flip_v) sign = -sign;
    out[plane + static_cast<size_t>(jj) * g.mx + ii] =
        sign * in[plane + static_cast<size_t>(js + kGhosts) * g.mx + is + kGhosts];
  }
}

__global__ void k_zero(double* p, size_t n) {
  for (size_t q = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; q < n;
       q += static_cast<size_t>(gridDim.x) * blockDim.x)
    p[q] = 0.0;
}

}  // namespace ugrid

// =============================================================================================
// Host side
// =============================================================================================
using namespace ugrid;

struct ugrid_session {
  int device = 0;
  Grid g{};
  ugrid_params par{};
  size_t states = 0;      // doubles per state array (ghosts included)
  int launch_blocks = 0;  // padded to a multiple of 8
  double* R = nullptr;       // residual output of ugrid_rhs (allocated on first use)
  double* rhs_in = nullptr;  // input staging of ugrid_rhs (allocated on first use)
  std::vector<double> mco;   // host copy of the reference Mach numbers
  Control* host_ctrl = nullptr;  // pinned mirror of the control record
  hipStream_t stream = nullptr;
  hipGraphExec_t exec = nullptr;  // trials, or backward-Euler rounds of kUpdates updates
  bool few_checks = false;  // backward Euler: the last replay's steps needed kFewChecks updates or fewer
  std::vector<void*> owned;
};

namespace {

int fail(char* err, size_t len, const std::string& message) {
  if (err && len) {
    const size_t k = message.size() < len - 1 ? message.size() : len - 1;
    std::memcpy(err, message.data(), k);
    err[k] = 0;
  }
  return 3;
}

bool ok(hipError_t e, char* err, size_t len, const char* what) {
  if (e == hipSuccess) return true;
  fail(err, len, std::string(what) + ": " + hipGetErrorString(e));
  return false;
}

template <class T>
bool device_alloc(ugrid_session* s, T** p, size_t count, char* err, size_t len) {
  void* q = nullptr;
  if (!ok(hipMalloc(&q, (count ? count : 1) * sizeof(T)), err, len, "hipMalloc")) return false;
  s->owned.push_back(q);
  *p = static_cast<T*>(q);
  return true;
}

// Arrays of one device allocation, each on a 256-byte boundary.
struct SmallArrays {
  std::vector<std::pair<void*, size_t>> at;  // the pointer to set (its address), and its array's offset
  size_t bytes = 0;
  template <class T>
  void add(T** p, size_t count) {
    at.push_back({p, bytes});
    bytes += (count * sizeof(T) + 255) / 256 * 256;
  }
  bool allocate(ugrid_session* s, char* err, size_t len) {
    char* base = nullptr;
    if (!device_alloc(s, &base, bytes, err, len)) return false;
    for (const auto& a : at) {
      const char* array = base + a.second;
      std::memcpy(a.first, &array, sizeof(array));
    }
    return true;
  }
};

void release(ugrid_session* s) {
  if (!s) return;
  if (s->exec) (void)hipGraphExecDestroy(s->exec);
  for (void* p : s->owned) (void)hipFree(p);
  if (s->host_ctrl) (void)hipHostFree(s->host_ctrl);
  if (s->stream) (void)hipStreamDestroy(s->stream);
  delete s;
}

// Fill the two ghost layers of every plane from the interior as the reference's boundary kernel
// does (src/euler2d_cuda.cu:153-180): both indices mapped, normal momentum negated on reflection.
void fill_ghosts(const Grid& g, double* u) {
  const int ng = kGhosts;
  for (int c = 0; c < g.ncase; ++c)
    for (int v = 0; v < 4; ++v) {
      double* q = u + (static_cast<size_t>(c) * 4 + v) * g.plane;
      for (int j = -ng; j < g.ny + ng; ++j)
        for (int i = -ng; i < g.nx + ng; ++i) {
          if (i >= 0 && i < g.nx && j >= 0 && j < g.ny) continue;
          int ii = i, jj = j;
          double sign = 1.0;
          if (ii < 0) {
            if (g.bc[0] == BC_PERIODIC) ii += g.nx;
            else if (g.bc[0] == BC_REFLECT) { ii = -ii - 1; if (v == 1) sign = -sign; }
            else ii = 0;
          } else if (ii >= g.nx) {
            if (g.bc[1] == BC_PERIODIC) ii -= g.nx;
            else if (g.bc[1] == BC_REFLECT) { ii = 2 * g.nx - 1 - ii; if (v == 1) sign = -sign; }
            else ii = g.nx - 1;
          }
          if (jj < 0) {
            if (g.bc[2] == BC_PERIODIC) jj += g.ny;
            else if (g.bc[2] == BC_REFLECT) { jj = -jj - 1; if (v == 2) sign = -sign; }
            else jj = 0;
          } else if (jj >= g.ny) {
            if (g.bc[3] == BC_PERIODIC) jj -= g.ny;
            else if (g.bc[3] == BC_REFLECT) { jj = 2 * g.ny - 1 - jj; if (v == 2) sign = -sign; }
            else jj = g.ny - 1;
          }
          q[static_cast<size_t>(j + ng) * g.mx + i + ng] = sign * q[static_cast<size_t>(jj + ng) * g.mx + ii + ng];
        }
    }
}

// Blocks per case of k_bound: about 2048 blocks over the batch, at most one per 256 cells.
void launch_bound(ugrid_session* s) {
  const Grid& g = s->g;
  const long long inner = static_cast<long long>(g.nx) * g.ny;
  const long long cap = (inner + kThreads - 1) / kThreads;
  const int per_case = static_cast<int>(std::max<long long>(1, std::min<long long>(cap, 2048 / g.ncase)));
  hipLaunchKernelGGL(k_bound, dim3(per_case * g.ncase), dim3(kThreads), 0, s->stream, g, per_case, -1);
}

int grid_blocks(const Grid& g, size_t items) {
  return static_cast<int>(std::max<size_t>(1, std::min<size_t>((items + kThreads - 1) / kThreads, 8192)));
}

// A stage kernel in the regular or the cut-grid instantiation.
template <int MODE>
void launch_stage(ugrid_session* s, hipStream_t stream, const double* in = nullptr, double* out = nullptr) {
  const dim3 blocks(s->launch_blocks), threads(kThreads);
  if (s->g.has_cut && s->g.ausm)
    hipLaunchKernelGGL((k_stage<MODE, true, true>), blocks, threads, 0, stream, s->g, in, out);
  else if (s->g.has_cut)
    hipLaunchKernelGGL((k_stage<MODE, true, false>), blocks, threads, 0, stream, s->g, in, out);
  else if (s->g.ausm)
    hipLaunchKernelGGL((k_stage<MODE, false, true>), blocks, threads, 0, stream, s->g, in, out);
  else
    hipLaunchKernelGGL((k_stage<MODE, false, false>), blocks, threads, 0, stream, s->g, in, out);
}

// A stage kernel followed, on a cut grid with small cells, by the redistribution of its candidate.
template <int MODE>
void launch_stage_srd(ugrid_session* s, hipStream_t stream) {
  const Grid& g = s->g;
  if (MODE == 1 && g.has_cut && g.n_pre > 0) {
    // The pre-check and its rejections; a failure of its last step is left to the trial's commit
    // (the stage kernels then return at once).
    const dim3 pre_blocks(grid_blocks(g, static_cast<size_t>(g.ncase) * g.n_pre));
    if (g.ausm)
      hipLaunchKernelGGL(k_stage1_precheck<true>, pre_blocks, dim3(kThreads), 0, stream, g);
    else
      hipLaunchKernelGGL(k_stage1_precheck<false>, pre_blocks, dim3(kThreads), 0, stream, g);
    hipLaunchKernelGGL(k_precheck_reject, dim3(1), dim3(kLanes), 0, stream, g);
  }
  launch_stage<MODE>(s, stream);
  if (!g.has_cut || g.nsmall == 0) return;
  hipLaunchKernelGGL(k_srd_avg<MODE>, dim3(grid_blocks(g, static_cast<size_t>(g.ncase) * g.nsmall)), dim3(kThreads), 0,
                     stream, g);
  hipLaunchKernelGGL(k_srd_apply<MODE>, dim3(grid_blocks(g, static_cast<size_t>(g.ncase) * g.n_srd)),
                     dim3(kThreads), 0, stream, g);
}

// One backward-Euler round: the kernels that open a step, then `updates` pseudo updates.  A launch that
// finds nothing to do costs about 3.5 us.  A step of tens of updates wants long rounds: with kUpdates it
// pays the three opening kernels once in eight updates, and at most a round less one of empty updates
// at its end.  A step that needs kFewChecks updates or fewer (a nearly steady flow) wastes less in
// rounds of one: 3 launches for each update but the first instead of 2 for each one missing of eight.
// One case of 64 x 64 whose steps converge at their first check takes 45 us a step in long rounds and 27
// in rounds of one, 8 cases of 256 x 256 98 and 59.  The host chooses by the updates a step of the
// session's last replay.
constexpr int kUpdates = 8;
constexpr int kFewChecks = 3;
constexpr int kShortRounds = 8;  // rounds of one update between polls
int launch_be_round(ugrid_session* s, hipStream_t stream, int updates) {
  const Grid& g = s->g;
  const long long inner = static_cast<long long>(g.nx) * g.ny;
  const long long blocks = (inner + 4 * kThreads - 1) / (4 * kThreads);
  const int per_case = static_cast<int>(blocks < 1 ? 1 : blocks > 256 ? 256 : blocks);
  const size_t cells = static_cast<size_t>(inner) * g.ncase;
  hipLaunchKernelGGL(k_bound, dim3(per_case * g.ncase), dim3(kThreads), 0, stream, g, per_case, PH_BOUND);
  hipLaunchKernelGGL(k_be_open, dim3(1), dim3(kLanes), 0, stream, g);
  hipLaunchKernelGGL(k_be_copy, dim3(grid_blocks(g, 4 * cells)), dim3(kThreads), 0, stream, g);
  for (int u = 0; u < updates; ++u) {
    launch_stage<4>(s, stream);
    hipLaunchKernelGGL(k_be_decide, dim3(1), dim3(kDecide), 0, stream, g);
  }
  return 3 + 2 * updates;
}

int launch_trial(ugrid_session* s, hipStream_t stream) {
  launch_stage_srd<1>(s, stream);
  launch_stage_srd<2>(s, stream);
  launch_stage_srd<3>(s, stream);
  hipLaunchKernelGGL(k_commit, dim3(1), dim3(kDecide), 0, stream, s->g);
  return 4;
}

// `count` trials, or backward-Euler rounds, as a graph.
bool build_graph(ugrid_session* s, int count, char* err, size_t len) {
  hipGraph_t graph = nullptr;
  if (!ok(hipStreamBeginCapture(s->stream, hipStreamCaptureModeThreadLocal), err, len, "begin capture")) return false;
  for (int k = 0; k < count; ++k) {
    if (s->par.time_integrator == 1)
      launch_be_round(s, s->stream, kUpdates);
    else
      launch_trial(s, s->stream);
  }
  const hipError_t launched = hipGetLastError();
  const hipError_t ended = hipStreamEndCapture(s->stream, &graph);
  if (!ok(launched, err, len, "trial launch") || !ok(ended, err, len, "end capture")) {
    if (graph) (void)hipGraphDestroy(graph);
    return false;
  }
  const hipError_t inst = hipGraphInstantiate(&s->exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  return ok(inst, err, len, "graph instantiate");
}

// Cut-cell arrays of the device: per-cell data, apertures, and the SRD lists (members of each
// neighbourhood; the cells SRD rewrites, each with its neighbourhoods in ascending order).
bool upload_cut(ugrid_session* s, const ugrid_cut_view& c, const double* dx, const double* dy, char* err, size_t len) {
  Grid& g = s->g;
  const size_t cells = g.plane, nfx = static_cast<size_t>(g.nx + 1) * g.ny, nfy = static_cast<size_t>(g.nx) * (g.ny + 1);
  std::vector<int> mem_off(1, 0), mem_idx;
  std::vector<std::vector<int>> groups(cells);
  for (int q = 0; q < c.nsmall; ++q) {
    const int count = static_cast<int>(c.scnt[q]);
    if (count < 1 || count > 25) {
      fail(err, len, "ugrid_create: invalid SRD neighbourhood size");
      return false;
    }
    for (int m = 0; m < count; ++m) {
      const double r = c.smem[25 * static_cast<size_t>(q) + m];
      if (!(r >= 0.0) || r >= static_cast<double>(cells)) {
        fail(err, len, "ugrid_create: invalid SRD member");
        return false;
      }
      mem_idx.push_back(static_cast<int>(r));
      groups[static_cast<size_t>(r)].push_back(q);
    }
    mem_off.push_back(static_cast<int>(mem_idx.size()));
  }
  std::vector<int> srd_cell, grp_off(1, 0), grp_idx;
  for (int j = 0; j < g.ny; ++j)
    for (int i = 0; i < g.nx; ++i) {
      const size_t k = static_cast<size_t>(j + kGhosts) * g.mx + i + kGhosts;
      if (c.vol[k] <= 0.0 || (c.smallpos[k] < 0.0 && c.nbrcount[k] == 1.0)) continue;
      srd_cell.push_back(static_cast<int>(k));
      grp_idx.insert(grp_idx.end(), groups[k].begin(), groups[k].end());
      grp_off.push_back(static_cast<int>(grp_idx.size()));
    }
  // Cell codes of the stage kernels (see Grid::code).  An aperture is coded 1 only when it equals
  // the full width bit for bit, 0 only when it is +0, so the kernels read the same values.
  std::vector<uint8_t> code(cells, 0);
  const auto face_state = [](double a, double full) -> unsigned {
    if (a == 0.0 && !std::signbit(a)) return 0u;
    return a == full ? 1u : 2u;
  };
  for (int jj = 0; jj < g.my; ++jj)
    for (int ii = 0; ii < g.mx; ++ii) {
      const size_t k = static_cast<size_t>(jj) * g.mx + ii;
      const int j = jj - kGhosts, i = ii - kGhosts;
      unsigned v = 0;
      if (c.vol[k] <= 0.0) v |= 1u;
      if (c.flag[k] != 0.0) v |= 2u;
      if (c.smallpos[k] >= 0.0 || c.nbrcount[k] != 1.0) v |= 4u;
      if (j >= 0 && j < g.ny && i >= 0 && i <= g.nx)
        v |= face_state(c.axl[static_cast<size_t>(j) * (g.nx + 1) + i], dy[jj]) << 3;
      if (j >= 0 && j <= g.ny && i >= 0 && i < g.nx)
        v |= face_state(c.ayl[static_cast<size_t>(j) * g.nx + i], dx[ii]) << 5;
      code[k] = static_cast<uint8_t>(v);
    }
  std::vector<int> pre_cell;  // interior cut cells, for the first-stage precheck
  for (int j = 0; j < g.ny; ++j)
    for (int i = 0; i < g.nx; ++i) {
      const size_t k = static_cast<size_t>(j + kGhosts) * g.mx + i + kGhosts;
      if (c.flag[k] != 0.0 && c.vol[k] > 0.0) pre_cell.push_back(static_cast<int>(k));
    }
  g.has_cut = 1;
  g.nsmall = c.nsmall;
  g.n_srd = static_cast<int>(srd_cell.size());
  g.n_pre = static_cast<int>(pre_cell.size());
  double *vol, *flag, *axl, *ayl, *wax, *way, *nbr, *pos, *svhat, *qh;
  int *moff, *midx, *scell, *goff, *gidx, *pcell;
  uint8_t* dcode;
  auto up = [&](void* dst, const void* src, size_t bytes) {
    return ok(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s->stream), err, len, "upload cut geometry");
  };
  const size_t nq = static_cast<size_t>(std::max(c.nsmall, 1));
  if (!device_alloc(s, &vol, cells, err, len) || !device_alloc(s, &flag, cells, err, len) ||
      !device_alloc(s, &axl, nfx, err, len) || !device_alloc(s, &ayl, nfy, err, len) ||
      !device_alloc(s, &wax, cells, err, len) || !device_alloc(s, &way, cells, err, len) ||
      !device_alloc(s, &nbr, cells, err, len) || !device_alloc(s, &pos, cells, err, len) ||
      !device_alloc(s, &svhat, nq, err, len) || !device_alloc(s, &qh, nq * 4 * g.ncase, err, len) ||
      !device_alloc(s, &moff, mem_off.size(), err, len) || !device_alloc(s, &midx, std::max<size_t>(mem_idx.size(), 1), err, len) ||
      !device_alloc(s, &scell, std::max<size_t>(srd_cell.size(), 1), err, len) ||
      !device_alloc(s, &goff, grp_off.size(), err, len) || !device_alloc(s, &gidx, std::max<size_t>(grp_idx.size(), 1), err, len) ||
      !device_alloc(s, &pcell, std::max<size_t>(pre_cell.size(), 1), err, len) ||
      !device_alloc(s, &dcode, cells, err, len))
    return false;
  const size_t d = sizeof(double), n = sizeof(int);
  if (!up(vol, c.vol, cells * d) || !up(flag, c.flag, cells * d) || !up(axl, c.axl, nfx * d) ||
      !up(ayl, c.ayl, nfy * d) || !up(wax, c.wax, cells * d) || !up(way, c.way, cells * d) ||
      !up(nbr, c.nbrcount, cells * d) || !up(pos, c.smallpos, cells * d) ||
      (c.nsmall > 0 && !up(svhat, c.svhat, c.nsmall * d)) || !up(moff, mem_off.data(), mem_off.size() * n) ||
      (!mem_idx.empty() && !up(midx, mem_idx.data(), mem_idx.size() * n)) ||
      (!srd_cell.empty() && !up(scell, srd_cell.data(), srd_cell.size() * n)) ||
      !up(goff, grp_off.data(), grp_off.size() * n) || (!grp_idx.empty() && !up(gidx, grp_idx.data(), grp_idx.size() * n)) ||
      (!pre_cell.empty() && !up(pcell, pre_cell.data(), pre_cell.size() * n)) || !up(dcode, code.data(), cells) ||
      !ok(hipStreamSynchronize(s->stream), err, len, "upload cut geometry"))
    return false;
  g.vol = vol;
  g.flag = flag;
  g.axl = axl;
  g.ayl = ayl;
  g.wax = wax;
  g.way = way;
  g.nbrcount = nbr;
  g.smallpos = pos;
  g.svhat = svhat;
  g.Qh = qh;
  g.mem_off = moff;
  g.mem_idx = midx;
  g.srd_cell = scell;
  g.grp_off = goff;
  g.grp_idx = gidx;
  g.pre_cell = pcell;
  g.code = dcode;
  return true;
}

// Rows per strip.  A strip of r rows costs its wave about r + 1 row times (the halo row's
// primitives and y flux), and a CU that holds n = 1, 2, 3 blocks (three is what the registers admit)
// takes kRowTime[n] microseconds a row, as fitted to launches of 1 to 64 rows on five grids (a cut grid's
// HLLC pseudo update has two blocks in a CU; its strips are chosen as for three).  Long
// strips waste least on the halo, short ones spread a small grid over the chip, and a launch that
// leaves its last round of blocks nearly empty pays for a whole one: the count with the least estimate
// is chosen, of counts that tie the smallest.  Against 32 rows, halved down to 4 while a CU held fewer
// than 16 waves: 8 cases of 1024 x 1024 682 us a step at 32 rows, 587 at the 23 that it takes (6120
// strips, two rounds of three blocks a CU) and 596 at 47 (2992, one round; the same estimate), 3 of 200 x 131
// 39.4 us at 4 rows and 27.6 at 1, 4 of 400 x 311 70.6 us at 4 and 62.3 at 3.
int choose_rows(int nx, int ny, int ncase, bool cut) {
  constexpr int kCus = 256, kResident = 3, kLongest = 64;
  constexpr double kRowTime[2][kResident + 1] = {{0.0, 1.95, 2.8, 3.6}, {0.0, 3.1, 4.1, 5.0}};
  const double* row_time = kRowTime[cut ? 1 : 0];
  const long long sx = (nx + kStripCells - 1) / kStripCells;
  int best = 1;
  double least = HUGE_VAL;
  for (int rows = 1; rows <= std::min(kLongest, ny); ++rows) {
    const long long strips = sx * ((ny + rows - 1) / rows) * ncase;
    const long long blocks = (strips + kWaves - 1) / kWaves, per_cu = (blocks + kCus - 1) / kCus;
    const double cost = (rows + 1) * (static_cast<double>(per_cu / kResident) * row_time[kResident] +
                                      row_time[per_cu % kResident]);
    if (cost < least) least = cost, best = rows;
  }
  return best;
}

}  // namespace

extern "C" int ugrid_create(const ugrid_setup* setup, const double* u, uint64_t u_len, const double* t,
                            const double* dt, ugrid_session** out, char* err, size_t err_len) {
  if (!out) return fail(err, err_len, "ugrid_create: null output handle");
  *out = nullptr;
  if (!setup || !u || !setup->dx || !setup->dy) return fail(err, err_len, "ugrid_create: null argument");
  const ugrid_params& p = setup->params;
  if (setup->nx < 1 || setup->ny < 1 || setup->ncase < 1)
    return fail(err, err_len, "ugrid_create: nx, ny and ncase must be positive");
  if (p.time_integrator != 0 && p.time_integrator != 1)
    return fail(err, err_len, "ugrid_create: time_integrator must be 0 (SSP-RK3) or 1 (backward Euler)");
  if (p.limiter != 3)
    return fail(err, err_len,
                "ugrid_create: the device backend requires the first-order limiter (3); refusing to change the method "
                "implicitly");
  for (int k = 0; k < 4; ++k)
    if (p.bc[k] < 0 || p.bc[k] > 2) return fail(err, err_len, "ugrid_create: boundary kinds are 0, 1 or 2");
  if ((p.bc[0] == BC_PERIODIC) != (p.bc[1] == BC_PERIODIC) || (p.bc[2] == BC_PERIODIC) != (p.bc[3] == BC_PERIODIC))
    return fail(err, err_len, "ugrid_create: periodic boundary must be set on both sides of an axis");
  if (setup->cut) {
    const ugrid_cut_view& c = *setup->cut;
    if (c.nbad_nbhd != 0)
      return fail(err, err_len, "ugrid_create: the device backend refuses " + std::to_string(c.nbad_nbhd) +
                                    " invalid SRD neighbourhoods");
    if (c.nsmall < 0 || !c.vol || !c.flag || !c.axl || !c.ayl || !c.wax || !c.way || !c.nbrcount || !c.smallpos ||
        (c.nsmall > 0 && (!c.scnt || !c.smem || !c.svhat)))
      return fail(err, err_len, "ugrid_create: incomplete cut-cell geometry");
    // The stage kernels take a ghost cell's state from the interior cell its boundary maps to,
    // which holds for the ghosts' own fluid volumes only while the body keeps three cells
    // clear of every side (as the geometry builders enforce).
    const int nx = setup->nx, ny = setup->ny;
    for (int j = -kGhosts; j < ny + kGhosts; ++j)
      for (int i = -kGhosts; i < nx + kGhosts; ++i) {
        const size_t k = static_cast<size_t>(j + kGhosts) * (nx + 2 * kGhosts) + (i + kGhosts);
        const bool near = i < 3 || i >= nx - 3 || j < 3 || j >= ny - 3;
        if (near && (c.flag[k] != 0.0 || !(c.vol[k] > 0.0)))
          return fail(err, err_len, "ugrid_create: cut-cell geometry within three cells of the domain boundary (cell " +
                                        std::to_string(i) + "," + std::to_string(j) + ")");
      }
    const double cells = static_cast<double>(nx + 2 * kGhosts) * (ny + 2 * kGhosts);
    for (int q = 0; q < c.nsmall; ++q) {
      const double count = c.scnt[q];
      if (!(count >= 1.0 && count <= 25.0) || count != static_cast<int>(count))
        return fail(err, err_len, "ugrid_create: invalid SRD neighbourhood size");
      for (int m = 0; m < static_cast<int>(count); ++m) {
        const double r = c.smem[25 * static_cast<size_t>(q) + m];
        if (!(r >= 0.0 && r < cells) || r != static_cast<double>(static_cast<long long>(r)))
          return fail(err, err_len, "ugrid_create: invalid SRD member");
      }
    }
  }
  const long long mx = setup->nx + 2LL * kGhosts, my = setup->ny + 2LL * kGhosts;
  if (mx * my > (1LL << 40) / setup->ncase) return fail(err, err_len, "ugrid_create: grid too large");
  const size_t states = static_cast<size_t>(setup->ncase) * 4 * static_cast<size_t>(mx * my);
  if (u_len != states) return fail(err, err_len, "ugrid_create: u length must be ncase * 4 * (nx + 4) * (ny + 4)");

  ugrid_session* s = new ugrid_session();
  s->par = p;
  s->states = states;
  Grid& g = s->g;
  g.nx = setup->nx;
  g.ny = setup->ny;
  g.mx = static_cast<int>(mx);
  g.my = static_cast<int>(my);
  g.ncase = setup->ncase;
  g.plane = static_cast<size_t>(mx * my);
  for (int k = 0; k < 4; ++k) g.bc[k] = p.bc[k];
  g.ausm = p.flux == 1;
  g.gamma = p.gamma;
  g.cfl = p.cfl;
  g.dt_fixed = p.dt_fixed;
  g.pseudo0 = p.pseudo_cfl;
  g.rtol = p.implicit_rtol;
  g.atol = p.implicit_atol;
  g.maxiter = p.implicit_maxiter;
  g.rows = choose_rows(g.nx, g.ny, g.ncase, setup->cut != nullptr);
  g.strips_x = (g.nx + kStripCells - 1) / kStripCells;
  g.strips_y = (g.ny + g.rows - 1) / g.rows;
  const long long strips = static_cast<long long>(g.strips_x) * g.strips_y * g.ncase;
  if (strips > (1LL << 30)) {
    release(s);
    return fail(err, err_len, "ugrid_create: grid too large");
  }
  g.strips = static_cast<int>(strips);
  g.blocks = (g.strips + kWaves - 1) / kWaves;
  g.use_part = g.ncase <= kPartCases ? 1 : 0;
  s->launch_blocks = (g.blocks + kXcds - 1) / kXcds * kXcds;

  std::vector<double> mco(g.ncase, p.ausm_mco);
  if (setup->mco)
    for (int c = 0; c < g.ncase; ++c) mco[c] = setup->mco[c];
  std::vector<double> t0(g.ncase, 0.0), dt0(g.ncase, 0.0);
  if (t)
    for (int c = 0; c < g.ncase; ++c) t0[c] = t[c];
  if (dt)
    for (int c = 0; c < g.ncase; ++c) dt0[c] = dt[c];

  const auto plain_value = [](double x) { return x > kPlainLow && x < kPlainHigh; };
  bool plain = plain_value(p.gamma - 1.0) && plain_value(p.gamma);
  for (int k = 0; k < g.mx; ++k) plain = plain && plain_value(setup->dx[k]);
  for (int k = 0; k < g.my; ++k) plain = plain && plain_value(setup->dy[k]);
  for (int c = 0; g.ausm && c < g.ncase; ++c) plain = plain && plain_value(mco[c]);  // (HLLC reads none)
  g.plain = plain ? 1 : 0;

  double *dxd = nullptr, *dyd = nullptr, *rdx = nullptr, *rdy = nullptr, *mcod = nullptr;
  if (!ok(hipGetDevice(&s->device), err, err_len, "hipGetDevice") ||
      !ok(hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking), err, err_len, "hipStreamCreate") ||
      !ok(hipHostMalloc(reinterpret_cast<void**>(&s->host_ctrl), sizeof(Control), hipHostMallocDefault), err, err_len,
          "hipHostMalloc") ||
      !device_alloc(s, &g.B[0], states, err, err_len) || !device_alloc(s, &g.B[1], states, err, err_len) ||
      !device_alloc(s, &g.B[2], states, err, err_len)) {
    release(s);
    return 3;
  }
  // The arrays that are small beside a state share one allocation (a hipMalloc each made the creation of a
  // small grid longer: one case of 40 x 40 350 -> 310 us).
  {
    SmallArrays small;
    const size_t cases = g.ncase;
    small.add(&dxd, g.mx), small.add(&rdx, g.mx), small.add(&dyd, g.my), small.add(&rdy, g.my);
    small.add(&mcod, cases), small.add(&g.t, cases), small.add(&g.dt, cases), small.add(&g.dt_out, cases);
    small.add(&g.smax, cases), small.add(&g.norm, cases), small.add(&g.initial, cases);
    small.add(&g.part, g.use_part ? g.strips : 1), small.add(&g.ctrl, 1);
    if (!small.allocate(s, err, err_len)) {
      release(s);
      return 3;
    }
  }
  g.dx = dxd;
  g.dy = dyd;
  g.rdx = rdx;
  g.rdy = rdy;
  g.mco = mcod;
  Control c0{};
  c0.status = 0;
  const hipMemcpyKind h2d = hipMemcpyHostToDevice;
  const size_t bytes = states * sizeof(double);
  // Every buffer that can come to hold the accepted state starts as the upload, so its ghost
  // cells are the entry values (only a download after the first step writes ghost cells).
  if (!ok(hipMemcpyAsync(g.B[0], u, bytes, h2d, s->stream), err, err_len, "upload state") ||
      !ok(hipMemcpyAsync(g.B[1], u, bytes, h2d, s->stream), err, err_len, "upload state") ||
      !ok(hipMemcpyAsync(g.B[2], u, bytes, h2d, s->stream), err, err_len, "upload state") ||
      !ok(hipMemsetAsync(g.norm, 0, g.ncase * sizeof(unsigned long long), s->stream), err, err_len, "clear norms") ||
      !ok(hipMemcpyAsync(dxd, setup->dx, g.mx * sizeof(double), h2d, s->stream), err, err_len, "upload dx") ||
      !ok(hipMemcpyAsync(dyd, setup->dy, g.my * sizeof(double), h2d, s->stream), err, err_len, "upload dy") ||
      !ok(hipMemcpyAsync(mcod, mco.data(), g.ncase * sizeof(double), h2d, s->stream), err, err_len, "upload mco") ||
      !ok(hipMemcpyAsync(g.t, t0.data(), g.ncase * sizeof(double), h2d, s->stream), err, err_len, "upload t") ||
      !ok(hipMemcpyAsync(g.dt, dt0.data(), g.ncase * sizeof(double), h2d, s->stream), err, err_len, "upload dt") ||
      !ok(hipMemcpyAsync(g.dt_out, dt0.data(), g.ncase * sizeof(double), h2d, s->stream), err, err_len,
          "upload dt") ||
      !ok(hipMemsetAsync(g.smax, 0, g.ncase * sizeof(unsigned long long), s->stream), err, err_len, "clear bound") ||
      !ok(hipMemcpyAsync(g.ctrl, &c0, sizeof(Control), h2d, s->stream), err, err_len, "upload control") ||
      !ok(hipStreamSynchronize(s->stream), err, err_len, "upload")) {
    release(s);
    return 3;
  }
  hipLaunchKernelGGL(k_recip, dim3(grid_blocks(g, g.mx + static_cast<size_t>(g.my))), dim3(kThreads), 0, s->stream, dxd,
                     rdx, g.mx, dyd, rdy, g.my);
  if (!ok(hipGetLastError(), err, err_len, "cell widths")) {
    release(s);
    return 3;
  }
  s->mco = mco;
  if (setup->cut && !upload_cut(s, *setup->cut, setup->dx, setup->dy, err, err_len)) {
    release(s);
    return 3;
  }
  const int trials = g.nx * static_cast<long long>(g.ny) * g.ncase >= (1 << 22) ? 4 : 16;
  const bool implicit = p.time_integrator == 1;
  if (!build_graph(s, implicit ? trials / 4 : trials, err, err_len)) {
    release(s);
    return 3;
  }
  *out = s;
  return 0;
}

extern "C" int ugrid_run(ugrid_session* s, double tend, int64_t maxsteps, ugrid_meta* meta, char* err,
                         size_t err_len) {
  if (!s) return fail(err, err_len, "ugrid_run: null session");
  const Grid& g = s->g;
  const bool implicit = s->par.time_integrator == 1;
  if (implicit) {
    // implicit2d_validate (src/implicit2d.cpp:11-35): controls, times and reference Mach numbers.
    const ugrid_params& p = s->par;
    std::vector<double> t(g.ncase);
    if (!ok(hipMemcpyAsync(t.data(), g.t, g.ncase * sizeof(double), hipMemcpyDeviceToHost, s->stream), err, err_len,
            "download t") ||
        !ok(hipStreamSynchronize(s->stream), err, err_len, "download t"))
      return 3;
    bool valid = std::isfinite(tend) && maxsteps >= 0 && p.gamma > 1.0 && std::isfinite(p.gamma) && p.cfl > 0.0 &&
                 std::isfinite(p.cfl) && p.dt_fixed >= 0.0 && std::isfinite(p.dt_fixed) && p.pseudo_cfl > 0.0 &&
                 std::isfinite(p.pseudo_cfl) && p.implicit_maxiter >= 1 && p.implicit_rtol >= 0.0 &&
                 std::isfinite(p.implicit_rtol) && p.implicit_atol > 0.0 && std::isfinite(p.implicit_atol);
    for (int c = 0; c < g.ncase; ++c)
      valid = valid && std::isfinite(t[c]) && s->mco[c] > 0.0 && std::isfinite(s->mco[c]);
    if (!valid) return fail(err, err_len, "invalid backward-Euler controls");
    const size_t cells = static_cast<size_t>(g.nx) * g.ny * g.ncase;
    hipLaunchKernelGGL(k_check_state, dim3(grid_blocks(g, cells)), dim3(kThreads), 0, s->stream, g);
    hipLaunchKernelGGL(k_be_start, dim3(1), dim3(kLanes), 0, s->stream, g, tend, static_cast<long long>(maxsteps));
  } else {
    launch_bound(s);
    hipLaunchKernelGGL(k_open, dim3(1), dim3(kThreads), 0, s->stream, g, tend, static_cast<long long>(maxsteps));
  }
  if (!ok(hipGetLastError(), err, err_len, "run start")) return 3;
  // Every replay of a running batch takes at least one decision (a commit, a rejection, a
  // phase change), so it must move the event count; a replay that does not is reported, not
  // waited on.
  long long progress = -1;
  long long steps = 0, used = 0;  // backward Euler: steps, and update kernels that they used, up to the last poll
  for (;;) {
    if (!ok(hipMemcpyAsync(s->host_ctrl, g.ctrl, sizeof(Control), hipMemcpyDeviceToHost, s->stream), err, err_len,
            "control copy") ||
        !ok(hipStreamSynchronize(s->stream), err, err_len, "trial"))
      return 3;
    const long long made = s->host_ctrl->nsteps - steps, tries = s->host_ctrl->checks + s->host_ctrl->iretries - used;
    steps += made;
    used += tries;
    if (implicit && progress != -1) s->few_checks = made > 0 && tries <= kFewChecks * made;
    if (s->host_ctrl->status != RUNNING) break;
    const long long now = s->host_ctrl->events;
    if (now == progress) return fail(err, err_len, "ugrid_run: device step control made no progress");
    progress = now;
    if (s->few_checks) {
      // (Launched directly: a second graph would take longer to make than short runs take.)
      const long long left = s->host_ctrl->maxsteps - s->host_ctrl->steps;
      const long long rounds = std::clamp<long long>(left, 1, kShortRounds);
      for (long long k = 0; k < rounds; ++k) launch_be_round(s, s->stream, 1);
      if (!ok(hipGetLastError(), err, err_len, "round launch")) return 3;
      continue;
    }
    if (!ok(hipGraphLaunch(s->exec, s->stream), err, err_len, "trial graph")) return 3;
  }
  const Control& c = *s->host_ctrl;
  if (meta) {
    meta->nsteps = c.nsteps;
    meta->nreject = c.nreject;
  }
  char line[256];
  line[0] = 0;
  if (implicit) {
    if (c.reason == WHY_INITIAL)
      std::snprintf(line, sizeof(line), "backward Euler: invalid initial fluid state");
    else if (c.reason == WHY_PSEUDO)
      std::snprintf(line, sizeof(line), "backward Euler: nonphysical pseudo candidate; physical step not accepted");
    else if (c.reason == WHY_DEFECT)
      std::snprintf(line, sizeof(line), "backward Euler: non-finite defect; physical step not accepted");
    else if (c.reason == WHY_MAXITER)
      std::snprintf(line, sizeof(line),
                    "backward Euler not converged: step=%lld updates=%d initial=%.6e defect=%.6e tolerance=%.6e; "
                    "physical step not accepted",
                    c.nsteps, c.iter, c.initial_defect, c.final_defect, c.tolerance);
    else if (c.reason == WHY_DT)
      std::snprintf(line, sizeof(line), "backward Euler: physical dt is invalid or cannot advance time");
  } else if (c.status == 2) {
    std::snprintf(line, sizeof(line), "non-physical RK candidate after %d retries at accepted step %lld", c.retries,
                  c.nsteps);
  }
  if (line[0]) fail(err, err_len, line);
  return c.status;
}

extern "C" int ugrid_download(ugrid_session* s, double* u, uint64_t u_len, double* t, double* dt, char* err,
                              size_t err_len) {
  if (!s) return fail(err, err_len, "ugrid_download: null session");
  if (u && u_len != s->states) return fail(err, err_len, "ugrid_download: u length mismatch");
  const Grid& g = s->g;
  Control c{};
  if (!ok(hipMemcpyAsync(&c, g.ctrl, sizeof(Control), hipMemcpyDeviceToHost, s->stream), err, err_len, "control") ||
      !ok(hipStreamSynchronize(s->stream), err, err_len, "control"))
    return 3;
  const size_t bytes = s->states * sizeof(double);
  // Once a step has begun, the ghosts are a boundary fill that the device makes in the accepted
  // state's own buffer (its kernels never read ghost cells): one copy, instead of a second state
  // beside it and two passes of the host over both (8 cases of 1024 x 1024: the Python pull, which
  // copies the state once more on the host, 123 -> 19 ms).
  if (u && c.ghost_from != 0 && g.nx >= 2 && g.ny >= 2 && g.my <= 65535 && 4LL * g.ncase <= 65535) {
    const double* from = c.ghost_from == 1 ? g.B[c.cur] : g.B[c.cur ^ 1];
    hipLaunchKernelGGL(k_fill_ghosts, dim3(g.my, 4 * g.ncase), dim3(kThreads), 0, s->stream, g, from, g.B[c.cur]);
    if (!ok(hipGetLastError(), err, err_len, "ghost cells") ||
        !ok(hipMemcpyAsync(u, g.B[c.cur], bytes, hipMemcpyDeviceToHost, s->stream), err, err_len, "download") ||
        !ok(hipStreamSynchronize(s->stream), err, err_len, "download"))
      return 3;
  } else if (u) {
    if (!ok(hipMemcpyAsync(u, g.B[c.cur], bytes, hipMemcpyDeviceToHost, s->stream), err, err_len, "download") ||
        !ok(hipStreamSynchronize(s->stream), err, err_len, "download"))
      return 3;
    // (Before the first step, and in backward Euler, every buffer's ghosts are still the uploaded ones.)
    std::vector<double> other;
    const double* ghosts = nullptr;
    if (c.ghost_from == 1) {
      fill_ghosts(g, u);
    } else if (c.ghost_from == 2) {
      other.resize(s->states);
      if (!ok(hipMemcpyAsync(other.data(), g.B[c.cur ^ 1], bytes, hipMemcpyDeviceToHost, s->stream), err, err_len,
              "download") ||
          !ok(hipStreamSynchronize(s->stream), err, err_len, "download"))
        return 3;
      fill_ghosts(g, other.data());
      ghosts = other.data();
    }
    if (ghosts)
      for (size_t cv = 0; cv < static_cast<size_t>(g.ncase) * 4; ++cv)
        for (int j = 0; j < g.my; ++j)
          for (int i = 0; i < g.mx; ++i) {
            if (i >= kGhosts && i < g.nx + kGhosts && j >= kGhosts && j < g.ny + kGhosts) continue;
            const size_t k = cv * g.plane + static_cast<size_t>(j) * g.mx + i;
            u[k] = ghosts[k];
          }
  }
  if (t && !ok(hipMemcpyAsync(t, g.t, g.ncase * sizeof(double), hipMemcpyDeviceToHost, s->stream), err, err_len,
                "download t"))
    return 3;
  if (dt && !ok(hipMemcpyAsync(dt, g.dt_out, g.ncase * sizeof(double), hipMemcpyDeviceToHost, s->stream), err,
                 err_len, "download dt"))
    return 3;
  return ok(hipStreamSynchronize(s->stream), err, err_len, "download") ? 0 : 3;
}

extern "C" int ugrid_rhs(ugrid_session* s, const double* u, uint64_t u_len, double* r, char* err, size_t err_len) {
  if (!s || !u || !r) return fail(err, err_len, "ugrid_rhs: null argument");
  if (u_len != s->states) return fail(err, err_len, "ugrid_rhs: u length mismatch");
  const size_t bytes = s->states * sizeof(double);
  if (!s->R && !device_alloc(s, &s->R, s->states, err, err_len)) return 3;
  if (!s->rhs_in && !device_alloc(s, &s->rhs_in, s->states, err, err_len)) return 3;
  hipLaunchKernelGGL(k_zero, dim3(1024), dim3(kThreads), 0, s->stream, s->R, s->states);
  if (!ok(hipMemcpyAsync(s->rhs_in, u, bytes, hipMemcpyHostToDevice, s->stream), err, err_len, "upload state"))
    return 3;
  launch_stage<0>(s, s->stream, s->rhs_in, s->R);
  if (!ok(hipGetLastError(), err, err_len, "residual launch") ||
      !ok(hipMemcpyAsync(r, s->R, bytes, hipMemcpyDeviceToHost, s->stream), err, err_len, "download residual") ||
      !ok(hipStreamSynchronize(s->stream), err, err_len, "residual"))
    return 3;
  return 0;
}

extern "C" int ugrid_implicit_stats(const ugrid_session* s, ugrid_implicit_info* out) {
  if (!s || !out) return 1;
  Control c{};
  if (hipMemcpyAsync(&c, s->g.ctrl, sizeof(Control), hipMemcpyDeviceToHost, s->stream) != hipSuccess ||
      hipStreamSynchronize(s->stream) != hipSuccess)
    return 1;
  out->updates = c.updates;
  out->retries = c.iretries;
  out->checks = c.checks;
  out->reason = c.reason;
  out->initial_defect = c.initial_defect;
  out->final_defect = c.final_defect;
  out->tolerance = c.tolerance;
  return 0;
}

extern "C" int ugrid_profile(ugrid_session* s, int32_t trials, double* stage_us, char* err, size_t err_len) {
  if (!s || !stage_us || trials < 1) return fail(err, err_len, "ugrid_profile: invalid argument");
  if (s->par.time_integrator != 0) return fail(err, err_len, "ugrid_profile: SSP-RK3 sessions only");
  const Grid& g = s->g;
  launch_bound(s);
  hipLaunchKernelGGL(k_open, dim3(1), dim3(kThreads), 0, s->stream, g, HUGE_VAL, (1LL << 62));
  std::vector<hipEvent_t> ev(4 * static_cast<size_t>(trials), nullptr);
  bool good = true;
  for (auto& e : ev) good = good && hipEventCreate(&e) == hipSuccess;
  for (int k = 0; good && k < trials; ++k) {
    hipEvent_t* e = &ev[4 * static_cast<size_t>(k)];
    (void)hipEventRecord(e[0], s->stream);
    launch_stage_srd<1>(s, s->stream);
    (void)hipEventRecord(e[1], s->stream);
    launch_stage_srd<2>(s, s->stream);
    (void)hipEventRecord(e[2], s->stream);
    launch_stage_srd<3>(s, s->stream);
    (void)hipEventRecord(e[3], s->stream);
    hipLaunchKernelGGL(k_commit, dim3(1), dim3(kDecide), 0, s->stream, g);
  }
  good = good && ok(hipGetLastError(), err, err_len, "profile launch") &&
         ok(hipStreamSynchronize(s->stream), err, err_len, "profile");
  double sum[3] = {0, 0, 0};
  for (int k = 0; good && k < trials; ++k)
    for (int q = 0; q < 3; ++q) {
      float ms = 0;
      good = good && ok(hipEventElapsedTime(&ms, ev[4 * static_cast<size_t>(k) + q], ev[4 * static_cast<size_t>(k) + q + 1]),
                        err, err_len, "profile events");
      sum[q] += ms;
    }
  for (auto& e : ev)
    if (e) (void)hipEventDestroy(e);
  if (!good) return 3;
  for (int q = 0; q < 3; ++q) stage_us[q] = 1e3 * sum[q] / trials;
  return 0;
}

extern "C" int ugrid_device_available(char* reason, size_t reason_len) {
  int count = 0;
  const hipError_t e = hipGetDeviceCount(&count);
  char line[256];
  if (e != hipSuccess || count <= 0) {
    std::snprintf(line, sizeof(line), "hipGetDeviceCount: %s (devices=%d)", hipGetErrorString(e), count);
    fail(reason, reason_len, line);
    return 0;
  }
  int device = 0;
  hipDeviceProp_t p{};
  if (hipGetDevice(&device) != hipSuccess || hipGetDeviceProperties(&p, device) != hipSuccess) {
    fail(reason, reason_len, "hipGetDeviceProperties failed");
    return 0;
  }
  std::snprintf(line, sizeof(line), "%s, %s", p.name, p.gcnArchName);
  fail(reason, reason_len, line);
  return 1;
}

extern "C" int ugrid_get_launch(const ugrid_session* s, ugrid_launch_info* out) {
  if (!s || !out) return 1;
  out->rows = s->g.rows;
  out->strips = s->g.strips;
  out->blocks = s->launch_blocks;
  out->threads = kThreads;
  return 0;
}

extern "C" void ugrid_destroy(ugrid_session* s) {
  if (!s) return;
  (void)hipSetDevice(s->device);
  (void)hipStreamSynchronize(s->stream);
  release(s);
}
