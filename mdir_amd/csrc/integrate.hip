// integrate.hip — velocity Verlet with SETTLE waters, in f64.
//
// Reference semantics: dyn.kick / dyn.drift (lib/Driver/DynamicsIR.cpp:102-112)
// fused as the integration run of MDExecKernels.cpp:1121 (08-gpu.md:112-121):
//   half kick, drift, SETTLE positions (ConstraintIR.cpp:473-593, the method
//   of Miyamoto & Kollman, J. Comput. Chem. 13, 952 (1992)), v += dx_c/dt,
//   the validity test |x - x_ref|^2 > (skin/2)^2 (ExposeValidity.cpp:23);
//   then after the forces: half kick and the velocity constraint
//   (ConstraintIR.cpp:392-471).
// A unit is a SETTLE water (3 consecutive atoms), a constraint cluster (an
// atom and up to four atoms bonded to it at fixed lengths, consecutive,
// M-SHAKE as ConstraintIR.cpp:595-747 takes it) or a free atom.  A block
// takes the atoms of its units a thread per atom (loads, half kick, noise,
// stores; the whole step of a free atom) and their constraints a thread per
// unit, through LDS (integrate_units).
#include "md_common.h"

namespace mdhip {

// The integrator's f64 arithmetic is rounded operation by operation as
// written (no contraction into fused multiply-adds): a step then gives the
// same bits whether its two halves run in one launch (kBetween) or two,
// and follows the oracle's integration, which rounds each operation.
#pragma clang fp contract(off)

struct IntParams {
  double dt;
  double skin_half2;     // (outer list buffer / 2)^2: rebuild beyond it
  double prune_half2;    // (pruned list buffer / 2)^2: prune again beyond it
  const double *x_prune; // positions at the last prune (atom order), or null
  double half_box[3];
  double m_o, m_h;
  double ra, rb, rc;   // SETTLE canonical triangle
  double d_oh, d_hh;
  // Langevin dynamics (langevin != 0): the g-BAOAB step with the O step
  // v <- decay v + spread / sqrt(m) R, decay = exp(-gamma dt) and
  // spread = sqrt((1 - decay^2) kB T); R from langevin_normals(seed, step,
  // atom).  A first half takes step number *step + offset; the launch that
  // closes a sequence of steps adds `advance`, their count, to *step (no
  // launch that reads the number runs beside it).
  int langevin;
  double decay, spread;
  unsigned long long seed;
  long long *step;
  int offset, advance;
  // constraint clusters: each member's bond length to its centre, by atom,
  // and the inverse masses (the descent step of a minimisation)
  const double *clen;
  const double *inv_mass;
};

// A unit's code (unit_size[u]): its atom count in bits 0-7, kUnitCluster
// for a constraint cluster, the cluster centre's offset from the unit's
// first atom in bits 12-15.
constexpr int kUnitCluster = 0x100;
constexpr int kUnitCentreShift = 12;

__device__ __forceinline__ void cross(const double *a, const double *b, double *c) {
  c[0] = a[1] * b[2] - a[2] * b[1];
  c[1] = a[2] * b[0] - a[0] * b[2];
  c[2] = a[0] * b[1] - a[1] * b[0];
}
__device__ __forceinline__ double dot(const double *a, const double *b) {
  return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}
__device__ __forceinline__ void unit(double *a) {
  const double s = rsqrt(dot(a, a));
  a[0] *= s;
  a[1] *= s;
  a[2] *= s;
}

// SETTLE of one water: old positions A0 B0 C0 (satisfying the constraints),
// new unconstrained A1 B1 C1 -> constrained, in place.
__device__ void settle_positions(const double *A0, const double *B0, const double *C0,
                                 double *A1, double *B1, double *C1,
                                 const IntParams &p) {
  const double total = p.m_o + 2.0 * p.m_h;
  double b0[3], c0[3], b1r[3], c1r[3];
  for (int k = 0; k < 3; ++k) {
    b0[k] = B0[k] - A0[k];
    c0[k] = C0[k] - A0[k];
    b1r[k] = B1[k] - A1[k];
    c1r[k] = C1[k] - A1[k];
  }
  double com[3], a1[3], b1[3], c1[3];
  for (int k = 0; k < 3; ++k) {
    com[k] = p.m_h / total * (b1r[k] + c1r[k]);
    a1[k] = -com[k];
    b1[k] = b1r[k] - com[k];
    c1[k] = c1r[k] - com[k];
  }
  double ez[3], ex[3], ey[3];
  cross(b0, c0, ez);
  unit(ez);
  cross(a1, ez, ex);
  unit(ex);
  cross(ez, ex, ey);
  const double xb0 = dot(b0, ex), yb0 = dot(b0, ey);
  const double xc0 = dot(c0, ex), yc0 = dot(c0, ey);
  const double za1 = dot(a1, ez);
  const double xb1 = dot(b1, ex), yb1 = dot(b1, ey), zb1 = dot(b1, ez);
  const double xc1 = dot(c1, ex), yc1 = dot(c1, ey), zc1 = dot(c1, ez);
  const double sinphi = za1 / p.ra;
  const double cosphi = sqrt(1.0 - sinphi * sinphi);
  const double sinpsi = (zb1 - zc1) / (2.0 * p.rc * cosphi);
  const double cospsi = sqrt(1.0 - sinpsi * sinpsi);
  const double ya2 = p.ra * cosphi;
  const double xb2 = -p.rc * cospsi;
  const double t1 = -p.rb * cosphi, t2 = p.rc * sinpsi * sinphi;
  const double yb2 = t1 - t2, yc2 = t1 + t2;
  const double alpha = xb2 * (xb0 - xc0) + yb0 * yb2 + yc0 * yc2;
  const double beta = xb2 * (yc0 - yb0) + xb0 * yb2 + xc0 * yc2;
  const double gamma = (xb0 * yb1 - xb1 * yb0) + (xc0 * yc1 - xc1 * yc0);
  const double both = alpha * alpha + beta * beta;
  const double sintheta = (alpha * gamma - beta * sqrt(both - gamma * gamma)) / both;
  const double costheta = sqrt(1.0 - sintheta * sintheta);
  const double xa3 = -ya2 * sintheta, ya3 = ya2 * costheta;
  const double xb3 = xb2 * costheta - yb2 * sintheta;
  const double yb3 = xb2 * sintheta + yb2 * costheta;
  const double xc3 = -xb2 * costheta - yc2 * sintheta;
  const double yc3 = -xb2 * sintheta + yc2 * costheta;
  double base[3] = {A1[0], A1[1], A1[2]};
  for (int k = 0; k < 3; ++k) {
    A1[k] = base[k] + xa3 * ex[k] + ya3 * ey[k] + za1 * ez[k] + com[k];
    B1[k] = base[k] + xb3 * ex[k] + yb3 * ey[k] + zb1 * ez[k] + com[k];
    C1[k] = base[k] + xc3 * ex[k] + yc3 * ey[k] + zc1 * ez[k] + com[k];
  }
}

__device__ __forceinline__ double det3(double m00, double m01, double m02, double m10,
                                       double m11, double m12, double m20, double m21,
                                       double m22) {
  return m00 * (m11 * m22 - m12 * m21) - m01 * (m10 * m22 - m12 * m20) +
         m02 * (m10 * m21 - m11 * m20);
}

// Impulses along the three bonds that zero the bond-relative velocities.
__device__ void settle_velocities(const double *xa, const double *xb, const double *xc,
                                  double *va, double *vb, double *vc,
                                  const IntParams &p) {
  const double io = 1.0 / p.m_o, ih = 1.0 / p.m_h;
  double e0[3], e1[3], e2[3], dvb[3], dvc[3], dvcb[3];
  for (int k = 0; k < 3; ++k) {
    e0[k] = xb[k] - xa[k];
    e1[k] = xc[k] - xa[k];
    e2[k] = xc[k] - xb[k];
    dvb[k] = vb[k] - va[k];
    dvc[k] = vc[k] - va[k];
    dvcb[k] = vc[k] - vb[k];
  }
  unit(e0);
  unit(e1);
  unit(e2);
  const double r0 = -dot(e0, dvb), r1 = -dot(e1, dvc), r2 = -dot(e2, dvcb);
  const double a00 = io + ih, a11 = io + ih, a22 = 2.0 * ih;
  const double a01 = dot(e0, e1) * io;
  const double a02 = -dot(e0, e2) * ih;
  const double a12 = dot(e1, e2) * ih;
  const double det = det3(a00, a01, a02, a01, a11, a12, a02, a12, a22);
  const double s0 = det3(r0, a01, a02, r1, a11, a12, r2, a12, a22) / det;
  const double s1 = det3(a00, r0, a02, a01, r1, a12, a02, r2, a22) / det;
  const double s2 = det3(a00, a01, r0, a01, a11, r1, a02, a12, r2) / det;
  for (int k = 0; k < 3; ++k) {
    const double i0 = s0 * e0[k], i1 = s1 * e1[k], i2 = s2 * e2[k];
    va[k] += -io * (i0 + i1);
    vb[k] += ih * (i0 - i2);
    vc[k] += ih * (i1 + i2);
  }
}

// The state of one unit of S atoms (a SETTLE water, S = 3, a constraint
// cluster, S = 2..5, with its centre at index 0): S is a compile-time constant
// so that the arrays stay in registers.
template <int S>
struct UnitState {
  double im[S], x[S][3], v[S][3];
  double len[S];  // clusters: index m's bond length to the centre
};

// Linear equations A y = b of at most 4 unknowns by elimination (the
// cluster equations are diagonally dominant: no pivoting).  One reciprocal
// per pivot: a chain of f64 divisions is what a sweep waits for.
template <int M>
__device__ __forceinline__ void solve_small(double (&A)[M][M], double (&b)[M]) {
  double inv[M];
#pragma unroll
  for (int i = 0; i < M; ++i) {
    inv[i] = 1.0 / A[i][i];
#pragma unroll
    for (int r = i + 1; r < M; ++r) {
      const double f = A[r][i] * inv[i];
#pragma unroll
      for (int c = i; c < M; ++c) A[r][c] -= f * A[i][c];
      b[r] -= f * b[i];
    }
  }
#pragma unroll
  for (int i = M - 1; i >= 0; --i) {
    double sum = b[i];
#pragma unroll
    for (int c = i + 1; c < M; ++c) sum -= A[i][c] * b[c];
    b[i] = sum * inv[i];
  }
}

// M-SHAKE of a cluster (centre at index 0): six Newton sweeps of the
// linearized bond equations sum_l 2 (r_k . s_l) w_kl lambda_l = d_k^2 -
// r_k . r_k, the members moving by +lambda_l s_l / m_l along the old bonds
// s_l and the centre by -sum_l lambda_l s_l / m_0 (w_kk = 1/m_0 + 1/m_k,
// w_kl = 1/m_0), the sweeps of the reference (ConstraintIR.cpp:595-747).
template <int S>
__device__ __forceinline__ void mshake_positions(const double (&x0)[S][3], double (&xn)[S][3],
                                                 const double (&im)[S],
                                                 const double (&len)[S]) {
  constexpr int M = S - 1;
  double sv[M][3], d2[M];
#pragma unroll
  for (int k = 0; k < M; ++k) {
    d2[k] = len[k + 1] * len[k + 1];
#pragma unroll
    for (int j = 0; j < 3; ++j) sv[k][j] = x0[k + 1][j] - x0[0][j];
  }
  for (int sweep = 0; sweep < 6; ++sweep) {
    double r[M][3], A[M][M], lam[M];
#pragma unroll
    for (int k = 0; k < M; ++k) {
#pragma unroll
      for (int j = 0; j < 3; ++j) r[k][j] = xn[k + 1][j] - xn[0][j];
      lam[k] = d2[k] - dot(r[k], r[k]);
    }
#pragma unroll
    for (int k = 0; k < M; ++k)
#pragma unroll
      for (int l = 0; l < M; ++l) A[k][l] = 2.0 * dot(r[k], sv[l]) * ((k == l) ? im[0] + im[k + 1] : im[0]);
    solve_small<M>(A, lam);
#pragma unroll
    for (int l = 0; l < M; ++l)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        xn[0][j] -= lam[l] * sv[l][j] * im[0];
        xn[l + 1][j] += lam[l] * sv[l][j] * im[l + 1];
      }
  }
}

// The velocity constraint of a cluster: impulses mu_l along the bonds r_l
// with sum_l (r_k . r_l) w_kl mu_l = -r_k . (v_k - v_0), one solve.
template <int S>
__device__ __forceinline__ void rattle_velocities(const double (&x)[S][3], double (&v)[S][3],
                                                  const double (&im)[S]) {
  constexpr int M = S - 1;
  double r[M][3], A[M][M], mu[M];
#pragma unroll
  for (int k = 0; k < M; ++k) {
    double dv[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      r[k][j] = x[k + 1][j] - x[0][j];
      dv[j] = v[k + 1][j] - v[0][j];
    }
    mu[k] = -dot(r[k], dv);
  }
#pragma unroll
  for (int k = 0; k < M; ++k)
#pragma unroll
    for (int l = 0; l < M; ++l) A[k][l] = dot(r[k], r[l]) * ((k == l) ? im[0] + im[k + 1] : im[0]);
  solve_small<M>(A, mu);
#pragma unroll
  for (int l = 0; l < M; ++l)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      v[0][j] -= mu[l] * r[l][j] * im[0];
      v[l + 1][j] += mu[l] * r[l][j] * im[l + 1];
    }
}

// The atoms of a block's units in LDS, slot t of every array belonging to
// thread t (a unit's members are consecutive slots): positions, velocities,
// the half kick dt/2 f/m, the noise spread/sqrt(m) R of a Langevin step, the
// inverse masses and the bond lengths.
constexpr int kIntThreads = 192;
struct UnitLds {
  double x[3][kIntThreads], v[3][kIntThreads], kick[3][kIntThreads], noise[3][kIntThreads];
  double im[kIntThreads], len[kIntThreads];
};

template <int S, bool CL>
__device__ __forceinline__ void constrain_velocities(UnitState<S> &s, const double (&x)[S][3],
                                                     const IntParams &p) {
  if constexpr (CL) rattle_velocities<S>(x, s.v, s.im);
  else if constexpr (S == 3) settle_velocities(x[0], x[1], x[2], s.v[0], s.v[1], s.v[2], p);
}

// A drift of length h from positions x0 (constrained): xn = x0 + h v,
// SETTLE or M-SHAKE from x0, and v += (xn_constrained - xn) / h.
template <int S, bool CL>
__device__ __forceinline__ void drift_settle(const UnitState<S> &s, const double (&x0)[S][3],
                                             double (&v)[S][3], double (&xn)[S][3], double h,
                                             const IntParams &p) {
#pragma unroll
  for (int m = 0; m < S; ++m)
#pragma unroll
    for (int k = 0; k < 3; ++k) xn[m][k] = x0[m][k] + h * v[m][k];
  if constexpr (CL || S == 3) {
    double xu[S][3];
#pragma unroll
    for (int m = 0; m < S; ++m)
#pragma unroll
      for (int k = 0; k < 3; ++k) xu[m][k] = xn[m][k];
    if constexpr (CL) mshake_positions<S>(x0, xn, s.im, s.len);
    else settle_positions(x0[0], x0[1], x0[2], xn[0], xn[1], xn[2], p);
    const double ih = 1.0 / h;
#pragma unroll
    for (int m = 0; m < S; ++m)
#pragma unroll
      for (int k = 0; k < 3; ++k) v[m][k] += (xn[m][k] - xu[m][k]) * ih;
  }
}

// Which halves of velocity Verlet a launch runs on each unit.
enum StepPart { kFirstHalf = 1, kSecondHalf = 2, kBetween = 3 };

// The unit whose members are slots t .. t + S - 1: kicks, constraints and
// drifts, LDS to LDS.  A step is a sequence of stages, each the velocity
// constraint at x and then a drift from x:
//   end of a step (kSecondHalf)   constraint; the kick that starts the next
//                                 step (kBetween)
//   velocity Verlet               drift of dt
//   Langevin                      constraint, drift of dt/2; O step; both
//                                 again
// (the g-BAOAB geodesic integrator of Leimkuhler and Matthews, Proc. R. Soc.
// A 472, 20160138, 2016, as the reference's Langevin step with constraints
// takes it, lib/Driver/DynamicsIR.cpp, the geodesic branch: project v onto
// the constraints; A: half drift, SETTLE, v += dx_c / (dt/2); O: v <- decay
// v + spread / sqrt(m) R, projected again at the new positions; A: half
// drift from there.  The closing B, kick and projection, is the second half
// of the step, as in velocity Verlet.)  One loop over the stages holds the
// constraint and the drift once: the kernel runs its code once per launch,
// so what it waits for is its instructions' way to the CU.
template <int PART, int S, bool CL>
__device__ __forceinline__ void step_unit(UnitLds &l, int t, const IntParams &p) {
  UnitState<S> s;
#pragma unroll
  for (int m = 0; m < S; ++m) {
    s.im[m] = l.im[t + m];
    s.len[m] = CL ? l.len[t + m] : 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      s.x[m][k] = l.x[k][t + m];
      s.v[m][k] = l.v[k][t + m] + l.kick[k][t + m];
    }
  }
  const bool langevin = (PART & kFirstHalf) && p.langevin;
  const int drifts = PART & kFirstHalf ? (langevin ? 2 : 1) : 0;
  const double h = langevin ? 0.5 * p.dt : p.dt;
#pragma unroll 1
  for (int stage = PART & kSecondHalf ? 0 : 1; stage <= drifts; ++stage) {
    if (stage == 0 || langevin) constrain_velocities<S, CL>(s, s.x, p);
    if (stage == 0) {
      if (PART == kBetween) {
#pragma unroll
        for (int m = 0; m < S; ++m)
#pragma unroll
          for (int k = 0; k < 3; ++k) s.v[m][k] = s.v[m][k] + l.kick[k][t + m];
      }
      continue;
    }
    double xn[S][3];
    drift_settle<S, CL>(s, s.x, s.v, xn, h, p);
#pragma unroll
    for (int m = 0; m < S; ++m)
#pragma unroll
      for (int k = 0; k < 3; ++k) s.x[m][k] = xn[m][k];
    if (stage == 1 && langevin) {
#pragma unroll
      for (int m = 0; m < S; ++m) {
        if (!(s.im[m] > 0.0)) continue;  // a particle without mass keeps its velocity
#pragma unroll
        for (int k = 0; k < 3; ++k) s.v[m][k] = p.decay * s.v[m][k] + l.noise[k][t + m];
      }
    }
  }
#pragma unroll
  for (int m = 0; m < S; ++m)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      if (PART & kFirstHalf) l.x[k][t + m] = s.x[m][k];
      l.v[k][t + m] = s.v[m][k];
    }
}

// The units of a launch: `clusters` constraint clusters, kClusterUnits per
// block, in the first blocks (their solves take longest), then the waters
// and free atoms, `threads` / width per block: kIntThreads and width 3 with
// waters, a wave and width 1 in a system of free atoms.
struct IntUnits {
  int clusters, cluster_blocks;
  const int *cluster_first, *cluster_code;
  int units, width, per_block;   // units per block: threads / width
  const int *first, *code;
};
constexpr int kClusterSlots = 5;
constexpr int kClusterUnits = kIntThreads / kClusterSlots;

// PART kFirstHalf: half kick with the force words (cleared), drift, SETTLE,
// v += dx_c/dt, f32 positions of the pair loop, validity flag.
// kSecondHalf: half kick with the new forces (not cleared: the next step's
// first half reads them) and the velocity constraint.  kBetween: both, the
// second half of one step and the first half of the next, in one pass over
// the state with the same operations in the same order.
//
// Thread per atom outside the constraints: consecutive threads load and
// store consecutive atoms, the three atoms of a water draw their noise side
// by side and while the loads are in flight, and 64 units make three waves
// of loads.  A thread per unit for all of it took 72-byte strides through
// every array and its noise in series.  CL: with constraint clusters (their
// solves take more registers).
//
// A launch is bound by its latencies (load, constraints, store) up to some
// 100,000 atoms and by memory beyond.  Langevin steps between two steps,
// a launch alone: 11.9 us at 14,000 atoms (a thread per unit, with a step
// counter that every block advanced behind a fence: 18.2), 90 us at
// 999,000 (520; 300 bytes an atom, 3.3 TB/s); 9.5 us without noise at
// 24,000 (11.8).  Beside waters a free atom takes the three slots of a unit:
// 16.4 us for 79,000 of them and one water, 12.6 us in a system of free
// atoms alone (a thread per unit: 64 and 57).
template <int PART, bool CL>
__global__ void __launch_bounds__(kIntThreads) integrate_units(
    IntUnits un, double *__restrict__ x, double *__restrict__ v,
    const double *__restrict__ inv_mass, long long *__restrict__ F,
    long long *__restrict__ Fr, const int *__restrict__ place_of,
    const double *__restrict__ shift, const double *__restrict__ xref,
    const double *__restrict__ q, float4 *__restrict__ xq, const float4 *__restrict__ gorig,
    double4 *__restrict__ xpq, double4 *__restrict__ xpa, IntParams p,
    int *__restrict__ flags) {
  __shared__ UnitLds l;
  const int t = threadIdx.x;
  const bool cluster = CL && (int)blockIdx.x < un.cluster_blocks;
  const int block = blockIdx.x - (CL && !cluster ? un.cluster_blocks : 0);
  const int width = cluster ? kClusterSlots : un.width;
  const int per_block = cluster ? kClusterUnits : un.per_block;
  const int count = cluster ? un.clusters : un.units;
  const int *__restrict__ ufirst = cluster ? un.cluster_first : un.first;
  const int *__restrict__ ucode = cluster ? un.cluster_code : un.code;
  if (PART == kSecondHalf && p.langevin && blockIdx.x == 0 && t == 0) *p.step += p.advance;

  // this thread's atom
  const int ul = cluster ? t / kClusterSlots : (width == 3 ? t / 3 : t), m = t - ul * width;
  const int u = block * per_block + ul;
  int at = -1;
  bool free = false;   // a free atom: its thread takes it through the step
  if (ul < per_block && u < count) {
    const int first = ufirst[u], code = ucode[u];
    free = code == 1;
    if (m < (code & 0xff)) {
      // clusters: the centre first, then the others in their order
      const int centre = (code >> kUnitCentreShift) & 15;
      at = cluster ? first + (m == 0 ? centre : (m - 1 < centre ? m - 1 : m)) : first + m;
    }
  }
  int pl = 0;
  double xa[3], va[3], sh[3], xr[3], xp[3], qa = 0.0;
  float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (at >= 0) {
    pl = place_of[at];
    const double im = inv_mass[at];
    long long w[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      w[k] = Fr ? Fr[3 * at + k] : 0;
      va[k] = v[3 * at + k];
      xa[k] = x[3 * at + k];
      if (PART & kFirstHalf) {
        sh[k] = shift[3 * at + k];
        xr[k] = xref[3 * at + k];
        xp[k] = p.x_prune ? p.x_prune[3 * at + k] : 0.0;
      }
    }
    if (PART & kFirstHalf) {
      qa = q[at];
      if (gorig) o = gorig[pl / (kCluster * kGroup)];
    }
    // Fr (or null): reciprocal force words by atom, added to the
    // place-ordered words as integers before the conversion, so the force
    // is the one a single word would hold.  The words are cleared by the
    // launch that reads them last.
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      w[k] += F[3 * pl + k];
      if (PART != kSecondHalf) {
        F[3 * pl + k] = 0;
        if (Fr) Fr[3 * at + k] = 0;
      }
    }
    double kick[3], noise[3] = {0.0, 0.0, 0.0};
    if ((PART & kFirstHalf) && p.langevin && im > 0.0) {
      langevin_normals(p.seed, *p.step + p.offset, (uint32_t)at, noise);
      const double spread = p.spread * sqrt(im);
#pragma unroll
      for (int k = 0; k < 3; ++k) noise[k] = spread * noise[k];
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) kick[k] = 0.5 * p.dt * ((double)w[k] * kForceUnscale) * im;
    if (free) {  // step_unit without constraints
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        va[k] = va[k] + kick[k];
        if (PART == kBetween) va[k] = va[k] + kick[k];
        if ((PART & kFirstHalf) && p.langevin) {
          const double h = 0.5 * p.dt;
          xa[k] = xa[k] + h * va[k];
          if (im > 0.0) va[k] = p.decay * va[k] + noise[k];
          xa[k] = xa[k] + h * va[k];
        } else if (PART & kFirstHalf) {
          xa[k] = xa[k] + p.dt * va[k];
        }
      }
    } else {
      l.im[t] = im;
      if (cluster) l.len[t] = m > 0 ? p.clen[at] : 0.0;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        l.x[k][t] = xa[k];
        l.v[k][t] = va[k];
        l.kick[k][t] = kick[k];
        l.noise[k][t] = noise[k];
      }
    }
  }
  if (width > 1) {
    __syncthreads();
    // this thread's unit
    const int mine = block * per_block + t;
    if (t < per_block && mine < count) {
      const int code = ucode[mine], t0 = t * width;
      if (cluster) {
        if constexpr (CL) {
          switch (code & 0xff) {
            case 2: step_unit<PART, 2, true>(l, t0, p); break;
            case 3: step_unit<PART, 3, true>(l, t0, p); break;
            case 4: step_unit<PART, 4, true>(l, t0, p); break;
            default: step_unit<PART, 5, true>(l, t0, p); break;
          }
        }
      } else if (code == 3) {
        step_unit<PART, 3, false>(l, t0, p);
      }
    }
    __syncthreads();
  }
  if (at < 0) return;
  if (!free) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      xa[k] = l.x[k][t];
      va[k] = l.v[k][t];
    }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) v[3 * at + k] = va[k];
  if (PART & kFirstHalf) {
    double d2 = 0.0, d2p = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      x[3 * at + k] = xa[k];
      const double d = xa[k] - xr[k];
      d2 += d * d;
      if (p.x_prune) {
        const double dp = xa[k] - xp[k];
        d2p += dp * dp;
      }
    }
    // beyond half the list's buffer since the build, beyond half the pruned
    // list's since the last prune
    if (d2 > p.skin_half2) atomicOr(&flags[kFlagRebuild], 1);
    if (d2p > p.prune_half2) atomicOr(&flags[kFlagPrune], 1);
    xq[pl] = make_float4((float)(xa[0] - sh[0] - p.half_box[0] - (double)o.x),
                         (float)(xa[1] - sh[1] - p.half_box[1] - (double)o.y),
                         (float)(xa[2] - sh[2] - p.half_box[2] - (double)o.z), (float)qa);
    if (xpq) xpq[pl] = make_double4(xa[0], xa[1], xa[2], qa);
    if (xpa) xpa[at] = make_double4(xa[0], xa[1], xa[2], qa);
  }
}

// The isotropic or axis-wise scaling of a Monte Carlo volume move: each
// unit (a rigid water or a free atom) moves with its centre of mass,
// X -> s X, and keeps its shape: x_i += (s - 1) X (per axis).  Masses come
// from the inverse masses (a massless atom has weight 0; a unit without
// mass moves with the mean of its positions).
__global__ void scale_units(int nunits, const int *__restrict__ unit_first,
                            const int *__restrict__ unit_size, const double *__restrict__ inv_mass,
                            double *__restrict__ x, double s0, double s1, double s2) {
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= nunits) return;
  const int first = unit_first[u], size = unit_size[u] & 0xff;
  double com[3] = {0.0, 0.0, 0.0}, total = 0.0;
  for (int m = 0; m < size; ++m) {
    const double im = inv_mass[first + m];
    const double w = im > 0.0 ? 1.0 / im : 0.0;
    total += w;
    for (int k = 0; k < 3; ++k) com[k] += w * x[3 * (first + m) + k];
  }
  if (total > 0.0) {
    for (int k = 0; k < 3; ++k) com[k] /= total;
  } else {
    for (int k = 0; k < 3; ++k) com[k] = 0.0;
    for (int m = 0; m < size; ++m)
      for (int k = 0; k < 3; ++k) com[k] += x[3 * (first + m) + k] / size;
  }
  const double s[3] = {s0, s1, s2};
  for (int m = 0; m < size; ++m)
    for (int k = 0; k < 3; ++k) x[3 * (first + m) + k] += (s[k] - 1.0) * com[k];
}

// Positions and charges by atom for PME in atom order (evaluations outside
// the step sequence, where no integration writes them).
__global__ void pme_pack_atoms(int n, const double *__restrict__ x, const double *__restrict__ q,
                               double4 *__restrict__ xpa) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) xpa[i] = make_double4(x[3 * i], x[3 * i + 1], x[3 * i + 2], q[i]);
}

// The pair loop's f32 positions (and the f64 ones of PME in place order) of
// every atom at its place in the current list, from x: the values a drift
// stores (integrate_units, the same expressions without contraction), for
// positions set outside the steps while the list stays.
__global__ void refresh_places(int n, const double *__restrict__ x,
                               const double *__restrict__ shift, const double *__restrict__ q,
                               const int *__restrict__ place_of,
                               const float4 *__restrict__ gorig, double hx, double hy,
                               double hz, float4 *__restrict__ xq,
                               double4 *__restrict__ xpq) {
  const int at = blockIdx.x * blockDim.x + threadIdx.x;
  if (at >= n) return;
  const int pl = place_of[at];
  const float4 o = gorig ? gorig[pl / (kCluster * kGroup)] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const double x0 = x[3 * at], x1 = x[3 * at + 1], x2 = x[3 * at + 2];
  xq[pl] = make_float4((float)(x0 - shift[3 * at + 0] - hx - (double)o.x),
                       (float)(x1 - shift[3 * at + 1] - hy - (double)o.y),
                       (float)(x2 - shift[3 * at + 2] - hz - (double)o.z), (float)q[at]);
  if (xpq) xpq[pl] = make_double4(x0, x1, x2, q[at]);
}

// Reciprocal force words by atom added into the place-ordered words (and
// cleared): integer sums, so the result is the word a single buffer holds.
__global__ void pme_fold_atoms(int n, const int *__restrict__ place_of,
                               long long *__restrict__ Fr, long long *__restrict__ F) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int pl = place_of[i];
  for (int k = 0; k < 3; ++k) {
    F[3 * pl + k] += Fr[3 * i + k];
    Fr[3 * i + k] = 0;
  }
}

// Force words (place order) -> f64 forces (atom order).
__global__ void forces_to_atoms(int n, const int *__restrict__ place_of,
                                const long long *__restrict__ F, double *__restrict__ out,
                                size_t fs) {
  place_of = frame_at(place_of, fs);
  F = frame_at(F, fs);
  out = frame_at(out, fs);
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int pl = place_of[i];
  for (int k = 0; k < 3; ++k) out[3 * i + k] = (double)F[3 * pl + k] * kForceUnscale;
}

__global__ void clear_words(long long *__restrict__ w, size_t count, size_t fs) {
  w = frame_at(w, fs);
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < count; i += stride) w[i] = 0;
}

// Steepest descent of rigid waters (setup only): x_new = x + h F / |F|max,
// constrained from the old positions; the step is kept by the host when the
// energy falls.
// A descent step of a constraint cluster: each atom along its force, then
// M-SHAKE against the cluster's positions before the step.
template <int S>
__device__ void descend_cluster(int first, int code, const double *__restrict__ x0,
                                double *__restrict__ x, const long long *__restrict__ F,
                                const int *__restrict__ place_of, double step,
                                const IntParams &p) {
  const int centre = (code >> kUnitCentreShift) & 15;
  double xo[S][3], xn[S][3], im[S], len[S];
  int at[S];
#pragma unroll
  for (int m = 0; m < S; ++m) {
    at[m] = first + (m == 0 ? centre : (m - 1 < centre ? m - 1 : m));
    im[m] = p.inv_mass[at[m]];
    len[m] = m > 0 ? p.clen[at[m]] : 0.0;
    const int pl = place_of[at[m]];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      xo[m][k] = x0[3 * at[m] + k];
      xn[m][k] = xo[m][k] + step * (double)F[3 * pl + k] * kForceUnscale;
    }
  }
  mshake_positions<S>(xo, xn, im, len);
#pragma unroll
  for (int m = 0; m < S; ++m)
#pragma unroll
    for (int k = 0; k < 3; ++k) x[3 * at[m] + k] = xn[m][k];
}

__global__ void descend(int nunits, const int *__restrict__ unit_first,
                        const int *__restrict__ unit_size, const double *__restrict__ x0,
                        double *__restrict__ x, const long long *__restrict__ F,
                        const int *__restrict__ place_of, double step, IntParams p) {
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= nunits) return;
  const int first = unit_first[u], code = unit_size[u];
  if (code & kUnitCluster) {
    switch (code & 0xff) {
      case 2: descend_cluster<2>(first, code, x0, x, F, place_of, step, p); break;
      case 3: descend_cluster<3>(first, code, x0, x, F, place_of, step, p); break;
      case 4: descend_cluster<4>(first, code, x0, x, F, place_of, step, p); break;
      default: descend_cluster<5>(first, code, x0, x, F, place_of, step, p); break;
    }
    return;
  }
  const int size = code & 0xff;
  double xo[3][3], xn[3][3];
  for (int m = 0; m < size; ++m) {
    const int at = first + m;
    const int pl = place_of[at];
    for (int k = 0; k < 3; ++k) {
      xo[m][k] = x0[3 * at + k];
      xn[m][k] = xo[m][k] + step * (double)F[3 * pl + k] * kForceUnscale;
    }
  }
  if (size == 3) settle_positions(xo[0], xo[1], xo[2], xn[0], xn[1], xn[2], p);
  for (int m = 0; m < size; ++m)
    for (int k = 0; k < 3; ++k) x[3 * (first + m) + k] = xn[m][k];
}

// Back to the default contraction for the kernels that follow.
#pragma clang fp contract(fast)

}  // namespace mdhip
