// pme.hip — the smooth PME reciprocal chain for gfx950.
//
// Reference semantics (docs/paper/05-electrostatics.md:95-279):
//   places    u = K frac(x/L) in f64, first point (floor(u) - n + 1) mod K
//             (PMEWeights.cpp:8)
//   spread    Q(l) = sum_j q_j prod_a M_n(u_aj - l_a)  (PMESpread.cpp; the
//             deterministic mode adds q prod M scaled by 2^40 with 64-bit
//             integer atomics, docs/pme.md:310-331) — done that way here,
//             in LDS, by bricks of grid rows fused with the z transform
//   R2C FFT   unnormalised, half spectrum along z
//   product   Q^ <- BC Q^, BC = t1 t2 t3 / m^2, C(0) = 0; energy
//             sum h BC |Q^|^2 with h = 1/2 on the k3 = 0 and Nyquist planes
//             (PMETables/PMEConvolve.cpp; the influence fused into the
//             transform as pme_callback.cu:5-21 fuses it into cuFFT's load)
//   C2R FFT   unnormalised: phi
//   gather    F_ja = -q_j (K_a/L_a) sum_l phi(l) M'(u_a - l_a) prod M
//             (PMEGather.cpp)
// The FFT is the LDS Stockham of fft.h; the forward z pass runs in the
// spread kernel on the brick it has just accumulated, and the x pass does
// forward transform, influence product and backward transform of each x
// line in one LDS residency.
#include "fft.h"
#include "md_common.h"

namespace mdhip {

struct PmeParams {
  int K[3];
  int order;
  double box[3];
  double inv_box[3];
};

// The arithmetic of an atom's stencil (weights, spread, gather, and their
// adjoints in adjoint.hip) fuses products into sums where an expression says
// so, not where the code around an instance happens to allow it: instances
// with one and with two threads to an atom then give the same bits, which a
// frame in batches of different sizes needs.
#pragma clang fp contract(on)

// B-spline weights M[t] of the points first + t, t = 0..n-1, and their
// derivatives in u, for fraction w (recursion of PMECode.h:147-186; closed
// forms of 05-electrostatics.md:290 at order 4).
template <typename T>
__device__ __forceinline__ void bspline(T w, int order, T *M, T *dM) {
  if (order == 4) {
    const T w2 = w * w, w3 = w2 * w, om = (T)1 - w;
    const T s6 = (T)1 / (T)6;
    M[0] = om * om * om * s6;
    M[1] = ((T)3 * w3 - (T)6 * w2 + (T)4) * s6;
    M[2] = ((T)-3 * w3 + (T)3 * w2 + (T)3 * w + (T)1) * s6;
    M[3] = w3 * s6;
    if (dM) {
      dM[0] = -(T)0.5 * om * om;
      dM[1] = (T)1.5 * w2 - (T)2 * w;
      dM[2] = (T)-1.5 * w2 + w + (T)0.5;
      dM[3] = (T)0.5 * w2;
    }
    return;
  }
  T A[9] = {0}, B[9] = {0};
  A[0] = w;
  A[1] = (T)1 - w;
  for (int nn = 3; nn <= order; ++nn) {
    for (int k = 0; k <= nn; ++k) B[k] = A[k];
    for (int k = 0; k < nn; ++k) {
      const T prev = k > 0 ? B[k - 1] : (T)0;
      A[k] = ((w + (T)k) * B[k] + ((T)nn - w - (T)k) * prev) / (T)(nn - 1);
    }
  }
  for (int k = 0; k < order; ++k) {
    M[order - 1 - k] = A[k];
    if (dM) dM[order - 1 - k] = B[k] - (k > 0 ? B[k - 1] : (T)0);
  }
}

__device__ __forceinline__ void pme_place(double x, double L, double invL, int K,
                                          int order, int &first, float &w) {
  const double s = x * invL;
  const double frac = s - floor(s);
  const double u = (double)K * frac;
  const double fl = floor(u);
  w = (float)(u - fl);
  // fl is in [0, K] (K only when frac rounds up to 1), so f is in
  // [1 - order, K - order + 1] and one wrap suffices
  int f = (int)fl - order + 1;
  if (f < 0) f += K;
  first = f;
}

#pragma clang fp contract(fast)

// ---- spread fused with the forward z transform ---------------------------
//
// A block owns a brick of BX x BY grid rows (all of z) and produces their
// half spectra along z.  pme_bin first lists, for every brick, the atoms
// whose B-spline stencil touches it (thread per atom, from the atom's own
// stencil, so no atom can be missed); each listed atom then adds the part
// of its stencil that lies in the brick as 64-bit fixed point (2^40 per e)
// by LDS integer atomics, so the sums do not depend on the order of the
// adds or of the list; the brick's rows are converted to f32 and
// transformed in place in LDS.  Every grid point belongs to one brick: no
// global atomics on the grid, no grid to clear, no real-space grid in HBM.

struct BrickParams {
  int nbx, nby;             // bricks along x and y
  int cap;                  // list capacity per brick
  int *count;               // atoms listed per brick; the gather clears it
  int *list;                // places of each brick's atoms, cap per brick
  int plane_major;          // half spectrum as [kz][x][y] instead of [x][y][kz]
};

template <int TL> struct BrickShape {
  static constexpr int R = 2 * TL;                  // real rows of a brick
  static constexpr int BY = R >= 8 ? 4 : 2;
  static constexpr int BX = R / BY;
};

// The bricks along one axis, nb of B points each (the last one may hold
// fewer of the K), that the stencil f .. f+N-1 (mod K) touches: `count`
// bricks from `first` on, mod nb.  A stencil of at most K/2 points never
// comes back to its first brick.
template <int N, int B>
__device__ __forceinline__ void stencil_bricks(int f, int K, int nb, int &first, int &count) {
  const int l = f + N - 1;
  first = f / B;
  count = l < K ? l / B - first + 1 : nb - first + (l - K) / B + 1;
}

// Thread per place: list the place with every brick its stencil touches.
// Places run in column order, so a block touches few bricks: it counts its
// entries per brick in LDS, takes one range of each brick's list with one
// global atomic, then writes (the order within a list may vary from run to
// run; nothing downstream depends on it).
constexpr int kBinLdsBricks = 8192;
template <int N, int TL>
__device__ __forceinline__ void bin_block(int block, const int *__restrict__ counts,
                                          const double4 *__restrict__ xpq, const PmeParams &pp,
                                          BrickParams bp, int *__restrict__ flags, size_t fs) {
  constexpr int BX = BrickShape<TL>::BX, BY = BrickShape<TL>::BY;
  __shared__ int s_count[kBinLdsBricks];
  counts = frame_at(counts, fs);
  xpq = frame_at(xpq, fs);
  bp.count = frame_at(bp.count, fs);
  bp.list = frame_at(bp.list, fs);
  flags = frame_at(flags, fs);
  const int nbricks = bp.nbx * bp.nby;
  const bool lds = nbricks <= kBinLdsBricks;
  if (lds)
    for (int k = threadIdx.x; k < nbricks; k += blockDim.x) s_count[k] = 0;
  const int place = block * blockDim.x + threadIdx.x;
  // at most this many bricks per axis: whole ones, one more at each end, a
  // partial one at the wrap
  constexpr int MX = (N - 2) / BX + 3 < N ? (N - 2) / BX + 3 : N;
  constexpr int MY = (N - 2) / BY + 3 < N ? (N - 2) / BY + 3 : N;
  int bx = 0, by = 0, nx = 0, ny = 0;
  if (place < counts[0]) {
    const double4 pq = xpq[place];
    if (pq.w != 0.0) {  // not padding, not an uncharged atom
      int f0, f1;
      float w;
      pme_place(pq.x, pp.box[0], pp.inv_box[0], pp.K[0], N, f0, w);
      pme_place(pq.y, pp.box[1], pp.inv_box[1], pp.K[1], N, f1, w);
      stencil_bricks<N, BX>(f0, pp.K[0], bp.nbx, bx, nx);
      stencil_bricks<N, BY>(f1, pp.K[1], bp.nby, by, ny);
    }
  }
  auto brick_at = [&](int i, int j) {
    const int x = bx + i, y = by + j;
    return (y < bp.nby ? y : y - bp.nby) * bp.nbx + (x < bp.nbx ? x : x - bp.nbx);
  };
  // unrolled to the most bricks, so that `local` stays in registers
  int local[MX * MY];
  if (lds) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < MY; ++j)
#pragma unroll
      for (int i = 0; i < MX; ++i)
        if (i < nx && j < ny) local[j * MX + i] = atomicAdd(&s_count[brick_at(i, j)], 1);
    __syncthreads();
    for (int k = threadIdx.x; k < nbricks; k += blockDim.x) {
      const int c = s_count[k];
      if (c) s_count[k] = atomicAdd(&bp.count[k], c);
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < MY; ++j)
#pragma unroll
    for (int i = 0; i < MX; ++i) {
      if (i >= nx || j >= ny) continue;
      const int brick = brick_at(i, j);
      const int slot = lds ? s_count[brick] + local[j * MX + i] : atomicAdd(&bp.count[brick], 1);
      if (slot < bp.cap)
        bp.list[(size_t)brick * bp.cap + slot] = place;
      else
        atomicOr(&flags[kFlagBrickOverflow], 1);
    }
}

template <int N, int TL>
__global__ void __launch_bounds__(256) pme_bin(const int *__restrict__ counts,
                                               const double4 *__restrict__ xpq,
                                               PmeParams pp, BrickParams bp,
                                               int *__restrict__ flags, size_t fs) {
  bin_block<N, TL>(blockIdx.x, counts, xpq, pp, bp, flags, fs);
}

// The bonded tuples as the launch's first `tuples` blocks, then the bins:
// both read only what the integration wrote by atom (x and xpa), so the
// tuples' forces go to the reciprocal part's words by atom (Fr) and neither
// waits for a list build.  A launch of their own before the pair loop (one
// wave of f64 work per SIMD, 8.6 us at 25,000 atoms) lengthened the list
// branch by that.  The bins' blocks then hold the tuples' registers too (150
// instead of 31 to 64, three waves per SIMD instead of five), which a large
// box with few tuples shows in this launch alone: 1,017,000 atoms with one
// flexible water 38.8 instead of 34.0 us, 20 steps 36.5 ms with and without.
template <int N, int TL>
__global__ void __launch_bounds__(256) pme_bin_tuples(
    const int *__restrict__ counts, const double4 *__restrict__ xpq, PmeParams pp,
    BrickParams bp, int *__restrict__ flags, TupleArgs ta, int tuples,
    const double *__restrict__ x, long long *__restrict__ Fr) {
  if ((int)blockIdx.x < tuples)
    tuple_block(blockIdx.x, tuples, ta, x, nullptr, pp.box, Fr);
  else
    bin_block<N, TL>(blockIdx.x - tuples, counts, xpq, pp, bp, flags, 0);
}

// The spread, the gather and their adjoints come with SP = 1 and SP = 2
// threads to a listed atom, each taking every SP-th x plane of its stencil,
// in blocks of SP kBrickThreads.  A brick lists a few hundred atoms: while
// the GPU holds all blocks at once, what a block waits for is the serial
// chain of one atom's stencil and of its own rows' transform, and two
// threads halve both; beyond that the second thread's own weights, and
// blocks twice as large to find room for beside the pair loop, cost more.
constexpr int kBrickThreads = 256;

// The word nearest p 2^40, ties to even, as __double2ll_rn(p 2^40) gives
// it, for |p| < 2^11: the sum with 1.5 2^52 is rounded at its last bit, a
// unit, and holds the integer in its mantissa: two f64 operations instead
// of eight.
__device__ __forceinline__ unsigned long long grid_word_small(float p) {
  const double d = fma((double)p, kGridScale, 0x1.8p52);
  return (unsigned long long)(__double_as_longlong(d) - 0x4338000000000000ll);
}
template <bool SMALL>
__device__ __forceinline__ unsigned long long grid_word(float p) {
  if (SMALL) return grid_word_small(p);
  return (unsigned long long)__double2ll_rn((double)p * kGridScale);
}

#pragma clang fp contract(on)

// The x planes `half`, half + SP, .. of one atom's stencil (first
// points f, weights M, charge q), the part that lies in the brick at (bx0,
// by0), added to the brick's accumulators.  SMALL: every product is below
// 2^11.
template <int N, int BX, int BY, int SP, bool SMALL>
__device__ __forceinline__ void spread_part(const int (&f)[3], const float (&M)[3][N], float qf,
                                            int half, const PmeParams &pp, int bx0, int by0,
                                            unsigned long long *acc) {
  const int K0 = pp.K[0], K1 = pp.K[1], K2 = pp.K[2];
  int z[N];
#pragma unroll
  for (int k = 0; k < N; ++k) z[k] = f[2] + k < K2 ? f[2] + k : f[2] + k - K2;
#pragma unroll
  for (int ii = 0; ii < N / SP; ++ii) {
    int gx = f[0] + ii * SP + half;
    if (gx >= K0) gx -= K0;
    const int tx = gx - bx0;
    if (tx < 0 || tx >= BX) continue;
    float mx = M[0][ii * SP];
#pragma unroll
    for (int h = 1; h < SP; ++h)
      if (h == half) mx = M[0][ii * SP + h];
    const float wx = mx * qf;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      int gy = f[1] + j;
      if (gy >= K1) gy -= K1;
      const int ty = gy - by0;
      if (ty < 0 || ty >= BY) continue;
      const float wxy = M[1][j] * wx;
      unsigned long long *row = acc + (tx * BY + ty) * K2;
#pragma unroll
      for (int k = 0; k < N; ++k) atomicAdd(row + z[k], grid_word<SMALL>(wxy * M[2][k]));
    }
  }
}

template <int N, int BX, int BY, int SP>
__device__ __forceinline__ void spread_atom(double4 pq, int half, const PmeParams &pp, int bx0,
                                            int by0, unsigned long long *acc) {
  int f[3];
  float w[3];
  pme_place(pq.x, pp.box[0], pp.inv_box[0], pp.K[0], N, f[0], w[0]);
  pme_place(pq.y, pp.box[1], pp.inv_box[1], pp.K[1], N, f[1], w[1]);
  pme_place(pq.z, pp.box[2], pp.inv_box[2], pp.K[2], N, f[2], w[2]);
  float M[3][N];
#pragma unroll
  for (int d = 0; d < 3; ++d) bspline<float>(w[d], N, M[d], nullptr);
  const float qf = (float)pq.w;
  // the weights are at most 1; the second test is false for a position
  // that is not finite
  if (fabsf(qf) < 1024.0f && w[0] + w[1] + w[2] <= 3.0f)
    spread_part<N, BX, BY, SP, true>(f, M, qf, half, pp, bx0, by0, acc);
  else
    spread_part<N, BX, BY, SP, false>(f, M, qf, half, pp, bx0, by0, acc);
}

#pragma clang fp contract(fast)

// The brick's R accumulated real rows (64-bit words in acc) to their half
// spectra along z in `out`: rows 2t and 2t+1 as the real and imaginary
// parts of one complex line t, one LDS transform, then the two spectra
// split apart.  a, b hold TL K2 complex values each, tw the K2 twiddles.
template <int TL>
__device__ __forceinline__ void brick_forward_z(const unsigned long long *acc,
                                                cpx<float> *a, cpx<float> *b,
                                                const cpx<float> *tw, const FftAxis &az,
                                                const PmeParams &pp, const BrickParams &bp,
                                                int bx0, int by0, cpx<float> *__restrict__ out) {
  constexpr int R = BrickShape<TL>::R, BY = BrickShape<TL>::BY;
  const int K0 = pp.K[0], K1 = pp.K[1], K2 = pp.K[2], H = K2 / 2 + 1;
  for (int w = threadIdx.x; w < R * K2; w += blockDim.x) {
    const int rr = div_by(w, az.mk), z = w - rr * K2;
    const float v = (float)((double)(long long)acc[w] * kGridUnscale);
    if (rr & 1)
      a[z * TL + (rr >> 1)].y = v;
    else
      a[z * TL + (rr >> 1)].x = v;
  }
  __syncthreads();
  cpx<float> *res = lds_fft<float, TL, -1>(a, b, az, tw);
  const uint32_t mh = div_magic((uint32_t)H);
  for (int w = threadIdx.x; w < TL * H; w += blockDim.x) {
    const int t = div_by(w, mh), k = w - t * H;
    const cpx<float> zk = res[k * TL + t];
    const cpx<float> zm = res[(k ? K2 - k : 0) * TL + t];
    const int r1 = 2 * t, r2 = r1 + 1;
    const int ix1 = bx0 + r1 / BY, iy1 = by0 + r1 % BY;
    const int ix2 = bx0 + r2 / BY, iy2 = by0 + r2 % BY;
    const size_t rows = (size_t)K0 * K1;
    if (ix1 < K0 && iy1 < K1) {
      const size_t row = (size_t)ix1 * K1 + iy1;
      out[bp.plane_major ? k * rows + row : row * H + k] = {(zk.x + zm.x) * 0.5f,
                                                            (zk.y - zm.y) * 0.5f};
    }
    if (ix2 < K0 && iy2 < K1) {
      const size_t row = (size_t)ix2 * K1 + iy2;
      out[bp.plane_major ? k * rows + row : row * H + k] = {(zk.y + zm.y) * 0.5f,
                                                            (zm.x - zk.x) * 0.5f};
    }
  }
}

template <int N, int TL, int SP>
__global__ void __launch_bounds__(SP * kBrickThreads) pme_spread_rows(
    const double4 *__restrict__ xpq, PmeParams pp, BrickParams bp,
    cpx<float> *__restrict__ out, FftAxis az, size_t fs) {
  constexpr int R = BrickShape<TL>::R, BX = BrickShape<TL>::BX, BY = BrickShape<TL>::BY;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  xpq = frame_at(xpq, fs);
  bp.count = frame_at(bp.count, fs);
  bp.list = frame_at(bp.list, fs);
  out = frame_at(out, fs);
  const int K2 = pp.K[2];
  unsigned long long *acc = reinterpret_cast<unsigned long long *>(smem);
  cpx<float> *a = reinterpret_cast<cpx<float> *>(acc + (size_t)R * K2);
  cpx<float> *b = a + TL * K2;
  cpx<float> *tw = b + TL * K2;  // the z twiddles, read by every pass
  const int brick = blockIdx.x;
  const int bx0 = (brick % bp.nbx) * BX, by0 = (brick / bp.nbx) * BY;
  for (int w = threadIdx.x; w < R * K2; w += blockDim.x) acc[w] = 0ull;
  for (int w = threadIdx.x; w < K2; w += blockDim.x)
    tw[w] = static_cast<const cpx<float> *>(az.tw)[w];
  int nat = bp.count[brick];
  nat = nat < bp.cap ? nat : bp.cap;
  const int *lst = bp.list + (size_t)brick * bp.cap;
  __syncthreads();
  // the next atom's load is in flight while this one is spread
  const int half = threadIdx.x % SP, step = blockDim.x / SP;
  int i = threadIdx.x / SP;
  double4 pq = i < nat ? xpq[lst[i]] : make_double4(0, 0, 0, 0);
  while (i < nat) {
    i += step;
    const double4 next = i < nat ? xpq[lst[i]] : make_double4(0, 0, 0, 0);
    spread_atom<N, BX, BY, SP>(pq, half, pp, bx0, by0, acc);
    pq = next;
  }
  __syncthreads();
  brick_forward_z<TL>(acc, a, b, tw, az, pp, bp, bx0, by0, out);
}

// ---- backward z transform fused with the gather ---------------------------
//
// A block owns the same brick of grid rows as the spread: it transforms the
// brick's half-spectrum rows back to real potential rows in LDS, and every
// listed atom adds the part of its force that comes from the brick's points,
// as 64-bit fixed point (each part is a fixed f32 sum, so the total does not
// depend on the order of the adds).  The real potential grid never goes to
// HBM.  The block clears its brick's list count for the next step.

#pragma clang fp contract(on)

// One atom's force from the potential rows of the brick at (bx0, by0):
// -q (K/L) sum phi M' M M over the stencil points in the brick, summed over
// the SP neighbouring threads that share the atom and added as
// 64-bit fixed point.  phi of brick row r at z is phi[z TL + r/2], .x for
// even r and .y for odd r.
template <int N, int TL, int BX, int BY, int SP>
__device__ __forceinline__ void gather_atom(double4 pq, int half, int place, const PmeParams &pp,
                                            int bx0, int by0, const cpx<float> *phi,
                                            long long *__restrict__ F) {
  const int K0 = pp.K[0], K1 = pp.K[1], K2 = pp.K[2];
  int f[3];
  float w[3];
  pme_place(pq.x, pp.box[0], pp.inv_box[0], K0, N, f[0], w[0]);
  pme_place(pq.y, pp.box[1], pp.inv_box[1], K1, N, f[1], w[1]);
  pme_place(pq.z, pp.box[2], pp.inv_box[2], K2, N, f[2], w[2]);
  float M[3][N], dM[3][N];
#pragma unroll
  for (int d = 0; d < 3; ++d) bspline<float>(w[d], N, M[d], dM[d]);
  const float *flat = reinterpret_cast<const float *>(phi);
  int z[N];
#pragma unroll
  for (int k = 0; k < N; ++k) z[k] = 2 * TL * (f[2] + k < K2 ? f[2] + k : f[2] + k - K2);
  const float qf = (float)pq.w;
  const float s0 = -qf * (float)(K0 * pp.inv_box[0]), s1 = -qf * (float)(K1 * pp.inv_box[1]),
              s2 = -qf * (float)(K2 * pp.inv_box[2]);
  // the even and the odd x planes are summed apart and added as words, so
  // that one thread and two give the same bits
  long long w0 = 0, w1 = 0, w2 = 0;
#pragma unroll
  for (int h = 0; h < 2 / SP; ++h) {
    const int par = SP == 2 ? half : h;
    float g0 = 0.0f, g1 = 0.0f, g2 = 0.0f;
#pragma unroll
    for (int ii = 0; ii < N / 2; ++ii) {
      int gx = f[0] + 2 * ii + par;
      if (gx >= K0) gx -= K0;
      const int tx = gx - bx0;
      if (tx < 0 || tx >= BX) continue;
      const float mx = par ? M[0][2 * ii + 1] : M[0][2 * ii];
      const float dmx = par ? dM[0][2 * ii + 1] : dM[0][2 * ii];
#pragma unroll
      for (int j = 0; j < N; ++j) {
        int gy = f[1] + j;
        if (gy >= K1) gy -= K1;
        const int ty = gy - by0;
        if (ty < 0 || ty >= BY) continue;
        const float my = M[1][j], dmy = dM[1][j];
        const float *row = flat + tx * BY + ty;
        float sz = 0.0f, dsz = 0.0f;
#pragma unroll
        for (int k = 0; k < N; ++k) {
          const float pv = row[z[k]];
          sz += pv * M[2][k];
          dsz += pv * dM[2][k];
        }
        g0 += dmx * my * sz;
        g1 += mx * dmy * sz;
        g2 += mx * my * dsz;
      }
    }
    w0 += to_fixed(s0 * g0);
    w1 += to_fixed(s1 * g1);
    w2 += to_fixed(s2 * g2);
  }
  if (SP == 2) {
    w0 += __shfl_xor(w0, 1);
    w1 += __shfl_xor(w1, 1);
    w2 += __shfl_xor(w2, 1);
    if (half) return;
  }
  unsigned long long *u = reinterpret_cast<unsigned long long *>(F + 3 * (size_t)place);
  atomicAdd(u + 0, (unsigned long long)w0);
  atomicAdd(u + 1, (unsigned long long)w1);
  atomicAdd(u + 2, (unsigned long long)w2);
}

#pragma clang fp contract(fast)

// The brick's half-spectrum rows of `in` back to real rows in LDS (one
// complex line t per pair of rows 2t, 2t+1): returns the buffer (a or b)
// holding the rows, phi of brick row r at z being phi[z TL + r/2], .x for
// even r and .y for odd r.
template <int TL>
__device__ __forceinline__ const cpx<float> *brick_backward_z(
    const cpx<float> *__restrict__ in, cpx<float> *a, cpx<float> *b, const cpx<float> *tw,
    const FftAxis &az, const PmeParams &pp, const BrickParams &bp, int bx0, int by0) {
  constexpr int BY = BrickShape<TL>::BY;
  const int K0 = pp.K[0], K1 = pp.K[1], K2 = pp.K[2], H = K2 / 2 + 1;
  const size_t rows = (size_t)K0 * K1;
  for (int w = threadIdx.x; w < TL * K2; w += blockDim.x) {
    const int t = div_by(w, az.mk), k = w - t * K2;
    const int r1 = 2 * t, r2 = r1 + 1;
    const int ix1 = bx0 + r1 / BY, iy1 = by0 + r1 % BY;
    const int ix2 = bx0 + r2 / BY, iy2 = by0 + r2 % BY;
    const int m = k < H ? k : K2 - k;
    cpx<float> x1 = {0.0f, 0.0f}, x2 = {0.0f, 0.0f};
    if (ix1 < K0 && iy1 < K1) {
      const size_t row = (size_t)ix1 * K1 + iy1;
      x1 = in[bp.plane_major ? m * rows + row : row * H + m];
    }
    if (ix2 < K0 && iy2 < K1) {
      const size_t row = (size_t)ix2 * K1 + iy2;
      x2 = in[bp.plane_major ? m * rows + row : row * H + m];
    }
    if (m == 0 || (K2 % 2 == 0 && m == K2 / 2)) {
      x1.y = 0.0f;
      x2.y = 0.0f;
    }
    a[k * TL + t] = k < H ? cpx<float>{x1.x - x2.y, x1.y + x2.x}
                          : cpx<float>{x1.x + x2.y, -x1.y + x2.x};
  }
  __syncthreads();
  return lds_fft<float, TL, 1>(a, b, az, tw);
}

template <int N, int TL, int SP>
__global__ void __launch_bounds__(SP * kBrickThreads) pme_gather_rows(
    const double4 *__restrict__ xpq, PmeParams pp, BrickParams bp,
    const cpx<float> *__restrict__ in, FftAxis az, long long *__restrict__ F, size_t fs) {
  constexpr int BX = BrickShape<TL>::BX, BY = BrickShape<TL>::BY;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  xpq = frame_at(xpq, fs);
  bp.count = frame_at(bp.count, fs);
  bp.list = frame_at(bp.list, fs);
  in = frame_at(in, fs);
  F = frame_at(F, fs);
  const int K2 = pp.K[2];
  cpx<float> *a = reinterpret_cast<cpx<float> *>(smem);
  cpx<float> *b = a + TL * K2;
  cpx<float> *tw = b + TL * K2;  // the z twiddles, read by every pass
  const int brick = blockIdx.x;
  const int bx0 = (brick % bp.nbx) * BX, by0 = (brick / bp.nbx) * BY;
  for (int w = threadIdx.x; w < K2; w += blockDim.x)
    tw[w] = static_cast<const cpx<float> *>(az.tw)[w];
  int nat = bp.count[brick];
  nat = nat < bp.cap ? nat : bp.cap;
  const int *lst = bp.list + (size_t)brick * bp.cap;
  // the first atoms load while the rows are transformed
  const int half = threadIdx.x % SP, step = blockDim.x / SP;
  int i = threadIdx.x / SP;
  int place = i < nat ? lst[i] : 0;
  double4 pq = xpq[place];
  const cpx<float> *phi = brick_backward_z<TL>(in, a, b, tw, az, pp, bp, bx0, by0);
  while (i < nat) {
    i += step;
    const int next_place = i < nat ? lst[i] : 0;
    const double4 next = xpq[next_place];
    gather_atom<N, TL, BX, BY, SP>(pq, half, place, pp, bx0, by0, phi, F);
    place = next_place;
    pq = next;
  }
  __syncthreads();  // every thread has read the count
  if (threadIdx.x == 0) bp.count[brick] = 0;
}

// ---- FFT passes ---------------------------------------------------------

template <typename T>
constexpr int tile_lines() { return sizeof(T) == 4 ? 16 : 8; }

// LDS of a tile of lines of length k: two buffers, and the axis' twiddles
// where they fit in the 64 KB a launch takes without asking for more, beside
// 2 KB of its own (every pass reads them: edges up to 240 in f32, 233 in f64).
template <typename T>
__host__ __device__ __forceinline__ bool tile_twiddles_fit(int k) {
  return (size_t)(2 * tile_lines<T>() + 1) * k * sizeof(cpx<T>) <= 65536 - 2048;
}
template <typename T>
inline size_t tile_lds(int k) {
  return (size_t)(2 * tile_lines<T>() + (tile_twiddles_fit<T>(k) ? 1 : 0)) * k * sizeof(cpx<T>);
}
// The twiddles copied to `at`, or the axis' own table; the caller's next
// barrier orders the copy.
template <typename T>
__device__ __forceinline__ const cpx<T> *tile_twiddles(cpx<T> *at, const FftAxis &ax) {
  const cpx<T> *own = static_cast<const cpx<T> *>(ax.tw);
  if (!tile_twiddles_fit<T>(ax.K)) return own;
  for (int w = threadIdx.x; w < ax.K; w += blockDim.x) at[w] = own[w];
  return at;
}

// Forward along z of pairs of real rows packed as one complex line, split
// into the two half spectra.  SRC_FIXED reads (and clears) 64-bit charge
// words; otherwise a real T grid.
template <typename T, bool SRC_FIXED>
__global__ void __launch_bounds__(256) fft_rows_r2c(
    const void *__restrict__ src_v, cpx<T> *__restrict__ out, int nrows,
    FftAxis az) {
  constexpr int TL = tile_lines<T>();
  extern __shared__ unsigned char smem[];
  cpx<T> *a = reinterpret_cast<cpx<T> *>(smem);
  const int K = az.K, H = K / 2 + 1;
  cpx<T> *b = a + TL * K;
  const int row0 = blockIdx.x * 2 * TL;
  for (int w = threadIdx.x; w < 2 * TL * K; w += blockDim.x) {
    const int z = w % K, rr = w / K;  // rr: row within the tile
    const int row = row0 + rr;
    T v = (T)0;
    if (row < nrows) {
      const size_t idx = (size_t)row * K + z;
      if (SRC_FIXED) {
        unsigned long long *src = (unsigned long long *)src_v;
        v = (T)((double)(long long)src[idx] * kGridUnscale);
        src[idx] = 0ull;
      } else {
        v = ((const T *)src_v)[idx];
      }
    }
    const int t = rr >> 1;
    if (rr & 1)
      a[z * TL + t].y = v;
    else
      a[z * TL + t].x = v;
  }
  __syncthreads();
  cpx<T> *res = lds_fft<T, TL, -1>(a, b, az);
  for (int w = threadIdx.x; w < TL * H; w += blockDim.x) {
    const int k = w % H, t = w / H;
    const cpx<T> zk = res[k * TL + t];
    const cpx<T> zm = res[((K - k) % K) * TL + t];
    const int r1 = row0 + 2 * t, r2 = r1 + 1;
    if (r1 < nrows)
      out[(size_t)r1 * H + k] = {(zk.x + zm.x) * (T)0.5, (zk.y - zm.y) * (T)0.5};
    if (r2 < nrows)
      out[(size_t)r2 * H + k] = {(zk.y + zm.y) * (T)0.5, (zm.x - zk.x) * (T)0.5};
  }
}

// Backward along z: two half spectra as one complex line, real part to the
// first row and imaginary part to the second.  The imaginary parts of the
// zero and (even K) Nyquist terms are ignored (mdrt_fft.c:149-157).
template <typename T>
__global__ void __launch_bounds__(256) fft_rows_c2r(const cpx<T> *__restrict__ in,
                                                    T *__restrict__ dst, int nrows,
                                                    FftAxis az, int plane_major) {
  constexpr int TL = tile_lines<T>();
  extern __shared__ unsigned char smem[];
  cpx<T> *a = reinterpret_cast<cpx<T> *>(smem);
  const int K = az.K, H = K / 2 + 1;
  cpx<T> *b = a + TL * K;
  const int row0 = blockIdx.x * 2 * TL;
  for (int w = threadIdx.x; w < TL * K; w += blockDim.x) {
    const int k = w % K, t = w / K;
    const int r1 = row0 + 2 * t, r2 = r1 + 1;
    const int m = k < H ? k : K - k;
    cpx<T> x1 = {(T)0, (T)0}, x2 = {(T)0, (T)0};
    // half spectrum [row][k], or kz-plane major [k][row]
    if (r1 < nrows) x1 = in[plane_major ? (size_t)m * nrows + r1 : (size_t)r1 * H + m];
    if (r2 < nrows) x2 = in[plane_major ? (size_t)m * nrows + r2 : (size_t)r2 * H + m];
    if (m == 0 || (K % 2 == 0 && m == K / 2)) {
      x1.y = (T)0;
      x2.y = (T)0;
    }
    cpx<T> zv;
    if (k < H)
      zv = {x1.x - x2.y, x1.y + x2.x};
    else
      zv = {x1.x + x2.y, -x1.y + x2.x};
    a[k * TL + t] = zv;
  }
  __syncthreads();
  cpx<T> *res = lds_fft<T, TL, 1>(a, b, az);
  for (int w = threadIdx.x; w < 2 * TL * K; w += blockDim.x) {
    const int z = w % K, rr = w / K;
    const int row = row0 + rr;
    if (row >= nrows) continue;
    const cpx<T> v = res[z * TL + (rr >> 1)];
    dst[(size_t)row * K + z] = (rr & 1) ? v.y : v.x;
  }
}

// Complex lines along y (axis 1: stride H) of the half spectrum, in place.
template <typename T>
__global__ void __launch_bounds__(256) fft_cols_y(cpx<T> *__restrict__ data, int K2,
                                                  int H, FftAxis ay, int sign) {
  constexpr int TL = tile_lines<T>();
  extern __shared__ unsigned char smem[];
  cpx<T> *a = reinterpret_cast<cpx<T> *>(smem);
  cpx<T> *b = a + TL * K2;
  const cpx<T> *tw = tile_twiddles<T>(b + TL * K2, ay);
  const int tiles = (H + TL - 1) / TL;
  const int i0 = blockIdx.x / tiles, z0 = (blockIdx.x % tiles) * TL;
  cpx<T> *base = data + (size_t)i0 * K2 * H + z0;
  for (int w = threadIdx.x; w < TL * K2; w += blockDim.x) {
    const int t = w % TL, y = w / TL;
    a[y * TL + t] = (z0 + t < H) ? base[(size_t)y * H + t] : cpx<T>{(T)0, (T)0};
  }
  __syncthreads();
  cpx<T> *res = sign < 0 ? lds_fft<T, TL, -1>(a, b, ay, tw) : lds_fft<T, TL, 1>(a, b, ay, tw);
  for (int w = threadIdx.x; w < TL * K2; w += blockDim.x) {
    const int t = w % TL, y = w / TL;
    if (z0 + t < H) base[(size_t)y * H + t] = res[y * TL + t];
  }
}

// Complex lines along x (stride K2 H): forward, influence product (and its
// energy), backward (mode 0); the product and backward only (mode 2); or a
// single direction (mode -1 forward, +1 backward) for the transform entry
// points of the runtime ABI.
struct ConvTables {
  const void *t[3];   // t_a(k) = exp(-pi^2 m_a^2 / beta^2) |b_a(k)|^2, t_0 * f/(pi V)
  const void *m[3];   // m_a(k) = signed k / L_a
  int K3;
  float pb2;          // pi^2 / beta^2 (the reciprocal virial)
};

template <typename T>
__global__ void __launch_bounds__(256) fft_x_conv(cpx<T> *__restrict__ data, int K1,
                                                  int K2, int H, FftAxis ax,
                                                  ConvTables ct, int mode,
                                                  double *__restrict__ energy_partial) {
  constexpr int TL = tile_lines<T>();
  extern __shared__ unsigned char smem[];
  cpx<T> *a = reinterpret_cast<cpx<T> *>(smem);
  cpx<T> *b = a + TL * K1;
  const cpx<T> *tw = tile_twiddles<T>(b + TL * K1, ax);
  __shared__ double s_e[256];
  const int tiles = (H + TL - 1) / TL;
  const int i1 = blockIdx.x / tiles, z0 = (blockIdx.x % tiles) * TL;
  const size_t stride = (size_t)K2 * H;
  cpx<T> *base = data + (size_t)i1 * H + z0;
  for (int w = threadIdx.x; w < TL * K1; w += blockDim.x) {
    const int t = w % TL, xx = w / TL;
    a[xx * TL + t] = (z0 + t < H) ? base[xx * stride + t] : cpx<T>{(T)0, (T)0};
  }
  __syncthreads();
  if (mode == -1 || mode == 1) {  // single direction: -1 forward, +1 backward
    cpx<T> *res = mode < 0 ? lds_fft<T, TL, -1>(a, b, ax, tw) : lds_fft<T, TL, 1>(a, b, ax, tw);
    for (int w = threadIdx.x; w < TL * K1; w += blockDim.x) {
      const int t = w % TL, xx = w / TL;
      if (z0 + t < H) base[xx * stride + t] = res[xx * TL + t];
    }
    return;
  }
  // mode 0: forward, product, backward; mode 2: product, backward (the
  // spectrum is already transformed along x)
  cpx<T> *res = mode == 0 ? lds_fft<T, TL, -1>(a, b, ax, tw) : a;
  const T *t0 = (const T *)ct.t[0], *t1 = (const T *)ct.t[1], *t2 = (const T *)ct.t[2];
  const T *m0 = (const T *)ct.m[0], *m1 = (const T *)ct.m[1], *m2 = (const T *)ct.m[2];
  double e = 0.0;
  for (int w = threadIdx.x; w < TL * K1; w += blockDim.x) {
    const int t = w % TL, kx = w / TL;
    const int kz = z0 + t;
    cpx<T> v = res[kx * TL + t];
    T bc = (T)0;
    if (kz < H && (kx | i1 | kz) != 0) {
      const T msq = m0[kx] * m0[kx] + m1[i1] * m1[i1] + m2[kz] * m2[kz];
      bc = t0[kx] * t1[i1] * t2[kz] / msq;
      if (energy_partial) {
        const double h = (kz == 0 || (ct.K3 % 2 == 0 && kz == ct.K3 / 2)) ? 0.5 : 1.0;
        e += h * (double)bc * ((double)v.x * v.x + (double)v.y * v.y);
      }
    }
    res[kx * TL + t] = {v.x * bc, v.y * bc};
  }
  __syncthreads();
  cpx<T> *other = (res == a) ? b : a;
  cpx<T> *res2 = lds_fft<T, TL, 1>(res, other, ax, tw);
  for (int w = threadIdx.x; w < TL * K1; w += blockDim.x) {
    const int t = w % TL, xx = w / TL;
    if (z0 + t < H) base[xx * stride + t] = res2[xx * TL + t];
  }
  if (energy_partial) {
    s_e[threadIdx.x] = e;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
      if (threadIdx.x < s) s_e[threadIdx.x] += s_e[threadIdx.x + s];
      __syncthreads();
    }
    if (threadIdx.x == 0) energy_partial[blockIdx.x] = s_e[0];
  }
}

constexpr int kPlaneAxisMax = 256;

// The y and x passes of one kz plane, whole in LDS, for grids whose planes
// fit (K1 K2 <= 4096 points, K1, K2 <= 256): forward y, forward x,
// influence product (and its energy), backward x, backward y.  The half
// spectrum is kz-plane major ([kz][x][y]), so a plane is one contiguous read
// and write.
// CK1, CK2: the plane's edges at compile time (0: the run-time K1, K2 and
// the axes' radix lists).
template <int CK1, int CK2>
__global__ void __launch_bounds__(512) fft_plane_conv(cpx<float> *__restrict__ data, int K1,
                                                      int K2, FftAxis ax, FftAxis ay,
                                                      ConvTables ct,
                                                      double *__restrict__ energy_partial,
                                                      double *__restrict__ virial_partial,
                                                      size_t fs) {
  if (CK1 > 0) {
    K1 = CK1;
    K2 = CK2;
  }
  extern __shared__ unsigned char smem[];
  __shared__ double s_e[512];
  data = frame_at(data, fs);
  energy_partial = frame_at(energy_partial, fs);
  virial_partial = frame_at(virial_partial, fs);
  __shared__ cpx<float> s_twx[kPlaneAxisMax], s_twy[kPlaneAxisMax];
  __shared__ float s_t0[kPlaneAxisMax], s_m0[kPlaneAxisMax];
  __shared__ float s_t1[kPlaneAxisMax], s_m1[kPlaneAxisMax];
  const int np = K1 * K2;
  cpx<float> *a = reinterpret_cast<cpx<float> *>(smem);
  cpx<float> *b = a + np;
  const int kz = blockIdx.x;
  cpx<float> *plane = data + (size_t)kz * np;
  const int swz = K2 % 16 == 0 ? 15 : 0;
  // element w of the plane: its x, y and place in LDS
  auto at = [&](int w, int &x, int &y) {
    x = CK2 > 0 ? w / CK2 : div_by(w, ay.mk);
    y = w - x * K2;
    return plane_index(x, y, K2, swz);
  };
  int kx, ky;
  // the plane (unrolled, so that the loads are issued together)
#pragma unroll 8
  for (int w = threadIdx.x; w < np; w += blockDim.x) a[at(w, kx, ky)] = plane[w];
  // twiddles and influence tables in LDS: every pass reads them
  for (int w = threadIdx.x; w < K1; w += blockDim.x) {
    s_twx[w] = static_cast<const cpx<float> *>(ax.tw)[w];
    s_t0[w] = static_cast<const float *>(ct.t[0])[w];
    s_m0[w] = static_cast<const float *>(ct.m[0])[w];
  }
  for (int w = threadIdx.x; w < K2; w += blockDim.x) {
    s_twy[w] = static_cast<const cpx<float> *>(ay.tw)[w];
    s_t1[w] = static_cast<const float *>(ct.t[1])[w];
    s_m1[w] = static_cast<const float *>(ct.m[1])[w];
  }
  __syncthreads();
  cpx<float> *r;
  if constexpr (CK1 > 0) {
    r = lds_fft_plane_k<float, 1, -1, CK1, CK2>(a, b, swz, s_twy);
    r = lds_fft_plane_k<float, 0, -1, CK1, CK2>(r, r == a ? b : a, swz, s_twx);
  } else {
    r = lds_fft_plane<float, 1, -1>(a, b, ay, K1, K2, swz, ay.mk, s_twy);
    r = lds_fft_plane<float, 0, -1>(r, r == a ? b : a, ax, K1, K2, swz, ay.mk, s_twx);
  }
  const float t2 = static_cast<const float *>(ct.t[2])[kz];
  const float m2 = static_cast<const float *>(ct.m[2])[kz];
  const double h = (kz == 0 || (ct.K3 % 2 == 0 && kz == ct.K3 / 2)) ? 0.5 : 1.0;
  double e = 0.0;
  // the reciprocal virial sum_m E_m [delta_ab - 2 (1/m^2 + pi^2/beta^2) m_a m_b]
  // (05-electrostatics.md:262-279): xx yy zz xy xz yz
  double vir[6] = {0, 0, 0, 0, 0, 0};
  for (int w = threadIdx.x; w < np; w += blockDim.x) {
    const int i = at(w, kx, ky);
    const cpx<float> v = r[i];
    float bc = 0.0f;
    if ((kx | ky | kz) != 0) {
      const float msq = s_m0[kx] * s_m0[kx] + s_m1[ky] * s_m1[ky] + m2 * m2;
      bc = s_t0[kx] * s_t1[ky] * t2 / msq;
      if (energy_partial || virial_partial) {
        const double em = h * (double)bc * ((double)v.x * v.x + (double)v.y * v.y);
        e += em;
        if (virial_partial) {
          const double c = 2.0 * (1.0 / (double)msq + (double)ct.pb2);
          const double mx = s_m0[kx], my = s_m1[ky], mz = m2;
          vir[0] += em * (1.0 - c * mx * mx);
          vir[1] += em * (1.0 - c * my * my);
          vir[2] += em * (1.0 - c * mz * mz);
          vir[3] -= em * c * mx * my;
          vir[4] -= em * c * mx * mz;
          vir[5] -= em * c * my * mz;
        }
      }
    }
    r[i] = {v.x * bc, v.y * bc};
  }
  __syncthreads();
  if constexpr (CK1 > 0) {
    r = lds_fft_plane_k<float, 0, 1, CK1, CK2>(r, r == a ? b : a, swz, s_twx);
    r = lds_fft_plane_k<float, 1, 1, CK1, CK2>(r, r == a ? b : a, swz, s_twy);
  } else {
    r = lds_fft_plane<float, 0, 1>(r, r == a ? b : a, ax, K1, K2, swz, ay.mk, s_twx);
    r = lds_fft_plane<float, 1, 1>(r, r == a ? b : a, ay, K1, K2, swz, ay.mk, s_twy);
  }
  for (int w = threadIdx.x; w < np; w += blockDim.x)
    plane[w] = r[at(w, kx, ky)];
  if (energy_partial) {
    s_e[threadIdx.x] = e;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
      if (threadIdx.x < s) s_e[threadIdx.x] += s_e[threadIdx.x + s];
      __syncthreads();
    }
    if (threadIdx.x == 0) energy_partial[blockIdx.x] = s_e[0];
  }
  if (virial_partial) {
    for (int c = 0; c < 6; ++c) {
      __syncthreads();
      s_e[threadIdx.x] = vir[c];
      __syncthreads();
      for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) s_e[threadIdx.x] += s_e[threadIdx.x + s];
        __syncthreads();
      }
      if (threadIdx.x == 0) virial_partial[6 * blockIdx.x + c] = s_e[0];
    }
  }
}

template __global__ void fft_rows_r2c<float, true>(const void *, cpx<float> *, int, FftAxis);
#define MDHIP_SPREAD_SP(N, TL, SP)                                                       \
  template __global__ void pme_spread_rows<N, TL, SP>(const double4 *, PmeParams,        \
      BrickParams, cpx<float> *, FftAxis, size_t);                                       \
  template __global__ void pme_gather_rows<N, TL, SP>(const double4 *, PmeParams,        \
      BrickParams, const cpx<float> *, FftAxis, long long *, size_t);
#define MDHIP_SPREAD(N, TL)                                                              \
  template __global__ void pme_bin<N, TL>(const int *, const double4 *, PmeParams,       \
      BrickParams, int *, size_t);                                                       \
  template __global__ void pme_bin_tuples<N, TL>(const int *, const double4 *,           \
      PmeParams, BrickParams, int *, TupleArgs, int, const double *, long long *);       \
  MDHIP_SPREAD_SP(N, TL, 1) MDHIP_SPREAD_SP(N, TL, 2)
#define MDHIP_SPREAD_N(N) MDHIP_SPREAD(N, 8) MDHIP_SPREAD(N, 4) MDHIP_SPREAD(N, 2) MDHIP_SPREAD(N, 1)
MDHIP_SPREAD_N(4)
MDHIP_SPREAD_N(6)
MDHIP_SPREAD_N(8)
template __global__ void fft_rows_r2c<float, false>(const void *, cpx<float> *, int, FftAxis);
template __global__ void fft_rows_r2c<double, false>(const void *, cpx<double> *, int, FftAxis);
template __global__ void fft_rows_c2r<float>(const cpx<float> *, float *, int, FftAxis, int);
template __global__ void fft_rows_c2r<double>(const cpx<double> *, double *, int, FftAxis, int);
template __global__ void fft_cols_y<float>(cpx<float> *, int, int, FftAxis, int);
template __global__ void fft_cols_y<double>(cpx<double> *, int, int, FftAxis, int);
template __global__ void fft_x_conv<float>(cpx<float> *, int, int, int, FftAxis, ConvTables, int, double *);
template __global__ void fft_x_conv<double>(cpx<double> *, int, int, int, FftAxis, ConvTables, int, double *);

}  // namespace mdhip
