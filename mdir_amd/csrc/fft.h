// fft.h — LDS-resident mixed-radix Stockham FFT for the PME grids.
//
// Conventions of the reference's transforms (runtime/mdrt_fft.c:110-256,
// cuFFT calls of runtime/mdrt_cuda.c:2901-2991): forward exp(-2 pi i k m/K),
// backward exp(+2 pi i k m/K), unnormalised; the real grid K1 x K2 x K3 is
// row-major (z fastest) and its half spectrum K1 x K2 x (K3/2+1) complex
// numbers, interleaved.
//
// A workgroup holds a tile of TL lines of one axis in LDS (element e of line
// t at [e * TL + t], so a row of the tile is TL consecutive complex numbers
// of the grid and the global loads of a tile are coalesced) and runs every
// radix pass of the line there; only the first load and the last store touch
// HBM.  The passes are bound by their LDS round trips, so an axis takes the
// fewest passes that radices 2 to 10 allow (216 = 6 6 6, 36 = 6 6, 70 = 10 7;
// 64 = 8 8), in registers, with twiddles from a table of exp(-2 pi i m / K)
// computed in f64 on the host.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mdhip {

template <typename T>
struct cpx {
  T x, y;
};

template <typename T>
__device__ __forceinline__ cpx<T> cmul(cpx<T> a, cpx<T> b) {
  return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <typename T>
__device__ __forceinline__ cpx<T> cadd(cpx<T> a, cpx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ __forceinline__ cpx<T> csub(cpx<T> a, cpx<T> b) { return {a.x - b.x, a.y - b.y}; }
// a * (S i), S = +-1
template <int S, typename T>
__device__ __forceinline__ cpx<T> cmuli(cpx<T> a) {
  return S > 0 ? cpx<T>{-a.y, a.x} : cpx<T>{a.y, -a.x};
}

constexpr int kMaxRadices = 8;

// Quotients by run-time divisors without a division: w / d is the high word
// of w * magic, magic = floor((2^32 - 1) / d) + 1, exact while w d < 2^32 (the
// product exceeds w 2^32 / d by less than w d / (2^32 d)); a divisor of 1 has
// magic 0 (2^32 mod 2^32) and is the caller's case.  The index arithmetic
// of a pass with its true divisions cost more than its butterflies.
__host__ __device__ __forceinline__ uint32_t div_magic(uint32_t d) {
  return 0xFFFFFFFFu / d + 1u;
}
__device__ __forceinline__ int div_by(int w, uint32_t magic) {
  return magic ? (int)__umulhi((uint32_t)w, magic) : w;
}

struct FftAxis {
  int K;
  int nrad;
  int rad[kMaxRadices];
  uint32_t mk;                // div_magic(K)
  uint32_t mkr[kMaxRadices];  // of K / rad[s], the butterflies of a line
  uint32_t mns[kMaxRadices];  // of the product of the radices before s
  const void *tw;             // cpx<T>[K]: exp(-2 pi i m / K)
};

// The passes of a length: the fewest factors among 2 .. 10, of those the
// ones with the smallest sum (the most butterflies side by side), the
// largest first (the first pass has no twiddles).  False when K has a prime
// factor above 7, or more factors 8, 4, 2, 3, 5, 7 (taken in that order)
// than kMaxRadices.
inline bool factor_axis(int K, FftAxis &ax) {
  int rest = K, plain = 0;
  for (int r : {8, 4, 2, 3, 5, 7})
    while (rest % r == 0) {
      ++plain;
      rest /= r;
    }
  if (rest != 1 || plain > kMaxRadices) return false;
  struct Search {
    int best[kMaxRadices], n = kMaxRadices + 1, sum = 0, cur[kMaxRadices];
    void go(int rest, int most, int depth, int total) {
      if (rest == 1) {
        if (depth < n || (depth == n && total < sum)) {
          n = depth;
          sum = total;
          for (int i = 0; i < depth; ++i) best[i] = cur[i];
        }
        return;
      }
      if (depth == kMaxRadices || depth >= n) return;
      for (int r = most; r >= 2; --r)
        if (rest % r == 0) {
          cur[depth] = r;
          go(rest / r, r, depth + 1, total + r);
        }
    }
  } s;
  s.go(K, 10, 0, 0);
  ax.K = K;
  ax.nrad = s.n;
  ax.mk = div_magic((uint32_t)K);
  int ns = 1;
  for (int i = 0; i < s.n; ++i) {
    ax.rad[i] = s.best[i];
    ax.mkr[i] = div_magic((uint32_t)(K / s.best[i]));
    ax.mns[i] = div_magic((uint32_t)ns);
    ns *= s.best[i];
  }
  return true;
}

// v[k] <- sum_r v[r] exp(S 2 pi i r k / R), R and the sign S known at compile
// time so that v stays in registers.
template <typename T, int R, int S>
__device__ __forceinline__ void butterfly(cpx<T> *v) {
  if constexpr (R == 2) {
    cpx<T> a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  } else if constexpr (R == 4) {
    cpx<T> a0 = cadd(v[0], v[2]), a1 = csub(v[0], v[2]);
    cpx<T> b0 = cadd(v[1], v[3]), b1 = cmuli<S>(csub(v[1], v[3]));
    v[0] = cadd(a0, b0);
    v[2] = csub(a0, b0);
    v[1] = cadd(a1, b1);
    v[3] = csub(a1, b1);
  } else if constexpr (R == 8) {
    const T h = (T)0.70710678118654752440;
    cpx<T> e[4] = {v[0], v[2], v[4], v[6]};
    cpx<T> o[4] = {v[1], v[3], v[5], v[7]};
    butterfly<T, 4, S>(e);
    butterfly<T, 4, S>(o);
    constexpr T ss = (T)S;
    cpx<T> t1 = {h * (o[1].x - ss * o[1].y), h * (o[1].y + ss * o[1].x)};
    cpx<T> t2 = cmuli<S>(o[2]);
    cpx<T> t3 = {h * (-o[3].x - ss * o[3].y), h * (-o[3].y + ss * o[3].x)};
    v[0] = cadd(e[0], o[0]);
    v[4] = csub(e[0], o[0]);
    v[1] = cadd(e[1], t1);
    v[5] = csub(e[1], t1);
    v[2] = cadd(e[2], t2);
    v[6] = csub(e[2], t2);
    v[3] = cadd(e[3], t3);
    v[7] = csub(e[3], t3);
  } else if constexpr (R == 6 || R == 10) {
    // 2 x 3 and 2 x 5, coprime: in n = (P n1 + 2 n2) mod R, out the k with
    // k mod 2 = k1 and k mod P = k2 (Good's indices: no twiddles between)
    constexpr int P = R / 2;
    cpx<T> u[2][P];
#pragma unroll
    for (int n2 = 0; n2 < P; ++n2) {
      const cpx<T> a = v[(2 * n2) % R], b = v[(P + 2 * n2) % R];
      u[0][n2] = cadd(a, b);
      u[1][n2] = csub(a, b);
    }
    butterfly<T, P, S>(u[0]);
    butterfly<T, P, S>(u[1]);
#pragma unroll
    for (int k = 0; k < R; ++k) v[k] = u[k % 2][k % P];
  } else if constexpr (R == 9) {
    // 3 x 3: in n = 3 n1 + n2, out k = k1 + 3 k2, twiddles w9^(n2 k1) between
    cpx<T> u[3][3];
#pragma unroll
    for (int n2 = 0; n2 < 3; ++n2) {
      u[n2][0] = v[n2];
      u[n2][1] = v[3 + n2];
      u[n2][2] = v[6 + n2];
      butterfly<T, 3, S>(u[n2]);
    }
#pragma unroll
    for (int n2 = 1; n2 < 3; ++n2)
#pragma unroll
      for (int k1 = 1; k1 < 3; ++k1) {
        const T c = (T)__builtin_cos(6.283185307179586476925286766559 * (n2 * k1) / 9.0);
        const T s = (T)__builtin_sin(6.283185307179586476925286766559 * (n2 * k1) / 9.0);
        u[n2][k1] = cmul(u[n2][k1], cpx<T>{c, (T)S * s});
      }
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
      cpx<T> w[3] = {u[0][k1], u[1][k1], u[2][k1]};
      butterfly<T, 3, S>(w);
#pragma unroll
      for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = w[k2];
    }
  } else {
    // radices 3, 5, 7 by their conjugate pairs: with p_r = v_r + v_{R-r} and
    // m_r = v_r - v_{R-r}, out k and R - k are v_0 + sum_r cos p_r +- S i
    // sum_r sin m_r, constants folded at compile time
    constexpr int H = R / 2;
    cpx<T> p[H], m[H];
    const cpx<T> v0 = v[0];
    cpx<T> all = v0;
#pragma unroll
    for (int r = 1; r <= H; ++r) {
      p[r - 1] = cadd(v[r], v[R - r]);
      m[r - 1] = csub(v[r], v[R - r]);
      all = cadd(all, p[r - 1]);
    }
    v[0] = all;
#pragma unroll
    for (int k = 1; k <= H; ++k) {
      cpx<T> re = v0, im = {(T)0, (T)0};
#pragma unroll
      for (int r = 1; r <= H; ++r) {
        const int a = (r * k) % R;
        const T c = (T)__builtin_cos(6.283185307179586476925286766559 * a / R);
        const T s = (T)__builtin_sin(6.283185307179586476925286766559 * a / R);
        re.x += c * p[r - 1].x;
        re.y += c * p[r - 1].y;
        im.x += s * m[r - 1].x;
        im.y += s * m[r - 1].y;
      }
      const cpx<T> t = cmuli<S>(im);
      v[k] = cadd(re, t);
      v[R - k] = csub(re, t);
    }
  }
}

// v[r] *= w^{k r tstep} of the twiddle table (its conjugate backward).
template <typename T, int R, int S>
__device__ __forceinline__ void twiddle(cpx<T> *v, const cpx<T> *tw, int kt) {
#pragma unroll
  for (int r = 1; r < R; ++r) {
    cpx<T> t = tw[kt * r];
    if (S > 0) t.y = -t.y;
    v[r] = cmul(v[r], t);
  }
}

// One Stockham pass of radix R over TL lines (Govindaraju et al., SC'08):
// after sub-transforms of length Ns, v[r] = in[j + r K/R] is twiddled by
// w^{(j mod Ns) r K/(Ns R)} and written to out[(j/Ns) Ns R + j mod Ns + r Ns].
template <typename T, int TL, int R, int S>
__device__ __forceinline__ void stockham_pass(const cpx<T> *in, cpx<T> *out, int K, int Ns,
                                              uint32_t mns, const cpx<T> *tw) {
  const int Kr = K / R;
  const int tstep = Kr / Ns;
  for (int w = threadIdx.x; w < TL * Kr; w += blockDim.x) {
    const int line = w % TL, j = w / TL;
    cpx<T> v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = in[(j + r * Kr) * TL + line];
    const int k = j - div_by(j, mns) * Ns;
    if (Ns > 1) twiddle<T, R, S>(v, tw, k * tstep);
    butterfly<T, R, S>(v);
    const int base = (j - k) * R + k;
#pragma unroll
    for (int r = 0; r < R; ++r) out[(base + r * Ns) * TL + line] = v[r];
  }
}

// The pass of a run-time radix.
#define MDHIP_RADIX_SWITCH(R, PASS) \
  switch (R) {                      \
    case 2: PASS(2); break;         \
    case 3: PASS(3); break;         \
    case 4: PASS(4); break;         \
    case 5: PASS(5); break;         \
    case 6: PASS(6); break;         \
    case 7: PASS(7); break;         \
    case 8: PASS(8); break;         \
    case 9: PASS(9); break;         \
    default: PASS(10); break;       \
  }

// Runs all passes of TL lines of length ax.K held in `a` (scratch `b`),
// sign S -1 forward / +1 backward.  Returns the buffer holding the result.
// tw: the twiddles to read (a copy in LDS), or null for the axis' own.
template <typename T, int TL, int S>
__device__ cpx<T> *lds_fft(cpx<T> *a, cpx<T> *b, const FftAxis &ax,
                           const cpx<T> *tw = nullptr) {
  const int K = ax.K;
  if (!tw) tw = static_cast<const cpx<T> *>(ax.tw);
  int Ns = 1;
  cpx<T> *in = a, *out = b;
  for (int s = 0; s < ax.nrad; ++s) {
    const int R = ax.rad[s];
#define MDHIP_PASS(R_) stockham_pass<T, TL, R_, S>(in, out, K, Ns, ax.mns[s], tw)
    MDHIP_RADIX_SWITCH(R, MDHIP_PASS)
#undef MDHIP_PASS
    __syncthreads();
    cpx<T> *t = in;
    in = out;
    out = t;
    Ns *= R;
  }
  return in;
}

// A K1 x K2 plane of complex numbers held whole in LDS, element (x, y) at
// x K2 + (y ^ s(x)), s(x) = (x & 1) << 3 | (x >> 1) & 7 when 16 divides K2
// (swz != 0), else 0: the rows a y-pass wave touches land in all 16 LDS
// bank pairs instead of 8.
__device__ __forceinline__ int plane_index(int x, int y, int K2, int swz) {
  return x * K2 + (y ^ (swz & (((x & 1) << 3) | ((x >> 1) & 7))));
}

// One Stockham pass over the lines of a plane: along y (AXIS 1: K1 lines of
// K2) or along x (AXIS 0: K2 lines of K1).  Threads run along the elements
// of a line for y and along the lines for x, so a wave's accesses are
// consecutive up to the swizzle.  mdiv: of the number the thread index
// divides by (the butterflies of a line along y, the lines along x).
template <typename T, int R, int AXIS, int S>
__device__ __forceinline__ void stockham_pass_plane(const cpx<T> *in, cpx<T> *out, int K1,
                                                    int K2, int swz, int Ns, uint32_t mdiv,
                                                    uint32_t mns, const cpx<T> *tw) {
  const int K = AXIS == 1 ? K2 : K1, nlines = AXIS == 1 ? K1 : K2;
  const int Kr = K / R;
  const int tstep = Kr / Ns;
  for (int w = threadIdx.x; w < nlines * Kr; w += blockDim.x) {
    const int q = div_by(w, mdiv);
    const int line = AXIS == 1 ? q : w - q * nlines;
    const int j = AXIS == 1 ? w - q * Kr : q;
    cpx<T> v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int e = j + r * Kr;
      v[r] = in[AXIS == 1 ? plane_index(line, e, K2, swz) : plane_index(e, line, K2, swz)];
    }
    const int k = j - div_by(j, mns) * Ns;
    if (Ns > 1) twiddle<T, R, S>(v, tw, k * tstep);
    butterfly<T, R, S>(v);
    const int base = (j - k) * R + k;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int e = base + r * Ns;
      out[AXIS == 1 ? plane_index(line, e, K2, swz) : plane_index(e, line, K2, swz)] = v[r];
    }
  }
}

// All passes along one axis of the plane in `a` (scratch `b`); returns the
// buffer holding the result.  tw: the axis' twiddles (in LDS); mlines:
// div_magic of the lines of an x pass (K2).
template <typename T, int AXIS, int S>
__device__ cpx<T> *lds_fft_plane(cpx<T> *a, cpx<T> *b, const FftAxis &ax, int K1, int K2,
                                 int swz, uint32_t mlines, const cpx<T> *tw) {
  int Ns = 1;
  cpx<T> *in = a, *out = b;
  for (int s = 0; s < ax.nrad; ++s) {
    const int R = ax.rad[s];
    const uint32_t mdiv = AXIS == 1 ? ax.mkr[s] : mlines;
#define MDHIP_PASS(R_) \
  stockham_pass_plane<T, R_, AXIS, S>(in, out, K1, K2, swz, Ns, mdiv, ax.mns[s], tw)
    MDHIP_RADIX_SWITCH(R, MDHIP_PASS)
#undef MDHIP_PASS
    __syncthreads();
    cpx<T> *t = in;
    in = out;
    out = t;
    Ns *= R;
  }
  return in;
}

// The same passes with the plane's edges known at compile time (the grids
// the bench and its configs use): every index division is by a constant,
// and the pass loop unrolls.
constexpr int next_radix(int rest) {
  return rest % 8 == 0 ? 8 : rest % 4 == 0 ? 4 : rest % 2 == 0 ? 2 : rest % 3 == 0 ? 3
                                                                 : rest % 5 == 0 ? 5 : 7;
}

template <typename T, int R, int AXIS, int K1, int K2, int NS, int S>
__device__ __forceinline__ void stockham_pass_plane_k(const cpx<T> *in, cpx<T> *out, int swz,
                                                      const cpx<T> *tw) {
  constexpr int K = AXIS == 1 ? K2 : K1, nlines = AXIS == 1 ? K1 : K2;
  constexpr int Kr = K / R;
  constexpr int tstep = K / (NS * R);
  for (int w = threadIdx.x; w < nlines * Kr; w += blockDim.x) {
    int line, j;
    if (AXIS == 1) {
      j = w % Kr;
      line = w / Kr;
    } else {
      line = w % nlines;
      j = w / nlines;
    }
    cpx<T> v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int e = j + r * Kr;
      v[r] = in[AXIS == 1 ? plane_index(line, e, K2, swz) : plane_index(e, line, K2, swz)];
    }
    const int k = j % NS;
    if (NS > 1) twiddle<T, R, S>(v, tw, k * tstep);
    butterfly<T, R, S>(v);
    const int base = (j / NS) * NS * R + k;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int e = base + r * NS;
      out[AXIS == 1 ? plane_index(line, e, K2, swz) : plane_index(e, line, K2, swz)] = v[r];
    }
  }
}

template <typename T, int AXIS, int S, int K1, int K2, int NS = 1>
__device__ __forceinline__ cpx<T> *lds_fft_plane_k(cpx<T> *in, cpx<T> *out, int swz,
                                                   const cpx<T> *tw) {
  constexpr int K = AXIS == 1 ? K2 : K1;
  if constexpr (NS >= K) {
    return in;
  } else {
    constexpr int R = next_radix(K / NS);
    stockham_pass_plane_k<T, R, AXIS, K1, K2, NS, S>(in, out, swz, tw);
    __syncthreads();
    return lds_fft_plane_k<T, AXIS, S, K1, K2, NS * R>(out, in, swz, tw);
  }
}

}  // namespace mdhip
