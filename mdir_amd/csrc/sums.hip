// sums.hip — the energies of an evaluation and the kinetic energy, summed on
// the GPU from the kernels' partial sums and the velocities.
//
// Every sum is taken in a fixed order: a thread's share at a fixed stride, a
// tree over the block's threads, the blocks in order on the host.
#include "md_common.h"

namespace mdhip {

constexpr int kSumBlocks = 128;
constexpr int kSumWidth = 5;   // components per entry at most
enum SumKind { kSumPairs = 0, kSumSpecial = 1, kSumTuples = 2, kSumRecip = 3, kSumKinetic = 4,
               kSumKinds = 5 };

struct SumArgs {
  const double *src[kSumKinetic];   // entries of `width` doubles each
  long long count[kSumKinetic];
  int width[kSumKinetic];
  const double *v, *mass;           // of the kinetic energy, n atoms (0: none)
  int n;
};

// Grid: kSumBlocks x kSumKinds blocks; out[kind][block][component].  One
// launch and a copy of 26 KB in place of the copies of every partial sum
// and of the velocities: at 999,000 atoms those are 30 MB per evaluation.
__global__ void __launch_bounds__(256) energy_sums(SumArgs a, double *__restrict__ out) {
  __shared__ double s_w[4][kSumWidth];
  const int kind = blockIdx.y;
  const long long first = (long long)blockIdx.x * 256 + threadIdx.x,
                  stride = (long long)kSumBlocks * 256;
  double e[kSumWidth] = {0.0, 0.0, 0.0, 0.0, 0.0};
  if (kind == kSumKinetic) {
    for (long long i = first; i < a.n; i += stride) {
      const double x = a.v[3 * i], y = a.v[3 * i + 1], z = a.v[3 * i + 2];
      e[0] += 0.5 * a.mass[i] * (x * x + y * y + z * z);
    }
  } else {
    const double *src = a.src[kind];
    const int width = a.width[kind];
    for (long long i = first; i < a.count[kind]; i += stride) {
#pragma unroll
      for (int c = 0; c < kSumWidth; ++c)
        if (c < width) e[c] += src[i * width + c];
    }
  }
#pragma unroll
  for (int c = 0; c < kSumWidth; ++c) {
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) e[c] += __shfl_xor(e[c], s);
    if (threadIdx.x % 64 == 0) s_w[threadIdx.x / 64][c] = e[c];
  }
  __syncthreads();
  if (threadIdx.x < kSumWidth)
    out[((size_t)kind * kSumBlocks + blockIdx.x) * kSumWidth + threadIdx.x] =
        (s_w[0][threadIdx.x] + s_w[1][threadIdx.x]) + (s_w[2][threadIdx.x] + s_w[3][threadIdx.x]);
}

}  // namespace mdhip
