// Right-padding masks: the valid length of every row of a boolean mask [B, T],
// or -1 for a row whose valid tokens are no prefix (src/kda/utils.py:8-29 checks
// the same with tensor operations and two host reads).  One workgroup per row
// and one launch: the mask's reductions, comparisons and type copies took about
// 50 us in ten launches for 8 x 1000 tokens, between two waits of the host; this
// is one launch of 4 us and one wait.
#include "kda_launch.h"

namespace kda {

constexpr int kMaskThreads = 256;

__global__ __launch_bounds__(kMaskThreads) void mask_lengths_kernel(const uint8_t* mask, int64_t T, int32_t* lengths) {
  __shared__ int32_t count[kMaskThreads / 64];
  __shared__ int32_t top[kMaskThreads / 64];
  const uint8_t* row = mask + static_cast<int64_t>(blockIdx.x) * T;
  const int tid = threadIdx.x;
  // a prefix: as many valid tokens as the last valid one's position says
  int32_t n = 0, last = 0;
  for (int64_t t = tid; t < T; t += kMaskThreads)
    if (row[t] != 0) {
      ++n;
      last = static_cast<int32_t>(t) + 1;
    }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    n += __shfl_xor(n, off);
    const int32_t other = __shfl_xor(last, off);
    last = other > last ? other : last;
  }
  if ((tid & 63) == 0) {
    count[tid >> 6] = n;
    top[tid >> 6] = last;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < kMaskThreads / 64; ++w) {
      n += count[w];
      last = top[w] > last ? top[w] : last;
    }
    lengths[blockIdx.x] = n == last ? n : -1;
  }
}

}  // namespace kda

namespace kda_host {

int launch_mask_lengths(const uint8_t* mask, int64_t batch, int64_t tokens, int32_t* lengths, hipStream_t stream) {
  hipLaunchKernelGGL(kda::mask_lengths_kernel, dim3(static_cast<unsigned>(batch)), dim3(kda::kMaskThreads), 0, stream,
                     mask, tokens, lengths);
  return check_launch("mask_lengths_kernel");
}

}  // namespace kda_host
