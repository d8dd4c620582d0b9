// Device code for sums over the rows of a matrix, as source text for hipRTC.
#pragma once

namespace tc {
namespace hip {

// O(n) = sum over r of A(r, n), in kernels the mapper gives to it (mapper.cc, takeColumnSums).
//
// A block sums 16 columns: a wavefront reads four rows of them (64 bytes of each) at a time, kWaves wavefronts take turns, and
// the partial sums of the lanes meet in LDS.  With one thread a column, 64 columns a block, the loads of a thread are a serial chain
// of batches as long as the unroll budget, on as many compute units as there are 64 columns.  The gradient of a bias over 1024 x 1024 took
// 13.5 us and takes 2.8, 700 x 2500 34.6 and 4.6, 1024 x 4096 18.0 and 6.8, 100 x 300 2.8 and 2.3; 64 rows take the 2.1 to 2.3 us of a launch
// either way.  What bounds this form is one or two round trips to memory behind the launch.
constexpr const char* kDeviceColumnSums = R"HIP(
namespace __tc {
template <int R, int N, int kWaves> __device__ __forceinline__ void columnSums(float* pO, const float* pA, float* sums) {
  constexpr int kLanes = 4 * kWaves, kTurns = (R + kLanes - 1) / kLanes, kFlight = kTurns < 16 ? kTurns : 16;
  const int column = threadIdx.x & 15, row = 4 * threadIdx.y + (threadIdx.x >> 4), n = 16 * blockIdx.x + column;
  const float* p = pA + tmin(n, N - 1);
  float part[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
  for (int t0 = 0; t0 < kTurns; t0 += kFlight) {
    float v[kFlight];
#pragma unroll
    for (int t = 0; t < kFlight; ++t) v[t] = p[tmin(row + (t0 + t) * kLanes, R - 1) * N];
#pragma unroll
    for (int t = 0; t < kFlight; ++t) part[t & 3] += row + (t0 + t) * kLanes < R ? v[t] : 0.0f;
  }
  sums[row * 16 + column] = (part[0] + part[1]) + (part[2] + part[3]);
  __syncthreads();
  if (threadIdx.y != 0) return;
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) sum += sums[(row + 4 * i) * 16 + column];
  // (what a wavefront writes to LDS it reads in order)
  sums[row * 16 + column] = sum;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  if (row == 0 && n < N) pO[n] = (sums[column] + sums[16 + column]) + (sums[32 + column] + sums[48 + column]);
}
}
)HIP";

} // namespace hip
} // namespace tc
