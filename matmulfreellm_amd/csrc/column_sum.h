// The column sums of per-workgroup partial rows, for the weight gradients of the row kernels.
#pragma once
#include "mmf_common.h"

namespace {

// out[k] = T(sum_g part[g, k]).  A workgroup owns 32 columns; its 32 lanes per column each add every 32nd group in index order and
// the 32 lane sums are then added in lane order, so the result depends on the shape only.
constexpr int kColsumCols = 32, kColsumLanes = 32;
template <typename T>
__global__ __launch_bounds__(kColsumCols * kColsumLanes) void colsum_kernel(const float* __restrict__ part, int groups, int K,
                                                                            T* __restrict__ out) {
    __shared__ float lane_sum[kColsumLanes][kColsumCols + 1];
    const int c = (int)threadIdx.x % kColsumCols, l = (int)threadIdx.x / kColsumCols;
    const int k = (int)blockIdx.x * kColsumCols + c;
    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
    if (k < K) {
        int g = l;
        for (; g + 3 * kColsumLanes < groups; g += 4 * kColsumLanes) {
            const float a0 = part[(int64_t)g * K + k], a1 = part[(int64_t)(g + kColsumLanes) * K + k];
            const float a2 = part[(int64_t)(g + 2 * kColsumLanes) * K + k], a3 = part[(int64_t)(g + 3 * kColsumLanes) * K + k];
            s0 += a0; s1 += a1; s2 += a2; s3 += a3;
        }
        for (; g < groups; g += kColsumLanes) s0 += part[(int64_t)g * K + k];
    }
    lane_sum[l][c] = (s0 + s1) + (s2 + s3);
    __syncthreads();
    if (l == 0 && k < K) {
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < kColsumLanes; ++i) s += lane_sum[i][c];
        out[k] = mmf_from_float<T>(s);
    }
}
template <typename T>
void launch_colsum(const float* part, int groups, int64_t K, T* out, hipStream_t s) {
    colsum_kernel<T><<<(unsigned)mmf_ceil_div(K, kColsumCols), kColsumCols * kColsumLanes, 0, s>>>(part, groups, (int)K, out);
}

}  // namespace
