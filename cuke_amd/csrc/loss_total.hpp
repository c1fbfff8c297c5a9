// The last sum of the margin loss, for the kernels that carry it.
#pragma once

#include "common.hpp"

namespace kge {

constexpr int kLossBlocks = 1024;  // partial losses of a batch, at most

#ifdef __HIPCC__
// One workgroup of 256 threads; s: 256 doubles of LDS.
__device__ __forceinline__ void loss_total_block(const kge_loss_total &total, double *s)
{
    const int n = (int)total.n;
    double acc = 0.0;
    if (n > 0) {  // uniform; an empty batch has no partial, and may have no workspace, to read
        double v[kLossBlocks / 256];  // all loads of a thread in flight together
#pragma unroll
        for (int q = 0; q < kLossBlocks / 256; ++q) {
            const int i = threadIdx.x + 256 * q;
            v[q] = total.parts[i < n ? i : 0];
            if (i >= n) v[q] = 0.0;
        }
#pragma unroll
        for (int q = 0; q < kLossBlocks / 256; ++q) acc += v[q];
    }
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) s[threadIdx.x] += s[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) total.loss[0] = (float)(s[0] * total.scale);
}
#endif

}  // namespace kge
