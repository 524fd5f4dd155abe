// dense_reduce.h -- the final reduction of the dense kernels' per-block
// records, in one order for every kernel that ends with it (dense_f64.hip,
// run_io.hip).
#ifndef SPM_DENSE_REDUCE_H
#define SPM_DENSE_REDUCE_H

#include "spm_device.h"

namespace spm {

// One block of 256 threads; `stride` doubles per record, `comps`
// double-double components per record.  Thread 0 gets out[3 comps]; red holds
// 12 doubles of LDS.
__device__ __forceinline__ void reduce_partials(const double* __restrict__ partial, int nrec, int stride, int comps,
                                                double* out, double* red)
{
    for (int q = 0; q < comps; ++q) {
        double h = 0.0, l = 0.0, a = 0.0;
        for (int i = threadIdx.x; i < nrec; i += blockDim.x) {
            const double* p = partial + (size_t)i * stride + 3 * q;
            dd_add(h, l, p[0], p[1]);
            a += p[2];
        }
        block_reduce_dd(h, l, a, red);
        if (threadIdx.x == 0) {
            out[3 * q + 0] = h;
            out[3 * q + 1] = l;
            out[3 * q + 2] = a;
        }
        __syncthreads();
    }
}

}  // namespace spm

#endif
