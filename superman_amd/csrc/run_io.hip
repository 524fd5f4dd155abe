// run_io.hip -- the first and the last kernel of every single-matrix run
// (capi.cpp): the matrix from the host's pinned memory into the plan's device
// memory, and the reduced sums back into pinned memory behind a flag the host
// polls.  With the plan's memory from a pool (workspace.cpp) a call then makes
// no allocation, no copy command and no stream synchronization: order 8 from
// 77-97 to 20 us a call, of which 9 us are three launches and a flag.
#include "dense_reduce.h"
#include "spm_kernels.h"

namespace spm {
namespace {

// 100 MHz counter common to the device's compute dies.
__device__ __forceinline__ unsigned long long ticks() { return __builtin_amdgcn_s_memrealtime(); }

__device__ __forceinline__ void store_host(unsigned long long* p, unsigned long long v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The finishing thread's stores: `words` result words, the run's ticks, then
// the flag.
__device__ __forceinline__ void publish(const unsigned long long* w, int words, const unsigned long long* t0,
                                        RunResult* host, unsigned int seq)
{
    for (int i = 0; i < words; ++i) store_host(&host->word[i], w[i]);
    store_host(&host->ticks, ticks() - *t0);
    __hip_atomic_store(&host->flag, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

// words 16-byte words from src (pinned host memory) to dst, zwords of zeros
// to zero, and the run's start time.
__global__ void __launch_bounds__(256)
run_begin_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst, unsigned int words, uint4* __restrict__ zero,
                 unsigned int zwords, unsigned long long* __restrict__ t0)
{
    const unsigned int t = blockIdx.x * 256 + threadIdx.x, step = gridDim.x * 256;
    for (unsigned int i = t; i < words; i += step) dst[i] = src[i];
    for (unsigned int i = t; i < zwords; i += step) zero[i] = make_uint4(0u, 0u, 0u, 0u);
    if (t == 0) *t0 = ticks();
}

// Double-double records (reduce_partials, as spm_dense_f64_noalloc's).
__global__ void __launch_bounds__(256)
run_end_dd_kernel(const double* __restrict__ partial, int nrec, int stride, int comps,
                  const unsigned long long* __restrict__ t0, RunResult* host, unsigned int seq)
{
    __shared__ double red[3 * (256 / kWave)];
    double out[6];
    reduce_partials(partial, nrec, stride, comps, out, red);
    if (threadIdx.x == 0) {
        unsigned long long w[6];
        for (int i = 0; i < 3 * comps; ++i) w[i] = (unsigned long long)__double_as_longlong(out[i]);
        publish(w, 3 * comps, t0, host, seq);
    }
}

// Integer records, summed mod 2^128.
__global__ void __launch_bounds__(256)
run_end_i128_kernel(const unsigned long long* __restrict__ partial, int nrec,
                    const unsigned long long* __restrict__ t0, RunResult* host, unsigned int seq)
{
    __shared__ unsigned long long red[2 * (256 / kWave)];
    unsigned __int128 t = 0;
    for (int i = threadIdx.x; i < nrec; i += 256)
        t += ((unsigned __int128)partial[2 * i + 1] << 64) | partial[2 * i];
    unsigned long long lo = (unsigned long long)t, hi = (unsigned long long)(t >> 64);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const unsigned long long olo = __shfl_xor(lo, off, kWave);
        const unsigned long long ohi = __shfl_xor(hi, off, kWave);
        const unsigned long long s = lo + olo;
        hi = hi + ohi + (s < lo ? 1ull : 0ull);
        lo = s;
    }
    if ((threadIdx.x & (kWave - 1)) == 0) {
        red[2 * (threadIdx.x / kWave)] = lo;
        red[2 * (threadIdx.x / kWave) + 1] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned __int128 s = 0;
        for (int i = 0; i < 256 / kWave; ++i) s += ((unsigned __int128)red[2 * i + 1] << 64) | red[2 * i];
        const unsigned long long w[2] = {(unsigned long long)s, (unsigned long long)(s >> 64)};
        publish(w, 2, t0, host, seq);
    }
}

const void* run_begin_kernel_ptr() { return reinterpret_cast<const void*>(&run_begin_kernel); }
const void* run_end_dd_kernel_ptr() { return reinterpret_cast<const void*>(&run_end_dd_kernel); }
const void* run_end_i128_kernel_ptr() { return reinterpret_cast<const void*>(&run_end_i128_kernel); }

}  // namespace spm
