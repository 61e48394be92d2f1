// Vectors between the caller's DOF order and the library's, on the device: the
// host's array crosses the bus as it is and one kernel permutes it (and zeroes
// prescribed DOFs, apply_zero!).  A host loop over the permutation ran at the
// latency of its scattered side, 34 ms each way for 12.8 million DOFs; a load of that
// length is now set, checked and permuted in 3.5 ms, of which the bus takes 3.3.
#include "k_common.h"

namespace tohip {

// out[i] = in[perm[i]] (in[i] without perm); 0 where mask has DOF i prescribed.
__global__ __launch_bounds__(kThreads) void k_order_gather(int64_t n, int dim,
                                                           const int* __restrict__ perm,
                                                           const uint8_t* __restrict__ mask,
                                                           const double* __restrict__ in,
                                                           double* __restrict__ out) {
    for (int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kThreads) {
        const double v = in[perm ? perm[i] : i];
        out[i] = mask && ((mask[i / dim] >> (i % dim)) & 1) ? 0.0 : v;
    }
}

// out[perm[i]] = in[i].
__global__ __launch_bounds__(kThreads) void k_order_scatter(int64_t n, const int* __restrict__ perm,
                                                            const double* __restrict__ in,
                                                            double* __restrict__ out) {
    for (int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kThreads)
        out[perm[i]] = in[i];
}

// {hi, lo} += {a, b}: Knuth's two-sum of the high parts, low parts alongside.
__device__ __forceinline__ void add_pair(double& hi, double& lo, double a, double b) {
    const double s = hi + a, t = s - hi;
    lo += ((hi - (s - t)) + (a - t)) + b;
    hi = s;
}

// Per-block partials {sum of squares as high + low part, count of non-finite
// values}.  The squares are summed in twice double precision, as on the host in
// extended precision: the stopping tolerances scale with the root.
__global__ __launch_bounds__(kThreads) void k_values_check(int64_t n, const double* __restrict__ x,
                                                           double* __restrict__ part) {
    __shared__ double sh[kThreads], sl[kThreads], sb[kThreads];
    double hi = 0.0, lo = 0.0, bad = 0.0;
    for (int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kThreads) {
        const double v = x[i], p = v * v;
        add_pair(hi, lo, p, __builtin_fma(v, v, -p));
        bad += isfinite(v) ? 0.0 : 1.0;
    }
    const int t = threadIdx.x;
    sh[t] = hi;
    sl[t] = lo;
    sb[t] = bad;
    for (int w = kThreads / 2; w > 0; w >>= 1) {
        __syncthreads();
        if (t < w) {
            add_pair(sh[t], sl[t], sh[t + w], sl[t + w]);
            sb[t] += sb[t + w];
        }
    }
    if (t == 0) {
        part[3 * (size_t)blockIdx.x] = sh[0];
        part[3 * (size_t)blockIdx.x + 1] = sl[0];
        part[3 * (size_t)blockIdx.x + 2] = sb[0];
    }
}

static unsigned order_blocks(int64_t n) {
    const int64_t b = (n + kThreads - 1) / kThreads;
    return (unsigned)(b < 1 ? 1 : b > 4096 ? 4096 : b);
}

hipError_t launch_order_gather(int64_t n, int dim, const int* perm, const uint8_t* mask,
                               const double* in, double* out, hipStream_t s) {
    hipLaunchKernelGGL(k_order_gather, dim3(order_blocks(n)), dim3(kThreads), 0, s, n, dim, perm,
                       mask, in, out);
    return hipGetLastError();
}

hipError_t launch_order_scatter(int64_t n, const int* perm, const double* in, double* out,
                                hipStream_t s) {
    hipLaunchKernelGGL(k_order_scatter, dim3(order_blocks(n)), dim3(kThreads), 0, s, n, perm, in,
                       out);
    return hipGetLastError();
}

hipError_t values_check(int64_t n, const double* x, double* partials, long double* sumsq,
                        double* bad, hipStream_t s) {
    hipLaunchKernelGGL(k_values_check, dim3(kVecBlocks), dim3(kThreads), 0, s, n, x, partials);
    hipError_t e = hipGetLastError();
    double h[3 * kVecBlocks];
    if (e == hipSuccess)
        e = hipMemcpyAsync(h, partials, sizeof(h), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return e;
    *sumsq = 0.0L;
    *bad = 0.0;
    for (int b = 0; b < kVecBlocks; ++b) {
        *sumsq += (long double)h[3 * b] + h[3 * b + 1];
        *bad += h[3 * b + 2];
    }
    return hipSuccess;
}

}  // namespace tohip
