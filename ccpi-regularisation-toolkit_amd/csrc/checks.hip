// checks.hip -- self-checks of the library's own arithmetic building blocks
// on the device they run on.
#include "runtime.hpp"
#include "../../include/cilreg_ext.h"

namespace cilreg {

namespace {

// Every 32-bit pattern [lo, hi) as a float: sqrt_rn against sqrtf, bit for
// bit (any NaN matching any NaN).  Mismatches and checked values are summed
// per workgroup, then added to the two counters.
__global__ __launch_bounds__(256) void check_sqrt_kernel(unsigned long long lo, unsigned long long hi,
                                                         unsigned long long* counts) {
    __shared__ unsigned long long red[2][4];
    unsigned long long bad = 0, seen = 0;
    for (unsigned long long u = lo + (unsigned long long)blockIdx.x * 256 + threadIdx.x; u < hi;
         u += (unsigned long long)gridDim.x * 256) {
        const float x = __uint_as_float((uint32_t)u);
        const float a = sqrt_rn(x), b = sqrtf(x);
        const bool same = __float_as_uint(a) == __float_as_uint(b) || (a != a && b != b);
        bad += same ? 0 : 1;
        seen += 1;
    }
    #pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        bad += __shfl_xor(bad, off, 64);
        seen += __shfl_xor(seen, off, 64);
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { red[0][w] = bad; red[1][w] = seen; }
    __syncthreads();
    if (threadIdx.x == 0) {
        atomicAdd(&counts[0], red[0][0] + red[0][1] + red[0][2] + red[0][3]);
        atomicAdd(&counts[1], red[1][0] + red[1][1] + red[1][2] + red[1][3]);
    }
}

// Every 32-bit pattern [lo, hi) as a float s: Mixed<float>::rof_sqrt_d(s,
// eps) against (float)sqrt((double)s + eps), bit for bit (any NaN matching any
// NaN).  Negative s (which the fluxes never produce) is skipped.
__global__ __launch_bounds__(256) void check_rof_sqrt_d_kernel(unsigned long long lo, unsigned long long hi,
                                                               double eps, unsigned long long* counts) {
    __shared__ unsigned long long red[2][4];
    unsigned long long bad = 0, seen = 0;
    for (unsigned long long u = lo + (unsigned long long)blockIdx.x * 256 + threadIdx.x; u < hi;
         u += (unsigned long long)gridDim.x * 256) {
        const float x = __uint_as_float((uint32_t)u);
        const float a = Mixed<float>::rof_sqrt_d(x, eps), b = (float)sqrt((double)x + eps);
        const bool same = __float_as_uint(a) == __float_as_uint(b) || (a != a && b != b);
        bad += same ? 0 : 1;
        seen += 1;
    }
    #pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        bad += __shfl_xor(bad, off, 64);
        seen += __shfl_xor(seen, off, 64);
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { red[0][w] = bad; red[1][w] = seen; }
    __syncthreads();
    if (threadIdx.x == 0) {
        atomicAdd(&counts[0], red[0][0] + red[0][1] + red[0][2] + red[0][3]);
        atomicAdd(&counts[1], red[1][0] + red[1][1] + red[1][2] + red[1][3]);
    }
}

__device__ inline void add_counts(unsigned long long bad, unsigned long long seen, unsigned long long* counts) {
    __shared__ unsigned long long red[2][4];
    #pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        bad += __shfl_xor(bad, off, 64);
        seen += __shfl_xor(seen, off, 64);
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { red[0][w] = bad; red[1][w] = seen; }
    __syncthreads();
    if (threadIdx.x == 0) {
        atomicAdd(&counts[0], red[0][0] + red[0][1] + red[0][2] + red[0][3]);
        atomicAdd(&counts[1], red[1][0] + red[1][1] + red[1][2] + red[1][3]);
    }
}

// rcp_in against 1 / y for every positive float y in [2^-125, 2^125].
__global__ __launch_bounds__(256) void check_rcp_in_kernel(unsigned long long* counts) {
    unsigned long long bad = 0, seen = 0;
    for (uint32_t u = (2u << 23) + blockIdx.x * 256u + threadIdx.x; u <= (252u << 23); u += gridDim.x * 256u) {
        const float y = __uint_as_float(u);
        bad += __float_as_uint(rcp_in(y)) != __float_as_uint(1.0f / y);
        seen += 1;
    }
    add_counts(bad, seen, counts);
}

// div_in against a / y: every significand of y (exponents cycling over
// [2^-60, 2^60]) with every stride-th significand of a, the offset moving with
// y (exponents cycling over [2^-60, 2^60], both signs).
__global__ __launch_bounds__(256) void check_div_in_kernel(uint32_t stride, unsigned long long* counts) {
    unsigned long long bad = 0, seen = 0;
    for (uint32_t m = blockIdx.x; m < (1u << 23); m += gridDim.x) {
        const float y = __uint_as_float(((67u + m % 121u) << 23) | m);
        const float r = rcp_in(y);
        for (uint32_t k = m % stride + stride * threadIdx.x; k < (1u << 23); k += stride * 256u) {
            const uint32_t h = (m ^ k) * 2654435761u;
            const float a = __uint_as_float((h & 0x80000000u) | ((67u + (h >> 8) % 121u) << 23) | k);
            bad += __float_as_uint(div_in(a, y, r)) != __float_as_uint(a / y);
            seen += 1;
        }
    }
    add_counts(bad, seen, counts);
}

// Runs a counting kernel and reads its two counters.
template <class F>
int run_counts(F&& launch, unsigned long long* mismatches, unsigned long long* checked) {
    if (!mismatches || !checked) { set_error("null pointer argument"); return -1; }
    hipStream_t s = device_stream();
    if (!s) { set_error("no stream"); return -1; }
    Arena ar;
    const size_t oc = ar.reserve(2 * sizeof(unsigned long long));
    if (ar.allocate() != 0) return -1;
    unsigned long long* d = (unsigned long long*)ar.at(oc);
    launch_zero(d, 2 * sizeof(unsigned long long), s);
    launch(d, s);
    unsigned long long h[2] = {0, 0};
    CILREG_CK(hipGetLastError());
    CILREG_CK(hipMemcpyAsync(h, d, sizeof h, hipMemcpyDeviceToHost, s));
    CILREG_CK(hipStreamSynchronize(s));
    *mismatches = h[0];
    *checked = h[1];
    return 0;
}

}  // namespace

}  // namespace cilreg

using namespace cilreg;

extern "C" {

int cilreg_check_sqrt_rn(unsigned long long* mismatches, unsigned long long* checked) {
    if (!mismatches || !checked) { set_error("null pointer argument"); return -1; }
    hipStream_t s = device_stream();
    if (!s) { set_error("no stream"); return -1; }
    Arena ar;
    const size_t oc = ar.reserve(2 * sizeof(unsigned long long));
    if (ar.allocate() != 0) return -1;
    unsigned long long* d = (unsigned long long*)ar.at(oc);
    launch_zero(d, 2 * sizeof(unsigned long long), s);
    hipLaunchKernelGGL(check_sqrt_kernel, dim3(16384), dim3(256), 0, s, 0ULL, 1ULL << 32, d);
    unsigned long long h[2] = {0, 0};
    CILREG_CK(hipGetLastError());
    CILREG_CK(hipMemcpyAsync(h, d, sizeof h, hipMemcpyDeviceToHost, s));
    CILREG_CK(hipStreamSynchronize(s));
    *mismatches = h[0];
    *checked = h[1];
    return 0;
}

int cilreg_check_rof_sqrt_d(double eps, unsigned long long* mismatches, unsigned long long* checked) {
    if (!mismatches || !checked) { set_error("null pointer argument"); return -1; }
    if (!(eps > 0.0)) { set_error("eps must be positive"); return -1; }
    hipStream_t s = device_stream();
    if (!s) { set_error("no stream"); return -1; }
    Arena ar;
    const size_t oc = ar.reserve(2 * sizeof(unsigned long long));
    if (ar.allocate() != 0) return -1;
    unsigned long long* d = (unsigned long long*)ar.at(oc);
    launch_zero(d, 2 * sizeof(unsigned long long), s);
    // non-negative patterns: +0 .. +inf and the positive NaNs
    hipLaunchKernelGGL(check_rof_sqrt_d_kernel, dim3(16384), dim3(256), 0, s, 0ULL, 1ULL << 31, eps, d);
    unsigned long long h[2] = {0, 0};
    CILREG_CK(hipGetLastError());
    CILREG_CK(hipMemcpyAsync(h, d, sizeof h, hipMemcpyDeviceToHost, s));
    CILREG_CK(hipStreamSynchronize(s));
    *mismatches = h[0];
    *checked = h[1];
    return 0;
}

int cilreg_check_rcp_in(unsigned long long* mismatches, unsigned long long* checked) {
    return run_counts([](unsigned long long* d, hipStream_t s) {
        hipLaunchKernelGGL(check_rcp_in_kernel, dim3(16384), dim3(256), 0, s, d);
    }, mismatches, checked);
}

int cilreg_check_div_in(unsigned stride, unsigned long long* mismatches, unsigned long long* checked) {
    if (stride == 0 || stride > 4096) { set_error("stride must be 1..4096"); return -1; }
    return run_counts([stride](unsigned long long* d, hipStream_t s) {
        hipLaunchKernelGGL(check_div_in_kernel, dim3(65536), dim3(256), 0, s, stride, d);
    }, mismatches, checked);
}

}  // extern "C"
