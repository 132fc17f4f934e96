// Element loads and stores shared by the kernels that take DftArgs (dft_unit_kernel,
// bluestein_kernel): every prologue / epilogue as a uniform run-time branch, since these kernels
// are compiled once per length and not per layout.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_kernel_args.h"

namespace asdfft {

// Index of the workgroup: the grid has rows of row_blocks (launch_dft_direct).
__device__ __forceinline__ int64_t dft_block(const DftArgs& a)
{
    return (int64_t)blockIdx.y * a.row_blocks + blockIdx.x;
}

__device__ __forceinline__ float2 dft_load(const DftArgs& a, int64_t base, int i)
{
    const float2* in2 = reinterpret_cast<const float2*>(a.in);
    const int64_t s = a.in_stride;
    float2 x;
    if (a.prologue == kProReal) {
        x = make_float2(reinterpret_cast<const float*>(a.in)[base + i * s], 0.0f);
    } else if (a.prologue == kProPlanar) {
        x = make_float2(reinterpret_cast<const float*>(a.in)[base + i * s], a.in_im[base + i * s]);
    } else if (a.prologue == kProHerm) {
        const int h = a.n >> 1;
        if (i <= h) {
            x = in2[base + i * s];
            if (i == 0 || 2 * i == a.n) x.y = 0.0f;
        } else {
            x = in2[base + (a.n - i) * s];
            x.y = -x.y;
        }
    } else {
        x = in2[base + i * s];
    }
    if (a.conj_in) x.y = -x.y;
    return x;
}

__device__ __forceinline__ void dft_store(const DftArgs& a, int64_t base, int k, float2 x)
{
    if (a.epilogue == kEpiReal) {
        reinterpret_cast<float*>(a.out)[base + k] = x.x;
        return;
    }
    if (a.conj_out) x.y = -x.y;
    if (a.epilogue == kEpiPlanar) {
        reinterpret_cast<float*>(a.out)[base + k] = x.x;
        a.out_im[base + k] = x.y;
    } else if (a.epilogue != kEpiHalf) {
        reinterpret_cast<float2*>(a.out)[base + k] = x;
    } else if (2 * k <= a.n) {
        // A real input's bins 0 and n/2 are real.  The chirp transform leaves rounding there; the product
        // keeps what is not finite visible in both parts.
        if (k == 0 || 2 * k == a.n) x.y = 0.0f * x.x + 0.0f;
        reinterpret_cast<float2*>(a.out)[base + k] = x;
    }
}

}  // namespace asdfft
