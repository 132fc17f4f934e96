// Lengths with prime factors above 19 (32 < n <= 8192, of those to 127 the batches above 2048): the chirp
// transform (L. Bluestein, 1970).
//
//   X_k = w_k sum_i (x_i w_i) conj(w_(k - i)),   w_k = e^(-i pi k^2 / n)
//
// is a convolution, computed as two M-point Stockham transforms (M >= 2n - 1, a power of two)
// around a product with the transformed chirp, all in one launch: one workgroup holds `tpb`
// transforms, each on M / 16 threads with 16 points per thread in registers.
//
// The second transform runs the first one's radices in reverse order.  Its first pass then reads
// exactly the positions that the first transform's last pass left in the thread's registers, so
// the product needs no exchange through LDS, and its last pass leaves result i in the thread that
// loaded input i.  Transforms on at most 64 threads lie in one wavefront and exchange without
// workgroup barriers.  Points x_i, i >= n, are zero: M >= 2n - 1 puts them in the upper half, so
// the upper half of the first pass's loads and of the last pass's stores does not exist.
//
// What bounds it: the latency of 2 x (2..4) passes; the data (16 n bytes per transform) is a few
// per cent of that.  It took the place of an O(n^2) sum, whose n dependent loads per output were
// 886 us at 997 x 256 (now 8.6), 611 us at 829 x 241 (8.2) and 40.9 us at 47 x 3230 (5.7; device
// times, launch included); the error against 64 bits is smaller too (997: 1.8e-7 against 5.7e-7).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dft_direct.h"
#include "kernels.h"
#include "stockham_impl.h"

namespace asdfft {

namespace {

constexpr int kBlPoints = 16;  // points per thread

template <int... Rs>
struct Radices {};

template <int T>
__device__ __forceinline__ void bl_sync()
{
    if constexpr (T <= 64) {
        wave_lds_sync();
    } else {
        lds_barrier();
    }
}

// Passes of one M-point transform on the points in v (pass layout: butterfly b of the thread is
// j = tid + b T, its point r is j + r M / R); the last pass's outputs stay in v.
template <int M, int T, int SPAN, int TWOFF, int R, int... Rest>
__device__ __forceinline__ void bl_passes(float2 (&v)[kBlPoints], const float2* tw, float2* lds, int tid)
{
    constexpr int B = kBlPoints / R;
    static_assert(B * R == kBlPoints && T * kBlPoints == M, "every pass fills the thread's points");
#pragma unroll
    for (int b = 0; b < B; ++b) {
        if constexpr (SPAN > 1) {
            const float2* w = tw + TWOFF + ((tid + b * T) % SPAN) * (R - 1);
#pragma unroll
            for (int r = 1; r < R; ++r) v[b * R + r] = cmul(v[b * R + r], w[r - 1]);
        }
        Dft<R>::run(&v[b * R]);
    }
    if constexpr (sizeof...(Rest) > 0) {
        constexpr int RN = First<Rest...>::value;
        constexpr int BN = kBlPoints / RN;
        bl_sync<T>();  // the previous exchange's reads are done before its slots are overwritten
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const int j = tid + b * T;
            const int k = j % SPAN;
            const int base = (j - k) * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) lds[pad16(base + r * SPAN)] = v[b * R + r];
        }
        bl_sync<T>();
#pragma unroll
        for (int b = 0; b < BN; ++b) {
#pragma unroll
            for (int r = 0; r < RN; ++r) v[b * RN + r] = lds[pad16(tid + b * T + r * (M / RN))];
        }
        bl_passes<M, T, SPAN * R, TWOFF + (SPAN > 1 ? SPAN * (R - 1) : 0), Rest...>(v, tw, lds, tid);
    }
}

template <int M, int T, int... Rs>
__device__ __forceinline__ void bl_transform(Radices<Rs...>, float2 (&v)[kBlPoints], const float* tw, float2* lds,
                                             int tid)
{
    bl_passes<M, T, 1, 0, Rs...>(v, reinterpret_cast<const float2*>(tw), lds, tid);
}

template <int T>
constexpr int bl_block()
{
    return T > 256 ? T : 256;
}

// R1: first radix of the forward sequence F (the last of the reversed sequence I), RL: its last.
template <int M, int R1, int RL, typename F, typename I>
__global__ void __launch_bounds__((bl_block<M / kBlPoints>())) bluestein_kernel(const DftArgs a)
{
    extern __shared__ float smem[];
    constexpr int T = M / kBlPoints;
    constexpr int B1 = kBlPoints / R1, BL = kBlPoints / RL;
    const int tt = threadIdx.x / T;
    const int tid = threadIdx.x % T;
    float2* lds = reinterpret_cast<float2*>(smem) + tt * (M + M / 16 + 1);
    const int64_t t = dft_block(a) * a.tpb + tt;
    const bool live = t < a.count;
    const int n = live ? a.n : 0;  // lanes of a transform past the batch load and store nothing
    int64_t ib = t * a.in_dist;
    if (a.in_cols != 1) {  // uniform
        int64_t q, c;
        divmod_nonneg(t, a.in_cols, q, c);
        ib = c + q * a.in_dist;
    }
    const float2* chirp = reinterpret_cast<const float2*>(a.roots);
    float2 v[kBlPoints];
#pragma unroll
    for (int b = 0; b < B1; ++b) {
#pragma unroll
        for (int r = 0; r < R1; ++r) {
            const int i = tid + b * T + r * (M / R1);
            v[b * R1 + r] = make_float2(0.0f, 0.0f);
            if (r < R1 / 2 && i < n) v[b * R1 + r] = cmul(dft_load(a, ib, i), chirp[i]);
        }
    }
    bl_transform<M, T>(F{}, v, a.tw_first, lds, tid);
    const float2* filter = reinterpret_cast<const float2*>(a.filter);
#pragma unroll
    for (int b = 0; b < BL; ++b) {
#pragma unroll
        for (int r = 0; r < RL; ++r)
            v[b * RL + r] = conjf2(cmul(v[b * RL + r], filter[tid + b * T + r * (M / RL)]));
    }
    bl_transform<M, T>(I{}, v, a.tw_second, lds, tid);
#pragma unroll
    for (int b = 0; b < B1; ++b) {
#pragma unroll
        for (int r = 0; r < R1 / 2; ++r) {
            const int i = tid + b * T + r * (M / R1);
            if (i < n) dft_store(a, t * a.out_dist, i, cmul(conjf2(v[b * R1 + r]), chirp[i]));
        }
    }
}

}  // namespace

// Convolution lengths and their radices.  A sequence that reads the same in both directions
// needs one twiddle table for both transforms.
#define ASDFFT_BLUESTEIN(X)                        \
    X(128, 16, 8, (16, 8), (8, 16))                \
    X(256, 16, 16, (16, 16), (16, 16))             \
    X(512, 8, 8, (8, 8, 8), (8, 8, 8))             \
    X(1024, 8, 8, (8, 16, 8), (8, 16, 8))          \
    X(2048, 16, 16, (16, 8, 16), (16, 8, 16))      \
    X(4096, 16, 16, (16, 16, 16), (16, 16, 16))    \
    X(8192, 16, 8, (16, 8, 8, 8), (8, 8, 8, 16))   \
    X(16384, 16, 16, (16, 8, 8, 16), (16, 8, 8, 16))

#define ASDFFT_LIST(...) __VA_ARGS__

std::vector<int> bluestein_radices(int64_t m, bool second)
{
#define ASDFFT_BL_RADICES(M, R1, RL, F, I) \
    if (m == M) return second ? std::vector<int>{ASDFFT_LIST I} : std::vector<int>{ASDFFT_LIST F};
    ASDFFT_BLUESTEIN(ASDFFT_BL_RADICES)
#undef ASDFFT_BL_RADICES
    return {};
}

hipError_t launch_bluestein(const LaunchShape& s, const DftArgs& args, dim3 grid, hipStream_t stream)
{
#define ASDFFT_BL_LAUNCH(M, R1, RL, F, I)                                                                       \
    if (args.m == M) {                                                                                          \
        if (s.block > bl_block<M / kBlPoints>() || s.block != args.tpb * (M / kBlPoints)) return hipErrorInvalidConfiguration; \
        auto kern = bluestein_kernel<M, R1, RL, Radices<ASDFFT_LIST F>, Radices<ASDFFT_LIST I>>;                \
        if (s.lds_bytes > 65536) {                                                                              \
            static std::atomic<uint64_t> raised{0};                                                             \
            hipError_t e = raise_lds_limit_once(reinterpret_cast<const void*>(kern), raised);                   \
            if (e != hipSuccess) return e;                                                                      \
        }                                                                                                       \
        hipLaunchKernelGGL(kern, grid, dim3((unsigned)s.block), s.lds_bytes, stream, args);                     \
        return hipGetLastError();                                                                               \
    }
    ASDFFT_BLUESTEIN(ASDFFT_BL_LAUNCH)
#undef ASDFFT_BL_LAUNCH
    return hipErrorInvalidValue;
}

}  // namespace asdfft
