// Transforms of lengths 1, 23, 29, 31 and of others to 127 as sums over pairs, and the launch dispatcher
// for the Stockham variants.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dft_direct.h"
#include "kernels.h"
#include "stockham_impl.h"

namespace asdfft {

// Length 1: every element through its layout's load and store (an identity axis, a plan of N == 1).
__global__ void __launch_bounds__(256) dft_unit_kernel(const DftArgs a)
{
    const int64_t t = dft_block(a) * 256 + threadIdx.x;
    if (t >= a.count) return;
    dft_store(a, t * a.out_dist, 0, dft_load(a, (t % a.in_cols) + (t / a.in_cols) * a.in_dist, 0));
}

// Primes 23, 29, 31 as a sum over pairs: with a_i = x_i + x_(N-i) and b_i = x_i - x_(N-i),
//   X_k, X_(N-k) = x_0 + sum_i a_i cos(2 pi i k / N) -+ i sum_i b_i sin(2 pi i k / N).
// Sixteen lanes take one transform: lane k loads x_k and x_(N-k), shares the pair through LDS and
// stores X_k and X_(N-k).  At these lengths the sum of at most 15 pairs is quicker than the chirp
// transform (31 x 8451: 3.3 against 6.4 us, 29 x 7717: 2.9 against 6.3, launch included; one thread
// per output over all N terms took 33.0 and 30.2) and more exact (0.8-0.9e-7 against 1.2-1.3e-7).
constexpr int kPairLanes = 16;

template <int N>
__global__ void __launch_bounds__(256) dft_pairs_kernel(const DftArgs a)
{
    constexpr int H = (N - 1) / 2;
    static_assert(H < kPairLanes && N % 2 == 1, "lanes cover the pairs");
    __shared__ float4 pairs[256 / kPairLanes][kPairLanes];
    __shared__ float2 roots[N];
    const int tt = threadIdx.x / kPairLanes;
    const int k = threadIdx.x % kPairLanes;
    const int64_t t = dft_block(a) * (256 / kPairLanes) + tt;
    const bool live = t < a.count && k <= H;
    if (threadIdx.x < N) roots[threadIdx.x] = reinterpret_cast<const float2*>(a.roots)[threadIdx.x];
    if (live) {
        const int64_t ib = (t % a.in_cols) + (t / a.in_cols) * a.in_dist;
        const float2 x = dft_load(a, ib, k);
        const float2 y = (k == 0) ? make_float2(0.0f, 0.0f) : dft_load(a, ib, N - k);
        pairs[tt][k] = make_float4(x.x + y.x, x.y + y.y, x.x - y.x, x.y - y.y);
    }
    __syncthreads();
    if (!live) return;
    const float4 x0 = pairs[tt][0];
    float2 p = make_float2(x0.x, x0.y), s = make_float2(0.0f, 0.0f);
    int m = 0;
#pragma unroll
    for (int i = 1; i <= H; ++i) {
        m += k;
        if (m >= N) m -= N;
        const float2 w = roots[m];  // cos, -sin
        const float4 v = pairs[tt][i];
        p.x += v.x * w.x;
        p.y += v.y * w.x;
        s.x += v.z * w.y;
        s.y += v.w * w.y;
    }
    dft_store(a, t * a.out_dist, k, make_float2(p.x - s.y, p.y + s.x));
    if (k > 0) dft_store(a, t * a.out_dist, N - k, make_float2(p.x + s.y, p.y - s.x));
}

// The same sum at any length to 127, one transform per wavefront (lane k: X_k and X_(n-k)).  Its 63 terms
// at most take less than the passes of a chirp transform until the batch fills the chip: 43 x 4 4.3 us
// (chirp 6.2, the sum over all terms before that 4.4), 127 x 4 5.5 (7.0), 127 x 2048 7.0 (8.0).  Bound by
// the latency of the loads and of one LDS read of a root and a pair per term.
__global__ void __launch_bounds__(64) dft_sum_kernel(const DftArgs a)
{
    __shared__ float4 pairs[64];
    __shared__ float2 roots[kMaxSum];
    const int64_t t = dft_block(a);
    if (t >= a.count) return;  // the whole workgroup
    const int n = a.n, half = n / 2, k = threadIdx.x;
    const bool twice = k > 0 && 2 * k < n;  // x_k and x_(n-k) are two elements
    for (int m = threadIdx.x; m < n; m += 64) roots[m] = reinterpret_cast<const float2*>(a.roots)[m];
    if (k <= half) {
        const int64_t ib = (t % a.in_cols) + (t / a.in_cols) * a.in_dist;
        const float2 x = dft_load(a, ib, k);
        float4 v = make_float4(x.x, x.y, 0.0f, 0.0f);
        if (twice) {
            const float2 y = dft_load(a, ib, n - k);
            v = make_float4(x.x + y.x, x.y + y.y, x.x - y.x, x.y - y.y);
        }
        pairs[k] = v;
    }
    __syncthreads();
    if (k > half) return;
    // four running sums, added at the end: their error is half that of one
    float2 p[4], s[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) p[q] = s[q] = make_float2(0.0f, 0.0f);
    int m = 0;
    const auto add = [&](int i, int q) __attribute__((always_inline)) {
        m += k;
        if (m >= n) m -= n;
        const float2 w = roots[m];  // cos, -sin
        const float4 v = pairs[i];
        p[q].x += v.x * w.x;
        p[q].y += v.y * w.x;
        s[q].x += v.z * w.y;
        s[q].y += v.w * w.y;
    };
    int i = 1;
    for (; i + 3 <= half; i += 4) {
#pragma unroll
        for (int q = 0; q < 4; ++q) add(i + q, q);
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        if (i + q <= half) add(i + q, q);
    }
    const float2 u = cadd(make_float2(pairs[0].x, pairs[0].y), cadd(cadd(p[0], p[1]), cadd(p[2], p[3])));
    const float2 d = cadd(cadd(s[0], s[1]), cadd(s[2], s[3]));
    dft_store(a, t * a.out_dist, k, make_float2(u.x - d.y, u.y + d.x));
    if (twice) dft_store(a, t * a.out_dist, n - k, make_float2(u.x + d.y, u.y - d.x));
}

bool dft_pairs_length(int64_t n) { return n == 23 || n == 29 || n == 31; }

int dft_pairs_per_block() { return 256 / kPairLanes; }

hipError_t launch_dft_direct(const LaunchShape& s, const DftArgs& dft, hipStream_t stream)
{
    // A workgroup holds few of these transforms (16 of 23 points), and one dimension of a grid less
    // than 2^32 threads: 2^28 transforms of 23 points, 49 GB.  Rows of up to 65536 workgroups, of
    // equal length, so that at most one workgroup a row has nothing to do.
    const int64_t rows = (s.grid + 65535) / 65536;
    if (s.grid <= 0 || rows > 65535 || s.block <= 0 || s.block > 1024) return hipErrorInvalidConfiguration;
    DftArgs args = dft;
    args.row_blocks = (int)((s.grid + rows - 1) / rows);
    const dim3 grid((unsigned)args.row_blocks, (unsigned)rows);
    const bool sum = args.m == 0 && args.n > 1 && !dft_pairs_length(args.n);
    if (args.m > 0) return launch_bluestein(s, args, grid, stream);
    if (s.block != (sum ? 64 : 256) || (sum && args.n > kMaxSum)) return hipErrorInvalidConfiguration;
    auto kern = sum ? dft_sum_kernel : args.n == 23 ? dft_pairs_kernel<23> : args.n == 29 ? dft_pairs_kernel<29>
              : args.n == 31 ? dft_pairs_kernel<31> : dft_unit_kernel;
    hipLaunchKernelGGL(kern, grid, dim3((unsigned)s.block), 0, stream, args);
    return hipGetLastError();
}

#define ASDFFT_DECL(V, E) hipError_t launch_stockham_v##V##_e##E(const LaunchShape&, const FftArgs&, hipStream_t);
ASDFFT_FOR_EACH_INSTANCE(ASDFFT_DECL)
#undef ASDFFT_DECL

hipError_t launch_stockham(const LaunchShape& s, const FftArgs& args, hipStream_t stream)
{
    if (s.grid <= 0 || s.block <= 0 || s.block > 1024) return hipErrorInvalidConfiguration;
    if (s.static_id >= 0) {
        if (s.static_id >= kNumStaticInstances) return hipErrorInvalidValue;
        return kStaticInstances[s.static_id].launch(s, args, stream);
    }
#define ASDFFT_CASE(V, E) \
    if (s.variant == V && s.emax == E) return launch_stockham_v##V##_e##E(s, args, stream);
    ASDFFT_FOR_EACH_INSTANCE(ASDFFT_CASE)
#undef ASDFFT_CASE
    return hipErrorInvalidValue;
}

int find_static(int variant, int emax, int n, int threads, int tpb, const int* radices, int nradices)
{
    for (int i = 0; i < kNumStaticInstances; i++) {
        const StaticEntry& e = kStaticInstances[i];
        if (e.variant != variant || e.emax != emax || e.n != n || e.threads != threads || e.nradices != nradices) continue;
        if (e.tpb != 0 && e.tpb != tpb) continue;
        bool same = true;
        for (int p = 0; p < nradices; p++) same = same && (e.radices[p] == radices[p]);
        if (same) return i;
    }
    return -1;
}

}  // namespace asdfft
