// ISTFT in one launch: inverse frame transforms and overlap-add without the frames in memory.
//
// A workgroup makes `chunk_frames * hop` consecutive output samples of one channel.  It walks the
// frames that reach them in groups of F = fft.tpb: F adjacent columns of the (nfft, nframes)
// spectrum are transformed with the run-time column passes, the last pass leaves them in LDS, and
// the group's first F * hop samples, which no later frame reaches, are summed, normalised and
// stored.  Samples that later frames still add to stay in LDS as the next group's carry.  The
// first `halo` frames of a workgroup only fill the carry (the workgroup before transforms them
// too), so a chunk costs chunk_frames + halo frames.  The next group's spectrum is loaded into
// registers while the current one is transformed; twiddles and window are in LDS.
//
// Each sample adds its frames in ascending order, as istft_ola_kernel does.
//
// The separate launches also write and read every frame (16 bytes a point): 118 us for 16
// channels of 1000 frames of 1024 points at hop 256, 82.7 here.  VALU issue is 55% of that (65
// instructions a point), the rest are the barriers of 16 wavefronts per CU: 16 frames of 1024
// points with their tables fill the LDS.  16 frames are whole 128-byte lines of the spectrum;
// groups of 8 with two workgroups per CU took 94 us.  With the later passes' twiddles in global
// memory their wait also waited for the next group's spectrum (91 us); frames as padded rows in
// LDS conflicted on its banks (103 us).
#include "stockham_impl.h"

namespace asdfft {

namespace {

constexpr int kEmax = 16;

// q / hop for 0 <= q < 2^16
__device__ __forceinline__ int div_hop(int q, uint32_t magic, int hop)
{
    return hop == 1 ? q : (int)__umulhi((uint32_t)q, magic);
}

struct Walk {
    const float2* in;  // the channel's spectrum
    int64_t nframes;
    int n, T, F, tt, tid;
    // copies that the compiler cannot see through: it would otherwise keep the addresses of every
    // radix case in registers across the group loop
    __device__ __forceinline__ void opaque()
    {
        asm volatile("" : "+s"(n), "+s"(T), "+s"(F));
        asm volatile("" : "+v"(tid), "+v"(tt));
    }
};

// Point at a byte offset (the steps between a butterfly's points are uniform: one add each).
__device__ __forceinline__ float2& point(float2* frame, int bytes)
{
    return *reinterpret_cast<float2*>(reinterpret_cast<char*>(frame) + bytes);
}

// Points of pass 0 (radix R) of frame t: butterfly b of a thread takes elements j + r n / R,
// j = tid + b T.  Frames outside the signal are zero.
template <int R>
__device__ __forceinline__ void load_frame(Walk w, int64_t t, float2 (&pre)[kEmax])
{
    constexpr int B = kEmax / R;
    w.opaque();
    const int nr = w.n / R;
    const bool live = t >= 0 && t < w.nframes;
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int j = w.tid + b * w.T;
        const float2* at = w.in + j * w.nframes + t;
        const int64_t step = nr * w.nframes;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            pre[b * R + r] = make_float2(0.0f, 0.0f);
            if (live && j < nr) pre[b * R + r] = *at;
            at += step;
        }
    }
}

// Pass 0 on the loaded points (conjugated: the transform is inverse), then the loads of frame
// t_next.
template <int R>
__device__ __forceinline__ void first_pass(Walk w, int64_t t_next, bool more, float2 (&pre)[kEmax], float2* frame)
{
    constexpr int B = kEmax / R;
    w.opaque();
    const int nr = w.n / R, pitch = (w.F + 1) * 8;
    float2 v[B * R];
#pragma unroll
    for (int e = 0; e < B * R; ++e) v[e] = make_float2(pre[e].x, -pre[e].y);
    if (more) load_frame<R>(w, t_next, pre);
#pragma unroll
    for (int b = 0; b < B; ++b) Dft<R>::run(&v[b * R]);
    lds_barrier();  // the group before has been summed
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int j = w.tid + b * w.T;
        if (j < nr) {
#pragma unroll
            for (int r = 0; r < R; ++r) point(frame, j * R * pitch + r * pitch) = v[b * R + r];
        }
    }
    lds_barrier();
}

// A later pass, LDS to LDS.  Its twiddles are in LDS too: a wait on a global load would also wait
// for the next group's spectrum, which was asked for first.
template <int R>
__device__ __forceinline__ void later_pass(const FftArgs& a, Walk w, int p, float2* frame, const float2* tw)
{
    constexpr int B = kEmax / R;
    w.opaque();
    const int span = __builtin_amdgcn_readfirstlane(a.pass[p].span);
    const uint32_t magic = (uint32_t)__builtin_amdgcn_readfirstlane((int)a.pass[p].magic);
    tw += __builtin_amdgcn_readfirstlane(a.pass[p].tw_offset);
    const int nr = w.n / R, pitch = (w.F + 1) * 8;
    float2 v[B * R];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int j = w.tid + b * w.T;
        if (j < nr) {
            const float2* wk = tw + (j - (int)__umulhi((uint32_t)j, magic) * span) * (R - 1);
#pragma unroll
            for (int r = 0; r < R; ++r) v[b * R + r] = point(frame, j * pitch + r * nr * pitch);
#pragma unroll
            for (int r = 1; r < R; ++r) v[b * R + r] = cmul(v[b * R + r], wk[r - 1]);
            Dft<R>::run(&v[b * R]);
        }
    }
    lds_barrier();
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const int j = w.tid + b * w.T;
        if (j < nr) {
            const int k = j - (int)__umulhi((uint32_t)j, magic) * span;
            const int base = (j - k) * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) point(frame, base * pitch + r * span * pitch) = v[b * R + r];
        }
    }
    lds_barrier();
}

#define ASDFFT_ISTFT_RADICES(X) X(16) X(12) X(10) X(9) X(8) X(6) X(4) X(2) X(13) X(11) X(7) X(5) X(3)

__global__ void __launch_bounds__(1024) istft_fused_kernel(const IstftFusedArgs a)
{
    extern __shared__ float smem[];
    const FftArgs& f = a.fft;
    const OlaArgs& o = a.ola;
    const int F = f.tpb, n = f.n, hop = o.hop;
    const int tt = (int)threadIdx.x % F, tid = (int)threadIdx.x / F;
    const int nthreads = f.threads * F;
    float2* tile = reinterpret_cast<float2*>(smem);  // element i of frame e at i (F + 1) + e
    float2* frame = tile + tt;
    float2* carry = tile + n * (F + 1);
    const int ncarry = n - hop;  // hop <= n
    const int64_t blk = logical_block(1);
    const int64_t ch = blk / a.chunks, c = blk - ch * a.chunks;
    const int64_t f0 = c * a.chunk_frames - a.halo;
    const int64_t m_lo = c * a.chunk_frames * hop;
    const int64_t total = n + (int64_t)hop * (o.nframes - 1);
    const int radix0 = __builtin_amdgcn_readfirstlane(f.pass[0].radix);
    const int passes = __builtin_amdgcn_readfirstlane(f.passes);
    const int reach = a.halo + 1;  // frames that reach one sample, at most
    const Walk w{reinterpret_cast<const float2*>(a.spec) + ch * (int64_t)n * o.nframes, o.nframes, n, f.threads, F, tt, tid};
    float2* out = reinterpret_cast<float2*>(o.out) + ch * o.out_len;
    const int tw_count =
        passes > 1 ? f.pass[passes - 1].tw_offset + f.pass[passes - 1].span * (f.pass[passes - 1].radix - 1) : 0;
    float2* tw = carry + ncarry;
    float* window = reinterpret_cast<float*>(tw + tw_count);
    float* envelope = window + n;

    float2 pre[kEmax];
    switch (radix0) {
#define ASDFFT_CASE(RR) \
    case RR: load_frame<RR>(w, f0 + tt, pre); break;
        ASDFFT_ISTFT_RADICES(ASDFFT_CASE)
#undef ASDFFT_CASE
        default: break;
    }
    for (int j = threadIdx.x; j < ncarry; j += nthreads) carry[j] = make_float2(0.0f, 0.0f);
    for (int j = threadIdx.x; j < tw_count; j += nthreads) tw[j] = reinterpret_cast<const float2*>(f.tw)[j];
    for (int j = threadIdx.x; j < n; j += nthreads) window[j] = o.window[j];
    // squared-window sum of a sample q = j modulo hop that every frame around it reaches, in the
    // frames' ascending order
    for (int j = threadIdx.x; j < hop; j += nthreads) {
        float env = 0.0f;
        for (int k = j + div_hop(n - 1 - j, a.hop_magic, hop) * hop; k >= 0; k -= hop) env += o.window[k] * o.window[k];
        envelope[j] = env;
    }

    for (int grp = 0; grp < a.groups; ++grp) {
        const int64_t fb = f0 + (int64_t)grp * F;  // the group's first frame
        if (fb * hop >= total) break;              // past the signal (uniform)
        const bool more = grp + 1 < a.groups;
        switch (radix0) {
#define ASDFFT_CASE(RR) \
    case RR: first_pass<RR>(w, fb + F + tt, more, pre, frame); break;
            ASDFFT_ISTFT_RADICES(ASDFFT_CASE)
#undef ASDFFT_CASE
            default: break;
        }
        for (int p = 1; p < passes; ++p) {
            switch (__builtin_amdgcn_readfirstlane(f.pass[p].radix)) {
#define ASDFFT_CASE(RR) \
    case RR: later_pass<RR>(f, w, p, frame, tw); break;
                ASDFFT_ISTFT_RADICES(ASDFFT_CASE)
#undef ASDFFT_CASE
                default: break;
            }
        }
        // frames [e_first, e_last] of this group (numbered from its first) lie in the signal;
        // those before the group (negative) are in the carry
        const int e_first = fb < 0 ? (int)-fb : fb < reach ? (int)-fb : -reach;
        const int e_last = (int)(o.nframes - 1 - fb < F - 1 ? o.nframes - 1 - fb : F - 1);
        const int64_t m0 = fb * hop;
        const bool inside = e_first == -reach && e_last == F - 1;  // every frame around is in the signal
        // y += the group's frames lo .. hi at sample q, conjugated, times the window
        const auto add_frames = [&](int q, int lo, int hi, float2& y) __attribute__((always_inline)) {
            const float* wk = window + (q - lo * hop);
            const float2* v = tile + (q - lo * hop) * (F + 1) + lo;
            for (int e = lo; e <= hi; ++e) {
                y.x += v->x * *wk;
                y.y -= v->y * *wk;
                wk -= hop;
                v -= hop * (F + 1) - 1;
            }
        };
        for (int q = threadIdx.x; q < F * hop; q += nthreads) {
            const int64_t m = m0 + q;
            const int64_t i = m - o.start;
            if (m < m_lo || i < 0 || i >= o.out_len) continue;
            // first and last frame that cover the sample: q - n < e hop <= q
            const int last = div_hop(q, a.hop_magic, hop);
            const int lo = max(div_hop(q - n + reach * hop, a.hop_magic, hop) - reach + 1, e_first);
            const int hi = min(last, e_last);
            float env = 0.0f;
            if (inside) {
                env = envelope[q - last * hop];
            } else {
                for (int e = lo; e <= hi; ++e) env += window[q - e * hop] * window[q - e * hop];
            }
            float2 y = q < ncarry ? carry[q] : make_float2(0.0f, 0.0f);
            add_frames(q, max(lo, 0), hi, y);
            const float s = o.scale / env;
            out[i] = make_float2(y.x * s, y.y * s);
        }
        if (more) {
            lds_barrier();  // the carry has been read
            for (int j = threadIdx.x; j < ncarry; j += nthreads) {
                const int q = F * hop + j;
                const int lo = max(div_hop(q - n + reach * hop, a.hop_magic, hop) - reach + 1, max(e_first, 0));
                float2 y = make_float2(0.0f, 0.0f);
                add_frames(q, lo, e_last, y);
                carry[j] = y;
            }
        }
    }
}

}  // namespace

bool istft_fused_radix(int radix)
{
#define ASDFFT_HAS(RR) \
    if (radix == RR) return true;
    ASDFFT_ISTFT_RADICES(ASDFFT_HAS)
#undef ASDFFT_HAS
    return false;
}

hipError_t launch_istft_fused(const IstftFusedArgs& args, int64_t grid, size_t lds_bytes, hipStream_t stream)
{
    const int block = args.fft.tpb * args.fft.threads;
    if (grid <= 0 || block <= 0 || block > 1024 || grid > 0xffffffff / block || args.ola.hop <= 0 || args.ola.hop > args.fft.n ||
        args.groups <= 0 || args.chunk_frames <= 0)
        return hipErrorInvalidValue;
    if (lds_bytes > 65536) {
        static std::atomic<uint64_t> raised{0};
        const hipError_t e = raise_lds_limit_once(reinterpret_cast<const void*>(istft_fused_kernel), raised);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(istft_fused_kernel, dim3((unsigned)grid), dim3((unsigned)block), lds_bytes, stream, args);
    return hipGetLastError();
}

}  // namespace asdfft
