// The spectral front end over the real FFT, fused (the reference's hesap-dsp spectral.hpp:43-126, :140-172,
// :334-386: Welch PSD, spectrogram, periodogram and STFT, which there run frame by frame as detrend + window loops,
// a RealFftPlan rfft and a |X|^2 loop).
//
// k_spec<H, E, MODE>: one real frame of N = 2H samples per group of T = H/E threads (several frames per workgroup
// below 256 threads). Each thread loads the sample pairs of its complex slots j = i + T m straight from the signal
// (frame s starts at s * hop, any hop), subtracts the frame mean (a workgroup tree reduction, fixed order) when
// asked, multiplies by the window, runs the H-point Stockham core on z[j] = x[2j] + i x[2j+1], and does the
// Hermitian recombine X[k] = E[k] + W_N^k O[k], E = (Z[k] + conj Z[H-k])/2, O = (Z[k] - conj Z[H-k])/(2i), with
// Z[H-k] read back through LDS; X[H] = Re Z[0] - Im Z[0] comes from the k = 0 slot. The epilogue then writes
//   MODE 0  the complex bins (STFT; with no window, no detrend and hop = the row distance, a batch of R2C rows),
//   MODE 1  the density periodogram scale |X|^2, doubled except DC and Nyquist (spectrogram rows),
//   MODE 2  nothing per frame: lane group g sums the periodograms of frames g, g + G, g + 2G, ... in registers and
//           writes one partial row; k_spec_sum adds the G partial rows in order (Welch, bit-identical run to run).
//           Frames of 32768 samples run MODE 1 in chunks of rows instead, each chunk added in order.
//   MODE 3  R2C rows below 512 points: X[0] as the plain sum, as the separate pass forms it. The product with W^0 = 1 is
//           exact for finite values but makes NaN of an infinity; in the other modes and lengths the select costs 2-4 %.
// HBM traffic: the signal once per frame that covers it (twice at 50% overlap) and the output; no framed copy of
// the signal, no spectrum round trip.
#include "buffer.hpp"
#include "fft_core.hpp"
#include "kernels.hpp"
#include "spectral.hpp"

#include <algorithm>

namespace crdfft
{
using namespace dev;

namespace
{

constexpr int round_up(int v, int m) { return (v + m - 1) / m * m; }

template <int H, int E> struct SpecCfg
{
    static constexpr int T = H / E;
    static constexpr int M = T >= 256 ? 1 : 256 / T; // frames per workgroup
    static constexpr int threads = T * M;
    static constexpr int LF = lds_floats(H);
    static constexpr int RS = round_up(2 * LF, 64) + (T < 64 ? T : 0); // per-frame region (re then im)
    static constexpr int lds_floats_total = RS * M + threads;         // + the mean reduction
    static constexpr int lds_bytes = lds_floats_total * 4;
};

template <int H, int E, int MODE>
__global__ __launch_bounds__((SpecCfg<H, E>::threads)) void k_spec(SpecArgs a)
{
    using C = SpecCfg<H, E>;
    constexpr int T = C::T;
    extern __shared__ float lds[];
    const int tid = threadIdx.x;
    const int local = slot_of<T>(tid);
    const int i = tid - local * T;
    const LdsView<1> view{lds + local * C::RS, C::LF};
    float* red = lds + C::RS * C::M;
    const uint64_t group = static_cast<uint64_t>(blockIdx.x) * C::M + local;
    const uint64_t groups = static_cast<uint64_t>(gridDim.x) * C::M;
    // Welch accumulators (MODE 2 exists for H <= 8192: the largest core needs every register of its 1024 threads)
    static_assert(MODE != 2 || H <= kSpecWelchMaxH, "Welch lane groups up to H = 8192");
    float acc[E + 1];
#pragma unroll
    for (int m = 0; m <= E; ++m)
    {
        acc[m] = 0.0f;
    }
    // MODE 0/1/3: one frame per lane group; MODE 2: frames group, group + groups, ... (uniform trip count per
    // workgroup: every lane group runs the same number of iterations, idle ones on a masked frame)
    const uint64_t iters = MODE == 2 ? (a.frames + groups - 1) / groups : 1;
    // 8-byte sample pairs when every frame starts 8-byte aligned (an even hop from an 8-byte aligned signal)
    const bool pairs = (reinterpret_cast<uintptr_t>(a.x) & 7u) == 0 && (a.hop & 1u) == 0;
#pragma unroll 1
    for (uint64_t it = 0; it < iters; ++it)
    {
        const uint64_t f = group + it * groups;
        const bool active = f < a.frames;
        // the tables are the same for every frame; an empty asm hides that from the frame loop, so the compiler reloads them
        // per frame (L1/L2 hits) instead of holding every butterfly's twiddles in registers across the frame loop
        const cf* tw = reinterpret_cast<const cf*>(a.tw);
        const cf* wk = reinterpret_cast<const cf*>(a.wtab);
        const float* win = a.window;
        if constexpr (MODE == 2)
        {
            asm volatile("" : "+s"(tw), "+s"(wk), "+s"(win));
        }
        // From 64 threads a frame on a buffer resource: an inactive frame gets no records, so its loads read zeros and touch no
        // memory. Below, plain loads: an inactive slot reads the first frame's samples. Its results go nowhere either way
        // (`active` at every store and accumulation).
        const Row<(T >= 64)> xr(a.x + (active ? f * a.hop : 0), active ? 8u * H : 0u);
        cf v[E];
        if (pairs)
        {
#pragma unroll
            for (int m = 0; m < E; ++m)
            {
                v[m] = xr.ld64(8u * static_cast<uint32_t>(i), 8u * T * m);
            }
        }
        else
        {
#pragma unroll
            for (int m = 0; m < E; ++m)
            {
                const uint32_t j = 8u * static_cast<uint32_t>(i);
                v[m] = cf{xr.ld32(j, 8u * T * m), xr.ld32(j + 4u, 8u * T * m)};
            }
        }
        if (MODE != 3 && a.detrend != 0)
        {
            // the frame mean, in a fixed order: a butterfly over the frame's lanes of one wave (each step adds the
            // same two partial sums in both lanes, so every lane ends with the same bits), then the waves' sums in
            // wave order through LDS
            float part = 0.0f;
#pragma unroll
            for (int m = 0; m < E; ++m)
            {
                part += v[m].x + v[m].y;
            }
            constexpr int W = T < 64 ? T : 64;
#pragma unroll
            for (int o = W / 2; o > 0; o >>= 1)
            {
                part += __shfl_xor(part, o, 64);
            }
            if constexpr (T > 64)
            {
                if ((tid & 63) == 0)
                {
                    red[tid >> 6] = part;
                }
                __syncthreads();
                const int w0 = (local * T) >> 6;
                part = 0.0f;
#pragma unroll
                for (int w = 0; w < T / 64; ++w)
                {
                    part += red[w0 + w];
                }
                __syncthreads();
            }
            const float mean = part / static_cast<float>(2 * H);
#pragma unroll
            for (int m = 0; m < E; ++m)
            {
                v[m].x -= mean;
                v[m].y -= mean;
            }
        }
        if (MODE != 3 && a.window != nullptr)
        {
            const __amdgpu_buffer_rsrc_t wr = make_rsrc(win, 8u * H);
#pragma unroll
            for (int m = 0; m < E; ++m)
            {
                const cf wv = bld<0>(wr, 8u * static_cast<uint32_t>(i + T * m), 0);
                v[m].x *= wv.x;
                v[m].y *= wv.y;
            }
        }
        fft_core<H, E, false, 1>(v, i, view, tw);
        // Z through LDS for the recombine (fft_core's last LDS read is behind a barrier; with H == E it used none)
        __syncthreads();
#pragma unroll
        for (int m = 0; m < E; ++m)
        {
            view.put_at(pad16(i), T * m, v[m]);
        }
        __syncthreads();
        // recombine and epilogue per slot (nothing but the accumulators outlives the frame)
        const uint64_t row = f * a.ostride;
#pragma unroll
        for (int m = 0; m < E; ++m)
        {
            const int k = i + T * m;
            const cf zk = v[m];
            // element H - k = (T - i) + T (E - 1 - m): pads apart, as T - i carries into no higher part for i > 0; slot 0 is
            // its own mirror
            const cf zh = m == 0 ? view.get(k == 0 ? 0 : H - k)
                                 : (T >= 16 ? view.get_at(pad16(T - i), T * (E - 1 - m)) : view.get(H - k));
            const cf e = {(zk.x + zh.x) * 0.5f, (zk.y - zh.y) * 0.5f};
            const cf o = {(zk.y + zh.y) * 0.5f, (zh.x - zk.x) * 0.5f};
            const cf xk = MODE == 3 && m == 0 && k == 0 ? cf{zk.x + zk.y, 0.0f} : cadd(e, cmul(o, wk[k]));
            // k == 0 also yields the Nyquist bin: W_N^H = -1, X[H] = Re Z0 - Im Z0 (read only where k == 0)
            const cf xn = {zk.x - zk.y, 0.0f};
            if constexpr (MODE == 0 || MODE == 3)
            {
                if (active)
                {
                    cf* out = reinterpret_cast<cf*>(a.out) + row;
                    out[k] = xk;
                    if (m == 0 && k == 0)
                    {
                        out[H] = xn;
                    }
                }
            }
            else
            {
                const float p = a.scale * (xk.x * xk.x + xk.y * xk.y) * (m == 0 && k == 0 ? 1.0f : 2.0f);
                const float pn = a.scale * (xn.x * xn.x);
                if constexpr (MODE == 1)
                {
                    if (active)
                    {
                        float* out = reinterpret_cast<float*>(a.out) + row;
                        out[k] = p;
                        if (m == 0 && k == 0)
                        {
                            out[H] = pn;
                        }
                    }
                }
                else
                {
                    acc[m] += active ? p : 0.0f;
                    if (m == 0 && k == 0)
                    {
                        acc[E] += active ? pn : 0.0f;
                    }
                }
            }
        }
        __syncthreads(); // LDS free for the next frame
    }
    if constexpr (MODE == 2)
    {
        // one partial row per lane group
        float* prow = reinterpret_cast<float*>(a.out) + group * static_cast<uint64_t>(H + 1);
#pragma unroll
        for (int m = 0; m < E; ++m)
        {
            prow[i + T * m] = acc[m];
        }
        if (i == 0)
        {
            prow[H] = acc[E];
        }
    }
}

// k_welch<N, E>: the Welch sum over pairs of frames. Frames 2 p and 2 p + 1 are the real and imaginary parts of one
// N-point transform Z, and |A[k]|^2 + |B[k]|^2 = (|Z[k]|^2 + |Z[N-k]|^2) / 2, so nothing has to be told apart per
// frame: a lane group of T = N/E threads adds |Z[k]|^2 of its pairs g, g + G, ... to its E slots, folds k onto
// N - k through LDS once at the end and the workgroup writes one partial row of N/2 + 1 densities. Per frame that is half an N-point
// transform (12 levels of 4096 points for two frames) in place of a half-length one, a recombine and its LDS exchange.
// Measured, 2^26 samples at 50 % overlap: N = 4096 257 -> 163 us, 1024 200 -> 111, 256 298 -> 90, 64 683 -> 88 (floor by bytes
// 44). What bounds it at N = 4096, E = 16, by counters: the vector unit issues 56 % of the time, LDS is busy 32 % (9 % in bank
// conflicts), and of the 3.3 waves a SIMD holds (LDS allows four) each spends a third of its time at waits and barriers and
// another 43 % waiting to issue. Loading the next pair ahead (32 more registers) measured no better, nor did
// reloading the twiddles per pair instead of keeping them.
template <int N, int E> struct WelchCfg
{
    static constexpr int T = N / E;
    static constexpr int M = T >= 256 ? 1 : 256 / T; // pairs per workgroup
    static constexpr int threads = T * M;
    static constexpr int LF = lds_floats(N);
    static constexpr int RS = round_up(2 * LF, 64) + (T < 64 ? T : 0); // per-pair region (re then im)
    static constexpr int lds_bytes = (RS * M + 2 * threads / 64 + 2) * 4;
};

template <int N, int E>
__global__ __launch_bounds__((WelchCfg<N, E>::threads)) void k_welch(SpecArgs a)
{
    using C = WelchCfg<N, E>;
    constexpr int T = C::T;
    extern __shared__ float lds[];
    const int tid = threadIdx.x;
    const int local = slot_of<T>(tid);
    const int i = tid - local * T;
    const LdsView<1> view{lds + local * C::RS, C::LF};
    float* red = lds + C::RS * C::M;
    const uint64_t group = static_cast<uint64_t>(blockIdx.x) * C::M + local;
    const uint64_t groups = static_cast<uint64_t>(gridDim.x) * C::M;
    const uint64_t pairs = (a.frames + 1) / 2;
    const uint64_t iters = (pairs + groups - 1) / groups; // the same for every lane group: idle ones read no records
    float acc[E];
#pragma unroll
    for (int m = 0; m < E; ++m)
    {
        acc[m] = 0.0f;
    }
    const __amdgpu_buffer_rsrc_t wr = make_rsrc(a.window, a.window != nullptr ? 4u * N : 0u);
    const uint32_t o4 = 4u * static_cast<uint32_t>(i);
    auto load = [&](cf (&d)[E], uint64_t it) {
        const uint64_t f = 2 * (group + it * groups);
        const bool one = f < a.frames, two = f + 1 < a.frames;
        const Row<(T >= 64)> ra(a.x + (one ? f * a.hop : 0), one ? 4u * N : 0u);
        const Row<(T >= 64)> rb(a.x + (two ? (f + 1) * a.hop : 0), two ? 4u * N : 0u);
#pragma unroll
        for (int m = 0; m < E; ++m)
        {
            d[m] = cf{ra.ld32(o4, 4u * T * m), rb.ld32(o4, 4u * T * m)};
            if constexpr (T < 64)
            {
                d[m] = cf{one ? d[m].x : 0.0f, two ? d[m].y : 0.0f};
            }
        }
    };
    float win[E];
#pragma unroll
    for (int m = 0; m < E; ++m)
    {
        win[m] = (a.window != nullptr ? bld32<0>(wr, o4, 4u * T * m) : 1.0f) * a.scale; // a power of two
    }
#pragma unroll 1
    for (uint64_t it = 0; it < iters; ++it)
    {
        cf v[E];
        load(v, it);
        if (a.detrend != 0)
        {
            // both means in a fixed order: lane butterflies within a wave, then the waves' sums in wave order
            cf part = {0.0f, 0.0f};
#pragma unroll
            for (int m = 0; m < E; ++m)
            {
                part = cadd(part, v[m]);
            }
            constexpr int W = T < 64 ? T : 64;
#pragma unroll
            for (int o = W / 2; o > 0; o >>= 1)
            {
                part.x += __shfl_xor(part.x, o, 64);
                part.y += __shfl_xor(part.y, o, 64);
            }
            if constexpr (T > 64)
            {
                cf* const sums = reinterpret_cast<cf*>(red);
                if ((tid & 63) == 0)
                {
                    sums[tid >> 6] = part;
                }
                __syncthreads();
                part = cf{0.0f, 0.0f};
#pragma unroll
                for (int w = 0; w < T / 64; ++w)
                {
                    part = cadd(part, sums[((local * T) >> 6) + w]);
                }
            }
            const cf mean = {part.x / static_cast<float>(N), part.y / static_cast<float>(N)};
#pragma unroll
            for (int m = 0; m < E; ++m)
            {
                v[m] = csub(v[m], mean);
            }
        }
        if (a.window != nullptr || a.scale != 1.0f)
        {
#pragma unroll
            for (int m = 0; m < E; ++m)
            {
                v[m].x *= win[m];
                v[m].y *= win[m];
            }
        }
        fft_core<N, E, false, 1>(v, i, view, reinterpret_cast<const cf*>(a.tw));
        // an idle lane group or half of a pair: the samples are zeros, less a mean of zero
#pragma unroll
        for (int m = 0; m < E; ++m)
        {
            acc[m] += v[m].x * v[m].x + v[m].y * v[m].y;
        }
    }
    // the lane groups' sums in group order, k folded onto N - k: P[k] = S[k] + S[N - k] (the one-sided doubling of the
    // halves), P[0] and P[N/2] alone; one partial row per workgroup
    __syncthreads();
#pragma unroll
    for (int m = 0; m < E; ++m)
    {
        lds[local * N + i + T * m] = acc[m];
    }
    __syncthreads();
    float* prow = reinterpret_cast<float*>(a.out) + static_cast<uint64_t>(blockIdx.x) * (N / 2 + 1);
    for (int k = tid; k <= N / 2; k += C::threads)
    {
        float p = 0.0f;
#pragma unroll 4
        for (int g = 0; g < C::M; ++g)
        {
            p += lds[g * N + k] + (k == 0 || k == N / 2 ? 0.0f : lds[g * N + N - k]);
        }
        prow[k] = p;
    }
}

// acc[k] = ((first ? 0 : acc[k]) + sum over the rows of rows[r][k]) * scale, in a fixed order: a workgroup owns 64
// bins, its 16 row groups sum rows g, g + 16, ... (AHEAD loads in flight per step), and the 16 partial sums are added
// in group order, so the result does not depend on timing. The sums carry their rounding errors along, so thousands of
// rows add none of their own.
constexpr int kSumBins = 64;
constexpr int kSumGroups = 16;

// s += x, the rounding error collected in c (Knuth's two-sum)
__device__ __forceinline__ void add_compensated(float& s, float& c, float x)
{
    const float t = s + x;
    const float b = t - s;
    c += (s - (t - b)) + (x - b);
    s = t;
}

template <int AHEAD>
__global__ __launch_bounds__(kSumBins * kSumGroups) void k_spec_sum(const float* rows, float* acc, uint32_t nfreq,
                                                                    uint32_t nrows, int first, float scale, float scale_lo)
{
    __shared__ float part[kSumGroups][kSumBins], rest[kSumGroups][kSumBins];
    const int kk = threadIdx.x % kSumBins;
    const int g = threadIdx.x / kSumBins;
    const uint32_t k = blockIdx.x * kSumBins + kk;
    float s = 0.0f, c = 0.0f;
    if (k < nfreq)
    {
        // one 32-bit offset a load and no checks: a row past the last one reads zero
        const __amdgpu_buffer_rsrc_t in = make_rsrc(rows, nrows * nfreq * 4u);
        const uint32_t step = kSumGroups * nfreq * 4u;
        uint32_t off = (g * nfreq + k) * 4u;
        for (uint32_t r = 0; r < nrows; r += AHEAD * kSumGroups)
        {
            float x[AHEAD];
#pragma unroll
            for (int q = 0; q < AHEAD; ++q)
            {
                x[q] = bld32<0>(in, off + q * step, 0);
            }
            __builtin_amdgcn_sched_barrier(0); // all on their way before the first one is waited for
#pragma unroll
            for (int q = 0; q < AHEAD; ++q)
            {
                add_compensated(s, c, x[q]);
            }
            off += AHEAD * step;
        }
    }
    part[g][kk] = s;
    rest[g][kk] = c;
    __syncthreads();
    if (g == 0 && k < nfreq)
    {
        s = first != 0 ? 0.0f : acc[k];
        c = 0.0f;
        for (int q = 0; q < kSumGroups; ++q)
        {
            add_compensated(s, c, part[q][kk]);
            c += rest[q][kk];
        }
        // (s + c) (scale + scale_lo) rounded once; a sum that has left the range of the type has no rest (inf - inf)
        const float plain = (c - c == 0.0f ? s + c : s) * scale;
        acc[k] = plain - plain == 0.0f ? __fmaf_rn(s, scale, __fmaf_rn(c, scale, s * scale_lo)) : plain;
    }
}

// (H, E): the per-length values per thread of the real-transform cores (the same choice as the DCT kernels', whose
// load / core / recombine structure this kernel shares)
#define CRDFFT_SPEC_LIST(X)                                                                                            \
    X(2, 2) X(4, 4) X(8, 8) X(16, 4) X(32, 4) X(64, 4) X(128, 4) X(256, 4) X(512, 8) X(1024, 8) X(2048, 8) X(4096, 8)  \
        X(8192, 8) X(16384, 16)

// (N, E) of the pair kernel: the fastest per length over a 2^26-sample signal at 50 % overlap (us at E = 8 / 16 / 32; 4
// values per thread were slower still): 64 87 / - / -, 128 108 / 107 / -, 256 116 / 97 / -, 512 114 / 131 / 106,
// 1024 151 / 158 / 112, 2048 155 / 161 / 153, 4096 170 / 168 / 167, 8192 - / 226 / 198.
#define CRDFFT_WELCH_LIST(X)                                                                                           \
    X(8, 4) X(16, 8) X(32, 8) X(64, 8) X(128, 16) X(256, 16) X(512, 32) X(1024, 32) X(2048, 32) X(4096, 16) X(8192, 32)

template <typename K> hipError_t set_lds(K kernel, unsigned bytes)
{
    if (bytes > 64 * 1024)
    {
        return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   static_cast<int>(bytes));
    }
    return hipSuccess;
}

} // namespace

bool spec_shape(uint64_t h, int* e, unsigned* frames_per_group)
{
#define X(H, E)                                                                                                        \
    if (h == H)                                                                                                        \
    {                                                                                                                  \
        *e = E;                                                                                                        \
        *frames_per_group = SpecCfg<H, E>::M;                                                                          \
        return true;                                                                                                   \
    }
    CRDFFT_SPEC_LIST(X)
#undef X
    return false;
}

hipError_t launch_spec(uint64_t h, int mode, const SpecArgs& a, uint64_t groups, hipStream_t s)
{
#define X(H, E)                                                                                                        \
    if (h == H)                                                                                                        \
    {                                                                                                                  \
        using C = SpecCfg<H, E>;                                                                                       \
        if (mode == 2 && H > kSpecWelchMaxH)                                                                           \
            return hipErrorInvalidValue;                                                                               \
        auto kern = mode == 3 && H < 256 ? k_spec<H, E, (H < 256 ? 3 : 0)>                                             \
                    : mode == 0 || mode == 3 ? k_spec<H, E, 0>                                                         \
                              : (mode == 1 ? k_spec<H, E, 1> : k_spec<H, E, (H <= kSpecWelchMaxH ? 2 : 1)>);        \
        hipError_t err = set_lds(kern, C::lds_bytes);                                                                  \
        if (err != hipSuccess)                                                                                         \
            return err;                                                                                                \
        if (groups == 0 || groups > 0xFFFFFFFFull)                                                                     \
            return hipErrorInvalidValue;                                                                               \
        hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(groups)), dim3(C::threads), C::lds_bytes, s, a);        \
        return hipGetLastError();                                                                                      \
    }
    CRDFFT_SPEC_LIST(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t spec_welch_residency(uint64_t h, int* per_cu)
{
#define X(H, E)                                                                                                        \
    if (h == H)                                                                                                        \
    {                                                                                                                  \
        using C = SpecCfg<H, E>;                                                                                       \
        if (H > kSpecWelchMaxH)                                                                                        \
            return hipErrorInvalidValue;                                                                               \
        auto kern = k_spec<H, E, (H <= kSpecWelchMaxH ? 2 : 1)>;                                                       \
        hipError_t err = set_lds(kern, C::lds_bytes);                                                                  \
        if (err != hipSuccess)                                                                                         \
            return err;                                                                                                \
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, kern, C::threads, C::lds_bytes);                   \
    }
    CRDFFT_SPEC_LIST(X)
#undef X
    return hipErrorInvalidValue;
}

bool welch_pair_shape(uint64_t n, int* e, unsigned* pairs_per_group)
{
#define X(N, E)                                                                                                        \
    if (n == N)                                                                                                        \
    {                                                                                                                  \
        *e = E;                                                                                                        \
        *pairs_per_group = WelchCfg<N, E>::M;                                                                          \
        return true;                                                                                                   \
    }
    CRDFFT_WELCH_LIST(X)
#undef X
    return false;
}

hipError_t launch_welch_pairs(uint64_t n, const SpecArgs& a, uint64_t groups, hipStream_t s)
{
#define X(N, E)                                                                                                        \
    if (n == N)                                                                                                        \
    {                                                                                                                  \
        using C = WelchCfg<N, E>;                                                                                      \
        hipError_t err = set_lds(k_welch<N, E>, C::lds_bytes);                                                         \
        if (err != hipSuccess)                                                                                         \
            return err;                                                                                                \
        if (groups == 0 || groups > 0xFFFFFFFFull)                                                                     \
            return hipErrorInvalidValue;                                                                               \
        hipLaunchKernelGGL((k_welch<N, E>), dim3(static_cast<unsigned>(groups)), dim3(C::threads), C::lds_bytes, s, a); \
        return hipGetLastError();                                                                                      \
    }
    CRDFFT_WELCH_LIST(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t welch_pair_residency(uint64_t n, int* per_cu)
{
#define X(N, E)                                                                                                        \
    if (n == N)                                                                                                        \
    {                                                                                                                  \
        using C = WelchCfg<N, E>;                                                                                      \
        const hipError_t err = set_lds(k_welch<N, E>, C::lds_bytes);                                                   \
        if (err != hipSuccess)                                                                                         \
            return err;                                                                                                \
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, k_welch<N, E>, C::threads, C::lds_bytes);          \
    }
    CRDFFT_WELCH_LIST(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t launch_spec_sum(const float* rows, float* acc, uint64_t nfreq, uint64_t nrows, bool first, float scale,
                           hipStream_t s, float scale_lo)
{
    // the last step's offsets as well are 32 bits wide
    if ((nrows + 2 * 8 * kSumGroups) * nfreq >= (uint64_t{1} << 30))
    {
        return hipErrorInvalidValue;
    }
    // Eight rows ahead where the few workgroups wait for memory (Welch us of 8 / 4 rows ahead: nperseg 4, 4096 frames
    // 18.2 / 27.0, 1024, 1000 frames 11.5 / 14.2); four where one step of them covers the rows or the bins fill the chip
    // (16, 1024 frames 10.1 / 9.9; 32768, 4096 frames 505 / 497).
    const unsigned blocks = static_cast<unsigned>((nfreq + kSumBins - 1) / kSumBins);
    auto kern = nrows > 4 * kSumGroups && blocks < 256 ? k_spec_sum<8> : k_spec_sum<4>;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(kSumBins * kSumGroups), 0, s, rows, acc, static_cast<uint32_t>(nfreq),
                       static_cast<uint32_t>(nrows), first ? 1 : 0, scale, scale_lo);
    return hipGetLastError();
}

} // namespace crdfft
