// The spectral front end's C-ABI (crdfft_spectral_*, crdfft_stft, crdfft_spectrogram, crdfft_welch): the GPU form of
// the reference's hesap-dsp stft / spectrogram / welch_psd / periodogram (engine/numerics/hesap-dsp/include/crd/
// hesap/dsp/spectral.hpp:43-222, :334-386) over its RealFftPlan, each one fused launch (spectral_kernels.hip).
#include <algorithm>
#include <cmath>
#include <new>
#include <vector>

#include <hip/hip_runtime.h>

#include "../../include/crdfft.h"
#include "kernels.hpp"
#include "planner.hpp"
#include "scratch.hpp"
#include "real.hpp"
#include "spectral.hpp"

namespace
{

// Welch: the lane-group kernel runs one resident round (CUs x workgroups per CU, at most this many workgroups); the
// grid is fixed per device and frame count, so the PSD is bit-identical run to run. The chunked path for the
// largest frames writes this many rows per chunk.
constexpr uint64_t kWelchWorkgroups = 2048;

crdfft_status st_of(hipError_t e)
{
    if (e == hipSuccess)
    {
        return CRDFFT_OK;
    }
    return e == hipErrorOutOfMemory ? CRDFFT_OUT_OF_MEMORY : CRDFFT_HIP_ERROR;
}

#define SPEC_TRY(expr)                                                                                                 \
    do                                                                                                                 \
    {                                                                                                                  \
        const hipError_t spec_e_ = (expr);                                                                             \
        if (spec_e_ != hipSuccess)                                                                                     \
            return st_of(spec_e_);                                                                                     \
    } while (0)

} // namespace

struct crdfft_spectral_plan_s
{
    uint64_t nperseg = 0, noverlap = 0, hop = 0, h = 0;
    uint64_t welch_wgs = 0; // the resident round of the Welch kernel
    int32_t window = CRDFFT_WINDOW_HANN;
    uint32_t flags = 0;
    int e = 0;
    unsigned fpg = 1; // frames per workgroup
    // Welch over pairs of frames: workgroups of one resident round (0: frames one by one), pairs per workgroup
    uint64_t pair_wgs = 0;
    unsigned ppg = 1;
    double pair_gain = 1.0; // mean gain of the pairs' transform
    crdfft::DeviceBuffer pair_tw;
    double winsum2 = 0.0;
    crdfft::DeviceBuffer win, wtab, tw, partial;
    crdfft::PerStream partial_of;
};

namespace
{

// The mean gain over all paths of a register DFT of r values (dft.hpp: 8 = 2 x 4, 16 = 4 x 4, 32 = 8 x 4): a path through
// W_r^e is shortened by what rounding its two parts takes off its length, a signed 0.7e-8 .. 3e-8 that adds up over stages.
double dft_gain(int r)
{
    if (r < 8)
    {
        return 1.0;
    }
    const int r1 = r / 4;
    double sum = 0.0;
    for (int n2 = 0; n2 < 4; ++n2)
    {
        for (int k1 = 0; k1 < r1; ++k1)
        {
            const double a = 2.0 * M_PI * n2 * k1 / r;
            const double c = std::cos(a), s = std::sin(a);
            sum += static_cast<double>(static_cast<float>(c)) * c + static_cast<double>(static_cast<float>(s)) * s;
        }
    }
    return dft_gain(r1) * sum / r;
}

// The same for fft_core of n points at e values per thread: a first stage of n's remainder, then stages of e.
double core_gain(uint64_t n, int e)
{
    double g = 1.0;
    for (; n > 1 && n % static_cast<uint64_t>(e) == 0; n /= static_cast<uint64_t>(e))
    {
        g *= dft_gain(e);
    }
    return g * dft_gain(static_cast<int>(n));
}

uint64_t frames_of(const crdfft_spectral_plan_s* p, uint64_t len)
{
    return len < p->nperseg ? 0 : (len - p->noverlap) / p->hop;
}

crdfft_status run(crdfft_spectral_plan p, const float* x, uint64_t len, int mode, double fs, void* out, void* stream)
{
    if (p == nullptr || x == nullptr || out == nullptr || (mode != 0 && !(fs > 0.0)))
    {
        return CRDFFT_INVALID_ARGUMENT;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const uint64_t frames = frames_of(p, len);
    const uint64_t nfreq = p->h + 1;
    crdfft::SpecArgs a{x,
                       p->window == CRDFFT_WINDOW_HANN ? p->win.as<float>() : nullptr,
                       p->wtab.as<crdfft::cfloat>(),
                       p->tw.as<crdfft::cfloat>(),
                       out,
                       frames,
                       p->hop,
                       mode == 0 ? 1.0f : static_cast<float>(1.0 / (fs * p->winsum2)),
                       (p->flags & CRDFFT_SPECTRAL_DETREND) != 0 ? 1 : 0,
                       nfreq};
    if (mode != 2)
    {
        if (frames == 0)
        {
            return CRDFFT_OK;
        }
        SPEC_TRY(crdfft::launch_spec(p->h, mode, a, (frames + p->fpg - 1) / p->fpg, s));
        return CRDFFT_OK;
    }
    float* psd = static_cast<float*>(out);
    if (frames == 0)
    {
        SPEC_TRY(crdfft::launch_fill_bytes(psd, 0, nfreq * sizeof(float), s)); // a kernel: safe in a captured graph
        return CRDFFT_OK;
    }
    float* partial = static_cast<float*>(p->partial_of.get(p->partial, s));
    if (partial == nullptr)
    {
        return CRDFFT_OUT_OF_MEMORY;
    }
    const float inv = static_cast<float>(1.0 / static_cast<double>(frames));
    // pairs of frames leave half as many lane groups to fill the chip: measured us of pairs / single frames at 50 % overlap,
    // nperseg 64: 256 frames 7.8 / 6.7, 512 6.8 / 8.0, 32768 8.9 / 172; 1024: 512 11.5 / 10.0, 1024 11.5 / 13.5, 32768
    // 37 / 78; 4096: 512 15.3 / 13.1, 1024 16.8 / 20.9, 32768 168 / 225. 8192: 768 24.4 / 23.9; one frame more than a round of
    // lane groups (768 on 256 CUs) takes single frames a second round, 777 25.2 / 33.1, 1000 25.4 / 32.3
    const uint64_t pairs_from = p->nperseg <= 256 ? 512 : p->nperseg <= 4096 ? 1024 : std::min<uint64_t>(p->welch_wgs + 1, 1024);
    if (p->pair_wgs > 0 && frames >= pairs_from)
    {
        const uint64_t pairs = (frames + 1) / 2;
        const uint64_t wgs = std::min<uint64_t>((pairs + p->ppg - 1) / p->ppg, p->pair_wgs);
        a.out = partial;
        a.tw = p->pair_tw.as<crdfft::cfloat>();
        // The window carries a power of two whose square is at most 1 / (fs sum w^2), exactly, and the row sum is scaled by the
        // rest over the frame count in two parts: rounded scales would be one error common to all bins. A bin of a pair can
        // be |A| + |B|, so its square unscaled would leave the range at half the amplitude of a single frame's; scaled it is
        // at most twice the scaled squares of A and B, which the sum adds up in any case (from a scale of 1 on as it is).
        const double scale = 1.0 / (fs * p->winsum2);
        double fold = 1.0;
        if (scale < 1.0)
        {
            fold = std::exp2(std::max(std::floor(0.5 * std::log2(scale)), -60.0));
        }
        a.scale = static_cast<float>(fold);
        // The radix-16 and radix-32 butterflies of the pairs lose more of a tone's power to their rounded constants than the
        // radix-8 ones of single frames, in every frame alike (nperseg 4096 6.9e-8, 8192 8.1e-8; single 2.6e-8, 3.4e-8): the
        // scale gives the mean back. Rel-L2 error against FP64, mean over 120 random tone pairs in noise, without / with it /
        // single frames: 4096 1.10e-7 / 4.6e-8 / 8.1e-8, 8192 1.16e-7 / 5.0e-8 / 8.2e-8, 256..2048 5.5-8.3e-8 / 3.2-3.7e-8 /
        // 6.7-7.6e-8.
        const double rest = scale / (fold * fold) / (p->pair_gain * p->pair_gain) / static_cast<double>(frames);
        const float rest_hi = static_cast<float>(rest);
        const float rest_lo = std::isfinite(rest_hi) ? static_cast<float>(rest - static_cast<double>(rest_hi)) : 0.0f;
        SPEC_TRY(crdfft::launch_welch_pairs(p->nperseg, a, wgs, s));
        SPEC_TRY(crdfft::launch_spec_sum(partial, psd, nfreq, wgs, true, rest_hi, s, rest_lo));
        return CRDFFT_OK;
    }
    if (p->h <= static_cast<uint64_t>(crdfft::kSpecWelchMaxH))
    {
        const uint64_t wgs = std::min<uint64_t>((frames + p->fpg - 1) / p->fpg, p->welch_wgs);
        a.out = partial;
        SPEC_TRY(crdfft::launch_spec(p->h, 2, a, wgs, s));
        SPEC_TRY(crdfft::launch_spec_sum(partial, psd, nfreq, wgs * p->fpg, true, inv, s));
        return CRDFFT_OK;
    }
    // the largest frames: density rows for chunks of frames into the scratch, each chunk added in order
    const uint64_t chunk = kWelchWorkgroups * p->fpg;
    for (uint64_t f0 = 0; f0 < frames; f0 += chunk)
    {
        const uint64_t cnt = std::min(chunk, frames - f0);
        crdfft::SpecArgs c = a;
        c.x = x + f0 * p->hop;
        c.frames = cnt;
        c.out = partial;
        SPEC_TRY(crdfft::launch_spec(p->h, 1, c, (cnt + p->fpg - 1) / p->fpg, s));
        SPEC_TRY(crdfft::launch_spec_sum(partial, psd, nfreq, cnt, f0 == 0, f0 + cnt == frames ? inv : 1.0f, s));
    }
    return CRDFFT_OK;
}

} // namespace

extern "C" {

crdfft_status crdfft_spectral_plan_create(crdfft_spectral_plan* plan, uint64_t nperseg, uint64_t noverlap,
                                          int32_t window, uint32_t flags)
{
    if (plan == nullptr || (window != CRDFFT_WINDOW_BOXCAR && window != CRDFFT_WINDOW_HANN) ||
        (flags & ~CRDFFT_SPECTRAL_DETREND) != 0)
    {
        return CRDFFT_INVALID_ARGUMENT;
    }
    *plan = nullptr;
    if (nperseg < 4 || (nperseg & (nperseg - 1)) != 0 || noverlap >= nperseg)
    {
        return CRDFFT_INVALID_SIZE; // a RealFftPlan: a power of two >= 4 (real_fft.hpp:24)
    }
    int e = 0;
    unsigned fpg = 0;
    if (!crdfft::spec_shape(nperseg / 2, &e, &fpg))
    {
        return CRDFFT_UNSUPPORTED;
    }
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
    {
        return CRDFFT_NO_DEVICE;
    }
    auto* p = new (std::nothrow) crdfft_spectral_plan_s;
    if (p == nullptr)
    {
        return CRDFFT_OUT_OF_MEMORY;
    }
    p->nperseg = nperseg;
    p->noverlap = noverlap;
    p->hop = nperseg - noverlap;
    p->h = nperseg / 2;
    p->window = window;
    p->flags = flags;
    p->e = e;
    p->fpg = fpg;
    // periodic hann (windows.hpp:63-124, sym = false): 0.5 + 0.5 cos(-pi + 2 pi i / nperseg), from FP64
    std::vector<float> w(nperseg, 1.0f);
    if (window == CRDFFT_WINDOW_HANN)
    {
        for (uint64_t i = 0; i < nperseg; ++i)
        {
            const double fac = -M_PI + 2.0 * M_PI * static_cast<double>(i) / static_cast<double>(nperseg);
            w[i] = static_cast<float>(0.5 + 0.5 * std::cos(fac));
        }
    }
    for (float v : w)
    {
        p->winsum2 += static_cast<double>(v) * static_cast<double>(v);
    }
    if (p->h <= static_cast<uint64_t>(crdfft::kSpecWelchMaxH))
    {
        int dev = 0, cus = 0, per_cu = 0;
        hipError_t re = hipGetDevice(&dev);
        if (re == hipSuccess)
            re = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        if (re == hipSuccess)
            re = crdfft::spec_welch_residency(p->h, &per_cu);
        if (re != hipSuccess)
        {
            delete p;
            return st_of(re);
        }
        p->welch_wgs = std::max<uint64_t>(1, std::min<uint64_t>(static_cast<uint64_t>(cus) * std::max(per_cu, 1),
                                                                kWelchWorkgroups));
    }
    int pair_e = 0;
    if (crdfft::welch_pair_shape(nperseg, &pair_e, &p->ppg))
    {
        int dev = 0, cus = 0, per_cu = 0;
        hipError_t re = hipGetDevice(&dev);
        if (re == hipSuccess)
            re = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        if (re == hipSuccess)
            re = crdfft::welch_pair_residency(nperseg, &per_cu);
        if (re != hipSuccess)
        {
            delete p;
            return st_of(re);
        }
        p->pair_wgs = std::min<uint64_t>(static_cast<uint64_t>(cus) * std::max(per_cu, 1), kWelchWorkgroups);
        p->pair_gain = core_gain(nperseg, pair_e);
    }
    const uint64_t entries = crdfft::stage_twiddle_entries(p->h, e);
    hipError_t err = p->win.alloc(nperseg * sizeof(float));
    if (err == hipSuccess)
        err = hipMemcpy(p->win.ptr, w.data(), nperseg * sizeof(float), hipMemcpyHostToDevice);
    if (err == hipSuccess)
        err = p->wtab.alloc((p->h + 1) * sizeof(crdfft::cfloat));
    if (err == hipSuccess)
        err = crdfft::build_roots(p->wtab.as<crdfft::cfloat>(), p->h + 1, 1, nperseg, nullptr);
    if (err == hipSuccess)
        err = p->tw.alloc(std::max<uint64_t>(entries, 1) * sizeof(crdfft::cfloat));
    if (err == hipSuccess && entries > 0)
        err = crdfft::build_stage_twiddles(p->tw.as<crdfft::cfloat>(), p->h, e, nullptr);
    if (err == hipSuccess && p->pair_wgs > 0)
    {
        const uint64_t pair_entries = crdfft::stage_twiddle_entries(nperseg, pair_e);
        err = p->pair_tw.alloc(std::max<uint64_t>(pair_entries, 1) * sizeof(crdfft::cfloat));
        if (err == hipSuccess && pair_entries > 0)
            err = crdfft::build_stage_twiddles(p->pair_tw.as<crdfft::cfloat>(), nperseg, pair_e, nullptr);
    }
    if (err == hipSuccess)
        err = p->partial.alloc(kWelchWorkgroups * fpg * (p->h + 1) * sizeof(float));
    if (err == hipSuccess)
        err = hipStreamSynchronize(nullptr);
    if (err != hipSuccess)
    {
        delete p;
        return st_of(err);
    }
    *plan = p;
    return CRDFFT_OK;
}

crdfft_status crdfft_spectral_plan_destroy(crdfft_spectral_plan plan)
{
    if (plan == nullptr)
    {
        return CRDFFT_INVALID_ARGUMENT;
    }
    delete plan;
    return CRDFFT_OK;
}

uint64_t crdfft_spectral_frames(crdfft_spectral_plan plan, uint64_t len)
{
    return plan == nullptr ? 0 : frames_of(plan, len);
}

crdfft_status crdfft_stft(crdfft_spectral_plan plan, const float* x, uint64_t len, void* out, void* stream)
{
    return run(plan, x, len, 0, 0.0, out, stream);
}

crdfft_status crdfft_spectrogram(crdfft_spectral_plan plan, const float* x, uint64_t len, double fs, float* out,
                                 void* stream)
{
    return run(plan, x, len, 1, fs, out, stream);
}

crdfft_status crdfft_welch(crdfft_spectral_plan plan, const float* x, uint64_t len, double fs, float* psd,
                           void* stream)
{
    return run(plan, x, len, 2, fs, psd, stream);
}

} // extern "C"
