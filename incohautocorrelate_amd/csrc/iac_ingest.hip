// iac_ingest.hip -- the averaged-intensity pass over a stack of dense frames
// (Detector::LoadAndAverageIntensity, IAC/Detector.cpp:687-790) on gfx950, with
// the reference's float arithmetic: pixel mask multiply, threshold or photon
// discretisation, per-pixel accumulation over frames in frame order, the
// 1/N scale, and the per-event MeanIntensity / PhotonCount sums.
#include <algorithm>
#include <cmath>

#include "iac_fpexact.h"
#include "iac_internal.h"
#include "iac_serial_sum.h"

#pragma clang fp contract(off)

namespace {

// ArrayOperators::DiscretizeToPhotons, IAC/ArrayOperators.h:138-148
__device__ __forceinline__ float discretize(float I, float T, float S) { return ceilf((I - T) / S) * (float)(I >= T); }

// The per-frame value tmpIntensity[j] after masking and the branch of
// Detector.cpp:718-760 (the value the event sums see).
__device__ __forceinline__ float frame_value(float I, int m, bool has_mask, float T, float S)
{
    float v = has_mask ? I * (float)m : I;
    if (S > 0) return v >= T ? discretize(v, T, S) : 0.0f;
    if (T > 0 && v < T) return 0.0f;
    return v;
}

// Frames a thread reads ahead of its chain of adds.
constexpr uint32_t kAhead = 8;

// One thread per pixel, frames in order: adds to the float sum (ParAdd with
// threshold) or to the long photon tally; calls over consecutive frame stacks
// continue the same per-pixel sequence.  avg != null: the stack is the whole run, the
// sequence starts at zero and ends as finish_kernel ends it (no accumulator in memory).
// HBM bound; kAhead loads are in flight per thread, since a stack of few pixels holds few
// waves per SIMD (200 frames of 517 x 512, 212 MB: 84 us one
// load at a time, 32 us this way, the frames partly still in the last-level cache).
template <bool kPhotons>
__global__ void __launch_bounds__(256)
    accumulate_pixels_kernel(const float *__restrict__ frames, uint32_t nframes, uint32_t npix,
                             const int *__restrict__ mask, float T, float S, float *__restrict__ sum,
                             long long *__restrict__ tally, float *__restrict__ avg)
{
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= npix) return;
    const int m = mask ? mask[j] : 1;
    long long n = 0;
    float s = 0.0f;
    if (!avg) {
        if (kPhotons) n = tally[j]; else s = sum[j];
    }
    auto add = [&](float I) {
        const float v = frame_value(I, m, mask != nullptr, T, kPhotons ? S : 0.0f);
        if (kPhotons) {
            if (v != 0.0f) n += (long long)floor((double)v + 0.5);
        } else {
            if (v >= T) s += v;
        }
    };
    const float *p = frames + j;
    uint32_t f = 0;
    for (; f + kAhead <= nframes; f += kAhead) {
        float I[kAhead];
#pragma unroll
        for (uint32_t k = 0; k < kAhead; k++) I[k] = p[(size_t)(f + k) * npix];
#pragma unroll
        for (uint32_t k = 0; k < kAhead; k++) add(I[k]);
    }
    for (; f < nframes; f++) add(p[(size_t)f * npix]);
    if (avg) {
        avg[j] = (kPhotons ? (float)n : s) * (1.0f / (float)nframes);
    } else {
        if (kPhotons) tally[j] = n; else sum[j] = s;
    }
}

// Intensity = (float)tally (discretised) or the float sum, x (1.0f / N)
__global__ void finish_kernel(uint32_t npix, uint32_t ntotal, float S, const float *__restrict__ sum,
                              const long long *__restrict__ tally, float *__restrict__ avg)
{
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= npix) return;
    const float v = S > 0 ? (float)tally[j] : sum[j];
    avg[j] = v * (1.0f / (float)ntotal);
}

// One block per frame: ArrayOperators::Sum<float> (IAC/ArrayOperators.h:260-268) of the frame's
// values, a serial float sum in pixel order; MeanIntensity = sum / P and, with photon
// discretisation, PhotonCount = (int) sum.  kShort: one wave per frame.
template <bool kMask, bool kPhotons, class Index, bool kShort>
__global__ void __launch_bounds__(kShort ? 64 : iac::kSumThreads)
    frame_sums_kernel(const float *__restrict__ frames, uint32_t npix, const int *__restrict__ mask, float T, float S,
                      float *__restrict__ mean_intensity, int *__restrict__ photon_count)
{
    __shared__ iac::SerialSumShared sh;
    const uint32_t f = blockIdx.x;
    auto value = [=](float v, int m) { return frame_value(v, m, kMask, T, kPhotons ? S : 0.0f); };
    const float *fr = frames + (size_t)f * npix;
    float s;
    if constexpr (kShort) s = iac::serial_sum_wave<kMask>(fr, mask, npix, value);
    else s = iac::serial_sum_block<kMask, Index>(fr, mask, npix, sh, value);
    if (threadIdx.x != 0) return;
    if (mean_intensity) mean_intensity[f] = s / (float)npix;
    if (photon_count && kPhotons) photon_count[f] = iac::cvtt_i32(s);
}

// A stack's frame sums, then its pixel sequences (into d_avg, or the accumulators).
int accumulate_stack(iac_ctx *ctx, const float *d_frames, uint32_t nframes, uint32_t npix, const int *d_mask, float T,
                     float S, float *d_sum, int64_t *d_tally, float *d_avg, float *d_mean_intensity,
                     int *d_photon_count)
{
    if (d_mean_intensity || d_photon_count) {
        if (nframes > 0x7fffffffu) return iac::fail(IAC_ERR_LIMIT, "too many frames in one stack");
        auto pick = [&](auto index, auto is_short) {
            using I = decltype(index);
            constexpr bool B = decltype(is_short)::value;
            return S > 0 ? (d_mask ? frame_sums_kernel<true, true, I, B> : frame_sums_kernel<false, true, I, B>)
                         : (d_mask ? frame_sums_kernel<true, false, I, B> : frame_sums_kernel<false, false, I, B>);
        };
        const bool few = iac::sum_short(npix, nframes, ctx->num_cus);
        auto sums = few ? pick(uint32_t{}, std::true_type{})
                        : (iac::sum_in_64(npix) ? pick(uint64_t{}, std::false_type{}) : pick(uint32_t{}, std::false_type{}));
        hipLaunchKernelGGL(sums, dim3(nframes), dim3(few ? 64 : iac::kSumThreads), 0, ctx->stream, d_frames, npix,
                           d_mask, T, S, d_mean_intensity, d_photon_count);
        IAC_HIP(hipGetLastError());
    }
    auto kern = S > 0 ? accumulate_pixels_kernel<true> : accumulate_pixels_kernel<false>;
    hipLaunchKernelGGL(kern, dim3((npix + 255) / 256), dim3(256), 0, ctx->stream, d_frames, nframes, npix, d_mask, T, S,
                       d_sum, reinterpret_cast<long long *>(d_tally), d_avg);
    IAC_HIP(hipGetLastError());
    return IAC_OK;
}

}  // namespace

extern "C" {

int iac_intensity_accumulate(iac_ctx *ctx, const float *d_frames, uint32_t nframes, uint32_t npix, const int *d_mask,
                             float threshold, float step, float *d_sum, int64_t *d_tally, float *d_mean_intensity,
                             int *d_photon_count)
{
    IAC_TRY(iac::bind(ctx));
    if (!d_frames || npix == 0) return iac::fail(IAC_ERR_INVALID_ARG, "bad averaging request");
    if (step > 0 ? !d_tally : !d_sum) return iac::fail(IAC_ERR_INVALID_ARG, "missing accumulator");
    if (nframes == 0) return IAC_OK;
    return accumulate_stack(ctx, d_frames, nframes, npix, d_mask, threshold, step, d_sum, d_tally, nullptr,
                            d_mean_intensity, d_photon_count);
}

int iac_intensity_finish(iac_ctx *ctx, uint32_t npix, uint32_t ntotal_frames, float step, const float *d_sum,
                         const int64_t *d_tally, float *d_avg)
{
    IAC_TRY(iac::bind(ctx));
    if (!d_avg || npix == 0) return iac::fail(IAC_ERR_INVALID_ARG, "bad averaging request");
    if (ntotal_frames == 0) return iac::fail(IAC_ERR_PRECONDITION, "event list is empty, nothing to average");
    if (step > 0 ? !d_tally : !d_sum) return iac::fail(IAC_ERR_INVALID_ARG, "missing accumulator");
    hipLaunchKernelGGL(finish_kernel, dim3((npix + 255) / 256), dim3(256), 0, ctx->stream, npix, ntotal_frames, step,
                       d_sum, reinterpret_cast<const long long *>(d_tally), d_avg);
    IAC_HIP(hipGetLastError());
    return IAC_OK;
}

int iac_average_intensity(iac_ctx *ctx, const float *d_frames, uint32_t nframes, uint32_t npix, const int *d_mask,
                          float threshold, float step, float *d_avg, float *d_mean_intensity, int *d_photon_count)
{
    IAC_TRY(iac::bind(ctx));
    if (!d_frames || !d_avg || npix == 0) return iac::fail(IAC_ERR_INVALID_ARG, "bad averaging request");
    if (nframes == 0) return iac::fail(IAC_ERR_PRECONDITION, "event list is empty, nothing to average");
    return accumulate_stack(ctx, d_frames, nframes, npix, d_mask, threshold, step, nullptr, nullptr, d_avg,
                            d_mean_intensity, d_photon_count);
}

}  // extern "C"
