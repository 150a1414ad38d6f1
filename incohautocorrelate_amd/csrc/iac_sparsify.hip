// iac_sparsify.hip -- frame sparsification on gfx950: the mask multiply
// (ArrayOperators::ParMultiplyElementwise, IAC/ArrayOperators.h:120-127), the
// hit test and photon discretisation of Detector::CreateSparseHitList
// (IAC/Detector.cpp:926-958, ArrayOperators::DiscretizeToPhotons :138-148),
// producing {kx, ky, kz, value} records in pixel order per frame.
#include <algorithm>
#include <cmath>

#include "iac_internal.h"

#pragma clang fp contract(off)

namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ bool is_hit(float I, float T) { return I >= T && I > 0; }

__device__ __forceinline__ float discretize(float I, float T, float S)
{
    return S > 0 ? ceilf((I - T) / S) * (float)(I >= T) : I;
}

// A frame is cut into slices of `slice` pixels (a power of two, 2048..16384), a block each, so
// that few frames fill the chip too.  The hit test runs once: mark_kernel leaves one bit per
// pixel (1/32 of the frames' bytes) and a count per slice, and emit_kernel reads those and only
// the hit pixels.  Bound: HBM, the frames read once.  One block per frame, the whole frame read
// in both passes and four barriers per 256 pixels took 344 + 748 us for 200 frames of 517 x 512
// (212 MB), this way 64 + 25 us.
constexpr uint32_t kSliceMax = 16384, kSliceMin = 2048;
constexpr uint32_t kWordsAhead = 8;  // 64-pixel words a wave reads at once

// bits[(f ns + s) slice / 64 + i]: hits of pixels 64 i .. 64 i + 63 of slice s; count[f ns + s]
// their number.  Grid: nframes * ns blocks.
__global__ void __launch_bounds__(kBlock)
    mark_kernel(const float *__restrict__ frames, const int *__restrict__ mask, uint32_t npix, uint32_t ns,
                uint32_t slice, float T, unsigned long long *__restrict__ bits, uint32_t *__restrict__ count)
{
    __shared__ uint32_t part[kBlock / 64];
    const uint32_t f = blockIdx.x / ns, p0 = (blockIdx.x - f * ns) * slice;
    const uint32_t len = min(slice, npix - p0);
    const float *fr = frames + (size_t)f * npix + p0;
    const int *mk = mask ? mask + p0 : nullptr;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t words = slice / 64 / (kBlock / 64);  // per wave, a multiple of kWordsAhead
    unsigned long long *out = bits + (size_t)blockIdx.x * (slice / 64);
    uint32_t c = 0;
    for (uint32_t w = wave * words; w < (wave + 1) * words && w * 64 < len; w += kWordsAhead) {
        float I[kWordsAhead];
        int m[kWordsAhead];
#pragma unroll
        for (uint32_t k = 0; k < kWordsAhead; k++) {
            const uint32_t i = (w + k) * 64 + lane;
            I[k] = i < len ? fr[i] : 0.0f;
            m[k] = mk && i < len ? mk[i] : 1;
        }
        unsigned long long mine = 0;
#pragma unroll
        for (uint32_t k = 0; k < kWordsAhead; k++) {
            const bool h = (w + k) * 64 + lane < len && is_hit(mk ? I[k] * (float)m[k] : I[k], T);
            const unsigned long long b = __ballot(h);
            c += (uint32_t)__popcll(b);
            if (lane == k) mine = b;
        }
        if (lane < kWordsAhead) out[w + lane] = mine;
    }
    if (lane == 0) part[wave] = c;
    __syncthreads();
    if (threadIdx.x == 0) count[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// exclusive scan of the frames' counts (ns slices each) -> off[0..n]
__global__ void __launch_bounds__(1024) scan_kernel(const uint32_t *__restrict__ count, uint32_t ns, uint32_t n,
                                                    uint64_t *__restrict__ off)
{
    __shared__ uint64_t part[1024];
    const uint32_t t = threadIdx.x, per = (n + 1023) / 1024;
    const uint32_t f0 = min(n, t * per), f1 = min(n, f0 + per);
    uint64_t s = 0;
    auto frame = [&](uint32_t f) {
        uint64_t c = 0;
#pragma unroll 4
        for (uint32_t k = 0; k < ns; k++) c += count[(size_t)f * ns + k];
        return c;
    };
    for (uint32_t f = f0; f < f1; f++) s += frame(f);
    part[t] = s;
    __syncthreads();
    for (uint32_t o = 1; o < 1024; o <<= 1) {
        const uint64_t v = t >= o ? part[t - o] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    uint64_t run = t ? part[t - 1] : 0;
    for (uint32_t f = f0; f < f1; f++) {
        off[f] = run;
        run += frame(f);
    }
    if (t == 1023) off[n] = part[1023];
}

// The hits of one slice as records, in pixel order from off[f] plus the counts of the slices
// before it: the set bits expand into a list of pixels in LDS (2 bytes per pixel of the slice),
// which consecutive threads then follow.
__global__ void __launch_bounds__(kBlock)
    emit_kernel(const float *__restrict__ frames, const int *__restrict__ mask, const float *__restrict__ kmap,
                uint32_t npix, uint32_t ns, uint32_t slice, float T, float S,
                const unsigned long long *__restrict__ bits, const uint32_t *__restrict__ count,
                const uint64_t *__restrict__ off, float4 *__restrict__ rec)
{
    extern __shared__ uint16_t list[];
    __shared__ uint32_t part[kBlock / 64];
    __shared__ uint32_t before_s[kBlock / 64];
    const uint32_t n = count[blockIdx.x];
    if (n == 0) return;
    const uint32_t f = blockIdx.x / ns, s = blockIdx.x - f * ns, p0 = s * slice;
    const uint32_t len = min(slice, npix - p0), lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    // mark_kernel writes whole groups of words up to the frame's end
    unsigned long long b = threadIdx.x * 64 < len ? bits[(size_t)blockIdx.x * (slice / 64) + threadIdx.x] : 0ull;
    uint32_t before = 0;
    for (uint32_t k = threadIdx.x; k < s; k += kBlock) before += count[(size_t)f * ns + k];
    const uint32_t mine = (uint32_t)__popcll(b);
    uint32_t x = mine;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= (uint32_t)o) x += y;
    }
    for (int o = 32; o > 0; o >>= 1) before += __shfl_down(before, o, 64);
    if (lane == 63) part[wave] = x;
    if (lane == 0) before_s[wave] = before;
    __syncthreads();
    uint32_t at = x - mine;
    for (uint32_t w = 0; w < wave; w++) at += part[w];
    for (; b; b &= b - 1) list[at++] = (uint16_t)(threadIdx.x * 64 + (uint32_t)__builtin_ctzll(b));
    __syncthreads();
    float4 *out = rec + off[f] + before_s[0] + before_s[1] + before_s[2] + before_s[3];
    const float *fr = frames + (size_t)f * npix;
    for (uint32_t i = threadIdx.x; i < n; i += kBlock) {
        const size_t p = (size_t)p0 + list[i];
        float I = fr[p];
        if (mask) I = I * (float)mask[p];
        out[i] = make_float4(kmap[3 * p], kmap[3 * p + 1], kmap[3 * p + 2], discretize(I, T, S));
    }
}

}  // namespace

extern "C" {

int iac_sparse_hit_list(iac_ctx *ctx, const float *d_kmap, uint32_t npix, const float *d_frames, uint32_t nframes,
                        const int *d_mask, float threshold, float step, float *d_rec4, uint64_t *d_frame_off,
                        uint64_t *n_total)
{
    IAC_TRY(iac::bind(ctx));
    if (!d_kmap || !d_frames || !d_rec4 || !d_frame_off || !n_total || npix == 0)
        return iac::fail(IAC_ERR_INVALID_ARG, "null input");
    *n_total = 0;
    if (nframes == 0) return IAC_OK;
    // the largest slice that still makes four blocks per CU
    uint32_t slice = kSliceMax;
    auto slices = [&](uint32_t n) { return (uint32_t)(((uint64_t)npix + n - 1) / n); };
    while (slice > kSliceMin && (uint64_t)nframes * slices(slice) < 4ull * ctx->num_cus) slice /= 2;
    const uint32_t ns = slices(slice);
    const uint64_t blocks = (uint64_t)nframes * ns;
    if (blocks > 0x7fffffffull) return iac::fail(IAC_ERR_LIMIT, "frame stack too large");
    void *work = nullptr;  // hit bits, then slice counts
    const size_t bit_bytes = blocks * (slice / 8);
    IAC_TRY(iac::scratch(ctx, 1, bit_bytes + blocks * sizeof(uint32_t), &work));
    auto *bits = static_cast<unsigned long long *>(work);
    auto *cnt = reinterpret_cast<uint32_t *>(static_cast<char *>(work) + bit_bytes);
    hipLaunchKernelGGL(mark_kernel, dim3((unsigned)blocks), dim3(kBlock), 0, ctx->stream, d_frames, d_mask, npix, ns,
                       slice, threshold, bits, cnt);
    hipLaunchKernelGGL(scan_kernel, dim3(1), dim3(1024), 0, ctx->stream, cnt, ns, nframes, d_frame_off);
    IAC_TRY(iac::timer_begin(ctx));
    hipLaunchKernelGGL(emit_kernel, dim3((unsigned)blocks), dim3(kBlock), slice * sizeof(uint16_t), ctx->stream,
                       d_frames, d_mask, d_kmap, npix, ns, slice, threshold, step, bits, cnt, d_frame_off,
                       reinterpret_cast<float4 *>(d_rec4));
    IAC_HIP(hipGetLastError());
    IAC_TRY(iac::timer_end(ctx));
    void *n = nullptr;
    IAC_TRY(iac::pinned(ctx, 0, sizeof(uint64_t), &n));
    IAC_HIP(hipMemcpyAsync(n, d_frame_off + nframes, sizeof(uint64_t), hipMemcpyDeviceToHost, ctx->stream));
    IAC_HIP(hipStreamSynchronize(ctx->stream));
    *n_total = *static_cast<const uint64_t *>(n);
    return IAC_OK;
}

}  // extern "C"
