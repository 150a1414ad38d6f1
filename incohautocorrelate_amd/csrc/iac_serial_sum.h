// iac_serial_sum.h -- ArrayOperators::Sum<float> (IAC/ArrayOperators.h:260-268) of one frame per
// block: the float sum in pixel order, bit for bit, without walking the frame value by value.
//
// While the running sum s stays inside one binade it is m ulps, m in [2^23, 2^24), and adding v
// takes m to the integer nearest m + v / ulp, a tie to the even one.  So a run of values adds a
// number d that depends on m only through its parity, and such maps compose.  1,024 threads form
// the maps of 16 consecutive values each -- by adding v / ulp to 1.5 * 2^23 and to its odd
// neighbour in float, which rounds the same way --, a scan composes them, and every thread learns
// the exact m in front of its values.  A thread whose values could leave the binade (or hold
// NaN, infinities or a step of a quarter binade) stops the scan: the values in front of it count,
// its own 16 are added in float, and the threads behind it go on in the new binade, at first in
// a window as long as what lies behind (a steady sum doubles once per window).  A growing sum
// leaves a binade ~20 times per frame; after kSumRetries such stops (a sum that wanders about
// zero) wave 0 adds the rest of the frame value by value.
//
// Bound: the frame's bytes for many frames, the chunks' serial chain (a scan of 16,384 values
// each) for few.  200 frames of 517 x 512 (212 MB): 3,085 us with one wave per frame feeding
// v_readlane into a serial chain (one add per value), 109 us this way.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace iac {

constexpr uint32_t kSumThreads = 1024;
constexpr uint32_t kSumPer = 16;                         // consecutive values per thread
constexpr uint32_t kSumChunk = kSumThreads * kSumPer;    // values per scan
constexpr uint32_t kSumWaves = kSumThreads / 64;
constexpr uint32_t kSumRetries = 96;

// A run of values: m -> m + d where m is even, m + d + e where it is odd (e is -1, 0 or 1).
struct UlpMap {
    int d, e;
};
__device__ __forceinline__ int ulp_apply(const UlpMap &a, int m) { return m + a.d + ((m & 1) ? a.e : 0); }
// a, then b
__device__ __forceinline__ UlpMap ulp_then(const UlpMap &a, const UlpMap &b)
{
    const int from_even = a.d + b.d + ((a.d & 1) ? b.e : 0);
    const int odd = a.d + a.e;  // an odd m becomes odd + m: even where odd is
    const int from_odd = odd + b.d + ((odd & 1) ? 0 : b.e);
    return UlpMap{from_even, from_odd - from_even};
}

struct SerialSumShared {
    UlpMap wave[kSumWaves];
    uint32_t stop[kSumWaves];
    float s, rest;
};

// 16 bytes at any float's address (the hardware needs 4-byte alignment for them)
template <class T>
struct __attribute__((packed, aligned(4))) Four {
    T x[4];
};
template <class T>
__device__ __forceinline__ void load_run(const T *__restrict__ p, T *v)
{
#pragma unroll
    for (uint32_t i = 0; i < kSumPer / 4; i++) {
        const Four<T> q = reinterpret_cast<const Four<T> *>(p)[i];
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) v[4 * i + k] = q.x[k];
    }
}

// Frames whose last chunk's pixel numbers may pass 2^32 count them in 64 bits (which costs 2 %:
// 252 -> 257 us for averaging and sparsifying the frames above).
inline bool sum_in_64(uint32_t npix) { return npix > UINT32_MAX - kSumChunk; }

// Short frames are added value by value by one wave: a growing sum leaves its first ten binades within
// them, a stop each.  Averages of 20 frames of 1,000 pixels 31.6 us by the scan, 15.6 so; of 2,560
// 33.7 and 21.0, of 4,096 32.5 and 29.1; with more frames than CUs the scans' blocks queue up:
// 300 frames of 4,096 pixels 70.9 and 41.6, of 8,192 76.0 and 64.4.
inline bool sum_short(uint32_t npix, uint32_t nframes, int cus) { return npix <= (nframes > (uint32_t)cus ? 8192u : 4096u); }

// The same sum by a one-wave block: 64 values at once, fed in order into a sum that every lane holds.
// Bound: the chain of adds, an add and a lane read per value.
template <bool kMask, class V>
__device__ __forceinline__ float serial_sum_wave(const float *__restrict__ fr, const int *__restrict__ mask,
                                                 uint32_t npix, V value)
{
    float s = 0.0f;
    int m = 1;
    float v = fr[min(threadIdx.x, npix - 1)];
    if (kMask) m = mask[min(threadIdx.x, npix - 1)];
    for (uint32_t j0 = 0; j0 < npix; j0 += 64) {
        const int x = __float_as_int(j0 + threadIdx.x < npix ? value(v, m) : 0.0f);
        const uint32_t next = min(j0 + 64 + threadIdx.x, npix - 1);  // loads under the adds
        v = fr[next];
        if (kMask) m = mask[next];
        // a lane is read one add ahead: its scalar is ready when the chain of adds gets there
        int a = __builtin_amdgcn_readlane(x, 0);
#pragma unroll
        for (int i = 1; i < 64; i++) {
            const int b = __builtin_amdgcn_readlane(x, i);
            s += __int_as_float(a);
            a = b;
        }
        s += __int_as_float(a);
    }
    return s;
}

// value(v, m): what a pixel of value v and mask m (1 without kMask) adds to the sum.  Index: of pixels,
// uint32_t or, where sum_in_64, uint64_t.  Called by all threads of a block of kSumThreads; returns the
// frame's sum in every thread.
template <bool kMask, class Index, class V>
__device__ __forceinline__ float serial_sum_block(const float *__restrict__ fr, const int *__restrict__ mask,
                                                  Index npix, SerialSumShared &sh, V value)
{
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    constexpr float kMid = 12582912.0f;  // 1.5 * 2^23, even: floats within 2^22 of it are 1 apart
    auto load = [&](Index j0, float *v) {
        const Index j = j0 + t * kSumPer;
        int m[kSumPer];
        if (npix - j0 >= kSumChunk) {
            load_run(fr + j, v);
            if (kMask) load_run(mask + j, m);
#pragma unroll
            for (uint32_t i = 0; i < kSumPer; i++) v[i] = value(v[i], kMask ? m[i] : 1);
        } else {  // past the frame: +0 adds nothing (a sum that starts at +0 is never -0)
#pragma unroll
            for (uint32_t i = 0; i < kSumPer; i++) {
                v[i] = j + i < npix ? fr[j + i] : 0.0f;
                m[i] = kMask && j + i < npix ? mask[j + i] : 1;
            }
#pragma unroll
            for (uint32_t i = 0; i < kSumPer; i++) v[i] = j + i < npix ? value(v[i], m[i]) : 0.0f;
        }
    };
    float s = 0.0f, v[kSumPer], next[kSumPer];
    uint32_t retries = 0;
    load(0, v);
    for (Index j0 = 0; j0 < npix; j0 += kSumChunk) {
        if (npix - j0 > kSumChunk) load(j0 + kSumChunk, next);
        for (uint32_t first = 0; first < kSumThreads;) {  // threads below `first` are in s
            // s = m ulps; an s near zero (no such binade), infinite or NaN takes only zeros
            const bool flat = !(fabsf(s) >= 0x1p-100f && fabsf(s) < __builtin_inff());
            const int ex = (int)((__float_as_uint(s) >> 23) & 0xffu) - 127;
            const float per_ulp = flat ? 0.0f : copysignf(__uint_as_float((uint32_t)(127 + 23 - ex) << 23), s);
            const float ulp = flat ? 0.0f : copysignf(__uint_as_float((uint32_t)(127 - 23 + ex) << 23), s);
            const int m0 = flat ? 0 : (int)((__float_as_uint(s) & 0x7fffffu) | 0x800000u);
            // the window: as many values as the frame has behind it, in whole waves
            const uint32_t behind = (uint32_t)((j0 / kSumPer + first) / 64) + 1;
            const uint32_t end = min(kSumThreads, (first / 64 + behind) * 64);
            UlpMap own{0, 0};
            int lo = 0, hi = 0;
            bool bad = false, down = false;
            if (wave * 64 < end && wave * 64 + 63 >= first) {
                float x0 = kMid, x1 = kMid + 1.0f, xlo = kMid, xhi = kMid;
                uint32_t any = 0;
#pragma unroll
                for (uint32_t i = 0; i < kSumPer; i++) {
                    const float f = v[i] * per_ulp;
                    x0 += f;
                    x1 += f;
                    xlo = fminf(xlo, x0);
                    xhi = fmaxf(xhi, x0);
                    any |= flat ? __float_as_uint(v[i]) << 1 : __float_as_uint(f);
                }
                // inside 2^22 of kMid throughout (with 2 to spare for x1), or not to be trusted
                bad = !(xlo > kMid - 4194300.0f && xhi < kMid + 4194300.0f && x0 == x0) || (flat && any);
                if (!bad && t >= first) {
                    down = (any >> 31) != 0;  // a negative step
                    own = UlpMap{(int)(x0 - kMid), 0};
                    own.e = (int)(x1 - kMid) - 1 - own.d;
                    lo = (int)(xlo - kMid);
                    hi = (int)(xhi - kMid);
                }
                bad = bad && t >= first;
            }
            UlpMap in = own;  // inclusive scan over the wave
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const UlpMap p{__shfl_up(in.d, o, 64), __shfl_up(in.e, o, 64)};
                if (lane >= (uint32_t)o) in = ulp_then(p, in);
            }
            // beyond 2^24 something in the wave stops the scan: only the sign of the total counts
            if (lane == 63) sh.wave[wave] = UlpMap{max(-(1 << 26), min(1 << 26, in.d)), in.e};
            UlpMap front{__shfl_up(in.d, 1, 64), __shfl_up(in.e, 1, 64)};
            if (lane == 0) front = UlpMap{0, 0};
            __syncthreads();
            UlpMap all = lane < kSumWaves ? sh.wave[lane] : UlpMap{0, 0};  // inclusive scan over the waves
#pragma unroll
            for (int o = 1; o < (int)kSumWaves; o <<= 1) {
                const UlpMap p{__shfl_up(all.d, o, 64), __shfl_up(all.e, o, 64)};
                if (lane >= (uint32_t)o) all = ulp_then(p, all);
            }
            auto waves = [&](int w) {
                return UlpMap{__builtin_amdgcn_readlane(all.d, w), __builtin_amdgcn_readlane(all.e, w)};
            };
            const int uw = __builtin_amdgcn_readfirstlane((int)wave);
            int m = uw ? ulp_apply(waves(uw - 1), m0) : m0;
            m = ulp_apply(front, m);  // in front of the thread's values
            // lo and hi belong to an even m, an odd one differs by at most 1.  A step down at the
            // binade's lower edge would round on the finer ulps below it.
            const bool out = bad || (hi > 0 && m + hi + 1 >= (1 << 24)) || (down && m + lo - 1 <= (1 << 23));
            const uint64_t outs = __ballot(out);
            if (lane == 0) sh.stop[wave] = outs ? wave * 64 + (uint32_t)__builtin_ctzll(outs) : kSumThreads;
            __syncthreads();
            uint32_t stop = kSumThreads;
            for (uint32_t w = 0; w < kSumWaves; w++) stop = min(stop, sh.stop[w]);
            if (stop == kSumThreads) {
                if (!flat) s = (float)ulp_apply(waves(kSumWaves - 1), m0) * ulp;
                first = end;
                continue;
            }
            if (t == stop) {
                float x = flat ? s : (float)m * ulp;
#pragma unroll
                for (uint32_t i = 0; i < kSumPer; i++) x += v[i];
                sh.s = x;
            }
            __syncthreads();
            s = sh.s;
            first = stop + 1;
            if (++retries > kSumRetries) {
                // the rest value by value, fed in order into wave 0's running sum
                if (wave == 0) {
                    for (Index j = j0 + first * kSumPer; j < npix; j += 64) {
                        const bool in = lane < npix - j;
                        const int x = __float_as_int(in ? value(fr[j + lane], kMask ? mask[j + lane] : 1) : 0.0f);
#pragma unroll
                        for (int i = 0; i < 64; i++) s += __int_as_float(__builtin_amdgcn_readlane(x, i));
                    }
                    if (lane == 0) sh.rest = s;
                }
                __syncthreads();
                return sh.rest;
            }
        }
#pragma unroll
        for (uint32_t i = 0; i < kSumPer; i++) v[i] = next[i];
    }
    return s;
}

}  // namespace iac
