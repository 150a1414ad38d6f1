// iac_cq.hip -- C(q): dense pixel-pair normalisation mesh, rotation merge and
// the final AC/C(q) division, on gfx950.
//
//   iac_cq_small / iac_cq_dense_frames: AutoCorr_CQ_small (IAC/kernel.cl:27-184)
//     by region tiles where they suit the images, else through the LDS cell-box pair
//     engine's walk (one record per pixel).
//   iac_merge_cq: Merge_CQ (IAC/kernel.cl:189-344), bricks of the big mesh in LDS, or
//     scattered adds where the updates are few.
//   iac_merge_ac_cq: RunIAC::Merge_ACandCQ (IAC/RunIAC.cpp:120-158).
#include <algorithm>
#include <cmath>
#include <cstring>

#include "iac_binning.h"
#include "iac_internal.h"
#include "iac_pairs.h"

#pragma clang fp contract(off)

namespace {

// records {k[p], I[f][p]} of dense frames; off[f] = f * npix
__global__ void gather_dense_kernel(const float *__restrict__ kmap, const float *__restrict__ frames,
                                    uint32_t npix, uint32_t nframes, float4 *__restrict__ rec,
                                    uint64_t *__restrict__ off)
{
    const uint64_t n = (uint64_t)npix * nframes;
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t p = (uint32_t)(i % npix);
        rec[i] = make_float4(kmap[3 * (size_t)p], kmap[3 * (size_t)p + 1], kmap[3 * (size_t)p + 2], frames[i]);
    }
    for (uint64_t f = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; f <= nframes; f += (uint64_t)gridDim.x * blockDim.x)
        off[f] = f * npix;
}

__global__ void u64_to_f64_kernel(const unsigned long long *__restrict__ in, size_t n, double mult,
                                  double *__restrict__ out)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        out[i] = (double)in[i] / mult;
}

// ---- Merge_CQ ------------------------------------------------------------------------
// Every small-mesh voxel, rotated by every event, adds to the cubic big mesh (its slow-scan index
// uses size_ab's centre too).  A scattered add is one L2 atomic request (2.4e10/s, 1,656 us for
// 1,000 events of a 129 x 129 x 3 mesh), so the big mesh is cut into bricks held in LDS: a block
// takes a brick and a slice of the events, finds per event the small voxels that can reach the
// brick (the brick turned back by the transposed matrix), bins exactly those and flushes the
// brick with contiguous adds: 284 us and 39 us for the rest.  Bound: VALU issue, most of it for
// the rows of candidates, whose 54 updates per brick and event lie in about 50 rows.  Other bricks
// and events per block measured (whole call, 315 us): 16 x 8 x 8 with 32, 128 or 256 events 340,
// 326, 378 us; 16 x 16 x 16 with 128 events 358; 16 x 8 x 4 459; the z rows of a y row in one
// thread 353 (rows of unequal length side by side).
// The transposed matrix is the inverse only of a rotation.  Events whose matrix is not
// orthonormal to kOrtho, and the count of updates that leave the mesh (voxels near or beyond its
// inscribed sphere), go through merge_rest_kernel.

constexpr float kOrtho = 1e-4f;               // largest |(R^T R - 1)_ij| the bricks take
constexpr int kBrX = 16, kBrY = 8, kBrZ = 8;  // 8 KB: 16 voxels are two 64-byte segments to flush
constexpr int kBrick = kBrX * kBrY * kBrZ;
constexpr uint32_t kBrickEvents = 6;       // log2 of the events that reach a brick, per block (about), at most
constexpr uint32_t kBrickEventsLeast = 2;  // and at least, where the bricks alone leave CUs idle

__device__ __forceinline__ bool orthonormal(const float *R)
{
    float worst = 0.0f;
    bool finite = true;
    for (int i = 0; i < 3; i++)
        for (int j = i; j < 3; j++) {
            const float d = (R[i] * R[j] + R[3 + i] * R[3 + j]) + R[6 + i] * R[6 + j] - (i == j ? 1.0f : 0.0f);
            worst = fmaxf(worst, fabsf(d));
            finite = finite && fabsf(d) < 1.0f;  // false for NaN
        }
    return finite && worst <= kOrtho;
}

constexpr int kRowAhead = 4;  // small voxels of a row read at once

// (unsigned long long)x, the usual values below 2^32 in one instruction
__device__ __forceinline__ unsigned long long fixed_u64(double x)
{
    if (__builtin_amdgcn_ballot_w64(!(x >= 0.0 && x < 4294967296.0)) != 0) {
        asm volatile("");
        return (unsigned long long)x;
    }
    return (uint32_t)x;
}

// What one small voxel of value val_in at the rotated (q0, q1, q2) adds (kernel.cl:262-341):
// add(fs, ms, ss, value) once, or per corner.  kFinite: no q is NaN (a NaN's voxel is index 0, what
// its conversion to an integer gives).
template <bool kLinear, bool kFinite, class Add>
__device__ __forceinline__ void merge_voxel(float q0, float q1, float q2, double val_in, double w, double mult,
                                            int cab, Add add)
{
    if (!kLinear) {
        // roundf(q) for |q| < 2^22: half away from zero is x + copysign(0.49999997f, x), truncated
        auto voxel = [cab](float x) {
            const int n = (int)(x + copysignf(0.49999997f, x)) + cab;
            return kFinite || x == x ? n : 0;
        };
        add(voxel(q0), voxel(q1), voxel(q2), fixed_u64((val_in * w) * mult));
        return;
    }
    const double sfs = (double)(1.0f - (q0 - floorf(q0)));
    const double sms = (double)(1.0f - (q1 - floorf(q1)));
    const double sss = (double)(1.0f - (q2 - floorf(q2)));
    const int fs = (int)(floorf(q0) + (float)cab);
    const int ms = (int)(floorf(q1) + (float)cab);
    const int ss = (int)(floorf(q2) + (float)cab);
    const double vmw = (val_in * mult) * w;
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const int ex = (c >> 1) & 1, ey = c >> 2, ez = c & 1;
        add(fs + ex, ms + ey, ss + ez,
            fixed_u64(vmw * (((ex ? 1 - sfs : sfs) * (ey ? 1 - sms : sms)) * (ez ? 1 - sss : sss))));
    }
}

// The event's candidates for a brick: rows (y, z) of small voxels along k_a, y of ny from y0
// (k_b), z of nz from z0 (k_c); row0 is the number of rows of the events listed before it.
struct BrickEvent {
    uint32_t event, row0;
    int16_t y0, ny, z0, nz;
};

// Grid: x bricks, y slices of the events; a brick takes as many slices as events reach it.
template <bool kLinear>
__global__ void __launch_bounds__(256)
    merge_brick_kernel(const double *__restrict__ small, size_t small_stride, int sab, int sc, int ka, int kb, int kc,
                       const float *__restrict__ rw, uint32_t nev, uint32_t per_log2, double mult, int nbx, int nby,
                       unsigned long long *__restrict__ big)
{
    __shared__ unsigned long long box[kBrick];
    __shared__ BrickEvent list[256];
    __shared__ uint32_t wev[4], wrow[4];
    const int cab = (sab - 1) / 2, cc = (sc - 1) / 2;
    const int bi = (int)blockIdx.x, b0 = (bi % nbx) * kBrX, b1 = (bi / nbx % nby) * kBrY, b2 = bi / (nbx * nby) * kBrZ;
    const int e0_ = min(kBrX, sab - b0), e1_ = min(kBrY, sab - b1), e2_ = min(kBrZ, sab - b2);
    // the q that reach the brick: its voxels' range (nearest: half a voxel more, linear: one),
    // with a margin for the float arithmetic of either side
    const float reach = (kLinear ? 1.0f : 0.5f) + 0.01f;
    const float lo[3] = {(float)(b0 - cab) - reach, (float)(b1 - cab) - reach, (float)(b2 - cab) - reach};
    const float hi[3] = {(float)(b0 + e0_ - 1 - cab) + reach, (float)(b1 + e1_ - 1 - cab) + reach,
                         (float)(b2 + e2_ - 1 - cab) + reach};
    const float mid[3] = {0.5f * (lo[0] + hi[0]), 0.5f * (lo[1] + hi[1]), 0.5f * (lo[2] + hi[2])};
    const float half[3] = {0.5f * (hi[0] - lo[0]), 0.5f * (hi[1] - lo[1]), 0.5f * (hi[2] - lo[2])};
    // events whose slab (cc planes each side) reaches a brick at distance r: about the share
    // (its half diagonal + cc) / r
    const float r = sqrtf(mid[0] * mid[0] + mid[1] * mid[1] + mid[2] * mid[2]);
    const float share = fminf(1.0f, (11.0f + (float)cc) / fmaxf(r, 1.0f));
    const uint32_t slices = min(gridDim.y, ((uint32_t)((float)nev * share) >> per_log2) + 1);
    if (blockIdx.y >= slices) return;
    const uint32_t ev0 = (uint32_t)((uint64_t)nev * blockIdx.y / slices);
    const uint32_t ev1 = (uint32_t)((uint64_t)nev * (blockIdx.y + 1) / slices);
    const float qmax = sqrtf(2.0f * (float)cab * (float)cab + (float)cc * (float)cc);
    const float margin = 0.02f + 3.0f * kOrtho * qmax;  // |R^T q - q_in| of a small voxel
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    bool any = false;
    for (uint32_t first = ev0; first < ev1; first += 256) {
        const uint32_t e = first + threadIdx.x;
        int l[3] = {0, 0, 0}, n[3] = {0, 0, 0};
        if (e < ev1) {
            float R[9];
            for (int i = 0; i < 9; i++) R[i] = rw[10 * (size_t)e + i];
            if (orthonormal(R)) {
                const int c[3] = {ka, kb, kc}, ext[3] = {cab, cab, cc};
#pragma unroll
                for (int j = 0; j < 3; j++) {
                    const float r0 = c[j] == 0 ? R[0] : (c[j] == 1 ? R[1] : R[2]);
                    const float r1 = c[j] == 0 ? R[3] : (c[j] == 1 ? R[4] : R[5]);
                    const float r2 = c[j] == 0 ? R[6] : (c[j] == 1 ? R[7] : R[8]);
                    const float p = r0 * mid[0] + r1 * mid[1] + r2 * mid[2];
                    const float h = fabsf(r0) * half[0] + fabsf(r1) * half[1] + fabsf(r2) * half[2] + margin;
                    l[j] = max(-ext[j], (int)ceilf(p - h));
                    n[j] = min(ext[j], (int)floorf(p + h)) - l[j] + 1;
                }
            }
        }
        const bool hit = n[0] > 0 && n[1] > 0 && n[2] > 0;
        const uint32_t rows = hit ? (uint32_t)(n[1] * n[2]) : 0u;
        const uint64_t hits = __ballot(hit);
        uint32_t x = rows;  // inclusive scan
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o, 64);
            if (lane >= (uint32_t)o) x += y;
        }
        if (lane == 63) {
            wev[wave] = (uint32_t)__popcll(hits);
            wrow[wave] = x;
        }
        __syncthreads();
        uint32_t at = (uint32_t)__popcll(hits & ((1ull << lane) - 1)), row = x - rows, nlist = 0, total = 0;
        for (uint32_t w = 0; w < 4; w++) {
            if (w < wave) {
                at += wev[w];
                row += wrow[w];
            }
            nlist += wev[w];
            total += wrow[w];
        }
        if (hit)
            list[at] = BrickEvent{e, row, (int16_t)l[1], (int16_t)n[1], (int16_t)l[2], (int16_t)n[2]};
        if (total && !any) {
            any = true;
            for (int v = threadIdx.x; v < kBrick; v += 256) box[v] = 0ull;
        }
        __syncthreads();
        for (uint32_t t = threadIdx.x; t < total; t += 256) {
            uint32_t a = 0, end = nlist;  // the event of row t
            while (end - a > 1) {
                const uint32_t m = (a + end) / 2;
                if (list[m].row0 <= t) a = m; else end = m;
            }
            const BrickEvent E = list[a];
            const uint32_t k = t - E.row0, iz = k / (uint32_t)E.ny;
            const int y = E.y0 + (int)(k - iz * (uint32_t)E.ny), z = E.z0 + (int)iz;
            const float *Re = rw + 10 * (size_t)E.event;
            const double w = (double)Re[9];
            // q_i = (slope x + u) + v in the order of the components, x the voxel along k_a
            float slope[3], u[3], v[3], x0 = (float)-cab, x1 = (float)cab;
#pragma unroll
            for (int i = 0; i < 3; i++) {
                slope[i] = Re[3 * i + ka];
                const float py = Re[3 * i + kb] * (float)y, pz = Re[3 * i + kc] * (float)z;
                const float first_p = kb < kc ? py : pz, second_p = kb < kc ? pz : py;
                u[i] = ka == 2 ? first_p + second_p : first_p;
                v[i] = ka == 2 ? 0.0f : second_p;
                const float s = py + pz;
                if (fabsf(slope[i]) > 1e-6f) {
                    const float inv = __builtin_amdgcn_rcpf(slope[i]), xa = (lo[i] - s) * inv, xb = (hi[i] - s) * inv;
                    x0 = fmaxf(x0, fminf(xa, xb));
                    x1 = fminf(x1, fmaxf(xa, xb));
                } else if (s < lo[i] - 0.01f || s > hi[i] + 0.01f) {
                    x1 = x0 - 1.0f;
                }
            }
            const int i0 = max((int)ceilf(x0 - 0.02f), -cab), i1 = min((int)floorf(x1 + 0.02f), cab);
            const double *src = small + small_stride * E.event + ((size_t)(z + cc) * sab + (size_t)(y + cab)) * sab + cab;
            for (int i = i0; i <= i1; i += kRowAhead) {
                double val[kRowAhead];
#pragma unroll
                for (int j = 0; j < kRowAhead; j++) val[j] = i + j <= i1 ? src[i + j] : 0.0;
#pragma unroll
                for (int j = 0; j < kRowAhead; j++) {
                    if (val[j] < (double)1e-37f) continue;
                    const float xf = (float)(i + j);
                    const float q0 = (slope[0] * xf + u[0]) + v[0];
                    const float q1 = (slope[1] * xf + u[1]) + v[1];
                    const float q2 = (slope[2] * xf + u[2]) + v[2];
                    merge_voxel<kLinear, true>(q0, q1, q2, val[j], w, mult, cab,
                                         [&](int fs, int ms, int ss, unsigned long long x) {
                                             const int lx = fs - b0, ly = ms - b1, lz = ss - b2;
                                             if ((unsigned)lx < (unsigned)e0_ && (unsigned)ly < (unsigned)e1_ &&
                                                 (unsigned)lz < (unsigned)e2_)
                                                 atomicAdd(&box[lx + kBrX * (ly + kBrY * lz)], x);
                                         });
                }
            }
        }
        __syncthreads();
    }
    if (!any) return;
    for (int v = threadIdx.x; v < kBrick; v += 256) {
        const unsigned long long x = box[v];
        if (x) {
            const size_t fs = b0 + v % kBrX, ms = b1 + v / kBrX % kBrY, ss = b2 + v / (kBrX * kBrY);
            atomicAdd(big + fs + ms * sab + ss * sab * sab, x);
        }
    }
}

constexpr uint32_t kRestEvents = 16;  // at most 64

// Small voxel `ind` under the events of this block row: every update of an event the bricks
// do not take (kBricks false: all events), of the others only the count of updates outside
// the mesh, which voxels well inside its inscribed sphere do not have.
template <bool kLinear, bool kBricks>
__global__ void __launch_bounds__(256)
    merge_rest_kernel(const double *__restrict__ small, size_t small_stride, int sab, int sc, int ka, int kb, int kc,
                      const float *__restrict__ rw, uint32_t nev, double mult,
                      unsigned long long *__restrict__ big, unsigned long long *__restrict__ dropped)
{
    __shared__ uint64_t taken;  // bit k: the bricks take event e0 + k
    const size_t nsmall = (size_t)sab * sab * sc;
    const size_t ind = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    const uint32_t e0 = blockIdx.y * kRestEvents, e1 = min(nev, e0 + kRestEvents);
    if (kBricks && threadIdx.x < 64) {
        const uint32_t e = e0 + threadIdx.x;
        const uint64_t b = __ballot(e < e1 && orthonormal(rw + 10 * (size_t)e));
        if (threadIdx.x == 0) taken = b;
    }
    if (kBricks) __syncthreads();
    if (ind >= nsmall) return;
    const int cab = (sab - 1) / 2, cc = (sc - 1) / 2;
    const int ss_in = (int)(ind / ((size_t)sab * sab));
    const int ms_in = (int)((ind - (size_t)ss_in * sab * sab) / sab);
    const int fs_in = (int)(ind - (size_t)ss_in * sab * sab - (size_t)ms_in * sab);
    const float qa = (float)(fs_in - cab), qb = (float)(ms_in - cab), qc = (float)(ss_in - cc);
    const float qi0 = ka == 0 ? qa : (kb == 0 ? qb : qc), qi1 = ka == 1 ? qa : (kb == 1 ? qb : qc);
    const float qi2 = ka == 2 ? qa : (kb == 2 ? qb : qc);
    // |R q| <= |q| sqrt(1 + 3 kOrtho); the farthest corner is within one voxel of it per axis
    const float inner = (float)cab - 1.5f;
    const bool inside = inner > 0.0f && (qa * qa + qb * qb + qc * qc) * (1.0f + 4.0f * kOrtho) < inner * inner;
    const uint64_t skip = kBricks ? taken : 0;
    const uint32_t n = e1 - e0;
    if (kBricks && inside && skip == (n < 64 ? (1ull << n) - 1 : ~0ull)) return;
    for (uint32_t i = e0; i < e1; i++) {
        const float *R = rw + 10 * (size_t)i;
        const bool in_bricks = kBricks && ((skip >> (i - e0)) & 1);
        if (in_bricks && inside) continue;
        const double val_in = small[small_stride * i + ind];  // stride 0: one mesh for all events
        if (val_in < (double)1e-37f) continue;
        const float q0 = R[0] * qi0 + R[1] * qi1 + R[2] * qi2;
        const float q1 = R[3] * qi0 + R[4] * qi1 + R[5] * qi2;
        const float q2 = R[6] * qi0 + R[7] * qi1 + R[8] * qi2;
        auto add = [&](int fs, int ms, int ss, unsigned long long v) {
            if ((unsigned)fs < (unsigned)sab && (unsigned)ms < (unsigned)sab && (unsigned)ss < (unsigned)sab) {
                if (v && !in_bricks) atomicAdd(big + (size_t)fs + (size_t)ms * sab + (size_t)ss * sab * sab, v);
            } else {
                atomicAdd(dropped, 1ull);
            }
        };
        if (in_bricks) merge_voxel<kLinear, true>(q0, q1, q2, val_in, (double)R[9], mult, cab, add);
        else merge_voxel<kLinear, false>(q0, q1, q2, val_in, (double)R[9], mult, cab, add);
    }
}

// Merge_ACandCQ: AC = IntToFloat(Mesh) (a float) / CQ in double, 0 where CQ <= 0
// or the quotient is NaN.
__global__ void merge_ac_cq_kernel(const unsigned long long *__restrict__ ac, const double *__restrict__ cq,
                                   size_t n, double *__restrict__ out)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float a = ((float)ac[i] * 0.001f) - 0.0f;
        const double c = cq[i];
        double o = c <= 0 ? 0.0 : (double)a / c;
        if (isnan(o)) o = 0.0;
        out[i] = o;
    }
}

int check_small(const iac_mesh_shape *s)
{
    if (!s) return iac::fail(IAC_ERR_INVALID_ARG, "null mesh shape");
    if (s->size_ab % 2 == 0 || s->size_c % 2 == 0 || s->size_ab < 5)
        return iac::fail(IAC_ERR_EVEN_MESH, "Meshsize must be odd for each dimension");
    if (s->k_a > 2 || s->k_b > 2 || s->k_c > 2 || s->k_a == s->k_b || s->k_a == s->k_c || s->k_b == s->k_c)
        return iac::fail(IAC_ERR_INVALID_ARG, "mesh axis alignment must be a permutation of 0,1,2");
    return IAC_OK;
}

unsigned blocks_for(size_t n) { return (unsigned)std::max<size_t>(1, std::min<size_t>(65535, (n + 255) / 256)); }

int cq_frames(iac_ctx *ctx, const float *d_kmap, uint32_t npix, const float *d_frames, uint32_t nframes,
              const uint32_t *h_group_off, uint32_t ngroups, const iac_mesh_shape *shape, int interp, double mult,
              uint64_t *d_meshes)
{
    IAC_TRY(iac::bind(ctx));
    IAC_TRY(check_small(shape));
    if (!d_kmap || !d_frames || !d_meshes || npix == 0) return iac::fail(IAC_ERR_INVALID_ARG, "null input");
    if (interp != IAC_NEAREST && interp != IAC_LINEAR) return iac::fail(IAC_ERR_INVALID_ARG, "bad interpolation");
    if (!(mult > 0)) return iac::fail(IAC_ERR_INVALID_ARG, "multiplicator must be > 0");
    if (nframes == 0) return IAC_OK;
    const uint64_t n = (uint64_t)npix * nframes;
    iac::PairRun R;
    std::memset(&R.spec, 0, sizeof(R.spec));
    R.spec.kind = iac::kKindCq;
    R.spec.ka = (int)shape->k_a;
    R.spec.kb = (int)shape->k_b;
    R.spec.kc = (int)shape->k_c;
    R.spec.interp = interp;
    R.spec.mult = mult;
    R.spec.P.cut_sq = iac::cut_sq(shape->max_q);
    R.spec.P.vox = (float)shape->voxel_per_dq;
    R.spec.P.c0 = (int)(shape->size_ab - 1) / 2;
    R.spec.P.c1 = (int)(shape->size_ab - 1) / 2;
    R.spec.P.c2 = (int)(shape->size_c - 1) / 2;
    R.spec.P.sab = (int)shape->size_ab;
    R.spec.P.sc = (int)shape->size_c;
    R.spec.P.rot_identity = 1;
    R.ordered = interp == IAC_LINEAR;
    R.d_kmap = d_kmap;
    R.npix = npix;
    R.rec = nullptr;
    R.d_frame_off = nullptr;
    R.nframes = nframes;
    R.n_total = n;
    R.h_group_off = h_group_off;
    R.ngroups = ngroups;
    R.d_mesh = d_meshes;
    bool done = false;
    IAC_TRY(iac::cq_tiles_run(ctx, R, d_frames, &done));
    if (done) return IAC_OK;
    // records, then the frame offsets, in scratch slot 0
    void *rec = nullptr;
    IAC_TRY(iac::scratch(ctx, 0, n * sizeof(float4) + (nframes + 1) * sizeof(uint64_t), &rec));
    void *off = static_cast<char *>(rec) + n * sizeof(float4);
    hipLaunchKernelGGL(gather_dense_kernel, dim3(blocks_for(n)), dim3(256), 0, ctx->stream, d_kmap, d_frames,
                       npix, nframes, static_cast<float4 *>(rec), static_cast<uint64_t *>(off));
    IAC_HIP(hipGetLastError());
    R.rec = static_cast<const float4 *>(rec);
    R.d_frame_off = static_cast<const uint64_t *>(off);
    return iac::pairs_run(ctx, R);
}

}  // namespace

extern "C" {

int iac_cq_small_multiplicator(const float *intensity, uint32_t npix, double *mult)
{
    if (!intensity || !mult || npix == 0) return iac::fail(IAC_ERR_INVALID_ARG, "null input");
    double t = 0;
    for (uint32_t i = 0; i < npix; i++) t += intensity[i];
    t = t / npix;
    const float mean = (float)t;
    if (mean <= 0)
        return iac::fail(IAC_ERR_PRECONDITION, "No intensity > 0 found in averaged intensity");
    double m = 1e-10;
    for (; 1 > mean * mean * m;) m *= 10;
    *mult = m * 100000;
    return IAC_OK;
}

int iac_cq_small(iac_ctx *ctx, const float *d_kmap, uint32_t npix, const float *d_intensity,
                 const iac_mesh_shape *small_shape, int interp, double mult, uint64_t *d_mesh)
{
    const uint32_t goff[2] = {0, 1};
    return cq_frames(ctx, d_kmap, npix, d_intensity, 1, goff, 1, small_shape, interp, mult, d_mesh);
}

int iac_cq_dense_frames(iac_ctx *ctx, const float *d_kmap, uint32_t npix, const float *d_frames,
                        uint32_t nframes, const uint32_t *h_group_off, uint32_t ngroups,
                        const iac_mesh_shape *shape, int interp, double mult, uint64_t *d_meshes)
{
    if (!h_group_off || ngroups == 0) return iac::fail(IAC_ERR_INVALID_ARG, "no frame groups");
    if (h_group_off[0] != 0 || h_group_off[ngroups] != nframes)
        return iac::fail(IAC_ERR_SHAPE, "frame groups must cover [0, nframes)");
    for (uint32_t g = 0; g < ngroups; g++)
        if (h_group_off[g + 1] < h_group_off[g]) return iac::fail(IAC_ERR_SHAPE, "frame groups must be sorted");
    return cq_frames(ctx, d_kmap, npix, d_frames, nframes, h_group_off, ngroups, shape, interp, mult, d_meshes);
}

int iac_u64_to_f64(iac_ctx *ctx, const uint64_t *d_in, size_t n, double mult, double *d_out)
{
    IAC_TRY(iac::bind(ctx));
    if (!d_in || !d_out) return iac::fail(IAC_ERR_INVALID_ARG, "null pointer");
    if (n == 0) return IAC_OK;
    hipLaunchKernelGGL(u64_to_f64_kernel, dim3(blocks_for(n)), dim3(256), 0, ctx->stream,
                       reinterpret_cast<const unsigned long long *>(d_in), n, mult, d_out);
    IAC_HIP(hipGetLastError());
    return IAC_OK;
}

int iac_merge_prepare(const float *rot9, const float *mean_intensity, uint32_t nev, const double *small_cq,
                      size_t nsmall, float *rw10, double *mult_out)
{
    if (!rot9 || !mean_intensity || !small_cq || !rw10 || !mult_out || nev == 0 || nsmall == 0)
        return iac::fail(IAC_ERR_INVALID_ARG, "null input");
    double max_weight = 0.0;
    for (uint32_t i = 0; i < nev; i++) {
        for (int k = 0; k < 9; k++) rw10[10 * (size_t)i + k] = rot9[9 * (size_t)i + k];
        rw10[10 * (size_t)i + 9] = (float)((double)mean_intensity[i] * (double)mean_intensity[i]);
        if (mean_intensity[i] > max_weight) max_weight = mean_intensity[i];
    }
    double t = 0;
    for (size_t i = 0; i < nsmall; i++) t += small_cq[i];
    const double mean_cq = t / nsmall;
    double m = 1e-12;
    for (; 1 > max_weight * max_weight * mean_cq * m;) m *= 10;
    uint64_t oom = 1;
    for (; oom < (uint64_t)nev;) oom *= 10;
    m = m / oom;
    m *= 1e10;
    if (m > 0.6) m = std::round(m);
    if (m < 1 && m > 0.1) m = 1;
    if (m < 1e-12) m = 1e-12;
    for (uint32_t i = 0; i < nev; i++) {
        float red = (float)m;
        if (m > 0.6) red = std::round((float)m);
        float w = rw10[10 * (size_t)i + 9];
        w *= red;
        w = std::floor((float)((double)w + 0.5));
        rw10[10 * (size_t)i + 9] = w / red;
    }
    *mult_out = m;
    return IAC_OK;
}

static int merge_launch(iac_ctx *ctx, const double *d_small_cq, bool per_event, const iac_mesh_shape *small_shape,
                        const float *d_rw10, uint32_t nev, int interp, double mult, uint64_t *d_big)
{
    IAC_TRY(iac::bind(ctx));
    IAC_TRY(check_small(small_shape));
    if (!d_small_cq || !d_rw10 || !d_big) return iac::fail(IAC_ERR_INVALID_ARG, "null pointer");
    if (interp != IAC_NEAREST && interp != IAC_LINEAR) return iac::fail(IAC_ERR_INVALID_ARG, "bad interpolation");
    if (nev == 0) return IAC_OK;
    const size_t nsmall = (size_t)small_shape->size_ab * small_shape->size_ab * small_shape->size_c;
    const size_t stride = per_event ? nsmall : (size_t)0;
    const int sab = (int)small_shape->size_ab, sc = (int)small_shape->size_c;
    const int ka = (int)small_shape->k_a, kb = (int)small_shape->k_b, kc = (int)small_shape->k_c;
    auto *big = reinterpret_cast<unsigned long long *>(d_big);
    // Bricks cost a fixed time and a little each before their first candidate, scattered adds cost by
    // their number.  Whole calls, scattered and in bricks: 944,000 adds of 53 x 53 x 7 (196 bricks)
    // 34 and 35 us, 1,258,000 46 and 36; 855,000 of 89 x 89 x 3 (864) 33 and 35, 1,140,000 42 and 40;
    // 1,341,000 of 193 x 193 x 3 (8,125) 44 and 42, 1,788,000 60 and 45.  96 linear events of
    // 65 x 65 x 3, 129 x 129 x 3 and 193 x 193 x 3: 409, 1,358 and 2,521 us scattered, 74, 186 and 292
    // in bricks.  The candidate ranges are 16 bits.
    const uint64_t nbx = (sab + kBrX - 1) / kBrX, nby = (sab + kBrY - 1) / kBrY, nbz = (sab + kBrZ - 1) / kBrZ;
    const uint64_t nbricks = nbx * nby * nbz;
    const uint64_t cus = (uint64_t)std::max(1, ctx->num_cus);
    const uint64_t least = nbricks >= 8 * cus ? 600000 + 75 * nbricks : (nbricks >= cus ? 850000 : 1200000);
    const bool bricks = (uint64_t)nev * nsmall * (interp ? 8 : 1) >= least && sab < 32768 && sc < 32768 &&
                        nbricks < (1u << 31);
    const dim3 rest((unsigned)((nsmall + 255) / 256), (nev + kRestEvents - 1) / kRestEvents);
    IAC_TRY(iac::timer_begin(ctx));
    if (bricks) {
        // Fewer bricks than eight per CU: blocks of fewer events, so that there are about as many (share:
        // of the events, those that reach a brick, on average).  64 linear events of 31 x 31 x 7 (32
        // bricks): 167 us with 64 each, 50 so (107 scattered); 96 nearest of 129 x 129 x 3 (2,601): 69 and 71.
        const double share = std::min(1.0, 1.3 * (11 + sc / 2) / (0.5 * sab));
        const double per = nev * share * nbricks / (8.0 * cus);
        const uint32_t least_log2 = nbricks >= 4 * cus ? kBrickEventsLeast + 2 : kBrickEventsLeast;
        uint32_t per_log2 = kBrickEvents;
        if (nbricks < 8 * cus)
            while (per_log2 > least_log2 && per < (double)(1u << per_log2)) per_log2--;
        const dim3 grid((unsigned)nbricks, std::min<uint32_t>(65535, (nev >> per_log2) + 1));
        hipLaunchKernelGGL(interp ? merge_brick_kernel<true> : merge_brick_kernel<false>, grid, dim3(256), 0,
                           ctx->stream, d_small_cq, stride, sab, sc, ka, kb, kc, d_rw10, nev, per_log2, mult, (int)nbx,
                           (int)nby, big);
        IAC_HIP(hipGetLastError());
    }
    auto kern = interp ? (bricks ? merge_rest_kernel<true, true> : merge_rest_kernel<true, false>)
                       : (bricks ? merge_rest_kernel<false, true> : merge_rest_kernel<false, false>);
    hipLaunchKernelGGL(kern, rest, dim3(256), 0, ctx->stream, d_small_cq, stride, sab, sc, ka, kb, kc, d_rw10, nev, mult,
                       big, ctx->d_counters);
    IAC_HIP(hipGetLastError());
    IAC_TRY(iac::timer_end(ctx));
    return IAC_OK;
}

int iac_merge_cq(iac_ctx *ctx, const double *d_small_cq, const iac_mesh_shape *small_shape, const float *d_rw10,
                 uint32_t nev, int interp, double mult, uint64_t *d_big)
{
    return merge_launch(ctx, d_small_cq, false, small_shape, d_rw10, nev, interp, mult, d_big);
}

int iac_merge_cq_multi(iac_ctx *ctx, const double *d_small_meshes, const iac_mesh_shape *small_shape,
                       const float *d_rw10, uint32_t nev, int interp, double mult, uint64_t *d_big)
{
    return merge_launch(ctx, d_small_meshes, true, small_shape, d_rw10, nev, interp, mult, d_big);
}

int iac_merge_ac_cq(iac_ctx *ctx, const uint64_t *d_ac, const double *d_cq, size_t n, double *d_out)
{
    IAC_TRY(iac::bind(ctx));
    if (!d_ac || !d_cq || !d_out) return iac::fail(IAC_ERR_INVALID_ARG, "null pointer");
    if (n == 0) return IAC_OK;
    hipLaunchKernelGGL(merge_ac_cq_kernel, dim3(blocks_for(n)), dim3(256), 0, ctx->stream,
                       reinterpret_cast<const unsigned long long *>(d_ac), d_cq, n, d_out);
    IAC_HIP(hipGetLastError());
    return IAC_OK;
}

}  // extern "C"
