// iac_pairs.hip -- the LDS cell-box pair engine shared by the 3D AC_uw path
// (Detector::AutoCorrelateSparseList) and the dense C(q) path
// (AutoCorr_CQ_small, IAC/kernel.cl:27-184).
//
// Input: photon or pixel records {kx, ky, kz, value} of nframes frames; frames
// form groups (frame range -> one output mesh each).  Three ways to take the pairs, to the same
// bits: detector strips (AC_uw nearest neighbour, runs of many pairs; "AC_uw strips" below), region
// tiles (dense C(q) images; "Region tiles" below), and the cell-offset walk for the rest:
//   1. plan (cached): the k-map's extents define a cell grid over its two
//      widest k axes (cell side `cell_vox` voxels); per-cell k extents bound
//      the voxel box reached by the pairs of every cell offset delta.
//   2. cell_sort: per frame, counting sort of its records by cell, dropping
//      zero-valued records (they add nothing in any mode), and the record count
//      of its fullest cell; in symmetric mode the frame's self-pair value is
//      summed for its group.
//   3. pairs: one block per (delta [, region of cells], chunk of frames of one
//      group).  The block privatises delta's voxel box in LDS across the chunk
//      and bins
//        symmetric modes: each unordered pair of distinct records once
//          (deltas of the positive half plane; within-cell pairs for 0),
//        ordered modes: every ordered pair (all deltas; self pairs in 0),
//      flushing the box with one atomic per nonzero voxel.  A pair outside
//      the box adds to global memory directly, except on in-box tasks of the
//      AC_uw specialised path, whose exact box provably holds every pair.
//      Work inside a block goes by groups of (frame, cell) items: the items'
//      pair counts are scanned (32-bit), then AC_uw runs walk the group's pairs
//      with the lanes of a wave on consecutive pairs (coalesced record loads)
//      and C(q) runs give each thread a contiguous pair range (either on
//      request).  A chunk with a frame whose fullest cell could push a group
//      past 2^32 pairs bins its items one after another instead.
//   4. symmetric modes: mesh[v] += H[v] + H[mirror v], centre += self.
// Nearest-neighbour binning is odd in q (iac_binning.h): the (b,a) pair lands
// on the point reflection of (a,b) with the same value, so step 4 restores
// the ordered-pair mesh exactly.  Linear modes are not odd and run ordered.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "iac_binning.h"
#include "iac_internal.h"
#include "iac_pairs.h"

#pragma clang fp contract(off)

namespace iac {
namespace {

constexpr int kBlock = 256;
// LDS box capacity (uint64 voxels): 4096 (32 KiB, 1024 items per scan group, 3 blocks
// per CU), 1920 (15 KiB, 512 items: 25.9 KB in all, so 6 blocks per CU) or 1024 (8 KiB,
// 512 items); chosen per plan.  1920 holds the tight boxes of 6-voxel cells (at most
// 1,859 voxels on a 1024^2 detector).
constexpr int kBoxMax = 4096;
constexpr int kBoxSmall = 1920;
constexpr int kBoxTiny = 1024;
// waves per SIMD the specialised-path kernels are compiled for: 6 keeps them within
// 85 VGPRs (no spills) so that 6 blocks fit a CU
template <bool FAST, int BOX>
struct Occupancy {
    static constexpr int blocks = FAST && BOX != kBoxMax ? 6 : 1;
};
template <int BOX>
struct BoxCfg {
    static constexpr int group = BOX == kBoxMax ? 1024 : 512;  // items per scan group
    static constexpr int ipt = group / kBlock;                  // items per thread
};
constexpr int kMaxCells = 4096;                    // NC_u * NC_v
// blocks per pair-kernel launch (tasks x chunks): 2^22 blocks of 256 threads keep
// the grid's work-item count far below 2^32; longer runs launch in chunk slices
constexpr uint32_t kMaxGridBlocks = 1u << 22;

struct CellGeom {
    int au, av;    // k axes spanned by the cell grid
    float u0, v0;  // grid origin
    float inv_wu;  // 1 / cell width along u (k units)
    float inv_wv;  // 1 / cell width along v
    int ncu, ncv;  // cells per axis
};

struct Task {
    int du, dv;         // cell offset delta (u, v)
    int iu0, iv0;       // first cell i whose partner i - delta is on the grid
    int nu, nv;         // extent of that cell range
    int bx0, by0, bz0;  // LDS box origin (voxel indices)
    int bx, by, bz;     // LDS box extent; bx == 0 -> no box, every add goes to global
    int inbox;          // the box lies inside the mesh: every nearest-neighbour pair lands in it
    int allin;          // the task's q box lies inside the cut sphere: no pair fails the cut
};

struct Chunk {
    uint32_t f0, f1, group;
};

__device__ __forceinline__ uint32_t fkey(float f)
{
    const uint32_t b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

inline float unkey(uint32_t k)
{
    uint32_t b = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
    float f;
    std::memcpy(&f, &b, 4);
    return f;
}

__device__ __forceinline__ int cell_of(const CellGeom &g, float ku, float kv)
{
    int cu = (int)floorf((ku - g.u0) * g.inv_wu);
    int cv = (int)floorf((kv - g.v0) * g.inv_wv);
    cu = min(max(cu, 0), g.ncu - 1);
    cv = min(max(cv, 0), g.ncv - 1);
    return cv * g.ncu + cu;
}

__device__ __forceinline__ float comp(const float4 &r, int a) { return a == 0 ? r.x : (a == 1 ? r.y : r.z); }

// q = u / d, r = u % d for u < 2^24, d >= 1, from the float reciprocal inv = 1.0f / d:
// the estimate is within one of the quotient, one correction step makes it exact.
__device__ __forceinline__ void divmod24(uint32_t u, uint32_t d, float inv, uint32_t &q, uint32_t &r)
{
    uint32_t t = (uint32_t)((float)u * inv);
    int32_t m = (int32_t)(u - __umul24(t, d));
    if (m < 0) {
        t--;
        m += (int32_t)d;
    } else if (m >= (int32_t)d) {
        t++;
        m -= (int32_t)d;
    }
    q = t;
    r = (uint32_t)m;
}

// (int)roundf(x) (half away from zero) for |x| < 2^23: x + copysign(0.49999997f, x)
// rounded to nearest, truncated.  Equal to roundf for every float in that range
// (checked exhaustively over all 2.5e9 of them); 3 instructions instead of 7.
__device__ __forceinline__ int round_away(float x)
{
    return (int)(x + copysignf(0.49999997f, x));
}

// round_away of an x in [0, 2^22) in one instruction: v_cvt_rpi_i32_f32 is floor(x + 1/2) without an
// intermediate rounding (checked over all floats of that range)
__device__ __forceinline__ int round_up(float x)
{
    int r;
    asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

// pair_val with the integer fast path in a 24-bit multiply
__device__ __forceinline__ uint32_t pair_val_small(float p)
{
    if (p >= 0.0f && p < 21054.0f && p == truncf(p)) return __umul24((uint32_t)p, 1000u);
    return pair_val(p);
}

// AC_uw with a double map, a linear first level and the identity rotation: a pair's
// eight first-level corners are its voxels.  A linear second level over such an
// integral corner keeps one corner of weight 1 (Sep = 1), valued FloatToInt(double)
// of the corner's float value; a nearest one takes FloatToInt(float).
__host__ __device__ __forceinline__ bool lin_first_identity(const BinParams &P)
{
    return P.double_map && P.interp1 == 1 && P.rot_identity;
}

// the value of a symmetric AC_uw pair: FloatToInt(float), or FloatToInt(double)
// for a linear second level over an integral first-level voxel (BinParams::dval)
__device__ __forceinline__ uint32_t sym_val(const BinParams &P, float p)
{
    return P.dval ? pair_val_d((double)p) : pair_val_small(p);
}

// ---- binning policies -------------------------------------------------------

// C(q) fixed point of AutoCorr_CQ_small (kernel.cl:93-101): (ulong)((double)(Ia*Ib) * M),
// pairs below 1e-37f skipped.
__device__ __forceinline__ bool cq_value(const PairSpec &S, float p, double &val)
{
    val = (double)p;
    return !(val < (double)1e-37f);
}

// Symmetric (nearest-neighbour) binning of one pair: voxel + value.
template <int KIND>
__device__ __forceinline__ bool bin_sym(const PairSpec &S, const float4 &a, const float4 &b, int &fs,
                                        int &ms, int &ss, uint64_t &v)
{
    if (KIND == kKindAc3d) {
        int dx, dy, dz;
        if (!bin_nn(a.x, a.y, a.z, b.x, b.y, b.z, S.P, S.R, dx, dy, dz)) return false;
        v = sym_val(S.P, a.w * b.w);
        fs = dx + S.P.c0;
        ms = dy + S.P.c1;
        ss = dz + S.P.c2;
        return true;
    } else {
        double val;
        if (!cq_value(S, a.w * b.w, val)) return false;
        float q[3] = {a.x - b.x, a.y - b.y, a.z - b.z};
        const float s = (q[0] * q[0] + q[1] * q[1]) + q[2] * q[2];
        if (!(s < S.P.cut_sq)) return false;
        q[0] = q[0] * S.P.vox;
        q[1] = q[1] * S.P.vox;
        q[2] = q[2] * S.P.vox;
        fs = (int)(roundf(q[S.ka]) + (float)S.P.c0);
        ms = (int)(roundf(q[S.kb]) + (float)S.P.c1);
        ss = (int)(roundf(q[S.kc]) + (float)S.P.c2);
        v = (uint64_t)(val * S.mult);
        return true;
    }
}

template <int KIND>
__device__ __forceinline__ uint64_t self_value(const PairSpec &S, float c)
{
    if (KIND == kKindAc3d) return sym_val(S.P, c * c);
    double val;
    return cq_value(S, c * c, val) ? (uint64_t)(val * S.mult) : 0ull;
}

// Ordered (linear-mode) binning of one pair into a sink.
template <int KIND, class Sink>
__device__ __forceinline__ void bin_ordered(const PairSpec &S, const float4 &a, const float4 &b, Sink &sink)
{
    if (KIND == kKindAc3d) {
        add_q_entry(sink, a.x, a.y, a.z, b.x, b.y, b.z, a.w * b.w, S.P, S.R);
    } else {
        double val;
        if (!cq_value(S, a.w * b.w, val)) return;
        float q[3] = {a.x - b.x, a.y - b.y, a.z - b.z};
        const float s = (q[0] * q[0] + q[1] * q[1]) + q[2] * q[2];
        if (!(s < S.P.cut_sq)) return;
        q[0] = q[0] * S.P.vox;
        q[1] = q[1] * S.P.vox;
        q[2] = q[2] * S.P.vox;
        if (S.interp == 0) {
            sink.add((int)(roundf(q[S.ka]) + (float)S.P.c0), (int)(roundf(q[S.kb]) + (float)S.P.c1),
                     (int)(roundf(q[S.kc]) + (float)S.P.c2), (uint64_t)(val * S.mult));
            return;
        }
        // kernel.cl:136-181: `1 - (q - floor(q))` in float, weights in double
        const float qa = q[S.ka], qb = q[S.kb], qc = q[S.kc];
        const double sfs = (double)(1.0f - (qa - floorf(qa)));
        const double sms = (double)(1.0f - (qb - floorf(qb)));
        const double sss = (double)(1.0f - (qc - floorf(qc)));
        const int fs = (int)(floorf(qa) + (float)S.P.c0);
        const int ms = (int)(floorf(qb) + (float)S.P.c1);
        const int ss = (int)(floorf(qc) + (float)S.P.c2);
        const double vm = val * S.mult;
        sink.add(fs + 0, ms + 0, ss + 0, (uint64_t)(vm * ((sfs * sms) * sss)));
        sink.add(fs + 0, ms + 0, ss + 1, (uint64_t)(vm * ((sfs * sms) * (1 - sss))));
        sink.add(fs + 1, ms + 0, ss + 0, (uint64_t)(vm * (((1 - sfs) * sms) * sss)));
        sink.add(fs + 1, ms + 0, ss + 1, (uint64_t)(vm * (((1 - sfs) * sms) * (1 - sss))));
        sink.add(fs + 0, ms + 1, ss + 0, (uint64_t)(vm * ((sfs * (1 - sms)) * sss)));
        sink.add(fs + 0, ms + 1, ss + 1, (uint64_t)(vm * ((sfs * (1 - sms)) * (1 - sss))));
        sink.add(fs + 1, ms + 1, ss + 0, (uint64_t)(vm * (((1 - sfs) * (1 - sms)) * sss)));
        sink.add(fs + 1, ms + 1, ss + 1, (uint64_t)(vm * (((1 - sfs) * (1 - sms)) * (1 - sss))));
    }
}

// ---- small kernels -------------------------------------------------------------

__global__ void fill_u32_kernel(uint32_t *p, uint32_t v, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = v;
}

__global__ void fill_u64_kernel(unsigned long long *p, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = 0ull;
}

// per-cell extents start empty: min keys at the top, max keys at the bottom
__global__ void init_cell_ext_kernel(uint32_t *ext, int ncell)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c < ncell)
        for (int d = 0; d < 3; d++) {
            ext[6 * c + d] = 0xffffffffu;
            ext[6 * c + 3 + d] = 0u;
        }
}

// the k-map's extents start empty; what dense_scan_kernel counts starts at none, its flags at 1
__global__ void cq_begin_kernel(uint32_t *ext, unsigned long long *kept, uint32_t *plain)
{
    if (threadIdx.x < 6) ext[threadIdx.x] = threadIdx.x < 3 ? 0xffffffffu : 0u;
    if (threadIdx.x < 2) plain[threadIdx.x] = 1u;
    if (threadIdx.x == 0) kept[0] = 0ull;
}

// min/max of each k component: ext[0..2] min keys, ext[3..5] max keys, reduced over the block: all
// blocks' atomics fall on these six words (one per wave took 20 us for 16,384 pixels, so 2 us)
__global__ void __launch_bounds__(256) kext_kernel(const float *__restrict__ kmap, uint32_t npix, uint32_t *ext)
{
    __shared__ uint32_t red[4][6];
    uint32_t m[6] = {0xffffffffu, 0xffffffffu, 0xffffffffu, 0u, 0u, 0u};
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < npix; i += gridDim.x * blockDim.x)
        for (int d = 0; d < 3; d++) {
            const uint32_t k = fkey(kmap[3 * (size_t)i + d]);
            m[d] = min(m[d], k);
            m[3 + d] = max(m[3 + d], k);
        }
    for (int d = 0; d < 6; d++)
        for (int o = 32; o > 0; o >>= 1) {
            const uint32_t v = (uint32_t)__shfl_xor(m[d], o, 64);
            m[d] = d < 3 ? min(m[d], v) : max(m[d], v);
        }
    if ((threadIdx.x & 63u) == 0)
        for (int d = 0; d < 6; d++) red[threadIdx.x >> 6][d] = m[d];
    __syncthreads();
    if (threadIdx.x < 6) {
        const int d = threadIdx.x;
        uint32_t v = red[0][d];
        for (int w = 1; w < 4; w++) v = d < 3 ? min(v, red[w][d]) : max(v, red[w][d]);
        if (d < 3) atomicMin(ext + d, v);
        else atomicMax(ext + d, v);
    }
}

// per-cell k extents: ext[6c + d] min key of component d, ext[6c + 3 + d] max key.
// LDS: the block's extents of every cell (6 ncell keys, dynamic), merged into ext with one
// atomic per touched cell and key.  A thread takes four pixels in a row and adds the extents of
// those in one cell together: the pixels of a wave lie in few cells, whose words its lanes share.
__global__ void __launch_bounds__(256)
    cell_ext_lds_kernel(const float *__restrict__ kmap, uint32_t npix, CellGeom g, uint32_t *ext)
{
    extern __shared__ uint32_t sext[];
    const int ncell = g.ncu * g.ncv;
    for (int c = threadIdx.x; c < ncell; c += blockDim.x)
        for (int d = 0; d < 3; d++) {
            sext[6 * c + d] = 0xffffffffu;
            sext[6 * c + 3 + d] = 0u;
        }
    __syncthreads();
    const uint64_t step = 4ull * gridDim.x * blockDim.x;
    for (uint64_t i0 = 4ull * (blockIdx.x * blockDim.x + threadIdx.x); i0 < npix; i0 += step) {
        int cell = -1;
        uint32_t m[6];
        auto put = [&]() {
            if (cell < 0) return;
            for (int d = 0; d < 3; d++) {
                atomicMin(sext + 6 * cell + d, m[d]);
                atomicMax(sext + 6 * cell + 3 + d, m[3 + d]);
            }
        };
        for (uint64_t i = i0; i < min(i0 + 4, (uint64_t)npix); i++) {
            const float k[3] = {kmap[3 * i], kmap[3 * i + 1], kmap[3 * i + 2]};
            const int c = cell_of(g, k[g.au], k[g.av]);
            const bool same = c == cell;
            if (!same) put();
            for (int d = 0; d < 3; d++) {
                const uint32_t key = fkey(k[d]);
                m[d] = same ? min(m[d], key) : key;
                m[3 + d] = same ? max(m[3 + d], key) : key;
            }
            cell = c;
        }
        put();
    }
    __syncthreads();
    for (int c = threadIdx.x; c < ncell; c += blockDim.x)
        if (sext[6 * c] != 0xffffffffu)
            for (int d = 0; d < 3; d++) {
                atomicMin(ext + 6 * c + d, sext[6 * c + d]);
                atomicMax(ext + 6 * c + 3 + d, sext[6 * c + 3 + d]);
            }
}

// the same with global atomics only (grids too large for the LDS copy)
__global__ void cell_ext_kernel(const float *__restrict__ kmap, uint32_t npix, CellGeom g, uint32_t *ext)
{
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < npix; i += gridDim.x * blockDim.x) {
        const float k[3] = {kmap[3 * (size_t)i], kmap[3 * (size_t)i + 1], kmap[3 * (size_t)i + 2]};
        const int c = cell_of(g, k[g.au], k[g.av]);
        for (int d = 0; d < 3; d++) {
            atomicMin(ext + 6 * c + d, fkey(k[d]));
            atomicMax(ext + 6 * c + 3 + d, fkey(k[d]));
        }
    }
}

// One block per frame: counting sort of the frame's nonzero records by cell.
// cs[f*(ncell+1) + c] = first sorted position of cell c relative to off[f];
// cs[f*(ncell+1) + ncell] = number of kept records; cmax[f] = records of the
// frame's fullest cell.  In symmetric mode the frame's self-pair values are added
// to self[group of f].  paths: the passes taken by this walk, then by strips.
template <int KIND, bool ORD>
__global__ void __launch_bounds__(kBlock)
    cell_sort_kernel(const float4 *__restrict__ rec, const uint64_t *__restrict__ off, CellGeom g,
                     float4 *__restrict__ srec, uint32_t *__restrict__ cs, PairSpec S,
                     const uint32_t *__restrict__ group_off, uint32_t ngroups,
                     unsigned long long *__restrict__ self, uint32_t *__restrict__ wflag,
                     uint32_t *__restrict__ cmax, const uint32_t *__restrict__ strips,
                     unsigned long long *__restrict__ paths)
{
    const bool by_strips = strips && strips[0];
    if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(paths + (by_strips ? 1 : 0), 1ull);
    if (by_strips) return;
    __shared__ uint32_t cnt[kMaxCells];
    __shared__ uint32_t part[kBlock];
    __shared__ unsigned long long sred[kBlock / 64];
    __shared__ uint32_t smax[kBlock / 64];
    const uint32_t f = blockIdx.x;
    const int ncell = g.ncu * g.ncv;
    const uint64_t base = off[f];
    const uint32_t n = (uint32_t)(off[f + 1] - base);
    for (int c = threadIdx.x; c < ncell; c += kBlock) cnt[c] = 0;
    __syncthreads();
    unsigned long long sv = 0;
    bool small = true;  // every kept weight an integer in [1, 129]
    for (uint32_t i = threadIdx.x; i < n; i += kBlock) {
        const float4 r = rec[base + i];
        if (r.w == 0.0f) continue;
        atomicAdd(&cnt[cell_of(g, comp(r, g.au), comp(r, g.av))], 1u);
        if (!ORD) sv += self_value<KIND>(S, r.w);
        small = small && r.w >= 1.0f && r.w <= 129.0f && r.w == truncf(r.w);
    }
    if (!small) wflag[0] = 0u;  // the run's flag starts at 1
    if (!ORD) {
        for (int o = 32; o > 0; o >>= 1) sv += __shfl_down(sv, o, 64);
        if ((threadIdx.x & 63) == 0) sred[threadIdx.x >> 6] = sv;
    }
    __syncthreads();
    if (!ORD && threadIdx.x == 0) {
        unsigned long long t = 0;
        for (int w = 0; w < kBlock / 64; w++) t += sred[w];
        if (t) {
            uint32_t lo = 0, hi = ngroups;  // group of f: largest gi with group_off[gi] <= f
            while (hi - lo > 1) {
                const uint32_t mid = (lo + hi) >> 1;
                if (group_off[mid] <= f) lo = mid; else hi = mid;
            }
            atomicAdd(self + lo, t);
        }
    }
    // exclusive scan of cnt[0..ncell)
    const int per = (ncell + kBlock - 1) / kBlock;
    const int c0 = min(ncell, (int)threadIdx.x * per), c1 = min(ncell, c0 + per);
    uint32_t s = 0, m = 0;
    for (int c = c0; c < c1; c++) {
        s += cnt[c];
        m = max(m, cnt[c]);
    }
    part[threadIdx.x] = s;
    for (int o = 32; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_down(m, o, 64));
    if ((threadIdx.x & 63) == 0) smax[threadIdx.x >> 6] = m;
    __syncthreads();
    for (int o = 1; o < kBlock; o <<= 1) {
        const uint32_t v = threadIdx.x >= (unsigned)o ? part[threadIdx.x - o] : 0u;
        __syncthreads();
        part[threadIdx.x] += v;
        __syncthreads();
    }
    uint32_t run = threadIdx.x ? part[threadIdx.x - 1] : 0u;
    uint32_t *csf = cs + (size_t)f * (ncell + 1);
    for (int c = c0; c < c1; c++) {
        const uint32_t v = cnt[c];
        csf[c] = run;
        cnt[c] = run;  // becomes the scatter cursor
        run += v;
    }
    if (threadIdx.x == kBlock - 1) csf[ncell] = part[kBlock - 1];
    if (threadIdx.x == 0) cmax[f] = max(max(smax[0], smax[1]), max(smax[2], smax[3]));
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n; i += kBlock) {
        const float4 r = rec[base + i];
        if (r.w == 0.0f) continue;
        const uint32_t pos = atomicAdd(&cnt[cell_of(g, comp(r, g.au), comp(r, g.av))], 1u);
        srec[base + pos] = r;
    }
}

// mesh[g][v] += H[g][v] + H[g][last - v]; the centre also receives self[g].
__global__ void symmetrize_kernel(const unsigned long long *__restrict__ H, unsigned long long *__restrict__ mesh,
                                  size_t nvox, uint32_t ngroups, size_t centre,
                                  const unsigned long long *__restrict__ self,
                                  const unsigned long long *__restrict__ strip_self,
                                  const uint32_t *__restrict__ strips)
{
    if (strips && strips[0]) self = strip_self;
    const size_t last = nvox - 1, total = nvox * ngroups;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const size_t gi = i / nvox, v = i - gi * nvox;
        const unsigned long long *h = H + gi * nvox;
        unsigned long long add = h[v] + h[last - v];
        if (v == centre) add += self[gi];
        if (add) mesh[i] += add;
    }
}

// A first-level voxel (mesh coordinates of the identity binning) under the frame's
// rotation: Atomic_Add_rotated_q_Entry's nearest second level (ACMesh.cpp:319-336)
// applied to the float voxel offsets, which equal the first level's roundf(q vox).
__device__ __forceinline__ void rotate_voxel(const float *r, int c0, int c1, int c2, int &fs, int &ms, int &ss)
{
    float q0 = (float)(fs - c0), q1 = (float)(ms - c1), q2 = (float)(ss - c2);
    rotate3(q0, q1, q2, r);
    fs = (int)roundf(q0) + c0;
    ms = (int)roundf(q1) + c1;
    ss = (int)roundf(q2) + c2;
}

struct BoxSink {
    unsigned long long *box;  // LDS
    unsigned long long *out;  // global mesh (group's H or mesh)
    unsigned long long *dropped;
    int bx0, by0, bz0, bx, by, bz;
    int S, SC;
    unsigned long long drop_weight;
    const float *rot;  // the chunk's rotation of first-level voxels, or null
    int c0, c1, c2;
    // an add outside the LDS box: the mesh voxel under the chunk's rotation, or the dropped
    // count when it leaves the mesh.  Target and value by selection, one atomic: nested
    // divergent branches here kept values live across the whole group loop (spills).
    __device__ __forceinline__ void add_outside(int fs, int ms, int ss, uint64_t v)
    {
        if (rot) rotate_voxel(rot, c0, c1, c2, fs, ms, ss);
        const bool ok = (unsigned)fs < (unsigned)S && (unsigned)ms < (unsigned)S && (unsigned)ss < (unsigned)SC;
        const size_t idx = ok ? (size_t)fs + (size_t)ms * S + (size_t)ss * S * S : 0;
        atomicAdd(ok ? out + idx : dropped, ok ? (unsigned long long)v : drop_weight);
    }
    __device__ __forceinline__ void add(int fs, int ms, int ss, uint64_t v)
    {
        if (!v) return;
        const unsigned lx = (unsigned)(fs - bx0), ly = (unsigned)(ms - by0), lz = (unsigned)(ss - bz0);
        if (lx < (unsigned)bx && ly < (unsigned)by && lz < (unsigned)bz)
            atomicAdd(box + lx + (size_t)bx * (ly + (size_t)by * lz), (unsigned long long)v);
        else
            add_outside(fs, ms, ss, v);
    }
};

// Pairs [p0, p0 + left) of a group on the specialised path (AC_uw, symmetric
// nearest-neighbour binning, identity rotation), records read from `src` (the
// LDS stage, or the sorted records in global memory).  Software pipelined: the
// next pair's records are requested before this pair is binned.  INBOX: every
// pair lands in the LDS box -- its voxel range covers the rounded q range of the
// task and lies inside the mesh -- so there is no bounds test and the box offset
// is two 24-bit multiply-adds on byte strides; otherwise the bounds test and the
// global sink.  SMALL: every weight of the run is an integer in [1, 129], so the
// fixed-point value 1000 wa wb (below 2^24) is exactly (1000 wa) * wb in float.
template <bool SMALL, bool INBOX>
__device__ __forceinline__ void fast_pairs(const float4 *__restrict__ src, const uint4 *item, const uint32_t *pre,
                                           int u, uint4 d, uint32_t ia, uint32_t ib, uint32_t left, bool tri,
                                           const PairSpec &S, unsigned long long *box, const Task &T,
                                           BoxSink &sink)
{
    const int fox = S.P.c0 - T.bx0, foy = S.P.c1 - T.by0, foz = S.P.c2 - T.bz0;
    const int bx8 = 8 * T.bx, bxby8 = 8 * T.bx * T.by;
    const int c8 = 8 * fox + bx8 * foy + bxby8 * foz;
    const float vox = S.P.vox, cut_sq = S.P.cut_sq;
    float4 ra = src[d.x + ia];
    float4 rb = src[d.z + ib];
    uint32_t bi = d.z + ib, bend = d.z + (tri ? d.y : d.w);
    char *const boxb = reinterpret_cast<char *>(box);
    for (;;) {
        const float4 ca = ra, cb = rb;
        if (left > 1) {
            if (++bi == bend) {  // row of a done: next a, or the next item with pairs
                ia++;
                uint32_t nb = tri ? ia + 1 : 0;
                if ((tri ? nb : ia) >= d.y) {
                    do {
                        u++;
                    } while (pre[u + 1] == pre[u]);
                    d = item[u];
                    ia = 0;
                    nb = tri ? 1 : 0;
                }
                ra = src[d.x + ia];
                bi = d.z + nb;
                bend = d.z + (tri ? d.y : d.w);
            }
            rb = src[bi];
        }
        asm volatile("" ::"v"(cb.w));  // one 16-byte load
        const float q0 = ca.x - cb.x, q1 = ca.y - cb.y, q2 = ca.z - cb.z;
        const float sq = (q0 * q0 + q1 * q1) + q2 * q2;
        if (sq < cut_sq) {
            const int dx = round_away(q0 * vox);
            const int dy = round_away(q1 * vox);
            const int dz = round_away(q2 * vox);
            const uint32_t v = SMALL ? (uint32_t)((ca.w * 1000.0f) * cb.w) : pair_val_small(ca.w * cb.w);
            if (INBOX) {
                const int o = __mul24(dz, bxby8) + (__mul24(dy, bx8) + (dx * 8 + c8));
                atomicAdd(reinterpret_cast<unsigned long long *>(boxb + o), (unsigned long long)v);
            } else {
                const uint32_t lx = (uint32_t)(dx + fox), ly = (uint32_t)(dy + foy), lz = (uint32_t)(dz + foz);
                if (lx < (uint32_t)T.bx && ly < (uint32_t)T.by && lz < (uint32_t)T.bz)
                    atomicAdd(box + lx + __umul24(ly, (uint32_t)T.bx) + __umul24(lz, (uint32_t)(T.bx * T.by)),
                              (unsigned long long)v);
                else
                    sink.add(dx + S.P.c0, dy + S.P.c1, dz + S.P.c2, v);
            }
        }
        if (--left == 0) break;
    }
}

template <bool INBOX>
__device__ __forceinline__ void fast_pairs_w(bool small, const float4 *__restrict__ src, const uint4 *item,
                                             const uint32_t *pre, int u, uint4 d, uint32_t ia, uint32_t ib,
                                             uint32_t left, bool tri, const PairSpec &S, unsigned long long *box,
                                             const Task &T, BoxSink &sink)
{
    if (small)
        fast_pairs<true, INBOX>(src, item, pre, u, d, ia, ib, left, tri, S, box, T, sink);
    else
        fast_pairs<false, INBOX>(src, item, pre, u, d, ia, ib, left, tri, S, box, T, sink);
}

// Pair r (row-major, ia < ib) of the distinct unordered pairs of n records.
__device__ __forceinline__ void tri_decode(uint32_t r, uint32_t n, uint32_t &ia, uint32_t &ib)
{
    // rows before row a: S(a) = a (2n - a - 1) / 2; a = the largest with S(a) <= r
    const double b = 2.0 * n - 1.0;
    uint32_t a = (uint32_t)fmax(0.0, floor((b - sqrt(fmax(0.0, b * b - 8.0 * (double)r))) * 0.5));
    auto S = [n](uint64_t x) { return x * (2ull * n - x - 1) / 2; };
    while (a > 0 && S(a) > r) a--;
    while (S(a + 1) <= r) a++;
    ia = a;
    ib = a + 1 + (uint32_t)(r - S(a));
}

// Phase 2 of a group on the specialised path with lanes on consecutive pairs:
// wave w walks the pair range [w0, w1) 64 at a time, lane l on pair P + l, so the
// records a wave loads lie in the few rows those 64 pairs span rather than in
// 64 unrelated rows (one or two cache lines per load instead of up to 64).
//
// Item lookup: the group's items are compacted (every item has pairs, so item
// starts are distinct) and followed by 64 sentinel starts (~0).  The starts in
// [P, P + 64) tag their positions with P in a per-wave LDS row; a lane's item is
// the item before the step plus the number of tagged positions up to the lane
// (ballot + mbcnt, the count's base and the next step's item in scalar registers).
//
// Division: a non-triangle item carries h = RN(1 / (2 nb)) in place of na and -nb
// in place of nb, and ia = trunc(f32(2r + 1) * h) is exactly r / nb for every
// r < 2^22: (r + 1/2) / nb lies at least 1 / (2 nb) from the integers, and the two
// roundings move it by at most (r + 1/2) / nb * 2^-23.  A group of more than 2^22
// pairs takes a correction step (below 2^24) or divides in integers.
//
// Records are read at 32-bit byte offsets from the chunk's first record, one step
// ahead of the binning.  Lanes past the range read a real pair (their position
// clamped to the group's last pair) and do not bin.
// a volatile LDS word: cross-lane tags stay LDS accesses, in program order
typedef volatile __attribute__((address_space(3))) uint32_t lds_tag_t;

// The binning: FASTBIN, the AC_uw specialised inline path (SMALL and INBOX apply
// there); otherwise bin_ordered for ordered runs and bin_sym for symmetric ones.
// EXACT: the group divides by h (non-triangle, at most 2^22 pairs); otherwise the
// triangle decode, or the reciprocal 2h with one correction step below 2^24 pairs,
// or an integer division.  CUT: FASTBIN tests the cut (false on an all-in task).
template <int KIND, bool ORD, bool FASTBIN, bool SMALL, bool INBOX, bool EXACT, bool CUT = true>
__device__ __forceinline__ void fast_walk(const float4 *__restrict__ src, const uint4 *item, const uint32_t *pre,
                                          uint32_t u0, uint32_t w0, uint32_t w1, uint32_t total, bool tri,
                                          const PairSpec &S, unsigned long long *box, const Task &T, BoxSink &sink,
                                          lds_tag_t *fl)
{
    const uint32_t lane = threadIdx.x & 63u;
    // wave-uniform values in scalar registers
    w0 = __builtin_amdgcn_readfirstlane(w0);
    w1 = __builtin_amdgcn_readfirstlane(w1);
    const uint32_t last = __builtin_amdgcn_readfirstlane(total) - 1u;
    uint32_t ub = __builtin_amdgcn_readfirstlane(u0);  // the item before the step's first start
    const int fox = S.P.c0 - T.bx0, foy = S.P.c1 - T.by0, foz = S.P.c2 - T.bz0;
    const int bx8 = 8 * T.bx, bxby8 = 8 * T.bx * T.by;
    const int c8 = 8 * fox + bx8 * foy + bxby8 * foz;
    // C(q): byte stride of the mesh axis that record component i bins along (k_a -> fs, k_b -> ms, k_c -> ss)
    const int cst0 = S.ka == 0 ? 8 : (S.kb == 0 ? bx8 : bxby8);
    const int cst1 = S.ka == 1 ? 8 : (S.kb == 1 ? bx8 : bxby8);
    const int cst2 = S.ka == 2 ? 8 : (S.kb == 2 ? bx8 : bxby8);
    const float vox = S.P.vox, cut_sq = S.P.cut_sq;
    const char *const srcb = reinterpret_cast<const char *>(src);
    char *const boxb = reinterpret_cast<char *>(box);

    fl[lane] = ~0u;  // untagged: a tag is a pair index, below 2^32 - 1
    // the item of pair P + lane; ub moves to the item of pair P + 63
    auto item_at = [&](uint32_t P) -> uint32_t {
        const uint32_t t = pre[ub + 1u + lane] - P;
        if (t < 64u) fl[t] = P;
        const uint64_t starts = __ballot(fl[lane] == P);
        const uint32_t base = ub + (uint32_t)(starts & 1ull);
        ub += (uint32_t)__popcll(starts);
        return __builtin_amdgcn_mbcnt_hi((uint32_t)(starts >> 33),
                                         __builtin_amdgcn_mbcnt_lo((uint32_t)(starts >> 1), base));
    };
    // the descriptor and first pair of the item of pair P + lane, a step before its decode
    struct Ahead {
        uint4 d;
        uint32_t pu;
    };
    auto lookup = [&](uint32_t P) -> Ahead {
        const uint32_t u = item_at(P);
        return Ahead{item[u], pre[u]};
    };
    // byte offsets of the two records of pair min(P + lane, last), which item A holds
    auto decode = [&](const Ahead &A, uint32_t P, uint32_t &oa, uint32_t &ob) {
        const uint4 d = A.d;
        const uint32_t r = min(P + lane, last) - A.pu;
        uint32_t ia, ib;
        if (EXACT) {
            // d.w = -nb: b's record index d.z + r - ia nb in one 24-bit multiply-add
            // (ia, nb <= r < 2^22)
            ia = (uint32_t)((float)(2u * r + 1u) * __uint_as_float(d.y));
            oa = (d.x + ia) << 4;
            ob = (uint32_t)(__mul24((int)ia, (int)d.w) + (int)(d.z + r)) << 4;
            return;
        }
        if (tri) {
            tri_decode(r, d.y, ia, ib);
        } else if (last < (1u << 24)) {
            divmod24(r, 0u - d.w, 2.0f * __uint_as_float(d.y), ia, ib);  // 2h = RN(1 / nb)
        } else {
            const uint32_t nb = 0u - d.w;
            ia = r / nb;
            ib = r - ia * nb;
        }
        oa = (d.x + ia) << 4;
        ob = (d.z + ib) << 4;
    };
    auto load = [&](uint32_t o) { return *reinterpret_cast<const float4 *>(srcb + o); };

    auto bin = [&](const float4 &ca, const float4 &cb, bool active) {
        if (FASTBIN) {
            asm volatile("" ::"v"(cb.w), "v"(ca.w));  // 16-byte loads
            const float q0 = ca.x - cb.x, q1 = ca.y - cb.y, q2 = ca.z - cb.z;
            const float sq = (q0 * q0 + q1 * q1) + q2 * q2;
            const bool in = active && (!CUT || sq < cut_sq);
            if (INBOX && SMALL) {
                // every pair of an in-box task (lanes past the range read pairs of the same task)
                // lands in the box: branch-free, a lane outside the range or the cut adds 0, so
                // the step is one basic block and the next step's item lookup interleaves with it
                const int dx = round_away(q0 * vox);
                const int dy = round_away(q1 * vox);
                const int dz = round_away(q2 * vox);
                const uint32_t v = (uint32_t)((ca.w * 1000.0f) * cb.w);
                const int o = __mul24(dz, bxby8) + (__mul24(dy, bx8) + (dx * 8 + c8));
                atomicAdd(reinterpret_cast<unsigned long long *>(boxb + o), (unsigned long long)(in ? v : 0u));
                return;
            }
            if (in) {
                const int dx = round_away(q0 * vox);
                const int dy = round_away(q1 * vox);
                const int dz = round_away(q2 * vox);
                const uint32_t v = SMALL ? (uint32_t)((ca.w * 1000.0f) * cb.w) : pair_val_small(ca.w * cb.w);
                if (INBOX) {
                    const int o = __mul24(dz, bxby8) + (__mul24(dy, bx8) + (dx * 8 + c8));
                    atomicAdd(reinterpret_cast<unsigned long long *>(boxb + o), (unsigned long long)v);
                } else {
                    const uint32_t lx = (uint32_t)(dx + fox), ly = (uint32_t)(dy + foy), lz = (uint32_t)(dz + foz);
                    if (lx < (uint32_t)T.bx && ly < (uint32_t)T.by && lz < (uint32_t)T.bz)
                        atomicAdd(box + lx + __umul24(ly, (uint32_t)T.bx) + __umul24(lz, (uint32_t)(T.bx * T.by)),
                                  (unsigned long long)v);
                    else if (v)
                        sink.add_outside(dx + S.P.c0, dy + S.P.c1, dz + S.P.c2, v);
                }
            }
            return;
        }
        if (!active) return;
        if (ORD && KIND == kKindAc3d && INBOX) {
            // a linear first level (identity) on a task whose box holds every corner: add_q_entry's
            // eight corners at one base byte offset plus constant strides, their values
            // ((v wx) wy) wz from a product tree in the same order
            const float q0 = ca.x - cb.x, q1 = ca.y - cb.y, q2 = ca.z - cb.z;
            const float sq = (q0 * q0 + q1 * q1) + q2 * q2;
            if (sq < cut_sq) {
                const float x0 = q0 * vox, x1 = q1 * vox, x2 = q2 * vox;
                const float f0 = floorf(x0), f1 = floorf(x1), f2 = floorf(x2);
                const double s0 = 1.0 - (double)(x0 - f0), s1 = 1.0 - (double)(x1 - f1);
                const double s2 = 1.0 - (double)(x2 - f2);
                const double v = (double)(ca.w * cb.w);
                const double vx[2] = {v * s0, v * (1 - s0)};
                const int o = __mul24((int)f2, bxby8) + (__mul24((int)f1, bx8) + ((int)f0 * 8 + c8));
                auto corners = [&](auto dval_c) {
                    constexpr bool kDouble = decltype(dval_c)::value;  // linear second level
#pragma unroll
                    for (int c = 0; c < 8; c++) {
                        const int ex = c & 1, ey = (c >> 1) & 1, ez = (c >> 2) & 1;
                        const double w = (vx[ex] * (ey ? 1 - s1 : s1)) * (ez ? 1 - s2 : s2);
                        const uint32_t u = kDouble ? pair_val_d((double)(float)w) : pair_val((float)w);
                        if (u)
                            atomicAdd(
                                reinterpret_cast<unsigned long long *>(boxb + o + ex * 8 + ey * bx8 + ez * bxby8),
                                (unsigned long long)u);
                    }
                };
                if (S.P.interp2) corners(std::true_type{}); else corners(std::false_type{});
            }
        } else if (ORD) {
            // ordered runs (linear second level): every corner through the checked box
            bin_ordered<KIND>(S, ca, cb, sink);
        } else if (KIND == kKindCq && INBOX) {
            // C(q) of a task whose box holds every voxel its pairs reach: the bin of
            // bin_sym (its value and axis order: round(q[ka] vox) + c0 is round_away
            // of the same product plus c0) as one byte offset, component i scaled by
            // the box stride of the mesh axis it maps to
            asm volatile("" ::"v"(cb.w), "v"(ca.w));  // 16-byte loads
            const float w = ca.w * cb.w;
            const float q0 = ca.x - cb.x, q1 = ca.y - cb.y, q2 = ca.z - cb.z;
            const float sq = (q0 * q0 + q1 * q1) + q2 * q2;
            if (sq < cut_sq && !(w < 1e-37f)) {
                const int o = __mul24(round_away(q2 * vox), cst2) +
                              (__mul24(round_away(q1 * vox), cst1) + (__mul24(round_away(q0 * vox), cst0) + c8));
                atomicAdd(reinterpret_cast<unsigned long long *>(boxb + o),
                          (unsigned long long)(uint64_t)((double)w * S.mult));
            }
        } else {
            // C(q) through the checked box, or the general symmetric binning
            int fs, ms, ss;
            uint64_t v;
            if (bin_sym<KIND>(S, ca, cb, fs, ms, ss, v)) sink.add(fs, ms, ss, v);
        }
    };

    // two steps per iteration, the next step's records in flight while one bins.  The
    // look-ahead is unconditional (past the range it reads the group's last pair, or the
    // next wave's), and so is the second step (past the range no lane bins): a load
    // behind a branch, or a second exit, would make the binning wait for the loads in
    // flight too.  The scheduling barriers keep the binning's first use of its records
    // after the issue of the next step's loads.
    // lane of step P in range: with the exact division every pair index stays below
    // 2^22 + 192, so P + lane cannot wrap (one compare on the decode's own sum)
    auto active = [&](uint32_t P) { return EXACT ? P + lane < w1 : lane < (w1 > P ? w1 - P : 0u); };
    uint32_t oa, ob;
    decode(lookup(w0), w0, oa, ob);
    float4 a0 = load(oa), b0 = load(ob);
    Ahead A = lookup(w0 + 64u);
    for (uint32_t P = w0;; P += 128u) {
        decode(A, P + 64u, oa, ob);
        const float4 a1 = load(oa), b1 = load(ob);
        __builtin_amdgcn_sched_barrier(0);
        A = lookup(P + 128u);
        bin(a0, b0, active(P));
        decode(A, P + 128u, oa, ob);
        a0 = load(oa);
        b0 = load(ob);
        __builtin_amdgcn_sched_barrier(0);
        A = lookup(P + 192u);
        bin(a1, b1, active(P + 64u));
        if (P + 128u >= w1) break;
    }
}

template <int KIND, bool ORD, bool FAST>
__device__ __forceinline__ void fast_walk_w(bool small, bool inbox, bool exact, const float4 *__restrict__ src,
                                            const uint4 *item, const uint32_t *pre, uint32_t u0, uint32_t w0,
                                            uint32_t w1, uint32_t total, bool tri, const PairSpec &S,
                                            unsigned long long *box, const Task &T, BoxSink &sink, lds_tag_t *fl)
{
    // the triangle task and groups of more than 2^22 pairs: one general instance (the
    // checked box and the general value), so the rare decodes add one walk loop, not four
    if (!exact) {
        fast_walk<KIND, ORD, FAST, false, false, false>(src, item, pre, u0, w0, w1, total, tri, S, box, T, sink, fl);
        return;
    }
    auto go = [&](auto fastbin_c, auto small_c, auto inbox_c) {
        constexpr bool kFastbin = decltype(fastbin_c)::value, kSmall = decltype(small_c)::value;
        constexpr bool kInbox = decltype(inbox_c)::value;
        fast_walk<KIND, ORD, kFastbin, kSmall, kInbox, true>(src, item, pre, u0, w0, w1, total, tri, S, box, T, sink,
                                                             fl);
    };
    using T_ = std::true_type;
    using F_ = std::false_type;
    if (!FAST) {
        if (((KIND == kKindCq && !ORD && S.interp == 0) || (KIND == kKindAc3d && ORD && lin_first_identity(S.P))) &&
            inbox)
            go(F_{}, F_{}, T_{});
        else
            go(F_{}, F_{}, F_{});
    } else if (inbox) {
        if (small && T.allin)  // the headline case: no cut test
            fast_walk<KIND, ORD, true, true, true, true, false>(src, item, pre, u0, w0, w1, total, tri, S, box, T,
                                                                sink, fl);
        else if (small) go(T_{}, T_{}, T_{});
        else go(T_{}, F_{}, T_{});
    } else {
        if (small) go(T_{}, T_{}, F_{});
        else go(T_{}, F_{}, F_{});
    }
}

// PF: 0 lanes on consecutive pairs (the walk), 1 a pair range per thread, pair by
// pair, 4 or 8 a range per thread in batches of PF pairs.  BEHIND: enqueued behind strips, whose
// flag ends it; a variant of its own, because the test costs the others 1.2 % (762 -> 771 us for 112
// frames of 756 photons).
template <int KIND, bool ORD, int PF, bool FAST, int BOX, bool BEHIND = false>
__global__ void __launch_bounds__(kBlock, (Occupancy<FAST, BOX>::blocks))
    pairs_kernel(const float4 *__restrict__ srec, const uint64_t *__restrict__ off,
                 const uint32_t *__restrict__ cs, const Chunk *__restrict__ chunks,
                 const Task *__restrict__ tasks, uint32_t ntasks, CellGeom g, PairSpec S,
                 unsigned long long *__restrict__ target, size_t nvox,
                 unsigned long long *__restrict__ dropped, const uint32_t *__restrict__ wflag,
                 const float *__restrict__ rots, const uint32_t *__restrict__ cmax,
                 const uint32_t *__restrict__ strips)
{
    if (BEHIND && strips[0]) return;  // the strips took the run
    constexpr int kGroup = BoxCfg<BOX>::group;
    constexpr int kItemsPerThread = BoxCfg<BOX>::ipt;
    __shared__ unsigned long long box[BOX];
    __shared__ uint4 item[kGroup];         // {a base, na (walk: h), b base, nb}, bases from the chunk's first record
    __shared__ uint32_t pre[kGroup + 64];  // exclusive prefix of pair counts (walk: then 64 sentinels)
    __shared__ uint32_t wtot[kBlock / 64];
    __shared__ uint32_t wnz[kBlock / 64];         // walk: items with pairs per wave
    __shared__ uint32_t wtags[kBlock / 64][64];   // walk: item-start tags per wave
    __shared__ uint32_t wfirst[kBlock / 64];      // walk: the item holding each wave's first pair
    __shared__ uint32_t s_total;                  // walk: pairs of the group
    __shared__ uint32_t s_heavy[kBlock / 64];     // per wave: the chunk holds an item of 2^32 / kGroup pairs or more

    const Task T = tasks[blockIdx.x % ntasks];
    const Chunk CH = chunks[blockIdx.x / ntasks];
    // the chunk's records: item bases count from its first record, so record byte
    // offsets stay below 2^32 (a chunk holds far fewer than 2^28 records)
    const uint64_t rec0 = off[CH.f0];
    const float4 *__restrict__ crec = srec + rec0;
    const int ncell = g.ncu * g.ncv;
    const bool zero_delta = (T.du == 0 && T.dv == 0);
    const bool tri = !ORD && zero_delta;  // distinct unordered pairs within a cell

    // per-frame rotations: a chunk holds frames of one rotation, applied to first-level voxels
    const float *crot = rots ? rots + 9 * (size_t)CH.f0 : nullptr;
    BoxSink sink{box, target + (size_t)CH.group * nvox, dropped, T.bx0, T.by0, T.bz0, T.bx, T.by, T.bz,
                 S.P.sab, S.P.sc, ORD ? 1ull : 2ull, crot, S.P.c0, S.P.c1, S.P.c2};
    const int vbox = T.bx * T.by * T.bz;
    const int fox = S.P.c0 - T.bx0, foy = S.P.c1 - T.by0, foz = S.P.c2 - T.bz0;  // fast path offsets
    const uint32_t fbxby = (uint32_t)(T.bx * T.by);
    // in-box tasks: the AC_uw specialised path, or symmetric nearest-neighbour C(q) (tight boxes)
    const bool inbox = (FAST || (KIND == kKindCq && !ORD && S.interp == 0) ||
                        (KIND == kKindAc3d && ORD && lin_first_identity(S.P))) &&
                       T.inbox != 0;
    const bool small = FAST && wflag[0] != 0u;
    // in-box C(q) on a pair range per thread: byte strides of the box axis each record
    // component bins along, and the centre's byte offset in the box
    const int cbx8 = 8 * T.bx, cbxby8 = 8 * T.bx * T.by;
    const int cc8 = 8 * fox + cbx8 * foy + cbxby8 * foz;
    const int cst0 = S.ka == 0 ? 8 : (S.kb == 0 ? cbx8 : cbxby8);
    const int cst1 = S.ka == 1 ? 8 : (S.kb == 1 ? cbx8 : cbxby8);
    const int cst2 = S.ka == 2 ? 8 : (S.kb == 2 ? cbx8 : cbxby8);
    char *const cboxb = reinterpret_cast<char *>(box);
    // pair counts and prefixes are 32-bit: a group of kGroup items each holding fewer
    // than 2^32 / kGroup pairs stays below 2^32.  A frame whose fullest cell holds M
    // records has items of at most M^2 pairs.
    constexpr uint64_t kHeavy = (1ull << 32) / kGroup;
    bool hv = false;
    for (uint32_t f = CH.f0 + threadIdx.x; f < CH.f1; f += kBlock) hv = hv || (uint64_t)cmax[f] * cmax[f] >= kHeavy;
    const bool whv = __ballot(hv) != 0ull;
    if ((threadIdx.x & 63u) == 0) s_heavy[threadIdx.x >> 6] = whv;
    for (int v = threadIdx.x; v < vbox; v += kBlock) box[v] = 0ull;
    __syncthreads();
    const bool heavy = (s_heavy[0] | s_heavy[1] | s_heavy[2] | s_heavy[3]) != 0u;

    // items (frame, cell) of the chunk: fewer than 2^24 (at most 4096 frames x 4096 cells),
    // so quotients come from a float reciprocal with one correction step
    const uint32_t cells = (uint32_t)T.nu * (uint32_t)T.nv;
    const uint32_t nitems = (CH.f1 - CH.f0) * cells;
    const float inv_cells = 1.0f / (float)cells, inv_nu = 1.0f / (float)T.nu;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    // lanes on consecutive pairs (every mode unless a pair range per thread is asked for)
    constexpr bool walking = PF == 0;
    if (heavy) {
        // items one after another, each a grid of rows along its shorter side (triangle
        // items: row a, columns b > a) with the block's threads along a row and four
        // record loads in flight per thread; general binning through the checked box
        for (uint32_t u = 0; u < nitems; u++) {
            uint32_t fr, rem, row, col;
            divmod24(u, cells, inv_cells, fr, rem);
            divmod24(rem, (uint32_t)T.nu, inv_nu, row, col);
            const uint32_t f = CH.f0 + fr;
            const int iv = T.iv0 + (int)row, iu = T.iu0 + (int)col;
            const int ci = iv * g.ncu + iu;
            const int cj = (iv - T.dv) * g.ncu + (iu - T.du);
            const uint32_t *csf = cs + (size_t)f * (ncell + 1);
            const uint32_t base = (uint32_t)(off[f] - rec0);
            const uint32_t a0 = base + csf[ci], na = csf[ci + 1] - csf[ci];
            const uint32_t b0 = base + csf[cj], nb = csf[cj + 1] - csf[cj];
            const bool by_a = tri || na <= nb;  // rows are a records, columns b records
            const uint32_t nrow = by_a ? na : nb, ncol = by_a ? nb : na;
            const uint32_t rbase = by_a ? a0 : b0, cbase = by_a ? b0 : a0;
            if (ncol == 0) continue;
            for (uint32_t r = 0; r < nrow; r++) {
                const float4 rr = crec[rbase + r];
                for (uint32_t c = (tri ? r + 1 : 0) + threadIdx.x; c < ncol; c += 4 * kBlock) {
                    float4 rc[4];
#pragma unroll
                    for (int k = 0; k < 4; k++) rc[k] = crec[cbase + min(c + k * kBlock, ncol - 1)];
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        if (c + k * kBlock >= ncol) break;
                        const float4 &ra = by_a ? rr : rc[k];
                        const float4 &rb = by_a ? rc[k] : rr;
                        if (ORD) {
                            bin_ordered<KIND>(S, ra, rb, sink);
                        } else {
                            int fs, ms, ss;
                            uint64_t v;
                            if (bin_sym<KIND>(S, ra, rb, fs, ms, ss, v)) sink.add(fs, ms, ss, v);
                        }
                    }
                }
            }
        }
        __syncthreads();  // the box is complete before the flush
    }
    for (uint32_t ub = 0; ub < (heavy ? 0u : nitems); ub += kGroup) {
        // phase 1: item descriptors and pair counts (contiguous items per thread)
        uint32_t mycnt[kItemsPerThread];
        uint4 myd[kItemsPerThread];
        uint32_t tsum = 0, nz = 0;
#pragma unroll
        for (int k = 0; k < kItemsPerThread; k++) {
            const uint32_t li = threadIdx.x * kItemsPerThread + k;
            const uint32_t u = ub + li;
            uint4 d = make_uint4(0, 0, 0, 0);
            uint32_t c = 0;
            if (u < nitems) {
                uint32_t fr, rem, row, col;
                divmod24(u, cells, inv_cells, fr, rem);
                divmod24(rem, (uint32_t)T.nu, inv_nu, row, col);
                const uint32_t f = CH.f0 + fr;
                const int iv = T.iv0 + (int)row, iu = T.iu0 + (int)col;
                const int ci = iv * g.ncu + iu;
                const int cj = (iv - T.dv) * g.ncu + (iu - T.du);
                const uint32_t *csf = cs + (size_t)f * (ncell + 1);
                const uint32_t base = (uint32_t)(off[f] - rec0);
                const uint32_t a0 = csf[ci], na = csf[ci + 1] - a0;
                const uint32_t b0 = csf[cj], nb = csf[cj + 1] - b0;
                d = make_uint4(base + a0, na, base + b0, nb);
                c = tri ? na * (na - 1) / 2 : na * nb;
                // the walk decodes (ia, ib) of a non-triangle item with h = RN(1 / (2 nb)) in
                // place of na (2 nb is exact in float: nb < 2^24) and -nb in place of nb
                if (walking && !tri && c) {
                    d.y = __float_as_uint(1.0f / (float)(2u * nb));
                    d.w = 0u - nb;
                }
            }
            if (!walking) item[li] = d;
            myd[k] = d;
            mycnt[k] = c;
            tsum += c;
            nz += c ? 1u : 0u;
        }
        // block exclusive scan of the per-thread sums: within each wave by shuffles,
        // then across the four waves through LDS (two barriers)
        uint32_t x = tsum, z = nz;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o, 64);
            const uint32_t yz = walking ? __shfl_up(z, o, 64) : 0u;
            if (lane >= (uint32_t)o) {
                x += y;
                z += yz;
            }
        }
        if (lane == 63) {
            wtot[wave] = x;
            wnz[wave] = z;
        }
        __syncthreads();
        if (walking) {
            // items with pairs only, in order: item starts become distinct
            uint32_t run = x - tsum, rz = z - nz, tot = 0, nzt = 0;
            for (uint32_t w = 0; w < kBlock / 64; w++) {
                if (w < wave) {
                    run += wtot[w];
                    rz += wnz[w];
                }
                tot += wtot[w];
                nzt += wnz[w];
            }
#pragma unroll
            for (int k = 0; k < kItemsPerThread; k++) {
                if (mycnt[k]) {
                    // the item holding the first pair of waves 1..3 (the walk splits the
                    // group's pairs in quarters)
                    for (uint32_t w = 1; w < kBlock / 64; w++) {
                        const uint32_t first = (uint32_t)(((uint64_t)tot * w) / (kBlock / 64));
                        if (first >= run && first - run < mycnt[k]) wfirst[w] = rz;
                    }
                    item[rz] = myd[k];
                    pre[rz] = run;
                    rz++;
                    run += mycnt[k];
                }
            }
            if (threadIdx.x < 64) pre[nzt + threadIdx.x] = ~0u;  // sentinel starts
            if (threadIdx.x == 0) {
                wfirst[0] = 0;
                s_total = tot;
            }
        } else {
            uint32_t run = x - tsum;
            for (uint32_t w = 0; w < wave; w++) run += wtot[w];
#pragma unroll
            for (int k = 0; k < kItemsPerThread; k++) {
                pre[threadIdx.x * kItemsPerThread + k] = run;
                run += mycnt[k];
            }
            if (threadIdx.x == kBlock - 1) pre[kGroup] = run;
        }
        __syncthreads();

        // phase 2: thread t bins the contiguous pair range [p0, p1).  PF == 1: pair
        // by pair, one load each.  PF > 1: PF pairs at a time with an integer-only
        // enumeration, so the 2 PF record loads of a batch are in flight together.
        const uint32_t total = walking ? s_total : pre[kGroup];
        if (walking) {
            // waves on quarters of the group's pairs, lanes on consecutive pairs
            const uint32_t w0 = (uint32_t)(((uint64_t)total * wave) / (kBlock / 64));
            const uint32_t w1 = (uint32_t)(((uint64_t)total * (wave + 1)) / (kBlock / 64));
            if (w0 < w1)
                fast_walk_w<KIND, ORD, FAST>(small, inbox, !tri && total <= (1u << 22), crec, item, pre, wfirst[wave],
                                             w0, w1, total, tri, S, box, T, sink, (lds_tag_t *)wtags[wave]);
            __syncthreads();
            continue;
        }
        const uint32_t p0 = (uint32_t)(((uint64_t)total * threadIdx.x) / kBlock);
        const uint32_t p1 = (uint32_t)(((uint64_t)total * (threadIdx.x + 1)) / kBlock);
        if (p0 < p1) {
            int lo = 0, hi = kGroup;  // the item holding p0: largest u with pre[u] <= p0
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (pre[mid] <= p0) lo = mid; else hi = mid;
            }
            int u = lo;
            uint4 d = item[u];
            uint32_t r = p0 - pre[u];
            uint32_t ia, ib;
            if (tri) {
                ia = 0;
                while (r >= d.y - 1 - ia) {
                    r -= d.y - 1 - ia;
                    ia++;
                }
                ib = ia + 1 + r;
            } else {
                ia = r / d.w;
                ib = r % d.w;
            }
            if (FAST && inbox) {
                fast_pairs_w<true>(small, crec, item, pre, u, d, ia, ib, p1 - p0, tri, S, box, T, sink);
            } else if (PF == 1) {
                // one record load per pair: the a record stays in a register along its row
                float4 ra = crec[d.x + ia];
                // in-box C(q): consecutive pairs of a row fall in runs on one voxel, so
                // a run's values add in a register and reach the box in one atomic
                int co = -1;
                unsigned long long cacc = 0;
                for (uint32_t p = p0;;) {
                    const float4 rb = crec[d.z + ib];
                    if (KIND == kKindCq && !ORD && inbox) {
                        asm volatile("" ::"v"(rb.w));  // one 16-byte load
                        const float w = ra.w * rb.w;
                        const float q0 = ra.x - rb.x, q1 = ra.y - rb.y, q2 = ra.z - rb.z;
                        const float sq = (q0 * q0 + q1 * q1) + q2 * q2;
                        if (sq < S.P.cut_sq && !(w < 1e-37f)) {
                            const int o = __mul24(round_away(q2 * S.P.vox), cst2) +
                                          (__mul24(round_away(q1 * S.P.vox), cst1) +
                                           (__mul24(round_away(q0 * S.P.vox), cst0) + cc8));
                            const unsigned long long v = (uint64_t)((double)w * S.mult);
                            if (o == co) {
                                cacc += v;
                            } else {
                                if (co >= 0) atomicAdd(reinterpret_cast<unsigned long long *>(cboxb + co), cacc);
                                co = o;
                                cacc = v;
                            }
                        }
                    } else if (FAST) {
                        // identity rotation, nearest neighbour: round(round(x)) == round(x), so every
                        // symmetric mode bins at (int)roundf(q * vox); box index in 24-bit multiplies
                        asm volatile("" ::"v"(rb.w));  // one 16-byte load, not xyz now and w later
                        const float q0 = ra.x - rb.x, q1 = ra.y - rb.y, q2 = ra.z - rb.z;
                        const float sq = (q0 * q0 + q1 * q1) + q2 * q2;
                        if (sq < S.P.cut_sq) {
                            const int dx = round_away(q0 * S.P.vox);
                            const int dy = round_away(q1 * S.P.vox);
                            const int dz = round_away(q2 * S.P.vox);
                            const uint64_t v = pair_val_small(ra.w * rb.w);
                            const uint32_t lx = (uint32_t)(dx + fox), ly = (uint32_t)(dy + foy),
                                           lz = (uint32_t)(dz + foz);
                            if (lx < (uint32_t)T.bx && ly < (uint32_t)T.by && lz < (uint32_t)T.bz)
                                atomicAdd(box + lx + __umul24(ly, (uint32_t)T.bx) + __umul24(lz, fbxby),
                                          (unsigned long long)v);
                            else
                                sink.add(dx + S.P.c0, dy + S.P.c1, dz + S.P.c2, v);
                        }
                    } else if (ORD) {
                        bin_ordered<KIND>(S, ra, rb, sink);
                    } else {
                        int fs, ms, ss;
                        uint64_t v;
                        if (bin_sym<KIND>(S, ra, rb, fs, ms, ss, v)) sink.add(fs, ms, ss, v);
                    }
                    if (++p == p1) break;
                    ib++;
                    if (ib >= (tri ? d.y : d.w)) {
                        ia++;
                        ib = tri ? ia + 1 : 0;
                        if ((tri ? ib : ia) >= d.y) {  // item exhausted: next item with pairs
                            do {
                                u++;
                            } while (pre[u + 1] == pre[u]);
                            d = item[u];
                            ia = 0;
                            ib = tri ? 1 : 0;
                        }
                        ra = crec[d.x + ia];
                    }
                }
                if (co >= 0) atomicAdd(reinterpret_cast<unsigned long long *>(cboxb + co), cacc);
            } else
            for (uint32_t p = p0; p < p1;) {
                const uint32_t nb = min((uint32_t)PF, p1 - p);
                float4 A[PF > 1 ? PF : 1], B[PF > 1 ? PF : 1];
#pragma unroll
                for (int k = 0; k < PF; k++) {
                    if ((uint32_t)k < nb) {
                        A[k] = crec[d.x + ia];
                        B[k] = crec[d.z + ib];
                        if (p + k + 1 < p1) {  // a next pair exists: advance the enumeration
                            ib++;
                            if (ib >= (tri ? d.y : d.w)) {
                                ia++;
                                ib = tri ? ia + 1 : 0;
                                if ((tri ? ib : ia) >= d.y) {  // item exhausted: next item with pairs
                                    do {
                                        u++;
                                    } while (pre[u + 1] == pre[u]);
                                    d = item[u];
                                    ia = 0;
                                    ib = tri ? 1 : 0;
                                }
                            }
                        }
                    }
                }
#pragma unroll
                for (int k = 0; k < PF; k++) {
                    if ((uint32_t)k < nb) {
                        if (ORD) {
                            bin_ordered<KIND>(S, A[k], B[k], sink);
                        } else {
                            int fs, ms, ss;
                            uint64_t v;
                            if (bin_sym<KIND>(S, A[k], B[k], fs, ms, ss, v)) sink.add(fs, ms, ss, v);
                        }
                    }
                }
                p += nb;
            }
        }
        __syncthreads();
    }

    // flush the LDS box (under the chunk's rotation, voxel by voxel: every pair of a box
    // voxel shares its first-level voxel, so the rotated second level bins them alike)
    unsigned long long *out = target + (size_t)CH.group * nvox;
    float rr[9];
    int ax = 0;  // the box axis consecutive lanes walk
    if (crot) {
        for (int i = 0; i < 9; i++) rr[i] = crot[i];
        // the axis whose rotated image moves most along the mesh's fast axis, so that
        // neighbouring lanes add to neighbouring voxels (one L2 request per 64-byte segment
        // a wave instruction touches)
        const float a0 = fabsf(rr[0]), a1 = fabsf(rr[1]), a2 = fabsf(rr[2]);
        ax = a1 > a0 ? (a2 > a1 ? 2 : 1) : (a2 > a0 ? 2 : 0);
    }
    const int e0 = ax == 0 ? T.bx : (ax == 1 ? T.by : T.bz), e1 = ax == 0 ? T.by : T.bx;
    for (int v = threadIdx.x; v < vbox; v += kBlock) {
        const int i0 = v % e0, rest = v / e0, i1 = rest % e1, i2 = rest / e1;
        const int lx = ax == 0 ? i0 : i1, ly = ax == 1 ? i0 : (ax == 0 ? i1 : i2), lz = ax == 2 ? i0 : i2;
        const unsigned long long x = box[lx + T.bx * (ly + T.by * lz)];
        if (x) {
            int fs = T.bx0 + lx, ms = T.by0 + ly, ss = T.bz0 + lz;
            if (crot) {
                rotate_voxel(rr, S.P.c0, S.P.c1, S.P.c2, fs, ms, ss);
                if ((unsigned)fs >= (unsigned)S.P.sab || (unsigned)ms >= (unsigned)S.P.sab ||
                    (unsigned)ss >= (unsigned)S.P.sc) {
                    atomicAdd(dropped, 1ull);  // excluded by the caller's bound check
                    continue;
                }
            }
            atomicAdd(out + (size_t)fs + (size_t)ms * S.P.sab + (size_t)ss * S.P.sab * S.P.sab, x);
        }
    }
}

// ---- dense C(q): region tiles -----------------------------------------------------
//
// Dense images hold many records per voxel, so the cell-offset tasks above spend their time on
// index work and on neighbouring pairs adding to one LDS word (20.6 ms for the 9.6e9 pairs of a
// 384 x 360 image into 129 x 129 x 3).  Here a task is a pair of regions (I, J) of the detector,
// up to 12 x 12 voxels each, whose whole range of q fits the LDS box: a wave owns 64 records of
// I, one per lane, spread evenly over the region so that they fall on different voxels, and takes
// J's records one by one from the scalar unit.  A pair is then its binning and nothing else:
// about 24 VALU instructions nearest, 67 linear.  Measured: the image above 20.6 -> 5.6 ms
// (nearest: VALU issue), 191 x 173 into 97 x 97 x 3 linear 14.6 -> 5.4 ms (bound by its eight LDS
// adds per pair, 23 clocks each: two or three of the 64 lanes share a voxel).

struct TileTask {
    int ci, cj;         // the regions of the a and b records; nearest neighbour: ci <= cj
    int bx0, by0, bz0;  // LDS box origin (voxel indices) and extent, as in Task
    int bx, by, bz;
    int inbox;  // every voxel the task's pairs add to lies in the box
    int allin;  // no pair fails the cut
    int sa, sb;  // the sign of q along the mesh's first two axes: 1 or -1, 0 where it varies
};

constexpr int kTileB = 16;  // b records per unit of work
constexpr int kTileParts = 144;  // voxel-sized parts of a region, at most
// b records per scalar load batch, unrolled: a linear pair's eight corners are work enough for the
// scheduler, and more of them spill
template <bool LINEAR>
struct TileBatch {
    static constexpr int n = LINEAR ? 2 : 8;
};

typedef float f4v __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) f4v *scalar_rec_t;
typedef const __attribute__((address_space(4))) uint32_t *scalar_u32_t;
typedef const __attribute__((address_space(4))) uint64_t *scalar_u64_t;

// The sort key of a k: its region, then its voxel-sized part of the region (side x side parts,
// so records of one region that lie far apart in its order lie on different voxels).
__device__ __forceinline__ uint32_t tile_key(const CellGeom &g, int side, float ku, float kv)
{
    const float xu = (ku - g.u0) * g.inv_wu, xv = (kv - g.v0) * g.inv_wv;
    const int cu = min(max((int)floorf(xu), 0), g.ncu - 1), cv = min(max((int)floorf(xv), 0), g.ncv - 1);
    const int su = min(max((int)((xu - (float)cu) * (float)side), 0), side - 1);
    const int sv = min(max((int)((xv - (float)cv) * (float)side), 0), side - 1);
    return (uint32_t)((cv * g.ncu + cu) * side + sv) * (uint32_t)side + (uint32_t)su;
}

// The nonzero values of all frames, counted into kept, and the run's flags: plain[0] is cleared by
// any value that could make a pair negative, NaN or 2^32 or more, plain[1] by one that could
// make it negative, NaN or 2^62 or more.  Bound: one read of the frames.
__global__ void __launch_bounds__(kBlock)
    dense_scan_kernel(const float *__restrict__ frames, uint64_t n, double mult, unsigned long long *__restrict__ kept,
                      uint32_t *__restrict__ plain)
{
    __shared__ unsigned long long kred[kBlock / 64];
    unsigned long long c = 0;
    bool ok = true, wide = 1e-37 * mult < 0.99;  // a product below 1e-37 adds nothing either way
    const uint64_t step = (uint64_t)gridDim.x * kBlock;
#pragma unroll 4
    for (uint64_t p = (uint64_t)blockIdx.x * kBlock + threadIdx.x; p < n; p += step) {
        const float I = frames[p];
        const double most = (double)(I * I) * mult;
        c += I != 0.0f ? 1u : 0u;
        ok = ok && (I == 0.0f || most < 4294967296.0);
        wide = wide && (I == 0.0f || (I > 0.0f && most < 0x1p62));
    }
    if (!ok || !wide) plain[0] = 0u;
    if (!wide) plain[1] = 0u;
    for (int o = 32; o > 0; o >>= 1) c += __shfl_down(c, o, 64);
    if ((threadIdx.x & 63) == 0) kred[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        c = 0;
        for (int w = 0; w < kBlock / 64; w++) c += kred[w];
        if (c) atomicAdd(kept, c);
    }
}

// Counts of the frames' nonzero pixels per key (cs, zeroed by the caller) and the groups' self
// values (symmetric modes).  Grid: ns blocks per frame.
template <bool ORD>
__global__ void __launch_bounds__(kBlock)
    tile_count_kernel(const float *__restrict__ kmap, const float *__restrict__ frames, uint32_t npix, uint32_t ns,
                      CellGeom g, int side, PairSpec S, const uint32_t *__restrict__ group_off, uint32_t ngroups,
                      uint32_t *__restrict__ cs, unsigned long long *__restrict__ self)
{
    __shared__ unsigned long long sred[kBlock / 64];
    const uint32_t f = blockIdx.x / ns;
    const size_t nkey = (size_t)g.ncu * g.ncv * side * side;
    uint32_t *csf = cs + f * (nkey + 1);
    unsigned long long sv = 0;
    for (uint32_t p = (blockIdx.x - f * ns) * kBlock + threadIdx.x; p < npix; p += ns * kBlock) {
        const float I = frames[(size_t)f * npix + p];
        if (I == 0.0f) continue;
        atomicAdd(csf + tile_key(g, side, kmap[3 * (size_t)p + g.au], kmap[3 * (size_t)p + g.av]), 1u);
        if (!ORD) sv += self_value<kKindCq>(S, I);
    }
    if (ORD) return;
    for (int o = 32; o > 0; o >>= 1) sv += __shfl_down(sv, o, 64);
    if ((threadIdx.x & 63) == 0) sred[threadIdx.x >> 6] = sv;
    __syncthreads();
    if (threadIdx.x == 0) {
        sv = 0;
        for (int w = 0; w < kBlock / 64; w++) sv += sred[w];
        if (sv) {
            uint32_t lo = 0, hi = ngroups;  // group of f: largest gi with group_off[gi] <= f
            while (hi - lo > 1) {
                const uint32_t mid = (lo + hi) >> 1;
                if (group_off[mid] <= f) lo = mid; else hi = mid;
            }
            atomicAdd(self + lo, sv);
        }
    }
}

// One block per frame: the key counts become first positions (cs[nkey] the frame's records), and
// the scatter's cursors.
__global__ void __launch_bounds__(1024) tile_scan_kernel(uint32_t *__restrict__ cs, uint32_t *__restrict__ cursor,
                                                         uint32_t nkey)
{
    __shared__ uint32_t part[16];
    uint32_t *csf = cs + (size_t)blockIdx.x * (nkey + 1);
    uint32_t *cur = cursor + (size_t)blockIdx.x * nkey;
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    uint32_t base = 0;
    for (uint32_t k0 = 0; k0 < nkey; k0 += 4096) {  // four keys per thread and step
        uint32_t v[4], s = 0;
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
            v[i] = k0 + 4 * t + i < nkey ? csf[k0 + 4 * t + i] : 0u;
            s += v[i];
        }
        uint32_t x = s;
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o, 64);
            if (lane >= (uint32_t)o) x += y;
        }
        if (lane == 63) part[wave] = x;
        __syncthreads();
        uint32_t run = base + x - s;
        for (uint32_t w = 0; w < 16; w++) {
            if (w < wave) run += part[w];
            base += part[w];
        }
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
            if (k0 + 4 * t + i < nkey) csf[k0 + 4 * t + i] = cur[k0 + 4 * t + i] = run;
            run += v[i];
        }
        __syncthreads();
    }
    if (t == 0) csf[nkey] = base;
}

// The nonzero pixels as records {k[ka], k[kb], k[kc], I} in key order, frame f from f npix.
__global__ void __launch_bounds__(kBlock)
    tile_scatter_kernel(const float *__restrict__ kmap, const float *__restrict__ frames, uint32_t npix, uint32_t ns,
                        CellGeom g, int side, int ka, int kb, int kc, uint32_t *__restrict__ cursor,
                        float4 *__restrict__ srec)
{
    const uint32_t f = blockIdx.x / ns;
    uint32_t *cur = cursor + f * ((size_t)g.ncu * g.ncv * side * side);
    for (uint32_t p = (blockIdx.x - f * ns) * kBlock + threadIdx.x; p < npix; p += ns * kBlock) {
        const float I = frames[(size_t)f * npix + p];
        if (I == 0.0f) continue;
        const float *k = kmap + 3 * (size_t)p;
        srec[(size_t)f * npix + atomicAdd(cur + tile_key(g, side, k[g.au], k[g.av]), 1u)] =
            make_float4(k[ka], k[kb], k[kc], I);
    }
}

constexpr uint32_t kPartBatch = 4;  // b records per scalar load batch

// A nearest-neighbour task of an image with many records per voxel.  For one a record the records
// of one part of J -- a voxel across -- fall on at most two voxels per axis, so a lane keeps the
// sums of its a with the part in registers and adds them to the box once per part: two compares in
// place of the rounding and the address, and no LDS add per pair.  Exact: subtraction, scaling and
// rounding are monotone, so the part's k extents give its first and last voxel; x rounds to n + 1
// or more where x >= n + 1/2 (n >= 0) or x > n + 1/2 (n < 0, half away from zero); the values are
// whole numbers below 2^32, whose sums a double holds.  A part that spans more voxels for some
// lane is binned pair by pair.
__device__ __forceinline__ void tile_by_parts(const float4 *__restrict__ rec, const uint32_t *__restrict__ csf,
                                              size_t parts, uint32_t a0, uint32_t na, const TileTask &T, float vox,
                                              double mult, int bx8, int bxby8, int c8, char *boxb,
                                              float (*ext)[kTileParts], uint32_t share, uint32_t shares)
{
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t *pj = csf + T.cj * parts;
    __syncthreads();  // the frame before may still be read
    for (uint32_t s = wave; s < parts; s += kBlock / 64) {
        const uint32_t s0 = pj[s], s1 = pj[s + 1];
        float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        for (uint32_t i = s0 + lane; i < s1; i += 64) {
            const float4 r = rec[i];
            lo[0] = fminf(lo[0], r.x);
            lo[1] = fminf(lo[1], r.y);
            lo[2] = fminf(lo[2], r.z);
            hi[0] = fmaxf(hi[0], r.x);
            hi[1] = fmaxf(hi[1], r.y);
            hi[2] = fmaxf(hi[2], r.z);
        }
        for (int o = 32; o > 0; o >>= 1)
            for (int d = 0; d < 3; d++) {
                lo[d] = fminf(lo[d], __shfl_xor(lo[d], o, 64));
                hi[d] = fmaxf(hi[d], __shfl_xor(hi[d], o, 64));
            }
        if (lane == 0)
            for (int d = 0; d < 3; d++) {
                ext[d][s] = lo[d];
                ext[3 + d][s] = hi[d];
            }
    }
    __syncthreads();
    const uint32_t groups = (na + 63) / 64, np = (uint32_t)parts;
    const uint64_t units = (uint64_t)groups * np;
    const uint64_t u0 = units * share / shares, u1 = units * (share + 1) / shares;
    uint32_t gr = (uint32_t)(u0 / np), s = (uint32_t)(u0 - (uint64_t)gr * np);
    float4 a = rec[a0 + min(gr * 64 + lane, na - 1)];
    // the float above n + 1/2 that the first x of voxel n + 1 reaches
    auto edge_of = [](int n) {
        const float t = (float)n + 0.5f;
        return n < 0 ? __uint_as_float(__float_as_uint(t) - 1u) : t;
    };
    // v, or next to nothing: only the high word is selected, and what the low word leaves (below
    // 2^-1021) vanishes in a sum of whole numbers or truncates to 0
    auto v_if = [](bool m, double v) {
        const uint64_t u = __builtin_bit_cast(uint64_t, v);
        const uint32_t h = m ? (uint32_t)(u >> 32) : 0u;
        return __builtin_bit_cast(double, ((uint64_t)h << 32) | (uint32_t)u);
    };
    auto add = [&](int o, double x) {
        if (x >= 1.0) atomicAdd(reinterpret_cast<unsigned long long *>(boxb + o), (unsigned long long)x);
    };
    for (uint64_t u = u0; u < u1; u++) {
        const uint32_t s0 = pj[s], s1 = pj[s + 1];
        if (s0 < s1 && gr * 64 + lane < na) {
            const scalar_rec_t b = (scalar_rec_t)(uintptr_t)(rec + s0);
            const uint32_t n = s1 - s0;
            const int a_n0 = round_away((a.x - ext[3][s]) * vox), a_n1 = round_away((a.x - ext[0][s]) * vox);
            const int b_n0 = round_away((a.y - ext[4][s]) * vox), b_n1 = round_away((a.y - ext[1][s]) * vox);
            const int c_n0 = round_away((a.z - ext[5][s]) * vox), c_n1 = round_away((a.z - ext[2][s]) * vox);
            const int o = __mul24(c_n0, bxby8) + (__mul24(b_n0, bx8) + (a_n0 * 8 + c8));
            const bool wide = a_n1 - a_n0 > 1 || b_n1 - b_n0 > 1 || c_n1 - c_n0 > 1;
            if (__ballot(wide) != 0 || n >= (1u << 20)) {
                for (uint32_t j = 0; j < n; j++) {
                    const f4v r = b[j];
                    const double v = (double)(a.w * r.w) * mult;
                    const int q = __mul24(round_away((a.z - r.z) * vox), bxby8) +
                                  (__mul24(round_away((a.y - r.y) * vox), bx8) + (round_away((a.x - r.x) * vox) * 8 + c8));
                    atomicAdd(reinterpret_cast<unsigned long long *>(boxb + q), (unsigned long long)(uint32_t)v);
                }
            } else {
                const float ta = edge_of(a_n0), tb = edge_of(b_n0), tc = edge_of(c_n0);
                // sums over the pairs beyond no, one or both edges: s00 all, s10 beyond a's, s01 b's, s11 both
                auto sums = [&](auto deep_c) {
                    constexpr bool kDeep = decltype(deep_c)::value;
                    double s00 = 0, s10 = 0, s01 = 0, s11 = 0, d00 = 0, d10 = 0, d01 = 0, d11 = 0;
                    for (uint32_t j0 = 0; j0 < n; j0 += kPartBatch) {
                        f4v r[kPartBatch];
#pragma unroll
                        for (uint32_t k = 0; k < kPartBatch; k++) {
                            r[k] = b[min(j0 + k, n - 1)];
                            if (j0 + k >= n) r[k].w = 0.0f;  // past the part: adds nothing
                        }
#pragma unroll
                        for (uint32_t k = 0; k < kPartBatch; k++) {
                            const bool ma = (a.x - r[k].x) * vox >= ta, mb = (a.y - r[k].y) * vox >= tb;
                            const double v = trunc((double)(a.w * r[k].w) * mult);
                            s00 += v;
                            s10 += v_if(ma, v);
                            s01 += v_if(mb, v);
                            s11 += v_if(ma && mb, v);
                            if (kDeep) {
                                const bool mc = (a.z - r[k].z) * vox >= tc;
                                d00 += v_if(mc, v);
                                d10 += v_if(mc && ma, v);
                                d01 += v_if(mc && mb, v);
                                d11 += v_if(mc && ma && mb, v);
                            }
                        }
                    }
                    auto plane = [&](int at, double p00, double p10, double p01, double p11) {
                        add(at, (p00 - p10) - (p01 - p11));
                        add(at + 8, p10 - p11);
                        add(at + bx8, p01 - p11);
                        add(at + bx8 + 8, p11);
                    };
                    if (kDeep) {
                        plane(o, s00 - d00, s10 - d10, s01 - d01, s11 - d11);
                        plane(o + bxby8, d00, d10, d01, d11);
                    } else {
                        plane(o, s00, s10, s01, s11);
                    }
                };
                if (__ballot(c_n1 != c_n0) != 0) sums(std::true_type{}); else sums(std::false_type{});
            }
        }
        if (++s == np) {
            s = 0;
            gr++;
            a = rec[a0 + min(gr * 64 + lane, na - 1)];
        }
    }
}

// Grid: ntasks per chunk of frames of one group.  Symmetric (nearest) runs bin each unordered pair
// once into the half mesh, linear ones every ordered pair, self pairs too, into the mesh.
// WIDE: values up to 2^62, converted in two halves (five instructions for one).  24 frames of 256^2 in
// 4 groups into 129 x 129 x 3 at a multiplicator of 1e10: 62.7 ms by the engine, 37.4 (31.4 at 1e6).
template <bool LINEAR, bool WIDE>
__global__ void __launch_bounds__(kBlock, LINEAR ? 4 : 8)
    cq_tile_kernel(const float4 *__restrict__ srec, uint32_t npix, const uint32_t *__restrict__ cs, int ncell, int side,
                   const Chunk *__restrict__ chunks, const TileTask *__restrict__ tasks, uint32_t ntasks, PairSpec S,
                   unsigned long long *__restrict__ target, size_t nvox, unsigned long long *__restrict__ dropped,
                   int by_parts, uint32_t splits)
{
    __shared__ float part_ext[LINEAR ? 1 : 6][LINEAR ? 1 : kTileParts];  // by parts: min a b c, max a b c
    extern __shared__ unsigned long long box[];  // the plan's largest box
    const uint32_t split = blockIdx.x % splits, ti = blockIdx.x / splits;
    const TileTask T = tasks[ti % ntasks];
    const Chunk CH = chunks[ti / ntasks];
    const int vbox = T.bx * T.by * T.bz;
    for (int v = threadIdx.x; v < vbox; v += kBlock) box[v] = 0ull;
    __syncthreads();
    // the wave's share of a task's units: contiguous, first by block, then by wave
    const uint32_t share = split * (kBlock / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t shares = splits * (kBlock / 64);
    const bool tri = !LINEAR && T.ci == T.cj;
    const bool fast = T.inbox, is_signed = T.sa != 0 && T.sb != 0;
    unsigned long long *const out = target + (size_t)CH.group * nvox;
    BoxSink sink{box, out, dropped, T.bx0, T.by0, T.bz0, T.bx, T.by, T.bz, S.P.sab, S.P.sc, LINEAR ? 1ull : 2ull,
                 nullptr, 0, 0, 0};
    // byte strides of the box, and the centre's byte offset in it
    const int bx8 = 8 * T.bx, bxby8 = 8 * T.bx * T.by;
    const int c8 = 8 * (S.P.c0 - T.bx0) + bx8 * (S.P.c1 - T.by0) + bxby8 * (S.P.c2 - T.bz0);
    const int cab8 = 8 * (S.P.c0 - T.bx0) + bx8 * (S.P.c1 - T.by0);  // in a plane of the box
    char *const boxb = reinterpret_cast<char *>(box);
    const float vox = S.P.vox, cut_sq = S.P.cut_sq;
    const uint32_t lane = threadIdx.x & 63u;

    // the pair's |q|^2 in the order of the k components (records hold them as the mesh's axes)
    auto norm2 = [&](float qa, float qb, float qc) {
        const float a2 = qa * qa, b2 = qb * qb, c2 = qc * qc;
        const float z = S.kc == 2 ? c2 : (S.kb == 2 ? b2 : a2);
        return ((S.kc == 2 ? a2 : (S.kb == 2 ? a2 : b2)) + (S.kc == 2 ? b2 : c2)) + z;
    };
    auto add8 = [&](int o, double x) {
        unsigned long long v = (uint32_t)x;
        if (WIDE) {  // the high word by an exact scaling, the rest of x without rounding
            const uint32_t hi = (uint32_t)(x * 0x1p-32);
            v = (unsigned long long)hi << 32 | (uint32_t)fma((double)hi, -0x1p32, x);
        }
        atomicAdd(reinterpret_cast<unsigned long long *>(boxb + o), v);
    };
    // signed voxel scale and byte stride of the first two axes: q times the first is not negative
    const float voxa = T.sa < 0 ? -vox : vox, voxb = T.sb < 0 ? -vox : vox;
    const int sta = T.sa < 0 ? -8 : 8, stb = T.sb < 0 ? -bx8 : bx8;
    // fast: the pair's voxels lie in the box; a pair that fails the cut
    // adds 0 (nearest) or is skipped (linear).  kSigned: q keeps its sign along the first two axes;
    // kThin: the box is one voxel deep along the third, whose voxel is then the same for all pairs.
    auto bin_fast = [&](const float4 &a, const f4v &b, auto cut_c, auto signed_c, auto thin_c) {
        constexpr bool kCut = decltype(cut_c)::value, kSigned = decltype(signed_c)::value;
        constexpr bool kThin = decltype(thin_c)::value;
        const float w = a.w * b.w, qa = a.x - b.x, qb = a.y - b.y, qc = a.z - b.z;
        if (!LINEAR) {
            const double x = (double)w * S.mult;
            int o = kSigned ? __mul24(round_up(qb * voxb), stb) + (__mul24(round_up(qa * voxa), sta) + (kThin ? cab8 : c8))
                            : __mul24(round_away(qb * vox), bx8) + (round_away(qa * vox) * 8 + (kThin ? cab8 : c8));
            if (!kThin) o += __mul24(round_away(qc * vox), bxby8);
            add8(o, !kCut || norm2(qa, qb, qc) < cut_sq ? x : 0.0);
            return;
        }
        if (kCut && !(norm2(qa, qb, qc) < cut_sq)) return;
        const float xa = qa * vox, xb = qb * vox, xc = qc * vox;
        const float fa = floorf(xa), fb = floorf(xb), fc = floorf(xc);
        const double sa = (double)(1.0f - (xa - fa)), sb = (double)(1.0f - (xb - fb)), sc = (double)(1.0f - (xc - fc));
        const double vm = (double)w * S.mult;
        const int o = __mul24((int)fc, bxby8) + (__mul24((int)fb, bx8) + ((int)fa * 8 + c8));
        const double p00 = sa * sb, p10 = (1 - sa) * sb, p01 = sa * (1 - sb), p11 = (1 - sa) * (1 - sb), tc = 1 - sc;
        add8(o, vm * (p00 * sc));
        add8(o + 8, vm * (p10 * sc));
        add8(o + bx8, vm * (p01 * sc));
        add8(o + bx8 + 8, vm * (p11 * sc));
        add8(o + bxby8, vm * (p00 * tc));
        add8(o + bxby8 + 8, vm * (p10 * tc));
        add8(o + bxby8 + bx8, vm * (p01 * tc));
        add8(o + bxby8 + bx8 + 8, vm * (p11 * tc));
    };
    // any pair, through the checked box
    auto bin_any = [&](const float4 &a, const f4v &b) {
        auto as_k = [&](float x, float y, float z, float w) {  // mesh axes -> k components
            return make_float4(S.ka == 0 ? x : (S.kb == 0 ? y : z), S.ka == 1 ? x : (S.kb == 1 ? y : z),
                               S.ka == 2 ? x : (S.kb == 2 ? y : z), w);
        };
        const float4 ra = as_k(a.x, a.y, a.z, a.w), rb = as_k(b.x, b.y, b.z, b.w);
        if (LINEAR) {
            bin_ordered<kKindCq>(S, ra, rb, sink);
        } else {
            int fs, ms, ss;
            uint64_t v;
            if (bin_sym<kKindCq>(S, ra, rb, fs, ms, ss, v)) sink.add(fs, ms, ss, v);
        }
    };

    for (uint32_t f = CH.f0; f < CH.f1; f++) {
        const size_t parts = (size_t)side * side;
        const uint32_t *csf = cs + f * (ncell * parts + 1);
        const float4 *rec = srec + (size_t)f * npix;
        const uint32_t a0 = csf[T.ci * parts], na = csf[(T.ci + 1) * parts] - a0;
        const uint32_t b0 = csf[T.cj * parts], nb = csf[(T.cj + 1) * parts] - b0;
        if (na == 0 || nb == 0) continue;
        const scalar_rec_t brec = (scalar_rec_t)(uintptr_t)(rec + b0);
        if constexpr (!LINEAR && !WIDE) {
            if (by_parts && fast && T.allin && !tri) {
                tile_by_parts(rec, csf, parts, a0, na, T, vox, S.mult, bx8, bxby8, c8, boxb, part_ext, share, shares);
                continue;
            }
        }
        // units: lane groups of the a records (group gr holds records gr + lane groups) times
        // runs of kTileB b records
        const uint32_t groups = (na + 63) / 64, runs = (nb + kTileB - 1) / kTileB;
        const uint64_t units = (uint64_t)groups * runs;
        const uint64_t u0 = units * share / shares, u1 = units * (share + 1) / shares;
        uint32_t gr = (uint32_t)(u0 / runs), run = (uint32_t)(u0 - (uint64_t)gr * runs);
        uint32_t ia = gr + lane * groups;
        float4 ra = rec[a0 + min(ia, na - 1)];
        auto unit = [&](auto edge_c, auto bin) {
            constexpr bool kEdge = decltype(edge_c)::value;
            constexpr int kTileBatch = TileBatch<LINEAR>::n;
#pragma unroll 1
            for (uint32_t j0 = run * kTileB; j0 < (run + 1) * kTileB; j0 += kTileBatch) {
                f4v rb[kTileBatch];
#pragma unroll
                for (int k = 0; k < kTileBatch; k++) rb[k] = brec[kEdge ? min(j0 + k, nb - 1) : j0 + k];
#pragma unroll
                for (int k = 0; k < kTileBatch; k++) {
                    // tri: each unordered pair of distinct records once
                    if (kEdge && (j0 + k >= nb || (tri && j0 + k <= ia))) continue;
                    bin(ra, rb[k]);
                }
            }
        };
        using T_ = std::true_type;
        using F_ = std::false_type;
        for (uint64_t u = u0; u < u1; u++) {
            if (ia < na) {
                const bool edge = tri || (run + 1) * kTileB > nb;
                auto go = [&](auto edge_c, auto cut_c, auto signed_c, auto thin_c) {
                    unit(edge_c, [&](const float4 &a, const f4v &b) { bin_fast(a, b, cut_c, signed_c, thin_c); });
                };
                if (!fast) {
                    unit(T_{}, bin_any);
                } else if (edge) {
                    go(T_{}, T_{}, F_{}, F_{});
                } else if (LINEAR) {
                    if (T.allin) go(F_{}, F_{}, F_{}, F_{}); else go(F_{}, T_{}, F_{}, F_{});
                } else if (T.allin && is_signed) {
                    if (T.bz == 1) go(F_{}, F_{}, T_{}, T_{}); else go(F_{}, F_{}, T_{}, F_{});
                } else if (T.allin) {
                    go(F_{}, F_{}, F_{}, F_{});
                } else {
                    go(F_{}, T_{}, F_{}, F_{});
                }
            }
            if (++run == runs) {
                run = 0;
                ia = ++gr + lane * groups;
                ra = rec[a0 + min(ia, na - 1)];
            }
        }
    }
    __syncthreads();
    for (int v = threadIdx.x; v < vbox; v += kBlock) {
        const unsigned long long x = box[v];
        if (!x) continue;
        const int fs = T.bx0 + v % T.bx, ms = T.by0 + v / T.bx % T.by, ss = T.bz0 + v / (T.bx * T.by);
        atomicAdd(out + (size_t)fs + (size_t)ms * S.P.sab + (size_t)ss * S.P.sab * S.P.sab, x);
    }
}

// ---- AC_uw strips ---------------------------------------------------------------------
//
// The walk above finds a pair's records through per-cell items of about 20 pairs, which costs twice
// what binning the pair does (58 VALU instructions and 7 LDS accesses per 64 pairs).  Where a box of
// 32-bit words can hold it, a task is instead a distance between strips of the detector (a few
// voxels tall, all of it wide): the records of strip j and those of the strips j + dv ..
// j + dv + nv - 1 pair completely, so a wave takes one side's records as lanes and the other's
// one by one from the scalar unit, with no index work: 22 VALU instructions and one LDS add per
// 64 pairs.  The box counts w_a w_b; the flush multiplies by the fixed point's 1000.
// 32 bits are exact: weights are integers in [1, 129] (else the walk runs) and a block flushes before
// the frames it has added could pass 2^32.  For one a the b of a voxel lie in a window one voxel
// tall, which meets two strips where they are taller than a voxel (three at one voxel, where rounding
// may reach over both edges), all of them in one task if it holds several distances; so a frame adds
// at most W A to a voxel, W the sum of its weights and A that of its fullest two (three)
// strips in a row.
// 3,000 frames of 2,090 photons on a 1024^2 detector into 257^3: 9.0 ms by the walk, 6.5 by strips
// (1.0e12 pairs/s); 800 frames with a rotation each 10.0 and 4.7 (a task of several distances
// flushes each voxel of its mesh 1.2 times, the walk's small boxes 2 to 3 times).  Bound: VALU issue
// at three quarters, a fifth of the lanes empty; with rotations the scattered atomics of the flush.
// Lanes without a record are off rather than adding 0: their zeros would meet in one address, 13
// clocks of LDS per 64 pairs instead of 6 (7.4 ms).

constexpr int kMaxStrips = 512;

// One block per frame, as cell_sort_kernel: records by strip, strip starts, self values; bound[f] =
// W A, the most a voxel can receive from the frame.  A record's w holds its integer weight and, above 8
// bits, its reach: no record of a strip fewer than reach strips away, wherever in it, is beyond the
// cut.  A strip's records are in order of falling reach (eight classes), so that
// most batches of b need no cut.  `usable` starts at 1 and is cleared by a weight that is no
// integer in [1, 129] or a frame whose bound passes 2^32 (any of 2^24 records does: 512 strips).
struct StripGeom {
    CellGeom g;
    float ulo, uhi, zext;  // extents of the k-map along the strips and the beam
    int span;              // strips that the window of a voxel can meet
};
constexpr int kReachClasses = 8;
__device__ inline uint32_t strip_reach(const StripGeom &G, float cut_sq, float u)
{
    const float du = fmaxf(u - G.ulo, G.uhi - u);
    const float left = cut_sq * (1.0f - 1e-5f) - (du * du + G.zext * G.zext) * (1.0f + 1e-5f);
    return left > 0.0f ? (uint32_t)min((float)(2 * kMaxStrips), sqrtf(left) * G.g.inv_wv * (1.0f - 1e-5f)) : 0u;
}
__global__ void __launch_bounds__(kBlock)
    strip_sort_kernel(const float4 *__restrict__ rec, const uint64_t *__restrict__ off, StripGeom G,
                      float4 *__restrict__ srec, uint32_t *__restrict__ cs, PairSpec S,
                      const uint32_t *__restrict__ group_off, uint32_t ngroups,
                      unsigned long long *__restrict__ self, uint32_t *__restrict__ usable,
                      uint32_t *__restrict__ bound)
{
    __shared__ uint32_t cnt[kMaxStrips * kReachClasses], wsum[kMaxStrips];
    __shared__ unsigned long long sred[kBlock / 64];
    __shared__ uint32_t wred[kBlock / 64], nred[kBlock / 64], sums[kBlock / 64];
    const CellGeom &g = G.g;
    const uint32_t f = blockIdx.x, lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const int ncell = g.ncv, nbin = ncell * kReachClasses;
    const uint64_t base = off[f];
    const uint32_t n = (uint32_t)(off[f + 1] - base);
    auto place = [&](const float4 &r, uint32_t reach) {
        const int cls = max(0, kReachClasses - 1 - (int)(reach * kReachClasses / (uint32_t)ncell));
        return cell_of(g, 0.0f, comp(r, g.av)) * kReachClasses + cls;
    };
    for (int c = threadIdx.x; c < kMaxStrips * kReachClasses; c += kBlock) cnt[c] = 0;
    for (int c = threadIdx.x; c < kMaxStrips; c += kBlock) wsum[c] = 0;
    __syncthreads();
    unsigned long long sv = 0;
    bool ok = n < (1u << 24);  // the sums of weights below fit 32 bits
    for (uint32_t i = threadIdx.x; i < n; i += kBlock) {
        const float4 r = rec[base + i];
        if (r.w == 0.0f) continue;
        const int bin = place(r, strip_reach(G, S.P.cut_sq, comp(r, g.au)));
        atomicAdd(&cnt[bin], 1u);
        sv += self_value<kKindAc3d>(S, r.w);
        const bool small = r.w >= 1.0f && r.w <= 129.0f && r.w == truncf(r.w);
        ok = ok && small;
        if (small) atomicAdd(&wsum[bin / kReachClasses], (uint32_t)r.w);
    }
    if (!ok) usable[0] = 0u;
    __syncthreads();
    // starts: consecutive bins per thread, whole strips each
    const int per = (nbin / kReachClasses + kBlock - 1) / kBlock;  // strips
    uint32_t tot = 0, most = 0, weight = 0;
    for (int k = 0; k < per; k++) {
        const int c = (int)threadIdx.x * per + k;
        if (c >= ncell) break;
        for (int e = 0; e < kReachClasses; e++) tot += cnt[c * kReachClasses + e];
        uint32_t window = 0;
        for (int e = c; e < min(c + G.span, ncell); e++) window += wsum[e];
        weight += wsum[c];
        most = max(most, window);
    }
    uint32_t x = tot;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= (uint32_t)o) x += y;
    }
    for (int o = 32; o > 0; o >>= 1) {
        sv += __shfl_down(sv, o, 64);
        weight += __shfl_down(weight, o, 64);
        most = max(most, (uint32_t)__shfl_down(most, o, 64));
    }
    if (lane == 63) sums[wave] = x;
    if (lane == 0) {
        sred[wave] = sv;
        wred[wave] = weight;
        nred[wave] = most;
    }
    __syncthreads();
    uint32_t run = x - tot, all = 0;
    for (uint32_t w = 0; w < kBlock / 64; w++) {
        if (w < wave) run += sums[w];
        all += sums[w];
    }
    uint32_t *csf = cs + (size_t)f * (ncell + 1);
    for (int k = 0; k < per; k++) {
        const int c = ((int)threadIdx.x * per + k) * kReachClasses;
        if (c >= nbin) break;
        csf[c / kReachClasses] = run;
        for (int e = 0; e < kReachClasses; e++) {
            const uint32_t v = cnt[c + e];
            cnt[c + e] = run;
            run += v;
        }
    }
    if (threadIdx.x == 0) {
        csf[ncell] = all;
        weight = most = 0;
        sv = 0;
        for (uint32_t k = 0; k < kBlock / 64; k++) {
            weight += wred[k];
            most = max(most, nred[k]);
            sv += sred[k];
        }
        const uint64_t b = (uint64_t)weight * most;
        if (b >> 32) usable[0] = 0u;
        bound[f] = (uint32_t)b;
        if (sv) {
            uint32_t lo = 0, hi = ngroups;  // group of f: largest gi with group_off[gi] <= f
            while (hi - lo > 1) {
                const uint32_t mid = (lo + hi) >> 1;
                if (group_off[mid] <= f) lo = mid; else hi = mid;
            }
            atomicAdd(self + lo, sv);
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n; i += kBlock) {
        float4 r = rec[base + i];
        if (r.w == 0.0f) continue;
        const uint32_t reach = strip_reach(G, S.P.cut_sq, comp(r, g.au));
        const uint32_t pos = atomicAdd(&cnt[place(r, reach)], 1u);
        r.w = __uint_as_float(((uint32_t)r.w & 255u) | reach << 8);
        srec[base + pos] = r;
    }
}

constexpr int kStripBatch = 4;  // scalar records per load batch

__device__ inline int mad24(int a, int b, int c)
{
    int r;
    asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));  // else two multiplies and an add3
    return r;
}

__device__ inline uint32_t uniform(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }

// Grid: ntasks per chunk of frames.  AV: the k component across the strips (0 or 1); the beam is
// the third.  A task pairs b in strip j with a in the strips j + dv .. j + dv + nv - 1.
template <int AV, int BLOCK>
__global__ void __launch_bounds__(BLOCK)
    strip_kernel(const float4 *__restrict__ srec, const uint64_t *__restrict__ off, const uint32_t *__restrict__ cs,
                 const Chunk *__restrict__ chunks, const Task *__restrict__ tasks, uint32_t ntasks, int ncell,
                 PairSpec S, unsigned long long *__restrict__ target, size_t nvox,
                 unsigned long long *__restrict__ dropped, const uint32_t *__restrict__ usable,
                 const uint32_t *__restrict__ bound, const float *__restrict__ rots)
{
    extern __shared__ uint32_t sbox[];
    if (!usable[0]) return;
    const Task T = tasks[blockIdx.x % ntasks];
    const Chunk CH = chunks[blockIdx.x / ntasks];
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr uint32_t kWaves = BLOCK / 64;
    const int vbox = T.bx * T.by * T.bz;
    for (int v = threadIdx.x; v < vbox; v += BLOCK) sbox[v] = 0u;
    const int bx4 = 4 * T.bx, bxby4 = 4 * T.bx * T.by;
    const int c4 = 4 * (S.P.c0 - T.bx0) + bx4 * (S.P.c1 - T.by0) + bxby4 * (S.P.c2 - T.bz0);
    char *const boxb = reinterpret_cast<char *>(sbox);
    const float cut_sq = S.P.cut_sq;
    unsigned long long *const out = target + (size_t)CH.group * nvox;
    const float *crot = rots ? rots + 9 * (size_t)CH.f0 : nullptr;

    auto flush = [&]() {
        float rr[9];
        int ax = 0;  // the box axis consecutive lanes walk (as the walk's flush)
        if (crot) {
            for (int i = 0; i < 9; i++) rr[i] = crot[i];
            const float a0 = fabsf(rr[0]), a1 = fabsf(rr[1]), a2 = fabsf(rr[2]);
            ax = a1 > a0 ? (a2 > a1 ? 2 : 1) : (a2 > a0 ? 2 : 0);
        }
        const int e0 = ax == 0 ? T.bx : (ax == 1 ? T.by : T.bz), e1 = ax == 0 ? T.by : T.bx;
        for (int v = threadIdx.x; v < vbox; v += BLOCK) {
            const int i0 = v % e0, rest = v / e0, i1 = rest % e1, i2 = rest / e1;
            const int lx = ax == 0 ? i0 : i1, ly = ax == 1 ? i0 : (ax == 0 ? i1 : i2), lz = ax == 2 ? i0 : i2;
            const uint32_t x = sbox[lx + T.bx * (ly + T.by * lz)];
            if (!x) continue;
            int fs = T.bx0 + lx, ms = T.by0 + ly, ss = T.bz0 + lz;
            if (crot) {
                rotate_voxel(rr, S.P.c0, S.P.c1, S.P.c2, fs, ms, ss);
                if ((unsigned)fs >= (unsigned)S.P.sab || (unsigned)ms >= (unsigned)S.P.sab ||
                    (unsigned)ss >= (unsigned)S.P.sc) {
                    atomicAdd(dropped, 1ull);  // excluded by the caller's bound check
                    continue;
                }
            }
            atomicAdd(out + (size_t)fs + (size_t)ms * S.P.sab + (size_t)ss * S.P.sab * S.P.sab, 1000ull * x);
        }
    };

    // lane record l with scalar record s; vox carries the sign that makes it b from a
    auto pair = [&](const float4 &l, uint32_t lw, const f4v &s, float vox, auto within_c, auto cut_c, bool on) {
        constexpr bool kWithin = decltype(within_c)::value;  // q across the strips has both signs
        const float dx = l.x - s.x, dy = l.y - s.y, dz = l.z - s.z;
        if (decltype(cut_c)::value) on = ((dx * dx + dy * dy) + dz * dz < cut_sq) && on;
        const float x = dx * vox, y = dy * vox, z = dz * vox;
        // a - b across strips dv > 0 apart is not negative
        const int nx = !kWithin && AV == 0 ? round_up(x) : round_away(x);
        const int ny = !kWithin && AV == 1 ? round_up(y) : round_away(y);
        const uint32_t v = __umul24(lw, __float_as_uint(s.w));
        const int o = mad24(round_away(z), bxby4, mad24(ny, bx4, nx * 4 + c4));
        atomicAdd(reinterpret_cast<uint32_t *>(boxb + o), on ? v : 0u);
    };
    // n lane records by m scalar ones; within: only pairs (l, s < l)
    auto item = [&](const float4 *lr, uint32_t n, scalar_rec_t sr, uint32_t m, float vox, auto within_c) {
        constexpr bool kWithin = decltype(within_c)::value;
        for (uint32_t g0 = 0; g0 < n; g0 += 64) {
            const uint32_t il = g0 + lane, me = kWithin ? min(m, g0 + 63) : m;
            if (il >= n) continue;  // empty lanes off: their zeros would all go to one address
            const float4 l = lr[il];
            const uint32_t lw = __float_as_uint(l.w) & 255u;
            // the next batch loads under the pairs of this one
            f4v next[kStripBatch];
#pragma unroll
            for (int k = 0; k < kStripBatch; k++) next[k] = sr[min((uint32_t)k, m - 1)];
            for (uint32_t j0 = 0; j0 < me; j0 += kStripBatch) {
                f4v s[kStripBatch];
                uint32_t least = ~0u;
#pragma unroll
                for (int k = 0; k < kStripBatch; k++) {
                    s[k] = next[k];
                    const uint32_t w = __float_as_uint(s[k].w);
                    least = min(least, w);
                    s[k].w = __uint_as_float(j0 + k < m ? w & 255u : 0u);
                }
#pragma unroll
                for (int k = 0; k < kStripBatch; k++) next[k] = sr[min(j0 + kStripBatch + k, m - 1)];
                if ((least >> 8) >= (uint32_t)(T.dv + T.nv)) {  // no pair of these strips beyond the cut
#pragma unroll
                    for (int k = 0; k < kStripBatch; k++)
                        pair(l, lw, s[k], vox, within_c, std::false_type{}, !kWithin || j0 + k < il);
                } else {
#pragma unroll
                    for (int k = 0; k < kStripBatch; k++)
                        pair(l, lw, s[k], vox, within_c, std::true_type{}, !kWithin || j0 + k < il);
                }
            }
        }
    };

    for (uint32_t fa = CH.f0; fa < CH.f1;) {
        // frames [fa, fb) cannot pass 2^32 in any voxel
        uint64_t most = bound[fa];
        uint32_t fb = fa + 1;
        while (fb < CH.f1 && most + bound[fb] < (1ull << 32)) most += bound[fb++];
        __syncthreads();  // the box is clear
        // items (frame, strip j of b), the waves in turn
        uint32_t f = uniform(fa);
        int j = (int)wave;
        for (;; j += (int)kWaves) {
            while (f < fb && j >= ncell - T.dv) {
                j -= ncell - T.dv;
                f++;
            }
            if (f >= fb) break;
            const scalar_u32_t csf = (scalar_u32_t)(uintptr_t)(cs + (size_t)f * (ncell + 1));
            const int i = j + T.dv, ie = min(i + T.nv, ncell);
            const uint32_t a0 = uniform(csf[i]), na = uniform(csf[ie]) - a0;
            const uint32_t b0 = uniform(csf[j]), nb = uniform(csf[j + 1]) - b0;
            if (na == 0 || nb == 0) continue;
            const uint64_t base = ((scalar_u64_t)(uintptr_t)off)[f];
            const float4 *fr = srec + (((uint64_t)uniform((uint32_t)(base >> 32)) << 32) | uniform((uint32_t)base));
            if (T.dv == 0)  // strip j itself and its neighbours: every a behind b in the order
                item(fr + a0, na, (scalar_rec_t)(uintptr_t)(fr + b0), nb, S.P.vox, std::true_type{});
            else if (((nb + 63) / 64) * na < ((na + 63) / 64) * nb)
                // the lanes take the side that leaves fewer of them empty
                item(fr + b0, nb, (scalar_rec_t)(uintptr_t)(fr + a0), na, -S.P.vox, std::false_type{});
            else
                item(fr + a0, na, (scalar_rec_t)(uintptr_t)(fr + b0), nb, S.P.vox, std::false_type{});
        }
        __syncthreads();
        flush();
        fa = fb;
        if (fa < CH.f1) {
            __syncthreads();
            for (int v = threadIdx.x; v < vbox; v += BLOCK) sbox[v] = 0u;
        }
    }
}

// ---- host planning ---------------------------------------------------------------

// The specialised pair path: AC_uw, symmetric (nearest-neighbour) binning, identity
// rotation; round_away needs |q * vox| < 2^23 and the cut bounds |q| by Max_Q.
inline bool fast_path(const PairSpec &S, bool ordered)
{
    // (its inline value is FloatToInt(float): the double-valued symmetric mode takes bin_sym)
    return S.kind == kKindAc3d && !ordered && S.P.rot_identity && !S.P.dval &&
           std::sqrt((double)S.P.cut_sq) * S.P.vox < 4194304.0;
}

// symmetric nearest-neighbour C(q): its voxels are round-half-away of the same
// fl(fl(ka - kb) * vox) products, so the tight boxes (and in-box tasks) apply
inline bool cq_tight(const PairSpec &S, bool ordered)
{
    return S.kind == kKindCq && !ordered && S.interp == 0 && std::sqrt((double)S.P.cut_sq) * S.P.vox < 4194304.0;
}

// interval of round(x) / of floor(x)+{0,1} for x in [lo, hi]
inline void nn_range(double &lo, double &hi)
{
    lo = std::floor(lo);
    hi = std::ceil(hi);
}
inline void lin_range(double &lo, double &hi)
{
    lo = std::floor(lo);
    hi = std::ceil(hi) + 1;
}

// Conservative voxel box (per mesh axis, relative to the centre) of the pairs
// whose q lies in [qlo, qhi].
void voxel_box(const PairSpec &S, const double qlo[3], const double qhi[3], double lo[3], double hi[3])
{
    const double vox = S.P.vox;
    double l[3], h[3];
    for (int d = 0; d < 3; d++) {
        l[d] = qlo[d] * vox;
        h[d] = qhi[d] * vox;
    }
    if (S.kind == kKindAc3d) {
        if (S.P.double_map) {
            for (int d = 0; d < 3; d++) (S.P.interp1 ? lin_range : nn_range)(l[d], h[d]);
        }
        if (!S.P.rot_identity) {
            double rl[3], rh[3];
            for (int i = 0; i < 3; i++) {
                rl[i] = rh[i] = 0;
                for (int j = 0; j < 3; j++) {
                    const double a = S.R[3 * i + j] * l[j], b = S.R[3 * i + j] * h[j];
                    rl[i] += std::min(a, b);
                    rh[i] += std::max(a, b);
                }
            }
            for (int d = 0; d < 3; d++) {
                l[d] = rl[d];
                h[d] = rh[d];
            }
        }
        for (int d = 0; d < 3; d++) {
            (S.P.interp2 ? lin_range : nn_range)(l[d], h[d]);
            lo[d] = l[d];
            hi[d] = h[d];
        }
    } else {
        const int ax[3] = {S.ka, S.kb, S.kc};
        for (int m = 0; m < 3; m++) {
            double a = l[ax[m]], b = h[ax[m]];
            (S.interp ? lin_range : nn_range)(a, b);
            lo[m] = a;
            hi[m] = b;
        }
    }
    for (int d = 0; d < 3; d++) {  // one voxel of slack for float rounding
        lo[d] -= 1;
        hi[d] += 1;
    }
}

}  // namespace
}  // namespace iac

struct iac_pair_plan {
    bool valid = false;
    // key
    const float *kmap = nullptr;
    uint32_t npix = 0;
    int cell_vox = 0;
    int box_cap = 0;  // LDS box capacity the tasks were sized for
    int region = 0;   // cells per task region side (0: whole grid)
    iac::PairSpec spec{};
    iac::CellGeom g{};
    std::vector<uint32_t> cell_ext;  // 6 keys per cell
    // product
    std::vector<iac::Task> tasks;
    iac::Task *d_tasks = nullptr;
    // region tiles (region == kRegionTiles): their tasks, and whether nearly all have a box
    std::vector<iac::TileTask> tiles;
    iac::TileTask *d_tiles = nullptr;
    bool tiles_fit = false;
    size_t tile_box = 0;  // voxels of the largest box
    int pins = 0;  // frame queues holding this plan (never evicted while > 0)
};

namespace iac {
namespace {

bool same_spec(const PairSpec &a, const PairSpec &b)
{
    return std::memcmp(&a, &b, sizeof(PairSpec)) == 0;
}

// Tasks: one per cell offset delta and region of first cells i.  A region of
// `region` x `region` cells (0: the whole grid) narrows the q range of its pairs
// -- q along the beam grows with the distance from the centre -- so larger cells
// still fit their voxel box.
void build_tasks(iac_pair_plan &pl, bool ordered)
{
    const CellGeom &g = pl.g;
    const PairSpec &S = pl.spec;
    const int nc = g.ncu * g.ncv;
    std::vector<char> has(nc, 0);
    std::vector<double> kmn(3 * (size_t)nc), kmx(3 * (size_t)nc);
    for (int c = 0; c < nc; c++) {
        const uint32_t *e = &pl.cell_ext[6 * (size_t)c];
        if (e[0] == 0xffffffffu) continue;  // no pixel in this cell
        has[c] = 1;
        for (int d = 0; d < 3; d++) {
            kmn[3 * c + d] = unkey(e[d]);
            kmx[3 * c + d] = unkey(e[3 + d]);
        }
    }
    const double maxq = std::sqrt((double)S.P.cut_sq);
    const int cen[3] = {S.P.c0, S.P.c1, S.P.c2};
    const int dim[3] = {S.P.sab, S.P.sab, S.P.sc};
    const int reg = pl.region > 0 ? pl.region : std::max(g.ncu, g.ncv);
    const bool fast = fast_path(S, ordered), tight_cq = cq_tight(S, ordered);
    const int cax[3] = {S.ka, S.kb, S.kc};  // C(q): the record component each mesh axis bins
    pl.tasks.clear();
    for (int dv = ordered ? -(g.ncv - 1) : 0; dv < g.ncv; dv++) {
        for (int du = -(g.ncu - 1); du < g.ncu; du++) {
            if (!ordered && dv == 0 && du < 0) continue;  // positive half plane
            const int iu0 = std::max(0, du), iv0 = std::max(0, dv);
            const int nu = std::min(g.ncu, g.ncu + du) - iu0, nv = std::min(g.ncv, g.ncv + dv) - iv0;
            if (nu <= 0 || nv <= 0) continue;
            for (int rv = iv0; rv < iv0 + nv; rv += reg) {
                for (int ru = iu0; ru < iu0 + nu; ru += reg) {
                    Task t{};
                    t.du = du;
                    t.dv = dv;
                    t.iu0 = ru;
                    t.iv0 = rv;
                    t.nu = std::min(reg, iu0 + nu - ru);
                    t.nv = std::min(reg, iv0 + nv - rv);
                    double qlo[3] = {1e30, 1e30, 1e30}, qhi[3] = {-1e30, -1e30, -1e30};
                    bool any = false;
                    for (int iv = t.iv0; iv < t.iv0 + t.nv; iv++)
                        for (int iu = t.iu0; iu < t.iu0 + t.nu; iu++) {
                            const int ci = iv * g.ncu + iu, cj = (iv - dv) * g.ncu + (iu - du);
                            if (!has[ci] || !has[cj]) continue;
                            any = true;
                            for (int d = 0; d < 3; d++) {
                                qlo[d] = std::min(qlo[d], kmn[3 * ci + d] - kmx[3 * cj + d]);
                                qhi[d] = std::max(qhi[d], kmx[3 * ci + d] - kmn[3 * cj + d]);
                            }
                        }
                    if (!any) continue;
                    double dist2 = 0;  // all pairs of the task are cut if the q box lies beyond Max_Q
                    for (int d = 0; d < 3; d++) {
                        const double m = qlo[d] > 0 ? qlo[d] : (qhi[d] < 0 ? -qhi[d] : 0.0);
                        dist2 += m * m;
                    }
                    if (std::sqrt(dist2) > maxq * (1.0 + 1e-5) + 1e-7) continue;
                    // the farthest corner of the q box inside the cut, with margin for the float
                    // rounding of the kernel's q and |q|^2 (a relative 3.1e-7 at most)
                    double far2 = 0;
                    for (int d = 0; d < 3; d++) far2 += std::max(qlo[d] * qlo[d], qhi[d] * qhi[d]);
                    t.allin = far2 * (1.0 + 1e-5) < (double)S.P.cut_sq ? 1 : 0;
                    double lo[3], hi[3];
                    if (fast || tight_cq) {
                        // the pair bins at round_away(fl(fl(ka - kb) * vox)): within eps of x in [l, h]
                        // (two float roundings, |x| < 2^22), so round-half-away lands in
                        // [ceil(l - eps - 1/2), floor(h + eps + 1/2)]
                        for (int d = 0; d < 3; d++) {
                            const int c = tight_cq ? cax[d] : d;
                            const double l = qlo[c] * S.P.vox, h = qhi[c] * S.P.vox;
                            const double eps = 1e-3 + 1e-6 * std::max(std::fabs(l), std::fabs(h));
                            lo[d] = std::ceil(l - eps - 0.5);
                            hi[d] = std::floor(h + eps + 0.5);
                        }
                    } else {
                        voxel_box(S, qlo, qhi, lo, hi);
                    }
                    int ilo[3], ihi[3];
                    for (int d = 0; d < 3; d++) {
                        ilo[d] = (int)std::max(0.0, lo[d] + cen[d]);
                        ihi[d] = (int)std::min((double)dim[d] - 1, hi[d] + cen[d]);
                    }
                    const long vol = (long)(ihi[0] - ilo[0] + 1) * (ihi[1] - ilo[1] + 1) * (ihi[2] - ilo[2] + 1);
                    if (ihi[0] >= ilo[0] && ihi[1] >= ilo[1] && ihi[2] >= ilo[2] && vol <= pl.box_cap) {
                        t.inbox = 1;
                        for (int d = 0; d < 3; d++)
                            if (lo[d] + cen[d] < 0.0 || hi[d] + cen[d] > (double)dim[d] - 1) t.inbox = 0;
                        if (S.kind == kKindCq && !tight_cq) t.inbox = 0;  // in-box C(q) bins need the tight boxes
                        t.bx0 = ilo[0];
                        t.by0 = ilo[1];
                        t.bz0 = ilo[2];
                        t.bx = ihi[0] - ilo[0] + 1;
                        t.by = ihi[1] - ilo[1] + 1;
                        t.bz = ihi[2] - ilo[2] + 1;
                    }
                    pl.tasks.push_back(t);
                }
            }
        }
    }
}

iac_pair_plan *find_plan(iac_ctx *ctx, const float *kmap, uint32_t npix, int cell_vox, int box_cap, int region,
                         const PairSpec &S)
{
    for (auto *p : ctx->pair_plans)
        if (p->valid && p->kmap == kmap && p->npix == npix && p->cell_vox == cell_vox && p->box_cap == box_cap &&
            p->region == region && same_spec(p->spec, S))
            return p;
    return nullptr;
}

constexpr size_t kMaxPlans = 20;   // cached plans of a context
constexpr int kRegionTiles = -1;   // iac_pair_plan::region of a region-tile plan
constexpr int kRegionStrips = -2;  // and less: of a strip plan, its distances per task with it
constexpr size_t kStripBox2 = 79 * 1024;  // LDS bytes of a strip box: two blocks per CU
constexpr size_t kStripBox1 = 158 * 1024; // one block per CU

// Tasks of the region tiles: pairs of regions (ci <= cj, or all ordered pairs of linear runs) that
// are not wholly beyond the cut, with the box of their voxels (linear: of their corners).
void build_tiles(iac_pair_plan &pl, bool ordered)
{
    const CellGeom &g = pl.g;
    const PairSpec &S = pl.spec;
    const int nc = g.ncu * g.ncv, cax[3] = {S.ka, S.kb, S.kc};
    const int cen[3] = {S.P.c0, S.P.c1, S.P.c2}, dim[3] = {S.P.sab, S.P.sab, S.P.sc};
    const long cap = pl.box_cap;
    const double maxq = std::sqrt((double)S.P.cut_sq);
    size_t boxed = 0;
    const size_t all = ordered ? (size_t)nc * nc : (size_t)nc * (nc + 1) / 2;
    for (int ci = 0; ci < nc; ci++) {
        if (pl.tiles.size() - boxed > all / 32) break;  // no longer to be made good
        const uint32_t *ea = &pl.cell_ext[6 * (size_t)ci];
        if (ea[0] == 0xffffffffu) continue;  // no pixel there
        for (int cj = ordered ? 0 : ci; cj < nc; cj++) {
            const uint32_t *eb = &pl.cell_ext[6 * (size_t)cj];
            if (eb[0] == 0xffffffffu) continue;
            double qlo[3], qhi[3], near2 = 0, far2 = 0;
            for (int d = 0; d < 3; d++) {
                qlo[d] = (double)unkey(ea[d]) - unkey(eb[3 + d]);
                qhi[d] = (double)unkey(ea[3 + d]) - unkey(eb[d]);
                const double m = qlo[d] > 0 ? qlo[d] : (qhi[d] < 0 ? -qhi[d] : 0.0);
                near2 += m * m;
                far2 += std::max(qlo[d] * qlo[d], qhi[d] * qhi[d]);
            }
            if (std::sqrt(near2) > maxq * (1.0 + 1e-5) + 1e-7) continue;
            TileTask t{};
            t.ci = ci;
            t.cj = cj;
            auto sign = [&](int d) { return qlo[d] >= 0.0 ? 1 : (qhi[d] <= 0.0 ? -1 : 0); };
            t.sa = sign(S.ka);
            t.sb = sign(S.kb);
            t.allin = far2 * (1.0 + 1e-5) < (double)S.P.cut_sq ? 1 : 0;
            // voxels round_away(x), or corners floor(x) and floor(x) + 1, of x within eps of
            // [l, h] (two float roundings)
            int lo[3], ext[3];
            bool box = true, inside = true;
            double vol = 1;
            for (int m = 0; m < 3; m++) {
                const double l = qlo[cax[m]] * S.P.vox, h = qhi[cax[m]] * S.P.vox;
                const double eps = 1e-3 + 1e-6 * std::max(std::fabs(l), std::fabs(h));
                const double v0 = (ordered ? std::floor(l - eps) : std::ceil(l - eps - 0.5)) + cen[m];
                const double v1 = (ordered ? std::floor(h + eps) + 1 : std::floor(h + eps + 0.5)) + cen[m];
                inside = inside && v0 >= 0.0 && v1 <= (double)dim[m] - 1;  // false for NaN
                const double c0 = std::max(0.0, v0), c1 = std::min((double)dim[m] - 1, v1);
                box = box && c1 >= c0;
                vol *= c1 - c0 + 1;
                lo[m] = box ? (int)c0 : 0;
                ext[m] = box ? (int)(c1 - c0) + 1 : 0;
            }
            if (box && vol <= (double)cap) {
                t.inbox = inside ? 1 : 0;
                t.bx0 = lo[0];
                t.by0 = lo[1];
                t.bz0 = lo[2];
                t.bx = ext[0];
                t.by = ext[1];
                t.bz = ext[2];
                pl.tile_box = std::max(pl.tile_box, (size_t)t.bx * t.by * t.bz);
                boxed++;
            }
            pl.tiles.push_back(t);
        }
    }
    pl.tiles_fit = !pl.tiles.empty() && boxed >= pl.tiles.size() - pl.tiles.size() / 32;
    if (!pl.tiles_fit) std::vector<TileTask>().swap(pl.tiles);
}

// One task per `per` strip distances, with the box of all of them.
void merge_strips(iac_pair_plan &pl, int per)
{
    std::vector<Task> out;
    for (const Task &t : pl.tasks) {  // in the order of dv
        // (a distance between them that is beyond the cut or has no pixels starts another task: its
        // pairs, if any, need not lie in the box)
        if (!out.empty() && out.back().dv / per == t.dv / per && t.dv == out.back().dv + out.back().nv) {
            Task &o = out.back();
            const int x1 = std::max(o.bx0 + o.bx, t.bx0 + t.bx), y1 = std::max(o.by0 + o.by, t.by0 + t.by),
                      z1 = std::max(o.bz0 + o.bz, t.bz0 + t.bz);
            o.bx0 = std::min(o.bx0, t.bx0);
            o.by0 = std::min(o.by0, t.by0);
            o.bz0 = std::min(o.bz0, t.bz0);
            o.bx = x1 - o.bx0;
            o.by = y1 - o.by0;
            o.bz = z1 - o.bz0;
            o.inbox = o.inbox && t.inbox;
            o.nv++;
        } else {
            out.push_back(t);
            out.back().nv = 1;
        }
    }
    for (Task &t : out) {
        t.inbox = t.inbox && (long)t.bx * t.by * t.bz <= pl.box_cap;
        pl.tile_box = std::max(pl.tile_box, (size_t)t.bx * t.by * t.bz * sizeof(uint32_t));
    }
    pl.tasks.swap(out);
}

// Page-locked read-back area of a plan: the k-map's extents (and a dense run's counts: kHead words),
// the cells', the strips', then more.
constexpr size_t kHead = 12;
struct PlanRead {
    uint32_t *kext, *cells, *strips;
    uint64_t *more;
};
int plan_read(iac_ctx *ctx, size_t more_bytes, PlanRead *out)
{
    void *p = nullptr;
    IAC_TRY(pinned(ctx, 0, (kHead + 6 * (size_t)(kMaxCells + kMaxStrips)) * sizeof(uint32_t) + more_bytes, &p));
    out->kext = static_cast<uint32_t *>(p);
    out->cells = out->kext + kHead;
    out->strips = out->cells + 6 * (size_t)kMaxCells;
    out->more = reinterpret_cast<uint64_t *>(out->strips + 6 * (size_t)kMaxStrips);
    return IAC_OK;
}

// Enqueues the extents of the k-map, d_ext initialised, and the copy of `words` words there to read.kext.
int kmap_extents_enqueue(hipStream_t st, const float *d_kmap, uint32_t npix, uint32_t *d_ext, const PlanRead &read,
                         size_t words = 6)
{
    const unsigned eb = std::max(1u, std::min<unsigned>(64, (npix + 1023) / 1024));
    hipLaunchKernelGGL(kext_kernel, dim3(eb), dim3(256), 0, st, d_kmap, npix, d_ext);
    IAC_HIP(hipGetLastError());
    IAC_HIP(hipMemcpyAsync(read.kext, d_ext, words * sizeof(uint32_t), hipMemcpyDeviceToHost, st));
    return IAC_OK;
}
void kmap_extents_read(const PlanRead &read, float kmin[3], float ext3[3])
{
    for (int d = 0; d < 3; d++) {
        kmin[d] = unkey(read.kext[d]);
        ext3[d] = unkey(read.kext[3 + d]) - kmin[d];
    }
}

// Extents of the k-map (one host round trip).
int kmap_extents(hipStream_t st, const float *d_kmap, uint32_t npix, uint32_t *d_ext, const PlanRead &read,
                 float kmin[3], float ext3[3])
{
    hipLaunchKernelGGL(init_cell_ext_kernel, dim3(1), dim3(64), 0, st, d_ext, 1);
    IAC_TRY(kmap_extents_enqueue(st, d_kmap, npix, d_ext, read));
    IAC_HIP(hipStreamSynchronize(st));
    kmap_extents_read(read, kmin, ext3);
    return IAC_OK;
}

// The grid of cells cell_vox % 1000 (u) by cell_vox / 1000 (v, 0: as u) voxels over the two widest
// axes, larger where it would exceed kMaxCells.
CellGeom cell_grid(const float kmin[3], const float ext3[3], float vox, int cell_vox)
{
    CellGeom g{};
    int order[3] = {0, 1, 2};
    std::sort(order, order + 3, [&](int a, int b) { return ext3[a] > ext3[b]; });
    g.au = std::min(order[0], order[1]);
    g.av = std::max(order[0], order[1]);
    double wu = (double)(cell_vox % 1000) / (double)vox;
    double wv = (double)(cell_vox / 1000 ? cell_vox / 1000 : cell_vox % 1000) / (double)vox;
    auto ncells = [&](int a, double w) { return std::max(1, (int)std::ceil(ext3[a] / w * (1 + 1e-6))); };
    while ((long)ncells(g.au, wu) * ncells(g.av, wv) > kMaxCells) {
        wu *= 1.25;
        wv *= 1.25;
    }
    g.inv_wu = (float)(1.0 / wu);
    g.inv_wv = (float)(1.0 / wv);
    g.u0 = kmin[g.au];
    g.v0 = kmin[g.av];
    g.ncu = ncells(g.au, wu);
    g.ncv = ncells(g.av, wv);
    return g;
}

// Frames per strip block: enough blocks to even out the last of them, few enough flushes (a 3,000
// frame run on 256 CUs: 7.0 ms with 12 blocks per CU, 6.8 with 24, 7.4 with 48).
constexpr double kStripBlocks = 24;
uint32_t strip_chunk(const iac_ctx *ctx, uint32_t nframes, size_t ntasks)
{
    return (uint32_t)std::max(1.0, std::min(64.0, (double)nframes * (double)ntasks / (kStripBlocks * ctx->num_cus)));
}

// Strips of an AC_uw run: ncv of them (0: strips do not pay), a task per `per` distances.
struct StripShape {
    CellGeom g;
    int per;
};

// The records of a run's frames: their root mean square, and the most of one frame.
struct FrameLoad {
    double rms, most;
};
FrameLoad frame_load(const uint64_t *off, uint32_t nframes)
{
    double sum = 0, most = 0;
    for (uint32_t f = 0; f < nframes; f++) {
        const double n = (double)(off[f + 1] - off[f]);
        sum += n * n;
        most = std::max(most, n);
    }
    return FrameLoad{std::sqrt(sum / std::max(1u, nframes)), most};
}

// Waves' loads of a Poisson number of lanes, L on average (erfc(6) is 2e-17).
double wave_loads(double L)
{
    if (L > 64.0 * 30) return L / 64 + 0.5;
    double groups = 1;
    const double sd = std::sqrt(2 * L);
    for (int k = 1; k < 32; k++) {
        const double z = (64.0 * k + 0.5 - L) / sd;
        if (z > 6) break;
        groups += z < -6 ? 1.0 : 0.5 * std::erfc(z);
    }
    return groups;
}

// Tall tasks waste little of their box (it spans per + 1 strips for per of lanes) and flush seldom;
// records of the lanes' strips should fill 64 lanes, or 128, and those of b outweigh the cost of
// starting an item.  The shape of least cost, in clocks of a CU per frame: 27 per 64 pairs (VALU
// issue; 34 with one block per CU, whose flush nothing covers), 7.5 pairs' worth for an item's start,
// 2.7 per voxel flushed to a rotated mesh (scattered atomics) or 1.5 to a plain one, shared
// by a chunk's frames.  Shapes that leave waves or CUs idle pay for it (60 frames of 21,000 photons in
// strips of half the detector: 90 ms, the walk 18), and no shape near the walk's cost
// is taken.  Measured: 34 picks seven-row boxes and 6.5 ms, 27 twelve-row ones and 6.8.  The frames
// count as if each held the root mean square of their records, and a frame of more than twice that
// as the time of its block, which takes a whole task of it (250 lognormal frames of up to 20,000
// photons, four draws: 4.4 to 7.1 ms in few tall strips by the mean alone, 1.6 to 2.3 so; the walk
// 3.2 to 4.2).
StripShape strip_shape(const iac_ctx *ctx, const float kmin[3], const float ext3[3], const PairRun &R,
                       const FrameLoad &load)
{
    StripShape best{};
    CellGeom &g = best.g;
    if (R.spec.kind != kKindAc3d || !fast_path(R.spec, R.ordered) || !(ext3[2] <= ext3[0] && ext3[2] <= ext3[1]))
        return best;
    g.av = ext3[1] >= ext3[0] ? 1 : 0;
    g.au = 1 - g.av;
    const double vox = R.spec.P.vox, wide = std::floor(2 * ext3[g.au] * vox + 2), deep = std::floor(2 * ext3[2] * vox + 2);
    const double tall = ext3[g.av] * vox, rms2 = load.rms * load.rms;
    // a second plan, sort and launch cost about 90 us, 0.3e-12 s per pair against the walk repay it
    // (a rotated mesh's smaller flushes more)
    const double pairs = 0.5 * rms2 * R.nframes;
    if (!(wide * deep * 4 * 3 <= kStripBox1) || !(pairs >= (R.h_rots ? 0x1p26 : 0x1p28))) return best;
    // What the walk takes for the pairs, and at its end for a task of the largest frame (its cells are six
    // voxels; the offset of most pairs holds 2 / cells of them).
    double walk = 0.5 * rms2 / 64 * 55;
    const bool uneven = load.most > 2 * load.rms;
    if (uneven) {
        const double cells = std::ceil(ext3[0] * vox / 6) * std::ceil(ext3[1] * vox / 6);
        walk += 0.5 * load.most * load.most / 64 * 55 * 2 / std::max(2.0, cells) * 3 * ctx->num_cus / R.nframes;
    }
    double least = 1e300, h_best = 0;
    for (int m = 1; m <= 8; m++)
        for (double h = 1; h <= 64; h *= 1.0905) {  // eighths of an octave
            const double rows = std::floor((m + 1) * h + 2), box = rows * wide * deep * 4, n = std::ceil(tall / h);
            if (box > kStripBox1) break;
            if (n > kMaxStrips || n < 2) continue;
            const double L = m * h * load.rms / std::max(1.0, tall), nb = L / m;
            const double items = n * (n + m) / (2.0 * m), tasks = std::ceil(n / m);
            const double frames = R.h_rots ? 1 : strip_chunk(ctx, R.nframes, (size_t)tasks);
            // idle waves where a block has few items, idle CUs where there are few blocks
            const double waves = box > kStripBox2 ? 16 : 8, slots = ctx->num_cus * (box > kStripBox2 ? 1 : 2);
            const double busy = std::min(1.0, frames * items / tasks / (3 * waves)) *
                                std::min(1.0, tasks * R.nframes / frames / (6 * slots));
            const double per_step = items * (box > kStripBox2 ? 34 : 27);
            // (the model is a sixth too high for strips)
            if (per_step * (nb + 7.5) / busy * 0.9 * std::max(1.0, std::min(L / 64, 30.0)) > std::min(1.3 * walk, least))
                continue;
            double pair_cost = per_step * (nb + 7.5) / busy * wave_loads(L);
            if (uneven) {
                // its block has a CU to itself in the end, half of one (of whose SIMDs it fills half) before
                const double x = load.most / load.rms;
                const double late = per_step / tasks * (x * nb + 7.5) * wave_loads(x * L) * (box > kStripBox2 ? 1.5 : 3);
                pair_cost += late * ctx->num_cus / R.nframes;
            }
            if (pair_cost > 1.3 * walk) continue;
            const double cost = pair_cost + tasks * box / 4 * (R.h_rots ? 2.7 : 1.5) / frames;
            if (cost < least) {
                least = cost;
                h_best = h;
                best.per = m;
                g.ncv = (int)n;
            }
        }
    if (g.ncv == 0) return best;
    g.u0 = 0.0f;
    g.inv_wu = 0.0f;
    g.ncu = 1;
    g.v0 = kmin[g.av];
    g.inv_wv = (float)(vox / h_best);
    return best;
}

// Enqueues the per-cell extents of the k-map and their copy to h_cells (valid after a sync).
int cell_extents(hipStream_t st, const float *d_kmap, uint32_t npix, const CellGeom &g, uint32_t *d_cell_ext,
                 uint32_t *h_cells)
{
    const int nc = g.ncu * g.ncv;
    hipLaunchKernelGGL(init_cell_ext_kernel, dim3((nc + 255) / 256), dim3(256), 0, st, d_cell_ext, nc);
    const size_t lds = 6 * sizeof(uint32_t) * (size_t)nc;
    if (lds <= 48 * 1024) {
        const unsigned lb = std::max(1u, std::min<unsigned>(512, (npix + 1023) / 1024));
        hipLaunchKernelGGL(cell_ext_lds_kernel, dim3(lb), dim3(256), lds, st, d_kmap, npix, g, d_cell_ext);
    } else {
        const unsigned eb = std::max(1u, std::min<unsigned>(1024, (npix + 255) / 256));
        hipLaunchKernelGGL(cell_ext_kernel, dim3(eb), dim3(256), 0, st, d_kmap, npix, g, d_cell_ext);
    }
    IAC_HIP(hipGetLastError());
    IAC_HIP(hipMemcpyAsync(h_cells, d_cell_ext, lds, hipMemcpyDeviceToHost, st));
    return IAC_OK;
}

// The plan of a grid and its cell extents, from the context's cache or made.
int plan_of(iac_ctx *ctx, const PairRun &R, int cell_vox, int box_cap, int region, const CellGeom &g,
            const uint32_t *cells, iac_pair_plan **out)
{
    const PairSpec &S = R.spec;
    std::vector<uint32_t> cext(cells, cells + 6 * (size_t)g.ncu * g.ncv);
    iac_pair_plan *pl = find_plan(ctx, R.d_kmap, R.npix, cell_vox, box_cap, region, S);
    if (pl && (std::memcmp(&pl->g, &g, sizeof(g)) != 0 || pl->cell_ext != cext)) pl = nullptr;
    if (!pl) {
        // reuse the oldest unpinned slot beyond the cached plans; a geometry holds at most five (the
        // walk's and the strips', or the walk's and four region sides that do not fit)
        if (ctx->pair_plans.size() >= kMaxPlans) {
            for (auto it = ctx->pair_plans.begin(); it != ctx->pair_plans.end(); ++it) {
                if ((*it)->pins > 0) continue;
                if ((*it)->d_tasks) IAC_HIP(hipFree((*it)->d_tasks));
                if ((*it)->d_tiles) IAC_HIP(hipFree((*it)->d_tiles));
                delete *it;
                ctx->pair_plans.erase(it);
                break;
            }
        }
        pl = new iac_pair_plan();
        ctx->pair_plans.push_back(pl);
        pl->kmap = R.d_kmap;
        pl->npix = R.npix;
        pl->cell_vox = cell_vox;
        pl->box_cap = box_cap;
        pl->region = region;
        pl->spec = S;
        pl->g = g;
        pl->cell_ext.swap(cext);
        if (region == kRegionTiles) {
            build_tiles(*pl, R.ordered);
            if (pl->tiles_fit) {
                IAC_HIP(hipMalloc(&pl->d_tiles, pl->tiles.size() * sizeof(TileTask)));
                IAC_HIP(hipMemcpy(pl->d_tiles, pl->tiles.data(), pl->tiles.size() * sizeof(TileTask),
                                  hipMemcpyHostToDevice));
            }
        } else {
            build_tasks(*pl, R.ordered);
            if (region <= kRegionStrips) merge_strips(*pl, kRegionStrips - region);
            if (pl->tasks.size() > kMaxGridBlocks)
                return fail(IAC_ERR_LIMIT,
                            "pair engine: more than 2^22 tasks (raise the task region or the cell size)");
            if (!pl->tasks.empty()) {
                IAC_HIP(hipMalloc(&pl->d_tasks, pl->tasks.size() * sizeof(Task)));
                IAC_HIP(hipMemcpy(pl->d_tasks, pl->tasks.data(), pl->tasks.size() * sizeof(Task),
                                  hipMemcpyHostToDevice));
            }
        }
        pl->valid = true;
    }
    *out = pl;
    return IAC_OK;
}

bool default_options(iac_ctx *ctx);

// Cell grid of the k-map (two host round trips for the extents) and the task
// table, from the context's cache when the geometry matches.  h_off: also the frames' offsets,
// read back with them (valid until the context's next call).
// strips (with h_off): also the plan of the run's strips (null where they do not suit it).
int get_plan(iac_ctx *ctx, hipStream_t st, const PairRun &R, int cell_vox, int box_cap, int region,
             iac_pair_plan **out, const uint64_t **h_off = nullptr, iac_pair_plan **strips = nullptr)
{
    void *ext = nullptr;
    IAC_TRY(scratch(ctx, 3, (6 + 6 * (size_t)(kMaxCells + kMaxStrips)) * sizeof(uint32_t), &ext));
    uint32_t *d_ext = static_cast<uint32_t *>(ext);
    const size_t off_bytes = h_off ? ((size_t)R.nframes + 1) * sizeof(uint64_t) : 0;
    PlanRead read;
    IAC_TRY(plan_read(ctx, off_bytes, &read));
    if (h_off) {
        IAC_HIP(hipMemcpyAsync(read.more, R.d_frame_off, off_bytes, hipMemcpyDeviceToHost, st));
        *h_off = read.more;
    }
    float kmin[3], ext3[3];
    IAC_TRY(kmap_extents(st, R.d_kmap, R.npix, d_ext, read, kmin, ext3));
    const CellGeom g = cell_grid(kmin, ext3, R.spec.P.vox, cell_vox);
    IAC_TRY(cell_extents(st, R.d_kmap, R.npix, g, d_ext + 6, read.cells));
    StripShape shape{};
    const CellGeom &sg = shape.g;
    if (strips) {
        *strips = nullptr;
        if (default_options(ctx)) shape = strip_shape(ctx, kmin, ext3, R, frame_load(*h_off, R.nframes));
        if (sg.ncv > 0) IAC_TRY(cell_extents(st, R.d_kmap, R.npix, sg, d_ext + 6 + 6 * kMaxCells, read.strips));
    }
    IAC_HIP(hipStreamSynchronize(st));
    IAC_TRY(plan_of(ctx, R, cell_vox, box_cap, region, g, read.cells, out));
    if (sg.ncv > 0) {
        (*out)->pins++;  // stays while the strips' plan takes a place in the cache
        iac_pair_plan *sp = nullptr;
        const int rc = plan_of(ctx, R, sg.ncv, (int)(kStripBox1 / 4), kRegionStrips - shape.per, sg, read.strips, &sp);
        (*out)->pins--;
        if (rc != IAC_OK) return rc;
        bool fit = !sp->tasks.empty();
        for (const Task &t : sp->tasks) fit = fit && t.inbox;  // every pair lands in the box, inside the mesh
        if (fit) *strips = sp;
    }
    return IAC_OK;
}

// A context without engine options set: the options name the walk's settings, so they select it
// (the autotuner's, which were measured on AC_uw, say nothing about the tiles of C(q)).
bool default_options(iac_ctx *ctx)
{
    return !(ctx->pair_mode || ctx->cell_vox || ctx->cell_vox_v || ctx->box_cap || ctx->task_region ||
             ctx->pair_prefetch || ctx->frame_chunk);
}

// Frame chunks inside each group, balanced by pair work: a chunk closes once its
// frames' n^2 reach fchunk times the mean per frame, or at 4 fchunk frames.
std::vector<Chunk> make_chunks(const uint64_t *off, uint32_t nframes, const uint32_t *group_off, uint32_t ngroups,
                               uint32_t fchunk, const float *h_rots = nullptr)
{
    double total = 0;
    for (uint32_t f = 0; f < nframes; f++) {
        const double n = (double)(off[f + 1] - off[f]);
        total += n * n;
    }
    // fchunk mean frames of pair work, at most 2^28 pairs: dense frames (C(q) images hold
    // P^2 pairs) become chunks of one frame, so a run still spreads over many blocks
    const double budget = std::max(1.0, std::min(total / std::max(1u, nframes) * fchunk, 268435456.0));
    const uint32_t fmax = std::min<uint32_t>(4 * fchunk, 4096);  // items per chunk < 2^24 (pairs_kernel)
    std::vector<Chunk> chunks;
    for (uint32_t gi = 0; gi < ngroups; gi++) {
        uint32_t f0 = group_off[gi];
        double acc = 0;
        for (uint32_t f = group_off[gi]; f < group_off[gi + 1]; f++) {
            const double n = (double)(off[f + 1] - off[f]);
            acc += n * n;
            // per-frame rotations: a chunk ends where the next frame's rotation differs
            const bool rot_break = h_rots && f + 1 < group_off[gi + 1] &&
                                   std::memcmp(h_rots + 9 * (size_t)f0, h_rots + 9 * (size_t)(f + 1), 36) != 0;
            if (acc >= budget || f + 1 - f0 >= fmax || rot_break) {
                chunks.push_back(Chunk{f0, f + 1, gi});
                f0 = f + 1;
                acc = 0;
            }
        }
        if (f0 < group_off[gi + 1]) chunks.push_back(Chunk{f0, group_off[gi + 1], gi});
    }
    return chunks;
}

// The pair kernel reads a chunk's records at 32-bit byte offsets from its first record: every
// chunk spans fewer than 2^28 records (the chunk budget keeps a chunk's other frames to a few
// million records, so only a single frame of ~2^28 records can break this).
int check_chunks(const uint64_t *off, const std::vector<Chunk> &chunks)
{
    for (const Chunk &c : chunks)
        if (off[c.f1] - off[c.f0] >= (1ull << 28))
            return fail(IAC_ERR_LIMIT, "pair engine: a frame chunk of 2^28 or more records (split the frame)");
    return IAC_OK;
}

struct Bufs {
    float4 *srec;
    uint32_t *cs;
    unsigned long long *H;  // symmetric modes: ngroups half-mesh accumulators
    uint32_t *d_goff;
    unsigned long long *d_self;
    uint32_t *d_flag;  // 1 while every weight of the run is a small integer (after d_self)
    Chunk *d_chunks;
    uint32_t nchunks;
    const Task *d_tasks;
    uint32_t ntasks;
    CellGeom g;
    int box_cap;
    // strips (nst == 0: none)
    float4 *st_rec;
    uint32_t *st_cs, *st_bound, *st_usable;
    unsigned long long *st_self;
    Chunk *st_chunks;
    uint32_t st_nchunks;
    const Task *st_tasks;
    uint32_t nst;
    StripGeom st_g;
    size_t st_box;  // bytes of the largest box
};

// per frame, the records of its fullest cell: after the frames' cell starts
uint32_t *cell_max(const PairRun &R, const Bufs &b)
{
    return b.cs + (size_t)R.nframes * (b.g.ncu * b.g.ncv + 1);
}

template <int K, bool O, int BOX>
void launch_pairs_box(int pf, bool fast, int walk, dim3 grid, hipStream_t st, const PairRun &R, const Bufs &b,
                      unsigned long long *target, size_t nvox, unsigned long long *dropped)
{
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(kBlock), 0, st, b.srec, R.d_frame_off, b.cs, b.d_chunks, b.d_tasks,
                           b.ntasks, b.g, R.spec, target, nvox, dropped, b.d_flag, R.d_rots, cell_max(R, b),
                           b.nst ? b.st_usable : nullptr);
    };
    constexpr bool kFast = K == kKindAc3d && !O;
    if constexpr (kFast && BOX == kBoxSmall) {
        if (b.nst) return go(pairs_kernel<K, O, 0, kFast, BOX, true>);
    }
    if ((O || pf == 1) && fast) {
        if (walk) go(pairs_kernel<K, O, 0, kFast, BOX>);
        else go(pairs_kernel<K, O, 1, kFast, BOX>);
    } else if (O || pf == 1 || BOX != kBoxMax) {
        if (walk) go(pairs_kernel<K, O, 0, false, BOX>);
        else go(pairs_kernel<K, O, 1, false, BOX>);
    } else if (pf == 4) {
        go(pairs_kernel<K, O, O ? 1 : 4, false, BOX>);
    } else {
        go(pairs_kernel<K, O, O ? 1 : 8, false, BOX>);
    }
}

// walk: lanes on consecutive pairs (1) or a contiguous pair range per thread (0)
template <int K, bool O>
void launch_pairs(int pf, int walk, dim3 grid, hipStream_t st, const PairRun &R, const Bufs &b,
                  unsigned long long *target, size_t nvox, unsigned long long *dropped)
{
    const bool fast = fast_path(R.spec, O);
    if (b.box_cap == kBoxSmall)
        launch_pairs_box<K, O, kBoxSmall>(pf, fast, walk, grid, st, R, b, target, nvox, dropped);
    else if (b.box_cap == kBoxTiny)
        launch_pairs_box<K, O, kBoxTiny>(pf, fast, walk, grid, st, R, b, target, nvox, dropped);
    else
        launch_pairs_box<K, O, kBoxMax>(pf, fast, walk, grid, st, R, b, target, nvox, dropped);
}

// Everything after planning, enqueue only (no host synchronisation, no
// allocation, fills by kernel): capturable into a graph.
bool walks(iac_ctx *ctx, const PairRun &R);

int enqueue(iac_ctx *ctx, hipStream_t st, const PairRun &R, const Bufs &prepared, bool timed)
{
    // a batch prepared with strips, launched with an engine option set since: the option's walk
    Bufs b = prepared;
    if (!default_options(ctx)) b.nst = 0;
    const PairSpec &S = R.spec;
    const bool ordered = R.ordered;
    const size_t nvox = (size_t)S.P.sab * S.P.sab * S.P.sc;
    const unsigned zb = (unsigned)std::max<size_t>(1, std::min<size_t>(4096, (nvox * R.ngroups + 255) / 256));
    if (!ordered) {
        hipLaunchKernelGGL(fill_u64_kernel, dim3(zb), dim3(256), 0, st, b.H, nvox * R.ngroups);
        hipLaunchKernelGGL(fill_u64_kernel, dim3(1), dim3(256), 0, st, b.d_self, (size_t)R.ngroups);
    }
    hipLaunchKernelGGL(fill_u32_kernel, dim3(1), dim3(64), 0, st, b.d_flag, 1u, (size_t)1);
    if (b.nst) {
        hipLaunchKernelGGL(fill_u64_kernel, dim3(1), dim3(256), 0, st, b.st_self, (size_t)R.ngroups);
        hipLaunchKernelGGL(fill_u32_kernel, dim3(1), dim3(64), 0, st, b.st_usable, 1u, (size_t)1);
        hipLaunchKernelGGL(strip_sort_kernel, dim3(R.nframes), dim3(kBlock), 0, st, R.rec, R.d_frame_off, b.st_g,
                           b.st_rec, b.st_cs, S, b.d_goff, R.ngroups, b.st_self, b.st_usable, b.st_bound);
        IAC_HIP(hipGetLastError());
    }
    if (S.kind == kKindAc3d) {
        if (ordered)
            hipLaunchKernelGGL((cell_sort_kernel<kKindAc3d, true>), dim3(R.nframes), dim3(kBlock), 0, st, R.rec,
                               R.d_frame_off, b.g, b.srec, b.cs, S, b.d_goff, R.ngroups, b.d_self, b.d_flag, cell_max(R, b),
                               b.nst ? b.st_usable : nullptr, ctx->d_counters + kPathCounter);
        else
            hipLaunchKernelGGL((cell_sort_kernel<kKindAc3d, false>), dim3(R.nframes), dim3(kBlock), 0, st, R.rec,
                               R.d_frame_off, b.g, b.srec, b.cs, S, b.d_goff, R.ngroups, b.d_self, b.d_flag, cell_max(R, b),
                               b.nst ? b.st_usable : nullptr, ctx->d_counters + kPathCounter);
    } else {
        if (ordered)
            hipLaunchKernelGGL((cell_sort_kernel<kKindCq, true>), dim3(R.nframes), dim3(kBlock), 0, st, R.rec,
                               R.d_frame_off, b.g, b.srec, b.cs, S, b.d_goff, R.ngroups, b.d_self, b.d_flag, cell_max(R, b),
                               b.nst ? b.st_usable : nullptr, ctx->d_counters + kPathCounter);
        else
            hipLaunchKernelGGL((cell_sort_kernel<kKindCq, false>), dim3(R.nframes), dim3(kBlock), 0, st, R.rec,
                               R.d_frame_off, b.g, b.srec, b.cs, S, b.d_goff, R.ngroups, b.d_self, b.d_flag, cell_max(R, b),
                               b.nst ? b.st_usable : nullptr, ctx->d_counters + kPathCounter);
    }
    IAC_HIP(hipGetLastError());
    auto *target = ordered ? reinterpret_cast<unsigned long long *>(R.d_mesh) : b.H;
    if (b.ntasks && b.nchunks) {
        if (timed) IAC_TRY(timer_begin(ctx));
        // ordered (linear) binning holds eight corner adds per pair in registers: no batching there
        const int pf = ordered || ctx->pair_prefetch == 0 || ctx->pair_prefetch == 1 ? 1 : (ctx->pair_prefetch == 4 ? 4 : 8);
        // block = chunk * ntasks + task; whole chunks per launch, the slice's chunks by pointer
        const int walk = walks(ctx, R) ? 1 : 0;
        if (b.nst) {
            const bool wide = b.st_box > kStripBox2;  // one block of 1,024 threads per CU, or two of 512
            auto kern = b.st_g.g.av == 0 ? (wide ? strip_kernel<0, 1024> : strip_kernel<0, 512>)
                                       : (wide ? strip_kernel<1, 1024> : strip_kernel<1, 512>);
            const uint32_t sper = std::max<uint32_t>(1, kMaxGridBlocks / b.nst);
            for (uint32_t c0 = 0; c0 < b.st_nchunks; c0 += sper) {
                hipLaunchKernelGGL(kern, dim3(b.nst * std::min(sper, b.st_nchunks - c0)), dim3(wide ? 1024 : 512), b.st_box,
                                   st, b.st_rec, R.d_frame_off, b.st_cs, b.st_chunks + c0, b.st_tasks, b.nst, b.st_g.g.ncv,
                                   S, target, nvox, ctx->d_counters, b.st_usable, b.st_bound, R.d_rots);
                IAC_HIP(hipGetLastError());
            }
        }
        const uint32_t per = std::max<uint32_t>(1, kMaxGridBlocks / b.ntasks);
        for (uint32_t c0 = 0; c0 < b.nchunks; c0 += per) {
            Bufs bs = b;
            bs.d_chunks = b.d_chunks + c0;
            const dim3 grid(b.ntasks * std::min(per, b.nchunks - c0));
            if (S.kind == kKindAc3d) {
                if (ordered) launch_pairs<kKindAc3d, true>(pf, walk, grid, st, R, bs, target, nvox, ctx->d_counters);
                else launch_pairs<kKindAc3d, false>(pf, walk, grid, st, R, bs, target, nvox, ctx->d_counters);
            } else {
                if (ordered) launch_pairs<kKindCq, true>(pf, walk, grid, st, R, bs, target, nvox, ctx->d_counters);
                else launch_pairs<kKindCq, false>(pf, walk, grid, st, R, bs, target, nvox, ctx->d_counters);
            }
            IAC_HIP(hipGetLastError());
        }
        if (timed) IAC_TRY(timer_end(ctx));
    }
    if (!ordered) {
        const size_t centre = (size_t)S.P.c0 + (size_t)S.P.c1 * S.P.sab + (size_t)S.P.c2 * S.P.sab * S.P.sab;
        hipLaunchKernelGGL(symmetrize_kernel, dim3(zb), dim3(256), 0, st, b.H,
                           reinterpret_cast<unsigned long long *>(R.d_mesh), nvox, R.ngroups, centre, b.d_self,
                           b.nst ? b.st_self : b.d_self, b.nst ? b.st_usable : nullptr);
        IAC_HIP(hipGetLastError());
    }
    return IAC_OK;
}

// Defaults from the tuner (bench.py sweeps and the ordered-mode measurements):
//   AC_uw nearest neighbour, identity rotation: lanes on consecutive pairs, 6-voxel cells,
//     1920-voxel boxes (1024^2 sparse and lognormal workloads);
//   AC_uw linear (ordered): lanes on consecutive pairs, 5-voxel cells, 4096-voxel boxes
//     (64 LDS adds per pair with a linear first level: LDS-atomic bound);
//   C(q) nearest neighbour: lanes on consecutive pairs, 3-voxel cells, 1920-voxel boxes,
//     4 x 4-cell task regions (dense 256^2 images);
//   C(q) linear: a pair range per thread, 4-voxel cells, 4096-voxel boxes, regions of 4.
bool walks(iac_ctx *ctx, const PairRun &R)
{
    if (ctx->pair_mode == 1) return true;
    if (ctx->pair_mode == 2) return false;
    // C(q) of dense frames: a pair range per thread, whose runs of one voxel add in a register
    return R.spec.kind != kKindCq;
}
int cell_vox_of(iac_ctx *ctx, const PairRun &R)
{
    int dflt = 4;
    if (R.spec.kind == kKindCq && !R.ordered) dflt = 3;
    else if (walks(ctx, R)) dflt = R.ordered ? 5 : (fast_path(R.spec, R.ordered) ? 6 : 4);
    const int u = ctx->cell_vox > 0 ? ctx->cell_vox : dflt;
    return u + 1000 * (ctx->cell_vox_v > 0 ? ctx->cell_vox_v : u);
}
int box_cap_of(iac_ctx *ctx, const PairRun &R)
{
    if (ctx->box_cap == kBoxMax || ctx->box_cap == kBoxTiny) return ctx->box_cap;
    if (ctx->box_cap == kBoxSmall || ctx->box_cap == 2048) return kBoxSmall;
    return R.ordered ? kBoxMax : kBoxSmall;
}
int region_of(iac_ctx *ctx, const PairRun &R)
{
    if (ctx->task_region > 0) return ctx->task_region;
    if (R.spec.kind != kKindCq) return 0;
    return R.ordered ? 4 : 2;
}
uint32_t fchunk_of(iac_ctx *ctx) { return ctx->frame_chunk > 0 ? ctx->frame_chunk : 32; }

// byte sizes of the per-run buffers
struct Sizes {
    size_t srec, cs, h, goff, self, chunks;
};
Sizes sizes_of(const PairRun &R, int nc, size_t nchunks)
{
    const size_t nvox = (size_t)R.spec.P.sab * R.spec.P.sab * R.spec.P.sc;
    auto up = [](size_t x) { return (x + 255) / 256 * 256; };
    return Sizes{up(R.n_total * sizeof(float4)),
                 up((size_t)R.nframes * (nc + 2) * sizeof(uint32_t)),  // cell starts, then the fullest cells
                 R.ordered ? 0 : nvox * R.ngroups * sizeof(unsigned long long),
                 up((R.ngroups + 1) * sizeof(uint32_t)),
                 up(R.ngroups * sizeof(unsigned long long) + sizeof(uint32_t)),
                 up(std::max<size_t>(1, nchunks) * sizeof(Chunk))};
}

// Bytes of a run's strip buffers, and their places from p on.
size_t strip_bytes(const PairRun &R, const iac_pair_plan *sp, size_t nchunks)
{
    if (!sp) return 0;
    auto up = [](size_t x) { return (x + 255) / 256 * 256; };
    return up(R.n_total * sizeof(float4)) + up((size_t)R.nframes * (sp->g.ncv + 2) * sizeof(uint32_t)) +
           up((R.ngroups + 1) * sizeof(unsigned long long)) + up(std::max<size_t>(1, nchunks) * sizeof(Chunk));
}
void strip_place(Bufs &b, char *p, const PairRun &R, const iac_pair_plan *sp, size_t nchunks)
{
    b.nst = 0;
    if (!sp) return;
    auto up = [](size_t x) { return (x + 255) / 256 * 256; };
    b.st_rec = reinterpret_cast<float4 *>(p);
    p += up(R.n_total * sizeof(float4));
    b.st_cs = reinterpret_cast<uint32_t *>(p);
    b.st_bound = b.st_cs + (size_t)R.nframes * (sp->g.ncv + 1);
    p += up((size_t)R.nframes * (sp->g.ncv + 2) * sizeof(uint32_t));
    b.st_self = reinterpret_cast<unsigned long long *>(p);
    b.st_usable = reinterpret_cast<uint32_t *>(b.st_self + R.ngroups);
    p += up((R.ngroups + 1) * sizeof(unsigned long long));
    b.st_chunks = reinterpret_cast<Chunk *>(p);
    b.st_nchunks = (uint32_t)nchunks;
    b.st_tasks = sp->d_tasks;
    b.nst = (uint32_t)sp->tasks.size();
    // (strips are one voxel tall or at least 9 % taller)
    b.st_g = StripGeom{sp->g, FLT_MAX, -FLT_MAX, 0.0f, sp->g.inv_wv < 0.95f * R.spec.P.vox ? 2 : 3};
    float zlo = FLT_MAX, zhi = -FLT_MAX;
    for (int c = 0; c < sp->g.ncv; c++) {
        const uint32_t *e = &sp->cell_ext[6 * (size_t)c];
        if (e[0] == 0xffffffffu) continue;  // no pixel there
        b.st_g.ulo = std::min(b.st_g.ulo, unkey(e[sp->g.au]));
        b.st_g.uhi = std::max(b.st_g.uhi, unkey(e[3 + sp->g.au]));
        zlo = std::min(zlo, unkey(e[2]));
        zhi = std::max(zhi, unkey(e[5]));
    }
    b.st_g.zext = zhi - zlo;
    b.st_box = sp->tile_box;
}

}  // namespace

void free_pair_plans(iac_ctx *ctx)
{
    for (auto *p : ctx->pair_plans) {
        if (p->d_tasks) (void)hipFree(p->d_tasks);
        if (p->d_tiles) (void)hipFree(p->d_tiles);
        delete p;
    }
    ctx->pair_plans.clear();
}

namespace {
// The group offsets and the chunk tables to the device, through page-locked staging: the host does
// not wait for the copies.
int upload_tables(iac_ctx *ctx, hipStream_t st, const PairRun &R, const std::vector<Chunk> &chunks,
                  const std::vector<Chunk> &schunks, uint32_t *d_goff, Chunk *d_chunks, Chunk *d_schunks)
{
    const size_t bg = (R.ngroups + 1) * sizeof(uint32_t), bc = chunks.size() * sizeof(Chunk);
    const size_t bs = schunks.size() * sizeof(Chunk);
    void *p = nullptr;
    IAC_TRY(pinned(ctx, 1, bg + bc + bs, &p));
    char *c = static_cast<char *>(p);
    auto put = [&](void *dst, const void *src, size_t n) -> int {
        if (!n) return IAC_OK;
        std::memcpy(c, src, n);
        IAC_HIP(hipMemcpyAsync(dst, c, n, hipMemcpyHostToDevice, st));
        c += n;
        return IAC_OK;
    };
    IAC_TRY(put(d_goff, R.h_group_off, bg));
    IAC_TRY(put(d_chunks, chunks.data(), bc));
    IAC_TRY(put(d_schunks, schunks.data(), bs));
    return upload_done(ctx);
}
}  // namespace

int pairs_run(iac_ctx *ctx, const PairRun &R)
{
    hipStream_t st = ctx->stream;
    if (R.n_total >= (1ull << 32)) return fail(IAC_ERR_LIMIT, "pair engine: at most 2^32 - 1 records per call");
    iac_pair_plan *pl = nullptr;
    const uint64_t *off = nullptr;
    iac_pair_plan *sp = nullptr;
    IAC_TRY(get_plan(ctx, st, R, cell_vox_of(ctx, R), box_cap_of(ctx, R), region_of(ctx, R), &pl, &off, &sp));
    const std::vector<Chunk> chunks = make_chunks(off, R.nframes, R.h_group_off, R.ngroups, fchunk_of(ctx), R.h_rots);
    IAC_TRY(check_chunks(off, chunks));
    std::vector<Chunk> schunks;
    if (sp)
        schunks = make_chunks(off, R.nframes, R.h_group_off, R.ngroups, strip_chunk(ctx, R.nframes, sp->tasks.size()), R.h_rots);
    const int nc = pl->g.ncu * pl->g.ncv;
    const Sizes z = sizes_of(R, nc, chunks.size());
    // scratch: sorted records + cell offsets (slot 1), H + group offsets + self + chunks (slot 2)
    void *s1 = nullptr, *s2 = nullptr;
    if (sp) {
        IAC_TRY(scratch_if(ctx, 1, z.srec + z.cs + strip_bytes(R, sp, schunks.size()), &s1));
        if (!s1) {  // the walk needs 16 bytes per record less
            sp = nullptr;
            schunks.clear();
        }
    }
    if (!s1) IAC_TRY(scratch(ctx, 1, z.srec + z.cs, &s1));
    IAC_TRY(scratch(ctx, 2, z.h + z.goff + z.self + z.chunks, &s2));
    Bufs b{};
    strip_place(b, static_cast<char *>(s1) + z.srec + z.cs, R, sp, schunks.size());
    b.srec = static_cast<float4 *>(s1);
    b.cs = reinterpret_cast<uint32_t *>(static_cast<char *>(s1) + z.srec);
    char *p2 = static_cast<char *>(s2);
    b.H = reinterpret_cast<unsigned long long *>(p2);
    b.d_goff = reinterpret_cast<uint32_t *>(p2 + z.h);
    b.d_self = reinterpret_cast<unsigned long long *>(p2 + z.h + z.goff);
    b.d_flag = reinterpret_cast<uint32_t *>(b.d_self + R.ngroups);
    b.d_chunks = reinterpret_cast<Chunk *>(p2 + z.h + z.goff + z.self);
    b.nchunks = (uint32_t)chunks.size();
    b.d_tasks = pl->d_tasks;
    b.ntasks = (uint32_t)pl->tasks.size();
    b.g = pl->g;
    b.box_cap = pl->box_cap;
    IAC_TRY(upload_tables(ctx, st, R, chunks, schunks, b.d_goff, b.d_chunks, b.st_chunks));
    return enqueue(ctx, st, R, b, true);
}

int pairs_strips_suit(iac_ctx *ctx, const PairRun &R, const uint64_t *h_off, bool *suit)
{
    void *ext = nullptr;
    IAC_TRY(scratch(ctx, 3, 6 * sizeof(uint32_t), &ext));
    PlanRead read;
    IAC_TRY(plan_read(ctx, 0, &read));
    float kmin[3], ext3[3];
    IAC_TRY(kmap_extents(ctx->stream, R.d_kmap, R.npix, static_cast<uint32_t *>(ext), read, kmin, ext3));
    *suit = strip_shape(ctx, kmin, ext3, R, frame_load(h_off, R.nframes)).g.ncv > 0;
    return IAC_OK;
}

// ---- dense C(q) -----------------------------------------------------------------

// Region side in voxels: the largest of these that makes kTileTasks tasks or more (smaller regions
// flush more boxes per pair).
constexpr int kTileSides[] = {12, 8, 6, 4};
constexpr double kTileTasks = 2048;
// mean records per region and frame below which most of a wave's 64 lanes idle and the engine's
// pair ranges take the run
constexpr double kTileRecords = 32;
// Blocks wanted, and the least pairs per block: a 350 x 350 image into 35 x 35 x 3 has 325 tasks
// of 2.4e7 pairs and takes 46 ms with one block each, 7 ms split (384 x 360 into 129 x 129 x 3,
// 2,080 tasks of 5.3e6: 8.6 and 6.1 ms).
constexpr double kTileBlocks = 16384, kTileShare = 65536;
// Mean records per voxel-sized part from which tasks add up parts in registers, pair by pair
// below: 12.1 against 10.5 ms at 16 records (eight 256^2 images into 129 x 129 x 3), 5.6 against
// 6.1 ms at 33 (384 x 360), 5.1 against 7.0 ms at 306 (350 x 350 into 35 x 35 x 3).
constexpr double kPartRecords = 24;

int cq_tiles_run(iac_ctx *ctx, const PairRun &R, const float *d_frames, bool *done)
{
    *done = false;
    const PairSpec &S = R.spec;
    const bool ordered = R.ordered;
    if (!default_options(ctx) && !(ctx->tuned && ctx->pair_prefetch == 0)) return IAC_OK;
    // what the walk refuses (pairs_run, check_chunks) stays refused
    if (R.n_total >= (1ull << 32) || R.npix >= (1u << 28)) return IAC_OK;
    // round_away and the boxes' 24-bit products need |q vox| < 2^22
    if (!(std::sqrt((double)S.P.cut_sq) * S.P.vox < 4194304.0) || R.nframes == 0) return IAC_OK;
    hipStream_t st = ctx->stream;
    const uint32_t ns = std::min<uint32_t>(256, (R.npix + kBlock - 1) / kBlock);  // sort blocks per frame
    if ((uint64_t)ns * R.nframes > 0x7fffffffull) return IAC_OK;
    // the k-map's extents | kept, flags | the cells' extents, a grid for each side
    constexpr size_t nsides = sizeof(kTileSides) / sizeof(kTileSides[0]);
    void *ext = nullptr;
    IAC_TRY(scratch(ctx, 3, (kHead + 6 * (size_t)(nsides * kMaxCells)) * sizeof(uint32_t), &ext));
    uint32_t *d_ext = static_cast<uint32_t *>(ext);
    auto *d_kept = reinterpret_cast<unsigned long long *>(d_ext + 8);
    auto *d_plain = reinterpret_cast<uint32_t *>(d_kept + 1);
    uint32_t *d_cells = d_ext + kHead;
    float kmin[3], ext3[3];
    PlanRead read;
    IAC_TRY(plan_read(ctx, 0, &read));
    hipLaunchKernelGGL(cq_begin_kernel, dim3(1), dim3(64), 0, st, d_ext, d_kept, d_plain);
    hipLaunchKernelGGL(dense_scan_kernel, dim3((unsigned)std::min<uint64_t>(2048, (R.n_total + 4 * kBlock - 1) / (4 * kBlock))),
                       dim3(kBlock), 0, st, d_frames, R.n_total, S.mult, d_kept, d_plain);
    IAC_TRY(kmap_extents_enqueue(st, R.d_kmap, R.npix, d_ext, read, kHead));
    IAC_HIP(hipStreamSynchronize(st));
    kmap_extents_read(read, kmin, ext3);
    uint64_t kept = 0;
    std::memcpy(&kept, read.kext + 8, sizeof(kept));
    const uint32_t *flags = read.kext + 10;
    const bool wide = !flags[0];
    if (!flags[1]) return IAC_OK;  // negative values: the engine's pairs test each
    const int box_cap = ordered ? kBoxMax : kBoxSmall;
    const size_t nvox = (size_t)S.P.sab * S.P.sab * S.P.sc;
    // the sides of enough tasks whose regions hold enough records
    struct Side {
        int side;
        CellGeom g;
    } sides[nsides];
    size_t n = 0;
    for (size_t k = 0; k < nsides; k++) {
        const CellGeom g = cell_grid(kmin, ext3, S.P.vox, kTileSides[k]);
        const int nc = g.ncu * g.ncv;
        const double ntask = ordered ? (double)nc * nc : 0.5 * nc * (nc + 1.0);
        if (ntask > kMaxGridBlocks || (double)kept < kTileRecords * (double)R.nframes * nc) break;
        if (ntask * R.ngroups < kTileTasks && k + 1 < nsides) continue;
        sides[n++] = Side{kTileSides[k], g};
    }
    if (n == 0) return IAC_OK;
    // Boxes of regions this size fit wherever in the mesh they lie: the plan can wait for the sort's
    // read-back.  Otherwise (a detector near or tilted) the sides' extents come first, in one go, so
    // that nothing is sorted for a side that does not fit.
    auto fits = [&](const CellGeom &g) {
        const int third = 3 - g.au - g.av, more = ordered ? 3 : 2;
        const double u = S.P.vox / (double)g.inv_wu, v = S.P.vox / (double)g.inv_wv, z = ext3[third] * (double)S.P.vox;
        return (std::floor(2 * u) + more) * (std::floor(2 * v) + more) * (std::floor(2 * z) + more) <= box_cap;
    };
    size_t first = 0;
    iac_pair_plan *pl = nullptr;
    if (!fits(sides[0].g)) {
        const size_t each = 6 * (size_t)kMaxCells;
        IAC_TRY(plan_read(ctx, nsides * each * sizeof(uint32_t), &read));
        uint32_t *h_cells = reinterpret_cast<uint32_t *>(read.more);
        for (size_t k = 0; k < n; k++)
            IAC_TRY(cell_extents(st, R.d_kmap, R.npix, sides[k].g, d_cells + k * each, h_cells + k * each));
        IAC_HIP(hipStreamSynchronize(st));
        for (first = 0; first < n; first++) {
            IAC_TRY(plan_of(ctx, R, sides[first].side, box_cap, kRegionTiles, sides[first].g, h_cells + first * each, &pl));
            if (pl->tiles_fit) break;
        }
    }
    for (size_t k = first; k < n; k++) {
        const int side = sides[k].side;
        const CellGeom &g = sides[k].g;
        const int nc = g.ncu * g.ncv;
        const double ntask = ordered ? (double)nc * nc : 0.5 * nc * (nc + 1.0);
        // chunks: a group's frames in as many blocks as fill the chip
        const uint32_t split = (uint32_t)std::max(1.0, std::ceil(kTileTasks / (ntask * R.ngroups)));
        std::vector<Chunk> chunks;
        for (uint32_t gi = 0; gi < R.ngroups; gi++) {
            const uint32_t f0 = R.h_group_off[gi], n = R.h_group_off[gi + 1] - f0, parts = std::min(split, n);
            for (uint32_t c = 0; c < parts; c++)
                chunks.push_back(Chunk{f0 + (uint32_t)((uint64_t)n * c / parts),
                                       f0 + (uint32_t)((uint64_t)n * (c + 1) / parts), gi});
        }
        auto up = [](size_t x) { return (x + 255) / 256 * 256; };
        // records | region starts | cursors (slot 1); half meshes | group offsets | self | chunks (slot 2)
        const size_t nkey = (size_t)nc * side * side;
        const size_t brec = up((size_t)R.npix * R.nframes * sizeof(float4)),
                     bcs = up(R.nframes * (nkey + 1) * sizeof(uint32_t)),
                     bcur = up(R.nframes * nkey * sizeof(uint32_t));
        const size_t bh = ordered ? 0 : up(nvox * R.ngroups * sizeof(unsigned long long)),
                     bg = up((R.ngroups + 1) * sizeof(uint32_t)), bs = up(R.ngroups * sizeof(unsigned long long));
        void *s1 = nullptr, *s2 = nullptr;
        IAC_TRY(scratch_if(ctx, 1, brec + bcs + bcur, &s1));
        if (!s1) return IAC_OK;  // the keys take up to 36 bytes per pixel; the walk needs none
        IAC_TRY(scratch(ctx, 2, bh + bg + bs + chunks.size() * sizeof(Chunk) + 256, &s2));
        char *p1 = static_cast<char *>(s1), *p2 = static_cast<char *>(s2);
        auto *srec = reinterpret_cast<float4 *>(p1);
        auto *cs = reinterpret_cast<uint32_t *>(p1 + brec);
        auto *cursor = reinterpret_cast<uint32_t *>(p1 + brec + bcs);
        auto *H = reinterpret_cast<unsigned long long *>(p2);
        auto *d_goff = reinterpret_cast<uint32_t *>(p2 + bh);
        auto *d_self = reinterpret_cast<unsigned long long *>(p2 + bh + bg);
        auto *d_chunks = reinterpret_cast<Chunk *>(p2 + bh + bg + bs);
        IAC_TRY(upload_tables(ctx, st, R, chunks, {}, d_goff, d_chunks, nullptr));
        if (!pl) IAC_TRY(cell_extents(st, R.d_kmap, R.npix, g, d_cells, read.cells));
        auto blocks = [](size_t n) { return (unsigned)std::max<size_t>(1, std::min<size_t>(4096, (n + 255) / 256)); };
        const size_t ncs = R.nframes * (nkey + 1);
        hipLaunchKernelGGL(fill_u32_kernel, dim3(blocks(ncs)), dim3(256), 0, st, cs, 0u, ncs);
        hipLaunchKernelGGL(fill_u64_kernel, dim3(blocks(R.ngroups)), dim3(256), 0, st, d_self, (size_t)R.ngroups);
        const unsigned sblocks = ns * R.nframes;
        hipLaunchKernelGGL(ordered ? tile_count_kernel<true> : tile_count_kernel<false>, dim3(sblocks), dim3(kBlock), 0,
                           st, R.d_kmap, d_frames, R.npix, ns, g, side, S, d_goff, R.ngroups, cs, d_self);
        hipLaunchKernelGGL(tile_scan_kernel, dim3(R.nframes), dim3(1024), 0, st, cs, cursor, (uint32_t)nkey);
        hipLaunchKernelGGL(tile_scatter_kernel, dim3(sblocks), dim3(kBlock), 0, st, R.d_kmap, d_frames, R.npix, ns, g,
                           side, S.ka, S.kb, S.kc, cursor, srec);
        if (!ordered)
            hipLaunchKernelGGL(fill_u64_kernel, dim3(blocks(nvox * R.ngroups)), dim3(256), 0, st, H, nvox * R.ngroups);
        IAC_HIP(hipGetLastError());
        if (!pl) {
            IAC_HIP(hipStreamSynchronize(st));
            IAC_TRY(plan_of(ctx, R, side, box_cap, kRegionTiles, g, read.cells, &pl));
            if (!pl->tiles_fit) {  // boxes outside the mesh
                pl = nullptr;
                continue;
            }
        }
        const bool by_parts = !ordered && !wide && (double)kept >= kPartRecords * (double)R.nframes * (double)nkey;
        auto *target = ordered ? reinterpret_cast<unsigned long long *>(R.d_mesh) : H;
        const uint32_t ntasks = (uint32_t)pl->tiles.size(), nchunks = (uint32_t)chunks.size();
        // few tasks, or tasks of uneven work (dense regions, regions with themselves): several blocks
        // each, of at least kTileShare pairs
        const double recs = (double)kept / ((double)R.nframes * nc);
        const double pairs = recs * recs * std::max(1.0, (double)R.nframes / nchunks);
        const uint32_t splits = (uint32_t)std::max(
            1.0, std::min({std::ceil(kTileBlocks / ((double)ntasks * nchunks)), pairs / kTileShare, 4096.0}));
        const uint32_t per = std::max<uint32_t>(1, kMaxGridBlocks / ((uint64_t)ntasks * splits));
        auto kern = ordered ? (wide ? cq_tile_kernel<true, true> : cq_tile_kernel<true, false>)
                            : (wide ? cq_tile_kernel<false, true> : cq_tile_kernel<false, false>);
        IAC_TRY(timer_begin(ctx));
        for (uint32_t c0 = 0; c0 < nchunks; c0 += per) {
            const dim3 grid(ntasks * splits * std::min(per, nchunks - c0));
            hipLaunchKernelGGL(kern, grid, dim3(kBlock),
                               pl->tile_box * sizeof(unsigned long long), st, srec,
                               R.npix, cs, nc, side, d_chunks + c0, pl->d_tiles, ntasks, S, target, nvox, ctx->d_counters,
                               by_parts ? 1 : 0, splits);
            IAC_HIP(hipGetLastError());
        }
        IAC_TRY(timer_end(ctx));
        if (!ordered) {
            const size_t centre = (size_t)S.P.c0 + (size_t)S.P.c1 * S.P.sab + (size_t)S.P.c2 * S.P.sab * S.P.sab;
            hipLaunchKernelGGL(symmetrize_kernel, dim3(blocks(nvox * R.ngroups)), dim3(256), 0, st, H,
                               reinterpret_cast<unsigned long long *>(R.d_mesh), nvox, R.ngroups, centre, d_self, d_self,
                               (const uint32_t *)nullptr);
            IAC_HIP(hipGetLastError());
        }
        ctx->tile_passes++;
        *done = true;
        return IAC_OK;
    }
    return IAC_OK;
}

// ---- prepared runs -----------------------------------------------------------

struct PairBatch {
    iac_ctx *ctx = nullptr;
    PairRun R{};
    std::vector<uint32_t> group_off;
    void *mem = nullptr;     // srec | cs | H | goff | self | chunks | tasks | strips' tasks and buffers
    Bufs b{};
};

int pairs_prepare(iac_ctx *ctx, const PairRun &R0, PairBatch **out)
{
    *out = nullptr;
    hipStream_t st = ctx->stream;
    if (R0.n_total >= (1ull << 32)) return fail(IAC_ERR_LIMIT, "pair engine: at most 2^32 - 1 records per call");
    iac_pair_plan *pl = nullptr;
    iac_pair_plan *sp = nullptr;
    const uint64_t *off = nullptr;
    IAC_TRY(get_plan(ctx, st, R0, cell_vox_of(ctx, R0), box_cap_of(ctx, R0), region_of(ctx, R0), &pl, &off, &sp));
    const std::vector<Chunk> chunks = make_chunks(off, R0.nframes, R0.h_group_off, R0.ngroups, fchunk_of(ctx));
    IAC_TRY(check_chunks(off, chunks));
    std::vector<Chunk> schunks;
    if (sp)
        schunks = make_chunks(off, R0.nframes, R0.h_group_off, R0.ngroups, strip_chunk(ctx, R0.nframes, sp->tasks.size()));
    auto *B = new PairBatch();
    B->ctx = ctx;
    B->R = R0;
    B->group_off.assign(R0.h_group_off, R0.h_group_off + R0.ngroups + 1);
    B->R.h_group_off = B->group_off.data();
    const int nc = pl->g.ncu * pl->g.ncv;
    const Sizes z = sizes_of(B->R, nc, chunks.size());
    const size_t tbytes = std::max<size_t>(1, pl->tasks.size()) * sizeof(Task);
    auto up = [](size_t x) { return (x + 255) / 256 * 256; };
    const size_t base = up(z.srec + z.cs + z.h + z.goff + z.self + z.chunks + tbytes);
    const size_t stask = sp ? up(sp->tasks.size() * sizeof(Task)) : 0;
    hipError_t e = alloc_buffer(ctx, base + stask + strip_bytes(B->R, sp, schunks.size()), &B->mem);
    if (e == hipErrorOutOfMemory && sp) {  // the walk needs 16 bytes per record less
        sp = nullptr;
        schunks.clear();
        e = alloc_buffer(ctx, base, &B->mem);
    }
    if (e != hipSuccess) {
        delete B;
        return hip_fail(e, "pairs_prepare allocation", __FILE__, __LINE__);
    }
    char *p = static_cast<char *>(B->mem);
    Bufs &b = B->b;
    b.srec = reinterpret_cast<float4 *>(p);
    b.cs = reinterpret_cast<uint32_t *>(p + z.srec);
    b.H = reinterpret_cast<unsigned long long *>(p + z.srec + z.cs);
    b.d_goff = reinterpret_cast<uint32_t *>(p + z.srec + z.cs + z.h);
    b.d_self = reinterpret_cast<unsigned long long *>(p + z.srec + z.cs + z.h + z.goff);
    b.d_flag = reinterpret_cast<uint32_t *>(b.d_self + R0.ngroups);
    b.d_chunks = reinterpret_cast<Chunk *>(p + z.srec + z.cs + z.h + z.goff + z.self);
    Task *tasks = reinterpret_cast<Task *>(p + z.srec + z.cs + z.h + z.goff + z.self + z.chunks);
    b.nchunks = (uint32_t)chunks.size();
    b.d_tasks = tasks;
    b.ntasks = (uint32_t)pl->tasks.size();
    b.g = pl->g;
    b.box_cap = pl->box_cap;
    e = hipMemcpyAsync(b.d_goff, B->group_off.data(), B->group_off.size() * 4, hipMemcpyHostToDevice, st);
    if (e == hipSuccess && !chunks.empty())
        e = hipMemcpyAsync(b.d_chunks, chunks.data(), chunks.size() * sizeof(Chunk), hipMemcpyHostToDevice, st);
    if (e == hipSuccess && !pl->tasks.empty())
        e = hipMemcpyAsync(tasks, pl->tasks.data(), pl->tasks.size() * sizeof(Task), hipMemcpyHostToDevice, st);
    if (sp) {  // a copy of the strips' tasks too: the cache may drop their plan
        strip_place(b, p + base + stask, B->R, sp, schunks.size());
        b.st_tasks = reinterpret_cast<Task *>(p + base);
        if (e == hipSuccess)
            e = hipMemcpyAsync(p + base, sp->tasks.data(), sp->tasks.size() * sizeof(Task), hipMemcpyHostToDevice, st);
        if (e == hipSuccess && !schunks.empty())
            e = hipMemcpyAsync(b.st_chunks, schunks.data(), schunks.size() * sizeof(Chunk), hipMemcpyHostToDevice, st);
    }
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) {
        (void)hipFree(B->mem);
        delete B;
        return hip_fail(e, "pairs_prepare upload", __FILE__, __LINE__);
    }
    *out = B;
    return IAC_OK;
}

int pairs_enqueue(PairBatch *B, hipStream_t st, uint64_t *d_mesh)
{
    PairRun R = B->R;
    R.d_mesh = d_mesh;
    // the pair kernel is timed on the context's own stream (not inside a capture)
    return enqueue(B->ctx, st, R, B->b, st == B->ctx->stream);
}

void pairs_batch_free(PairBatch *B)
{
    if (!B) return;
    if (B->mem) (void)hipFree(B->mem);
    delete B;
}

// ---- frame queues --------------------------------------------------------------

struct PairQueue {
    iac_ctx *ctx = nullptr;
    PairRun R0{};
    iac_pair_plan *pl = nullptr;
    uint64_t max_records = 0;
    uint32_t max_frames = 0;
    void *mem = nullptr;        // srec | cs | H | goff | self | chunks (device)
    Bufs b{};
    Chunk *h_chunks = nullptr;  // pinned: the chunk table and group offsets of the last run
    uint32_t *h_goff = nullptr;
    hipEvent_t staged = nullptr;  // the last run's uploads from h_chunks / h_goff are done
};

int pairs_queue_create(iac_ctx *ctx, const PairRun &R0, uint64_t max_records, uint32_t max_frames, PairQueue **out)
{
    *out = nullptr;
    if (max_records == 0 || max_records >= (1ull << 32) || max_frames == 0)
        return fail(IAC_ERR_LIMIT, "pair engine queue: 1 .. 2^32 - 1 records and at least one frame");
    iac_pair_plan *pl = nullptr;
    IAC_TRY(get_plan(ctx, ctx->stream, R0, cell_vox_of(ctx, R0), box_cap_of(ctx, R0), region_of(ctx, R0), &pl));
    auto *Q = new PairQueue();
    Q->ctx = ctx;
    Q->R0 = R0;
    Q->R0.ngroups = 1;
    Q->R0.n_total = max_records;
    Q->R0.nframes = max_frames;
    Q->max_records = max_records;
    Q->max_frames = max_frames;
    const int nc = pl->g.ncu * pl->g.ncv;
    const Sizes z = sizes_of(Q->R0, nc, max_frames);
    hipError_t e = hipMalloc(&Q->mem, z.srec + z.cs + z.h + z.goff + z.self + z.chunks);
    if (e == hipSuccess)
        e = hipHostMalloc((void **)&Q->h_chunks, (size_t)max_frames * sizeof(Chunk) + 64, hipHostMallocDefault);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&Q->staged, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventRecord(Q->staged, ctx->stream);
    if (e != hipSuccess) {
        if (Q->mem) (void)hipFree(Q->mem);
        if (Q->h_chunks) (void)hipHostFree(Q->h_chunks);
        if (Q->staged) (void)hipEventDestroy(Q->staged);
        delete Q;
        return hip_fail(e, "pair engine queue allocation", __FILE__, __LINE__);
    }
    Q->h_goff = reinterpret_cast<uint32_t *>(Q->h_chunks + max_frames);
    char *p = static_cast<char *>(Q->mem);
    Bufs &b = Q->b;
    b.srec = reinterpret_cast<float4 *>(p);
    b.cs = reinterpret_cast<uint32_t *>(p + z.srec);
    b.H = reinterpret_cast<unsigned long long *>(p + z.srec + z.cs);
    b.d_goff = reinterpret_cast<uint32_t *>(p + z.srec + z.cs + z.h);
    b.d_self = reinterpret_cast<unsigned long long *>(p + z.srec + z.cs + z.h + z.goff);
    b.d_flag = reinterpret_cast<uint32_t *>(b.d_self + 1);
    b.d_chunks = reinterpret_cast<Chunk *>(p + z.srec + z.cs + z.h + z.goff + z.self);
    b.d_tasks = pl->d_tasks;
    b.ntasks = (uint32_t)pl->tasks.size();
    b.g = pl->g;
    b.box_cap = pl->box_cap;
    pl->pins++;
    Q->pl = pl;
    *out = Q;
    return IAC_OK;
}

int pairs_queue_run(PairQueue *Q, const PairRun &R, const uint64_t *h_off)
{
    if (R.nframes == 0 || R.n_total == 0) return IAC_OK;
    if (R.nframes > Q->max_frames || R.n_total > Q->max_records)
        return fail(IAC_ERR_LIMIT, "pair engine queue: run larger than the queue");
    hipStream_t st = Q->ctx->stream;
    const uint32_t goff[2] = {0, R.nframes};
    const std::vector<Chunk> chunks = make_chunks(h_off, R.nframes, goff, 1, fchunk_of(Q->ctx), R.h_rots);
    IAC_TRY(check_chunks(h_off, chunks));
    // the previous run's uploads read the pinned table: wait for them before rewriting it
    IAC_HIP(hipEventSynchronize(Q->staged));
    std::copy(chunks.begin(), chunks.end(), Q->h_chunks);
    Q->h_goff[0] = 0;
    Q->h_goff[1] = R.nframes;
    IAC_HIP(hipMemcpyAsync(Q->b.d_goff, Q->h_goff, 2 * sizeof(uint32_t), hipMemcpyHostToDevice, st));
    if (!chunks.empty())
        IAC_HIP(hipMemcpyAsync(Q->b.d_chunks, Q->h_chunks, chunks.size() * sizeof(Chunk), hipMemcpyHostToDevice, st));
    IAC_HIP(hipEventRecord(Q->staged, st));
    PairRun RR = Q->R0;
    RR.rec = R.rec;
    RR.d_frame_off = R.d_frame_off;
    RR.nframes = R.nframes;
    RR.n_total = R.n_total;
    RR.h_group_off = goff;
    RR.ngroups = 1;
    RR.d_mesh = R.d_mesh;
    RR.d_rots = R.d_rots;
    RR.h_rots = R.h_rots;
    Bufs b = Q->b;
    b.nchunks = (uint32_t)chunks.size();
    return enqueue(Q->ctx, st, RR, b, true);
}

void pairs_queue_free(PairQueue *Q)
{
    if (!Q) return;
    (void)hipStreamSynchronize(Q->ctx->stream);
    if (Q->pl) Q->pl->pins--;
    if (Q->mem) (void)hipFree(Q->mem);
    if (Q->h_chunks) (void)hipHostFree(Q->h_chunks);
    if (Q->staged) (void)hipEventDestroy(Q->staged);
    delete Q;
}

}  // namespace iac
