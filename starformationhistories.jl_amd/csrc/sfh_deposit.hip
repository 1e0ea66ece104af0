// sfh_deposit.hip -- smoothed Hess-diagram template deposition on gfx950:
// bin_cmd_smooth (src/StarFormationHistories.jl:574-621), one template or many
// templates per launch.
//
// Kernels of a call:
//   k_dep_prep    one thread per point: the reference's FP64 footprint / index
//                 math (bit-exact, no FMA contraction) and every per-point
//                 constant of the evaluation -> a 112-byte PointDesc.
//   k_dep_wide    the wide kernels' sums on every fourth column (see sfh_psf.h).
//   k_dep_gather  every other point, then the wide kernels' sums interpolated.
//                 Both are bin-owner gathers: a thread owns one row and kCPT =
//                 16 consecutive columns (or nodes) of one template, in
//                 registers; a workgroup 256 such strips.  Every wave walks its
//                 template's descriptors in order through scalar loads (the
//                 descriptor is uniform across the wave, so it sits in scalar
//                 registers: no LDS staging, no barriers), skips points whose
//                 rows miss its strips, and adds each point's contribution to
//                 its bins, so there are no atomics and every bin sums its
//                 points in a fixed order (deterministic).  Contributions
//                 accumulate in FP32 per 64 points and are flushed into FP64
//                 accumulators.
//   k_dep_finish  small launches, whose points are split into slices: their sums.
// The pair work is VALU bound; HBM traffic is the descriptors in, the wide sums
// out and in again (0.1 GB for 700 templates of 200 x 300 bins) and one write
// of each template.  700 such templates (2.8e10 pairs, most of them in rows of
// one node or two): 7.5 ms with three nodes per row and every column evaluated,
// 6.0 ms with the nodes merged, 4.0 ms (1.76 wide + 2.23) with the wide kernels
// on a quarter of their columns and the accumulators reached by LDS instead of
// flat accesses (VGPRs 112 -> 89), 3.4 ms with the sum form, 2.8 ms with the wide
// gather's FP64 sums in registers and its workgroups by cost, 2.7 ms (1.13 +
// 1.59) with 8-byte keys for the hit search; 2.9 ms (1.16 + 1.75) since every
// node of a masked strip forms its own multiplier and the merged rows and the
// sum form end where a template's tails would lose accuracy (sfh_psf.h).
#include "sfh_internal.h"
#include "sfh_psf.h"

#include <algorithm>
#include <type_traits>

namespace sfh {

using psf::PointCounts;
using psf::PointDesc;
using psf::PointKey;

constexpr int kDepBlock = 256;
constexpr int kCPT = psf::kCPT;  // columns per thread
constexpr int kChunk = 64;       // points between FP32 -> FP64 flushes
constexpr int64_t kWideBytes = (int64_t)512 << 20;   // scratch of the wide kernels' sums per launch
// Workgroups that a sliced launch aims at: four per CU, one resident round.  A
// launch of fewer splits its points: 50 templates of 75 x 100 bins are 100
// workgroups (0.50 ms -> 0.25 ms of gather plus 0.01 ms for the slices' sums),
// one of 100 x 151 bins 5 (0.45 -> 0.17 ms).
constexpr int64_t kGatherSlots = 1024;

__global__ __launch_bounds__(256) void k_dep_prep(
    const double* __restrict__ colors, const double* __restrict__ mags,
    const double* __restrict__ cerr, const double* __restrict__ merr,
    const double* __restrict__ weights, const double* __restrict__ cmult, double cov_mult,
    int64_t npoints, psf::Range ex, psf::Range ey, int asym, PointDesc* __restrict__ out,
    PointKey* __restrict__ keys, unsigned long long* __restrict__ pairs, int* __restrict__ bad)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    unsigned long long cnt = 0;
    if (p < npoints) {
        const double x = colors[p], y = mags[p], sx = cerr[p], sy = merr[p], A = weights[p];
        const double c = cmult ? cmult[p] : cov_mult;
        PointDesc d;
        if (!(isfinite(x) && isfinite(y) && isfinite(sx) && isfinite(sy) && isfinite(A) && isfinite(c))) {
            d = psf::empty_desc();
            atomicOr(bad, 1);
        } else if (asym) {
            cnt = (unsigned long long)psf::prep_asymmetric(x, y, sx, sy, A, ex, ey, &d);
        } else {
            cnt = (unsigned long long)psf::prep_covariant(x, y, sx, sy, c, A, ex, ey, &d);
        }
        out[p] = d;
        keys[p] = psf::point_key(d, (int)(ex.length - 1), asym != 0);
    }
    psf::add_count(pairs, blockIdx.x, cnt);
}

struct GatherArgs {
    int nx, ny;
    int ncg, nblk;               // strips per row, workgroups per template
    int wcg;                     // strips per row of the wide kernels' nodes (0: none)
    int wslices;                 // slices of the wide kernels' sums
    double* wide;                // their sums: [slice][template][ny][16 wcg]
    int64_t wstride;             // between slices
    double* part;                // sliced: [slice][template][ny * nx], else NULL
    float* out32;
    double* out64;
    int64_t ld_out;
};

// Workgroup -> (template, band): order[blockIdx.x] when an order is given (the
// pairs by decreasing cost, so the longest workgroups start first and the
// launch ends with short ones); otherwise template t's band j is (j + t) mod
// nblk: consecutive workgroups go to the 8 XCDs in turn, so without the
// rotation every template's band j would land on XCD j mod 8 and the populated
// bands of a diagram would load some XCDs far more than others.
__device__ __forceinline__ void gather_tile(const int32_t* __restrict__ order, int nblk, int64_t* t, int* blk)
{
    if (order) {
        const int id = order[blockIdx.x];
        *t = id / nblk;
        *blk = id - (int)*t * nblk;
    } else {
        *t = blockIdx.x / nblk;
        *blk = (int)((blockIdx.x - *t * nblk + *t) % nblk);
    }
}

// FP64 accumulators in LDS, [column][thread].  Volatile, so that they stay
// there instead of being promoted to registers, and through a pointer into the
// LDS address space (a volatile access is not moved out of the generic one by
// the compiler, and flat accesses would wait for the global loads too).
typedef volatile __attribute__((address_space(3))) double lds_double;
struct LdsAcc {
    lds_double* p;
    __device__ lds_double* operator[](int c) const { return p + c * kDepBlock; }
};

// One lane's point of a chunk (class none past the end).
__device__ inline PointKey key_of(const PointKey* __restrict__ keys, int p, int np)
{
    return p < np ? keys[p] : PointKey{1u, 0u};
}

// f(descriptor) for each of a chunk's points in hits, in order.  Descriptors
// are uniform across the wave, so they are read through scalar loads, two per
// wait.
template <class F>
__device__ __forceinline__ void each(const PointDesc* __restrict__ chunk, uint64_t hits, F f)
{
    while (hits) {
        const int i = __builtin_ctzll(hits);
        hits &= hits - 1;
        const bool two = hits != 0;
        const int j = two ? __builtin_ctzll(hits) : i;
        if (two) hits &= hits - 1;
        const PointDesc d0 = chunk[i];
        const PointDesc d1 = chunk[j];
        f(d0);
        if (two) f(d1);
    }
}

// The wide kernels (kWide1, kWide2) of a template on their nodes, every
// kStep-th column: the gather below with 16 nodes of one row per thread and
// one form per loop, into the FP64 sums [slice][template][row][node] that
// k_dep_gather (or k_dep_finish) interpolates.
// VALU bound: 6.3e8 wave instructions for 700 templates, 94% of their lanes
// active, 3.9 cycles each per SIMD; 1.16 ms (1.76 with the FP64 sums in LDS).
__global__ __launch_bounds__(kDepBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_dep_wide(
    const PointDesc* __restrict__ desc, const PointKey* __restrict__ keys, const int64_t* __restrict__ offsets,
    const int32_t* __restrict__ order, GatherArgs a)
{
    int64_t t;
    int blk;
    gather_tile(order, (a.wcg * a.ny + kDepBlock - 1) / kDepBlock, &t, &blk);
    const int64_t p0 = offsets[t], p1 = offsets[t + 1];
    const int slot = blk * kDepBlock + threadIdx.x;
    const int row = slot / a.wcg;
    const int col0 = (slot - row * a.wcg) * kCPT;
    const bool valid = row < a.ny;
    const int wslot = __builtin_amdgcn_readfirstlane(blk * kDepBlock + (int)(threadIdx.x & ~63u));
    const int row_lo = wslot / a.wcg, row_hi = (wslot + 63) / a.wcg;
    double acc[kCPT];
    float part[kCPT];
#pragma unroll
    for (int c = 0; c < kCPT; ++c) {
        acc[c] = 0.0;
        part[c] = 0.0f;
    }
    const PointDesc* __restrict__ td = desc + p0;
    const PointKey* __restrict__ tk = keys + p0;
    const int np = (int)(p1 - p0);
    const int nch = (np + kChunk - 1) / kChunk;
    const int c0 = (int)((int64_t)nch * blockIdx.y / gridDim.y);
    const int c1 = (int)((int64_t)nch * (blockIdx.y + 1) / gridDim.y);
    const int lane = threadIdx.x & 63;
    auto add = [&](const PointDesc& d, auto nodes) {
        constexpr int NODES = decltype(nodes)::value;
        if (!(valid && row >= d.ya && row <= d.yb)) return;
        float M[NODES], L[NODES], h[NODES];
        psf::merged_row<NODES>(d, row, M, L, h);
        psf::gauss_strip<NODES>(d, M, L, h, col0, part);
    };
    PointKey kn = key_of(tk, c0 * kChunk + lane, np);
    for (int ch = c0; ch < c1; ++ch) {
        const PointKey k = kn;
        kn = key_of(tk, (ch + 1) * kChunk + lane, np);              // next chunk's keys in flight
        const uint32_t cls = k.cls();
        const bool hit = k.ya() <= row_hi && k.yb() >= row_lo;
        const uint64_t h1 = __ballot(hit && cls == psf::kClsWide1), h2 = __ballot(hit && cls == psf::kClsWide2);
        if (!(h1 | h2)) continue;
        each(td + ch * kChunk, h1, [&](const PointDesc& d) { add(d, std::integral_constant<int, 1>{}); });
        each(td + ch * kChunk, h2, [&](const PointDesc& d) { add(d, std::integral_constant<int, 2>{}); });
#pragma unroll
        for (int c = 0; c < kCPT; ++c) {
            acc[c] += (double)part[c];
            part[c] = 0.0f;
        }
    }
    if (!valid) return;
    double* o = a.wide + blockIdx.y * a.wstride + (t * a.ny + row) * (int64_t)(a.wcg * kCPT) + col0;
#pragma unroll
    for (int c = 0; c < kCPT; c += 2)
        *reinterpret_cast<double2*>(o + c) = make_double2(acc[c], acc[c + 1]);
}

// kStep columns from col (a multiple of kStep) of one row of template t: v plus
// the wide kernels' sums interpolated from their nodes (slices added in
// order), written to the outputs.
__device__ inline void finish_cols(const GatherArgs& a, int64_t t, int row, int col, double* v)
{
    static constexpr psf::InterpWeights W = psf::interp_weights();
    if (a.wcg) {
        // column col + r lies r / kStep past node col / kStep + kLead
        const int ldw = a.wcg * kCPT;
        const double* w = a.wide + (t * a.ny + row) * (int64_t)ldw + col / psf::kStep;
        double n[psf::kTaps];
#pragma unroll
        for (int k = 0; k < psf::kTaps; ++k) n[k] = w[k];
        for (int s = 1; s < a.wslices; ++s) {
            w += a.wstride;
#pragma unroll
            for (int k = 0; k < psf::kTaps; ++k) n[k] += w[k];
        }
        v[0] += n[psf::kLead];
#pragma unroll
        for (int r = 1; r < psf::kStep; ++r)
#pragma unroll
            for (int k = 0; k < psf::kTaps; ++k) v[r] = fma(W.w[r][k], n[k], v[r]);
    }
    const int64_t base = t * a.ld_out + (int64_t)row * a.nx + col;
#pragma unroll
    for (int r = 0; r < psf::kStep; ++r) {
        if (col + r >= a.nx) continue;
        if (a.out32) a.out32[base + r] = (float)v[r];
        if (a.out64) a.out64[base + r] = v[r];
    }
}

// The FP64 accumulators live in LDS (16 per thread, 32 KiB per workgroup: five
// workgroups per CU), touched once per 64 points, so that the FP32 strip and
// the per-point constants fit the registers of five waves per SIMD (the sums
// in registers measured the same: 1577 against 1576 us for 700 templates).
// VALU bound: 1.03e9 wave instructions, 68% of their lanes active (the short
// footprints of the sum and erf-difference forms), 3.8 cycles each per SIMD.
template <bool kAsym>
__global__ __launch_bounds__(kDepBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_dep_gather(
    const PointDesc* __restrict__ desc, const PointKey* __restrict__ keys, const int64_t* __restrict__ offsets,
    const int32_t* __restrict__ order, GatherArgs a)
{
    __shared__ double sacc_[kCPT][kDepBlock];
    const LdsAcc sacc{(lds_double*)&sacc_[0][0]};
    int64_t t;
    int blk;
    gather_tile(order, a.nblk, &t, &blk);
    const int nx = a.nx, ncg = a.ncg;
    const int64_t p0 = offsets[t], p1 = offsets[t + 1];
    const int slot = blk * kDepBlock + threadIdx.x;
    const int row = slot / ncg;
    const int col0 = (slot - row * ncg) * kCPT;
    const bool valid = row < a.ny;
    // rows of this wave's 64 strips (wave-uniform)
    const int wslot = __builtin_amdgcn_readfirstlane(blk * kDepBlock + (int)(threadIdx.x & ~63u));
    const int row_lo = wslot / ncg, row_hi = (wslot + 63) / ncg;

    float part[kCPT];
#pragma unroll
    for (int c = 0; c < kCPT; ++c) {
        sacc[c][threadIdx.x] = 0.0;
        part[c] = 0.0f;
    }
    // Each chunk of 64 points: every lane reads one point's footprint and form,
    // ballots keep the points whose rows meet this wave's strips, and only
    // those descriptors are loaded.  The hits are taken in passes: first the
    // common cases (a Gaussian form with a footprint spanning the whole grid
    // width, one node per row, then two -- the asymmetric kernel's second is
    // the form with a y factor per row), then every other point but the wide
    // kernels.  Each pass has one code path, so the strip's registers carry
    // through it without copies; a bin sums a chunk's points pass by pass, each
    // in point order (deterministic).
    const PointDesc* __restrict__ td = desc + p0;
    const PointKey* __restrict__ tk = keys + p0;
    const int np = (int)(p1 - p0);
    const int nch = (np + kChunk - 1) / kChunk;
    const int c0 = (int)((int64_t)nch * blockIdx.y / gridDim.y);
    const int c1 = (int)((int64_t)nch * (blockIdx.y + 1) / gridDim.y);
    const int lane = threadIdx.x & 63;
    const int wave_id = (int)(threadIdx.x >> 6);
    auto in_rows = [&](const PointDesc& d) { return valid && row >= d.ya && row <= d.yb; };
    // the common forms: NODES merged nodes per row (0: the asymmetric kernel's
    // y factor), no column mask
    auto add_common = [&](const PointDesc& d, auto nodes) {
        constexpr int N = decltype(nodes)::value, NODES = N ? N : 1;
        if (!in_rows(d)) return;
        float M[NODES], L[NODES] = {}, h[NODES] = {};
        if constexpr (N == 0) M[0] = d.pref * psf::y_factor(fmaf((float)(row - d.ya), d.dv, d.ay), d.ey);
        else psf::merged_row<NODES>(d, row, M, L, h);
        psf::gauss_strip<NODES>(d, M, L, h, col0, part);
    };
    auto add = [&](const PointDesc& d) {
        if (!in_rows(d) || col0 > d.xb || col0 + kCPT - 1 < d.xa) return;
        psf::add_point<!kAsym>(d, row, col0, part);
    };
    // A point in the erf-difference form (a kernel narrower than 3 columns, 3.6
    // in the asymmetric case: a footprint of 45 or 37 columns at most) with the
    // whole wave cooperating, instead of strip code in which only the few lanes
    // whose strips meet the footprint would work: segments of 16, 32 or 64 lanes
    // take one of the point's rows inside this wave's strips each, lane l of a
    // segment footprint column xa + l; lanes 0 .. nc evaluate erfc at their
    // column's left edge (its sign that of the edge) and a column's right edge is
    // the next lane's.  A wider footprint (edges so far from 0 that adding steps
    // to them rounds) is taken in blocks of a segment's columns.  Each
    // bin's value (nodes summed in order, in FP32) is added to its owner's
    // FP64 accumulator in LDS: the bins are distinct, so no two lanes write one
    // word, and the owner's own flush comes later in program order.
    auto direct = [&](const PointDesc& d) {
        constexpr int NODES = kAsym ? 1 : 3;
        const int nc = d.xb - d.xa + 1;
        const int lw = nc < 16 ? 4 : nc < 32 ? 5 : 6;          // nc + 1 edges per segment
        const int ls = lane & ((1 << lw) - 1), wide = (1 << lw) - 1;
        const int r0 = d.ya > row_lo ? d.ya : row_lo, r1 = d.yb < row_hi ? d.yb : row_hi;
        for (int cb = 0; cb < nc; cb += wide)
        for (int rp = r0; rp <= r1; rp += 64 >> lw) {
            const int l = cb + ls, r = rp + (lane >> lw);
            float W[3], h[3] = {0.0f, 0.0f, 0.0f};
            if constexpr (kAsym) W[0] = d.pref * psf::y_factor(fmaf((float)(r - d.ya), d.dv, d.ay), d.ey);
            else psf::cov_row(d, r, W, h);
            float v = 0.0f;
#pragma unroll
            for (int k = 0; k < NODES; ++k) {
                const float e = psf::signed_erfc(psf::direct_edge(d, l, h[k]));
                // the next lane's value (wave_shl:1)
                const float e1 = __int_as_float(
                    __builtin_amdgcn_update_dpp(0, __float_as_int(e), 0x130, 0xf, 0xf, false));
                v = fmaf(W[k], psf::erf_diff(e, e1), v);
            }
            if (l < nc && ls < wide && r <= r1) {
                const int col = d.xa + l;
                const int o = r * ncg + col / kCPT - wslot;
                if (o >= 0 && o < 64) {
                    lds_double* p = &sacc[col % kCPT][wave_id * 64 + o];
                    *p = *p + (double)v;
                }
            }
        }
    };
    PointKey kn = key_of(tk, c0 * kChunk + lane, np);
    for (int ch = c0; ch < c1; ++ch) {
        const PointKey k = kn;
        kn = key_of(tk, (ch + 1) * kChunk + lane, np);              // next chunk's keys in flight
        const uint32_t cls = k.cls();
        const bool hit = k.ya() <= row_hi && k.yb() >= row_lo && cls >= psf::kClsOne;
        const uint64_t all = __ballot(hit);
        if (!all) continue;
        const uint64_t h1 = __ballot(hit && cls == psf::kClsOne), h2 = __ballot(hit && cls == psf::kClsSecond);
        const uint64_t h3 = __ballot(hit && cls == psf::kClsDirect);
        const PointDesc* __restrict__ chunk = td + ch * kChunk;
        each(chunk, h1, [&](const PointDesc& d) { add_common(d, std::integral_constant<int, 1>{}); });
        each(chunk, h2, [&](const PointDesc& d) { add_common(d, std::integral_constant<int, kAsym ? 0 : 2>{}); });
        each(chunk, all & ~(h1 | h2 | h3), add);
        each(chunk, h3, direct);
#pragma unroll
        for (int c = 0; c < kCPT; ++c) {
            sacc[c][threadIdx.x] += (double)part[c];
            part[c] = 0.0f;
        }
    }
    if (!valid) return;
    if (a.part) {
        double* o = a.part + ((blockIdx.y * (int64_t)(gridDim.x / a.nblk) + t) * a.ny + row) * nx + col0;
#pragma unroll
        for (int c = 0; c < kCPT; ++c)
            if (col0 + c < nx) o[c] = sacc[c][threadIdx.x];
        return;
    }
#pragma unroll 1
    for (int c = 0; c < kCPT && col0 + c < nx; c += psf::kStep) {
        double v[psf::kStep];
#pragma unroll
        for (int r = 0; r < psf::kStep; ++r) v[r] = sacc[c + r][threadIdx.x];
        finish_cols(a, t, row, col0 + c, v);
    }
}

// The templates from the gather's slices, added in order, and the wide
// kernels' sums: one thread per kStep columns of a row.
__global__ __launch_bounds__(kDepBlock) void k_dep_finish(GatherArgs a, int64_t ntemplates, int slices)
{
    const int64_t g = (int64_t)blockIdx.x * kDepBlock + threadIdx.x;
    const int nq = (a.nx + psf::kStep - 1) / psf::kStep;
    const int64_t per = (int64_t)nq * a.ny;
    if (g >= per * ntemplates) return;
    const int64_t t = g / per;
    const int row = (int)((g - t * per) / nq), col = (int)((g - t * per) % nq) * psf::kStep;
    const double* p = a.part + (t * a.ny + row) * a.nx + col;
    const int64_t stride = ntemplates * a.ny * a.nx;
    double v[psf::kStep] = {};
#pragma unroll 4
    for (int s = 0; s < slices; ++s)
#pragma unroll
        for (int r = 0; r < psf::kStep; ++r) v[r] += p[s * stride + (col + r < a.nx ? r : 0)];
    finish_cols(a, t, row, col, v);
}

// Relative cost per row strip of each x form (issue slots of the form's strip
// code over the Gaussian form's).
__device__ inline unsigned form_cost(int kind, bool full)
{
    if (kind == psf::kGauss1) return 2u;
    if (kind == psf::kGauss2) return 4u;
    if (kind == psf::kGauss) return full ? 5u : 6u;
    if (kind == psf::kSum) return 10u;
    return 32u;
}

// Adds a point's cost to every band of 256 strips (ncg per row) that its rows
// meet: the rows x strips inside the band, times w.
__device__ inline void band_cost(unsigned long long* band, int nblk, int ncg, int ya, int yb, unsigned w)
{
    const int b0 = (int)(((int64_t)ya * ncg) / kDepBlock);
    int b1 = (int)(((int64_t)yb * ncg + ncg - 1) / kDepBlock);
    if (b1 > nblk - 1) b1 = nblk - 1;
    for (int b = b0; b <= b1; ++b) {
        const int rlo = (int)(((int64_t)b * kDepBlock) / ncg);
        const int rhi = (int)(((int64_t)b * kDepBlock + kDepBlock - 1) / ncg);
        const int r0 = ya > rlo ? ya : rlo, r1 = yb < rhi ? yb : rhi;
        if (r1 >= r0) atomicAdd(&band[b], (unsigned long long)(r1 - r0 + 1) * w);
    }
}

// Estimated cost of every (template, row band) workgroup of the gather (cost)
// and of the wide kernels' gather (wcost).  One workgroup per template, the
// band sums in LDS (integer atomics: the sums do not depend on the order);
// (nblk + wblk) * 8 bytes of dynamic LDS.
__global__ __launch_bounds__(256) void k_dep_cost(const PointDesc* __restrict__ desc,
                                                  const int64_t* __restrict__ offsets, int nx, int ncg, int nblk,
                                                  int wcg, int wblk, unsigned long long* __restrict__ cost,
                                                  unsigned long long* __restrict__ wcost)
{
    extern __shared__ unsigned long long band[];
    const int64_t t = blockIdx.x;
    for (int b = threadIdx.x; b < nblk + wblk; b += blockDim.x) band[b] = 0;
    __syncthreads();
    for (int64_t p = offsets[t] + threadIdx.x; p < offsets[t + 1]; p += blockDim.x) {
        const int4 f = *reinterpret_cast<const int4*>(desc + p);
        if (f.x > f.y) continue;
        const int kind = desc[p].kind;
        if (kind >= psf::kWide1) {
            band_cost(band + nblk, wblk, wcg, f.z, f.w, (unsigned)wcg * (kind == psf::kWide1 ? 2u : 3u));
        } else {
            const unsigned w = form_cost(kind, f.x == 0 && f.y == nx - 1);
            band_cost(band, nblk, ncg, f.z, f.w, w * (unsigned)(f.y / kCPT - f.x / kCPT + 1));
        }
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nblk; b += blockDim.x) cost[t * nblk + b] = band[b];
    for (int b = threadIdx.x; b < wblk; b += blockDim.x) wcost[t * wblk + b] = band[nblk + b];
}

constexpr int kOrderMax = 16384;    // workgroups one ordering launch takes
constexpr int kOrderBuckets = 1024;

// order[] = the n workgroup ids by decreasing cost, to 1/1024 of the largest:
// a counting sort over 1024 cost buckets in one workgroup (the order inside
// a bucket is that of the LDS atomics; it only schedules the gather, whose
// workgroups each write their own band, so the templates do not depend on it).
// One workgroup per list: the gather's n costs, then the wide kernels' nwide.
__global__ __launch_bounds__(1024) void k_dep_order(const unsigned long long* __restrict__ cost, int n, int nwide,
                                                    int32_t* __restrict__ order)
{
    if (blockIdx.x == 1) {
        cost += n;
        order += n;
        n = nwide;
    }
    __shared__ unsigned long long smax[16];
    __shared__ int start[kOrderBuckets];
    __shared__ int wsum[16];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    unsigned long long mx = 0;
    for (int i = tid; i < n; i += blockDim.x) mx = cost[i] > mx ? cost[i] : mx;
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned long long o = __shfl_xor(mx, off, 64);
        mx = o > mx ? o : mx;
    }
    if (lane == 0) smax[wv] = mx;
    start[tid] = 0;
    __syncthreads();
    mx = 0;
    for (int w = 0; w < 16; ++w) mx = smax[w] > mx ? smax[w] : mx;
    int shift = 0;
    while ((mx >> shift) >= (unsigned long long)kOrderBuckets) ++shift;
    auto bucket = [&](int i) { return kOrderBuckets - 1 - (int)(cost[i] >> shift); };
    for (int i = tid; i < n; i += blockDim.x) atomicAdd(&start[bucket(i)], 1);
    __syncthreads();
    // exclusive prefix sum of the 1024 counts, one per thread
    const int c = start[tid];
    int incl = c;
    for (int off = 1; off < 64; off <<= 1) {
        const int o = __shfl_up(incl, off, 64);
        if (lane >= off) incl += o;
    }
    if (lane == 63) wsum[wv] = incl;
    __syncthreads();
    int base = 0;
    for (int w = 0; w < wv; ++w) base += wsum[w];
    start[tid] = base + incl - c;
    __syncthreads();
    for (int i = tid; i < n; i += blockDim.x) order[atomicAdd(&start[bucket(i)], 1)] = i;
}

// The gather over descriptors of npoints points (template t owns
// desc[offsets[t] .. offsets[t+1])): the wide kernels on their nodes, then
// everything else, with the workgroups in decreasing estimated cost when the
// launch is small enough to order in one pass.  Where a launch would leave the
// chip idle its points are split into slices, whose FP64 sums k_dep_finish
// adds in order.
static int launch_gather(sfh_ctx* ctx, const PointDesc* desc, const PointKey* keys, const int64_t* d_offsets,
                         int64_t ntemplates, int64_t npoints, bool asym, int nx, int ny, float* out32, double* out64,
                         int64_t ld_out)
{
    GatherArgs a{};
    a.nx = nx;
    a.ny = ny;
    a.ncg = (int)cdiv(nx, kCPT);
    a.nblk = (int)cdiv((int64_t)a.ncg * ny, kDepBlock);
    a.wcg = psf::wide_pays(nx) ? (int)cdiv(psf::wide_nodes(nx), kCPT) : 0;
    a.ld_out = ld_out;
    const int64_t wblk = cdiv((int64_t)a.wcg * ny, kDepBlock), wbins = (int64_t)a.wcg * kCPT * ny;
    SFH_ARG_CHECK(ctx, (int64_t)a.nblk * ntemplates < (int64_t)1 << 31, "too many templates for one launch");
    // templates per launch: the wide kernels' sums within kWideBytes
    const int64_t group = a.wcg ? std::max<int64_t>(1, std::min(ntemplates, kWideBytes / (wbins * 8))) : ntemplates;
    for (int64_t t0 = 0; t0 < ntemplates; t0 += group) {
        const int64_t nt = std::min(group, ntemplates - t0);
        const int64_t grid = (int64_t)a.nblk * nt, chunks = cdiv(cdiv(npoints, ntemplates), kChunk);
        auto slices = [&](int64_t workgroups) {
            return (int)std::max<int64_t>(1, std::min(chunks, kGatherSlots / std::max<int64_t>(workgroups, 1)));
        };
        const int ns = slices(grid);
        const int64_t* offsets = d_offsets + t0;
        const int32_t *order = nullptr, *worder = nullptr;
        a.out32 = out32 ? out32 + t0 * ld_out : nullptr;
        a.out64 = out64 ? out64 + t0 * ld_out : nullptr;
        a.part = nullptr;
        if (ns > 1) {
            void* p = nullptr;
            if (int rc = scratch(ctx, "dep_part", (size_t)ns * nt * nx * ny * sizeof(double), &p)) return rc;
            a.part = (double*)p;
        } else if (nt > 1 && grid <= kOrderMax && npoints > 0) {
            const int64_t wgrid = wblk * nt;
            void *pc = nullptr, *po = nullptr;
            if (int rc = scratch(ctx, "dep_cost", (size_t)(grid + wgrid) * sizeof(unsigned long long), &pc)) return rc;
            if (int rc = scratch(ctx, "dep_order", (size_t)(grid + wgrid) * sizeof(int32_t), &po)) return rc;
            {
                TimedLaunch tl(ctx, "deposit_order");
                hipLaunchKernelGGL(k_dep_cost, dim3((unsigned)nt), dim3(256),
                                   (size_t)(a.nblk + wblk) * sizeof(unsigned long long), ctx->stream, desc, offsets, nx,
                                   a.ncg, a.nblk, a.wcg, (int)wblk, (unsigned long long*)pc,
                                   (unsigned long long*)pc + grid);
                hipLaunchKernelGGL(k_dep_order, dim3(a.wcg ? 2 : 1), dim3(1024), 0, ctx->stream,
                                   (const unsigned long long*)pc, (int)grid, (int)wgrid, (int32_t*)po);
            }
            if (int rc = check_launch(ctx, "k_dep_order")) return rc;
            order = (const int32_t*)po;
            worder = order + grid;
        }
        if (a.wcg) {
            a.wslices = slices(wblk * nt);
            a.wstride = wbins * nt;
            void* p = nullptr;
            if (int rc = scratch(ctx, "dep_wide", (size_t)(a.wslices * a.wstride) * sizeof(double), &p)) return rc;
            a.wide = (double*)p;
            TimedLaunch tl(ctx, "deposit_wide");
            hipLaunchKernelGGL(k_dep_wide, dim3((unsigned)(wblk * nt), (unsigned)a.wslices), dim3(kDepBlock), 0,
                               ctx->stream, desc, keys, offsets, worder, a);
        }
        if (int rc = check_launch(ctx, "k_dep_wide")) return rc;
        {
            TimedLaunch tl(ctx, asym ? "deposit_asym" : "deposit_cov");
            const dim3 g((unsigned)grid, (unsigned)ns);
            hipLaunchKernelGGL(asym ? k_dep_gather<true> : k_dep_gather<false>, g, dim3(kDepBlock), 0, ctx->stream,
                               desc, keys, offsets, order, a);
        }
        if (int rc = check_launch(ctx, "k_dep_gather")) return rc;
        if (ns > 1) {
            hipLaunchKernelGGL(k_dep_finish, dim3((unsigned)cdiv(cdiv(nx, psf::kStep) * ny * nt, kDepBlock)),
                               dim3(kDepBlock), 0, ctx->stream, a, nt, ns);
            if (int rc = check_launch(ctx, "k_dep_finish")) return rc;
        }
    }
    return SFH_OK;
}

static int validate_ranges(sfh_ctx* ctx, sfh_range xe, sfh_range ye)
{
    SFH_ARG_CHECK(ctx, xe.length >= 2 && ye.length >= 2, "edge ranges need at least 2 edges");
    SFH_ARG_CHECK(ctx, (xe.length - 1) * (ye.length - 1) > 1, "length(image.weights) > 1 (:367)");
    SFH_ARG_CHECK(ctx, std::isfinite(xe.step) && std::isfinite(ye.step) && xe.step != 0.0 && ye.step != 0.0,
                  "edge steps must be finite and non-zero");
    SFH_ARG_CHECK(ctx, xe.length < (1 << 30) && ye.length < (1 << 30), "grid too large");
    return SFH_OK;
}

// Core launcher on device arrays.  out32 / out64: column t at base + t*ld_out.
static int deposit(sfh_ctx* ctx, const double* colors, const double* mags, const double* cerr,
                   const double* merr, const double* weights, const double* cmult,
                   const int64_t* d_offsets, int64_t ntemplates, int64_t npoints_total,
                   double cov_mult, sfh_range xe, sfh_range ye, float* out32, double* out64,
                   int64_t ld_out, int64_t* pairs_out)
{
    if (int rc = validate_ranges(ctx, xe, ye)) return rc;
    const int nx = (int)(xe.length - 1), ny = (int)(ye.length - 1);
    SFH_ARG_CHECK(ctx, ld_out >= (int64_t)nx * ny, "ld_out < nx*ny");
    const bool asym = (cov_mult == 0.0) && cmult == nullptr;
    void *pdesc = nullptr, *pcnt = nullptr;
    if (int rc = scratch(ctx, "dep_desc", (size_t)(npoints_total + 1) * (sizeof(PointDesc) + sizeof(PointKey)), &pdesc))
        return rc;
    PointKey* keys = (PointKey*)((PointDesc*)pdesc + npoints_total + 1);
    if (int rc = scratch(ctx, "dep_counters", sizeof(PointCounts), &pcnt)) return rc;
    SFH_HIP_TRY(ctx, hipMemsetAsync(pcnt, 0, sizeof(PointCounts), ctx->stream));
    PointCounts* dc = (PointCounts*)pcnt;
    psf::Range rx{xe.first, xe.step, xe.length}, ry{ye.first, ye.step, ye.length};
    if (npoints_total > 0) {
        TimedLaunch tl(ctx, "deposit_prep");
        hipLaunchKernelGGL(k_dep_prep, dim3((unsigned)cdiv(npoints_total, 256)), dim3(256), 0, ctx->stream,
                           colors, mags, cerr, merr, weights, cmult, cov_mult, npoints_total, rx, ry,
                           asym ? 1 : 0, (PointDesc*)pdesc, keys, dc->pairs, &dc->bad);
    }
    if (int rc = check_launch(ctx, "k_dep_prep")) return rc;
    if (int rc = launch_gather(ctx, (const PointDesc*)pdesc, keys, d_offsets, ntemplates, npoints_total, asym, nx, ny,
                               out32, out64, ld_out))
        return rc;
    // Non-finite inputs: the reference's round(Int, NaN) throws InexactError.
    PointCounts hc;
    SFH_HIP_TRY(ctx, hipMemcpyAsync(&hc, dc, sizeof(hc), hipMemcpyDeviceToHost, ctx->stream));
    SFH_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    if (hc.bad) return set_error(ctx, SFH_ERR_DOMAIN, "non-finite kernel parameter (InexactError in round(Int, ·))");
    if (pairs_out) *pairs_out = hc.total();
    return SFH_OK;
}

// The gather of descriptors already built (by the device preparation of
// partial_cmd_smooth): template t owns desc[koff[t] .. koff[t+1]).
int deposit_from_desc(sfh_ctx* ctx, const void* desc, const void* keys, const int64_t* d_koff, int64_t ntemplates,
                      int64_t npoints, bool asym, sfh_range xe, sfh_range ye, float* out32, int64_t ld_out)
{
    if (int rc = validate_ranges(ctx, xe, ye)) return rc;
    const int nx = (int)(xe.length - 1), ny = (int)(ye.length - 1);
    SFH_ARG_CHECK(ctx, ld_out >= (int64_t)nx * ny, "ld_out < nx*ny");
    return launch_gather(ctx, (const PointDesc*)desc, (const PointKey*)keys, d_koff, ntemplates, npoints, asym, nx, ny,
                         out32, nullptr, ld_out);
}

}  // namespace sfh

using namespace sfh;

extern "C" {

int sfh_bin_cmd_smooth(sfh_ctx* ctx, const double* colors, const double* mags,
                       const double* color_err, const double* mag_err, const double* weights,
                       int64_t npoints, int cov_mult, sfh_range xedges, sfh_range yedges,
                       double* out)
{
    if (!ctx) return SFH_ERR_ARGUMENT;
    std::lock_guard<std::recursive_mutex> g(ctx->mu);
    if (int rc = bind(ctx)) return rc;
    SFH_ARG_CHECK(ctx, cov_mult == -1 || cov_mult == 0 || cov_mult == 1, "cov_mult in (-1, 0, 1) (:579)");
    SFH_ARG_CHECK(ctx, npoints >= 0, "npoints must be >= 0");
    SFH_ARG_CHECK(ctx, out && (npoints == 0 || (colors && mags && color_err && mag_err && weights)),
                  "null pointer");
    if (int rc = validate_ranges(ctx, xedges, yedges)) return rc;
    const int64_t nbins = (xedges.length - 1) * (yedges.length - 1);
    const int64_t np = npoints > 0 ? npoints : 1;
    void* p = nullptr;
    if (int rc = scratch(ctx, "bcs_in", (size_t)np * 5 * sizeof(double) + 2 * sizeof(int64_t), &p)) return rc;
    double* d = (double*)p;
    const double* srcs[5] = {colors, mags, color_err, mag_err, weights};
    for (int k = 0; k < 5 && npoints > 0; ++k)
        SFH_HIP_TRY(ctx, hipMemcpyAsync(d + k * np, srcs[k], (size_t)npoints * sizeof(double),
                                        hipMemcpyHostToDevice, ctx->stream));
    int64_t* doff = (int64_t*)(d + 5 * np);
    int64_t hoff[2] = {0, npoints};
    SFH_HIP_TRY(ctx, hipMemcpyAsync(doff, hoff, sizeof(hoff), hipMemcpyHostToDevice, ctx->stream));
    void* po = nullptr;
    if (int rc = scratch(ctx, "bcs_out", (size_t)nbins * sizeof(double), &po)) return rc;
    int rc = deposit(ctx, d, d + np, d + 2 * np, d + 3 * np, d + 4 * np, nullptr, doff, 1, npoints,
                     (double)cov_mult, xedges, yedges, nullptr, (double*)po, nbins, nullptr);
    if (rc) return rc;
    SFH_HIP_TRY(ctx, hipMemcpyAsync(out, po, (size_t)nbins * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    SFH_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return SFH_OK;
}

int sfh_bin_cmd_smooth_batch_device(sfh_ctx* ctx, const double* d_colors, const double* d_mags,
                                    const double* d_color_err, const double* d_mag_err,
                                    const double* d_weights, const double* d_cmult,
                                    const int64_t* d_offsets, int64_t ntemplates, double cov_mult,
                                    sfh_range xedges, sfh_range yedges, float* d_out, int64_t ld_out,
                                    int64_t* pairs_out)
{
    if (!ctx) return SFH_ERR_ARGUMENT;
    std::lock_guard<std::recursive_mutex> g(ctx->mu);
    if (int rc = bind(ctx)) return rc;
    SFH_ARG_CHECK(ctx, ntemplates >= 1, "ntemplates must be >= 1");
    SFH_ARG_CHECK(ctx, d_offsets && d_out, "null pointer");
    SFH_ARG_CHECK(ctx, std::isfinite(cov_mult), "cov_mult must be finite");
    // The gather kernel trusts the offsets to index the descriptor array, so
    // check them all on the host first (ntemplates+1 integers).
    std::vector<int64_t> hoff((size_t)ntemplates + 1);
    SFH_HIP_TRY(ctx, hipMemcpyAsync(hoff.data(), d_offsets, hoff.size() * sizeof(int64_t),
                                    hipMemcpyDeviceToHost, ctx->stream));
    SFH_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    SFH_ARG_CHECK(ctx, hoff[0] == 0, "offsets[0] must be 0");
    for (int64_t t = 0; t < ntemplates; ++t)
        SFH_ARG_CHECK(ctx, hoff[t + 1] >= hoff[t], "offsets must be non-decreasing (t=%lld)", (long long)t);
    const int64_t last = hoff[ntemplates];
    SFH_ARG_CHECK(ctx, last == 0 || (d_colors && d_mags && d_color_err && d_mag_err && d_weights),
                  "null point array");
    return deposit(ctx, d_colors, d_mags, d_color_err, d_mag_err, d_weights, d_cmult, d_offsets,
                   ntemplates, last, cov_mult, xedges, yedges, d_out, nullptr, ld_out, pairs_out);
}

}  // extern "C"
