// sfh_psf.h -- per-point footprint preparation (FP64, bit-exact index math)
// and per-bin evaluation (FP32) of the two pixel-integrated Gaussian kernels of
// StarFormationHistories.jl, shared by the gfx950 kernels and a host build
// used to check the FP32 arithmetic against the FP64 oracle on the CPU.
//
// Reference: src/StarFormationHistories.jl
//   GaussianPSFCovariant + gaussian_psf_covariant  :272-338
//   addstar!(::Histogram, ::RealSpaceKernel)        :366-408
//   GaussianPSFAsymmetric + gaussian_int_general     :191-265
//   addstar!(::AbstractMatrix, ::PixelSpaceKernel)  :348-364
//   bin_cmd_smooth                                  :574-621
//
// Both kernels reduce to D(u, e) = erf(u + e) - erf(u - e) at a bin centre u
// (in units of sqrt(2) sigma) and half bin width e:
//   covariant  : A hy / (2 sqrt(2 pi) sy) * sum_k w_k exp(-t_k^2/2) D(u_i + g t_k, ex)
//                with t_k = (y_j + xi_k hy - y0)/sy (3-point Gauss-Legendre, :303-304),
//                g = c sy / (sqrt(2) sx)  (the reference's Δx = dx + c Δy, :328);
//   asymmetric : A/4 * D(u_i, ex) * D(v_j, ey)  (:203-204; the two sign flips cancel).
// For e < kSumEps (kSumEpsAsym for asymmetric kernels), D is evaluated without the
// erf-difference cancellation as
//   D = (4 e / sqrt(pi)) <exp(-(u+s)^2)>, the mean over |s| < e:
// e < 0.026, the Gaussian form: the mean is exp(-u^2) S(u^2), S(w) =
//   sum_n H_2n(sqrt w) e^2n / (2n+1)! = s0 exp(b w) (1 + O(b^2 w^2)), b = s1 / s0
//   = 2e^2/3 + O(e^4), so D = (4 e / sqrt(pi)) s0 exp(-(1 - b) u^2), one Gaussian
//   of a rescaled coordinate.  ln S(w) = ln s0 + b w - (4/45) e^4 w^2 + ..., so the
//   dropped term is (4/45) e^4 w^2 relative to the local value: <= 1.1e-5 at
//   |u| = 4 for e < 0.026; relative to the kernel's peak it is at most
//   (4/45) e^4 max(w^2 e^-w) = 0.048 e^4, below 2.2e-8, under the FP32 rounding of
//   the sums.  On the 700-template workload 97% of the pairs take this form.
// 0.026 <= e < kSumEps, the sum form: the mean as two Gaussians (e < kPairEps),
//   whose first wrong term of ln is 3e-5 (2 u e)^6, at most 2.6e-3 e^6 of the
//   peak, or three, with 1.4e-7 (2 u e)^8, at most 1.7e-4 e^8 (set_sum).  Relative
//   to the local value at |u| = 3.7, where a kernel is 1e-6 of its peak, that is
//   1.4e-7 (two) and 5e-8 (three, e = 0.12); at e = 0.2 it would be 3.2e-6, and
//   a template's worst bin above 1e-6 of its maximum 4e-6 off instead of 1.6e-6.
// Both run in scaled coordinates a = u sqrt(log2 e) times the square root of
// their Gaussian's own factor, so a Gaussian is one hardware exp2 of -a^2.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <type_traits>

namespace sfh {
namespace psf {

constexpr float kSeriesEps = 0.1f;    // an asymmetric kernel's y factor as a series below this half height
constexpr float kPairEps = 0.055f;    // x: the sum form's two Gaussians below this half width, three above
constexpr float kSumEps = 0.12f;      // the sum form below, erf differences above: covariant kernels ...
constexpr float kSumEpsAsym = 0.1f;   // ... and asymmetric ones
constexpr float kGaussEps = 0.026f;   // the Gaussian form below this half width
// Covariant kernels in the Gaussian form: the row's three Gauss-Legendre nodes
// merged into one node or two (set_row_nodes) up to these values of
// h^2 (1 + 2 g^2), h = half row height / sigma_y.  Two nodes up to 0.03 keep the
// peak's error as small, but put templates' worst bin above 1e-6 of the maximum
// at 2.7e-6 instead of the three nodes' 2.5e-6 (0.018: 2.5e-6); 700 templates of
// 200 x 300 bins take 3.81 ms up to 0.03, 3.86 up to 0.018, 4.02 up to 0.01.
constexpr double kOneNodeEta = 0.00135;
constexpr double kTwoNodeEta = 0.018;
// ... and where the strips' multipliers 2^(+-2 m du) stay finite (gauss_strip)
constexpr double kMaxLogB = 120.0;
// Wide kernels (merged Gaussian forms whose footprint spans the grid's width)
// are evaluated on every kStep-th column only, and the sum over all of them is
// interpolated to the columns between with kTaps-point Lagrange weights
// (interp_weights).  A row of such a kernel is one Gaussian or two of the same
// width sigma; the interpolation's largest error over all offsets is 2.0e-8 of
// its peak for a step of sigma / 5 and 3.4e-9 for sigma / 6.  kStepDu: the
// largest step in the scaled coordinate (where sigma = 0.849): sigma / 5.3.
constexpr int kStep = 4;
constexpr int kTaps = 10;
constexpr int kLead = kTaps / 2 - 1;            // nodes before the first column
constexpr double kStepDu = 0.16;
constexpr double kGLNode = 0.7745966692414834;   // :303
constexpr float kW0 = 0.5555555555555556f;      // :304
constexpr float kW1 = 0.8888888888888888f;
constexpr double kLog2e = 1.4426950408889634;
constexpr int kCPT = 16;                        // consecutive columns evaluated per thread

// Evaluation of a point: the erf difference, the Gaussian form (its rows'
// Gauss-Legendre nodes one by one, or merged into one node or two), or the
// sum form (kWide1, kWide2: the merged forms on every kStep-th column)
enum : int32_t { kDirect = 0, kGauss = 1, kSum = 2, kGauss1 = 3, kGauss2 = 4, kWide1 = 5, kWide2 = 6 };

// One prepared kernel: the clipped footprint and its FP32 parameters.
// Footprint indices are 0-based and inclusive; xa > xb marks "nothing to
// deposit" (the reference's length>1 guard, :359 / :401).
// All kinds but kDirect store ax, du and g in a scaled coordinate (see header).
struct alignas(16) PointDesc {
    int32_t xa, xb, ya, yb;
    float ax;     // x coordinate of the first footprint column centre
    float du;     // x step per column
    float ex;     // half column width in u (direct form)
    float g;      // covariant: shear c*sy/(sqrt2 sx); asymmetric: 0
    float ay;     // covariant: t of first footprint row centre; asymmetric: v of first row
    float dv;     // t (or v) step per row
    float ey;     // covariant: GL node offset xi*hy/sy; asymmetric: half row width in v
    float pref;   // amplitude prefactor (see header), with the series form factors
    float s1, s2, s3;       // a row's y weight, kGauss1: 2^(s1 t^2 + s2 t^4), kGauss2: 2^(s1 t^2 +-
                            // s2 t) and the nodes' x shifts g t -+ s3; kSum: the outer Gaussians' x
                            // shifts -+ s3 and the middle one's amplitude s1 over theirs
    int32_t kind;
    float gf, gfi;          // kGauss2: 2^(2 s3 du) and its inverse, the nodes' strip multipliers
                            // relative to the middle's
    int32_t terms;          // kGauss: 1; kSum: 2 or 3 Gaussians
    int32_t pad0;
    float q[8];             // Gaussian forms: q[j] = 2^-(du (j + 1/2))^2, the strip's column factors
};

// What the gather reads of every point to find its hits: the rows of its
// footprint and the class of its evaluation, in 8 bytes.
enum : uint32_t { kClsNone = 0, kClsWide1, kClsWide2, kClsOne, kClsSecond, kClsRest, kClsDirect };
struct PointKey {
    uint32_t a, b;     // ya | low two bits of the class << 30, yb | its high bits << 30
    __host__ __device__ int ya() const { return (int)(a & 0x3FFFFFFFu); }
    __host__ __device__ int yb() const { return (int)(b & 0x3FFFFFFFu); }
    __host__ __device__ uint32_t cls() const { return (a >> 30) | (b >> 30) << 2; }
};

// The class of a point on a grid of nx columns: kClsOne, one merged node per
// row; kClsSecond, the other common form (a covariant kernel's two nodes, an
// asymmetric one of the grid's width with a y factor per row); kClsRest,
// masked strips.
__host__ __device__ inline PointKey point_key(const PointDesc& d, int nx, bool asym)
{
    if (d.xa > d.xb) return PointKey{1u, 0u};
    const bool full = d.xa == 0 && d.xb == nx - 1;
    const uint32_t c = d.kind == kWide1    ? kClsWide1
                       : d.kind == kWide2  ? kClsWide2
                       : d.kind == kDirect ? kClsDirect
                       : d.kind == kGauss1 ? kClsOne
                       : d.kind == kGauss2 || (asym && full && d.kind == kGauss) ? kClsSecond
                                                                                 : kClsRest;
    return PointKey{(uint32_t)d.ya | (c & 3u) << 30, (uint32_t)d.yb | (c >> 2) << 30};
}

// What the preparation counts besides: the (point, bin) pairs, over as many
// words as keep same-address atomics rare (24,000 waves adding to one word
// took 0.25 ms), and a flag for inputs that are refused.
constexpr int kCountSlots = 256;
struct PointCounts {
    unsigned long long pairs[kCountSlots];
    int bad;
    int64_t total() const
    {
        unsigned long long s = 0;
        for (unsigned long long v : pairs) s += v;
        return (int64_t)s;
    }
};

#if defined(__HIPCC__)
// Adds a wave's counts to the slot of its workgroup.
__device__ inline void add_count(unsigned long long* pairs, unsigned workgroup, unsigned long long cnt)
{
    for (int off = 32; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, 64);
    if ((threadIdx.x & 63) == 0 && cnt) atomicAdd(&pairs[workgroup % kCountSlots], cnt);
}
#endif

struct Range {
    double first, step;
    int64_t length;
};

// Julia round(Int, x) (ties to even) with the argument clamped so the cast
// is defined; callers flag non-finite input separately.
__host__ __device__ inline int64_t jl_round(double x)
{
    if (x > 4.0e15) x = 4.0e15;
    if (x < -4.0e15) x = -4.0e15;
    return (int64_t)rint(x);
}

__host__ __device__ inline int64_t jl_ceil(double x)
{
    if (x > 4.0e15) x = 4.0e15;
    if (x < -4.0e15) x = -4.0e15;
    return (int64_t)ceil(x);
}

__host__ __device__ inline int64_t imax(int64_t a, int64_t b) { return a > b ? a : b; }
__host__ __device__ inline int64_t imin(int64_t a, int64_t b) { return a < b ? a : b; }

__host__ __device__ inline PointDesc empty_desc()
{
    PointDesc d{};
    d.xa = 1;
    d.xb = 0;
    d.ya = 1;
    d.yb = 0;
    return d;
}

// Coefficients of S(w) = s0 + s1 w + s2 w^2 + s3 w^3 + s4 w^4 (w = u^2) for
// the series D = (4e/sqrt(pi)) exp(-w) S(w).
struct Series {
    float s0, s1, s2, s3, s4;
};

__host__ __device__ inline Series series_coeffs(float e)
{
    const float q = e * e;
    const float c1 = q / 6.0f, c2 = q * q / 120.0f, c3 = q * q * q / 5040.0f,
                c4 = q * q * q * q / 362880.0f;
    Series s;
    s.s0 = 1.0f - 2.0f * c1 + 12.0f * c2 - 120.0f * c3 + 1680.0f * c4;
    s.s1 = 4.0f * c1 - 48.0f * c2 + 720.0f * c3 - 13440.0f * c4;
    s.s2 = 16.0f * c2 - 480.0f * c3 + 13440.0f * c4;
    s.s3 = 64.0f * c3 - 3584.0f * c4;
    s.s4 = 256.0f * c4;
    return s;
}

// Nodes of a wide kernel's row on a grid of nx columns (node k at column
// kStep (k - kLead)), and whether they take fewer strips than the columns.
__host__ __device__ inline int wide_nodes(int nx) { return (nx + kStep - 1) / kStep + kTaps - 1; }
__host__ __device__ inline bool wide_pays(int nx)
{
    return (wide_nodes(nx) + kCPT - 1) / kCPT < (nx + kCPT - 1) / kCPT;
}

// Lagrange weights of nodes -kLead .. kTaps - 1 - kLead at x = r / kStep.
struct InterpWeights {
    double w[kStep][kTaps];
};
__host__ __device__ constexpr InterpWeights interp_weights()
{
    InterpWeights t{};
    for (int r = 0; r < kStep; ++r)
        for (int i = 0; i < kTaps; ++i) {
            double w = 1.0;
            for (int j = 0; j < kTaps; ++j)
                if (j != i) w *= ((double)r / kStep - (j - kLead)) / (double)(i - j);
            t.w[r][i] = w;
        }
    return t;
}

// The column factors of a Gaussian form's strips, from the rounded step du that
// the kernel uses (gauss_strip).
__host__ __device__ inline void set_strip(PointDesc* d)
{
    // (j + 3/2)^2 - (j + 1/2)^2 = 2 (j + 1): two exp2 and products in FP64 instead
    // of an exp2 per column (they were most of a descriptor's cost)
    const double du = (double)d->du, w = exp2(-2.0 * du * du);
    double q = exp2(-0.25 * du * du), p = w;
    for (int j = 0; j < 8; ++j) {
        d->q[j] = (float)q;
        q *= p;
        p *= w;
    }
}

// The x coordinates of a merged Gaussian form (ax, du: scaled), whose footprint
// spans the nx columns: on the wide kernels' nodes where the kernel is smooth
// enough, else on the columns.
__host__ __device__ inline void set_merged_x(PointDesc* d, int32_t kind, double ax, double du, int nx)
{
    d->kind = kind;
    if (wide_pays(nx) && fabs(kStep * du) <= kStepDu) {
        d->kind = kind == kGauss1 ? kWide1 : kWide2;
        du *= kStep;
        ax -= kLead * du;
    }
    d->ax = (float)ax;
    d->du = (float)du;
    set_strip(d);
    const double r = exp2(2.0 * (double)d->s3 * (double)d->du);
    d->gf = (float)r;
    d->gfi = (float)(1.0 / r);
}

// A covariant kernel in the Gaussian form with its rows' Gauss-Legendre nodes
// merged (only for a footprint that spans the grid's width); false where the
// row is too high for that, or its shear too large (the three nodes stay).
// Around a row centre t, phi = t^2/2 + gam (u + g t)^2 (gam = 1 - b) has the
// t-derivative s = k2 t + 2 gam g u, k2 = 1 + 2 gam g^2, and the three nodes at
// t, t +- dl (dl = xi hy / sy) sum exactly to
//   S exp(-phi) F(x),  F = 1 - p + p cosh x,  x = dl s,
//   S = 8/9 + (10/9) exp(-dl^2 k2 / 2),  p = 1 - (8/9) / S.
// One node: F = exp(p x^2 / 2), the x^2 joining the quadratic form, which
// stays one Gaussian of a rescaled coordinate, shear and y weight.  The first
// dropped term of ln F, 0.0154 x^4, is (h^2 k2 = eta) at most 0.012 eta^2 =
// 2.2e-8 of the kernel's peak for eta < 0.00135: the bound of the Gaussian form
// itself at its limit e = 0.026 (e^2 = eta / 2).
// Two nodes: F = exp(al x^2) cosh(be x) with the x^2 and x^4 terms of ln F
// (be^4 = (3 p^2 - p) / 2, al = p/2 - be^2/2): two Gaussians with the shifts
// g' t -+ v.  Its first dropped term, 2.9e-4 x^6, is at most 6.6e-4 eta^3 =
// 3.9e-9 of the peak for eta < 0.018.
__host__ __device__ inline bool set_row_nodes(PointDesc* d, double ax, double du, double gam, double g, int nx)
{
    const double dl = (double)d->ey, k2 = 1.0 + 2.0 * gam * g * g;
    const double eta = dl * dl * k2 / (kGLNode * kGLNode);
    if (!(eta <= kTwoNodeEta)) return false;
    const bool one = eta <= kOneNodeEta;
    const double e2 = (10.0 / 9.0) * exp(-0.5 * dl * dl * k2);
    const double S = 8.0 / 9.0 + e2, p = e2 / S;
    const double be2 = one ? 0.0 : sqrt(0.5 * p * (3.0 * p - 1.0));
    const double q = 0.5 * (p - be2) * dl * dl;            // the x^2 term's share in the exponent: q s^2
    const double A = gam * (1.0 - 4.0 * q * gam * g * g);
    const double g1 = gam * g * (1.0 - 2.0 * q * k2) / A;
    const double rho = 0.5 + gam * g * g - q * k2 * k2 - A * g1 * g1;
    const double scale = sqrt(A * kLog2e);
    double v = 0.0, lam = 0.0, pre = S;
    if (!one) {
        const double bd = sqrt(be2) * dl;
        v = bd * gam * g / A;
        lam = bd * (k2 - 2.0 * gam * g * g1);
        pre *= 0.5 * exp(A * v * v);
    }
    // |2 m du| over every strip: m reaches the rows' shear, the nodes' shift and the
    // x range of the columns (and of up to eight strips' width past them)
    const double tm = fmax(fabs((double)d->ay), fabs((double)d->ay + (double)(d->yb - d->ya) * (double)d->dv));
    const double span = fabs(ax) + (double)(nx + 8 * kCPT) * fabs(du);
    if (!(2.0 * kStep * fabs(du) * scale * scale * (fabs(g1) * tm + fabs(v) + span) <= kMaxLogB)) return false;
    d->pref = (float)((double)d->pref * pre);
    d->g = (float)(g1 * scale);
    d->s1 = (float)(-rho * kLog2e);
    d->s2 = (float)(lam * kLog2e);        // (0 for one node)
    d->s3 = (float)(v * scale);
    set_merged_x(d, one ? kGauss1 : kGauss2, ax * scale, du * scale, nx);
    return true;
}

// The sum form of half column width e.  With r = 2u, the mean over the column is
//   <exp(-(u+s)^2)> = exp(-u^2) Z exp(k2 r^2 / 2 + k4 r^4 / 24 + k6 r^6 / 720 + ...),
// Z the mean and k_n the cumulants of s under the weight exp(-s^2) on |s| < e.
// exp(a r^2) (1 - P + P cosh(b r)) has the cumulants 2a + P b^2, P (1 - 3P) b^4 and
// P (1 - 15 P + 30 P^2) b^6.  P = 1 (two Gaussians) with b and a from k4 and k2
// leaves k6 off by 0.08 of its value for the uniform weight, 16 e^6 / 63; P =
// 0.63747 (three) gives that value too, and its k8 to half a percent.
__host__ __device__ inline void set_sum(PointDesc* d, double ax, double du, double g)
{
    const double e = (double)d->ex;
    // the moments by 5-point Gauss-Legendre quadrature (exact to e^10)
    constexpr double x1 = 0.5384693101056831, x2 = 0.9061798459386640;
    constexpr double w0 = 0.2844444444444444, w1 = 0.2393143352496832, w2 = 0.1184634425280945;
    const double s1 = e * e * x1 * x1, s2 = e * e * x2 * x2;
    const double f1 = 2.0 * w1 * exp(-s1), f2 = 2.0 * w2 * exp(-s2);
    const double Z = w0 + f1 + f2;
    const double m2 = (f1 * s1 + f2 * s2) / Z, k4 = (f1 * s1 * s1 + f2 * s2 * s2) / Z - 3.0 * m2 * m2;
    const double P = d->ex < kPairEps ? 1.0 : 0.63747;
    const double b2 = sqrt(k4 / (P * (1.0 - 3.0 * P)));
    // exp(-u^2 + a r^2 -+ b r) = exp(b^2 / gam) exp(-gam (u +- b / gam)^2), gam = 1 - 4a
    const double gam = 1.0 - 2.0 * (m2 - P * b2), scale = sqrt(gam * kLog2e);
    const double grow = exp(b2 / gam);
    d->kind = kSum;
    d->terms = P < 1.0 ? 3 : 2;
    d->pref = (float)((double)d->pref * Z * 0.5 * P * grow);
    d->s1 = (float)(2.0 * (1.0 - P) / (P * grow));
    d->s3 = (float)(sqrt(b2) / gam * scale);
    d->ax = (float)(ax * scale);
    d->du = (float)(du * scale);
    d->g = (float)(g * scale);
    set_strip(d);
}

// The form of a point with x coordinate ax of its first column, column step du
// and half width d->ex (in u) on a grid of nx columns.  cov: a covariant
// kernel of shear g; else an asymmetric one, whose y factor joins a merged
// Gaussian form (one node, no shear) where it has the Gaussian form itself, with
// the next term of its ln S, -(4/45) e^4 v^4, in the row's weight (without it the
// RMS error of a template's bins was 1.8e-7 instead of 1.5e-7).
__host__ __device__ inline void set_x_form(PointDesc* d, double ax, double du, bool cov, double g, int nx)
{
    const float e = d->ex;
    if (!(e < (cov ? kSumEps : kSumEpsAsym))) {
        d->kind = kDirect;
        d->ax = (float)ax;
        d->du = (float)du;
        d->g = (float)g;
        return;
    }
    if (e >= kGaussEps) {
        set_sum(d, ax, du, g);
        return;
    }
    // s0 exp(-(1 - b) w), b = s1 / s0: the coordinates carry sqrt(1 - b), the
    // amplitude s0
    const Series s = series_coeffs(e);
    const double gam = 1.0 - (double)s.s1 / (double)s.s0, scale = sqrt(gam * kLog2e);
    d->kind = kGauss;
    d->terms = 1;
    d->pref = (float)((double)d->pref * (double)s.s0);
    const bool full = e > 0.0f && d->xa == 0 && d->xb == nx - 1;
    if (full && cov && set_row_nodes(d, ax, du, gam, g, nx)) return;
    if (full && !cov && d->ey > 0.0f && d->ey < kGaussEps) {
        const Series y = series_coeffs(d->ey);
        d->pref = (float)((double)d->pref * (double)y.s0);
        d->s1 = (float)(-(1.0 - (double)y.s1 / (double)y.s0) * kLog2e);
        const double ey2 = (double)d->ey * (double)d->ey;
        d->s2 = (float)(-4.0 / 45.0 * ey2 * ey2 * kLog2e);
        set_merged_x(d, kGauss1, ax * scale, du * scale, nx);
        return;
    }
    d->ax = (float)(ax * scale);
    d->du = (float)(du * scale);
    d->g = (float)(g * scale);
    set_strip(d);
}

// Covariant kernel centred at (x0, y0) (real units) -- addstar! :366-408.
// Returns the number of (point, bin) pairs in the footprint (0 if skipped).
// The FP64 expressions keep the reference's operation order; compile with
// fp-contract off so no FMA changes a rounding.
__host__ __device__ inline int64_t prep_covariant(double x0, double y0, double sx, double sy,
                                                  double c, double A, Range ex, Range ey,
                                                  PointDesc* out)
{
#pragma clang fp contract(off)
    const int64_t nx = ex.length - 1, ny = ey.length - 1;
    const int64_t xp = jl_round((x0 - ex.first) / ex.step + 1.0);   // histogram_pix :502, :378-379
    const int64_t yp = jl_round((y0 - ey.first) / ey.step + 1.0);
    const int64_t xo = imax(1, jl_round(15.0 * sx / ex.step / 2.0)); // size(obj) :293, :381
    const int64_t yo = imax(1, jl_round(10.0 * sy / ey.step / 2.0)); // :382
    const int64_t xa = imax(1, xp - xo), xb = imin(nx, xp + xo);    // :384
    const int64_t ya = imax(1, yp - yo), yb = imin(ny, yp + yo);    // :385
    const int64_t lx = xb - xa + 1, ly = yb - ya + 1;
    if (lx <= 1 || ly <= 1) {                                        // :401
        *out = empty_desc();
        return 0;
    }
    // xriter / yriter: range(histogram_data(first+1/2), histogram_data(last+1/2); length) :390-395
    const double xs = ((double)xa + 0.5 - 1.0) * ex.step + ex.first;
    const double xe = ((double)xb + 0.5 - 1.0) * ex.step + ex.first;
    const double ys = ((double)ya + 0.5 - 1.0) * ey.step + ey.first;
    const double ye = ((double)yb + 0.5 - 1.0) * ey.step + ey.first;
    const double xst = (xe - xs) / (double)(lx - 1), yst = (ye - ys) / (double)(ly - 1);
    const double hx = xst / 2.0, hy = yst / 2.0;
    const double s2x = 1.4142135623730951 * sx;
    PointDesc d{};
    d.xa = (int32_t)(xa - 1);
    d.xb = (int32_t)(xb - 1);
    d.ya = (int32_t)(ya - 1);
    d.yb = (int32_t)(yb - 1);
    d.ex = (float)(hx / s2x);
    d.ay = (float)((ys - y0) / sy);
    d.dv = (float)(yst / sy);
    d.ey = (float)(kGLNode * hy / sy);
    double pref = A * hy / (2.0 * 2.5066282746310002 * sy);          // prefac*h_y, :318,:323
    if (d.ex < kSumEps) pref *= 4.0 * hx / s2x / 1.7724538509055160;   // series form factor
    d.pref = (float)pref;
    set_x_form(&d, (xs - x0) / s2x, xst / s2x, true, c * sy / s2x, (int)nx);
    *out = d;
    return lx * ly;
}

// Asymmetric pixel-space kernel -- bin_cmd_smooth :598-609, addstar! :348-364.
// (x0, y0) in real units, converted to fractional pixels like the reference.
__host__ __device__ inline int64_t prep_asymmetric(double col, double mag, double cerr,
                                                   double merr, double A, Range ex, Range ey,
                                                   PointDesc* out)
{
#pragma clang fp contract(off)
    const int64_t nx = ex.length - 1, ny = ey.length - 1;
    const double x0 = (col - ex.first) / ex.step + 1.0;             // :601
    const double y0 = (mag - ey.first) / ey.step + 1.0;             // :602
    const double sx = cerr / ex.step, sy = merr / ey.step;          // :603-604
    const int64_t cx = jl_ceil(sx * 10.0), cy = jl_ceil(sy * 10.0); // size(obj) :247
    const int64_t x = jl_round(x0), y = jl_round(y0);               // :350
    const int64_t xo = imax(1, cx / 2), yo = imax(1, cy / 2);       // :351-352
    const int64_t xa = imax(1, x - xo), xb = imin(nx, x + xo);      // :356
    const int64_t ya = imax(1, y - yo), yb = imin(ny, y + yo);      // :357
    const int64_t lx = xb - xa + 1, ly = yb - ya + 1;
    if (lx <= 1 || ly <= 1) {                                        // :359
        *out = empty_desc();
        return 0;
    }
    const double s2x = 1.4142135623730951 * sx, s2y = 1.4142135623730951 * sy;
    PointDesc d{};
    d.xa = (int32_t)(xa - 1);
    d.xb = (int32_t)(xb - 1);
    d.ya = (int32_t)(ya - 1);
    d.yb = (int32_t)(yb - 1);
    d.ex = (float)(0.5 / s2x);
    d.ay = (float)(((double)ya + 0.5 - y0) / s2y);
    d.dv = (float)(1.0 / s2y);
    d.ey = (float)(0.5 / s2y);
    double pref = A / 4.0;
    if (d.ex < kSumEpsAsym) pref *= 4.0 * (0.5 / s2x) / 1.7724538509055160;
    if (d.ey < kSeriesEps) pref *= 4.0 * (0.5 / s2y) / 1.7724538509055160;
    d.pref = (float)pref;
    // evaluate at i + 1/2 :361
    set_x_form(&d, ((double)xa + 0.5 - x0) / s2x, 1.0 / s2x, false, 0.0, (int)nx);
    *out = d;
    return lx * ly;
}

__host__ __device__ inline float fast_exp(float x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __expf(x);
#else
    return std::exp(x);
#endif
}

__host__ __device__ inline float fast_exp2(float x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_exp2f(x);
#else
    return std::exp2(x);
#endif
}

__host__ __device__ inline float clamp126(float x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_fmed3f(x, -126.0f, 126.0f);
#else
    return fminf(fmaxf(x, -126.0f), 126.0f);
#endif
}

// exp(-u^2) * S(u^2)  (the full-degree series form of D without its 4e/sqrt(pi)
// factor; the asymmetric kernel's y factor)
__host__ __device__ inline float d_series(float u, const Series& s)
{
    float w = u * u;
    w = w < 100.0f ? w : 100.0f;
    const float poly = fmaf(fmaf(fmaf(fmaf(s.s4, w, s.s3), w, s.s2), w, s.s1), w, s.s0);
    return fast_exp(-w) * poly;
}

__host__ __device__ inline float fast_rcp(float x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcpf(x);
#else
    return 1.0f / x;
#endif
}

// erfc(x) for x >= 0, branch-free: the Chebyshev-fitted form of Numerical
// Recipes (Press et al., 2nd ed., section 6.2, erfcc), fractional error below
// 1.2e-7 for every x >= 0 in exact arithmetic.
__host__ __device__ inline float erfc_pos(float x)
{
    const float t = fast_rcp(fmaf(0.5f, x, 1.0f));
    float p = 0.17087277f;
    p = fmaf(p, t, -0.82215223f);
    p = fmaf(p, t, 1.48851587f);
    p = fmaf(p, t, -1.13520398f);
    p = fmaf(p, t, 0.27886807f);
    p = fmaf(p, t, -0.18628806f);
    p = fmaf(p, t, 0.09678418f);
    p = fmaf(p, t, 0.37409196f);
    p = fmaf(p, t, 1.00002368f);
    p = fmaf(p, t, -1.26551223f);
    return t * fast_exp(fmaf(-x, x, p));
}

// erfc(|b|) with the sign of b, and erf(b1) - erf(b0) of a column from its two
// edges' values: both >= 0: e0 - e1; both < 0: |e1| - |e0|; across 0: 2 - |e1| - |e0|
__host__ __device__ inline float signed_erfc(float b) { return copysignf(erfc_pos(fabsf(b)), b); }
__host__ __device__ inline float erf_diff(float e0, float e1)
{
    const float d = e0 - e1;
    return __builtin_signbitf(e0) && !__builtin_signbitf(e1) ? 2.0f + d : d;
}

// erf(u + e) - erf(u - e) through erfc of non-negative arguments (D is even
// in u), so that it keeps its relative accuracy in the tails
__host__ __device__ inline float d_direct(float u, float e)
{
    const float a = fabsf(u);
    const float hi = erfc_pos(a + e);
    return a >= e ? erfc_pos(a - e) - hi : 2.0f - hi - erfc_pos(e - a);
}

// The asymmetric kernel's y factor of a row at coordinate v (half height ey).
__host__ __device__ inline float y_factor(float v, float ey)
{
    return ey < kSeriesEps ? d_series(v, series_coeffs(ey)) : d_direct(v, ey);
}

// Row weights of the covariant kernel: W_k = pref w_k exp(-t_k^2/2) at the GL
// nodes t_k = tj + (k-1) ey, and the x shifts h_k = g t_k.
__host__ __device__ inline void cov_row(const PointDesc& d, int row, float* W, float* h)
{
    const float tj = fmaf((float)(row - d.ya), d.dv, d.ay);
    const float t0 = tj - d.ey, t2 = tj + d.ey;
    const float hl = (float)(-0.5 * kLog2e);
    W[0] = d.pref * kW0 * fast_exp2(hl * t0 * t0);
    W[1] = d.pref * kW1 * fast_exp2(hl * tj * tj);
    W[2] = d.pref * kW0 * fast_exp2(hl * t2 * t2);
    h[0] = d.g * t0;
    h[1] = d.g * tj;
    h[2] = d.g * t2;
}

// The covariant row in the Gaussian form's terms: M_k = pref w_k, the log2 of
// the node's y weight L_k = -(log2 e / 2) t_k^2 (it joins the exponent of the
// strip recurrence, so no exp2 of its own) and the x shifts h_k = g t_k.
__host__ __device__ inline void cov_row_log(const PointDesc& d, int row, float* M, float* L, float* h)
{
    const float tj = fmaf((float)(row - d.ya), d.dv, d.ay);
    const float t0 = tj - d.ey, t2 = tj + d.ey;
    const float hl = (float)(-0.5 * kLog2e);
    M[0] = d.pref * kW0;
    M[1] = d.pref * kW1;
    M[2] = M[0];
    L[0] = hl * t0 * t0;
    L[1] = hl * tj * tj;
    L[2] = hl * t2 * t2;
    h[0] = d.g * t0;
    h[1] = d.g * tj;
    h[2] = d.g * t2;
}

// The same for a row of merged nodes (kGauss1: one, kGauss2: two; see
// set_row_nodes).
template <int NODES>
__host__ __device__ inline void merged_row(const PointDesc& d, int row, float* M, float* L, float* h)
{
    const float t = fmaf((float)(row - d.ya), d.dv, d.ay);
    if constexpr (NODES == 1) {
        M[0] = d.pref;
        L[0] = fmaf(d.s2, t * t, d.s1) * (t * t);
        h[0] = d.g * t;
    } else {
        M[0] = M[1] = d.pref;
        L[0] = fmaf(d.s1, t, d.s2) * t;
        L[1] = fmaf(d.s1, t, -d.s2) * t;
        h[0] = fmaf(d.g, t, -d.s3);
        h[1] = fmaf(d.g, t, d.s3);
    }
}

// part = in ? v : part, as a select: v is computed for every lane first (the
// register barrier keeps the compiler from sinking its computation into a
// branch per column, which serialises the columns' dependency chains)
__host__ __device__ __forceinline__ void masked_set(float& part, float v, bool in)
{
#if defined(__HIP_DEVICE_COMPILE__)
    __asm__ volatile("" : "+v"(v));
#endif
    part = in ? v : part;
}

// f(integral_constant<int, C>) for C = I .. N-1, in order
template <int I, int N, typename F>
__host__ __device__ __forceinline__ void static_for(F&& f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// The Gaussian form over one row's strip: part[c] += sum_k M[k] 2^(L[k]) E_k(c),
// E_k(c) = 2^-(a_k(c))^2, by a product recurrence from the strip's middle.
// With m the x coordinate midway between columns 7 and 8 and s = c - 7.5,
//   (m + s du)^2 = m^2 + 2 s m du + s^2 du^2,
// so E(8 + j) = P B^j q[j] and E(7 - j) = P B^-(j+1) q[j], P = 2^-(m^2 + m du),
// B = 2^(-2 m du), q[j] = 2^-(du (j + 1/2))^2 (prepared per point).  A row takes
// three exp2 per node (the two merged nodes four) instead of one per column (an exp2 takes two
// VALU issue slots, an FMA or multiply one), and a column costs one FMA and one
// multiply per node.  Each column adds the nodes in order k = 0, 1, 2.
//
// B and 1/B have to stay finite: where a far strip's P has underflowed to 0, a
// product with an infinite one would be a NaN.  Without shear |m| stays within
// the footprint's 5.3 standard deviations and a strip, and the merged nodes'
// |2 m du| is bounded at the preparation (kMaxLogB, set_row_nodes).  The three GL
// nodes' m holds the rows' shear g t, which has no bound, so their exponent is
// clamped to +-126: du < 0.3 (half bin width e < 0.12), so |m| > 200 where the
// clamp acts, and P is 0 there, and stays 0.  Their B are computed node by node:
// a node's B is used where its own |m| is small, and as the middle node's B times
// a prepared 2^(2 g ey du) it would carry the rounding of an exponent as large as
// the nodes' distance (1e-5 of the peak in rows much higher than the kernel).
// The two merged nodes lie within 0.1 of each other and share one.
template <int NODES>
__host__ __device__ __forceinline__ void gauss_strip(const PointDesc& d, const float* M, const float* L,
                                                     const float* h, int col0, float* part)
{
    static_assert(kCPT == 16, "the recurrence runs 8 columns each way from the strip's middle");
    static_assert(NODES >= 1 && NODES <= 3, "one node, two merged ones or three GL nodes");
    const float base = fmaf((float)(col0 - d.xa), d.du, d.ax);
    const float du = d.du;
    float m[NODES], pf[NODES], B[NODES], Bi[NODES];
#pragma unroll
    for (int k = 0; k < NODES; ++k) {
        m[k] = fmaf(7.5f, du, base + h[k]);
        pf[k] = M[k] * fast_exp2(L[k] - m[k] * (m[k] + du));
    }
    if constexpr (NODES == 2) {
        const float md2 = (m[0] + m[1]) * du;
        const float Bm = fast_exp2(-md2), Bmi = fast_exp2(md2);
        B[0] = Bm * d.gf;
        Bi[0] = Bmi * d.gfi;
        B[1] = Bm * d.gfi;
        Bi[1] = Bmi * d.gf;
    } else {
#pragma unroll
        for (int k = 0; k < NODES; ++k) {
            const float md2 = NODES == 3 ? clamp126(2.0f * m[k] * du) : 2.0f * m[k] * du;
            B[k] = fast_exp2(-md2);
            Bi[k] = fast_exp2(md2);
        }
    }
#pragma unroll
    for (int k = 0; k < NODES; ++k) {
        float f = pf[k], b = pf[k] * Bi[k];
        const float Bk = B[k], Bik = Bi[k];
        static_for<0, 8>([&](auto jj) {
            constexpr int j = decltype(jj)::value;
            constexpr int cf = 8 + j, cb = 7 - j;
            part[cf] = fmaf(f, d.q[j], part[cf]);
            part[cb] = fmaf(b, d.q[j], part[cb]);
            if constexpr (j < 7) {
                f *= Bk;
                b *= Bik;
            }
        });
    }
}

// Left edge of footprint column l of a narrow kernel in the erf-difference
// form, for GL node shift h: x0 + l du + h, x0 = ax - ex (the wave-cooperative
// path: one column per lane, the right edge being the next column's left).
__host__ __device__ inline float direct_edge(const PointDesc& d, int l, float h)
{
    return fmaf((float)l, d.du, d.ax - d.ex) + h;
}

// A point in the Gaussian form (its rows' nodes not merged) or the sum form on
// one row's strip, only columns inside its footprint receiving anything.  COV:
// the covariant kernel (else the asymmetric one).  The sum form's Gaussians
// are one loop over the same code.
template <bool COV>
__host__ __device__ __forceinline__ void add_point(const PointDesc& d, int row, int col0, float* part)
{
    constexpr int NODES = COV ? 3 : 1;
    float M[NODES], L[NODES] = {}, h[NODES] = {}, sum[kCPT] = {};
    if constexpr (COV) cov_row_log(d, row, M, L, h);
    else M[0] = d.pref * y_factor(fmaf((float)(row - d.ya), d.dv, d.ay), d.ey);
    float shift = -d.s3;                                       // -s3, s3, then 0
    for (int i = 0;;) {
        float hs[NODES];
#pragma unroll
        for (int k = 0; k < NODES; ++k) hs[k] = h[k] + shift;
        gauss_strip<NODES>(d, M, L, hs, col0, sum);
        if (++i == d.terms) break;
        shift = i == 1 ? d.s3 : 0.0f;
        const float amp = i == 1 ? 1.0f : d.s1;
#pragma unroll
        for (int k = 0; k < NODES; ++k) M[k] *= amp;
    }
    const int lo = d.xa - col0, hi = d.xb - col0;
#pragma unroll
    for (int c = 0; c < kCPT; ++c) masked_set(part[c], part[c] + sum[c], c >= lo && c <= hi);
}

}  // namespace psf
}  // namespace sfh
