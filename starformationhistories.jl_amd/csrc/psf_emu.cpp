// psf_emu.cpp -- host build of the deposition kernel's arithmetic (the
// __host__ __device__ functions of sfh_psf.h) arranged exactly like
// k_dep_gather: FP32 per-point contributions summed per 64-point chunk -- the
// chunk's common-case points (Gaussian form with one node per row, then with
// two, footprint spanning the grid width) first, then the others, each in
// point order -- then flushed into FP64, the wide kernels' sums (on every
// kStep-th column) apart and interpolated at the end; erf-difference kernels
// add each bin straight into FP64.  Lets the CPU test-suite check the FP32
// formulation and the footprint index math against the FP64 oracle without a
// GPU.
#include "sfh_psf.h"

#include <cstring>
#include <vector>

using namespace sfh::psf;

extern "C" int64_t emu_bin_cmd_smooth(const double* colors, const double* mags, const double* cerr,
                                      const double* merr, const double* weights, const double* cmult,
                                      int64_t P, double cov_mult, Range ex, Range ey, double* out)
{
    const int nx = (int)(ex.length - 1), ny = (int)(ey.length - 1);
    const bool asym = cov_mult == 0.0 && cmult == nullptr;
    std::vector<PointDesc> desc((size_t)P);
    int64_t pairs = 0;
    for (int64_t p = 0; p < P; ++p) {
        const double c = cmult ? cmult[p] : cov_mult;
        pairs += asym ? prep_asymmetric(colors[p], mags[p], cerr[p], merr[p], weights[p], ex, ey, &desc[p])
                      : prep_covariant(colors[p], mags[p], cerr[p], merr[p], c, weights[p], ex, ey, &desc[p]);
    }
    // the kernel's strips: a row's columns in runs of kCPT from column 0
    const int ncg = (nx + kCPT - 1) / kCPT;
    std::vector<double> acc((size_t)ncg * kCPT * ny, 0.0);
    std::vector<float> part((size_t)ncg * kCPT * ny, 0.0f);
    const size_t ld = (size_t)ncg * kCPT;
    // the wide kernels' sums on their nodes
    const int wcg = wide_pays(nx) ? (wide_nodes(nx) + kCPT - 1) / kCPT : 0;
    std::vector<double> wacc((size_t)wcg * kCPT * ny, 0.0);
    std::vector<float> wpart((size_t)wcg * kCPT * ny, 0.0f);
    for (int64_t pc = 0; pc < P; pc += 64) {
        const int64_t pe = pc + 64 < P ? pc + 64 : P;
        for (int64_t q = pc; q < pe; ++q) {
            const PointDesc& d = desc[q];
            if (d.xa > d.xb || d.kind < kWide1) continue;
            for (int row = d.ya; row <= d.yb; ++row)
                for (int cg = 0; cg < wcg; ++cg) {
                    float M[2], L[2], h[2];
                    float* pp = &wpart[((size_t)row * wcg + cg) * kCPT];
                    if (d.kind == kWide1) {
                        merged_row<1>(d, row, M, L, h);
                        gauss_strip<1>(d, M, L, h, cg * kCPT, pp);
                    } else {
                        merged_row<2>(d, row, M, L, h);
                        gauss_strip<2>(d, M, L, h, cg * kCPT, pp);
                    }
                }
        }
        for (int pass = 0; pass < 3; ++pass) {
            for (int64_t q = pc; q < pe; ++q) {
                const PointDesc& d = desc[q];
                if (d.xa > d.xb || d.kind >= kWide1) continue;
                const bool full = d.xa == 0 && d.xb == nx - 1;
                const int in = d.kind == kGauss1 ? 0 : full && d.kind == (asym ? kGauss : kGauss2) ? 1 : 2;
                if (in != pass) continue;
                // erf-difference kernels: the kernel's wave-cooperative
                // path, one column at a time, each bin straight into FP64
                const bool coop = d.kind == kDirect;
                for (int row = d.ya; row <= d.yb; ++row) {
                    float W[3], L[3] = {0.0f, 0.0f, 0.0f}, h[3] = {0.0f, 0.0f, 0.0f};
                    if (pass == 0) merged_row<1>(d, row, W, L, h);
                    else if (asym) W[0] = d.pref * y_factor(fmaf((float)(row - d.ya), d.dv, d.ay), d.ey);
                    else if (pass == 1) merged_row<2>(d, row, W, L, h);
                    else cov_row(d, row, W, h);
                    if (coop) {
                        const int nodes = asym ? 1 : 3;
                        for (int l = 0; l <= d.xb - d.xa; ++l) {
                            float v = 0.0f;
                            for (int k = 0; k < nodes; ++k) {
                                const float e0 = signed_erfc(direct_edge(d, l, h[k]));
                                v = fmaf(W[k], erf_diff(e0, signed_erfc(direct_edge(d, l + 1, h[k]))), v);
                            }
                            acc[(size_t)row * ld + d.xa + l] += (double)v;
                        }
                        continue;
                    }
                    for (int cg = 0; cg < ncg; ++cg) {
                        const int col0 = cg * kCPT;
                        float* pp = &part[(size_t)row * ld + col0];
                        if (pass == 0 || (asym && pass == 1)) gauss_strip<1>(d, W, L, h, col0, pp);
                        else if (pass == 1) gauss_strip<2>(d, W, L, h, col0, pp);
                        else if (col0 <= d.xb && col0 + kCPT - 1 >= d.xa) {
                            if (asym) add_point<false>(d, row, col0, pp);
                            else add_point<true>(d, row, col0, pp);
                        }
                    }
                }
            }
        }
        for (size_t k = 0; k < wacc.size(); ++k) {
            wacc[k] += (double)wpart[k];
            wpart[k] = 0.0f;
        }
        for (size_t k = 0; k < acc.size(); ++k) {
            acc[k] += (double)part[k];
            part[k] = 0.0f;
        }
    }
    const InterpWeights iw = interp_weights();
    for (int row = 0; row < ny; ++row)
        for (int col = 0; col < nx; ++col) {
            double v = acc[(size_t)row * ld + col];
            const double* n = wcg ? &wacc[(size_t)row * wcg * kCPT + col / kStep] : nullptr;
            const int r = col % kStep;
            if (n && r == 0) v += n[kLead];
            else if (n)
                for (int k = 0; k < kTaps; ++k) v = fma(iw.w[r][k], n[k], v);
            out[(size_t)row * nx + col] = v;
        }
    return pairs;
}
