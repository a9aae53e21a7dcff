// Critical curves and caustics (reference: critical_and_caustic_curves,
// src/caustics/point_source.py:1582-1649): the critical-curve polynomial (:1482-1534) on a grid
// of phases, its roots from the reference's initial estimates, the roots continued along the
// phases (match_points, utils.py:15-40), mapped through the lens equation (:1536-1556) and
// shifted into the frame of the API.
//
// Three kernels around the root solver: coefficients, one phase per lane; solver; continuation
// with the map, one workgroup per lens.  A curve of 200 points has work for four waves, so the
// call is bound by latency: 120 us, of which the solve's iterations take 84-110.  With some 40
// elementwise launches around the solver (three lenses: 60) it took 415 us (one MI355X).
//
// Near phases 0 and pi the polynomial is real up to rounding, and so are the reference's
// initial estimates: which root each of them leads to there follows the rounding of the
// coefficients.  They are therefore formed operation by operation as elementwise tensor
// expressions form them, each product and sum rounded (a product with a real factor scales
// both components; a complex product rounds one of its two partial products).
#include "caustics_hip.h"
#include "chain.hpp"

using namespace caus;

namespace {

constexpr int kCurveBlock = 256;

// parameters of lens b: columns on the device (stride 0 or 1) or values
struct CurveParams {
    const double* p[5];
    int64_t st[5];
    double v[5];
    __device__ __forceinline__ double at(int k, int64_t b) const {
        return p[k] ? p[k][b * st[k]] : v[k];
    }
};

struct CurveLens {
    double a, x_cm, e1, e2;
    cd r3;
};

template <int NL>
__device__ __forceinline__ CurveLens curve_lens(const CurveParams& P, int64_t b) {
#pragma clang fp contract(off)
    CurveLens L;
    const double s = P.at(0, b), q = P.at(1, b);
    L.a = 0.5 * s;
    L.x_cm = L.a * (1.0 - q) / (1.0 + q);
    if constexpr (NL == 2) {
        L.e1 = 1.0 / (1.0 + q);
        L.e2 = 1.0 - L.e1;
    } else {
        const double q3 = P.at(2, b), R = P.at(3, b), psi = P.at(4, b);
        L.e1 = q / (1.0 + q + q3);
        L.e2 = q * L.e1;
        L.r3 = cd{R * cos(psi), R * sin(psi)};
    }
    return L;
}

// ascending coefficients at phase phi; four: the exponent 4, not known to the compiler, so that
// the power is taken by the library's pow
template <int NL>
__device__ __forceinline__ void curve_coeffs(const CurveLens& L, double phi, double four,
                                             cd (&c)[NL == 2 ? 5 : 7]) {
#pragma clang fp contract(off)
    const double a = L.a, a2 = a * a, a4 = pow(a, four), e1 = L.e1, e2 = L.e2;
    const cd x = cd{cos(-phi), sin(-phi)};
    if constexpr (NL == 2) {
        c[4] = x;
        c[3] = cd{0.0 * x.re, 0.0 * x.im};
        c[2] = (-2.0 * a2) * x - cd{1.0, 0.0};
        c[1] = cd{-4.0 * a * e1 + 2.0 * a, 0.0};
        c[0] = a4 * x - cd{a2, 0.0};
    } else {
        const cd r3 = L.r3, r32 = r3 * r3;
        const auto re = [](double v) { return cd{v, 0.0}; };
        c[6] = x;
        c[5] = (-2.0 * x) * r3;
        c[4] = (-2.0 * a2) * x - re(1.0) + x * r32;
        c[3] = ((4.0 * a2) * x) * r3 - re(2.0 * a * e1) + re(2.0 * a * e2) + (2.0 * e1) * r3 +
               (2.0 * e2) * r3;
        c[2] = a4 * x - re(3.0 * a2 * e1) - re(3.0 * a2 * e2) + re(2.0 * a2) -
               ((2.0 * a2) * x) * r32 + (4.0 * a * e1) * r3 - (4.0 * a * e2) * r3 - e1 * r32 -
               e2 * r32;
        c[1] = ((-2.0 * a4) * x) * r3 + (2.0 * a2 * e1) * r3 + (2.0 * a2 * e2) * r3 -
               (2.0 * a * e1) * r32 + (2.0 * a * e2) * r32;
        c[0] = re(a4 * e1 + a4 * e2 - a4) + (a4 * x) * r32 - (a2 * e1) * r32 - (a2 * e2) * r32;
    }
}

template <int NL>
__global__ __launch_bounds__(kCurveBlock) void k_curve_coeffs(CurveParams P, const double* phi,
                                                              int64_t npts, int64_t n, double four,
                                                              cd* coeffs) {
    constexpr int N1 = NL == 2 ? 5 : 7;
    for (int64_t i = (int64_t)blockIdx.x * kCurveBlock + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kCurveBlock) {
        const int64_t b = i / npts;
        cd c[N1];
        curve_coeffs<NL>(curve_lens<NL>(P, b), phi[i - b * npts], four, c);
#pragma unroll
        for (int k = 0; k < N1; ++k) coeffs[i * N1 + k] = c[k];
    }
}

// continuation of a lens' roots (chain.hpp), the curves row after row in the API's frame and
// their images in the source plane
template <int NL, int NT>
__global__ __launch_bounds__(NT) void k_curve_map(CurveParams P, const cd* __restrict__ roots,
                                                  int64_t npts, int64_t B, uint64_t* words,
                                                  cd* __restrict__ crit, cd* __restrict__ caus) {
    constexpr int N = NL == 2 ? 4 : 6;
    for (int64_t b = blockIdx.x; b < B; b += gridDim.x) {
        const cd* p = roots + b * npts * N;
        uint64_t* w = words + b * npts;
        auto get = [p](int64_t k, int r) { return p[k * N + r]; };
        auto word = [w](int64_t k) -> uint64_t& { return w[k]; };
        chain_perms<N, NT>(get, word, npts);
        const CurveLens L = curve_lens<NL>(P, b);
        for (int64_t k = threadIdx.x; k < npts; k += NT) {
            const uint64_t perm = w[k];
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const cd z = p[k * N + (int)((perm >> (4 * i)) & 0xF)];
                cd y = z - L.e1 * crcp<2>(conj(z) - cd{L.a, 0.0});
                y = y - L.e2 * crcp<2>(conj(z) + cd{L.a, 0.0});
                if constexpr (NL == 3) y = y - (1.0 - L.e1 - L.e2) * crcp<2>(conj(z) - conj(L.r3));
                const int64_t o = (b * N + i) * npts + k;
                crit[o] = z - cd{L.x_cm, 0.0};
                caus[o] = y - cd{L.x_cm, 0.0};
            }
        }
    }
}

template <int NL>
int curves(hipStream_t s, const CurveParams& P, int64_t B, const double* phi, int64_t npts,
           char* ws, cd* crit, cd* caus, int itmax) {
    constexpr int N = NL == 2 ? 4 : 6;
    const int64_t n = B * npts;
    cd* coeffs = reinterpret_cast<cd*>(ws);
    cd* roots = coeffs + n * (N + 1);
    uint64_t* words = reinterpret_cast<uint64_t*>(roots + n * N);
    const int64_t blocks = (n + kCurveBlock - 1) / kCurveBlock;
    hipLaunchKernelGGL((k_curve_coeffs<NL>), dim3((unsigned)(blocks < 65536 ? blocks : 65536)),
                       dim3(kCurveBlock), 0, s, P, phi, npts, n, 4.0, coeffs);
    const int rc = caus_roots(s, reinterpret_cast<const double*>(coeffs), nullptr,
                              reinterpret_cast<double*>(roots), nullptr, nullptr, n, N, itmax,
                              CAUS_MODE_FP64, CAUS_INIT_REFERENCE);
    if (rc != CAUS_OK) return rc;
    const dim3 g((unsigned)(B < (1 << 20) ? B : (1 << 20)));   // strides over the lenses
    if (npts <= 64)   // as k_match_chain: one wave up to 64 points
        hipLaunchKernelGGL((k_curve_map<NL, 64>), g, dim3(64), 0, s, P, roots, npts, B, words,
                           crit, caus);
    else
        hipLaunchKernelGGL((k_curve_map<NL, 256>), g, dim3(256), 0, s, P, roots, npts, B, words,
                           crit, caus);
    return hipGetLastError() == hipSuccess ? CAUS_OK : CAUS_ERR_LAUNCH;
}

}  // namespace

extern "C" int64_t caus_critical_curves_workspace_bytes(int32_t nlenses, int64_t B, int64_t npts) {
    if (nlenses < 2 || nlenses > 3 || B < 0 || npts < 0) return -1;
    const int64_t n = nlenses == 2 ? 4 : 6;
    return B * npts * ((2 * n + 1) * (int64_t)sizeof(cd) + (int64_t)sizeof(uint64_t));
}

extern "C" int caus_critical_curves(void* stream, int32_t nlenses, const double* const* params,
                                    const int64_t* strides, const double* values, int64_t B,
                                    const double* phi, int64_t npts, double* critical,
                                    double* caustic, void* workspace, int64_t workspace_bytes,
                                    int32_t itmax) {
    const int64_t need = caus_critical_curves_workspace_bytes(nlenses, B, npts);
    if (need < 0 || itmax < 0) return CAUS_ERR_ARG;
    if (B == 0 || npts == 0) return CAUS_OK;
    if (!params || !strides || !values || !phi || !critical || !caustic || !workspace ||
        workspace_bytes < need)
        return CAUS_ERR_ARG;
    CurveParams P{};
    for (int k = 0; k < (nlenses == 2 ? 2 : 5); ++k) {
        if (strides[k] < 0) return CAUS_ERR_ARG;
        P.p[k] = params[k];
        P.st[k] = strides[k];
        P.v[k] = values[k];
    }
    hipStream_t s = (hipStream_t)stream;
    char* ws = reinterpret_cast<char*>(workspace);
    cd* c = reinterpret_cast<cd*>(critical);
    cd* y = reinterpret_cast<cd*>(caustic);
    return nlenses == 2 ? curves<2>(s, P, B, phi, npts, ws, c, y, itmax)
                        : curves<3>(s, P, B, phi, npts, ws, c, y, itmax);
}
