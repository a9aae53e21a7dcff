// C-ABI entry points of the fused point-source magnification and light-curve kernels.
#include <atomic>

#include "ps_impl.hpp"

using namespace caus;

// Scratch of caus_lightcurve_point_source_noalloc: the per-(light curve, epoch chunk)
// partial gradient sums that the caller's workspace holds in
// caus_lightcurve_point_source.  Every GPU the library runs on holds one copy until the
// process ends; calls on one GPU share it.
static constexpr int64_t kLcScratchBytes = CAUS_LC_NOALLOC_MAX_BYTES;
static __device__ __align__(256) double scratch[kLcScratchBytes / sizeof(double)];

namespace {

constexpr uint32_t kAllDirs = ~0u;   // every direction's derivative

int np_for(int nl) { return nl == 1 ? 0 : (nl == 2 ? 2 : 5); }

int check_mode(int mode) {
    return (mode == CAUS_MODE_FP64 || mode == CAUS_MODE_FP64_COMP || mode == CAUS_MODE_CF32)
               ? CAUS_OK
               : CAUS_ERR_ARG;
}

int ps_dispatch(hipStream_t s, int nl, const cd* w, int64_t N, const PsCols& params,
                int64_t per, const double* g_mag, double* mag, double* jac, uint32_t dirs,
                double* g_w, double* g_params, uint8_t* status, int itmax, int mode, bool vjp) {
    switch (nl) {
        case 1:
            return mag_point_source_nl<1>(s, w, N, params, per, g_mag, mag, jac, dirs, g_w,
                                          g_params, status, itmax, mode, vjp);
        case 2:
            return mag_point_source_nl<2>(s, w, N, params, per, g_mag, mag, jac, dirs, g_w,
                                          g_params, status, itmax, mode, vjp);
        case 3:
            return mag_point_source_nl<3>(s, w, N, params, per, g_mag, mag, jac, dirs, g_w,
                                          g_params, status, itmax, mode, vjp);
        default:
            return CAUS_ERR_ARG;
    }
}

int lc_dispatch(hipStream_t s, int nl, const double* t, int64_t T, const PsCols& lcp, int64_t L,
                const double* g_mag, double* mag, double* jac, uint32_t dirs, double* ws,
                uint8_t* status, int itmax, int mode, bool vjp) {
    switch (nl) {
        case 1:
            return lightcurve_point_source_nl<1>(s, t, T, lcp, L, g_mag, mag, jac, dirs, ws,
                                                 status, itmax, mode, vjp);
        case 2:
            return lightcurve_point_source_nl<2>(s, t, T, lcp, L, g_mag, mag, jac, dirs, ws,
                                                 status, itmax, mode, vjp);
        default:
            return lightcurve_point_source_nl<3>(s, t, T, lcp, L, g_mag, mag, jac, dirs, ws,
                                                 status, itmax, mode, vjp);
    }
}

// ---- backward pass from a kept Jacobian ------------------------------------------------
// N items in G = N / R rows of R consecutive ones; planes jac[d * N + i], the first nw of
// them (0 or 2) the derivatives along Re w and Im w.  g_w[i] = g_i (J_0, J_1), and each
// further plane k summed over its row, g_p[k * G + row] = sum_i g_i J_{nw+k, i}, in an
// order that depends on N and R alone.
// Bound: one read of g and the planes (binary light curves 56 B an epoch), so the split only
// has to put enough loads in flight.  It replaces a second solve of every epoch in the
// backward pass and torch's one reduction per parameter: 512,000 binary epochs with their
// gradient 175 -> 109 us of kernels, 50,001 triple-lens positions with 7 gradients
// 250 -> 111 us (one MI355X).
constexpr int kJacPlanes = 9;        // 4 trajectory + 5 lens parameters
constexpr int kJacWaveRow = 512;     // rows up to this long are summed by one wave each
constexpr int64_t kJacChunk = 1024;  // longer ones in chunks of at least this (4 items a thread)

struct JacArgs {
    const double *jac, *g;
    double *g_w, *g_p;
    int64_t N, R, G;
    int nw, np, nchunk;
};

// rows of one item: no sums
__global__ __launch_bounds__(kPsBlock) void k_jac_items(JacArgs a) {
    const int64_t i = (int64_t)blockIdx.x * kPsBlock + threadIdx.x;
    if (i >= a.N) return;
    const double g = a.g[i];
    if (a.g_w) {
        a.g_w[2 * i] = g * a.jac[i];
        a.g_w[2 * i + 1] = g * a.jac[a.N + i];
    }
    if (a.g_p)
        for (int k = 0; k < a.np; ++k) a.g_p[k * a.N + i] = g * a.jac[(a.nw + k) * a.N + i];
}

// sums of items first, first + step, .. below end of one row, g_w on the way; four items at a
// time keep that many loads of every plane in flight
__device__ __forceinline__ void jac_sums(const JacArgs& a, int64_t first, int64_t end, int step,
                                         double (&s)[kJacPlanes]) {
#pragma unroll
    for (int k = 0; k < kJacPlanes; ++k) s[k] = 0.0;
    for (int64_t i = first; i < end; i += 4 * (int64_t)step) {
        int64_t at[4];
        double g[4], w0[4], w1[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t j = i + (int64_t)u * step;
            at[u] = j < end ? j : first;
            g[u] = a.g[at[u]];
        }
        if (a.g_w) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                w0[u] = a.jac[at[u]];
                w1[u] = a.jac[a.N + at[u]];
            }
        }
#pragma unroll
        for (int k = 0; k < kJacPlanes; ++k)
            if (k < a.np) {
                double v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = a.jac[(a.nw + k) * a.N + at[u]];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (i + (int64_t)u * step < end) s[k] += g[u] * v[u];
            }
        if (a.g_w) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (i + (int64_t)u * step < end) {
                    a.g_w[2 * at[u]] = g[u] * w0[u];
                    a.g_w[2 * at[u] + 1] = g[u] * w1[u];
                }
        }
    }
#pragma unroll
    for (int k = 0; k < kJacPlanes; ++k)
        if (k < a.np) s[k] = wave_sum(s[k]);
}

// one wave per row
__global__ __launch_bounds__(kPsBlock) void k_jac_wave_rows(JacArgs a) {
    const int64_t row = (int64_t)blockIdx.x * (kPsBlock / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= a.G) return;
    double s[kJacPlanes];
    jac_sums(a, row * a.R + lane, (row + 1) * a.R, 64, s);
#pragma unroll
    for (int k = 0; k < kJacPlanes; ++k)
        if (k < a.np && lane == 0 && a.g_p) a.g_p[k * a.G + row] = s[k];
}

// one workgroup per chunk of a row; partial sums of chunk c go to ws[(k * G + row) * nchunk + c]
__global__ __launch_bounds__(kPsBlock) void k_jac_chunks(JacArgs a, double* out) {
    __shared__ double red[kPsBlock / 64][kJacPlanes];
    const int64_t row = blockIdx.x / a.nchunk;
    const int c = (int)(blockIdx.x % a.nchunk);
    const int64_t lo = row * a.R + a.R * c / a.nchunk, hi = row * a.R + a.R * (c + 1) / a.nchunk;
    double s[kJacPlanes];
    jac_sums(a, lo + threadIdx.x, hi, kPsBlock, s);
#pragma unroll
    for (int k = 0; k < kJacPlanes; ++k)
        if ((threadIdx.x & 63) == 0 && k < a.np) red[threadIdx.x >> 6][k] = s[k];
    __syncthreads();
    const int k = threadIdx.x;
    if (k < a.np && out) {
        double v = 0.0;
#pragma unroll
        for (int q = 0; q < kPsBlock / 64; ++q) v += red[q][k];
        out[(k * a.G + row) * a.nchunk + c] = v;
    }
}

// g_p[j] = sum of the nchunk partial sums of output j, one workgroup of one wave each
__global__ __launch_bounds__(64) void k_jac_finalize(const double* ws, double* g_p, int nchunk) {
    double v = 0.0;
    for (int c = threadIdx.x; c < nchunk; c += 64) v += ws[(int64_t)blockIdx.x * nchunk + c];
    v = wave_sum(v);
    if (threadIdx.x == 0) g_p[blockIdx.x] = v;
}

// Chunks per row: 256 rows and more give every CU a workgroup and are summed in one launch
// (a second one costs 4 us); fewer are cut, up to 1024 workgroups in all.
int jac_chunks(int64_t N, int64_t R) {
    const int64_t G = N / R;
    const int64_t by_size = (R + kJacChunk - 1) / kJacChunk, by_fill = (1024 + G - 1) / G;
    return (int)(G >= 256 ? 1 : (by_size < by_fill ? by_size : by_fill));
}

}  // namespace

extern "C" int64_t caus_jacobian_workspace_bytes(int32_t np, int64_t N, int64_t R) {
    if (np < 0 || np > kJacPlanes || N < 0 || R < 1 || N % R != 0) return -1;
    if (N == 0 || np == 0 || R <= kJacWaveRow) return 0;
    const int nchunk = jac_chunks(N, R);
    return nchunk == 1 ? 0 : (N / R) * np * nchunk * (int64_t)sizeof(double);
}

extern "C" int caus_jacobian_vjp(void* stream, const double* jac, int64_t N, int32_t nw,
                                 int32_t np, int64_t R, const double* g, double* g_w,
                                 double* g_params, double* workspace, int64_t workspace_bytes) {
    const int64_t need = caus_jacobian_workspace_bytes(np, N, R);
    if (need < 0 || (nw != 0 && nw != 2) || (nw == 0 && g_w)) return CAUS_ERR_ARG;
    if (N == 0) return CAUS_OK;
    if (!jac || !g || workspace_bytes < need || (need > 0 && !workspace)) return CAUS_ERR_ARG;
    hipStream_t s = (hipStream_t)stream;
    JacArgs a{jac, g, g_w, g_params, N, R, N / R, nw, np, 1};
    if (R == 1) {
        const int64_t blocks = (N + kPsBlock - 1) / kPsBlock;
        if (blocks > INT32_MAX) return CAUS_ERR_ARG;
        hipLaunchKernelGGL(k_jac_items, dim3((unsigned)blocks), dim3(kPsBlock), 0, s, a);
    } else if (R <= kJacWaveRow) {
        const int64_t blocks = (a.G + kPsBlock / 64 - 1) / (kPsBlock / 64);
        if (blocks > INT32_MAX) return CAUS_ERR_ARG;
        hipLaunchKernelGGL(k_jac_wave_rows, dim3((unsigned)blocks), dim3(kPsBlock), 0, s, a);
    } else {
        a.nchunk = jac_chunks(N, R);
        if (a.G * a.nchunk > INT32_MAX) return CAUS_ERR_ARG;
        const bool two = a.nchunk > 1 && np > 0 && g_params;
        hipLaunchKernelGGL(k_jac_chunks, dim3((unsigned)(a.G * a.nchunk)), dim3(kPsBlock), 0, s,
                           a, two ? workspace : (a.nchunk > 1 ? nullptr : g_params));
        if (two)
            hipLaunchKernelGGL(k_jac_finalize, dim3((unsigned)(a.G * np)), dim3(64), 0, s,
                               workspace, g_params, a.nchunk);
    }
    return hipGetLastError() == hipSuccess ? CAUS_OK : CAUS_ERR_LAUNCH;
}

// n caller columns; false if one is missing or a stride is negative
static bool user_cols(const double* const* p, const int64_t* st, int n, PsCols& c) {
    if (n > 0 && (!p || !st)) return false;
    for (int k = 0; k < n; ++k) {
        if (!p[k] || st[k] < 0) return false;
        c.p[k] = p[k];
        c.st[k] = st[k];
    }
    return true;
}

extern "C" int caus_mag_point_source_jac_planes(void* stream, int32_t nlenses, const double* w,
                                                int64_t N, const double* const* params,
                                                const int64_t* strides, int64_t per,
                                                double* mag, double* jac, uint32_t planes,
                                                int32_t itmax, int32_t mode) {
    if (N < 0 || itmax < 0 || nlenses < 1 || nlenses > 3 || check_mode(mode) != CAUS_OK ||
        per < 1)
        return CAUS_ERR_ARG;
    if (N == 0) return CAUS_OK;
    PsCols c{};
    if (!w || !mag || !user_cols(params, strides, np_for(nlenses), c)) return CAUS_ERR_ARG;
    return ps_dispatch((hipStream_t)stream, nlenses, reinterpret_cast<const cd*>(w), N, c, per,
                       nullptr, mag, jac, planes, nullptr, nullptr, nullptr, itmax, mode,
                       jac != nullptr);
}

extern "C" int caus_mag_point_source_jac(void* stream, int32_t nlenses, const double* w,
                                         int64_t N, const double* const* params,
                                         const int64_t* strides, int64_t per, double* mag,
                                         double* jac, int32_t itmax, int32_t mode) {
    return caus_mag_point_source_jac_planes(stream, nlenses, w, N, params, strides, per, mag, jac,
                                            kAllDirs, itmax, mode);
}

extern "C" int caus_lightcurve_point_source_jac_planes(
    void* stream, int32_t nlenses, const double* t, int64_t T, const double* const* params,
    const int64_t* strides, int64_t L, double* mag, double* jac, uint32_t planes, int32_t itmax,
    int32_t mode) {
    if (T < 0 || L < 0 || itmax < 0 || nlenses < 1 || nlenses > 3 || check_mode(mode) != CAUS_OK)
        return CAUS_ERR_ARG;
    if (T == 0 || L == 0) return CAUS_OK;
    PsCols c{};
    if (L > 65535 || !t || !mag || !user_cols(params, strides, 4 + np_for(nlenses), c))
        return CAUS_ERR_ARG;
    return lc_dispatch((hipStream_t)stream, nlenses, t, T, c, L, nullptr, mag, jac, planes,
                       nullptr, nullptr, itmax, mode, jac != nullptr);
}

extern "C" int caus_lightcurve_point_source_jac(void* stream, int32_t nlenses, const double* t,
                                                int64_t T, const double* const* params,
                                                const int64_t* strides, int64_t L, double* mag,
                                                double* jac, int32_t itmax, int32_t mode) {
    return caus_lightcurve_point_source_jac_planes(stream, nlenses, t, T, params, strides, L, mag,
                                                   jac, kAllDirs, itmax, mode);
}

extern "C" int caus_mag_point_source(void* stream, int32_t nlenses, const double* w, int64_t N,
                                     const double* params, int64_t params_stride, double* mag,
                                     uint8_t* status, int32_t itmax, int32_t mode) {
    if (N < 0 || itmax < 0 || nlenses < 1 || nlenses > 3 || check_mode(mode) != CAUS_OK)
        return CAUS_ERR_ARG;
    if (N == 0) return CAUS_OK;
    if (!w || !mag || (nlenses > 1 && !params) || params_stride < 0) return CAUS_ERR_ARG;
    return ps_dispatch((hipStream_t)stream, nlenses, reinterpret_cast<const cd*>(w), N,
                       ps_rows(params, params_stride), 1, nullptr, mag, nullptr, kAllDirs,
                       nullptr, nullptr, status, itmax, mode, false);
}

extern "C" int caus_mag_point_source_vjp(void* stream, int32_t nlenses, const double* w,
                                         int64_t N, const double* params, int64_t params_stride,
                                         const double* g_mag, double* mag, double* g_w,
                                         double* g_params, uint8_t* status, int32_t itmax,
                                         int32_t mode) {
    if (N < 0 || itmax < 0 || nlenses < 1 || nlenses > 3 || check_mode(mode) != CAUS_OK)
        return CAUS_ERR_ARG;
    if (N == 0) return CAUS_OK;
    if (!w || !mag || !g_mag || (nlenses > 1 && !params) || params_stride < 0)
        return CAUS_ERR_ARG;
    return ps_dispatch((hipStream_t)stream, nlenses, reinterpret_cast<const cd*>(w), N,
                       ps_rows(params, params_stride), 1, g_mag, mag, nullptr, kAllDirs, g_w,
                       g_params, status, itmax, mode, true);
}

extern "C" int64_t caus_lightcurve_workspace_bytes(int32_t nlenses, int64_t T, int64_t L) {
    if (nlenses < 1 || nlenses > 3 || T < 0 || L < 0) return -1;
    const int64_t per_block = (int64_t)kPsBlock * lc_epochs_per_lane(T, L);
    const int64_t nchunk = (T + per_block - 1) / per_block;
    return nchunk * L * (4 + np_for(nlenses)) * (int64_t)sizeof(double);
}

extern "C" int caus_lightcurve_point_source(void* stream, int32_t nlenses, const double* t,
                                            int64_t T, const double* lc_params, int64_t L,
                                            const double* g_mag, double* mag, double* g_params,
                                            double* workspace, int64_t workspace_bytes,
                                            uint8_t* status, int32_t itmax, int32_t mode) {
    if (T < 0 || L < 0 || itmax < 0 || nlenses < 1 || nlenses > 3 || check_mode(mode) != CAUS_OK)
        return CAUS_ERR_ARG;
    if (T == 0 || L == 0) return CAUS_OK;
    if (L > 65535 || !t || !lc_params || !mag) return CAUS_ERR_ARG;
    const bool vjp = g_mag != nullptr;
    if (vjp && (!g_params || !workspace ||
                workspace_bytes < caus_lightcurve_workspace_bytes(nlenses, T, L)))
        return CAUS_ERR_ARG;
    hipStream_t s = (hipStream_t)stream;
    const int rc = lc_dispatch(s, nlenses, t, T, ps_rows(lc_params, 4 + np_for(nlenses)), L, g_mag,
                               mag, nullptr, kAllDirs, workspace, status, itmax, mode, vjp);
    if (rc != CAUS_OK || !vjp) return rc;
    const int nq = 4 + np_for(nlenses);
    const int64_t per_block = (int64_t)kPsBlock * lc_epochs_per_lane(T, L);
    const int nchunk = (int)((T + per_block - 1) / per_block);
    const int64_t n = L * nq;
    hipLaunchKernelGGL(k_lightcurve_finalize, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                       workspace, g_params, L, nchunk, nq);
    return hipGetLastError() == hipSuccess ? CAUS_OK : CAUS_ERR_LAUNCH;
}

namespace {
// device address of `scratch` on the current device, looked up once per device (the
// host-side name of a __device__ array is not a device address)
double* lc_scratch_ptr() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
    static std::atomic<double*> cached[64];
    double* p = cached[dev].load(std::memory_order_acquire);
    if (!p) {
        void* q = nullptr;
        if (hipGetSymbolAddress(&q, HIP_SYMBOL(scratch)) != hipSuccess || !q) return nullptr;
        p = static_cast<double*>(q);
        cached[dev].store(p, std::memory_order_release);
    }
    return p;
}
}  // namespace

extern "C" int caus_lightcurve_point_source_noalloc(void* stream, int32_t nlenses,
                                                    const double* t, int64_t T,
                                                    const double* lc_params, int64_t L,
                                                    const double* g_mag, double* mag,
                                                    double* g_params, uint8_t* status,
                                                    int32_t itmax, int32_t mode) {
    if (nlenses < 1 || nlenses > 3 || T < 0 || L < 0) return CAUS_ERR_ARG;
    double* ws = nullptr;
    int64_t wsb = 0;
    if (g_mag && T > 0 && L > 0) {
        wsb = caus_lightcurve_workspace_bytes(nlenses, T, L);
        if (wsb < 0 || wsb > kLcScratchBytes) return CAUS_ERR_ARG;
        ws = lc_scratch_ptr();
        if (!ws) return CAUS_ERR_LAUNCH;
    }
    return caus_lightcurve_point_source(stream, nlenses, t, T, lc_params, L, g_mag, mag, g_params,
                                        ws, wsb, status, itmax, mode);
}
