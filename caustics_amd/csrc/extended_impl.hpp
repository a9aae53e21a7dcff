// Extended-source magnification by contour integration: one workgroup per source.
//
// Reference (fbartolic/caustics, src/caustics/):
//   limb sampling + 10 gap-bisection rounds .... extended_source.py:56-153
//   image continuation (greedy match_points) ... extended_source.py:34-53, utils.py:15-40
//   segments: closure test, split, ordering .... extended_source.py:156-309
//   stitching of open segments ................. extended_source.py:312-667
//   contours, magnification .................... extended_source.py:670-901
//   trapezoid / limb-darkened P,Q integrals .... integrate.py:18-121, utils.py:89-100
//
// Layout per source (workspace): limb angles, images (point-major: z[k*DEG + row]),
// per-point flag words (bit r: real image in row r; bit 16+r: det J < 0), all double
// buffered for the insertions of the refinement rounds, plus one 64-bit word per point
// for the image permutations and a P/Q scratch for limb darkening.
//
// Identity of images along the limb: every limb point is solved from the default
// initial estimates in parallel (one lane per point); image rows are then chained with
// the reference's greedy nearest-point assignment.  Where the nearest-neighbour map
// between consecutive points is a bijection the greedy result does not depend on the
// row order, so those steps compose as permutations; the rare steps where two images
// compete are resolved with the greedy rule on the actual carried rows (wave 0).
// Segments are kept as lists of pieces (row, first point, length, direction) instead
// of dense zero-padded arrays; stitching reproduces the reference's ordering rules.
#pragma once
#include "caustics_hip.h"
#include "chain.hpp"
#include "ps_impl.hpp"

namespace caus {

constexpr int kExtBlock = 256;    // block of the per-source integration kernel
constexpr int kExtWaveBlock = 64; // block of the per-source bookkeeping kernels (one wave)
constexpr int kExtMaxSeg = 32;     // >= 3 * (nlenses^2 + 1)
constexpr int kExtMaxPieces = 48;  // pieces of one stitched contour
constexpr int kExtSortMax = 4096;  // limb points per source (k_ext_select's register tiles)

template <int NL>
constexpr int ext_degree() {
    return NL == 1 ? 2 : NL * NL + 1;
}

__host__ __device__ inline int ext_npts_init(int npts) { return npts / 2; }
__host__ __device__ inline int ext_n_add(int npts) { return (npts / 2) / 10; }
__host__ __device__ inline int ext_mmax(int npts) { return ext_npts_init(npts) + 10 * ext_n_add(npts); }

__host__ __device__ inline size_t ext_align(size_t x) { return (x + 255) & ~size_t(255); }

// bytes of workspace per source
__host__ __device__ inline size_t ext_ws_bytes(int deg, int mmax) {
    size_t b = 0;
    b += ext_align(2 * (size_t)mmax * sizeof(double));            // theta x2
    b += ext_align(2 * (size_t)mmax * deg * sizeof(cd));          // z x2
    b += ext_align(2 * (size_t)mmax * sizeof(uint32_t));          // flags x2
    b += ext_align((size_t)(mmax + 1) * sizeof(uint64_t));        // permutations
    b += ext_align(2 * ((size_t)mmax * deg + 2) * sizeof(double)); // P, Q
    b += ext_align(2 * ((size_t)mmax * deg + 2) * sizeof(double)); // point cotangents
    b += ext_align(2 * ((size_t)mmax * deg + 2) * sizeof(double)); // centroid cotangent parts
    b += ext_align(2 * (size_t)mmax * sizeof(int32_t));             // limb order x2
    b += ext_align(2 * (size_t)mmax * sizeof(uint64_t));            // gap keys x2
    return b;
}

struct ExtWS {
    double* theta[2];
    cd* z[2];
    uint32_t* flg[2];
    uint64_t* perm;
    double* pq;
    double* xy;
    double* yz;
    int32_t* ord[2];   // refinement: limb order -> index of the point in append order
    uint64_t* gk[2];   // refinement: key of the gap after each point in limb order
};

__device__ inline ExtWS ext_ws(char* base, int deg, int mmax) {
    ExtWS w;
    size_t o = 0;
    w.theta[0] = (double*)(base + o);
    w.theta[1] = w.theta[0] + mmax;
    o += ext_align(2 * (size_t)mmax * sizeof(double));
    w.z[0] = (cd*)(base + o);
    w.z[1] = w.z[0] + (size_t)mmax * deg;
    o += ext_align(2 * (size_t)mmax * deg * sizeof(cd));
    w.flg[0] = (uint32_t*)(base + o);
    w.flg[1] = w.flg[0] + mmax;
    o += ext_align(2 * (size_t)mmax * sizeof(uint32_t));
    w.perm = (uint64_t*)(base + o);
    o += ext_align((size_t)(mmax + 1) * sizeof(uint64_t));
    w.pq = (double*)(base + o);
    o += ext_align(2 * ((size_t)mmax * deg + 2) * sizeof(double));
    w.xy = (double*)(base + o);
    o += ext_align(2 * ((size_t)mmax * deg + 2) * sizeof(double));
    w.yz = (double*)(base + o);
    o += ext_align(2 * ((size_t)mmax * deg + 2) * sizeof(double));
    w.ord[0] = (int32_t*)(base + o);
    w.ord[1] = w.ord[0] + mmax;
    o += ext_align(2 * (size_t)mmax * sizeof(int32_t));
    w.gk[0] = (uint64_t*)(base + o);
    w.gk[1] = w.gk[0] + mmax;
    return w;
}

// ---- permutations packed as 4-bit entries ------------------------------------
__device__ __forceinline__ int pget(uint64_t p, int i) { return (int)((p >> (4 * i)) & 0xF); }
// greedy match_points(a, b): for i in order, nearest unused b (ties -> lowest index)
template <int DEG>
__device__ __forceinline__ uint64_t greedy_match(const cd (&a)[DEG], const cd (&b)[DEG]) {
    unsigned used = 0;
    uint64_t p = 0;
#pragma unroll
    for (int i = 0; i < DEG; ++i) {
        double best = 0.0;
        int bj = -1;
#pragma unroll
        for (int j = 0; j < DEG; ++j) {
            const double d = norm2(b[j] - a[i]);
            if (!((used >> j) & 1u) && (bj < 0 || d < best)) {
                best = d;
                bj = j;
            }
        }
        used |= 1u << bj;
        p |= (uint64_t)bj << (4 * i);
    }
    return p;
}

// ---- limb sampling ------------------------------------------------------------
// Initial limb angle k of m (extended_source.py:101-103): numpy/jax linspace(-pi, pi,
// m, endpoint=False) is start + k * step with the product and the sum rounded
// separately, then pi - 1e-8 as the last angle; no FMA contraction, so the angles are
// the same doubles.
__device__ __forceinline__ double ext_limb_angle(int k, int m) {
#pragma clang fp contract(off)
    if (k == m) return 3.14159265358979323846 - 1e-8;
    const double step = (3.14159265358979323846 - -3.14159265358979323846) / (double)m;
    const double y = (double)k * step;
    return y + -3.14159265358979323846;
}
// Source-plane limb point w0 + rho e^{i th} (extended_source.py:79-98), each component a
// product then a sum as the reference's complex arithmetic rounds it.
__device__ __forceinline__ cd ext_limb_point(cd w0, double rho, double cs, double sn) {
#pragma clang fp contract(off)
    const double x = rho * cs, y = rho * sn;
    return cd{x + w0.re, y + w0.im};
}

// ---- point solve -----------------------------------------------------------
// warm = true: z holds initial roots (those of a nearby limb point).  The solve ends
// with the compensated polish, which takes converged roots to the doubles nearest the
// exact roots, so the result does not depend on where the iteration started and the
// rows are put in order afterwards by value (match_points).  first = true (limb point
// 0): the row order of this point seeds the continuation of every row along the limb
// (greedy matching resolves competing images in row order), so it is solved by the
// reference-compatible FP64 form from the reference's initial estimates
// (init_est.h:57-102, ehrlich_aberth.h:60-150), which puts the roots in the reference
// solver's order, in both precision forms.
template <int NL, int MODE>
__device__ __forceinline__ bool ext_solve_point(cd w, const LensFrame<NL>& lf,
                                                cd (&z)[ext_degree<NL>()], uint32_t& flags,
                                                int itmax, SolveStats* stats = nullptr,
                                                bool warm = false, bool first = false) {
    constexpr int DEG = ext_degree<NL>();
    bool ok = true;
    flags = 0;
    if constexpr (NL == 1) {
        const double sq = sqrt(1.0 + 4.0 * rcp(norm2(w)));
        z[0] = (0.5 * (1.0 + sq)) * w;
        z[1] = (0.5 * (1.0 - sq)) * w;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            flags |= 1u << j;
            // sign of det J; the reference's 1 - 1/|z|^2 has the same sign as 1 - 1/|z|^4
            if (norm2(z[j]) < 1.0) flags |= 1u << (16 + j);
        }
    } else {
        if (first)
            ok = solve_lens_refcompat<NL>(w, lf, z, itmax, stats);
        else
            ok = solve_lens<NL, MODE, true>(w, lf, z, itmax, warm, stats);
#pragma unroll
        for (int j = 0; j < DEG; ++j) {
            ImageTerms<NL> it = image_terms<NL>(z[j], lf);
            if (norm2(z[j] - it.G - w) < 1e-12) flags |= 1u << j;
            if (1.0 - norm2(it.K) < 0.0) flags |= 1u << (16 + j);
        }
    }
    return ok;
}

template <int DEG>
__device__ __forceinline__ void load_pt(const cd* zb, int k, cd (&z)[DEG]) {
#pragma unroll
    for (int r = 0; r < DEG; ++r) z[r] = zb[(size_t)k * DEG + r];
}
template <int DEG>
__device__ __forceinline__ void store_pt(cd* zb, int k, const cd (&z)[DEG]) {
#pragma unroll
    for (int r = 0; r < DEG; ++r) zb[(size_t)k * DEG + r] = z[r];
}
template <int DEG>
__device__ __forceinline__ uint32_t permute_flags(uint32_t f, uint64_t p) {
    uint32_t o = 0;
#pragma unroll
    for (int i = 0; i < DEG; ++i) {
        const int s = pget(p, i);
        o |= ((f >> s) & 1u) << i;
        o |= ((f >> (16 + s)) & 1u) << (16 + i);
    }
    return o;
}
__device__ inline double block_sum(double v, double* sh) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    v = wave_sum(v);
    if (lane == 0) sh[wv] = v;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < kExtBlock / 64; ++q) s += sh[q];
    __syncthreads();
    return s;
}

// ---- segments and contours ---------------------------------------------------
struct Seg {
    int row, start, len;  // points start..start+len-1 of image row `row`
    int par;              // parity of the segment (+1/-1)
    int empty;
    double length;        // sum of |z_{k+1} - z_k|
    cd head, tail;        // first and last point (0 for an empty segment)
};
struct Piece {
    int row, start, len, rev;
};

// Final limb points in limb order, row after row (image `row` of point k at row * ld + k):
// the continuation's last gather writes them so, and everything after it reads along rows.
struct ZRows {
    const cd* z;
    int ld;
};
template <int DEG>
__device__ __forceinline__ cd pt(ZRows zb, int k, int row) {
    return zb.z[(size_t)row * zb.ld + k];
}
// point k of a piece list
template <int DEG>
__device__ inline cd contour_point(ZRows zb, const Piece* pc, int np, int k) {
    for (int i = 0; i < np; ++i) {
        if (k < pc[i].len) {
            const int idx = pc[i].rev ? pc[i].start + pc[i].len - 1 - k : pc[i].start + k;
            return pt<DEG>(zb, idx, pc[i].row);
        }
        k -= pc[i].len;
    }
    return cd{0.0, 0.0};
}

}  // namespace caus

namespace caus {

// Node i of the n-point Gauss-Legendre rule on [-1,1] by Newton iteration on P_n; xw holds
// (node, weight) in ascending order
__device__ inline void gauss_legendre(int n, int i, double2* xw) {
    // root i counted from x = +1 downwards, stored ascending
    double z = cos(3.14159265358979323846 * (i + 0.75) / (n + 0.5));
    double pp = 1.0;
    for (int it = 0; it < 100; ++it) {
        double p1 = 1.0, p2 = 0.0;
        for (int j = 1; j <= n; ++j) {
            const double p3 = p2;
            p2 = p1;
            p1 = ((2.0 * j - 1.0) * z * p2 - (j - 1.0) * p3) / j;
        }
        pp = n * (z * p1 - p2) / (z * z - 1.0);
        const double dz = p1 / pp;
        z -= dz;
        if (fabs(dz) < 1e-16) break;
    }
    double p1 = 1.0, p2 = 0.0;
    for (int j = 1; j <= n; ++j) {
        const double p3 = p2;
        p2 = p1;
        p1 = ((2.0 * j - 1.0) * z * p2 - (j - 1.0) * p3) / j;
    }
    pp = n * (z * p1 - p2) / (z * z - 1.0);
    xw[n - 1 - i] = make_double2(z, 2.0 / ((1.0 - z * z) * pp * pp));
}

// s = sqrt(x) and h ~ 1/(2 sqrt x) for x > 0 in the normal range (x >= 2^-767): the
// v_rsq_f64 seed, one coupled Newton step, a residual correction of s, one more step on h.
__device__ __forceinline__ void sqrt_half_rsq(double x, double& s, double& h) {
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y;
    h = 0.5 * y;
    const double e = fma(-h, g, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    s = fma(fma(-g, g, x), h, g);
    h = fma(h, fma(-h, s, 0.5), h);
}

// wave-uniform value into scalar registers (every lane holds the same value)
__device__ __forceinline__ double uniform(double x) {
    const uint64_t b = (uint64_t)__double_as_longlong(x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// What a source's limb-darkened line integrals share, the same for every lane of the
// workgroup: lens frame (lenses 1 and 2 on the real axis, lens_frame), source and profile.
template <int NL>
struct LDSource {
    double e[NL];
    cd r[NL];
    cd w0;
    double rho, rho2x, irho, irho2, u1, c3;   // rho2x = 2 rho (infinite: see ld_source)
};
template <int NL>
__device__ __forceinline__ LDSource<NL> ld_source(const LensFrame<NL>& lf, cd w0, double rho,
                                                  double u1) {
    LDSource<NL> q;
#pragma unroll
    for (int j = 0; j < NL; ++j) {
        q.e[j] = uniform(lf.e[j]);
        q.r[j] = cd{uniform(lf.r[j].re), uniform(lf.r[j].im)};
    }
    q.w0 = cd{uniform(w0.re), uniform(w0.im)};
    q.rho = uniform(rho);
    q.irho = uniform(rcp(rho));
    // r = |D| / rho of a negative radius is never above 1: the profile's outer branch is off
    q.rho2x = uniform(rho < 0.0 ? INFINITY : 2.0 * rho);
    q.irho2 = uniform(q.irho * q.irho);
    q.u1 = uniform(u1);
    q.c3 = uniform(3.0 / (3.0 - u1));
    return q;
}

// One node of a line integral at z (integrate.py:29-44): r = |lens_eq(z) - w0| / rho,
// B = c3 (u1 B_r + 1 - 2 u1), c3 = 3/(3-u1), B_r = 1 + t with t = sqrt(1 - r^2) inside the
// disk (r <= 1) and t = -sqrt(1 - 1/r^2) outside.  Returned: v_j = 1/(conj z - conj r_j),
// D = lens_eq(z) - w0, n2 = |D|^2, t and p, with dB_r/dD = -(2/rho^2) p D.
// q = min(r, 1/r) serves both sides, |t| = sqrt(1 - q^2), and the derivative
//   -(dB_r/d|D|) / |D| = min(1, 1/r^2)^2 / (rho^2 |t|)
// needs no division by |D|.  Near the limb t keeps only the rounding of r and 1/r, so these
// are one multiplication each.  Contraction is off so that the forward-only and the
// forward+VJP kernels round alike.
template <int NL>
__device__ __forceinline__ void ld_node(cd z, const LDSource<NL>& q, cd (&v)[NL], cd& D,
                                        double& n2, double& t, double& p) {
#pragma clang fp contract(off)
    // v_j: the squared moduli share one reciprocal of their product
    double dx[NL], dy[NL], n[NL], sj[NL];
    const double yy = z.im * z.im;
#pragma unroll
    for (int j = 0; j < NL; ++j) {
        dx[j] = z.re - q.r[j].re;
        dy[j] = j < 2 ? z.im : z.im - q.r[j].im;
        n[j] = fma(dx[j], dx[j], j < 2 ? yy : dy[j] * dy[j]);
    }
    if constexpr (NL == 1) {
        sj[0] = rcp(n[0]);
    } else if constexpr (NL == 2) {
        const double rP = rcp(n[0] * n[1]);
        sj[0] = n[1] * rP;
        sj[1] = n[0] * rP;
    } else {
        const double n01 = n[0] * n[1];
        const double rP = rcp(n01 * n[2]);
        const double u = n[2] * rP;
        sj[0] = n[1] * u;
        sj[1] = n[0] * u;
        sj[2] = n01 * rP;
    }
#pragma unroll
    for (int j = 0; j < NL; ++j) v[j] = cd{dx[j] * sj[j], dy[j] * sj[j]};
    cd G = q.e[0] * v[0];
#pragma unroll
    for (int j = 1; j < NL; ++j) G = cd{fma(q.e[j], v[j].re, G.re), fma(q.e[j], v[j].im, G.im)};
    D = z - G - q.w0;
    n2 = norm2(D);
    double aD, hD;
    sqrt_half_rsq(fmax(n2, 0x1p-700), aD, hD);
    const double r = aD * q.irho, ir = q.rho2x * hD;
    const double k = fmin(r, ir);
    const double x = 1.0 - k * k;
    double s, h;
    sqrt_half_rsq(fmax(x, 0x1p-200), s, h);
    h = x > 0.0 ? h : 0.0;
    t = copysign(s, 1.0 - r);
    const double m = fmin(ir, 1.0), m2 = m * m;
    p = (h * m2) * m2;
}

// one trapezoid term of the limb-darkened contour integral (integrate.py:118-121),
// written with explicit fma so that both kernels that form it round it alike
__device__ __forceinline__ double ld_trapezoid(double Pk, double Pn, double Qk, double Qn, cd a,
                                               cd b, double acc) {
    return fma(0.5 * (Pk + Pn), b.re - a.re, fma(0.5 * (Qk + Qn), b.im - a.im, acc));
}

// Gauss-Legendre nodes and weights (x, w) of the two parts of a line
struct GLNodes {
    const double2 *a, *b;
    int n1, n2;
};

// sum_i w_i B_i of one part of a line from St = sum_i w_i t_i (the weights sum to 2)
template <int NL>
__device__ __forceinline__ double ld_sum(double St, int n, const LDSource<NL>& q) {
    return q.c3 * fma(q.u1, St, n > 0 ? fma(-2.0, q.u1, 2.0) : 0.0);
}

// split point of a line (integrate.py:50-66); explicit fma, both kernels round it alike
__device__ __forceinline__ double ld_split(double a, double b, double rho) {
    const double d = fabs(b - a);
    const double sp = (b > a) ? fma(-2.0, rho, b) : fma(2.0, rho, b);
    return 0.5 * d <= 2.0 * rho ? fma(0.5, d, a) : sp;
}

// -0.5 * int_{a}^{b} B(x + i y) dy  (P) or 0.5 * int_{a}^{b} B(x + i y) dx (Q), split at
// the reference's point (integrate.py:50-107)
template <int NL, bool ISP>
__device__ __forceinline__ double ld_line(double fixed, double a, double b,
                                          const LDSource<NL>& q, const GLNodes& g) {
    const double sp = ld_split(a, b, q.rho);
    double I = 0.0;
#pragma unroll 1
    for (int part = 0; part < 2; ++part) {
        const double lo = part == 0 ? a : sp, hi = part == 0 ? sp : b;
        const double2* xw = part == 0 ? g.a : g.b;
        const int n = part == 0 ? g.n1 : g.n2;
        const double h = 0.5 * (hi - lo), c = 0.5 * (hi + lo);
        double St = 0.0;
#pragma unroll 2
        for (int i = 0; i < n; ++i) {
            const double2 k = xw[i];
            const double y = fma(h, k.x, c);
            cd v[NL], D;
            double n2, t, p;
            ld_node<NL>(ISP ? cd{fixed, y} : cd{y, fixed}, q, v, D, n2, t, p);
            St = fma(k.y, t, St);
        }
        I = fma(h, ld_sum<NL>(St, n, q), I);
    }
    return ISP ? -0.5 * I : 0.5 * I;
}

// Uniform-source contour integral over points c_0..c_{L-1} (pieces), closed back to
// c_0: nterms trapezoid terms of (x dy - y dx)/2 (L, or L-1 for the single-lens quirk).
template <int NL, int DEG>
__device__ double integrate_contour(ZRows zb, const Piece* pc, int np, int L, int nterms,
                                    double* shd) {
    const int tid = threadIdx.x;
    double acc = 0.0;
    if (L <= 0) return block_sum(0.0, shd);
    for (int k = tid; k < nterms; k += kExtBlock) {
        const cd a = contour_point<DEG>(zb, pc, np, k);
        const cd b = contour_point<DEG>(zb, pc, np, (k + 1 == L) ? 0 : k + 1);
        acc += 0.5 * (0.5 * a.re + 0.5 * b.re) * (b.im - a.im) +
               0.5 * (-0.5 * a.im - 0.5 * b.im) * (b.re - a.re);
    }
    return block_sum(acc, shd);
}

// ---- stitching (extended_source.py:312-667), wave-uniform code on wave 0 ---------
struct ActSeg {
    Piece pc[kExtMaxPieces];
    int np, t, par, empty;
};

template <int DEG>
__device__ inline cd seg_point(ZRows zb, const Seg& s, int k) {
    if (s.empty || k < 0 || k >= s.len) return cd{0.0, 0.0};
    return pt<DEG>(zb, s.start + k, s.row);
}
// line ending at the head / tail (second element is the connection point).
// Dense-array semantics: points beyond the segment are zero, dynamic_slice clamps.
template <class F>
__device__ inline void head_line(F get, int t, cd& l0, cd& l1) {
    const cd x0 = get(0), x1 = get(1), x2 = get(2);
    const bool c = (norm2(x1 - x0) > 1e-10) || (t <= 1);
    if (c) {
        l0 = x1;
        l1 = x0;
    } else {
        l0 = x2;
        l1 = x1;
    }
}
template <class F>
__device__ inline void tail_line(F get, int t, int dense_len, cd& l0, cd& l1) {
    const bool c = (t <= 1) || (norm2(get(t) - get(t - 1)) > 1e-10);
    int s = c ? t - 1 : t - 2;
    s = s < 0 ? 0 : (s > dense_len - 2 ? dense_len - 2 : s);
    l0 = get(s);
    l1 = get(s + 1);
}

__device__ inline bool geom_condition(cd a0, cd a1, cd b0, cd b1) {
    const double dist = sqrt(norm2(a1 - b1));
    const bool c1 = dist < 1e-1;
    const cd v1 = a1 - a0, v2 = b1 - b0;
    const double n1 = sqrt(norm2(v1)), n2 = sqrt(norm2(v2));
    const double cosang = (v1.re / n1) * (v2.re / n2) + (v1.im / n1) * (v2.im / n2);
    const double alpha = acos(cosang);  // NaN outside [-1,1] or for a zero vector
    const bool c2 = (180.0 - alpha * (180.0 / 3.14159265358979323846)) < 60.0;
    const bool c3 = sqrt(norm2(a1 - b1)) < sqrt(norm2(a0 - b0));
    return (c1 && c2 && c3) || dist < 1e-5;
}

}  // namespace caus

// ============================================================================
// Reverse mode of the contour pipeline.  Directions (user order):
//   0 Re w0, 1 Im w0, 2 rho, 3 u1, 4.. lens parameters (s, q[, q3, r3, psi]).
// Discrete choices (limb angles, rows, segment structure) are piecewise constant;
// every contour point is the image z of a fixed limb angle, differentiated
// implicitly through the lens equation, and the Gauss-Legendre line integrals are
// differentiated exactly as discretised (moving end points and split point included).
// ============================================================================
namespace caus {

template <int NL>
constexpr int ext_nd() {
    return 4 + (NL == 1 ? 0 : n_user_params<NL>());
}

template <int NL>
struct ExtTangents {
    static constexpr int ND = ext_nd<NL>();
    cd dw0[ND];              // tangent of the lens-frame source centre
    LensTangent<NL> lt[ND];  // tangent of the lens frame
    double drho[ND], du1[ND];
};

template <int NL>
__device__ inline void ext_tangents(const double* prm, ExtTangents<NL>& T) {
    constexpr int ND = ext_nd<NL>();
#pragma unroll
    for (int d = 0; d < ND; ++d) {
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            T.lt[d].de[j] = 0.0;
            T.lt[d].dr[j] = cd{0.0, 0.0};
        }
        T.lt[d].dxcm = 0.0;
        T.dw0[d] = cd{0.0, 0.0};
        T.drho[d] = 0.0;
        T.du1[d] = 0.0;
    }
    T.dw0[0] = cd{1.0, 0.0};
    T.dw0[1] = cd{0.0, 1.0};
    T.drho[2] = 1.0;
    T.du1[3] = 1.0;
    if constexpr (NL > 1) {
        LensTangent<NL> up[n_user_params<NL>()];
        lens_frame_tangents<NL>(prm, up);
#pragma unroll
        for (int k = 0; k < n_user_params<NL>(); ++k) {
            T.lt[4 + k] = up[k];
            T.dw0[4 + k] = cd{up[k].dxcm, 0.0};
        }
    }
}

// point k of a piece list: value, limb index and row
template <int DEG>
__device__ inline cd contour_locate(ZRows zb, const Piece* pc, int np, int k, int& idx,
                                    int& row) {
    for (int i = 0; i < np; ++i) {
        if (k < pc[i].len) {
            idx = pc[i].rev ? pc[i].start + pc[i].len - 1 - k : pc[i].start + k;
            row = pc[i].row;
            return pt<DEG>(zb, idx, row);
        }
        k -= pc[i].len;
    }
    idx = 0;
    row = 0;
    return cd{0.0, 0.0};
}

// Reverse-mode accumulators of the direct (not through the contour points) dependence
// of the limb-darkened line integrals on the lens frame, the source centre, rho and u1.
// A direction with tangents (de_j, dr_j, dw0, drho, du1) receives
//   sum_j de_j ge_j + e_j Re(gr_j conj(dr_j)) + Re(gw conj(dw0)) + grho drho + gu1 du1
// (the mass e_j of the dr_j term is applied once, in along), so that each
// Gauss-Legendre node costs O(NL) instead of O(NL x directions).
template <int NL>
struct LDAdj {
    double ge[NL];
    cd gr[NL];
    cd gw;
    double grho, gu1;
    __device__ void zero() {
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            ge[j] = 0.0;
            gr[j] = cd{0.0, 0.0};
        }
        gw = cd{0.0, 0.0};
        grho = gu1 = 0.0;
    }
    __device__ void axpy(double s, const LDAdj& o) {
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            ge[j] += s * o.ge[j];
            gr[j] = gr[j] + s * o.gr[j];
        }
        gw = gw + s * o.gw;
        grho += s * o.grho;
        gu1 += s * o.gu1;
    }
    __device__ double along(const LensTangent<NL>& lt, const double (&e)[NL], cd dw0, double drho,
                            double du1) const {
        double v = grho * drho + gu1 * du1 + gw.re * dw0.re + gw.im * dw0.im;
#pragma unroll
        for (int j = 0; j < NL; ++j)
            v += lt.de[j] * ge[j] + e[j] * (gr[j].re * lt.dr[j].re + gr[j].im * lt.dr[j].im);
        return v;
    }
};

// P (ISP) or Q line integral with its partial derivatives along the fixed coordinate,
// the lower limit a and the upper limit b; wA * (direct parameter derivative) goes to A.
// With D = lens_eq(z) - w0 and p as ld_node gives it, dB = c3 u1 dB_r has the node terms
//   dD = -(dG + dw0), dG = sum_j de_j v_j + e_j v_j^2 conj(dr_j);  dD/dx = 1 + K,
//   dD/dy = i (1 - K), K = sum_j e_j v_j^2,
// so that with u = w_i p D every derivative is a linear function of the part's sums of
//   u, Re(conj(u) v_j), conj(u) v_j^2, w_i p |D|^2 and x_i (dB along the line):
// the derivatives along and across the line at weight w_i are Im / Re (u + conj(u) K)
// = components of sum u + sum_j e_j conj(sum conj(u) v_j^2).  The node loop therefore holds
// only these sums; the profile's constants and the line's scale are applied once a part.
// Bound: FP64 issue.  Per node of two lenses 87 FP64 operations and 3 quarter-rate seeds;
// with every derivative formed node by node it was 124 and 3.  Integration of 4,096 binary
// sources of 256-4096 limb points (3.2e9 nodes): 17.0 -> 11.8-12.2 ms, of 12,000 triple-lens
// sources (2.0e9 nodes): 17.8 -> 10.8 ms (of which 0.5 ms the Gauss-Legendre nodes).
template <int NL, bool ISP>
__device__ __forceinline__ double ld_line_adj(double fixed, double a, double b,
                                              const LDSource<NL>& q, const GLNodes& g, double wA,
                                              double& dfix, double& da, double& db,
                                              LDAdj<NL>& A) {
    const double d = fabs(b - a);
    const double sc = ISP ? -0.5 : 0.5;
    const double sp = ld_split(a, b, q.rho);
    double dsp_da, dsp_db, dsp_drho;
    if (0.5 * d <= 2.0 * q.rho) {
        const double sg = (b - a) > 0 ? 1.0 : ((b - a) < 0 ? -1.0 : 0.0);
        dsp_da = 1.0 - 0.5 * sg;
        dsp_db = 0.5 * sg;
        dsp_drho = 0.0;
    } else {
        dsp_da = 0.0;
        dsp_db = 1.0;
        dsp_drho = (b > a) ? -2.0 : 2.0;
    }
    const double kap = -2.0 * q.c3 * q.u1 * q.irho2;   // dB/dD = kap p D
    // B = c3 (u1 (1 + t) + 1 - 2 u1), c3' = c3^2/3: dB/du1 = bu0 + bu1 t
    const double dc3 = q.c3 * q.c3 / 3.0;
    const double bu0 = dc3 * (1.0 - q.u1) - q.c3, bu1 = dc3 * q.u1 + q.c3;
    double I = 0.0, dsp = 0.0;
    da = db = dfix = 0.0;
#pragma unroll 1
    for (int part = 0; part < 2; ++part) {
        const double lo = part == 0 ? a : sp, hi = part == 0 ? sp : b;
        const double2* xw = part == 0 ? g.a : g.b;
        const int n = part == 0 ? g.n1 : g.n2;
        const double h = 0.5 * (hi - lo), c = 0.5 * (hi + lo);
        double St = 0.0, S2 = 0.0, sq = 0.0, ge[NL];
        cd su = cd{0.0, 0.0}, gr[NL];
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            ge[j] = 0.0;
            gr[j] = cd{0.0, 0.0};
        }
#pragma unroll 1
        for (int i = 0; i < n; ++i) {
            const double2 k = xw[i];
            const double y = fma(h, k.x, c);
            cd v[NL], D;
            double n2, t, p;
            ld_node<NL>(ISP ? cd{fixed, y} : cd{y, fixed}, q, v, D, n2, t, p);
            St = fma(k.y, t, St);
            const double pw = k.y * p;
            sq = fma(pw, n2, sq);
            const cd u = pw * D;
            su = su + u;
            double along = ISP ? u.im : u.re;   // dB along the line
#pragma unroll
            for (int j = 0; j < NL; ++j) {
                const cd s = cd{fma(u.re, v[j].re, u.im * v[j].im),
                                fma(u.re, v[j].im, -(u.im * v[j].re))};   // conj(u) v
                ge[j] += s.re;
                if (ISP) {
                    const double im = fma(s.re, v[j].im, s.im * v[j].re);
                    gr[j].re = fma(s.re, v[j].re, fma(-s.im, v[j].im, gr[j].re));
                    gr[j].im += im;
                    along = fma(q.e[j], im, along);
                } else {
                    const double re = fma(s.re, v[j].re, -(s.im * v[j].im));
                    gr[j].re += re;
                    gr[j].im = fma(s.re, v[j].im, fma(s.im, v[j].re, gr[j].im));
                    along = fma(q.e[j], re, along);
                }
            }
            S2 = fma(k.x, along, S2);
        }
        cd sK = cd{0.0, 0.0};
#pragma unroll
        for (int j = 0; j < NL; ++j) sK = sK + q.e[j] * gr[j];
        const double S0 = ld_sum<NL>(St, n, q);
        const double Sx = kap * (su.re + sK.re), Sy = kap * (su.im + sK.im);
        const double S1 = ISP ? Sy : Sx, S3 = ISP ? Sx : Sy;   // along / across the line
        S2 *= kap;
        I = fma(h, S0, I);
        // d/dlo of h sum w B(c + h x) with dh/dlo = -1/2, dc/dlo = 1/2, and d/dhi
        const double dlo = fma(0.5 * h, S1 - S2, -0.5 * S0);
        const double dhi = fma(0.5 * h, S1 + S2, 0.5 * S0);
        if (part == 0) {
            da += dlo;
            dsp += dhi;
        } else {
            dsp += dlo;
            db += dhi;
        }
        dfix = fma(h, S3, dfix);
        const double cw = wA * sc * h, ck = cw * kap;
        A.gw = A.gw - ck * su;
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            A.ge[j] -= ck * ge[j];
            A.gr[j] = A.gr[j] - ck * gr[j];
        }
        A.grho -= ck * q.irho * sq;
        A.gu1 += cw * (n > 0 ? fma(bu1, St, 2.0 * bu0) : 0.0);
    }
    da += dsp * dsp_da;
    db += dsp * dsp_db;
    A.grho += wA * sc * dsp * dsp_drho;
    dfix *= sc;
    da *= sc;
    db *= sc;
    return sc * I;
}

// Adjoint of one contour integral: accumulates scale * dI/dtheta into g[ND] (per thread).
// pq holds P, Q of the contour points (limb darkening; written by the forward pass).
// Adjoint of the image z of limb angle th for the cotangent zbar = (bx, by) of z:
// dz = (u - K conj u)/det with u = dw0 + drho e^{i th} + sum_j de_j v_j + e_j v_j^2 conj(dr_j)
// gives zbar . dz = Re(c u), c = (conj(zbar) - zbar conj(K))/det, added to A.
template <int NL>
__device__ inline void image_adjoint(cd z, double th, const LensFrame<NL>& lf, double bx,
                                     double by, LDAdj<NL>& A) {
    const ImageTerms<NL> it = image_terms<NL>(z, lf);
    const double idet = rcp(1.0 - norm2(it.K));
    const cd zbar = cd{bx, by};
    const cd c = idet * (conj(zbar) - zbar * conj(it.K));
    double sn, cs;
    sincos(th, &sn, &cs);
    A.gw = A.gw + conj(c);
    A.grho += c.re * cs - c.im * sn;
#pragma unroll
    for (int j = 0; j < NL; ++j) {
        const cd v = it.inv[j];
        const cd cv = c * v;
        A.ge[j] += cv.re;
        A.gr[j] = A.gr[j] + cv * v;
    }
}

// Adjoint of one uniform-source contour integral: adds scale * dI/d(frame, w0, rho) to
// adj (per thread).  Each point's cotangent, from the two trapezoid terms it enters, is
// pushed through the image tangents.
template <int NL, int DEG>
__device__ void contour_adjoint(ZRows zb, const double* theta, const Piece* pc, int np, int L,
                                int nterms, const LensFrame<NL>& lf, double scale,
                                LDAdj<NL>& adj) {
    const int tid = threadIdx.x;
    for (int k = tid; k < L; k += kExtBlock) {
        int idx, row;
        const cd zk = contour_locate<DEG>(zb, pc, np, k, idx, row);
        const int kn = (k + 1 == L) ? 0 : k + 1;
        const int kp = (k == 0) ? L - 1 : k - 1;
        const cd zn = contour_point<DEG>(zb, pc, np, kn);
        const cd zp = contour_point<DEG>(zb, pc, np, kp);
        double xbar = 0.0, ybar = 0.0;
        if (k < nterms) {
            xbar += 0.5 * zn.im;
            ybar -= 0.5 * zn.re;
        }
        if (kp < nterms) {
            xbar -= 0.5 * zp.im;
            ybar += 0.5 * zp.re;
        }
        image_adjoint<NL>(zk, theta[idx], lf, scale * xbar, scale * ybar, adj);
    }
}

// One contour of a source as the integrals see it: its pieces, L points, nterms
// trapezoid terms, the divisor of its centroid sum, its parity, the offset of its
// points in the source's flat point list and (limb darkening) its centroid.
struct ExtCEntry {
    const Piece* pc;
    int np, L, nterms, off;
    double cdiv, par, zx, zy;
};
constexpr int kExtMaxContours = 16;  // >= nlenses^2 + 1 closed rows + 3 stitched contours

// Limb-darkened integrals of all nc contours of a source (integrate.py:47-121), their
// parity-weighted sum, and with VJP the reverse mode (adds to adj).  The P and Q line
// integrals of every point -- 2 npts_ld brightness evaluations per point, nearly all of
// the work -- run as one flat loop over the source's 2 T lines (all P lines, then all Q
// lines, so that all but one wave run one kind), and the workgroup idles only in its last
// iteration; the centroids before it and the trapezoid sums and the point adjoints after it
// run contour by contour.  The forward and forward+VJP kernels form P and Q alike (ld_line /
// ld_line_adj), so they return the same integral.
// pq, xy, xq, yz hold 2 T doubles each: P and Q, the points' cotangents from the P and from
// the Q lines, and the parts of the centroid's cotangent (Pbar dP/dy0, Qbar dQ/dx0).
// A workgroup takes every parts-th run of 256 neighbouring lines, from run `part` on, and with
// parts = 1 the sums after them; SUMS: only those sums, the lines being done.  Without the
// reverse mode P and Q do not depend on who forms them; its sums over a source's lines would, so
// there parts is 1.
template <int NL, int DEG, bool VJP, bool SUMS>
__device__ double integrate_source_ld(ZRows zb, const double* theta, ExtCEntry* ct, int nc,
                                      int T, double* pq, double* xy, double* xq, double* yz,
                                      const LensFrame<NL>& lf, const LDSource<NL>& q,
                                      const GLNodes& gl, LDAdj<NL>& adj, double* shd, int part,
                                      int parts) {
    const int tid = threadIdx.x;
    if constexpr (!SUMS) {
        // centroids (integrate.py:112); the closing point repeats c_0 in the sum
        for (int c = 0; c < nc; ++c) {
            const ExtCEntry& e = ct[c];
            double sx = 0.0, sy = 0.0;
            for (int k = tid; k < e.L; k += kExtBlock) {
                const cd a = contour_point<DEG>(zb, e.pc, e.np, k);
                sx += a.re;
                sy += a.im;
            }
            const cd c0 = (e.L > 0) ? contour_point<DEG>(zb, e.pc, e.np, 0) : cd{0.0, 0.0};
            const double zx = (block_sum(sx, shd) + c0.re) / e.cdiv;
            const double zy = (block_sum(sy, shd) + c0.im) / e.cdiv;
            if (tid == 0) {
                ct[c].zx = zx;
                ct[c].zy = zy;
            }
        }
        __syncthreads();
        // the P lines of every point, then the Q lines, flat over the contours
        for (int u = tid + part * kExtBlock; u < 2 * T; u += parts * kExtBlock) {
            const bool isP = u < T;
            const int gi = isP ? u : u - T;
            int c = 0;
            while (c + 1 < nc && gi >= ct[c + 1].off) ++c;
            const ExtCEntry& e = ct[c];
            const int k = gi - e.off;
            const cd zk = contour_point<DEG>(zb, e.pc, e.np, k);
            if constexpr (!VJP) {
                if (isP)
                    pq[2 * gi] = ld_line<NL, true>(zk.re, e.zy, zk.im, q, gl);
                else
                    pq[2 * gi + 1] = ld_line<NL, false>(zk.im, e.zx, zk.re, q, gl);
            } else {
                const int L = e.L;
                const int kn = (k + 1 == L) ? 0 : k + 1;
                const int kp = (k == 0) ? L - 1 : k - 1;
                const cd zn = contour_point<DEG>(zb, e.pc, e.np, kn);
                const cd zp = contour_point<DEG>(zb, e.pc, e.np, kp);
                // cotangent of P_k or Q_k from the two trapezoid terms it enters; P_k =
                // P(x_k; y0 .. y_k), Q_k = Q(y_k; x0 .. x_k), (x0, y0) the centroid
                double bar = 0.0, df, da, db;
                if (isP) {
                    if (k < e.nterms) bar += 0.5 * (zn.re - zk.re);
                    if (kp < e.nterms) bar += 0.5 * (zk.re - zp.re);
                    pq[2 * gi] = ld_line_adj<NL, true>(zk.re, e.zy, zk.im, q, gl, e.par * bar, df,
                                                       da, db, adj);
                    xy[2 * gi] = bar * df;
                    xy[2 * gi + 1] = bar * db;
                    yz[2 * gi] = bar * da;
                } else {
                    if (k < e.nterms) bar += 0.5 * (zn.im - zk.im);
                    if (kp < e.nterms) bar += 0.5 * (zk.im - zp.im);
                    pq[2 * gi + 1] = ld_line_adj<NL, false>(zk.im, e.zx, zk.re, q, gl, e.par * bar,
                                                            df, da, db, adj);
                    xq[2 * gi] = bar * db;
                    xq[2 * gi + 1] = bar * df;
                    yz[2 * gi + 1] = bar * da;
                }
            }
        }
        if (!VJP && parts > 1) return 0.0;
        __syncthreads();
    }
    double total = 0.0;
    for (int c = 0; c < nc; ++c) {
        const ExtCEntry& e = ct[c];
        const int L = e.L;
        const double* I = pq + 2 * e.off;
        double* v = xy + 2 * e.off;
        const double* vq = xq + 2 * e.off;
        const double* y = yz + 2 * e.off;
        double acc = 0.0, x0bar = 0.0, y0bar = 0.0;
        for (int k = tid; k < L; k += kExtBlock) {
            const int kn = (k + 1 == L) ? 0 : k + 1;
            if (k < e.nterms) {
                const cd a = contour_point<DEG>(zb, e.pc, e.np, k);
                const cd b = contour_point<DEG>(zb, e.pc, e.np, kn);
                acc = ld_trapezoid(I[2 * k], I[2 * kn], I[2 * k + 1], I[2 * kn + 1], a, b, acc);
            }
            if constexpr (VJP) {
                const int kp = (k == 0) ? L - 1 : k - 1;
                double xbar = v[2 * k] + vq[2 * k], ybar = v[2 * k + 1] + vq[2 * k + 1];
                if (k < e.nterms) {
                    xbar -= 0.5 * (I[2 * k] + I[2 * kn]);
                    ybar -= 0.5 * (I[2 * k + 1] + I[2 * kn + 1]);
                }
                if (kp < e.nterms) {
                    xbar += 0.5 * (I[2 * kp] + I[2 * k]);
                    ybar += 0.5 * (I[2 * kp + 1] + I[2 * k + 1]);
                }
                v[2 * k] = xbar;
                v[2 * k + 1] = ybar;
                y0bar += y[2 * k];
                x0bar += y[2 * k + 1];
            }
        }
        total += e.par * block_sum(acc, shd);
        if constexpr (VJP) {
            const double X0 = block_sum(x0bar, shd) / e.cdiv;
            const double Y0 = block_sum(y0bar, shd) / e.cdiv;
            // each thread reads back only the cotangents it wrote above
            for (int k = tid; k < L; k += kExtBlock) {
                int idx, row;
                const cd zk = contour_locate<DEG>(zb, e.pc, e.np, k, idx, row);
                const double wgt = (k == 0) ? 2.0 : 1.0;  // c_0 enters the centroid twice
                image_adjoint<NL>(zk, theta[idx], lf, e.par * (v[2 * k] + wgt * X0),
                                  e.par * (v[2 * k + 1] + wgt * Y0), adj);
            }
        }
    }
    return total;
}

}  // namespace caus

// ============================================================================
// Batch pipeline.  The contours of a batch of sources are computed by a fixed
// sequence of launches over the whole batch, so that the root solves (nearly all of
// the arithmetic) run one limb point per lane at the solver's occupancy:
//   k_ext_limb_init   1-2 + flat   effective npts, prefix offsets of the flat work lists;
//                                  Gauss-Legendre nodes; limb point 0 of every source
//   k_ext_limb_init   flat         the other initial limb angles, kExtPer consecutive ones
//                                  per lane
//   k_ext_chain       per source   image continuation (extended_source.py:34-53), limb
//                                  order and gap keys of the initial points
//   10 x k_ext_select per source   largest gaps, insertion shifts, next limb order, tasks
//        k_ext_solve_add flat      new points appended, matched to their left neighbour,
//                                  keys of their two gaps
//   (small batches: k_ext_init_grouped for the second launch, k_ext_refine for all rounds)
//   k_ext_chain       per source   points gathered in limb order, image continuation
//   k_ext_contours    per source   closure test, segments, stitching -> piece lists
//   k_ext_integrate   per source   contour integrals, magnification, reverse mode
// No launch allocates, synchronises with the host or clears memory with a memset, so
// the sequence can be captured in a HIP graph.
// ============================================================================
namespace caus {

// waves per SIMD that the register allocation of the reverse-mode integrate kernel
// targets (its per-thread adjoint state is large)
#ifndef CAUS_EXT_VJP_WAVES
#define CAUS_EXT_VJP_WAVES 3
#endif

constexpr int kExtMaxParts = 16;    // most workgroups of one source's line integrals
constexpr int kExtPer = 4;          // initial limb angles per lane of k_ext_limb_init
constexpr int kExtFlatBlock = 256;  // block of the flat kernels

struct ExtArgs {
    const cd* w0;
    int64_t S;
    const double* rho;
    const double* params;
    int64_t pstride;
    const int32_t* npts;
    int npts_def;
    const double* u1;
    int64_t u1stride;
    int npts_ld;
    double* mag;
    uint8_t* status;
    const double* g_mag;   // VJP only
    double* g_out;         // VJP only: (S, 4 + P)
    char* ws;              // batch header, then one block of ws_per_source bytes per source
    size_t ws_per_source;
    unsigned long long* work;  // optional counters: FP64 root-iterations, FP32
                               // root-iterations, compensated root-iterations, limb-point
                               // solves, contour points
    int mmax;
    int nadd_max;
    int itmax;
};

// contours of one source, written by k_ext_contours
struct ExtContours {
    unsigned closed;  // image rows that are closed contours by themselves
    int open;         // 1 when the three stitched contours in con[] are used
    ActSeg con[3];
};

// batch header of the workspace
struct ExtBatch {
    int64_t* off_init;  // S + 1: prefix of the lanes of k_ext_limb_init
    int64_t* off_add;   // S + 1: prefix of the new points of one refinement round
    int32_t* npts;      // S: effective limb resolution
    uint8_t* fail;      // S: a solve did not converge, or npts was out of range
    int32_t* t_src;     // new-point tasks of the current round (capacity S * nadd_max):
    int32_t* t_left;    // source, append index of the left and right limb neighbours,
    int32_t* t_right;   // limb-order position and append index of the new point, and
    int32_t* t_dst;     // its limb angle
    int32_t* t_app;
    double* t_th;
    double2* gl;        // 2 x 128 Gauss-Legendre nodes and weights (limb darkening)
};
constexpr int kExtGL = 128;   // most nodes of one part of a line (npts_ld <= 256)

__host__ __device__ inline size_t ext_task_cap(int64_t S, int nadd_max) {
    return (size_t)S * (size_t)(nadd_max > 0 ? nadd_max : 1);
}

__host__ __device__ inline size_t ext_header_bytes(int64_t S, int nadd_max) {
    const size_t cap = ext_task_cap(S, nadd_max);
    return ext_align(2 * (size_t)(S + 1) * sizeof(int64_t)) + ext_align((size_t)S * 4) +
           ext_align((size_t)S) + ext_align(5 * cap * sizeof(int32_t)) +
           ext_align(cap * sizeof(double)) + 2 * kExtGL * sizeof(double2);
}

__host__ __device__ inline size_t ext_source_bytes(int deg, int mmax) {
    return ext_ws_bytes(deg, mmax) + ext_align(sizeof(ExtContours));
}

__host__ __device__ inline size_t ext_total_bytes(int deg, int64_t S, int npts_max) {
    return ext_header_bytes(S, ext_n_add(npts_max)) +
           (size_t)S * ext_source_bytes(deg, ext_mmax(npts_max));
}

__device__ inline ExtBatch ext_batch(const ExtArgs& A) {
    ExtBatch b;
    char* p = A.ws;
    const size_t cap = ext_task_cap(A.S, A.nadd_max);
    b.off_init = (int64_t*)p;
    b.off_add = b.off_init + (A.S + 1);
    p += ext_align(2 * (size_t)(A.S + 1) * sizeof(int64_t));
    b.npts = (int32_t*)p;
    p += ext_align((size_t)A.S * 4);
    b.fail = (uint8_t*)p;
    p += ext_align((size_t)A.S);
    b.t_src = (int32_t*)p;
    b.t_left = b.t_src + cap;
    b.t_right = b.t_left + cap;
    b.t_dst = b.t_right + cap;
    b.t_app = b.t_dst + cap;
    p += ext_align(5 * cap * sizeof(int32_t));
    b.t_th = (double*)p;
    p += ext_align(cap * sizeof(double));
    b.gl = (double2*)p;
    return b;
}

template <int DEG>
__device__ inline char* ext_source_base(const ExtArgs& A, int64_t s) {
    return A.ws + ext_header_bytes(A.S, A.nadd_max) + (size_t)s * A.ws_per_source;
}
template <int DEG>
__device__ inline ExtContours* ext_contours(const ExtArgs& A, int64_t s) {
    return (ExtContours*)(ext_source_base<DEG>(A, s) + ext_ws_bytes(DEG, A.mmax));
}

// lens frame, lens-frame source centre and radius of source s
template <int NL>
__device__ inline void ext_source(const ExtArgs& A, int64_t s, LensFrame<NL>& lf, cd& w0,
                                  double& rho) {
    double x_cm = 0.0;
    if constexpr (NL == 1) {
        lf.e[0] = 1.0;
        lf.r[0] = cd{0.0, 0.0};
    } else {
        lens_frame<NL>(A.params + s * A.pstride, lf, x_cm);
    }
    w0 = A.w0[s] + cd{x_cm, 0.0};
    rho = A.rho[s];
}

__device__ inline void ext_count(unsigned long long* work, const SolveStats& st, int solves) {
    atomicAdd(work + 0, (unsigned long long)st.it64);
    atomicAdd(work + 1, (unsigned long long)st.it32);
    atomicAdd(work + 2, (unsigned long long)st.itcomp);
    atomicAdd(work + 3, (unsigned long long)solves);
}

// limb points of source s after `round` refinement rounds
__device__ inline int ext_points(int npts, int round) {
    return ext_npts_init(npts) + round * ext_n_add(npts);
}

constexpr double kExtPi = 3.14159265358979323846;

// effective limb resolution of source s: 0 (skipped) or 4..npts_def, out-of-range values
// clamped and flagged
__device__ __forceinline__ int ext_npts(const ExtArgs& A, int64_t s, bool& bad) {
    const int n = A.npts ? A.npts[s] : A.npts_def;
    bad = n != 0 && (n < 4 || n > A.npts_def);
    return bad ? (n < 4 ? 4 : A.npts_def) : n;
}

// effective npts and the prefix offsets of the flat work lists: one workgroup, each thread
// a run of consecutive sources
__device__ inline void ext_plan(const ExtArgs& A, const ExtBatch& B) {
    constexpr int NT = kExtFlatBlock;
    __shared__ int64_t s_a[NT / 64], s_b[NT / 64];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int64_t run = (A.S + NT - 1) / NT;
    const int64_t s0 = min(A.S, tid * run), s1 = min(A.S, s0 + run);
    int64_t ca = 0, cb = 0;
    for (int64_t s = s0; s < s1; ++s) {
        bool bad;
        const int n = ext_npts(A, s, bad);
        B.npts[s] = n;   // 0: the source is skipped (no limb points, no work)
        ca += (ext_npts_init(n) + kExtPer - 1) / kExtPer;
        cb += ext_n_add(n);
    }
    int64_t ia = ca, ib = cb;   // inclusive sums over the threads
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int64_t ta = __shfl_up(ia, off, 64), tb = __shfl_up(ib, off, 64);
        if (lane >= off) {
            ia += ta;
            ib += tb;
        }
    }
    if (lane == 63) {
        s_a[wv] = ia;
        s_b[wv] = ib;
    }
    __syncthreads();
    for (int q = 0; q < wv; ++q) {
        ia += s_a[q];
        ib += s_b[q];
    }
    int64_t oa = ia - ca, ob = ib - cb;
    for (int64_t s = s0; s < s1; ++s) {
        const int n = B.npts[s];
        B.off_init[s] = oa;
        B.off_add[s] = ob;
        oa += (ext_npts_init(n) + kExtPer - 1) / kExtPer;
        ob += ext_n_add(n);
    }
    if (tid == NT - 1) {
        B.off_init[A.S] = oa;
        B.off_add[A.S] = ob;
    }
}

// ---- initial limb points (extended_source.py:100-106), two launches.
// START: the first workgroup plans the batch, with limb darkening (ngl = npts_ld) the next
// one computes the Gauss-Legendre nodes, and the others solve limb point 0 of every source,
// flanes sources per workgroup while one wave of each suffices, and set the failure flags.
// Otherwise: the points after it, one run of kExtPer consecutive angles per lane.  The
// lane's first angle starts from the standard initial estimates (after point 0: from its
// roots), each later one from the previous angle's roots.  A warm start can leave two
// estimates inside one cluster of nearly double images (near a caustic), where the FP64
// stopping test accepts both before they separate; the compensated polish that ends every
// solve continues the Aberth iteration there and takes them to the cluster's distinct roots.
// Point 0 is solved in the reference's root order (ext_solve_point, first).  That solve costs
// as much as the rest of a run, and one lane of it holds its whole wave: with the points 0
// inside the runs 12,000 triple-lens sources took 5.6 ms, apart 4.5 ms for both launches (4,096
// binary ones 0.71 and 0.67 ms).  The nodes were found by a wave of every source before its
// integration (some 30 us each).  Both launches run one kernel, so that the ill-conditioned
// solves of all points are compiled, and round, alike.
template <int NL, int MODE>
__global__ __launch_bounds__(kExtFlatBlock)
__attribute__((amdgpu_waves_per_eu(2)))  // 2 waves/SIMD measured faster than 1
void k_ext_limb_init(ExtArgs A, int start, int ngl, int flanes) {
    constexpr int DEG = ext_degree<NL>();
    const ExtBatch B = ext_batch(A);
    int64_t blk = blockIdx.x, per_block = kExtFlatBlock, total, stride;
    if (start) {
        if (blk == 0) {
            ext_plan(A, B);
            return;
        }
        if (ngl && blk == 1) {
            static_assert(kExtFlatBlock == 2 * kExtGL, "one thread per node");
            const int part = threadIdx.x / kExtGL, i = threadIdx.x % kExtGL;
            const int n = part == 0 ? ngl / 2 : ngl - ngl / 2;
            if (i < n) gauss_legendre(n, i, B.gl + part * kExtGL);
            return;
        }
        blk -= ngl ? 2 : 1;
        if ((int)threadIdx.x >= flanes) return;
        per_block = flanes;
        total = A.S;
        stride = total;
    } else {
        total = B.off_init[A.S];
        stride = (int64_t)gridDim.x * kExtFlatBlock;
    }
    for (int64_t t = blk * per_block + threadIdx.x; t < total; t += stride) {
        int64_t lo = t;
        int n, k0 = 0, kb = 0;
        bool bad = false;
        if (start) {
            n = ext_npts(A, t, bad);
        } else {
            lo = 0;
            int64_t hi = A.S;  // off_init[lo] <= t < off_init[hi]
            while (hi - lo > 1) {
                const int64_t mid = (lo + hi) >> 1;
                if (B.off_init[mid] <= t) lo = mid;
                else hi = mid;
            }
            n = B.npts[lo];
            k0 = (int)(t - B.off_init[lo]) * kExtPer;
            kb = max(k0, 1);
        }
        const int64_t s = lo;
        const int M0 = ext_npts_init(n);
        const int k1 = start ? (n == 0 ? 0 : 1) : min(M0, k0 + kExtPer);
        LensFrame<NL> lf;
        cd w0;
        double rho;
        ext_source<NL>(A, s, lf, w0, rho);
        ExtWS W = ext_ws(ext_source_base<DEG>(A, s), DEG, A.mmax);
        cd z[DEG];
        if (kb > k0) load_pt<DEG>(W.z[0], 0, z);
        SolveStats st{0, 0, 0, 0};
        bool fail = bad;
        for (int k = kb; k < k1; ++k) {
            const double th = ext_limb_angle(k, M0 - 1);
            double sn, cs;
            sincos(th, &sn, &cs);
            uint32_t f;
            if (!ext_solve_point<NL, MODE>(ext_limb_point(w0, rho, cs, sn), lf, z, f, A.itmax,
                                           A.work ? &st : nullptr, k > k0, k == 0))
                fail = true;
            W.theta[0][k] = th;
            store_pt<DEG>(W.z[0], k, z);
            W.flg[0][k] = f;
        }
        if (start || fail) B.fail[s] = fail ? 1 : 0;
        if (A.work) ext_count(A.work, st, k1 - kb);
    }
}

// key of the gap between limb points a and b (rows as stored): the largest image step
// |b_r - a_r| over rows real at either end, as an ordered bit pattern
// (extended_source.py:112-116)
template <int DEG>
__device__ __forceinline__ uint64_t gap_key(const cd* za, uint32_t fa, const cd* zb_,
                                            uint32_t fb_) {
    const uint32_t m = (fa | fb_) & 0xFFFFu;
    double dmax = 0.0;
#pragma unroll
    for (int r = 0; r < DEG; ++r)
        if ((m >> r) & 1u) dmax = fmax(dmax, norm2(zb_[r] - za[r]));
    return (uint64_t)__double_as_longlong(sqrt(dmax));   // sqrt is monotone: one for all rows
}

// ---- image continuation (chain.hpp), one workgroup per source.  FINAL = false: over the
// initial points (buffer 0, limb order = append order), in place, then the limb order and
// the gap keys of round 0.  FINAL = true: over the refined points, read through the limb
// order ord[cur] and gathered once into buffer 1, row after row.
// Measured on 24,000 triple-lens sources (256-4096 limb points), both launches of two
// chunks: one wave per source with the points gathered before and after the scan, every
// conflict searched by shuffles row by row, 10.6 ms; this form 3.9 ms.
template <int NL, bool FINAL>
__global__ __launch_bounds__(kExtBlock) void k_ext_chain(ExtArgs A, int cur) {
    constexpr int DEG = ext_degree<NL>();
    const int tid = threadIdx.x;
    const int64_t s = blockIdx.x;
    const ExtBatch B = ext_batch(A);
    if (B.npts[s] == 0) return;   // skipped source
    ExtWS W = ext_ws(ext_source_base<DEG>(A, s), DEG, A.mmax);
    uint64_t* perm = W.perm;
    auto word = [perm](int k) -> uint64_t& { return perm[k]; };
    cd* z0 = W.z[0];
    if constexpr (!FINAL) {
        const int M = ext_points(B.npts[s], 0);
        auto get = [z0](int k, int r) { return z0[(size_t)k * DEG + r]; };
        chain_perms<DEG, kExtBlock>(get, word, M);
        for (int k = tid; k < M; k += kExtBlock) {
            const uint64_t p = perm[k];
            cd z[DEG];
#pragma unroll
            for (int i = 0; i < DEG; ++i) z[i] = get(k, pget(p, i));
            store_pt<DEG>(z0, k, z);
            W.flg[0][k] = permute_flags<DEG>(W.flg[0][k], p);
        }
        __syncthreads();
        for (int k = tid; k < M; k += kExtBlock) {
            W.ord[0][k] = k;
            if (k + 1 < M)
                W.gk[0][k] = gap_key<DEG>(z0 + (size_t)k * DEG, W.flg[0][k],
                                          z0 + (size_t)(k + 1) * DEG, W.flg[0][k + 1]);
        }
    } else {
        const int M = ext_points(B.npts[s], 10);
        const int32_t* ord = W.ord[cur];
        auto get = [z0, ord](int k, int r) { return z0[(size_t)ord[k] * DEG + r]; };
        chain_perms<DEG, kExtBlock>(get, word, M);
        cd* z1 = W.z[1];
        for (int k = tid; k < M; k += kExtBlock) {
            const uint64_t p = perm[k];
            const int a = ord[k];
#pragma unroll
            for (int i = 0; i < DEG; ++i)
                z1[(size_t)i * A.mmax + k] = z0[(size_t)a * DEG + pget(p, i)];
            W.flg[1][k] = permute_flags<DEG>(W.flg[0][a], p);
            W.theta[1][k] = W.theta[0][a];
        }
    }
}

// ---- one refinement round, part 1 (extended_source.py:108-135): the n_add largest
// image gaps (descending by (gap, position)), insertion shifts, the next limb order and the
// carried-over gap keys, one task per new point.  Points stay where they are (append
// order); only the order and keys move.
//
// Only the set of the n_add largest keys matters (the append order of the new points is
// never seen again: everything later goes through the limb order), so the keys are not
// sorted.  Each thread holds its PER keys (limb position tid + i NT) in registers and the
// threshold is found by bisection on the key's bit pattern, one ballot and popcount per
// register and step; some 15-20 steps isolate the n_add-th key, and equal keys are taken
// from the last position on, as a descending sort by (key, position) takes them.  The
// shifts come from the same ballots.
// NT threads per source: one wave for short contours, four above kExtSelWave points.
// Bound: latency of the bisection's dependent steps.  A bitonic sort of all keys in LDS
// took 15.5 us at 150 limb points (one source) and 361 us for 4,096 binary sources of
// 256-4096 points.
constexpr int kExtSelWave = 512;
// LDS written by some lanes of a wave, read by others of the same wave
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
template <int NT, int PER>
struct ExtSelLds {
    int cnt[2][NT / 64];           // bisection counts, double buffered (one barrier a step)
    uint64_t max[NT / 64];
    int sel[PER * (NT / 64)];      // selected / tied keys per (register, wave)
};
// the NT threads tid = 0 .. NT-1 of a workgroup run it together (one wave of a larger
// workgroup where NT is 64)
template <int NL, int NT, int PER>
__device__ __forceinline__ void ext_select(const ExtArgs& A, const ExtBatch& B, int64_t src, int n,
                                           int cur, int round, int tid, ExtSelLds<NT, PER>& sh) {
    constexpr int DEG = ext_degree<NL>();
    constexpr int NW = NT / 64;
    auto sync = [] {
        if constexpr (NW > 1) __syncthreads();
        else wave_sync();
    };
    int (&s_cnt)[2][NW] = sh.cnt;
    uint64_t (&s_max)[NW] = sh.max;
    int (&s_sel)[PER * NW] = sh.sel;
    const int lane = tid & 63, wv = tid >> 6;
    const int M = ext_points(n, round), nadd = ext_n_add(n);   // M <= PER * NT
    ExtWS W = ext_ws(ext_source_base<DEG>(A, src), DEG, A.mmax);
    const int nxt = cur ^ 1;
    const int32_t* ord = W.ord[cur];
    const uint64_t* gk = W.gk[cur];
    uint64_t key[PER];
    uint64_t mx = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int k = tid + i * NT;
        key[i] = k < M - 1 ? gk[k] : 0ull;
        mx = key[i] > mx ? key[i] : mx;
    }
    int par = 0;
    // number of keys >= t (t >= 1, so the padding's zero keys never count)
    auto count = [&](uint64_t t) -> int {
        int c = 0;
#pragma unroll
        for (int i = 0; i < PER; ++i) c += __popcll(__ballot(key[i] >= t));
        if constexpr (NW > 1) {
            if (lane == 0) s_cnt[par][wv] = c;
            __syncthreads();
            c = 0;
#pragma unroll
            for (int q = 0; q < NW; ++q) c += s_cnt[par][q];
            par ^= 1;
        }
        return c;
    };
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const uint64_t o = __shfl_xor(mx, off, 64);
        mx = o > mx ? o : mx;
    }
    if constexpr (NW > 1) {
        if (lane == 0) s_max[wv] = mx;
        __syncthreads();
#pragma unroll
        for (int q = 0; q < NW; ++q) mx = s_max[q] > mx ? s_max[q] : mx;
    }
    // count(>= lo) >= nadd > count(>= hi) = chi; keys are non-negative doubles' bits
    uint64_t lo = 0, hi = mx + 1;
    int chi = 0;
    bool exact = false;
    if (nadd == 0) {
        lo = hi;       // nothing is selected
        exact = true;
    }
    const uint64_t low = 24ull << 52;   // a first step 24 binades below the largest gap
    bool probe = mx > low;
    while (!exact && hi - lo > 1) {
        const uint64_t mid = probe ? mx - low : lo + ((hi - lo) >> 1);
        probe = false;
        const int c = count(mid);
        if (c == nadd) exact = true;
        if (c >= nadd) {
            lo = mid;
        } else {
            hi = mid;
            chi = c;
        }
    }
    // keys >= lo are selected when that is exactly nadd of them; otherwise the chi keys
    // above lo and the last nadd - chi of the keys equal to lo
    unsigned sel = 0;   // bit i: the gap after point tid + i NT is refined
    if (exact) {
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (key[i] >= lo && tid + i * NT < M - 1) sel |= 1u << i;
    } else {
        int tot = 0;    // all keys equal to lo
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const uint64_t m = __ballot(key[i] == lo && tid + i * NT < M - 1);
            if (lane == 0) s_sel[i * NW + wv] = __popcll(m);
        }
        sync();
        for (int q = 0; q < PER * NW; ++q) tot += s_sel[q];
        int before = 0;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const bool tie = key[i] == lo && tid + i * NT < M - 1;
            const uint64_t m = __ballot(tie);
            int b = before;
            for (int q = 0; q < NW; ++q) {
                if (q < wv) b += s_sel[i * NW + q];
                before += s_sel[i * NW + q];
            }
            const int rank = b + __popcll(m & ((1ull << lane) - 1ull));   // ties before this one
            if (key[i] > lo || (tie && tot - rank <= nadd - chi)) sel |= 1u << i;
        }
        sync();
    }
    // insertion shift of every point = selected gaps before it
    uint64_t bal[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        bal[i] = __ballot((sel >> i) & 1u);
        if (NW > 1 && lane == 0) s_sel[i * NW + wv] = __popcll(bal[i]);
    }
    if constexpr (NW > 1) __syncthreads();
    const int64_t t0 = B.off_add[src];
    int run = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        if (i * NT >= M) break;
        int b = run;
        if constexpr (NW > 1) {
            for (int q = 0; q < NW; ++q) {
                if (q < wv) b += s_sel[i * NW + q];
                run += s_sel[i * NW + q];
            }
        } else {
            run += __popcll(bal[i]);
        }
        const int k = tid + i * NT;
        if (k >= M) continue;
        const int c = b + __popcll(bal[i] & ((1ull << lane) - 1ull));
        const int d = k + c;
        const int a = ord[k];
        W.ord[nxt][d] = a;
        if ((sel >> i) & 1u) {
            const int e = ord[k + 1];
            const int64_t t = t0 + c;
            B.t_src[t] = (int32_t)src;
            B.t_left[t] = a;
            B.t_right[t] = e;
            B.t_dst[t] = d + 1;
            B.t_app[t] = M + c;
            B.t_th[t] = 0.5 * (W.theta[0][a] + W.theta[0][e]);
            W.ord[nxt][d + 1] = M + c;
        } else if (k + 1 < M) {
            W.gk[nxt][d] = key[i];
        }
    }
}
template <int NL, int NT, int PER>
__global__ __launch_bounds__(NT) void k_ext_select(ExtArgs A, int cur, int round) {
    __shared__ ExtSelLds<NT, PER> sh;
    const int64_t src = blockIdx.x;
    const ExtBatch B = ext_batch(A);
    const int n = B.npts[src];
    if (n == 0) return;   // skipped source
    ext_select<NL, NT, PER>(A, B, src, n, cur, round, threadIdx.x, sh);
}

// ---- one refinement round, part 2: every new point of the batch, one per lane,
// solved, matched to its left neighbour's images (match_points), appended, and the
// keys of its two gaps
template <int NL, int MODE>
__global__ __launch_bounds__(kExtFlatBlock)
__attribute__((amdgpu_waves_per_eu(2)))  // 2 waves/SIMD measured faster than 1
void k_ext_solve_add(ExtArgs A, int cur) {
    constexpr int DEG = ext_degree<NL>();
    const ExtBatch B = ext_batch(A);
    const int64_t total = B.off_add[A.S];
    const int64_t stride = (int64_t)gridDim.x * kExtFlatBlock;
    const int nxt = cur ^ 1;
    for (int64_t t = (int64_t)blockIdx.x * kExtFlatBlock + threadIdx.x; t < total; t += stride) {
        const int64_t s = B.t_src[t];
        const int a = B.t_left[t], b = B.t_right[t], d = B.t_dst[t], e = B.t_app[t];
        const double th = B.t_th[t];
        LensFrame<NL> lf;
        cd w0;
        double rho;
        ext_source<NL>(A, s, lf, w0, rho);
        ExtWS W = ext_ws(ext_source_base<DEG>(A, s), DEG, A.mmax);
        double sn, cs;
        sincos(th, &sn, &cs);
        cd z[DEG], left[DEG];
        load_pt<DEG>(W.z[0], a, left);
#pragma unroll
        for (int r = 0; r < DEG; ++r) z[r] = left[r];   // start from the left neighbour
        uint32_t f;
        SolveStats st{0, 0, 0, 0};
        if (!ext_solve_point<NL, MODE>(ext_limb_point(w0, rho, cs, sn), lf, z, f, A.itmax,
                                       A.work ? &st : nullptr, true))
            B.fail[s] = 1;
        if (A.work) ext_count(A.work, st, 1);
        const uint64_t p = greedy_match<DEG>(left, z);
        // scatter raw row j to row pinv[j] (output row i = raw row p[i])
        uint64_t pinv = 0;
#pragma unroll
        for (int i = 0; i < DEG; ++i) pinv |= (uint64_t)i << (4 * pget(p, i));
        cd* ze = W.z[0] + (size_t)e * DEG;
#pragma unroll
        for (int j = 0; j < DEG; ++j) ze[pget(pinv, j)] = z[j];
        f = permute_flags<DEG>(f, p);
        W.flg[0][e] = f;
        W.theta[0][e] = th;
        // gaps (left, new) at d-1 and (new, right) at d, from the stored rows
        cd zn[DEG];
#pragma unroll
        for (int i = 0; i < DEG; ++i) zn[i] = z[pget(p, i)];
        W.gk[nxt][d - 1] = gap_key<DEG>(left, W.flg[0][a], zn, f);
        cd right[DEG];
        load_pt<DEG>(W.z[0], b, right);
        W.gk[nxt][d] = gap_key<DEG>(zn, f, right, W.flg[0][b]);
    }
}

// ---- one polynomial per group of lanes, one root per lane -------------------------------
// A small batch has too few limb points to fill the device with one polynomial per lane, and
// a launch then lasts as long as one lane needs for all DEG roots after each other.  Here lane
// j of a group of 8 (two lenses) or 16 (three) holds root j: an Ehrlich-Aberth sweep and a
// sweep of the compensated polish take one root's instructions.  Roots are exchanged through
// LDS within a wave.  All roots move together (Jacobi form), where the one-lane solver moves
// them one after the other; both end in the compensated polish, which takes every root to the
// double nearest the exact one whatever led there.  A nearly double pair can still move when
// the polish's sweeps end, so the results are the same to rounding (of 19,200 sources at caustics
// 1 magnification and 4 gradients differed, by up to 5e-12; all others were the same bits).
template <int NL>
constexpr int ext_group() {
    return NL == 3 ? 16 : 8;
}

// sweeps of the group's polish: only clusters need more than two, and there all roots moving
// together take more of them than one after the other (kPolishSweeps)
constexpr int kGroupPolishSweeps = 40;
template <int NL>
struct GroupSolve {
    static constexpr int DEG = ext_degree<NL>();
    static constexpr int GL = ext_group<NL>();
    static_assert(DEG < GL, "a lane per coefficient");
    double2* zs;   // this group's GL slots
    int j;         // root of this lane (valid below DEG)

    __device__ __forceinline__ void put(cd z) const {
        wave_sync();
        zs[j] = make_double2(z.re, z.im);
        wave_sync();
    }
    __device__ __forceinline__ cd get(int i) const {
        const double2 v = zs[i];
        return cd{v.x, v.y};
    }
    // sum over the other roots of 1/(x - z_i); they are read from the group's slots
    template <int RCP_STEPS>
    __device__ __forceinline__ cd aberth(cd x) const {
        cd S = cd{0.0, 0.0};
#pragma unroll
        for (int i = 0; i < DEG; ++i) {
            cd d = x - get(i);
            const bool own = i == j;
            d.re = own ? 1.0 : d.re;   // keeps the reciprocal finite
            const cd r = crcp<RCP_STEPS>(d);
            S = S + cd{own ? 0.0 : r.re, own ? 0.0 : r.im};
        }
        return S;
    }
    // plain FP64 sweeps until every root of every group of the wave has met the stopping test
    // (fast_step); returns whether this lane's root has
    __device__ __forceinline__ bool iterate(const cd (&p)[DEG + 1], cd& z, int itmax,
                                            SolveStats& st) const {
        double al[DEG + 1];
#pragma unroll
        for (int i = 0; i <= DEG; ++i) al[i] = cabs(p[i]);
#pragma unroll
        for (int i = 0; i <= DEG; ++i) al[i] = al[i] * fma(ALPHA_W, (double)i, 1.0);
        bool done = j >= DEG;
        for (int it = 0; it < itmax && __ballot(!done) != 0ull; ++it) {
            put(z);
            if (done) continue;
            ++st.it64;
            const cd x = z;
            const double ax = __builtin_amdgcn_sqrt(norm2(x));
            double b = al[DEG];
#pragma unroll
            for (int k = DEG - 1; k >= 0; --k) b = fma(b, ax, al[k]);
            cd h = p[DEG], hd = cd{0.0, 0.0};
#pragma unroll
            for (int k = DEG - 1; k >= 0; --k) {
                hd = cfma(hd, x, h);
                h = cfma(h, x, p[k]);
            }
            const double tb = EA_EPS * b;
            if (norm2(h) > tb * tb)
                z = x - cdiv<2>(h, hd - h * aberth<0>(x));
            else
                done = true;
        }
        return done;
    }
    // polish_roots, every root of a sweep at once
    __device__ __forceinline__ void polish(const cd (&p)[DEG + 1], cd& z) const {
        bool act = j < DEG;
        for (int sweep = 0; sweep < kGroupPolishSweeps && __ballot(act) != 0ull; ++sweep) {
            put(z);
            if (!act) continue;
            cd h, hd;
            if (sweep == 0)
                horner_comp_value<DEG>(p, z, h, hd);
            else
                horner_comp_vd<DEG>(p, z, h, hd);
            const cd den = hd - h * aberth<2>(z);
            act = false;
            if (norm2(den) > 0.0) {
                const cd corr = cdiv<2>(h, den);
                const cd zn = z - corr;
                if (isfinite(zn.re) && isfinite(zn.im)) {
                    act = norm2(corr) > 0x1p-80 * norm2(z);
                    z = zn;
                }
            }
        }
    }
};

// this lane's group within its wave: the lanes' bits of a ballot
template <int GL>
__device__ __forceinline__ uint32_t group_bits(uint64_t ballot) {
    const int base = (threadIdx.x & 63) & ~(GL - 1);
    return (uint32_t)(ballot >> base) & ((1u << GL) - 1u);
}

// limb point at angle th of one source by one group: the roots (one a lane, left in the
// group's slots) and the flag word; false if one did not converge
template <int NL>
__device__ __forceinline__ bool ext_group_point(const GroupSolve<NL>& G, cd w,
                                                const LensFrame<NL>& lf, cd& z, int itmax,
                                                uint32_t& flags, SolveStats& st) {
    constexpr int DEG = ext_degree<NL>();
    constexpr int GL = ext_group<NL>();
    bool ok = true, real = true, neg = false;
    if constexpr (NL == 1) {
        const double sq = sqrt(1.0 + 4.0 * rcp(norm2(w)));
        z = (G.j == 0 ? 0.5 * (1.0 + sq) : 0.5 * (1.0 - sq)) * w;
        neg = norm2(z) < 1.0;
    } else {
        cd p[DEG + 1];
        lens_poly<NL>(w, lf, p);
        ok = G.iterate(p, z, itmax, st);
        ok = ok && (G.j >= DEG || (isfinite(z.re) && isfinite(z.im)));
        G.polish(p, z);
        const ImageTerms<NL> it = image_terms<NL>(z, lf);
        real = norm2(z - it.G - w) < 1e-12;
        neg = 1.0 - norm2(it.K) < 0.0;
    }
    const uint32_t in = (1u << DEG) - 1u;
    const uint32_t fr = group_bits<GL>(__ballot(real)) & in;
    const uint32_t fn = group_bits<GL>(__ballot(neg)) & in;
    flags = fr | (fn << 16);
    G.put(z);
    return (group_bits<GL>(__ballot(ok)) & in) == in;
}

// The third lens' position from its polar form again, where the solve's coefficients are
// formed: there the compiler contracts the products into the sums that take them, as it does
// in k_ext_solve_add, and the ill-conditioned roots near a lens of small mass follow an ulp of
// a coefficient by up to its square root.
__device__ __forceinline__ void lens3_refresh(const double* prm, double sp, double cp,
                                              LensFrame<3>& lf) {
    double R = prm[3];
    asm volatile("" : "+v"(R));   // not hoisted out of the caller's loop
    lf.r[2] = cd{R * cp, R * sp};
}

// ---- the initial limb points after point 0, one a group of lanes, each from point 0's roots;
// per_source workgroups for every source.  Used where the batch is small (ext_grouped).
template <int NL>
__global__ __launch_bounds__(kExtBlock) void k_ext_init_grouped(ExtArgs A, int per_source) {
    constexpr int DEG = ext_degree<NL>();
    constexpr int GL = ext_group<NL>();
    __shared__ double2 s_z[kExtBlock];
    const int tid = threadIdx.x;
    const int64_t src = blockIdx.x / per_source;
    const ExtBatch B = ext_batch(A);
    const int M0 = ext_npts_init(B.npts[src]);
    const int k0 = 1 + (int)(blockIdx.x % per_source) * (kExtBlock / GL);
    if (k0 >= M0) return;
    const int kq = k0 + tid / GL;
    const bool mine = kq < M0;
    const int k = mine ? kq : M0 - 1;   // groups past the last point repeat it, write nothing
    LensFrame<NL> lf;
    cd w0;
    double rho;
    ext_source<NL>(A, src, lf, w0, rho);
    ExtWS W = ext_ws(ext_source_base<DEG>(A, src), DEG, A.mmax);
    const int j = tid & (GL - 1);
    const GroupSolve<NL> G{s_z + (tid & ~(GL - 1)), j};
    const double th = ext_limb_angle(k, M0 - 1);
    double sn, cs;
    sincos(th, &sn, &cs);
    cd z = j < DEG ? W.z[0][j] : cd{0.0, 0.0};
    uint32_t f;
    SolveStats st{0, 0, 0, 0};
    const bool ok = ext_group_point<NL>(G, ext_limb_point(w0, rho, cs, sn), lf, z, A.itmax,
                                        f, st);
    if (!mine) return;
    if (j < DEG) W.z[0][(size_t)k * DEG + j] = z;
    if (j == 0) {
        W.theta[0][k] = th;
        W.flg[0][k] = f;
        if (!ok) B.fail[src] = 1;
    }
    if (A.work) ext_count(A.work, st, j == 0 ? 1 : 0);
}

// ---- all ten refinement rounds of one source by one workgroup: ext_select, then the new
// points one a group of lanes.  Used where the batch is small (ext_grouped).
// Bound: latency of the rounds' serial steps (figures: ext_grouped).
template <int NL, int SELT, int PER>
__global__ __launch_bounds__(kExtBlock) void k_ext_refine(ExtArgs A) {
    constexpr int DEG = ext_degree<NL>();
    constexpr int GL = ext_group<NL>();
    __shared__ ExtSelLds<SELT, PER> sh;
    __shared__ double2 s_z[kExtBlock], s_left[kExtBlock];
    const int tid = threadIdx.x;
    const int64_t src = blockIdx.x;
    const ExtBatch B = ext_batch(A);
    const int n = B.npts[src];
    if (n == 0) return;   // skipped source
    const int nadd = ext_n_add(n);
    const int64_t t0 = B.off_add[src];
    LensFrame<NL> lf;
    cd w0;
    double rho;
    ext_source<NL>(A, src, lf, w0, rho);
    ExtWS W = ext_ws(ext_source_base<DEG>(A, src), DEG, A.mmax);
    double sp3 = 0.0, cp3 = 0.0;
    if constexpr (NL == 3) sincos(A.params[src * A.pstride + 4], &sp3, &cp3);
    const int j = tid & (GL - 1), base = tid & ~(GL - 1);
    const GroupSolve<NL> G{s_z + base, j};
    double2* const lefts = s_left + base;
    SolveStats st{0, 0, 0, 0};
    bool fail = false;
    int cur = 0;
    for (int round = 0; round < 10; ++round, cur ^= 1) {
        if (tid < SELT) ext_select<NL, SELT, PER>(A, B, src, n, cur, round, tid, sh);
        __syncthreads();
        const int nxt = cur ^ 1;
        for (int q0 = 0; q0 < nadd; q0 += kExtBlock / GL) {
            // groups past the last point repeat it and write nothing
            const int q = q0 + tid / GL;
            const bool mine = q < nadd;
            const int64_t t = t0 + (mine ? q : nadd - 1);
            const int a = B.t_left[t], b = B.t_right[t], d = B.t_dst[t], e = B.t_app[t];
            const double th = B.t_th[t];
            const cd left = j < DEG ? W.z[0][(size_t)a * DEG + j] : cd{0.0, 0.0};
            const cd right = j < DEG ? W.z[0][(size_t)b * DEG + j] : cd{0.0, 0.0};
            const uint32_t fa = W.flg[0][a], fb = W.flg[0][b];
            lefts[j] = make_double2(left.re, left.im);
            double sn, cs;
            sincos(th, &sn, &cs);
            if constexpr (NL == 3) lens3_refresh(A.params + src * A.pstride, sp3, cp3, lf);
            cd z = left;   // start from the left neighbour
            uint32_t f;
            SolveStats s1{0, 0, 0, 0};
            const bool ok = ext_group_point<NL>(G, ext_limb_point(w0, rho, cs, sn), lf, z, A.itmax,
                                                f, s1);
            if (mine) {
                st.it64 += s1.it64;
                fail |= !ok;
            }
            // nearest new image of left row j; rows that take distinct ones follow them
            // whatever the row order, otherwise row by row (greedy_match)
            int bj = 0;
            double best = 0.0;
            bool nan = false;
#pragma unroll
            for (int i = 0; i < DEG; ++i) {
                const double dd = norm2(G.get(i) - left);
                nan |= dd != dd;
                if (i == 0 || dd < best) {
                    best = dd;
                    bj = i;
                }
            }
            const bool odd = group_bits<GL>(__ballot(nan && j < DEG)) != 0;
            uint32_t hit = j < DEG ? 1u << bj : 0u;
#pragma unroll
            for (int off = 1; off < GL; off <<= 1) hit |= __shfl_xor(hit, off, 64);
            if (odd || hit != (1u << DEG) - 1u) {
                unsigned used = 0;
#pragma unroll 1
                for (int i = 0; i < DEG; ++i) {
                    const double2 lv = lefts[i];
                    double bd = 0.0;
                    int bi = -1;
#pragma unroll 1
                    for (int c = 0; c < DEG; ++c) {
                        const double dd = norm2(G.get(c) - cd{lv.x, lv.y});
                        if (!((used >> c) & 1u) && (bi < 0 || dd < bd)) {
                            bd = dd;
                            bi = c;
                        }
                    }
                    used |= 1u << bi;
                    if (i == j) bj = bi;
                }
            }
            // output row j = raw row bj
            const cd zn = G.get(bj);
            const uint32_t in = (1u << DEG) - 1u;
            const uint32_t fo =
                (group_bits<GL>(__ballot((f >> bj) & 1u)) & in) |
                ((group_bits<GL>(__ballot((f >> (16 + bj)) & 1u)) & in) << 16);
            // keys of the gaps (left, new) at d-1 and (new, right) at d (gap_key)
            double d1 = j < DEG && (((fa | fo) >> j) & 1u) ? norm2(zn - left) : 0.0;
            double d2 = j < DEG && (((fo | fb) >> j) & 1u) ? norm2(right - zn) : 0.0;
#pragma unroll
            for (int off = 1; off < GL; off <<= 1) {
                d1 = fmax(d1, __shfl_xor(d1, off, 64));
                d2 = fmax(d2, __shfl_xor(d2, off, 64));
            }
            if (mine && j < DEG) W.z[0][(size_t)e * DEG + j] = zn;
            if (mine && j == 0) {
                W.flg[0][e] = fo;
                W.theta[0][e] = th;
                W.gk[nxt][d - 1] = (uint64_t)__double_as_longlong(sqrt(fmax(0.0, d1)));
                W.gk[nxt][d] = (uint64_t)__double_as_longlong(sqrt(fmax(0.0, d2)));
            }
        }
        __syncthreads();
    }
    if (fail) B.fail[src] = 1;
    if (A.work) ext_count(A.work, st, tid == 0 ? 10 * nadd : 0);
}

// ---- closed rows, segments and stitching (extended_source.py:156-727) for the final
// points in buffer `buf`; writes the source's ExtContours.  One workgroup per source: its
// four waves take a quarter of the boundaries each, wave by wave the segments' lengths, and
// the first one stitches with one remaining segment per lane: the sort is a rank count, each
// lane tests its segment's four connections, and the nearest admissible one among the four
// nearest is one wave reduction and a count.
// Bound: latency of the merge steps.  With every lane of one wave repeating the serial sort
// and search over records in LDS: one source 45 us, 4,096 binary sources 0.86 ms, 12,000
// triple-lens sources 3.0 ms; this form 13 us, 0.18 ms, 2.2 ms.
struct ExtCand {          // a candidate segment
    Seg s;
    cd h0, h1, t0, t1;    // its lines at the head and at the tail (head_line, tail_line)
};
template <int NL>
__global__ __launch_bounds__(kExtBlock) void k_ext_contours(ExtArgs A, int buf) {
    constexpr int DEG = ext_degree<NL>();
    constexpr int NIMG = NL * NL + 1;
    constexpr int NSEG = 3 * NIMG;  // nr_of_segments
    constexpr int NRUN = 10;        // starts / ends kept per row (the reference's split)
    constexpr int NW = kExtBlock / 64;
    static_assert(NSEG <= kExtMaxSeg && NSEG < 64, "one segment per lane");
    __shared__ ActSeg s_con[3];
    __shared__ ExtCand s_cand[NSEG];
    __shared__ int s_st[NW][DEG][NRUN], s_en[NW][DEG][NRUN], s_nst[NW][DEG], s_nen[NW][DEG];
    __shared__ int s_ord[64];
    __shared__ unsigned s_allmask;
    __shared__ int s_nc;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wv = tid >> 6;
    const int64_t src = blockIdx.x;
    const ExtBatch B = ext_batch(A);
    if (B.npts[src] == 0) return;   // skipped source
    const int M = ext_points(B.npts[src], 10);
    ExtWS W = ext_ws(ext_source_base<DEG>(A, src), DEG, A.mmax);
    ExtContours* C = ext_contours<DEG>(A, src);
    const ZRows zb{W.z[buf], A.mmax};
    const uint32_t* fb = W.flg[buf];
    // closure test (extended_source.py:289-291)
    if (tid == 0) s_allmask = 0xFFFFu;
    if (tid < NW * DEG) (&s_nst[0][0])[tid] = (&s_nen[0][0])[tid] = 0;
    __syncthreads();
    unsigned am = 0xFFFFu;
    for (int k = tid; k < M; k += kExtBlock) am &= fb[k];
    atomicAnd(&s_allmask, am);
    __syncthreads();
    unsigned closed = 0;
#pragma unroll
    for (int r = 0; r < DEG; ++r) {
        if ((s_allmask >> r) & 1u) {
            if (norm2(pt<DEG>(zb, 0, r) - pt<DEG>(zb, M - 1, r)) < 1e-10) closed |= 1u << r;
        }
    }
    const bool all_closed = closed == (1u << DEG) - 1u;
    if (!all_closed) {
        // changepoints per boundary c in [0, M] (extended_source.py:163-188), a quarter of the
        // boundaries per wave; rows that are closed contribute nothing (their segments were
        // zeroed).  Each wave keeps the first NRUN starts and ends of every row.
        const unsigned open = ((1u << DEG) - 1u) & ~closed;
        const int share = ((M + 1 + NW - 1) / NW + 63) & ~63;
        const int c0 = wv * share, c1 = min(M + 1, c0 + share);
        for (int base = c0; base < c1; base += 64) {
            const int c = base + lane;
            unsigned word = 0;
            if (c < c1) {
                const unsigned fp = (c > 0) ? fb[c - 1] : 0u, fc = (c < M) ? fb[c] : 0u;
#pragma unroll
                for (int r = 0; r < DEG; ++r) {
                    if (!((open >> r) & 1u)) continue;
                    const int mp = (int)((fp >> r) & 1u), mc = (int)((fc >> r) & 1u);
                    bool cp;
                    int dm;
                    if (c == 0) {
                        cp = mc != 0;
                        dm = mc ? 1 : 0;
                    } else if (c == M) {
                        cp = mp != 0;
                        dm = mp ? -1 : 0;
                    } else {
                        const cd za = mp ? pt<DEG>(zb, c - 1, r) : cd{0.0, 0.0};
                        const cd zc = mc ? pt<DEG>(zb, c, r) : cd{0.0, 0.0};
                        const int pa = mp ? (((fp >> (16 + r)) & 1u) ? -1 : 1) : 0;
                        const int pc_ = mc ? (((fc >> (16 + r)) & 1u) ? -1 : 1) : 0;
                        dm = mc - mp;
                        cp = (norm2(zc - za) > 0.01) || (pc_ != pa) || (dm != 0);
                    }
                    if (cp && dm >= 0) word |= 1u << r;
                    if (cp && dm <= 0) word |= 1u << (16 + r);
                }
            }
            if (__ballot(word != 0) == 0ull) continue;
            const uint64_t below = (1ull << lane) - 1ull;
            for (int r = 0; r < DEG; ++r) {
                const uint64_t ms = __ballot((word >> r) & 1u);
                const uint64_t me = __ballot((word >> (16 + r)) & 1u);
                if ((ms | me) == 0ull) continue;
                const int ns = s_nst[wv][r], ne = s_nen[wv][r];
                if ((word >> r) & 1u) {
                    const int rank = ns + __popcll(ms & below);
                    if (rank < NRUN) s_st[wv][r][rank] = c;
                }
                if ((word >> (16 + r)) & 1u) {
                    const int rank = ne + __popcll(me & below);
                    if (rank < NRUN) s_en[wv][r][rank] = c;
                }
                wave_sync();
                if (lane == 0) {
                    s_nst[wv][r] = min(NRUN, ns + __popcll(ms));
                    s_nen[wv][r] = min(NRUN, ne + __popcll(me));
                }
                wave_sync();
            }
        }
        __syncthreads();
        if (wv == 0) {
            // candidate index row*10+slot; nonempty (>= 2 points) ones in descending index
            // order (:222-240), one index per lane
            auto nth = [&](const int (&l)[NW][DEG][NRUN], const int (&n)[NW][DEG], int r,
                           int q) -> int {   // q-th start / end of row r over the waves
                for (int w = 0; w < NW; ++w) {
                    if (q < n[w][r]) return l[w][r][q];
                    q -= n[w][r];
                }
                return 0;
            };
            int nc = 0;
            for (int base = 0; base < DEG * NRUN; base += 64) {
                const int idx = DEG * NRUN - 1 - (base + lane);
                const int r = max(idx, 0) / NRUN, q = max(idx, 0) % NRUN;
                const int l = nth(s_st, s_nst, r, q), rr = nth(s_en, s_nen, r, q);
                const bool ok = idx >= 0 && ((open >> r) & 1u) && rr - l >= 2;
                const uint64_t m = __ballot(ok);
                const int rank = nc + __popcll(m & ((1ull << lane) - 1ull));
                if (ok && rank < NSEG) {
                    Seg sg;
                    sg.row = r;
                    sg.start = l;
                    sg.len = rr - l;
                    sg.par = ((fb[l] >> (16 + r)) & 1u) ? -1 : 1;
                    sg.empty = 0;
                    sg.length = 0.0;
                    sg.head = pt<DEG>(zb, l, r);
                    sg.tail = pt<DEG>(zb, rr - 1, r);
                    ExtCand& o = s_cand[rank];
                    o.s = sg;
                    auto get = [&](int k) { return seg_point<DEG>(zb, sg, k); };
                    head_line(get, sg.len - 1, o.h0, o.h1);
                    tail_line(get, sg.len - 1, 4 * M, o.t0, o.t1);
                }
                nc = min(NSEG, nc + __popcll(m));
            }
            if (lane >= nc && lane < NSEG) {
                ExtCand& o = s_cand[lane];
                o.s.empty = 1;
                o.s.len = 0;
                o.s.length = 0.0;
                o.s.par = 0;
                o.s.row = 0;
                o.s.start = 0;
                o.s.head = o.s.tail = o.h0 = o.h1 = o.t0 = o.t1 = cd{0.0, 0.0};
            }
            if (lane == 0) s_nc = nc;
        }
        __syncthreads();
        // segment lengths, a segment per wave in turn, lanes over points
        for (int q = wv; q < s_nc; q += NW) {
            const Seg sg = s_cand[q].s;
            double L = 0.0;
            for (int k = lane; k + 1 < sg.len; k += 64)
                L += sqrt(norm2(pt<DEG>(zb, sg.start + k + 1, sg.row) -
                                pt<DEG>(zb, sg.start + k, sg.row)));
            L = wave_sum(L);
            if (lane == 0) s_cand[q].s.length = L;
        }
        __syncthreads();
        if (wv == 0) {
            // stitching, 3 contours, merge scans of 20, 18, 16 (:495-667, :690); lane q < R
            // holds the q-th remaining segment
            int R = NSEG, id = lane < NSEG ? lane : 0;
            int maxm = 20;
            for (int ci = 0; ci < 3; ++ci, maxm -= 2) {
                // stable sort by length, empties (length 0) last
                {
                    const bool xe = s_cand[id].s.empty || s_cand[id].s.length == 0.0;
                    const double xl = s_cand[id].s.length;
                    s_ord[lane] = id;
                    wave_sync();
                    int rank = 0;
                    for (int p = 0; p < R; ++p) {
                        const Seg& o = s_cand[s_ord[p]].s;
                        const double yl = o.length;
                        const bool ye = o.empty || yl == 0.0;
                        // p sorts before this lane's segment
                        const bool before = xe != ye ? xe : (!xe && xl > yl);
                        const bool after = xe != ye ? ye : (!xe && yl > xl);
                        rank += (before || (!after && p < lane)) ? 1 : 0;
                    }
                    wave_sync();
                    if (lane < R) s_ord[rank] = id;
                    wave_sync();
                }
                const int i0 = s_ord[0];
                R -= 1;
                id = lane < R ? s_ord[lane + 1] : i0;
                wave_sync();
                const Seg c0 = s_cand[i0].s;
                ActSeg& act = s_con[ci];
                // the contour so far, the same in every lane; its pieces in LDS
                const int aempty = c0.empty;
                int np = 1, at_ = c0.empty ? 0 : c0.len - 1, apar = c0.par;
                if (lane == 0) act.pc[0] = Piece{c0.row, c0.start, c0.len, 0};
                wave_sync();
                cd ah = c0.head, at = c0.tail;  // its first and last point
                const ExtCand me = s_cand[id];
                cd head = me.s.head, tail = me.s.tail;
                bool empty = me.s.empty != 0 || lane >= R;
                for (int it = 0; it < maxm; ++it) {
                    if (__ballot(!empty) == 0ull) break;
                    // lines at the contour's ends (head_line, tail_line) from its points 0, 1, 2
                    // and t, t-1, t-2 and the last two of the reference's dense array, a
                    // lane each
                    cd e = cd{0.0, 0.0};
                    if (lane < 8 && !aempty) {
                        const int k =
                            lane < 3 ? lane : lane < 6 ? at_ - (lane - 3) : 4 * M - 8 + lane;
                        if (k >= 0 && k <= at_) e = contour_point<DEG>(zb, act.pc, np, k);
                    }
                    cd hx[3], tx[3];
#pragma unroll
                    for (int u = 0; u < 3; ++u) {
                        hx[u] = cd{__shfl(e.re, u, 64), __shfl(e.im, u, 64)};
                        tx[u] = cd{__shfl(e.re, 3 + u, 64), __shfl(e.im, 3 + u, 64)};
                    }
                    const bool hc = (norm2(hx[1] - hx[0]) > 1e-10) || (at_ <= 1);
                    cd ah0 = hc ? hx[1] : hx[2], ah1 = hc ? hx[0] : hx[1];
                    const bool tc = (at_ <= 1) || (norm2(tx[0] - tx[1]) > 1e-10);
                    // t = 0 clamps the line's start to point 0
                    cd at0 = tc ? (at_ == 0 ? tx[0] : tx[1]) : tx[2];
                    cd at1 = tc ? (at_ == 0 ? cd{0.0, 0.0} : tx[0]) : tx[1];
                    if ((tc ? at_ - 1 : at_ - 2) > 4 * M - 2) {   // the slice is clamped there
                        at0 = cd{__shfl(e.re, 6, 64), __shfl(e.im, 6, 64)};
                        at1 = cd{__shfl(e.re, 7, 64), __shfl(e.im, 7, 64)};
                    }
                    // the four connections of this lane's segment
                    double dd[4];
                    dd[0] = sqrt(norm2(at - head));
                    dd[1] = sqrt(norm2(ah - tail));
                    dd[2] = sqrt(norm2(ah - head));
                    dd[3] = sqrt(norm2(at - tail));
                    double best = 0.0;
                    int bf = -1;
                    if (!empty) {   // zero segments connect only within 1e-5 of 0
                        const bool same = apar * me.s.par > 0;
#pragma unroll
                        for (int ct = 0; ct < 4; ++ct) {
                            if ((ct < 2) != same) continue;
                            const bool hd = ct == 1 || ct == 2;   // at the contour's head
                            const bool sh = ct == 0 || ct == 2;   // at the segment's head
                            if ((bf < 0 || dd[ct] < best) &&
                                geom_condition(hd ? ah0 : at0, hd ? ah1 : at1,
                                               sh ? me.h0 : me.t0, sh ? me.h1 : me.t1)) {
                                best = dd[ct];
                                bf = ct * R + lane;
                            }
                        }
                    }
                    if (__ballot(bf >= 0) == 0ull) break;   // nothing connects, now or later
                    // nearest admissible connection by (distance, ctype-major index)
                    uint64_t bk = bf >= 0 ? (uint64_t)__double_as_longlong(best) : ~0ull;
                    int f = bf >= 0 ? bf : 0x7fffffff;
#pragma unroll
                    for (int off = 32; off >= 1; off >>= 1) {
                        const uint64_t ok = __shfl_xor(bk, off, 64);
                        const int of = __shfl_xor(f, off, 64);
                        if (ok < bk || (ok == bk && of < f)) {
                            bk = ok;
                            f = of;
                        }
                    }
                    // it has to be among the four nearest of all, empty ones included
                    int nearer = 0;
#pragma unroll
                    for (int ct = 0; ct < 4; ++ct) {
                        const uint64_t k = (uint64_t)__double_as_longlong(dd[ct]);
                        const bool nr = lane < R && (k < bk || (k == bk && ct * R + lane < f));
                        nearer += __popcll(__ballot(nr));
                    }
                    if (nearer >= 4 || np >= kExtMaxPieces) break;
                    const int ct = f / R, q = f % R;
                    const int qi = __shfl(id, q, 64);
                    const Seg sq = s_cand[qi].s;
                    if (ct == 0 || ct == 3) {   // T-H: act + s;  T-T: act + reversed s
                        if (lane == 0) act.pc[np] = Piece{sq.row, sq.start, sq.len, ct == 3};
                        at = ct == 0 ? sq.tail : sq.head;
                    } else {                    // H-T: s + act;  H-H: reversed s + act
                        Piece mv{0, 0, 0, 0};
                        if (lane < np) mv = act.pc[lane];
                        wave_sync();
                        if (lane < np) act.pc[lane + 1] = mv;
                        if (lane == 0) act.pc[0] = Piece{sq.row, sq.start, sq.len, ct == 2};
                        ah = (ct == 1) ? sq.head : sq.tail;
                        apar = (ct == 1) ? sq.par : -sq.par;
                    }
                    np += 1;
                    at_ += sq.len;
                    wave_sync();   // every lane has read the segment
                    if (lane == q) {
                        // the reference zeroes a merged segment (rest[i] = 0): its ends
                        // then rank by their distance from the origin, not as the
                        // contour's own ends
                        empty = true;
                        head = tail = cd{0.0, 0.0};
                        s_cand[qi].s.empty = 1;
                        s_cand[qi].s.head = cd{0.0, 0.0};
                        s_cand[qi].s.tail = cd{0.0, 0.0};
                    }
                    wave_sync();
                }
                if (lane == 0) {
                    act.np = np;
                    act.t = at_;
                    act.par = apar;
                    act.empty = aempty;
                }
                wave_sync();
            }
        }
        __syncthreads();
    }
    if (tid == 0) {
        C->closed = closed;
        C->open = all_closed ? 0 : 1;
    }
    if (!all_closed) {
        // the used pieces and the fields after them
        for (int ci = 0; ci < 3; ++ci) {
            if (tid < s_con[ci].np) C->con[ci].pc[tid] = s_con[ci].pc[tid];
            if (tid == 0) {
                C->con[ci].np = s_con[ci].np;
                C->con[ci].t = s_con[ci].t;
                C->con[ci].par = s_con[ci].par;
                C->con[ci].empty = s_con[ci].empty;
            }
        }
    }
}

// ---- contour integrals, magnification and its reverse mode (extended_source.py:
// 860-901; integrate.py:18-121)
template <int NL, bool LD, bool VJP, bool SUMS = false>
__global__ __launch_bounds__(kExtBlock)
__attribute__((amdgpu_waves_per_eu(VJP ? CAUS_EXT_VJP_WAVES : 3)))
void k_ext_integrate(ExtArgs A, int buf, int maxparts, int per_part) {
    constexpr int DEG = ext_degree<NL>();
    constexpr int ND = ext_nd<NL>();
    __shared__ double s_d[8];
    __shared__ double2 s_gl[2 * kExtGL];
    const int tid = threadIdx.x;
    // parts of one source are S workgroups apart, so that the first parts of the largest
    // sources start first
    const int64_t src = VJP ? blockIdx.x : blockIdx.x % A.S;
    const int part = VJP ? 0 : (int)(blockIdx.x / A.S);
    const ExtBatch B = ext_batch(A);
    const int parts = LD && !VJP ? min(maxparts, max(1, B.npts[src] / per_part)) : 1;
    if (SUMS ? parts == 1 : part >= parts) return;
    if (B.npts[src] == 0) {   // skipped source: zero magnification and gradient
        if (tid == 0) {
            A.mag[src] = 0.0;
            if (A.status) A.status[src] = 1;
        }
        if constexpr (VJP) {
            if (tid < ND) A.g_out[src * ND + tid] = 0.0;
        }
        return;
    }
    const int M = ext_points(B.npts[src], 10);
    LensFrame<NL> lf;
    cd w0;
    double rho;
    ext_source<NL>(A, src, lf, w0, rho);
    const double u1 = LD ? A.u1[src * A.u1stride] : 0.0;
    ExtWS W = ext_ws(ext_source_base<DEG>(A, src), DEG, A.mmax);
    GLNodes g{};
    if constexpr (LD && !SUMS) {
        g.n1 = A.npts_ld / 2;
        g.n2 = A.npts_ld - g.n1;
        g.a = s_gl;
        g.b = s_gl + kExtGL;
        for (int i = tid; i < 2 * kExtGL; i += kExtBlock) s_gl[i] = B.gl[i];
    }
    __syncthreads();
    const ZRows zb{W.z[buf], A.mmax};
    const uint32_t* fb = W.flg[buf];
    const double* thb = W.theta[buf];
    // the source's contours (extended_source.py:860-899): NL == 1 both images (tail index
    // N-1, :860-866); otherwise every closed image row, then the three stitched contours
    __shared__ ExtCEntry s_ct[kExtMaxContours];
    __shared__ Piece s_one[DEG];
    __shared__ int s_nc, s_T;
    if (tid == 0) {
        int nc = 0, off = 0;
        auto add = [&](const Piece* pc, int np, int L, int nterms, double cdiv, double par) {
            s_ct[nc] = ExtCEntry{pc, np, L, nterms, off, cdiv, par, 0.0, 0.0};
            off += L;
            ++nc;
        };
        if constexpr (NL == 1) {
            for (int r = 0; r < 2; ++r) {
                s_one[r] = Piece{r, 0, M, 0};
                add(&s_one[r], 1, M, M - 1, (double)M, ((fb[0] >> (16 + r)) & 1u) ? -1.0 : 1.0);
            }
        } else {
            const ExtContours* C = ext_contours<DEG>(A, src);
            const unsigned closed = C->closed;
            for (int r = 0; r < DEG; ++r) {
                if ((closed >> r) & 1u) {
                    s_one[r] = Piece{r, 0, M, 0};
                    add(&s_one[r], 1, M, M, (double)(M + 1),
                        ((fb[0] >> (16 + r)) & 1u) ? -1.0 : 1.0);
                }
            }
            if (C->open) {
                for (int ci = 0; ci < 3; ++ci) {
                    const ActSeg& a = C->con[ci];
                    const int L = a.empty ? 0 : a.t + 1;
                    add(a.pc, a.np, L, L, (double)(L + 1), (double)a.par);
                }
            }
        }
        s_nc = nc;
        s_T = off;
    }
    __syncthreads();
    const int nc = s_nc, T = s_T;
    double gacc[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) gacc[d] = 0.0;
    LDAdj<NL> adj;
    adj.zero();
    double total = 0.0;
    if constexpr (LD) {
        // the append-order points (buffer 0) are not read any more: the Q lines' cotangents
        const LDSource<NL> q = ld_source<NL>(lf, w0, rho, u1);
        total = integrate_source_ld<NL, DEG, VJP, SUMS>(
            zb, thb, s_ct, nc, T, W.pq, W.xy, reinterpret_cast<double*>(W.z[buf ^ 1]), W.yz, lf, q,
            g, adj, s_d, part, parts);
    } else {
        for (int c = 0; c < nc; ++c) {
            const ExtCEntry& e = s_ct[c];
            total += e.par * integrate_contour<NL, DEG>(zb, e.pc, e.np, e.L, e.nterms, s_d);
            if constexpr (VJP)
                contour_adjoint<NL, DEG>(zb, thb, e.pc, e.np, e.L, e.nterms, lf, e.par, adj);
        }
    }
    if (LD && !VJP && !SUMS && parts > 1) return;
    const unsigned long long npoints = (unsigned long long)T;
    const double m = fabs(total) / (kExtPi * rho * rho);
    if constexpr (VJP) {
        const double base = (total >= 0.0 ? 1.0 : -1.0) / (kExtPi * rho * rho);
        const double gm = A.g_mag[src];
        ExtTangents<NL> T;
        ext_tangents<NL>(A.params + src * A.pstride, T);
#pragma unroll
        for (int d = 0; d < ND; ++d)
            gacc[d] = adj.along(T.lt[d], lf.e, T.dw0[d], T.drho[d], T.du1[d]);
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            double v = block_sum(gacc[d], s_d) * base;
            if (d == 2) v -= 2.0 * m / rho;
            if (tid == 0) A.g_out[src * ND + d] = gm * v;
        }
    }
    if (tid == 0) {
        A.mag[src] = m;
        if (A.status) A.status[src] = B.fail[src] ? 0 : 1;
        if (A.work) atomicAdd(A.work + 4, npoints);
    }
}

int ext_flat_grid(int64_t max_lanes);

// Whether a batch is small enough for one limb point per group of lanes (k_ext_init_grouped,
// k_ext_refine).  A group's eight or sixteen lanes issue about twice (two lenses) and three
// times (three) the instructions of one lane per point, so it pays while the flat kernels
// leave the device mostly idle.  Whole calls on one MI355X, flat -> grouped, uniform disks: two
// lenses 337 -> 164 us (one source of 150 limb points), 462 -> 289 (400 of 200), 738 -> 628
// (1,200 of 256), 961 -> 1436 (4,000 of 200); three lenses 1181 -> 780, 2026 -> 1353,
// 2477 -> 2058, 3586 -> 5706.  Sources with sizes of their own count for less, since most are
// far below the largest: 1,000 of 256-1024 points 624 -> 484 (two) and 1617 -> 1597 us (three),
// 1,200 of 256-4096 1016 -> 1373 and 3666 -> 4860.
// A limit on the sweeps that could stop a converging solve keeps the one-lane solver, whose
// roots move one after the other: it counts, and needs, other sweeps than the group, whose roots
// move together, and which sources of a call converge must not depend on how many there are.  Of
// 4,800 sources at caustics (up to q3 = 1e-6) none needed more than 25 sweeps either way.
template <int NL>
bool ext_grouped(const ExtArgs& a) {
    constexpr int64_t tasks = 16000, sources = 1200;
    constexpr int itmax = 250;
    if (a.itmax < itmax) return false;
    const int64_t share = a.npts ? (NL == 3 ? 2 : 4) : 1;
    return a.S <= sources && a.S * a.nadd_max <= tasks * share;
}

// Limb points per workgroup of a source's limb-darkened line integrals without the reverse mode
// (a source of n takes n / that many workgroups; their sums follow in a second launch).  One
// workgroup of four waves issues less than half of a CU's FP64 rate and needs 1.5 ms for a
// source of 4096 points, so small batches are cut until they fill the 768 resident workgroups,
// and batches of up to two fillings into parts of 256 points, so that the largest sources do not
// outlast the rest.  Sources with sizes of their own or skipped ones count half.  One MI355X,
// whole calls, one workgroup a source -> this: 20 binary epochs of 200 points 324 -> 276 us,
// 500-epoch mag() event 485 -> 467 us, 1,300 epochs of 256-4096 points 3.1 -> 1.8 ms, three
// lenses 5.3 -> 3.3 ms; 2,100 epochs of 256-1024 points 1.87 ms either way.  With the reverse
// mode, sums that do not depend on the cut cost large batches 2-4%, so it is not cut.
inline int ext_per_part(const ExtArgs& a) {
    if (a.S > 2 * 768) return INT32_MAX;
    const int64_t busy = a.npts ? a.S / 2 : a.S;
    const int64_t fill = a.npts_def * busy / 768;
    return (int)(fill < 32 ? 32 : (fill > 256 ? 256 : fill));
}

// the launch sequence for one batch of nlenses = NL
template <int NL, int MODE, bool LD, bool VJP>
int ext_run(hipStream_t s, const ExtArgs& a) {
    const int64_t S = a.S;
    const unsigned nb = (unsigned)S;
    // points 0: a wave of 16 sources per workgroup while those are few, then full workgroups
    const int flanes = S <= 16 * 1024 ? 16 : kExtFlatBlock, ngl = LD ? a.npts_ld : 0;
    hipLaunchKernelGGL((k_ext_limb_init<NL, MODE>),
                       dim3((unsigned)((S + flanes - 1) / flanes + (LD ? 2 : 1))),
                       dim3(kExtFlatBlock), 0, s, a, 1, ngl, flanes);
    const int64_t lanes_init = S * (int64_t)((ext_npts_init(a.npts_def) + kExtPer - 1) / kExtPer);
    const bool grouped = MODE == MODE_FP64 && ext_grouped<NL>(a);
    // three lenses keep k_ext_limb_init: its coefficients' rounding decides the ill-conditioned
    // roots near a lens of small mass
    bool init_grouped = false;
    if constexpr (NL < 3) init_grouped = grouped;
    if (init_grouped) {
        constexpr int per_block = kExtBlock / ext_group<NL>();
        const int n0 = ext_npts_init(a.npts_def) - 1;
        const int per_source = n0 > per_block ? (n0 + per_block - 1) / per_block : 1;
        if constexpr (NL < 3)
            hipLaunchKernelGGL((k_ext_init_grouped<NL>), dim3(nb * per_source), dim3(kExtBlock), 0,
                               s, a, per_source);
    } else {
        hipLaunchKernelGGL((k_ext_limb_init<NL, MODE>), dim3(ext_flat_grid(lanes_init)),
                           dim3(kExtFlatBlock), 0, s, a, 0, 0, 0);
    }
    hipLaunchKernelGGL((k_ext_chain<NL, false>), dim3(nb), dim3(kExtBlock), 0, s, a, 0);  // initial
    const int add_grid = ext_flat_grid(S * (int64_t)(a.nadd_max > 0 ? a.nadd_max : 1));
    int cur = 0;
    if (grouped) {
        if (a.mmax <= kExtSelWave)
            hipLaunchKernelGGL((k_ext_refine<NL, kExtWaveBlock, kExtSelWave / 64>), dim3(nb),
                               dim3(kExtBlock), 0, s, a);
        else
            hipLaunchKernelGGL((k_ext_refine<NL, kExtBlock, kExtSortMax / kExtBlock>), dim3(nb),
                               dim3(kExtBlock), 0, s, a);
    } else {
        static_assert(kExtSelWave % 64 == 0 && kExtSortMax % kExtBlock == 0,
                      "select register tiles");
        for (int round = 0; round < 10; ++round) {
            // one wave while its 8 registers of keys hold the contour (no barrier in the
            // bisection); four waves of 16 above
            if (a.mmax <= kExtSelWave)
                hipLaunchKernelGGL((k_ext_select<NL, kExtWaveBlock, kExtSelWave / 64>), dim3(nb),
                                   dim3(kExtWaveBlock), 0, s, a, cur, round);
            else
                hipLaunchKernelGGL((k_ext_select<NL, kExtBlock, kExtSortMax / kExtBlock>), dim3(nb),
                                   dim3(kExtBlock), 0, s, a, cur, round);
            hipLaunchKernelGGL((k_ext_solve_add<NL, MODE>), dim3(add_grid), dim3(kExtFlatBlock), 0,
                               s, a, cur);
            cur ^= 1;
        }
    }
    hipLaunchKernelGGL((k_ext_chain<NL, true>), dim3(nb), dim3(kExtBlock), 0, s, a, cur);  // final
    if constexpr (NL > 1)
        hipLaunchKernelGGL((k_ext_contours<NL>), dim3(nb), dim3(kExtBlock), 0, s, a, 1);
    const int per_part = ext_per_part(a);
    const int parts = LD && !VJP ? min(kExtMaxParts, max(1, a.npts_def / per_part)) : 1;
    hipLaunchKernelGGL((k_ext_integrate<NL, LD, VJP>), dim3(nb * (unsigned)parts), dim3(kExtBlock),
                       0, s, a, 1, parts, per_part);
    if constexpr (LD && !VJP) {
        if (parts > 1)
            hipLaunchKernelGGL((k_ext_integrate<NL, LD, VJP, true>), dim3(nb), dim3(kExtBlock), 0,
                               s, a, 1, parts, per_part);
    }
    return hipGetLastError() == hipSuccess ? CAUS_OK : CAUS_ERR_LAUNCH;
}

template <int NL>
int mag_extended_nl(hipStream_t s, const ExtArgs& a, int mode, bool ld, bool vjp);

#define CAUS_EXT_CASE(NL, MODE, LD, VJP) return ext_run<NL, MODE, LD, VJP>(s, a);
#define CAUS_DEFINE_EXT(NL)                                                                     \
    template <>                                                                                 \
    int mag_extended_nl<NL>(hipStream_t s, const ExtArgs& a, int mode, bool ld, bool vjp) {     \
        const int m = mode == MODE_FP64 ? 0 : mode == MODE_FP64_COMP ? 1 : 2;                \
        switch (m * 4 + (ld ? 2 : 0) + (vjp ? 1 : 0)) {                                         \
            case 0: CAUS_EXT_CASE(NL, MODE_FP64, false, false)                                  \
            case 1: CAUS_EXT_CASE(NL, MODE_FP64, false, true)                                   \
            case 2: CAUS_EXT_CASE(NL, MODE_FP64, true, false)                                   \
            case 3: CAUS_EXT_CASE(NL, MODE_FP64, true, true)                                    \
            case 4: CAUS_EXT_CASE(NL, MODE_FP64_COMP, false, false)                             \
            case 5: CAUS_EXT_CASE(NL, MODE_FP64_COMP, false, true)                              \
            case 6: CAUS_EXT_CASE(NL, MODE_FP64_COMP, true, false)                              \
            case 7: CAUS_EXT_CASE(NL, MODE_FP64_COMP, true, true)                               \
            case 8: CAUS_EXT_CASE(NL, MODE_CF32, false, false)                                  \
            case 9: CAUS_EXT_CASE(NL, MODE_CF32, false, true)                                   \
            case 10: CAUS_EXT_CASE(NL, MODE_CF32, true, false)                                  \
            case 11: CAUS_EXT_CASE(NL, MODE_CF32, true, true)                                   \
            default:                                                                            \
                return CAUS_ERR_ARG;                                                            \
        }                                                                                       \
    }

}  // namespace caus
