// Greedy continuation of image rows along a sequence of points (reference:
// match_points, src/caustics/utils.py:15-40, chained as in extended_source.py:34-53 and
// point_source.py:1628-1640): point k+1's rows are permuted so that row i continues row
// i of point k, rows taking their nearest unused image in row order.
//
// P_k, the permutation that puts raw point k in order, obeys P_{k+1} = greedy(P_k).
// Where the nearest-neighbour map m_k between the raw points k and k+1 is a bijection,
// greedy(P_k) = m_k o P_k whatever the row order, so runs of such steps compose by an
// associative scan; only steps where two rows want one image (a few per cent on caustic
// crossings) depend on the carried order.  Three phases, one workgroup per sequence:
//   1. all waves: nearest-neighbour maps, one point per lane, and a segmented inclusive
//      scan over each 64 points (a conflict starts a segment), written as one word a point;
//   2. wave 0 walks the 64-point batches: one composition per batch, and per conflict a
//      scalar walk over the rows in which a row takes its nearest image if that is still
//      free and only otherwise looks for the nearest free one;
//   3. the caller reads P_k per point and gathers.
// Permutations are composed in bytes (v_perm_b32 picks four entries an instruction: 27
// instructions for ten rows) and stored in nibbles.
// Bound: phase 1 by FP64 issue (100 squared distances a point for ten rows) and the read of
// the points, phase 2 by latency.
#pragma once
#include "cplx.hpp"

namespace caus {

template <int DEG>
struct RowPerm {
    static constexpr int NW = (DEG + 3) / 4;
    uint32_t w[NW];   // byte i: entry i; bytes past DEG hold the identity
};

template <int DEG>
__device__ __forceinline__ RowPerm<DEG> rp_ident() {
    RowPerm<DEG> r;
#pragma unroll
    for (int t = 0; t < RowPerm<DEG>::NW; ++t) r.w[t] = 0x03020100u + 0x04040404u * (unsigned)t;
    return r;
}

// (a o b)[i] = a[b[i]]
template <int DEG>
__device__ __forceinline__ RowPerm<DEG> rp_compose(const RowPerm<DEG>& a, const RowPerm<DEG>& b) {
    static_assert(DEG <= 12, "entries fit twelve bytes");
    constexpr int NW = RowPerm<DEG>::NW;
    RowPerm<DEG> r;
#pragma unroll
    for (int t = 0; t < NW; ++t) {
        const uint32_t s = b.w[t];
        if constexpr (NW == 1) {
            r.w[t] = __builtin_amdgcn_perm(0u, a.w[0], s);
        } else if constexpr (NW == 2) {
            r.w[t] = __builtin_amdgcn_perm(a.w[1], a.w[0], s);
        } else {
            const uint32_t lo = __builtin_amdgcn_perm(a.w[1], a.w[0], s & 0x07070707u);
            const uint32_t hi = __builtin_amdgcn_perm(0u, a.w[2], s & 0x03030303u);
            const uint32_t m8 = s & 0x08080808u;              // entries 8..11
            const uint32_t mask = (m8 << 5) - (m8 >> 3);      // 0xFF in those bytes
            r.w[t] = (hi & mask) | (lo & ~mask);
        }
    }
    return r;
}

// nibble i of the word <-> byte i
template <int DEG>
__device__ __forceinline__ uint64_t rp_pack(const RowPerm<DEG>& p) {
    uint64_t o = 0;
#pragma unroll
    for (int t = 0; t < RowPerm<DEG>::NW; ++t) {
        uint32_t x = p.w[t];
        x = (x | (x >> 4)) & 0x00FF00FFu;
        x = (x | (x >> 8)) & 0xFFFFu;
        o |= (uint64_t)x << (16 * t);
    }
    return o;
}
template <int DEG>
__device__ __forceinline__ RowPerm<DEG> rp_unpack(uint64_t n) {
    RowPerm<DEG> r;
#pragma unroll
    for (int t = 0; t < RowPerm<DEG>::NW; ++t) {
        uint32_t x = (uint32_t)(n >> (16 * t)) & 0xFFFFu;
        x = (x | (x << 8)) & 0x00FF00FFu;
        r.w[t] = (x | (x << 4)) & 0x0F0F0F0Fu;
    }
    return r;
}
template <int DEG>
__device__ __forceinline__ uint64_t rp_ident_word() {
    return rp_pack<DEG>(rp_ident<DEG>());
}

constexpr uint64_t kChainConflict = 1ull << 63;  // two rows have one nearest image
constexpr uint64_t kChainSlow = 1ull << 62;      // a value is not finite: every row searches

// Nearest-neighbour map from the rows of raw point k - 1 to those of raw point k (ties
// to the lowest row), with the conflict bits.  The rows of point k are streamed.
template <int DEG, class Get, class IT>
__device__ __forceinline__ uint64_t chain_nn(Get get, IT k) {
    cd a[DEG];
    double fin = 0.0;   // stays 0 while every component is finite
#pragma unroll
    for (int i = 0; i < DEG; ++i) {
        a[i] = get(k - 1, i);
        fin = fma(a[i].re, 0.0, fma(a[i].im, 0.0, fin));
    }
    double best[DEG];
    int bj[DEG];
#pragma unroll
    for (int j = 0; j < DEG; ++j) {
        const cd b = get(k, j);
        fin = fma(b.re, 0.0, fma(b.im, 0.0, fin));
#pragma unroll
        for (int i = 0; i < DEG; ++i) {
            const double d = norm2(b - a[i]);
            if (j == 0 || d < best[i]) {
                best[i] = d;
                bj[i] = j;
            }
        }
    }
    unsigned hit = 0;
    uint64_t p = 0;
#pragma unroll
    for (int i = 0; i < DEG; ++i) {
        hit |= 1u << bj[i];
        p |= (uint64_t)bj[i] << (4 * i);
    }
    if (hit != (1u << DEG) - 1u) p |= kChainConflict;
    if (!(fin == 0.0)) p |= kChainConflict | kChainSlow;
    return p;
}

// greedy match_points of the carried rows (prev, nibbles) of point k - 1 against point
// k; all lanes of one wave call it with the same arguments.  e: chain_nn of the step.
// A row whose nearest image is free takes it.  Otherwise lanes 0..DEG-1 hold the
// distances to point k's rows and the nearest free one is found (ties to the lowest
// row; a distance that is not a number is taken only when it comes first, as a scan over
// the free rows in order does).
template <int DEG, class Get, class IT>
__device__ __forceinline__ uint64_t chain_greedy(Get get, IT k, uint64_t prev, uint64_t e) {
    const int lane = threadIdx.x & 63;
    unsigned used = 0;
    uint64_t p = 0;
    cd b = cd{0.0, 0.0};
    bool have = false;
#pragma unroll 1
    for (int i = 0; i < DEG; ++i) {
        const int row = (int)(prev >> (4 * i)) & 0xF;
        int j = (int)(e >> (4 * row)) & 0xF;
        if ((e & kChainSlow) || ((used >> j) & 1u)) {
            if (!have) {
                if (lane < DEG) b = get(k, lane);
                have = true;
            }
            const cd a = get(k - 1, row);
            const bool freeRow = lane < DEG && !((used >> lane) & 1u);
            const double d = freeRow ? norm2(b - a) : INFINITY;
            const uint64_t cand = __ballot(freeRow);
            const uint64_t nan = __ballot(freeRow && d != d);
            double m = d != d ? INFINITY : d;
#pragma unroll
            for (int off = 8; off >= 1; off >>= 1) m = fmin(m, __shfl_xor(m, off, 64));
            m = __shfl(m, 0, 64);
            const uint64_t at = __ballot(freeRow && d == m);
            const int first = __ffsll((long long)cand) - 1;
            j = ((nan >> first) & 1u) || at == 0 ? first : __ffsll((long long)at) - 1;
        }
        used |= 1u << j;
        p |= (uint64_t)j << (4 * i);
    }
    return p;
}

// Phases 1 and 2 for a workgroup of NT threads (whole waves) and points 0..M-1: get(k, i)
// is raw row i of point k, word(k) a reference to a 64-bit word per point that receives
// P_k in nibbles (row i of point k <- raw row P_k[i]).  Ends with a barrier.
template <int DEG, int NT, class Get, class Word, class IT>
__device__ __forceinline__ void chain_perms(Get get, Word word, IT M) {
    const int lane = threadIdx.x & 63;
    const uint64_t idw = rp_ident_word<DEG>();
    for (IT base = (IT)(threadIdx.x & ~63); base < M; base += NT) {
        const IT k = base + lane;
        const uint64_t e = (k > 0 && k < M) ? chain_nn<DEG>(get, k) : idw;
        RowPerm<DEG> x = (e & kChainConflict) ? rp_ident<DEG>() : rp_unpack<DEG>(e);
        int head = (e & kChainConflict) ? 1 : 0;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            RowPerm<DEG> o;
#pragma unroll
            for (int t = 0; t < RowPerm<DEG>::NW; ++t) o.w[t] = __shfl_up(x.w[t], off, 64);
            const int oh = __shfl_up(head, off, 64);
            if (lane >= off && !head) {
                x = rp_compose<DEG>(x, o);
                head = oh;
            }
        }
        if (k < M) word(k) = (e & kChainConflict) ? e : rp_pack<DEG>(x);
    }
    __syncthreads();
    if (threadIdx.x < 64) {
        RowPerm<DEG> S = rp_ident<DEG>();   // P at the last point of the batch before
        uint64_t nw = lane < M ? word((IT)lane) : idw;
        for (IT base = 0; base < M; base += 64) {
            const IT k = base + lane;
            const uint64_t e = nw;
            nw = k + 64 < M ? word(k + 64) : idw;
            uint64_t rem = __ballot((e & kChainConflict) != 0);
            const RowPerm<DEG> x = (e & kChainConflict) ? rp_ident<DEG>() : rp_unpack<DEG>(e);
            RowPerm<DEG> P = rp_compose<DEG>(x, S);
            while (rem) {
                const int c = __ffsll((long long)rem) - 1;
                rem &= rem - 1;
                RowPerm<DEG> prev = S;
                if (c > 0) {
#pragma unroll
                    for (int t = 0; t < RowPerm<DEG>::NW; ++t)
                        prev.w[t] = __builtin_amdgcn_readlane(P.w[t], c - 1);
                }
                const uint64_t ec =
                    (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)e, c) |
                    ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(e >> 32), c)
                     << 32);
                const uint64_t g = chain_greedy<DEG>(get, base + c, rp_pack<DEG>(prev), ec);
                const RowPerm<DEG> G = rp_unpack<DEG>(g);
                if (lane >= c) P = rp_compose<DEG>(x, G);
            }
            if (k < M) word(k) = rp_pack<DEG>(P);
            const int last = M - base < 64 ? (int)(M - base) - 1 : 63;
#pragma unroll
            for (int t = 0; t < RowPerm<DEG>::NW; ++t)
                S.w[t] = __builtin_amdgcn_readlane(P.w[t], last);
        }
    }
    __syncthreads();
}

}  // namespace caus
