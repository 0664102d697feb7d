// p4g_site.h -- device functions the pruning kernels share: the site
// likelihood at the root and the weighted sum over sites.
#pragma once

#include "p4g_internal.h"

namespace p4g {

constexpr float SCALE_THRESH = 5.9604645e-08f;  // 2^-24

// s_waitcnt vmcnt(0) with the other counters left alone (gfx9 encoding:
// vmcnt bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8)
constexpr int VMCNT0 = 0x0F70;

// Site likelihood of pattern p from the root's category-summed
// sum_s pi_s cl_s (Lk) and the pattern's scale exponent e, as
// Pf/p4_tree.c:1029-1197: (1 - pInvar)/K * Lk plus the invariant-site term,
// or Lk/K without pInvar; adds count * log(like) to contrib.  In FP32 mode
// the partials carry 2^-e, so the variable-site part is unscaled in FP64
// before the invariant part is added; with no invariant part the log is
// taken in the scaled domain.
template <bool SCALE>
__device__ __forceinline__ void siteLogLike(const PruneArgs &a, double Lk, int e, int p, int K,
                                            const double *pi, double &contrib, int &bad)
{
    const size_t nPatPad = (size_t)a.nPatPad;
    const double LN2 = 0.69314718055994530942;
    double like, lnl;
    bool ok;
    if (a.pInvar != 0.0) {
        const double varS = Lk * ((1.0 - a.pInvar) / (double)K);
        double inv = 0.0;
        for (int w = 0; w < a.nWords; w++) {
            uint32_t mw = a.invMask[(size_t)w * nPatPad + p];
            while (mw) {
                const int b = __ffs(mw) - 1;
                mw &= mw - 1;
                inv += pi[w * 32 + b] * a.pInvar;
            }
        }
        if (SCALE && e != 0 && inv == 0.0) {
            ok = varS > 0.0;
            lnl = log(varS) - (double)e * LN2;
            like = ldexp(varS, -e);
        } else {
            like = ((SCALE && e != 0) ? ldexp(varS, -e) : varS) + inv;
            ok = like > 0.0;
            lnl = log(like);
        }
    } else {
        const double likeS = (K > 1) ? Lk / (double)K : Lk;
        ok = likeS > 0.0;
        lnl = log(likeS);
        like = likeS;
        if (SCALE && e != 0) {
            lnl -= (double)e * LN2;
            like = ldexp(likeS, -e);
        }
    }
    if (p < a.nPat) {
        if (!ok) bad = 1;
        contrib = a.counts[p] * lnl;
        if (a.patLikes) a.patLikes[p] = like;
    }
}

// The exponent a category brings to the root's common one: e, or none if its
// likelihood L is exactly 0.  Such a category was not rescaled from the point
// where its partial became 0, and its small exponent would shift the others
// out of a double's range.
constexpr int NO_EXPONENT = 0x3fffffff;
template <bool SCALE> __device__ __forceinline__ int rootExponent(double L, int e)
{
    return SCALE && L == 0.0 ? NO_EXPONENT : e;   // (a NaN keeps its place in the sum)
}

// A pattern's category sum, sum_k L(k) 2^-E(k), as the returned value times
// 2^-e; E as rootExponent gives it, e the smallest (NO_EXPONENT: the sum is 0).
template <bool SCALE, typename FL, typename FE>
__device__ __forceinline__ double sumCategories(int K, FL L, FE E, int &e)
{
    e = SCALE ? E(0) : 0;
    if (SCALE)
        for (int k = 1; k < K; k++) e = min(e, E(k));
    double sum = 0.0;
    for (int k = 0; k < K; k++) sum += SCALE ? ldexp(L(k), e - E(k)) : L(k);
    return sum;
}

// A workgroup's sum and flag for the workgroup that will add them all, and
// its ticket.  The two stores are agent-scope atomics (written through to
// memory) and acknowledged before the ticket is drawn, which is all the
// reader's agent-scope loads need.  A release fence in their place writes the
// XCD's whole L2 back to memory, once per workgroup, with the other
// workgroups' partials dirty in it: dirty paths of 24 parts x 4 chains took
// 303 us in the 4-state kernel with it and take 104 us, a 64-taxon,
// 38,184-pattern FP32 evaluation 88 us and 70.
__device__ __forceinline__ unsigned postBlockSum(const PruneArgs &a, double contrib, int bad, int blk)
{
    __hip_atomic_store(a.blockSums + blk, contrib, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(a.blockBad + blk, bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
    return __hip_atomic_fetch_add(a.counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The last workgroup of the item sums the per-workgroup partials (wave 0
// of each workgroup reports) in a fixed order with Neumaier compensation.
__device__ __forceinline__ void finishSiteSumWave(const PruneArgs &a, double contrib, int bad, int blk, int nBlk)
{
    const int lane = threadIdx.x & 63;
    for (int off = 32; off >= 1; off >>= 1) {
        contrib += __shfl_xor(contrib, off);
        bad |= __shfl_xor(bad, off);
    }
    unsigned prev = 0;
    if (lane == 0) prev = postBlockSum(a, contrib, bad, blk);
    prev = __shfl(prev, 0);
    if (prev != (unsigned)(nBlk - 1)) return;
    __threadfence();
    double s = 0.0, comp = 0.0;
    int b = 0;
    for (int i = lane; i < nBlk; i += 64) {
        const double x = __hip_atomic_load(a.blockSums + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        b |= __hip_atomic_load(a.blockBad + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const double t = s + x;  // Neumaier
        if (fabs(s) >= fabs(x))
            comp += (s - t) + x;
        else
            comp += (x - t) + s;
        s = t;
    }
    double v = s + comp;
    for (int off = 32; off >= 1; off >>= 1) {
        v += __shfl_xor(v, off);
        b |= __shfl_xor(b, off);
    }
    if (lane == 0) {
        a.result[0] = b ? -1.0e99 : v;
        a.result[1] = (double)b;
        *a.counter = 0u;
    }
}

}  // namespace p4g
