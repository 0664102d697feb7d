// p4g_deriv.hip -- branch-length derivatives of the log likelihood and the
// up-pass ("cl2") conditional likelihoods they need, in FP64.
//
//  k_pderiv       P' = r Q P and P'' = r^2 Q Q P for every (node, category),
//                 one thread per entry, from Q of the node's (comp, rMatrix)
//                 and the node's P (the reference evaluates the same
//                 derivatives as V diag(r lam e^(lam t)) V^-1,
//                 Pf/eig.c:294-395, called from Pf/p4_node.c:442-540).
//  k_edgeDerivs4, k_edgeDerivs20, k_edgeDerivs
//                 ONE launch per part for every branch: a wave owns the
//                 patterns of a tile in one gamma category and walks the
//                 tree in preorder.  For child n of node m it forms cl2[n] --
//                 the likelihood of everything outside n's subtree given the
//                 state of m -- from m's cl2 through m's P (or the root
//                 frequencies) times the siblings' downward messages
//                 (Pf/p4_node.c:858-1018 with the dispatch of
//                 Pf/p4_treeNewt.c:597-620), then the site likelihood across
//                 n's branch and its first and second derivatives with P, P'
//                 and P'' (Pf/p4_treeNewt.c:257-500).  The category waves of
//                 a workgroup combine each pattern's categories in LDS;
//                 per-workgroup sums go to a buffer.  k_edgeDerivs4 serves
//                 the 4-state wave layout, k_edgeDerivs20 the 20-state tiles
//                 (on the FP64 matrix cores), k_edgeDerivs everything else.
//  k_derivReduce  per node, the workgroups' sums in a fixed order with
//                 Neumaier compensation.
#include "p4g_internal.h"

#include <cmath>

namespace p4g {

// One workgroup per (node, category), Q, P^T and Q P staged in LDS: read from
// L2 per entry, the 20-state products were a chain of 400 dependent loads
// (103 us for 376 matrices).
__global__ __launch_bounds__(256) void k_pderiv(DerivPArgs a)
{
    extern __shared__ double pdSm[];   // [3][S][S]: Q, P^T, Q P
    const int S = a.dim, SS = S * S;
    const int it = blockIdx.x / a.K, k = blockIdx.x - it * a.K;
    const int node = a.nodeList[it];
    const double r = a.rateFac[(size_t)it * a.K + k];
    const double *Q = a.Q + (size_t)a.eigSlot[it] * SS;
    const size_t m0 = (size_t)node * a.K + k;
    const double *PT = a.PT64 + m0 * SS;   // PT[j][s] = P[s][j]
    double *sQ = pdSm, *sP = sQ + SS, *sQP = sP + SS;
    for (int e = threadIdx.x; e < SS; e += 256) {
        sQ[e] = Q[e];
        sP[e] = PT[e];
    }
    __syncthreads();
    // QP[m][j] = sum_l Q[m][l] P[l][j]; P' = r Q P; P'' = r^2 Q QP
    for (int e = threadIdx.x; e < SS; e += 256) {
        const int m = e / S, j = e - m * S;
        double v = 0.0;
        for (int l = 0; l < S; l++) v += sQ[m * S + l] * sP[j * S + l];
        sQP[e] = v;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < SS; e += 256) {
        const int j = e / S, s = e - j * S;   // stored transposed, like P^T
        double v = 0.0;
        for (int m = 0; m < S; m++) v += sQ[s * S + m] * sQP[m * S + j];
        const double p1 = r * sQP[s * S + j], p2 = r * r * v;
        a.P1T[m0 * SS + e] = p1;
        a.P2T[m0 * SS + e] = p2;
        if (a.D) {
            double *D = a.D + m0 * (3 * AA_MAT);
            D[aaPaIndex(j, s, false)] = sP[e];   // P^T: row j, column s
            D[AA_MAT + aaPaIndex(s, j, false)] = p1;
            D[2 * AA_MAT + aaPaIndex(s, j, false)] = p2;
        }
    }
}

hipError_t launchPderiv(const DerivPArgs &a, hipStream_t s)
{
    if (a.nItems <= 0) return hipSuccess;
    const size_t lds = sizeof(double) * 3 * a.dim * a.dim;
    if (lds > 64 * 1024) {   // more than 64 KB of LDS has to be asked for
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_pderiv),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k_pderiv, dim3(a.nItems * a.K), dim3(256), lds, s, a);
    return hipGetLastError();
}

// A pattern's category sums to its weighted lnL, d1 and d2 (Pf/p4_treeNewt.c:
// 257-500), with the penalty for an impossible site.
__device__ __forceinline__ void siteDerivs(const DerivArgs &a, int p, double likeS, double firstS, double secondS,
                                           double &lnL, double &d1, double &d2)
{
    const int K = a.K;
    const double *pi = a.rootPi;
    if (a.pInvar != 0.0) {
        const double f = (1.0 - a.pInvar) / (double)K;
        likeS *= f;
        firstS *= f;
        secondS *= f;
        for (int w = 0; w < a.nWords; w++) {
            uint32_t mw = a.invMask[(size_t)w * a.nPatPad + p];
            while (mw) {
                const int b = __ffs(mw) - 1;
                mw &= mw - 1;
                likeS += pi[w * 32 + b] * a.pInvar;
            }
        }
    } else if (K > 1) {
        likeS /= (double)K;
        firstS /= (double)K;
        secondS /= (double)K;
    }
    const double cnt = a.counts[p];
    if (likeS < 1.0e-300) {
        lnL = cnt * -100000.0;
        d1 = cnt * 1000000.0;
        d2 = cnt * 10000000.0;
    } else {
        lnL = cnt * log(likeS);
        d1 = cnt * (firstS / likeS);
        d2 = cnt * ((secondS * likeS - firstS * firstS) / (likeS * likeS));
    }
}

// The unit kernels keep the category values of DERIV_BATCH branches in LDS
// and finish them together, branch b of a batch by wave b % K: one pair of
// barriers per two units instead of two per branch, and the logarithms and
// divisions of a batch run on all waves instead of one.  Q: lanes that hold
// parts of one pattern's sums (1 or 4, 64 / Q lanes apart).
constexpr int DERIV_BATCH = 4;
template <int Q>
__device__ __forceinline__ void flushBatch(const DerivArgs &a, double (*red)[3][64], const int *outIdx, int n)
{
    const int K = a.K, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    __syncthreads();
    for (int b = wave; b < n; b += K) {
        double v[3] = {0.0, 0.0, 0.0};
        for (int k = 0; k < K; k++)
            for (int c = 0; c < 3; c++) v[c] += red[b * K + k][c][lane];
        for (int off = 64 / Q; off < 64; off <<= 1)
            for (int c = 0; c < 3; c++) v[c] += __shfl_xor(v[c], off);
        const int p = (int)blockIdx.x * (64 / Q) + lane % (64 / Q);
        double s[3] = {0.0, 0.0, 0.0};
        if (lane < 64 / Q && p < a.nPat) siteDerivs(a, p, v[0], v[1], v[2], s[0], s[1], s[2]);
        for (int off = 32 / Q; off >= 1; off >>= 1)
            for (int c = 0; c < 3; c++) s[c] += __shfl_xor(s[c], off);
        if (lane == 0) {
            double *o = a.partial + ((size_t)outIdx[b] * gridDim.x + blockIdx.x) * 3;
            for (int c = 0; c < 3; c++) o[c] = s[c];
        }
    }
    __syncthreads();
}

typedef const __attribute__((address_space(4))) int dcint;
typedef const __attribute__((address_space(4))) double dcdouble;
// (unit records and matrices were written before the launch: scalar loads)
__device__ __forceinline__ DerivUnit derivUnit(const DerivArgs &a, int i)
{
    dcint *u = (dcint *)a.units + 16 * i;
    DerivUnit r;
    r.nKids = u[0];
    r.src = u[1];
    r.parent = u[2];
    r.out = u[3];
#pragma unroll
    for (int c = 0; c < 2; c++) {
        r.node[c] = u[4 + c];
        r.tip[c] = u[6 + c];
        r.idx[c] = u[8 + c];
    }
    r.sibStart = u[10];
    r.nSib = u[11];
#pragma unroll
    for (int c = 0; c < 2; c++) {
        r.item[c] = u[12 + c];
        r.eig[c] = u[14 + c];
    }
    return r;
}

typedef double dvD4 __attribute__((ext_vector_type(4)));

// 4 states, wave layout: lane = pattern.  Bound by memory: per pattern and
// category every down partial is read once and every cl2 written once and,
// unless the next unit is its node, read once.  A unit's loads are issued
// one unit ahead and before that unit's stores; the matrices come by scalar
// loads, and of P, P' and P'' only P: with the message M = P x, P' x is r Q M
// and P'' x is r^2 Q Q M, and the few Q stay in the scalar cache.  38,184
// patterns, 4 categories, 126 nodes: 359 us, 1.2 GB at 3.4 TB/s (one branch at
// a time, with vector loads of P, P' and P'', two barriers per branch and the
// logarithms on one wave of four: 780 us).
__global__ __launch_bounds__(64 * WAVE_MAX_K) void k_edgeDerivs4(DerivArgs a)
{
    extern __shared__ double dvSm[];   // [DERIV_BATCH][K][3][64]
    double (*red)[3][64] = reinterpret_cast<double (*)[3][64]>(dvSm);
    __shared__ unsigned char ambL[256];
    const int K = a.K;
    const int cat = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int p = blockIdx.x * 64 + lane;
    const size_t nPP = (size_t)a.nPatPad;
    for (int j = threadIdx.x; j < a.nAmb && j < 256; j += blockDim.x) ambL[j] = (unsigned char)(a.ambMask[j] & 15u);
    __syncthreads();
    auto mat = [&](int node) -> dcdouble * { return (dcdouble *)a.PT64 + ((size_t)node * K + cat) * 16; };
    auto clAt = [&](int slot) { return *(const dvD4 *)(a.cl + (((size_t)slot * K + cat) * nPP + p) * 4); };
    auto cl2At = [&](int node) -> dvD4 * { return (dvD4 *)(a.cl2 + (((size_t)node * K + cat) * nPP + p) * 4); };
    auto codeAt = [&](int row) -> unsigned { return a.tips[(size_t)row * nPP + p]; };
    // M x (P^T stored: M[s][j] at j * 4 + s)
    auto apply = [&](dcdouble *M, const dvD4 &x) -> dvD4 {
        dvD4 v = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int s = 0; s < 4; s++) v[s] += x[j] * M[j * 4 + s];
        return v;
    };
    // the column of a tip's code; a gap: 1 for every state
    auto column = [&](dcdouble *M, unsigned code) -> dvD4 {
        const bool b0 = code & 1u, b1 = code & 2u;
        dvD4 v;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const double lo = b0 ? M[4 + s] : M[s], hi = b0 ? M[12 + s] : M[8 + s];
            v[s] = b1 ? hi : lo;
        }
        if (code >= 4u) {
            const unsigned m = code == TIP_ALL ? 0u : ambL[code - 4];
#pragma unroll
            for (int s = 0; s < 4; s++) {
                double x = 0.0;
#pragma unroll
                for (int j = 0; j < 4; j++) x += ((m >> j) & 1u) ? M[j * 4 + s] : 0.0;
                v[s] = code == TIP_ALL ? 1.0 : x;
            }
        }
        return v;
    };
    struct Kid {
        dvD4 x;
        unsigned code;
    };
    auto message = [&](int node, int tip, const Kid &kd) -> dvD4 {
        return tip ? column(mat(node), kd.code) : apply(mat(node), kd.x);
    };
    // a unit's loads; what a child does not need reads the part's first slot or row
    auto load = [&](const DerivUnit &u, Kid (&kd)[2], dvD4 &up) {
#pragma unroll
        for (int c = 0; c < 2; c++) {
            kd[c].x = clAt(u.tip[c] ? 0 : u.idx[c]);
            kd[c].code = codeAt(u.tip[c] ? u.idx[c] : 0);
        }
        up = *cl2At(u.src == DU_HBM ? u.parent : u.node[0]);
    };
    dvD4 prev = {0.0, 0.0, 0.0, 0.0};   // cl2 of the previous unit's child that the next unit may continue from
    __shared__ int outIdx[DERIV_BATCH];
    int nB = 0;
    // one branch: its sums to the batch, its cl2 to HBM
    auto branch = [&](int node, int item, int eig, const dvD4 &c2, const dvD4 &M, int out) {
        const double r = ((dcdouble *)a.rateFac)[(size_t)item * K + cat];
        dcdouble *Q = (dcdouble *)a.Q + 16 * eig;
        dvD4 q1;
        double like = 0.0, first = 0.0, second = 0.0;
#pragma unroll
        for (int s = 0; s < 4; s++) q1[s] = Q[4 * s] * M[0] + Q[4 * s + 1] * M[1] + Q[4 * s + 2] * M[2] + Q[4 * s + 3] * M[3];
#pragma unroll
        for (int s = 0; s < 4; s++) {
            like += c2[s] * M[s];
            first += c2[s] * q1[s];
            second += c2[s] * (Q[4 * s] * q1[0] + Q[4 * s + 1] * q1[1] + Q[4 * s + 2] * q1[2] + Q[4 * s + 3] * q1[3]);
        }
        red[nB * K + cat][0][lane] = like;
        red[nB * K + cat][1][lane] = first * r;
        red[nB * K + cat][2][lane] = second * (r * r);
        if (threadIdx.x == 0) outIdx[nB] = out;
        nB++;
        *cl2At(node) = c2;
    };
    uint64_t rm = ~0ull;
    if (a.rootLeafRow >= 0) {
        const unsigned code = codeAt(a.rootLeafRow);
        rm = code < 4u ? 1ull << code : code == TIP_ALL ? ~0ull : a.ambMask[code - 4];
    }
    // the root frequencies (Pf/p4_node.c:858-879); a leaf root's own data
    // enters here too
    dvD4 root;
#pragma unroll
    for (int s = 0; s < 4; s++) root[s] = ((rm >> s) & 1ull) ? a.rootPi[s] : 0.0;
    auto unit = [&](const DerivUnit &u, int next, const Kid (&kd)[2], const dvD4 &up) {   // next: the next unit's src
        if (nB + u.nKids > DERIV_BATCH) {
            flushBatch<1>(a, red, outIdx, nB);
            nB = 0;
        }
        dvD4 av = root;
        if (u.src != DU_ROOT) {
            // up through the parent's branch: sum_f cl2[parent][f] P[f][s]
            // (Pf/p4_node.c:883-937)
            dvD4 x;
#pragma unroll
            for (int s = 0; s < 4; s++) x[s] = u.src == DU_HBM ? up[s] : prev[s];
            dcdouble *P = mat(u.parent);
#pragma unroll
            for (int s = 0; s < 4; s++) av[s] = P[4 * s] * x[0] + P[4 * s + 1] * x[1] + P[4 * s + 2] * x[2] + P[4 * s + 3] * x[3];
        }
        const dvD4 M0 = message(u.node[0], u.tip[0], kd[0]);
        if (u.nKids == 2) {
            const dvD4 M1 = message(u.node[1], u.tip[1], kd[1]);
            const dvD4 c0 = av * M1, c1 = av * M0;
            branch(u.node[0], u.item[0], u.eig[0], c0, M0, u.out);
            branch(u.node[1], u.item[1], u.eig[1], c1, M1, u.out + 1);
#pragma unroll
            for (int s = 0; s < 4; s++) prev[s] = next == DU_PREV0 ? c0[s] : c1[s];
        } else {
            for (int q = 0; q < u.nSib; q++) {
                const DerivSib sb = a.sibs[u.sibStart + q];
                Kid k2{};
                if (sb.kind == 0)
                    k2.code = codeAt(sb.idx);
                else
                    k2.x = clAt(sb.idx);
                av *= message(sb.pnode, sb.kind == 0, k2);
            }
            branch(u.node[0], u.item[0], u.eig[0], av, M0, u.out);
            prev = av;
        }
    };
    DerivUnit u = derivUnit(a, 0);
    Kid A[2], B[2];
    dvD4 ua, ub;
    load(u, A, ua);
    for (int i = 0; i < a.nUnits; i += 2) {
        DerivUnit n = derivUnit(a, min(i + 1, a.nUnits - 1));
        load(n, B, ub);
        unit(u, n.src, A, ua);
        if (i + 1 >= a.nUnits) break;
        u = derivUnit(a, min(i + 2, a.nUnits - 1));
        load(u, A, ua);
        unit(n, u.src, B, ub);
    }
    flushBatch<1>(a, red, outIdx, nB);
}

// 20 states, tiles of 16 patterns: the layout and the matrix products of the
// pruning kernel (p4g_aa.hip), FP64: register r of lane (q, p) is state 4q + r
// of pattern p, register 4 state 16 + q.  Bound by the products: per node
// with two children up to seven (its P^T, and P, P' and P'' of each internal
// child), each ten v_mfma_f64_16x16x4f64 with the 20 rows padded to 32.
// 48 taxa x 2,003 patterns, 4 categories: 217 us (one lane per pattern and
// category, with register arrays in scratch memory: 10.2 ms).
struct DvPart {
    dvD4 x;
    double x4;
};
template <bool TIPLDS>
__global__ __launch_bounds__(64 * WAVE_MAX_K) __attribute__((amdgpu_waves_per_eu(2))) void k_edgeDerivs20(DerivArgs a)
{
    // [DERIV_BATCH][K][3][64], [nTax][16] tip codes
    extern __shared__ double dvSm[];
    double (*red)[3][64] = reinterpret_cast<double (*)[3][64]>(dvSm);
    __shared__ int outIdx[DERIV_BATCH];
    __shared__ unsigned ambL[256];
    const int K = a.K;
    const int cat = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, q = lane >> 4, pl = lane & 15;
    const int tile = blockIdx.x, p = tile * AA_TILE + pl;
    const size_t nPP = (size_t)a.nPatPad;
    const size_t nT = nPP / AA_TILE;
    uint8_t *tipL = (uint8_t *)(dvSm + DERIV_BATCH * K * 192);
    for (int j = threadIdx.x; j < a.nAmb && j < 256; j += blockDim.x) ambL[j] = (unsigned)a.ambMask[j];
    if (TIPLDS)
        for (int t = threadIdx.x; t < a.nTax; t += blockDim.x)
            *reinterpret_cast<uint4 *>(tipL + t * AA_TILE) =
                *reinterpret_cast<const uint4 *>(a.tips + (size_t)t * nPP + (size_t)tile * AA_TILE);
    __syncthreads();
    auto codeAt = [&](int row) -> unsigned { return TIPLDS ? tipL[row * AA_TILE + pl] : a.tips[(size_t)row * nPP + p]; };
    auto region = [&](size_t slot) -> size_t { return ((slot * nT + tile) * K + cat) * AA_PART; };
    typedef double d2v __attribute__((ext_vector_type(2)));
    auto loadPart = [&](const double *R) -> DvPart {
        const d2v lo = *(const d2v *)(R + lane * 2), hi = *(const d2v *)(R + 128 + lane * 2);
        return DvPart{dvD4{lo.x, lo.y, hi.x, hi.y}, R[256 + lane]};
    };
    struct Mat {
        dvD4 a0, a1;
        double b0, b1;
    };
    auto loadMat = [&](const double *M) -> Mat {
        return Mat{*(const dvD4 *)(M + lane * 4), *(const dvD4 *)(M + 320 + (q * 4 + (pl & 3)) * 4), M[256 + lane],
                   M[384 + q * 4 + (pl & 3)]};
    };
    constexpr int PS = aaMatStride(false);   // stride of the operand table (D's matrices are packed)
    const double *PA = a.PA + (size_t)cat * PS, *D = a.D + (size_t)cat * (3 * AA_MAT);
    auto matP = [&](int node) { return PA + (size_t)node * K * PS; };
    auto matD = [&](int node, int which) { return D + (size_t)node * K * (3 * AA_MAT) + which * AA_MAT; };
    auto product = [&](const Mat &m, const DvPart &y) -> DvPart {
        dvD4 d0 = {0, 0, 0, 0}, d1 = {0, 0, 0, 0};
#pragma unroll
        for (int t = 0; t < 4; t++) {
            d0 = __builtin_amdgcn_mfma_f64_16x16x4f64(m.a0[t], y.x[t], d0, 0, 0, 0);
            d1 = __builtin_amdgcn_mfma_f64_16x16x4f64(m.a1[t], y.x[t], d1, 0, 0, 0);
        }
        d0 = __builtin_amdgcn_mfma_f64_16x16x4f64(m.b0, y.x4, d0, 0, 0, 0);
        d1 = __builtin_amdgcn_mfma_f64_16x16x4f64(m.b1, y.x4, d1, 0, 0, 0);
        return DvPart{d0, d1[0]};
    };
    // the column of a tip's code from the transposed matrices; a gap: `all`
    auto column = [&](const double *base, int node, unsigned code, double all) -> DvPart {
        const double *T = base + ((size_t)node * K + cat) * (AA_S * AA_S);
        const unsigned j = code < (unsigned)AA_S ? code : 0u;
        DvPart v{*(const dvD4 *)(T + j * AA_S + 4 * q), T[j * AA_S + 16 + q]};
        if (code == TIP_ALL) {
            v = DvPart{dvD4{all, all, all, all}, all};
        } else if (code >= (unsigned)AA_S) {
            const unsigned m = ambL[code - AA_S];
            v = DvPart{dvD4{0, 0, 0, 0}, 0.0};
#pragma unroll 1
            for (int i = 0; i < AA_S; i++)
                if ((m >> i) & 1u) {
                    v.x += *(const dvD4 *)(T + i * AA_S + 4 * q);
                    v.x4 += T[i * AA_S + 16 + q];
                }
        }
        return v;
    };
    auto dot = [&](const DvPart &u, const DvPart &v) {
        return u.x[0] * v.x[0] + u.x[1] * v.x[1] + u.x[2] * v.x[2] + u.x[3] * v.x[3] + u.x4 * v.x4;
    };
    auto times = [&](const DvPart &u, const DvPart &v) { return DvPart{u.x * v.x, u.x4 * v.x4}; };
    int nB = 0;
    // M: the child's message; d1, d2: P' and P'' times its partial
    auto branch = [&](int node, const DvPart &c2, const DvPart &M, const DvPart &d1, const DvPart &d2, int out) {
        red[nB * K + cat][0][lane] = dot(c2, M);
        red[nB * K + cat][1][lane] = dot(c2, d1);
        red[nB * K + cat][2][lane] = dot(c2, d2);
        if (threadIdx.x == 0) outIdx[nB] = out;
        nB++;
        double *R = a.cl2 + region((size_t)node);
        *(d2v *)(R + lane * 2) = d2v{c2.x[0], c2.x[1]};
        *(d2v *)(R + 128 + lane * 2) = d2v{c2.x[2], c2.x[3]};
        R[256 + lane] = c2.x4;
    };
    // child c: message, P' and P'' products
    auto child = [&](int node, int tip, int idx, DvPart &M, DvPart &d1, DvPart &d2) {
        if (tip) {
            const unsigned code = codeAt(idx);
            M = column(a.PT64, node, code, 1.0);
            d1 = column(a.P1T, node, code, 0.0);   // (the rows of P' and P'' sum to zero)
            d2 = column(a.P2T, node, code, 0.0);
        } else {
            const DvPart x = loadPart(a.cl + region((size_t)idx));
            const Mat m0 = loadMat(matP(node)), m1 = loadMat(matD(node, 1)), m2 = loadMat(matD(node, 2));
            M = product(m0, x);
            d1 = product(m1, x);
            d2 = product(m2, x);
        }
    };
    DvPart root;
    {
        uint64_t rm = ~0ull;
        if (a.rootLeafRow >= 0) {
            const unsigned code = codeAt(a.rootLeafRow);
            rm = code < (unsigned)AA_S ? 1ull << code : code == TIP_ALL ? ~0ull : a.ambMask[code - AA_S];
        }
        for (int r = 0; r < 4; r++) root.x[r] = (rm >> (4 * q + r)) & 1ull ? a.rootPi[4 * q + r] : 0.0;
        root.x4 = (rm >> (16 + q)) & 1ull ? a.rootPi[16 + q] : 0.0;
    }
    DvPart prev0 = root, prev1 = root;
    for (int i = 0; i < a.nUnits; i++) {
        const DerivUnit u = derivUnit(a, i);
        if (nB + u.nKids > DERIV_BATCH) {
            flushBatch<4>(a, red, outIdx, nB);
            nB = 0;
        }
        DvPart av = root;
        if (u.src != DU_ROOT) {
            const Mat m = loadMat(matD(u.parent, 0));
            DvPart c2;
            if (u.src == DU_HBM) c2 = loadPart(a.cl2 + region((size_t)u.parent));
            else if (u.src == DU_PREV0) c2 = prev0;
            else c2 = prev1;
            av = product(m, c2);
        }
        DvPart M0, f0, s0;
        child(u.node[0], u.tip[0], u.idx[0], M0, f0, s0);
        if (u.nKids == 2) {
            DvPart M1, f1, s1;
            child(u.node[1], u.tip[1], u.idx[1], M1, f1, s1);
            prev0 = times(av, M1);
            prev1 = times(av, M0);
            branch(u.node[0], prev0, M0, f0, s0, u.out);
            branch(u.node[1], prev1, M1, f1, s1, u.out + 1);
        } else {
            for (int n = 0; n < u.nSib; n++) {
                const DerivSib sb = a.sibs[u.sibStart + n];
                const DvPart v = sb.kind == 0 ? column(a.PT64, sb.pnode, codeAt(sb.idx), 1.0)
                                              : product(loadMat(matP(sb.pnode)), loadPart(a.cl + region((size_t)sb.idx)));
                av = times(av, v);
            }
            prev0 = av;
            branch(u.node[0], prev0, M0, f0, s0, u.out);
        }
    }
    flushBatch<4>(a, red, outIdx, nB);
}

template <int SC>
__global__ __launch_bounds__(64 * DERIV_MAX_K) void k_edgeDerivs(DerivArgs a)
{
    constexpr int SM = SC ? SC : MAX_DIM;
    const int S = SC ? SC : a.dim;
    const int K = a.K;
    const int cat = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    const int p = blockIdx.x * 64 + lane;
    const size_t nPP = (size_t)a.nPatPad;
    const int SS = S * S;
    __shared__ double sL[DERIV_MAX_K][64], sF[DERIV_MAX_K][64], sS[DERIV_MAX_K][64];
    // element (slot, cat, pattern, state) of the down-pass partials
    auto clAt = [&](int slot, int s) -> double {
        const size_t o = (((size_t)slot * nPP + p) * K + cat) * S + s;
        return a.cl[o];
    };
    auto cl2At = [&](int node) -> double * { return a.cl2 + (((size_t)node * K + cat) * nPP + p) * S; };
    auto PT = [&](const double *base, int node) { return base + ((size_t)node * K + cat) * SS; };
    // mask of a tip code: 0 for none of S states (never), all bits for TIP_ALL
    auto tipMask = [&](unsigned code) -> uint64_t {
        if (code < (unsigned)S) return 1ull << code;
        if (code == TIP_ALL) return ~0ull;
        return a.ambMask[code - S];
    };
    const double *pi = a.rootPi;
    for (int e = 0; e < a.nOps; e++) {
        const DerivOp op = a.ops[e];
        double av[SM];
        if (op.flags & DOP_PARENT_ROOT) {
            // the root frequencies (Pf/p4_node.c:858-879); a leaf root's own
            // data enters here too
            uint64_t m = ~0ull;
            if (a.rootLeafRow >= 0) m = tipMask(a.tips[(size_t)a.rootLeafRow * nPP + p]);
#pragma unroll
            for (int s = 0; s < SM; s++)
                if (s < S) av[s] = ((m >> s) & 1ull) ? pi[s] : 0.0;
        } else {
            // up through the parent's branch: sum_from cl2[parent][from] P[from][s]
            // (Pf/p4_node.c:883-937)
            const double *c2 = cl2At(op.parent);
            const double *Pp = PT(a.PT64, op.parent);   // Pp[s][from] = P[from][s]
#pragma unroll
            for (int s = 0; s < SM; s++)
                if (s < S) {
                    double sum = 0.0;
                    for (int f = 0; f < S; f++) sum += Pp[s * S + f] * c2[f];
                    av[s] = sum;
                }
        }
        // times every sibling's message down its branch (Pf/p4_node.c:942-1018)
        for (int q = 0; q < op.nSib; q++) {
            const DerivSib sb = a.sibs[op.sibStart + q];
            const double *Ps = PT(a.PT64, sb.pnode);     // Ps[j][s] = P[s][j]
            if (sb.kind == 0) {
                const unsigned code = a.tips[(size_t)sb.idx * nPP + p];
                if (code == TIP_ALL) continue;
                const uint64_t m = tipMask(code);
#pragma unroll
                for (int s = 0; s < SM; s++)
                    if (s < S) {
                        double sum;
                        if (code < (unsigned)S) {
                            sum = Ps[code * S + s];
                        } else {
                            sum = 0.0;
                            for (int j = 0; j < S; j++)
                                if ((m >> j) & 1ull) sum += Ps[j * S + s];
                        }
                        av[s] *= sum;
                    }
            } else {
                double x[SM];
#pragma unroll
                for (int j = 0; j < SM; j++)
                    if (j < S) x[j] = clAt(sb.idx, j);
#pragma unroll
                for (int s = 0; s < SM; s++)
                    if (s < S) {
                        double sum = 0.0;
                        for (int j = 0; j < S; j++) sum += Ps[j * S + s] * x[j];
                        av[s] *= sum;
                    }
            }
        }
        double *c2n = cl2At(op.node);
#pragma unroll
        for (int s = 0; s < SM; s++)
            if (s < S) c2n[s] = av[s];
        // the site likelihood across the node's branch, and d/dt, d2/dt2
        const double *P0 = PT(a.PT64, op.node), *P1 = PT(a.P1T, op.node), *P2 = PT(a.P2T, op.node);
        double like = 0.0, first = 0.0, second = 0.0;
        if (op.flags & DOP_LEAF) {
            const unsigned code = a.tips[(size_t)op.idx * nPP + p];
            if (code < (unsigned)S) {
                for (int f = 0; f < S; f++) {
                    const double t2 = av[f];
                    like += t2 * P0[code * S + f];
                    first += t2 * P1[code * S + f];
                    second += t2 * P2[code * S + f];
                }
            } else if (code == TIP_ALL) {
                for (int f = 0; f < S; f++) {
                    const double t2 = av[f];
                    like += t2;
                    for (int t = 0; t < S; t++) {
                        first += t2 * P1[t * S + f];
                        second += t2 * P2[t * S + f];
                    }
                }
            } else {
                const uint64_t m = a.ambMask[code - S];
                for (int f = 0; f < S; f++) {
                    const double t2 = av[f];
                    for (int t = 0; t < S; t++)
                        if ((m >> t) & 1ull) {
                            like += t2 * P0[t * S + f];
                            first += t2 * P1[t * S + f];
                            second += t2 * P2[t * S + f];
                        }
                }
            }
        } else {
            double x[SM];
#pragma unroll
            for (int t = 0; t < SM; t++)
                if (t < S) x[t] = clAt(op.idx, t);
            for (int f = 0; f < S; f++)
                for (int t = 0; t < S; t++) {
                    const double t2 = av[f] * x[t];
                    like += t2 * P0[t * S + f];
                    first += t2 * P1[t * S + f];
                    second += t2 * P2[t * S + f];
                }
        }
        sL[cat][lane] = like;
        sF[cat][lane] = first;
        sS[cat][lane] = second;
        __syncthreads();
        if (cat == 0) {
            double lnL = 0.0, d1 = 0.0, d2 = 0.0;
            if (p < a.nPat) {
                double likeS = 0.0, firstS = 0.0, secondS = 0.0;
                for (int k = 0; k < K; k++) {
                    likeS += sL[k][lane];
                    firstS += sF[k][lane];
                    secondS += sS[k][lane];
                }
                siteDerivs(a, p, likeS, firstS, secondS, lnL, d1, d2);
            }
            for (int off = 32; off >= 1; off >>= 1) {
                lnL += __shfl_xor(lnL, off);
                d1 += __shfl_xor(d1, off);
                d2 += __shfl_xor(d2, off);
            }
            if (lane == 0) {
                double *o = a.partial + ((size_t)e * gridDim.x + blockIdx.x) * 3;
                o[0] = lnL;
                o[1] = d1;
                o[2] = d2;
            }
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(64) void k_derivReduce(const double *partial, int nBlk, const DerivOp *ops, int nOps,
                                                    double *out)
{
    const int e = blockIdx.x;
    const int lane = threadIdx.x;
    if (e >= nOps) return;
    double v[3];
    for (int c = 0; c < 3; c++) {
        double s = 0.0, comp = 0.0;
        for (int i = lane; i < nBlk; i += 64) {
            const double x = partial[((size_t)e * nBlk + i) * 3 + c];
            const double t = s + x;   // Neumaier
            if (fabs(s) >= fabs(x))
                comp += (s - t) + x;
            else
                comp += (x - t) + s;
            s = t;
        }
        double w = s + comp;
        for (int off = 32; off >= 1; off >>= 1) w += __shfl_xor(w, off);
        v[c] = w;
    }
    if (lane == 0) {
        const int node = ops[e].node;
        out[node * 3] = v[0];
        out[node * 3 + 1] = v[1];
        out[node * 3 + 2] = v[2];
    }
}

bool derivUsesUnits(int dim, int K, int layout)
{
    return K <= WAVE_MAX_K && ((dim == 4 && layout == CL_WAVE) || (dim == AA_S && layout == CL_TILED));
}

int derivBlockPatterns(int dim, int K, int layout)
{
    return derivUsesUnits(dim, K, layout) && layout == CL_TILED ? AA_TILE : 64;
}

hipError_t launchEdgeDerivs(const DerivArgs &a, int nBlocks, hipStream_t s)
{
    const dim3 block(64 * a.K);
    if (a.nUnits > 0) {
        const size_t lds = sizeof(double) * DERIV_BATCH * a.K * 192;
        constexpr int TIP_LDS_MAX_TAXA = 256;
        if (a.layout == CL_WAVE)
            hipLaunchKernelGGL(k_edgeDerivs4, dim3(nBlocks), block, lds, s, a);
        else if (a.nTax <= TIP_LDS_MAX_TAXA)
            hipLaunchKernelGGL(k_edgeDerivs20<true>, dim3(nBlocks), block, lds + (size_t)a.nTax * AA_TILE, s, a);
        else
            hipLaunchKernelGGL(k_edgeDerivs20<false>, dim3(nBlocks), block, lds, s, a);
    } else if (a.dim == 4)
        hipLaunchKernelGGL(k_edgeDerivs<4>, dim3(nBlocks), block, 0, s, a);
    else if (a.dim == 20)
        hipLaunchKernelGGL(k_edgeDerivs<20>, dim3(nBlocks), block, 0, s, a);
    else
        hipLaunchKernelGGL(k_edgeDerivs<0>, dim3(nBlocks), block, 0, s, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_derivReduce, dim3(a.nOps), dim3(64), 0, s, a.partial, nBlocks, a.ops, a.nOps, a.out);
    return hipGetLastError();
}

}  // namespace p4g
