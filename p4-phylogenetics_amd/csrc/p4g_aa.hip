// p4g_aa.hip -- 20-state pruning (protein) on the matrix cores, FP32 and
// FP64 partials, up to WAVE_MAX_K gamma categories.
//
// One wavefront per (tile of 16 site patterns, gamma category); the K
// category waves of a tile form a workgroup and meet only at the root.
// A partial (20 states x 16 patterns of one category) is five registers per
// lane: lane (q = l / 16, p = l % 16) holds states 4q .. 4q+3 and 16 + q of
// pattern p.  Per internal child, out = P x is five k-steps of
// v_mfma_f32_16x16x4f32 / v_mfma_f64_16x16x4f64 on two row tiles (states
// 0..15, and 16..19 padded to 16 rows), and the operands are ordered so that
// a result register is the next product's B operand as it stands:
//   k-step t < 4 contracts states {4q + t}, k-step 4 states {16 + q}, so B
//   of step t is register t of x;
//   the rows of A are permuted so that result register r of lane (q, p) is
//   state 4q + r (the FP32 result has row 4q + r there, the FP64 result row
//   q + 4r), and register 0 of the second row tile state 16 + q.
// A in that order is the operand table that the P kernels write (aaPaIndex):
// a lane's A operands are two vector and two scalar loads, contiguous over
// the wave, where the plain matrix takes ten gathers.  A tip child takes
// column `code` of P: its operands are loaded the same way, written to the
// wave's LDS scratch and gathered from there (gathers of 16-byte rows of P^T
// from memory, four lanes at a time, kept the texture path busy for 80% of
// the kernel).
#include "p4g_internal.h"
#include "p4g_site.h"

#include <algorithm>

namespace p4g {

typedef float aaF4 __attribute__((ext_vector_type(4)));
typedef double aaD4 __attribute__((ext_vector_type(4)));
template <typename T> struct AaT;
template <> struct AaT<float> {
    typedef aaF4 V4;
    typedef float VS __attribute__((ext_vector_type(4)));   // a 16-byte store
    static __device__ __forceinline__ V4 mfma(float a, float b, V4 c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
};
template <> struct AaT<double> {
    typedef aaD4 V4;
    typedef double VS __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ V4 mfma(double a, double b, V4 c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
};

// One child's operands: A of k-steps 0..3 and 4 of both row tiles; with G
// also its partial, if an earlier evaluation left it in HBM, and its tip code.
template <typename T> struct AaKid {
    typename AaT<T>::V4 a0, a1, x;
    T b0, b1, x4;
    int e;
    unsigned code;   // a tip's (with G)
};

// The node program runs one op at a time per wave; a full evaluation is a
// chain of some hundred ops, so what is not hidden inside an op is paid a
// hundred times.  An op therefore issues the NEXT op's loads (operands, and
// with G the partials of children that earlier evaluations left in HBM)
// before its own products, and its stores after them: the vector memory
// counter retires in issue order, so the next op's wait covers loads that
// are one op old and never the stores just issued.  For the compiler's wait
// counts to say so, every op issues the same loads and stores on every path,
// without a branch: the child's kind only selects addresses (a missing child
// repeats the first, a partial that is not in HBM reads a cached line), and
// the root, which stores nothing, is a step of its own after the loop.
// Results that a later op of the program reads go to an LDS slot of the wave
// (Sethi-Ullman order, see buildAaProgram) and always to HBM, where later
// evaluations read them.  There is no barrier in the chain: FP32 scale
// exponents are per (node, pattern, category), combined exactly at the root.
// Measured: 128 taxa, 19,877 patterns, 4 categories, FP32 300-322 us (430 with a
// barrier per op for a shared exponent, tip rows gathered from memory and
// loads waiting for stores); 48 taxa x 5,003 patterns FP64 77 us (1,124 on
// the general kernel, one lane per pattern and category).  The floors are
// the partials' stores (156 and 28 us at the rate of a large copy) and the
// padded matrix products (85 and 24 us).  What is left is issue: with the
// loads, the stores or the products taken out in turn each gives back 20 to
// 25% of the time, and one workgroup per CU alone takes 90 us of chain.
template <typename T, bool G, bool TIPLDS>
__device__ __forceinline__ void pruneAaBody(const PruneArgs &a, int tile, int nTiles)
{
    constexpr bool SCALE = sizeof(T) == 4;
    constexpr int V = 16 / (int)sizeof(T);   // values of a 16-byte store
    constexpr unsigned TS = (unsigned)sizeof(T);
    constexpr unsigned PB = AA_PART * TS;                    // bytes of a partial
    constexpr unsigned SB = PB + (SCALE ? AA_TILE * 4 : 0);  // and of an LDS slot: FP32 with the exponents
    constexpr unsigned MB = AA_MAT * TS;                     // bytes of a matrix
    constexpr unsigned MS = aaMatStride(SCALE) * TS;         // their stride in the table
    typedef typename AaT<T>::V4 V4;
    typedef typename AaT<T>::VS VS;
    __shared__ unsigned ambL[256];   // state masks of partial-ambiguity codes
    // [K][MB] a tip child's matrix (and at the end the root's sums),
    // [K][nLds][SB] slots, [nTax][16] tip codes
    extern __shared__ __align__(16) unsigned char aaSm[];
    const int tid = threadIdx.x;
    const int k = __builtin_amdgcn_readfirstlane(tid >> 6);   // category
    const int lane = tid & 63;
    const int q = lane >> 4, pl = lane & 15;
    const int K = a.K;
    const int p = tile * AA_TILE + pl;
    const size_t nPatPad = (size_t)a.nPatPad;
    const char *PA = (const char *)a.PA + (size_t)k * MS;     // this category's matrices
    char *tipM = (char *)aaSm + k * MB;                       // this wave's scratch and slots
    char *slots = (char *)aaSm + K * MB + (unsigned)(k * a.nLds) * SB;
    uint8_t *tipL = (uint8_t *)aaSm + K * MB + (unsigned)(K * a.nLds) * SB;
    // (a dirty path has a few ops: it loads its tip codes with the operands
    // and its launch waits for nothing)
    if (TIPLDS && !G)
        for (int t = tid; t < a.nTax; t += blockDim.x)
            *reinterpret_cast<uint4 *>(tipL + t * AA_TILE) =
                *reinterpret_cast<const uint4 *>(a.tips + (size_t)t * nPatPad + (size_t)tile * AA_TILE);
    if (a.nAmb)
        for (int j = tid; j < a.nAmb && j < 256; j += blockDim.x) ambL[j] = (unsigned)a.ambMask[j];
    if ((TIPLDS && !G) || a.nAmb) __syncthreads();
    const uint8_t *tips = a.tips + (size_t)tile * AA_TILE;
    auto tipCode = [&](int row) -> unsigned {
        if (TIPLDS && !G) return (unsigned)tipL[row * AA_TILE + pl];
        return (unsigned)(tips + (size_t)row * nPatPad)[(unsigned)pl];
    };
    // lane offsets: a matrix's operands (row pl of the second row tile holds
    // state 16 + i1), the same values in the scratch matrix [state][20], a
    // tip's column there, a partial, its exponents (in units of the tile)
    const int i1 = SCALE ? pl >> 2 : pl & 3;
    const int row0 = SCALE ? pl : (pl & 3) * 4 + (pl >> 2);
    const unsigned offA0 = (unsigned)lane * 4u * TS, offB0 = (256u + lane) * TS;
    const unsigned offA1 = (320u + (q * 4 + i1) * 4u) * TS, offB1 = (384u + q * 4 + i1) * TS;
    const unsigned rowA0 = (20u * row0 + 4u * q) * TS, rowA1 = (20u * (16 + i1) + 4u * q) * TS;
    const unsigned lane16 = (unsigned)lane * 16u, laneT = (unsigned)lane * TS;
    char *clT = (char *)a.cl + (size_t)tile * K * SB + (size_t)k * PB;   // + slot offset: this wave's partial
    const unsigned offE = (unsigned)(K - k) * PB + (unsigned)k * (AA_TILE * 4u) + (unsigned)pl * 4u;
    const V4 zero = {T(0), T(0), T(0), T(0)};
    typedef int i8v __attribute__((ext_vector_type(8)));
    typedef const __attribute__((address_space(4))) i8v ci8v;
    ci8v *recG = (ci8v *)a.aaRec;
    auto recAt = [&](int i) -> AaRec {
        const i8v r = recG[i];
        return AaRec{(unsigned)r[0], r[1], (unsigned)r[2], r[3], (unsigned)r[4], r[5], r[6], r[7]};
    };
    typedef int i4v __attribute__((ext_vector_type(4)));
    typedef const __attribute__((address_space(4))) i4v ci4v;
    ci4v *kidsG = (ci4v *)a.kids;
    auto kidAt = [&](int i) -> KidRec {
        const i4v r = kidsG[i];
        return KidRec{r.x, r.y, r.z, r.w};
    };
    auto kindOf = [](const AaRec &r, int c) { return (r.info >> (2 + 2 * c)) & 3; };
    auto kidsOf = [](const AaRec &r) { return r.info >> 6; };
    auto argOf = [](const AaRec &r, int c) { return c ? r.arg1 : r.arg0; };
    // (a wave-uniform base and an unsigned 32-bit lane offset: the
    // scalar-base form of the memory instructions)
    auto region = [&](int arg) -> char * { return clT + ((size_t)(unsigned)arg << AA_SLOT_SHIFT); };
    auto loadPart = [&](const char *R, V4 &x, T &x4) {
#pragma unroll
        for (int r = 0; r < 4; r += V) {
            const VS v = *(const VS *)(R + (r / V) * 1024 + lane16);
            for (int i = 0; i < V; i++) x[r + i] = v[i];
        }
        x4 = *(const T *)(R + 256 * TS + laneT);
    };
    auto loadMat = [&](const char *M, AaKid<T> &kd) {
        kd.a0 = *(const V4 *)(M + offA0);
        kd.b0 = *(const T *)(M + offB0);
        kd.a1 = *(const V4 *)(M + offA1);
        kd.b1 = *(const T *)(M + offB1);
    };
    // one op's loads
    auto issue = [&](const AaRec &op, AaKid<T> (&kd)[2]) {
#pragma unroll
        for (int c = 0; c < 2; c++) {
            loadMat(PA + ((size_t)(c ? op.mat1 : op.mat0) << 6), kd[c]);
            if (G) {
                const bool hbm = kindOf(op, c) == 1;
                const char *R = hbm ? region(argOf(op, c)) : PA;
                loadPart(R, kd[c].x, kd[c].x4);
                if (SCALE) kd[c].e = *(const int *)(R + (hbm ? offE : 0u));
                kd[c].code = tipCode(kindOf(op, c) == 0 ? argOf(op, c) : 0);
            }
        }
    };
    // The scratch matrix is written by some lanes and read by others of the
    // wave.  The hardware keeps a wave's LDS operations in order; the fence,
    // which has no instruction of its own, keeps the compiler from reordering
    // them (128 taxa x 19,877 patterns FP32 313 us with it and without; four
    // generations of 24 partitions x 4 chains 2.87 ms with and without).
    auto waveLdsFence = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    };
    // a tip child: column `code` of its matrix, 1 for every state if all are
    // allowed, the sum of the allowed columns for a partial ambiguity
    auto tipCol = [&](const AaKid<T> &kd, unsigned code, V4 &v, T &v4) {
        if constexpr (SCALE) {
            *(V4 *)(tipM + rowA0) = kd.a0;
            *(V4 *)(tipM + rowA1) = kd.a1;   // (four lanes each, the same values)
        } else {
            *(VS *)(tipM + rowA0) = VS{kd.a0[0], kd.a0[1]};
            *(VS *)(tipM + rowA0 + 16u) = VS{kd.a0[2], kd.a0[3]};
            *(VS *)(tipM + rowA1) = VS{kd.a1[0], kd.a1[1]};
            *(VS *)(tipM + rowA1 + 16u) = VS{kd.a1[2], kd.a1[3]};
        }
        *(T *)(tipM + rowA0 + (16u - 3u * q) * TS) = kd.b0;   // column 16 + q
        *(T *)(tipM + rowA1 + (16u - 3u * q) * TS) = kd.b1;
        waveLdsFence();   // (before the columns are read)
        auto colAt = [&](unsigned j, V4 &w, T &w4) {
            const char *C = tipM + (80u * q + j) * TS;
#pragma unroll
            for (int r = 0; r < 4; r++) w[r] = *(const T *)(C + 20 * r * TS);
            w4 = *(const T *)(tipM + (320u + 20u * q + j) * TS);
        };
        colAt(min(code, (unsigned)AA_S - 1u), v, v4);
        if (__builtin_amdgcn_ballot_w64(code >= (unsigned)AA_S)) {
            if (code == TIP_ALL) {
                v = V4{T(1), T(1), T(1), T(1)};
                v4 = T(1);
            } else if (code >= (unsigned)AA_S) {
                const unsigned m = ambL[code - AA_S];
                v = zero;
                v4 = T(0);
#pragma unroll 1
                for (unsigned j = 0; j < (unsigned)AA_S; j++)
                    if ((m >> j) & 1u) {
                        V4 w;
                        T w4;
                        colAt(j, w, w4);
                        v += w;
                        v4 += w4;
                    }
            }
        }
        waveLdsFence();   // (before the scratch is written again)
    };
    auto product = [&](const AaKid<T> &kd, const V4 &x, T x4, V4 &v, T &v4) {
        V4 d0 = zero, d1 = zero;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            d0 = AaT<T>::mfma(kd.a0[t], x[t], d0);
            d1 = AaT<T>::mfma(kd.a1[t], x[t], d1);
        }
        d0 = AaT<T>::mfma(kd.b0, x4, d0);
        d1 = AaT<T>::mfma(kd.b1, x4, d1);
        v = d0;
        v4 = d1[0];
    };
    auto loadSlot = [&](int arg, V4 &x, T &x4, int &e) {
        loadPart(slots + arg, x, x4);
        if (SCALE) e += *(const int *)(slots + arg + PB + (unsigned)pl * 4u);
    };
    auto slotKid = [&](const AaKid<T> &kd, int arg, V4 &v, T &v4, int &e) {
        V4 x;
        T x4;
        loadSlot(arg, x, x4, e);
        product(kd, x, x4, v, v4);
    };
    auto anyKid = [&](const AaKid<T> &kd, int kind, int arg, V4 &v, T &v4, int &e) {
        if (kind == 0) {
            tipCol(kd, G ? kd.code : tipCode(arg), v, v4);
        } else if (kind == 2) {
            slotKid(kd, arg, v, v4, e);
        } else if (G && kind == 1) {
            if (SCALE) e += kd.e;
            product(kd, kd.x, kd.x4, v, v4);
        } else {   // computed in this program, no slot: this wave's own stores
            V4 x;
            T x4;
            loadPart(region(arg), x, x4);
            if (SCALE) e += *(const int *)(region(arg) + offE);
            __builtin_amdgcn_s_waitcnt(VMCNT0);
            product(kd, x, x4, v, v4);
        }
    };
    V4 acc = zero;
    T acc4 = T(0);
    int e = 0;
    AaKid<T> A[2], B[2];
    AaRec op = recAt(0), nx = recAt(min(1, a.nOps - 1));
    issue(op, A);
    // op `op` from the operands cur; unless it is the last, the loads of
    // `nx` into nxt and the record after it
    auto step = [&](int i, bool last, AaKid<T> (&cur)[2], AaKid<T> (&nxt)[2]) {
        AaRec n2 = nx;
        if (!last) {
            issue(nx, nxt);
            n2 = recAt(min(i + 2, a.nOps - 1));
        }
        e = 0;
        V4 v;
        T v4;
        const int type = op.info & 3;
        if (!last && type == AA_TT) {
            // (LDS reads that the fences of a tip's scratch need not hold up
            // stand before it)
            const unsigned c0 = G ? cur[0].code : tipCode(op.arg0), c1 = G ? cur[1].code : tipCode(op.arg1);
            tipCol(cur[0], c0, acc, acc4);
            tipCol(cur[1], c1, v, v4);
            acc *= v;
            acc4 *= v4;
        } else if (!last && type == AA_TL) {
            const unsigned c0 = G ? cur[0].code : tipCode(op.arg0);
            V4 x;
            T x4;
            loadSlot(op.arg1, x, x4, e);
            tipCol(cur[0], c0, acc, acc4);
            product(cur[1], x, x4, v, v4);
            acc *= v;
            acc4 *= v4;
        } else if (!last && type == AA_LL) {
            slotKid(cur[0], op.arg0, acc, acc4, e);
            slotKid(cur[1], op.arg1, v, v4, e);
            acc *= v;
            acc4 *= v4;
        } else {
            // (children past the second, as a root's third, load here: the
            // first of them before the products of the first two)
            const int nK = kidsOf(op);
            AaKid<T> kk;
            KidRec kr{};
            auto extra = [&](int c) {
                kr = kidAt(op.kidStart + c);
                loadMat(PA + (size_t)kr.pnode * K * MS, kk);
                if (G) {
                    const bool hbm = kr.kind == 1;
                    const char *R = hbm ? region(kr.idx) : PA;
                    loadPart(R, kk.x, kk.x4);
                    if (SCALE) kk.e = *(const int *)(R + (hbm ? offE : 0u));
                    kk.code = tipCode(kr.kind == 0 ? kr.idx : 0);
                }
            };
            if (nK > 2) extra(2);
            anyKid(cur[0], kindOf(op, 0), op.arg0, acc, acc4, e);
            if (nK > 1) {
                anyKid(cur[1], kindOf(op, 1), op.arg1, v, v4, e);
                acc *= v;
                acc4 *= v4;
            }
            for (int c = 2; c < nK; ++c) {
                if (c > 2) extra(c);
                anyKid(kk, kr.kind, kr.idx, v, v4, e);
                acc *= v;
                acc4 *= v4;
            }
            if (nK > 2) __builtin_amdgcn_s_waitcnt(VMCNT0);
        }
        if (SCALE) {
            // rescale by the pattern's largest entry, an exact power of two.
            // Some pattern of the tile needs it at most ops, so there is no
            // branch; the maximum over the pattern's four lanes by lane swaps.
            float m = fmaxf(fmaxf(fmaxf(acc[0], acc[1]), fmaxf(acc[2], acc[3])), acc4);
            const unsigned u = __float_as_uint(m);
            const auto s16 = __builtin_amdgcn_permlane16_swap(u, u, false, false);
            m = fmaxf(__uint_as_float(s16[0]), __uint_as_float(s16[1]));
            const unsigned w = __float_as_uint(m);
            const auto s32 = __builtin_amdgcn_permlane32_swap(w, w, false, false);
            m = fmaxf(__uint_as_float(s32[0]), __uint_as_float(s32[1]));
            const int ex = m < SCALE_THRESH ? __builtin_amdgcn_frexp_expf(m) : 0;   // 0 for m = 0
#pragma unroll
            for (int r = 0; r < 4; r++) acc[r] = __builtin_amdgcn_ldexpf(acc[r], -ex);
            acc4 = __builtin_amdgcn_ldexpf(acc4, -ex);
            e -= ex;
        }
        if (!last) {
            char *D = region((int)op.dst);
            VS w[4 / V];
#pragma unroll
            for (int r = 0; r < 4; r++) w[r / V][r % V] = acc[r];
            if (op.ld >= 0) {
                char *L = slots + op.ld;
#pragma unroll
                for (int j = 0; j < 4 / V; j++) *(VS *)(L + j * 1024 + lane16) = w[j];
                *(T *)(L + 256 * TS + laneT) = acc4;
                if (SCALE) *(int *)(L + PB + (unsigned)pl * 4u) = e;   // the pattern's four lanes, one value
            }
            // Stored past L2 (non-temporal): nothing in this launch reads them
            // there, and they would evict the P table every op reads (four
            // generations of dirty paths, 24 parts x 4 chains: 4.50 ms against
            // 4.63 cached)
#pragma unroll
            for (int j = 0; j < 4 / V; j++) __builtin_nontemporal_store(w[j], (VS *)(D + j * 1024 + lane16));
            __builtin_nontemporal_store(acc4, (T *)(D + 256 * TS + laneT));
            if (SCALE) __builtin_nontemporal_store(e, (int *)(D + offE));
        }
        op = nx;
        nx = n2;
    };
    // The root, the last op, is a step of its own: inside the loop every
    // step then issues the same loads and the same stores
    const int nLast = a.nOps - 1;
    int i = 0;
    for (; i + 2 <= nLast; i += 2) {
        step(i, false, A, B);
        step(i + 1, false, B, A);
    }
    if (i < nLast) {
        step(i, false, A, B);
#pragma unroll
        for (int c = 0; c < 2; c++) A[c] = B[c];
    }
    step(nLast, true, A, B);
    // this category's sum_s pi_s cl_s across the four lanes of the pattern,
    // then wave 0 adds the categories
    const double *pi = a.rootPi;
    uint64_t msk = ~0ull;
    if (a.rootLeafRow >= 0) {
        const unsigned code = tipCode(a.rootLeafRow);
        msk = code < (unsigned)AA_S ? (1ull << code) : code == TIP_ALL ? ~0ull : a.ambMask[code - AA_S];
    }
    double Lk = 0.0;
#pragma unroll
    for (int r = 0; r < 4; r++)
        if ((msk >> (4 * q + r)) & 1ull) Lk += pi[4 * q + r] * (double)acc[r];
    if ((msk >> (16 + q)) & 1ull) Lk += pi[16 + q] * (double)acc4;
    Lk += __shfl_xor(Lk, 16);
    Lk += __shfl_xor(Lk, 32);
    if (q == 0) {
        ((double *)tipM)[pl] = Lk;
        ((int *)tipM)[2 * AA_TILE + pl] = rootExponent<SCALE>(Lk, e);
    }
    __syncthreads();
    double contrib = 0.0;
    int bad = 0;
    if (k == 0 && q == 0) {
        int eL;
        const double L = sumCategories<SCALE>(
            K, [&](int kk) { return ((const double *)(aaSm + kk * MB))[pl]; },
            [&](int kk) { return ((const int *)(aaSm + kk * MB))[2 * AA_TILE + pl]; }, eL);
        siteLogLike<SCALE>(a, L, eL, p, K, pi, contrib, bad);
    }
    if (k == 0) finishSiteSumWave(a, contrib, bad, tile, nTiles);
}

// Waves per SIMD: FP32 four (at most 128 VGPRs; five, at 96, spills and is no
// faster), FP64 three, with G two (its operands and slots are twice the size)
template <typename T, bool G> constexpr int aaWaves() { return sizeof(T) == 4 ? 4 : G ? 2 : 3; }

template <typename T, bool G, bool TIPLDS>
__global__ __launch_bounds__(64 * WAVE_MAX_K) __attribute__((amdgpu_waves_per_eu(aaWaves<T, G>())))
void k_pruneAa(PruneArgs a)
{
    pruneAaBody<T, G, TIPLDS>(a, blockIdx.x, gridDim.x);
}

// (items that could stage their tip codes are read from global memory by
// the other instance, which ignores tipLds)
template <typename T, bool G, bool TIPLDS>
__global__ __launch_bounds__(64 * WAVE_MAX_K) __attribute__((amdgpu_waves_per_eu(aaWaves<T, G>())))
void k_pruneAaBatch(const PruneArgs *args, const int *blockItem)
{
    const int item = blockItem[2 * blockIdx.x];
    const int local = blockItem[2 * blockIdx.x + 1];
    const PruneArgs a = args[item];
    pruneAaBody<T, G, TIPLDS>(a, local, a.nPatPad / AA_TILE);
}

bool pruneUsesMfma(int dim, int K, int precision) { return dim == AA_S && K <= WAVE_MAX_K; }

// LDS slot file: per slot, K x 320 values (FP32: and K x 16 exponents).
// Five slots for K = 4 are 26 KB in FP32; with the tip matrices (6 KB) and
// the tip codes of 128 taxa (2 KB) four workgroups, the four waves per SIMD
// the kernel is built for, fit a CU's 160 KB.  In FP64 five are 50 KB, and two
// workgroups fit.
static int g_aaLdsSlots = 5;
constexpr size_t AA_LDS_BUDGET = 28 * 1024, AA_LDS_BUDGET64 = 51 * 1024;
static size_t aaSlotBytes(int K, int precision)
{
    return (size_t)K * aaPartBytes(precision == FP32);
}
void setAaLdsSlots(int n) { g_aaLdsSlots = n < 0 ? 0 : n; }
int pruneAaLdsSlots(int K, int precision)
{
    const size_t fit = (precision == FP32 ? AA_LDS_BUDGET : AA_LDS_BUDGET64) / aaSlotBytes(K, precision);
    return (int)std::min<size_t>((size_t)g_aaLdsSlots, fit);
}
// the tile's tip codes go to LDS up to this many taxa (4 KB)
constexpr int AA_TIP_LDS_MAX_TAXA = 256;
bool pruneAaTipLds(int nTax) { return nTax <= AA_TIP_LDS_MAX_TAXA; }
size_t pruneAaLdsBytes(int K, int nLds, int tipTaxa, int precision)
{
    return (size_t)K * AA_MAT * (precision == FP32 ? 4 : 8) + (size_t)nLds * aaSlotBytes(K, precision) +
           (size_t)tipTaxa * AA_TILE;
}
bool pruneAaItemOk(const PruneArgs &a, int precision)
{
    return a.K >= 1 && a.K <= WAVE_MAX_K && a.nLds >= 0 && a.nLds <= pruneAaLdsSlots(a.K, precision) &&
           (!a.tipLds || pruneAaTipLds(a.nTax)) && a.aaRec != nullptr && a.PA != nullptr && a.nOps >= 1;
}

template <typename T>
static hipError_t launchAaT(const PruneArgs &a, int nBlocks, size_t lds, hipStream_t s)
{
    const dim3 g(nBlocks), b(64 * a.K);
    if (a.aaHbm) {
        if (a.tipLds) hipLaunchKernelGGL((k_pruneAa<T, true, true>), g, b, lds, s, a);
        else hipLaunchKernelGGL((k_pruneAa<T, true, false>), g, b, lds, s, a);
    } else {
        if (a.tipLds) hipLaunchKernelGGL((k_pruneAa<T, false, true>), g, b, lds, s, a);
        else hipLaunchKernelGGL((k_pruneAa<T, false, false>), g, b, lds, s, a);
    }
    return hipGetLastError();
}

hipError_t launchPruneAa(const PruneArgs &a, int precision, int nBlocks, hipStream_t s)
{
    if (nBlocks < 1 || nBlocks != a.nPatPad / AA_TILE || !pruneAaItemOk(a, precision)) return hipErrorInvalidValue;
    const size_t lds = pruneAaLdsBytes(a.K, a.nLds, a.tipLds ? a.nTax : 0, precision);
    return precision == FP32 ? launchAaT<float>(a, nBlocks, lds, s) : launchAaT<double>(a, nBlocks, lds, s);
}

template <typename T>
static hipError_t launchAaBatchT(const PruneArgs *d, const int *bi, int nBlocks, int K, bool hbm, size_t lds,
                                 bool tipLds, hipStream_t s)
{
    const dim3 g(nBlocks), b(64 * K);
    if (hbm) {
        if (tipLds) hipLaunchKernelGGL((k_pruneAaBatch<T, true, true>), g, b, lds, s, d, bi);
        else hipLaunchKernelGGL((k_pruneAaBatch<T, true, false>), g, b, lds, s, d, bi);
    } else {
        if (tipLds) hipLaunchKernelGGL((k_pruneAaBatch<T, false, true>), g, b, lds, s, d, bi);
        else hipLaunchKernelGGL((k_pruneAaBatch<T, false, false>), g, b, lds, s, d, bi);
    }
    return hipGetLastError();
}

// every item of the launch has exactly K categories and the same hbm (the
// batch groups by both); lds: the largest slot file and tip codes of its
// items; tipLds: every item stages its tip codes
hipError_t launchPruneAaBatch(const PruneArgs *d, const int *bi, int nBlocks, int K, int precision, bool hbm,
                              size_t lds, bool tipLds, hipStream_t s)
{
    if (K < 1 || K > WAVE_MAX_K ||
        lds > pruneAaLdsBytes(K, pruneAaLdsSlots(K, precision), AA_TIP_LDS_MAX_TAXA, precision))
        return hipErrorInvalidValue;
    return precision == FP32 ? launchAaBatchT<float>(d, bi, nBlocks, K, hbm, lds, tipLds, s)
                             : launchAaBatchT<double>(d, bi, nBlocks, K, hbm, lds, tipLds, s);
}

}  // namespace p4g
